// Chunked Palimpsa backward, local pass: chunk_bwd_tile_kernel (instantiated in chunk_bwd_tile_*.hip).
//
// Per (tile of 64 tokens, head), from the state at the start of the tile: dq, the tile's own parts of dv, db, dk and of
// the gate's gradient, and the carry R_loc = f_first dM_first that the tile hands to its predecessor (chunk_bwd.hip).
// With G_t = scale do_t q_t^T, r = 1 / I_t and mu = M_t r, per state entry and token (the reference's reverse
// recurrence, chunk_palimpsa_forgetting_scalar.py:360-434):
//   forward  M <- f_t M + v_t k_t        J <- f_t J + b_t k_t^2   (J = I - Ip)
//   reverse  dM <- f_{t+1} dM + G r      dJ <- f_{t+1} dJ - G r mu
//   dq = sum_d scale do mu    dv = sum_n dM k    db = sum_n dJ k^2    dk = sum_d dM v + 2 k sum_d dJ b
// all of it token by token in fp32 on the vector units.
//
// The reverse sweep needs mu and r of every token in reverse order.  A tile is worked in steps of kG tokens from its
// end: the state before a step is recomputed from the state before its half of the tile by two matrix products over at
// most 32 tokens (k weighted by the decay against v, and k^2 against b; bf16 operands, two halves of each for fp32
// rows), the step's tokens are advanced forward leaving their states in registers, then worked in reverse.
//
// Scaled form (bf16 rows without the uncertainty output): with F_t the decay since the start of the step, M = F M', J = F J' and
// dM' = F dM, dJ' = F dJ
//   M' <- M' + (v_t / F_t) k_t    J' <- J' + (b_t / F_t) k_t^2    r' = 1 / (J' + Ip / F_t) = F_t r    mu = M' r'
//   dM' <- dM' + (do_t r') q_t    dJ' <- dJ' - (do_t r' mu) q_t    dv = (1 / F_t) sum_n dM' k,  dk = sum_d dM' (v / F) + ...
// so that a decay costs nothing per entry (17 instructions instead of 20; dM, dJ take the step's whole decay once), v / F and
// b / F are formed where the rows are staged, and F dM of the step's first token is the carry that the step before it takes.
// A tile is worked in plain form where a step decays below 2^-48, the decay since the start of a step exceeds 1, or rows, the state
// at its start or Ip are large (kMaxV and so on): then nothing over F leaves fp32's range, and nothing times F that counts.  (Two
// copies of the loop: both forms of a step in one loop keep too many registers.)
// 1 / F (a product and a hardware reciprocal, one ulp) and the products with it round once more: under the rounding of bf16 rows that is
// nothing (gradients against a float64 recurrence: the same three digits), but fp32 rows' gradients were up to 12 % further off where
// tokens decay by e^-2 or more (dk, 96x96 and 64x64), for 4 % of the time (64x64 B=8 T=2048 H=8 444 us, plain 458).  With the
// uncertainty the scaled form was no faster (bf16 64x64 H=8 490 us, plain 459), and dovar / F needs a bound of its own.
//
// What bounds it: vector issue, of waves that are two to a SIMD (the registers).  By the counters 24 instructions per entry and
// token at 64x64, 16 of them fp32 arithmetic of the entry and one a reciprocal, 7 for the sums over lanes, the recomputed states,
// staging and the sums over waves; a wave alone issues one per 5 cycles, and waits (reads of LDS, barriers, what the other
// wave has in the way) for two fifths of its time.  B=8 T=2048 H=12 64x64 554 -> 515 us, 48x48 H=16 549 -> 491, 48x96 4 x 1531 456 -> 392,
// packed 32768 tokens 96x96 4050 -> 3600 (plain form throughout -> this, with the fetches and stores below), with every tile in plain
// form 552, 532, 428 and 3840; fp32 rows 64x64 H=8 604 -> 458 (slices of 32 value rows, fetches and stores), with the uncertainty bf16 64x64
// H=8 512 -> 459.  As products on the matrix cores (12 prefix and 12 suffix instructions of 16 cycles per 16 entries of a lane, operands
// exchanged through LDS between waves of different roles) the same pass took 822 us at 64x64.
// Waits that the compiler places (counted in order, for loads and stores alike) cost more than instructions here: rows are
// fetched by every wave on one path, nothing is stored between a fetch and its use, and a token's dq, dk leave from the four
// lanes of a quad that would otherwise hold the same sum, four tokens a store.
// Layout: a wave holds 4 DN columns x 16 DT rows of the state, a lane DN neighbouring columns of DT rows, the layout in
// which the matrix products leave the state (DN = 3: the fourth operand row of a lane group is empty), so that a head of
// 48 columns loads all four SIMDs.  As many tokens per step as the registers hold: the fixed cost of a step is what small
// pieces pay (profiles/tile_kernel_pieces.txt).
//
// Gate: gamma_t = f_t (<dM_t, M_{t-1}> + <dJ_t, J_{t-1}>) = <dM'_t, M'_{t-1}> + <dJ'_t, J'_{t-1}>, formed as it stands: where a
// token decays strongly, what is left of the state is of the order of f_t, and so is gamma.  (gamma_{t+1} + Ip sum(G r mu) -
// <dv_t, v_t> - <db_t, b_t> is the same number for one addition, but as a difference of terms of order 1: with every fifth token
// at f = e^-18 the gradients of these tokens were off by 200 times their size in fp32.)  The first token of a step sees the
// state after the step before it in time: its gamma is formed there, that of the tile's first token from the state at
// the start of the tile.
#pragma once
#include <type_traits>

#include "chunk_bwd.h"
#include "pal_host.h"
#include "pal_profile.h"

namespace pal {

// The sums of a token over lanes by DPP with a bank mask (see pair_bit3), in three stages so that the next token's arithmetic can be placed between them (each
// stage is a chain of dependent instructions).
//   o[2 DN] (dq, then dk of the lane's columns): over the 16 lanes of a row but for its quads, over which four tokens are
//     summed together (quad_tokens).  Lane bit 3 selects dq or dk, of which z0 is the first (lane bit 2 clear) or the third
//     column, z1 the second or the fourth (DN = 3: the second in both).
//   p[4], q[4] (dv, db of the lane's rows; DT < 3: dv0, dv1 or 0, db0, db1 or 0 in p): over the four rows of lanes, the
//     lanes of row g get p_g and q_g.
template <int DT, int DN>
struct TokSums {
  float o[2 * DN], p[4], q[4], X;
  float y0, y1, y2, y3, z0, z1;
  __device__ __forceinline__ void stage_a() {
    if constexpr (DN == 4) {
      asm("s_nop 1\n\t"
          "v_add_f32_dpp %0, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %1, %5, %5 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %2, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %3, %7, %7 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
          "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
          "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
          "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc"
          : "=&v"(y0), "=&v"(y1), "=&v"(y2), "=&v"(y3)
          : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "v"(o[4]), "v"(o[5]), "v"(o[2 * DN - 2]), "v"(o[2 * DN - 1]));
    } else {
      asm("s_nop 1\n\t"
          "v_add_f32_dpp %0, %3, %3 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %1, %4, %4 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %2, %5, %5 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
          "v_add_f32_dpp %0, %6, %6 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
          "v_add_f32_dpp %1, %7, %7 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
          "v_add_f32_dpp %2, %8, %8 row_ror:8 row_mask:0xf bank_mask:0xc"
          : "=&v"(y0), "=&v"(y1), "=&v"(y2)
          : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "v"(o[4]), "v"(o[5]));
      y3 = y1;
    }
    if constexpr (DT >= 3)
      asm("s_nop 1\n\t"
          "v_permlane32_swap_b32 %0, %2\n\t"
          "v_permlane32_swap_b32 %1, %3\n\t"
          "v_permlane32_swap_b32 %4, %6\n\t"
          "v_permlane32_swap_b32 %5, %7"
          : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]), "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]));
    else
      asm("s_nop 1\n\t"
          "v_permlane32_swap_b32 %0, %2\n\t"
          "v_permlane32_swap_b32 %1, %3" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
  }
  __device__ __forceinline__ void stage_b() {
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %2, %2 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %3, %3 row_shl:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %0, %4, %4 row_shr:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %1, %5, %5 row_shr:4 row_mask:0xf bank_mask:0xa"
        : "=&v"(z0), "=&v"(z1) : "v"(y0), "v"(y1), "v"(y2), "v"(y3));
    p[0] += p[2];
    p[1] += p[3];
    if constexpr (DT >= 3) {
      q[0] += q[2];
      q[1] += q[3];
      asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3" : "+v"(p[0]), "+v"(p[1]), "+v"(q[0]), "+v"(q[1]));
    } else {
      asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(p[0]), "+v"(p[1]));
    }
  }
  __device__ __forceinline__ void stage_c() {
    p[0] += p[1];
    if constexpr (DT >= 3) q[0] += q[1];
  }
};
// the values of four tokens, each summed over the quad: lane u of the quad gets token u's
__device__ __forceinline__ float quad_tokens(int lane, float z0, float z1, float z2, float z3) {
  const bool b0 = lane & 1, b1 = lane & 2;
  const float x = (b0 ? z1 : z0) + quad_move<0xB1>(b0 ? z0 : z1), y = (b0 ? z3 : z2) + quad_move<0xB1>(b0 ? z2 : z3);
  return (b1 ? y : x) + quad_move<0x4E>(b1 ? x : y);
}
template <int DT>
__device__ __forceinline__ void lds_vals(const float* p, float* out) {
  if constexpr (DT >= 3) {
    const f32x4 x = *(const f32x4*)p;
#pragma unroll
    for (int e = 0; e < DT; ++e) out[e] = x[e];
  } else if constexpr (DT == 2) {
    const f32x2 x = *(const f32x2*)p;
    out[0] = x[0]; out[1] = x[1];
  } else {
    out[0] = *p;
  }
}

// what both sweeps read of a token: its k, v and b (over F in scaled form), and in plain form f
template <int DT, bool SCALED, int DS>
struct TokFwd {
  f32x4 k;
  float v[DT], b[DT], f;
  __device__ __forceinline__ void load(const float* kq, const float* vb, const float* dec, int plane) {
    if constexpr (!SCALED) f = dec[DS - 1];
    k = *(const f32x4*)kq;
    lds_vals<DT>(vb, v);
    lds_vals<DT>(vb + plane, b);
  }
};
// and the reverse sweep: q, do, (dovar), Ip and 1 / F or, in plain form, the next token's f
template <int DT, bool VAR, bool SCALED, int DS>
struct TokRev {
  f32x4 q;
  float d_o[DT], d_ov[VAR ? DT : 1], ip, inv;
  __device__ __forceinline__ void load(const float* kq, const float* vb, const float* dec, float Ip, int plane) {
    q = *(const f32x4*)(kq + 16);
    lds_vals<DT>(vb + 2 * plane, d_o);
    if constexpr (VAR) lds_vals<DT>(vb + 3 * plane, d_ov);
    ip = SCALED ? dec[0] : Ip;
    inv = dec[SCALED ? 1 : 2 * DS - 1];
  }
};

// Least decay over a step, and largest entries of v, b, k and of the state at the tile's start (and Ip), for the scaled form.  At
// the upper end nothing over F then leaves fp32's range (M' < 2^80, J' + Ip / F < 2^68).  At the lower end a tile's precisions stay below
// 2^16 + 64 x 2^4 x 2^8 < 2^19, so that r' = F r is at least 2^-67, and what is left of a gradient's term do r mu q after F has
// 12 bits above fp32's last one (2^-149) for terms down to 2^-89: r, mu of 2^-19, 2^-22 and q of 2^-4 leave do down to 2^-44.
// (A step of eight tokens at gates of 0.5 and a rate of 4.5, strong for a layer, decays by 2^26 on average.)
constexpr float kMinStepDecay = 0x1p-48f, kMaxV = 0x1p20f, kMaxB = 0x1p4f, kMaxK = 0x1p4f, kMaxState = 0x1p16f;

// Waves per SIMD that a lane's E state entries leave registers for.  Three entries (48 columns by 16 rows) take 131 to 136 and are held to
// 128 (`four`), for up to four spilled: 80x80 at 192 tiles x heads 138 -> 123 us, with the uncertainty 172 -> 154, at 384 242 -> 232; but
// not where that spills 14 to 27: earlier launches' sums added, fp32 rows with the uncertainty.
constexpr int tile_waves(int E, bool four) { return E > 4 ? 2 : E == 3 && four ? 4 : 3; }

template <typename TIn, int DT, int DN, int NBW, bool VAR, int SLICE>
__global__ __attribute__((amdgpu_flat_work_group_size(NBW * 64, NBW * 64), amdgpu_waves_per_eu(tile_waves(DT * DN, SLICE != 2 && !(VAR && sizeof(TIn) == 4)))))
void chunk_bwd_tile_kernel(BwdArgs A, TileRect R) {
  const ChunkArgs& a = A.c;
  extern __shared__ float smem[];
  typedef typename Raw4<TIn>::type raw4;
  constexpr bool F32 = sizeof(TIn) == 4;
  constexpr int DTP = rows_pad(DT), DS = 16 * DT;   // value rows of a pass
  constexpr int plane = 16 * DTP, SV = vb_stride(DT, VAR);   // staged value rows of a token: v, b, do, (dovar)
  constexpr int WC = 4 * DN;                // key columns of a wave
  constexpr int NT = NBW * 64, DNG = WC * NBW;
  constexpr TileLds L = tile_lds(DT, DN, NBW, VAR, F32);
  constexpr int kG = tile_g(DT, DN), kSub = kC / kG;   // tokens per step, steps per tile
  constexpr bool kScaled = tile_scales(VAR, F32);
  constexpr int kDS = tile_decs(VAR, F32);   // numbers kept per token, f the last of them
  constexpr bool BOTH = L.both != 0;
  float* sC = smem;
  float* sDec = smem + L.oDec;   // [64] (scaled form: Ip / F_t, 1 / F_t, F_t,) f_t
  int* sPlain = (int*)(smem + L.oDec + kDS * kC);   // (scaled form) whether the tile is worked in plain form
  float* sW = smem + L.oW;
  float* sFB = smem + L.oFB;
  float* sX = smem + L.oX;
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.H, dk = a.dk, dv = a.dv;
  int cidx, h;
  if (!tile_head(a.total_chunks, H, (int)blockIdx.x, cidx, h)) return;
  int seq, t0, clen, cis;
  chunk_lookup(a, cidx, seq, t0, clen, cis);
  const float Ip = a.Ip[h], scale = a.scale;

  const int64_t qks = qk_stride(a), vs = (int64_t)H * dv, dks = (int64_t)H * dk;
  const int64_t tok0 = (int64_t)t0 * H + h;
  const TIn* kp = (const TIn*)a.k + qk_row(a, t0, h);
  const TIn* qp = (const TIn*)a.q + qk_row(a, t0, h);
  const TIn* vp = (const TIn*)a.v + tok0 * dv;
  const TIn* bp = (const TIn*)a.b + tok0 * dv;
  const TIn* dop = (const TIn*)A.d_o + tok0 * dv;
  const int64_t tile_off = ((int64_t)cidx * H + h) * dv * dk;
  float* base = smem + L.oBase + w * (2 * DT * 256) + 4 * lane;   // + 256 per piece of 16 value rows: M, then I
  const int last = (clen - 1) / kG;
  float ssum = 0.f;   // sum of S over the tile's tokens

  constexpr bool PARTS = SLICE == 3;           // a small pass: workgroups for every rectangle, outputs of their own
  const int n0 = R.n0 + (PARTS ? blockIdx.z * DNG : 0), r0 = R.r0 + (PARTS ? blockIdx.y * DS : 0);   // first key column, value row
  const int nw = n0 + WC * w;                  // of the wave (a lane has DN of its columns, from DN g on)
  {
    // Staging items, (token of the step, four columns): the first threads take k and q, the next ones (from a wave of their
    // own, if there are that many) v, b, do.  They are
    // decoded anew each time from an opaque copy of the thread index: kept, they would take registers.
    constexpr int nKQ = kG * DNG / 4, nVB = kG * DS / 4;
    constexpr int offV = ((nKQ + 63) & ~63) + nVB <= NT ? (nKQ + 63) & ~63 : nKQ;
    static_assert(nKQ + nVB <= NT, "one staging item per thread");
    // Where a wave stages rows of one kind, it fetches through descriptors that end with the step's last valid row: tokens beyond the
    // end read as zero, without a branch, a select or a register to clear (which would wait for all that is in flight).
    constexpr bool kByWave = offV % 64 == 0;
    constexpr int kStagers = (offV + nVB + 63) / 64;
    raw4 r1, r2, r3;
    float rdv[VAR ? 4 : 1];
    const bool kq_wave = w < offV / 64;
    const int64_t f_stride = kq_wave ? qks : vs;
    const TIn* f1 = (kq_wave ? kp + n0 : vp + r0) + kG * last * f_stride;   // of the step that is fetched next
    const TIn* f2 = (kq_wave ? qp + n0 : bp + r0) + kG * last * f_stride;
    const TIn* f3 = dop + r0 + kG * last * vs;
    const int f_width = kq_wave ? DNG : DS;
    const int f_full = w < kStagers ? (int)(((kG - 1) * (int)f_stride + f_width) * sizeof(TIn)) : 0;
    unsigned f_off = 0xf0000000u;
    if constexpr (kByWave) {
      const int it = kq_wave ? tid : tid - offV, t = it & (kG - 1), c = 4 * (it / kG);
      if (c < f_width) f_off = (unsigned)((t * (int)f_stride + c) * (int)sizeof(TIn));
    }
    auto fetch = [&](int j) {
      const int ntok = j < 0 ? 0 : min(kG, clen - kG * j);
      if constexpr (kByWave) {
        const int bytes = ntok <= 0 ? 0 : ntok == kG || f_full == 0 ? f_full : (int)(((ntok - 1) * (int)f_stride + f_width) * sizeof(TIn));
        auto take = [&](const TIn* p, int n) {
          const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, n, 0x00020000);
          if constexpr (F32) return __builtin_bit_cast(raw4, __builtin_amdgcn_raw_buffer_load_b128(rs, f_off, 0, 0));
          else return __builtin_bit_cast(raw4, __builtin_amdgcn_raw_buffer_load_b64(rs, f_off, 0, 0));
        };
        r1 = take(f1, bytes);
        r2 = take(f2, bytes);
        r3 = take(f3, kq_wave ? 0 : bytes);
        f1 -= kG * f_stride;
        f2 -= kG * f_stride;
        f3 -= kG * vs;
      }
      if (!kByWave || VAR) {
        int tx = tid;
        asm volatile("" : "+v"(tx));
        const int s = kG * j;
        const bool kq = kByWave ? kq_wave : tx < offV;
        const int it = kq ? tx : tx - offV, t = it & (kG - 1), c = 4 * (it / kG);
        if constexpr (!kByWave) {
          const bool on = t < ntok && c < (kq ? DNG : DS);
          if (ntok > 0) {
            const int64_t o = kq ? (int64_t)n0 + (on ? s * qks + t * qks + c : 0) : (int64_t)r0 + (on ? s * vs + t * vs + c : 0);
            const TIn *p1 = kp, *p2 = qp;   // (opaque: of a choice between two pointers the compiler makes one between places in scratch memory)
            asm volatile("" : "+s"(p1), "+s"(p2));
            r1 = *(const raw4*)((kq ? p1 : vp) + o);
            r2 = *(const raw4*)((kq ? p2 : bp) + o);
            r3 = *(const raw4*)(dop + (kq ? (int64_t)r0 : o));
          }
        }
        if (VAR && ntok > 0) {
          const int64_t o = tok0 * dv + r0 + s * vs + (!kq && t < ntok && c < DS ? t * (int)vs + c : 0);
#pragma unroll
          for (int e = 0; e < (VAR ? 4 : 0); ++e) rdv[e] = load_rt(A.d_o_var, o + e, a.var_bf16);
        }
      }
    };
    // value rows are staged with the DT rows of a lane next to each other; v and b over F
    bool plain = true;
    auto deposit = [&](int j) {
      int tx = tid;
      asm volatile("" : "+v"(tx));
      // (in every wave the fetched rows' registers are theirs until here: one that is reused earlier makes its wave wait for the fetch)
      asm volatile("" : "+v"(r1), "+v"(r2), "+v"(r3));
      const bool kq = kByWave ? w < offV / 64 : tx < offV;
      const int it = kq ? tx : tx - offV, t = it & (kG - 1), c = 4 * (it / kG);
      const bool ok = kByWave || kG * j + t < clen;
      if (kq) {
        if (c < DNG) {
          f32x4 x, y;
#pragma unroll
          for (int e = 0; e < 4; ++e) { x[e] = ok ? (float)r1[e] : 0.f; y[e] = ok ? (float)r2[e] : 0.f; }
          if constexpr (DN == 4) {
            float* p = smem + L.oKQ + (((j & 1) * NBW + (c >> 4)) * kG + t) * 32 + (c & 15);
            *(f32x4*)p = x;
            *(f32x4*)(p + 16) = y;
          } else {   // lane groups of three columns, four words apart
            const int wv = c / 12, c12 = c - 12 * wv;
            float* p = smem + L.oKQ + (((j & 1) * NBW + wv) * kG + t) * 32;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int o = (c12 + e) + (((c12 + e) * 11) >> 5);   // + (c12 + e) / 3
              p[o] = x[e];
              p[o + 16] = y[e];
            }
          }
        }
      } else if (c < DS) {
        float* p = smem + L.oVB + ((j & 1) * kG + t) * SV + (c & 15) * DTP + (c >> 4);
        const float inv = !kScaled || plain ? 1.f : sDec[4 * (kG * j + t) + 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[e * DTP] = ok ? inv * (float)r1[e] : 0.f;
          p[e * DTP + plane] = ok ? inv * (float)r2[e] : 0.f;
          p[e * DTP + 2 * plane] = ok ? scale * (float)r3[e] : 0.f;
          if constexpr (VAR) p[e * DTP + 3 * plane] = kG * j + t < clen ? scale * rdv[e] : 0.f;
        }
      }
    };
    // Transposed v, b of half hf for the matrix products, [tensor][plane][row][32 tokens]: fetched (two tokens, eight rows
    // of both tensors per item), then put into LDS.
    bf16_t* const sT = (bf16_t*)(smem + L.oT);
    constexpr int PL = F32 ? 2 : 1, groups = DS >> 3, HI = 16 * groups;   // items of a half
    // Rows come through descriptors that end with the tile's last token: what lies beyond reads as zero.
    auto tile_rows = [&](const TIn* p, int64_t stride, int width) {
      return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, clen > 0 ? (int)(unsigned)(((clen - 1) * stride + width) * sizeof(TIn)) : 0, 0x00020000);
    };
    struct HalfItem { TIn x[2][2][8]; };
    auto half_fetch = [&](int hf, int idx, HalfItem& y) {
      const int sp = idx / groups, c8 = idx - sp * groups;
      const __amdgpu_buffer_rsrc_t vrs = tile_rows(vp + r0, vs, DS), brs = tile_rows(bp + r0, vs, DS);
      const unsigned o = (unsigned)((kHalf * hf + 2 * sp) * (int)vs + 8 * c8) * (unsigned)sizeof(TIn);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int e = 0; e < (int)(sizeof(TIn) / 2); ++e) {
          const unsigned at = o + (unsigned)(u * (int)vs * (int)sizeof(TIn) + 16 * e);
          const auto xv = __builtin_amdgcn_raw_buffer_load_b128(vrs, at, 0, 0), xb = __builtin_amdgcn_raw_buffer_load_b128(brs, at, 0, 0);
          __builtin_memcpy((char*)y.x[0][u] + 16 * e, &xv, 16);
          __builtin_memcpy((char*)y.x[1][u] + 16 * e, &xb, 16);
        }
    };
    auto half_put = [&](int idx, const HalfItem& y, bf16_t* dst) {
      const int sp = idx / groups, c8 = idx - sp * groups;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a0 = (float)y.x[t][0][e], a1 = (float)y.x[t][1][e];
          bf16_t* p = dst + ((t * PL) * DS + 8 * c8 + e) * kHS + 2 * sp;
          const bf16x2 hi = pack2(a0, a1);
          *(bf16x2*)p = hi;
          if constexpr (F32) *(bf16x2*)(p + DS * kHS) = pack2(a0 - (float)hi[0], a1 - (float)hi[1]);
        }
    };
    float largest[3] = {0.f, 0.f, 0.f};   // |v|, |b|, |k| of the thread's items
    auto look = [&](const HalfItem& y) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          largest[t] = fmaxf(largest[t], fmaxf(__builtin_fabsf((float)y.x[t][0][e]), __builtin_fabsf((float)y.x[t][1][e])));
    };
    // the wave's k in operand layout (tokens 8g + j of the half; operand row i is column i & 3 of lane group i >> 2)
    TIn kt[8];
    auto load_kt = [&](int hf, TIn* kt) {
      int lx = lane;
      asm volatile("" : "+v"(lx));
      const int i = lx & 15, g = lx >> 4;
      const bool ok = DN == 4 || (i & 3) < DN;
      const __amdgpu_buffer_rsrc_t krs = tile_rows(kp + nw, qks, WC);
      const unsigned o = (unsigned)((kHalf * hf + 8 * g) * (int)qks + (ok ? DN * (i >> 2) + (i & 3) : 0)) * (unsigned)sizeof(TIn);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned at = o + (unsigned)(j * (int)qks * (int)sizeof(TIn));
        TIn x;
        if constexpr (F32) x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(krs, at, 0, 0));
        else x = __builtin_bit_cast(bf16_t, __builtin_amdgcn_raw_buffer_load_b16(krs, at, 0, 0));
        kt[j] = ok ? x : (TIn)0.f;
      }
    };
    float M[DT][DN], J[DT][DN];   // J = I - Ip
    // state before step `row` (or after token 31) from the base state in LDS
    auto state_at = [&](int row, const bf16_t* T) {
      const float fb = sFB[row];
      f32x4 accM[DT], accJ[DT];
#pragma unroll
      for (int x = 0; x < DT; ++x) {
        const f32x4 m = *(const f32x4*)(base + 256 * x), y = *(const f32x4*)(base + 256 * (DT + x));
#pragma unroll
        for (int r = 0; r < 4; ++r) { accM[x][r] = fb * m[r]; accJ[x][r] = fb * y[r]; }
      }
      if (row == kSub || (row & (kSub / 2 - 1)) != 0) {
        const f32x4 w0 = *(const f32x4*)&sW[row * kHalf + 8 * g], w1 = *(const f32x4*)&sW[row * kHalf + 8 * g + 4];
        float k1[8], k2[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float kv = (float)kt[j];
          k1[j] = kv * (j < 4 ? w0[j & 3] : w1[j & 3]);
          k2[j] = k1[j] * kv;
        }
        bf16x8 K1, K2, K1l, K2l;
        if constexpr (F32) {
          split_bf16(k1, K1, K1l);
          split_bf16(k2, K2, K2l);
        } else {
#pragma unroll
          for (int j = 0; j < 8; j += 2) {
            const bf16x2 x = pack2(k1[j], k1[j + 1]), y = pack2(k2[j], k2[j + 1]);
            K1[j] = x[0]; K1[j + 1] = x[1]; K2[j] = y[0]; K2[j + 1] = y[1];
          }
        }
        const bf16_t* p = T + i * kHS + 8 * g;
#pragma unroll
        for (int x = 0; x < DT; ++x) {
          const bf16x8 V = *(const bf16x8*)(p + 16 * x * kHS), B = *(const bf16x8*)(p + (PL * DS + 16 * x) * kHS);
          if constexpr (F32) {
            const bf16x8 Vl = *(const bf16x8*)(p + (DS + 16 * x) * kHS), Bl = *(const bf16x8*)(p + (3 * DS + 16 * x) * kHS);
            accM[x] = mfma16_split(K1, K1l, V, Vl, accM[x]);
            accJ[x] = mfma16_split(K2, K2l, B, Bl, accJ[x]);
          } else {
            accM[x] = mfma16(K1, V, accM[x]);
            accJ[x] = mfma16(K2, B, accJ[x]);
          }
        }
      }
#pragma unroll
      for (int x = 0; x < DT; ++x)
#pragma unroll
        for (int r = 0; r < DN; ++r) { M[x][r] = accM[x][r]; J[x][r] = accJ[x][r]; }
    };
    // base state of the first half: the state at the start of the tile
    struct BaseIn { f32x4 m[DT], y[DT]; };
    auto base_fetch = [&](BaseIn& z) {
      int lx = lane;
      asm volatile("" : "+v"(lx));
      const int i = lx & 15, nl = nw + DN * (lx >> 4);
      const float* cm = a.chunk_mu + tile_off;
      const float* cI = a.chunk_I + tile_off;
#pragma unroll
      for (int x = 0; x < DT; ++x) {
        const unsigned o = (unsigned)((r0 + 16 * x + i) * dk + nl);
        if constexpr (DN == 4) {
          z.m[x] = *(const f32x4*)(cm + o);
          z.y[x] = *(const f32x4*)(cI + o);
        } else {
#pragma unroll
          for (int r = 0; r < DN; ++r) {
            z.m[x][r] = cm[o + r];
            z.y[x][r] = cI[o + r];
          }
          z.m[x][3] = 0.f;
          z.y[x][3] = 1.f;
        }
      }
    };
    auto base_put = [&](BaseIn& z) {
#pragma unroll
      for (int x = 0; x < DT; ++x) {
#pragma unroll
        for (int r = 0; r < DN; ++r) { z.m[x][r] *= z.y[x][r]; z.y[x][r] -= Ip; }
        *(f32x4*)(base + 256 * x) = z.m[x];
        *(f32x4*)(base + 256 * (DT + x)) = z.y[x];
      }
    };
    // dv, db of a step: sums over the waves.  Item (token, dv or db, four rows) of a thread; the last waves take them,
    // the first ones have the staging.
    constexpr int nF = kG * DS / 2, offF = NT >= ((nF + 63) & ~63) ? NT - ((nF + 63) & ~63) : 0;
    auto flush_at = [&](int j, int it) {
      const int tok = kG * j + ((it & (2 * kG - 1)) >> 1), c = 4 * (it / (2 * kG));
      return (TIn*)((it & 1) ? A.db : A.dv) + tok0 * dv + (int64_t)tok * vs + r0 + c;
    };
    const bool cols_before = !PARTS && R.flags & kRectColsBefore;   // what the columns of the earlier launches gave is added to
    auto flush_sum = [&](int j, int it, f32x4& x, raw4& was) {
      const float* p = smem + L.oPart + (j & 1) * NBW * (kG * 32 * DT) + (it & (2 * kG - 1)) * DS + 4 * (it / (2 * kG));
      if (cols_before && kG * j + ((it & (2 * kG - 1)) >> 1) < clen) was = *(const raw4*)flush_at(j, it);
      f32x4 z[NBW];
#pragma unroll
      for (int y = 0; y < NBW; ++y) z[y] = *(const f32x4*)(p + y * (kG * 32 * DT));
      x = z[0];
#pragma unroll
      for (int y = 1; y < NBW; ++y) x += z[y];
    };
    auto flush_store = [&](int j, int it, f32x4 x, raw4 was) {
      if (kG * j + ((it & (2 * kG - 1)) >> 1) < clen) {
        if constexpr (PARTS) {
          const int tok = kG * j + ((it & (2 * kG - 1)) >> 1), c = 4 * (it / (2 * kG));
          const int64_t row = ((int64_t)(R.group + blockIdx.z) * A.tokens + t0 + tok) * H + h;
          *(f32x4*)(A.pVB + (row * 2 + (it & 1)) * dv + r0 + c) = x;
          return;
        }
        if (cols_before) {
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] += (float)was[e];
        }
        store_vec<4>(flush_at(j, it), (const float*)&x);
      }
    };
    // wave 0: a step's gates, of the first token of the step after in the place of its own first
    auto flush_xs = [&](int j) {
      if (lane < kG) {
        const float* p = smem + L.oXS + (j & 1) * NBW * kG + lane;
        float x = p[0];
#pragma unroll
        for (int y = 1; y < NBW; ++y) x += p[y * kG];
        sX[kG * j + (lane ? lane : kG)] = x;
      }
    };

    // Everything the pass starts from is requested at once.
    const bool two = clen > kHalf;
    {
      int tp = tid;   // opaque: nothing that depends on it is kept through the passes
      asm volatile("" : "+v"(tp));
      BaseIn bs;
      HalfItem y0, y1;
      bf16_t* const sT0 = BOTH || !two ? sT : (bf16_t*)(smem + L.oPart);
      bf16_t* const sT1 = BOTH ? sT + 2 * PL * DS * kHS : sT;
      // (the gates first: the decays are what the rest waits for)
      const int64_t gi = (int64_t)(t0 + (lane < clen ? lane : 0)) * H + h;
      const unsigned gate_word = load_gate_word(a.gt, gi, a.gate_bf16);
      const float gh = a.g[h] * kLog2e;
      fetch(last);
      // items of both halves: one of either for a thread, or one of each
      constexpr bool kOneEach = NT < 2 * HI;
      const int hf1 = kOneEach ? 0 : tp >= HI, it1 = kOneEach ? tp : tp - HI * hf1;
      half_fetch(hf1, min(it1, HI - 1), y0);
      if constexpr (kOneEach) half_fetch(1, min(tp, HI - 1), y1);
      base_fetch(bs);
      TIn kt1[8];
      load_kt(0, kt);
      load_kt(1, kt1);
      {
      if (w == 0) {
        const float gt = lane < clen ? gate_value(gate_word, gi, a.gate_bf16) : 0.f;
        const float c = wave_inclusive_scan(-gt * gh, lane);
        sC[lane] = c;
        sX[lane] = 0.f;
        if (lane == 63 && (!PARTS || (n0 | r0) == 0)) A.wFtot[(int64_t)cidx * H + h] = c;
        const float f = fast_exp2(-gt * gh);
        if constexpr (kScaled) {
          // decay since the start of the step: the product over its tokens
          float F = f;
          const int u = lane & (kG - 1);
          float y = row_shr_zero<1>(F);
          F = u >= 1 ? F * y : F;
          y = row_shr_zero<2>(F);
          F = u >= 2 ? F * y : F;
          if constexpr (kG == 8) {
            y = row_shr_zero<4>(F);
            F = u >= 4 ? F * y : F;
          }
          const float inv = fast_rcp(F);
          *(f32x4*)&sDec[4 * lane] = f32x4{Ip * inv, inv, F, f};
          const bool off = !__all(F >= kMinStepDecay && F <= 1.f);
          if (lane == 0) *sPlain = off;
        } else {
          sDec[lane] = f;
        }
      }
      __syncthreads();
      // row j < kSub: weights of the tokens of the half for the state before step j; row kSub: for the state after token 31
      {
        constexpr int kRows = NT / kHalf, kIts = (kSub + kRows) / kRows;
        const int s = tp % kHalf;
        const float c0 = sC[s], c1 = sC[kHalf + s], cm = sC[kHalf - 1];
        float ce[kIts];
#pragma unroll
        for (int e = 0; e < kIts; ++e) {
          const int j = min(tp / kHalf + e * kRows, kSub), at = j < kSub ? kG * j : kHalf;
          ce[e] = sC[max(at - 1, 0)];
        }
#pragma unroll
        for (int e = 0; e < kIts; ++e) {
          const int j = min(tp / kHalf + e * kRows, kSub), at = j < kSub ? kG * j : kHalf;
          const bool upper = j < kSub && j >= kSub / 2;
          const int hb = upper ? kHalf : 0;
          sW[j * kHalf + s] = hb + s < at ? fast_exp2(ce[e] - (upper ? c1 : c0)) : 0.f;
          if (s == 0) sFB[j] = at == hb ? 1.f : fast_exp2(ce[e] - (upper ? cm : 0.f));
        }
      }
      }
      if constexpr (kOneEach) {
        for (int idx = tp; idx < HI; idx += NT) {
          if (idx >= NT) { half_fetch(0, idx, y0); half_fetch(1, idx, y1); }
          half_put(idx, y0, sT0);
          if (two) half_put(idx, y1, sT1);
          if constexpr (kScaled) { look(y0); look(y1); }
        }
      } else if (it1 < HI && (two || hf1 == 0)) {
        half_put(it1, y0, hf1 ? sT1 : sT0);
        if constexpr (kScaled) look(y0);
      }
      base_put(bs);
      if constexpr (kScaled) {
#pragma unroll
        for (int e = 0; e < 8; ++e) largest[2] = fmaxf(largest[2], fmaxf(__builtin_fabsf((float)kt[e]), __builtin_fabsf((float)kt1[e])));
        float state = __builtin_fabsf(Ip);
#pragma unroll
        for (int x = 0; x < DT; ++x)
#pragma unroll
          for (int r = 0; r < DN; ++r) state = fmaxf(state, fmaxf(__builtin_fabsf(bs.m[x][r]), __builtin_fabsf(bs.y[x][r])));
        if (!(largest[0] <= kMaxV && largest[1] <= kMaxB && largest[2] <= kMaxK && state <= kMaxState)) *sPlain = 1;
      }
      __syncthreads();
      if constexpr (kScaled) plain = __builtin_amdgcn_readfirstlane(*sPlain) != 0;
      deposit(last);
      if (two) {
        state_at(kSub, sT0);
#pragma unroll
        for (int e = 0; e < 8; ++e) kt[e] = kt1[e];
#pragma unroll
        for (int x = 0; x < DT; ++x) {
          *(f32x4*)(base + 256 * x) = f32x4{M[x][0], M[x][1], M[x][2], DN == 4 ? M[x][DN - 1] : 0.f};
          *(f32x4*)(base + 256 * (DT + x)) = f32x4{J[x][0], J[x][1], J[x][2], DN == 4 ? J[x][DN - 1] : 0.f};
        }
      }
      __syncthreads();
    }

    // dM, dJ at a step's end in time: the carry of the tokens after it, with the decay of the first of them
    float dM[DT][DN], dJ[DT][DN];
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < DN; ++r) { dM[x][r] = 0.f; dJ[x][r] = 0.f; }
    // dq, dk: lane u of a quad stores the columns oc (and, out2, oc + 1) of token u (and, eight tokens a step, u + 4) of dq (lane
    // bit 3 clear) or dk
    int lo = lane;
    asm volatile("" : "+v"(lo));
    const int oc = nw + DN * (lo >> 4) + 2 * ((lo >> 2) & 1), ow = (lo >> 3) & 1, ou = lo & 3;
    const bool out2 = DN == 4 || (lo & 4) == 0;
    TIn* const po = (TIn*)(ow ? A.dk : A.dq) + tok0 * dk + oc + ou * (int)dks;
    // bf16 rows: sums over the launches so far
    const int accs = 2 * (PARTS ? dk : DNG) * H;   // per token
    float* const pacc = (PARTS ? A.pQK + ((int64_t)blockIdx.y * A.tokens * H + tok0) * (2 * dk) + ow * dk + oc
                               : A.wQK + tok0 * (2 * DNG) + ow * DNG + (oc - n0)) + ou * accs;
    auto steps = [&](auto form) {
    constexpr bool SCALED = decltype(form)::value;
    for (int j = last; j >= 0; --j) {
      if (j == kSub / 2 - 1 && two) {   // on to the first half
        BaseIn bs;
        base_fetch(bs);
        load_kt(0, kt);
        if constexpr (!BOTH) {
          int it0 = tid;
          asm volatile("" : "+v"(it0));
          for (int idx = it0; idx < HI; idx += NT) {
            HalfItem y;
            half_fetch(0, idx, y);
            half_put(idx, y, sT);
          }
        }
        base_put(bs);
        if constexpr (!BOTH) __syncthreads();
      }
      fetch(j - 1);   // (by every wave and also before the first step, when nothing is left: the registers are then set on one path)
      // what the step before left is summed over the waves here, beside the set-up of this step
      f32x4 fl = {0.f, 0.f, 0.f, 0.f};
      raw4 fw;
      int itF = tid - offF;
      asm volatile("" : "+v"(itF));
      const bool doF = w >= offF / 64 && (nF % 64 == 0 || itF < nF);
      if (j < last) {
        if (doF) flush_sum(j + 1, itF, fl, fw);
        if (w == 0) flush_xs(j + 1);
      }
      state_at(j, sT + (BOTH && j >= kSub / 2 ? 2 * PL * DS * kHS : 0));
      if (j < last && doF) {
        flush_store(j + 1, itF, fl, fw);
        if constexpr (NT < nF) for (int it = itF + NT; it < nF; it += NT) { flush_sum(j + 1, it, fl, fw); flush_store(j + 1, it, fl, fw); }
      }
      const float* krow = smem + L.oKQ + ((j & 1) * NBW + w) * kG * 32 + 4 * g;
      const float* vrow = smem + L.oVB + (j & 1) * kG * SV + i * DTP;
      const float* dec = sDec + kDS * kG * j;
      const int o_tok = kG * j * (int)dks;   // (64 tokens of a tile stay within 32 bits)
      float* part = smem + L.oPart + ((j & 1) * NBW + w) * (kG * 32 * DT);
      float was[kG / 4][2];
      float xs[kG / 2], xo, oz[kG][2], inv_last = 1.f;
      TokSums<DT, DN> ts[2];
      auto finish = [&](int u, TokSums<DT, DN>& z, float inv) {
        z.stage_c();
        oz[u][0] = z.z0;
        oz[u][1] = z.z1;
        float* pu = part + u * (32 * DT);
        if constexpr (DT >= 3) {
          if (lane < 16 * DT) {
            pu[lane] = z.p[0] * inv;
            pu[16 * DT + lane] = z.q[0] * inv;
          }
        } else {
          if (lane < 32 * DT) pu[lane] = z.p[0] * inv;
        }
        if (u & 1) xo = z.X;
        else xs[u >> 1] = pair_bit3(z.X, xo);
      };
      {
        float sM[kG][DT][DN], sJ[kG][DT][DN];   // state after each token; in reverse mu and 1 / I in their place
        // ---- forward over the step; a token's operands are requested during the arithmetic of the token before it
        TokFwd<DT, SCALED, kDS> xf[kG], xr[kG];
        TokRev<DT, VAR, SCALED, kDS> yr[kG];
        xf[0].load(krow, vrow, dec, plane);
#pragma unroll
        for (int u = 0; u < kG; ++u) {
          const TokFwd<DT, SCALED, kDS>& x = xf[u];
          __builtin_amdgcn_sched_barrier(0);
          if (u + 1 < kG) xf[u + 1].load(krow + (u + 1) * 32, vrow + (u + 1) * SV, dec + kDS * (u + 1), plane);
          else yr[u].load(krow + u * 32, vrow + u * SV, dec + kDS * u, Ip, plane);
#pragma unroll
          for (int r = 0; r < DN; ++r) {
            const float kk = x.k[r] * x.k[r];
#pragma unroll
            for (int d = 0; d < DT; ++d) {
              const float m = u ? sM[u ? u - 1 : 0][d][r] : M[d][r], y = u ? sJ[u ? u - 1 : 0][d][r] : J[d][r];
              sM[u][d][r] = fmaf(x.v[d], x.k[r], SCALED ? m : m * x.f);
              sJ[u][d][r] = fmaf(x.b[d], kk, SCALED ? y : y * x.f);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SCALED) {
          const float Fe = dec[4 * (kG - 1) + 2];
#pragma unroll
          for (int r = 0; r < DN; ++r)
#pragma unroll
            for (int d = 0; d < DT; ++d) { dM[d][r] *= Fe; dJ[d][r] *= Fe; }
        }
        // the gate of the first token of the step after, which saw the state after this one
        float next_gate = 0.f;
#pragma unroll
        for (int r = 0; r < DN; ++r)
#pragma unroll
          for (int d = 0; d < DT; ++d) next_gate = fmaf(dM[d][r], sM[kG - 1][d][r], fmaf(dJ[d][r], sJ[kG - 1][d][r], next_gate));
        asm volatile("" : "+v"(next_gate));
        __builtin_amdgcn_sched_barrier(0);
        // ---- and in reverse
        float S = 0.f, inv_before = 1.f;
        // SLICE 2: what the launches over earlier value rows left for the lane's token
        if constexpr (SLICE == 2) {
#pragma unroll
          for (int e = 0; e < kG / 4; ++e) {
            const bool on = kG * j + 4 * e + ou < clen;
            const int t = on ? kG * j + 4 * e : -ou;   // (or the first token)
            const float* acc = F32 ? (const float*)po + t * (int)dks : pacc + t * accs;
            was[e][0] = acc[0];
            was[e][1] = acc[out2 ? 1 : 0];
          }
        }
#pragma unroll
        for (int u = kG - 1; u >= 0; --u) {
          __builtin_amdgcn_sched_barrier(0);
          const TokFwd<DT, SCALED, kDS>& x = u + 1 < kG ? xr[u] : xf[u];
          const TokRev<DT, VAR, SCALED, kDS>& y = yr[u];
          float dq[DN], dqv[DN], dk[DN], dvp[DT], dbp[DT], St = 0.f, gate = 0.f;
          TokSums<DT, DN>& before = ts[(u + 1) & 1];   // of the token worked before this one
          if (u + 1 < kG) before.stage_a();
#pragma unroll
          for (int r = 0; r < DN; ++r) {
            if (r > 0) __builtin_amdgcn_sched_barrier(0);
            if (r == 1 && u + 1 < kG) before.stage_b();
            if (r == 2 && u + 1 < kG) finish(u + 1, before, inv_before);
            if (r == DN - 2 && u > 0) {   // half of mu, r of this token are dead: room for the next token's operands
              xr[u - 1].load(krow + (u - 1) * 32, vrow + (u - 1) * SV, dec + kDS * (u - 1), plane);
              yr[u - 1].load(krow + (u - 1) * 32, vrow + (u - 1) * SV, dec + kDS * (u - 1), Ip, plane);
            }
            __builtin_amdgcn_s_setprio(3);
#pragma unroll
            for (int d = 0; d < DT; ++d) {
              sJ[u][d][r] = fast_rcp(sJ[u][d][r] + y.ip);
              asm volatile("" : "+v"(sJ[u][d][r]));
            }
            __builtin_amdgcn_s_setprio(0);
#pragma unroll
            for (int d = 0; d < DT; ++d) sM[u][d][r] *= sJ[u][d][r];
            const float kk = x.k[r] * x.k[r];
            float dkM, dkJ, Sw;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
              const float ri = sJ[u][d][r], m = sM[u][d][r];
              const float fn = !SCALED && u + 1 < kG ? y.inv : 1.f;   // (plain form)
              if constexpr (VAR) {
                const float e = y.d_o[d] * m, n = y.d_ov[d] * ri, t = fmaf(n, y.q[r], e) * ri;   // G r mu over q
                dq[r] = d ? dq[r] + e : e;
                dqv[r] = d ? dqv[r] + n : n;
                Sw = d ? Sw + t : t;
                dM[d][r] = fmaf(dM[d][r], fn, y.d_o[d] * ri * y.q[r]);
                dJ[d][r] = fmaf(dJ[d][r], fn, -t * y.q[r]);
              } else {
                dq[r] = d ? fmaf(m, y.d_o[d], dq[r]) : m * y.d_o[d];
                if constexpr (SCALED) {
                  const float p = y.d_o[d] * ri, t = p * m;   // G r mu over q
                  Sw = d ? Sw + t : t;
                  dM[d][r] = fmaf(p, y.q[r], dM[d][r]);
                  dJ[d][r] = fmaf(-t, y.q[r], dJ[d][r]);
                } else {
                  const float p = y.d_o[d] * y.q[r] * ri, t = p * m;   // G r mu
                  Sw = d ? Sw + t : t;
                  dM[d][r] = fmaf(dM[d][r], fn, p);
                  dJ[d][r] = fmaf(dJ[d][r], fn, -t);
                }
              }
              if (u > 0) gate = fmaf(dM[d][r], sM[u ? u - 1 : 0][d][r], fmaf(dJ[d][r], sJ[u ? u - 1 : 0][d][r], gate));
              dkM = d ? fmaf(dM[d][r], x.v[d], dkM) : dM[d][r] * x.v[d];
              dkJ = d ? fmaf(dJ[d][r], x.b[d], dkJ) : dJ[d][r] * x.b[d];
              dvp[d] = r ? fmaf(dM[d][r], x.k[r], dvp[d]) : dM[d][r] * x.k[r];
              dbp[d] = r ? fmaf(dJ[d][r], kk, dbp[d]) : dJ[d][r] * kk;
            }
            St = VAR || SCALED ? fmaf(Sw, y.q[r], St) : St + Sw;
            dk[r] = fmaf(2.f * x.k[r], dkJ, dkM);
          }
          TokSums<DT, DN>& mine = ts[u & 1];
          inv_before = SCALED ? y.inv : 1.f;
          S = fmaf(St, inv_before, S);
          mine.X = u == 0 ? next_gate : SCALED ? gate : x.f * gate;
          asm volatile("" : "+v"(S), "+v"(mine.X));
#pragma unroll
          for (int r = 0; r < DN; ++r) {
            mine.o[r] = VAR ? fmaf(2.f * y.q[r], dqv[r], dq[r]) : dq[r];
            mine.o[DN + r] = dk[r];
          }
          if constexpr (DT >= 3) {
#pragma unroll
            for (int d = 0; d < 4; ++d) { mine.p[d] = d < DT ? dvp[d < DT ? d : 0] : 0.f; mine.q[d] = d < DT ? dbp[d < DT ? d : 0] : 0.f; }
          } else {
            mine.p[0] = dvp[0];
            mine.p[1] = DT == 2 ? dvp[DT - 1] : dbp[0];
            mine.p[2] = DT == 2 ? dbp[0] : 0.f;
            mine.p[3] = DT == 2 ? dbp[DT - 1] : 0.f;
          }
          if constexpr (!SCALED) {
            if (u == 0) {
#pragma unroll
              for (int r = 0; r < DN; ++r)
#pragma unroll
                for (int d = 0; d < DT; ++d) { dM[d][r] *= x.f; dJ[d][r] *= x.f; }
            }
          }
        }
        ssum += S;
        inv_last = inv_before;
      }
      __builtin_amdgcn_sched_barrier(0);
      ts[0].stage_a();
      ts[0].stage_b();
      finish(0, ts[0], inv_last);
      // gates: odd token of a pair by lane bit 3, pair of tokens by bit 2 (kG = 8: four of them by bit 5)
      {
        float x = quad_sum(pair_bit2(xs[0], xs[1]));
        if constexpr (kG == 8) {
          float y = quad_sum(pair_bit2(xs[kG / 2 - 2], xs[kG / 2 - 1]));
          swap_halves(x, y);
          x += y;
          y = x;
          swap_rows(x, y);
          x += y;
        } else {
          x = rows4_sum(x);
        }
        if ((lane & (kG == 8 ? 19 : 51)) == 0)
          smem[L.oXS + ((j & 1) * NBW + w) * kG + (kG == 8 ? (lane >> 5) * 4 : 0) + ((lane >> 2) & 1) * 2 + ((lane >> 3) & 1)] = x;
      }
      // (before the stores: what a wave waits for here, its fetched rows, would include stores that were just issued)
      if (j > 0) deposit(j - 1);
#pragma unroll
      for (int e = 0; e < kG / 4; ++e) {
        float x[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          x[c] = quad_tokens(lane, oz[4 * e][c], oz[4 * e + 1][c], oz[4 * e + 2][c], oz[4 * e + 3][c]);
          if constexpr (SLICE == 2) x[c] += was[e][c];
        }
        if (kG * j + 4 * e + ou < clen) {
          bool done = true;
          if constexpr (PARTS || (SLICE != 0 && !F32)) {   // the value rows of the launches add up, in fp32
            if (PARTS || (R.flags & kRectRowsAfter)) {
              float* acc = pacc + (kG * j + 4 * e) * accs;
              acc[0] = x[0];
              if (out2) acc[1] = x[1];
              done = false;
            }
          }
          if (done) {
            TIn* o = po + (o_tok + 4 * e * (int)dks);
            if constexpr (DN == 4) {
              store_vec<2>(o, x);
            } else {
              o[0] = from_f32<TIn>(x[0]);
              if (out2) o[1] = from_f32<TIn>(x[1]);
            }
          }
        }
      }
      __syncthreads();
    }
    // (vmcnt(0): to the compiler one loop may follow the other, which would then wait for what this one has requested)
    if constexpr (kScaled && !SCALED) __builtin_amdgcn_s_waitcnt(0x0f70);
    };
    if (plain) steps(std::false_type{});
    else if constexpr (kScaled) steps(std::true_type{});
    {
      f32x4 x;
      raw4 fw;
      int it0 = tid;
      asm volatile("" : "+v"(it0));
      for (int it = it0; it < nF; it += NT) { flush_sum(0, it, x, fw); flush_store(0, it, x, fw); }
      if (w == 0) flush_xs(0);
    }
    // gate of the tile's first token, which saw the state at the start of the tile
    {
      float y0 = 0.f;
#pragma unroll
      for (int x = 0; x < DT; ++x) {
        const f32x4 m = *(const f32x4*)(base + 256 * x), y = *(const f32x4*)(base + 256 * (DT + x));
#pragma unroll
        for (int r = 0; r < DN; ++r) y0 = fmaf(dM[x][r], m[r], fmaf(dJ[x][r], y[r], y0));
      }
      y0 = wave_sum(y0);
      ssum = wave_sum(ssum);
      if (lane == 0) {   // (the second buffer of partial sums is free)
        smem[L.oXS + NBW * kG + w] = y0;
        smem[L.oXS + NBW * kG + NBW + w] = ssum;
      }
    }
    // carry handed to the previous tile
    int lx = lane;
    asm volatile("" : "+v"(lx));
    const int ci = lx & 15, cn = nw + DN * (lx >> 4);
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const int64_t co = tile_off + (r0 + 16 * x + ci) * dk + cn;
      float rm[DN], rj[DN];
#pragma unroll
      for (int r = 0; r < DN; ++r) { rm[r] = dM[x][r]; rj[r] = dJ[x][r]; }
      if constexpr (DN == 4) {
        store_vec<4>((TIn*)A.wDM + co, rm);
        store_vec<4>((TIn*)A.wDJ + co, rj);
      } else {
#pragma unroll
        for (int r = 0; r < DN; ++r) {
          ((TIn*)A.wDM)[co + r] = from_f32<TIn>(rm[r]);
          ((TIn*)A.wDJ)[co + r] = from_f32<TIn>(rj[r]);
        }
      }
    }
  }
  __syncthreads();
  if (w == 0) {
    const float* p = smem + L.oXS + NBW * kG;
    float x = p[0], tot = -p[NBW];
#pragma unroll
    for (int y = 1; y < NBW; ++y) { x += p[y]; tot -= p[NBW + y]; }
    x = lane ? sX[lane] : x;
    const int rect = PARTS ? (R.group + blockIdx.z) * R.slices + blockIdx.y : 0;
    float* pe = (PARTS ? A.pE : A.wE) + ((int64_t)rect * H + h) * A.tokens + t0 + lane;
    float* ps = (PARTS ? A.pSig : A.wSig) + ((int64_t)rect * a.total_chunks + cidx) * H + h;
    const bool add = !PARTS && (R.flags & (kRectRowsBefore | kRectColsBefore));
    if (lane < clen) *pe = add ? x + *pe : x;
    if (lane == 0) *ps = add ? tot + *ps : tot;
  }
}

template <typename TIn, int DT, int DN, int NBW, bool VAR>
static int launch_tile_n(const BwdArgs& A, const TileRect& R, hipStream_t s) {
  const int64_t blocks = tile_head_blocks(A.c.total_chunks, A.c.H);
  if (blocks > 0x7fffffff) return PAL_E_DIM;
  constexpr size_t lds = sizeof(float) * (size_t)tile_lds(DT, DN, NBW, VAR, sizeof(TIn) == 4).total;
  static_assert(lds <= kMaxLds, "LDS of a compute unit");
  auto go = [&](auto kern) -> int {
    if (int rc = allow_lds((const void*)kern, lds)) return rc;
    PAL_TIMED_LAUNCH(kKernBwdLocal, s, kern, dim3((unsigned)blocks, (unsigned)R.slices, (unsigned)R.groups), dim3(64 * NBW), lds, s, A, R);
    return 0;
  };
  if constexpr (DT <= 2) {
    if (R.flags & kRectParts) {
      if (int rc = go(&chunk_bwd_tile_kernel<TIn, DT, DN, NBW, VAR, 3>)) return rc;
      PAL_HIP_LAUNCH_CHECK();
      return PAL_OK;
    }
  }
  if (int rc = R.flags & kRectRowsBefore  ? go(&chunk_bwd_tile_kernel<TIn, DT, DN, NBW, VAR, 2>)
               : R.flags & kRectRowsAfter ? go(&chunk_bwd_tile_kernel<TIn, DT, DN, NBW, VAR, 1>)
                                          : go(&chunk_bwd_tile_kernel<TIn, DT, DN, NBW, VAR, 0>))
    return rc;
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}
template <typename TIn, int DT, bool VAR>
static int launch_tile_d(const BwdArgs& A, const TileRect& R, hipStream_t s) {
  switch (R.cols) {
    case 64: return launch_tile_n<TIn, DT, 4, 4, VAR>(A, R, s);
    case 48: return launch_tile_n<TIn, DT, 3, 4, VAR>(A, R, s);
    case 32: return launch_tile_n<TIn, DT, 4, 2, VAR>(A, R, s);
    case 16: if constexpr (DT == 1 || DT == 3) return launch_tile_n<TIn, DT, 4, 1, VAR>(A, R, s);
  }
  return PAL_E_HEADDIM;
}

// The launches that make up the tile kernel: groups of key columns, in each the slices of value rows (a small pass: all of
// them side by side, a launch for each width that the groups have).
template <typename TIn, bool VAR>
int launch_tile_t(const BwdArgs& A, const TileParts& P, hipStream_t s) {
  const int dk = A.c.dk, dv = A.c.dv;
  TileRect R;
  R.group = 0;
  for (R.n0 = 0; R.n0 < dk; R.n0 += R.groups * R.cols) {
    R.cols = P.on ? parts_cols(dk, R.n0) : tile_piece(dk - R.n0);
    R.groups = P.on && dk % R.cols == 0 ? dk / R.cols : 1;
    R.slices = P.on ? P.slices : 1;
    int rows;
    for (R.r0 = 0; R.r0 < dv; R.r0 += rows * R.slices) {
      rows = P.on ? P.rows : tile_rows(R.cols, dv - R.r0, sizeof(TIn) == 4, P.few);
      R.flags = P.on ? kRectParts : (R.n0 ? kRectColsBefore : 0) | (R.r0 ? kRectRowsBefore : 0) | (R.r0 + rows < dv ? kRectRowsAfter : 0);
      int rc;
      switch (rows) {
        case 16: rc = launch_tile_d<TIn, 1, VAR>(A, R, s); break;
        case 32: rc = launch_tile_d<TIn, 2, VAR>(A, R, s); break;
        case 48: rc = launch_tile_d<TIn, 3, VAR>(A, R, s); break;
        case 64:
          if constexpr (sizeof(TIn) == 2) { rc = launch_tile_d<TIn, 4, VAR>(A, R, s); break; }   // (fp32 rows: slices of at most 48)
          [[fallthrough]];
        default: rc = PAL_E_HEADDIM;
      }
      if (rc) return rc;
    }
    R.group += R.groups;
  }
  return PAL_OK;
}

}  // namespace pal
