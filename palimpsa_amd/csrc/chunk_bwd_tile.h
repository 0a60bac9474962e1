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
// What bounds it: vector issue.  Per entry and token 19 fp32 instructions and a reciprocal, and 6 more for the sums over
// lanes, the recomputed states, staging and the sums over waves (64x64; 9 more in the smaller rectangles of 96x96); two waves per
// SIMD (the registers), which together issue an instruction per 4 cycles.  As products on the matrix cores (12 prefix and 12
// suffix instructions of 16 cycles per 16 entries of a lane, operands exchanged through LDS between waves of different roles)
// the same pass took 822 us at B=8 T=2048 H=12 64x64, this takes 555; 48x48 H=16 736 -> 555, packed 32768 tokens 96x96 4.91 -> 4.1 ms,
// fp32 rows 64x64 B=8 T=2048 H=8 (forward and backward together) 1.53 -> 0.95 ms.
// Layout: a wave holds 4 DN columns x 16 DT rows of the state, a lane DN neighbouring columns of DT rows, the layout in
// which the matrix products leave the state (DN = 3: the fourth operand row of a lane group is empty), so that a head of
// 48 columns loads all four SIMDs.  As many tokens per step as the registers hold: the fixed cost of a step (about
// 2600 cycles of a SIMD per wave beside 67 per entry and token of a lane) is what small pieces pay.
//
// Gate: gamma_t = f_t (<dM_t, M_{t-1}> + <dJ_t, J_{t-1}>), formed as it stands: where a token decays strongly, what is left of
// the state is of the order of f_t, and so is gamma.  (The states of the step are in registers, so that it takes two
// instructions per entry and token and the one that makes I out of J.  gamma_{t+1} + Ip sum(G r mu) - <dv_t, v_t> - <db_t, b_t>
// is the same number for one addition, but as a difference of terms of order 1: with every fifth token at f = e^-18 the
// gradients of these tokens were off by 200 times their size in fp32.  The definition costs 531 -> 555 us at B=8 T=2048 H=12
// 64x64; fp32 rows B=8 T=2048 H=8 64x64 went from 636 to 612, since the reciprocals of a token are now taken beside its
// products instead of with the forward sweep.)  The first token of a step sees the state after the step before it in time:
// its gamma is formed there, that of the tile's first token from the state at the start of the tile.
#pragma once
#include <type_traits>

#include "chunk_bwd.h"
#include "pal_host.h"
#include "pal_profile.h"

namespace pal {

// The sums of a token over lanes by DPP with a bank mask (see pair_bit3), in three stages so that the next token's arithmetic can be placed between them (each
// stage is a chain of dependent instructions).
//   o[2 DN] (dq, then dk of the lane's columns): over the 16 lanes of a row.  Lane bit 3 selects dq or dk, of which z0 is
//     the first (lane bit 2 clear) or the third column, z1 the second or the fourth (DN = 3: the second in both).
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
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0\n\t"
        "v_add_f32_dpp %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_add_f32_dpp %1, %1, %1 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
        : "+v"(z0), "+v"(z1));
    p[0] += p[1];
    if constexpr (DT >= 3) q[0] += q[1];
  }
};
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

// what both sweeps read of a token: its k, v, b and f
template <int DT>
struct TokFwd {
  f32x4 k;
  float v[DT], b[DT], f;
  __device__ __forceinline__ void load(const float* kq, const float* vb, const float* pf, int plane) {
    f = *pf;
    k = *(const f32x4*)kq;
    lds_vals<DT>(vb, v);
    lds_vals<DT>(vb + plane, b);
  }
};
// and the reverse sweep: q, do, (dovar), the next token's f
template <int DT, bool VAR>
struct TokRev {
  f32x4 q;
  float d_o[DT], d_ov[VAR ? DT : 1], fn;
  __device__ __forceinline__ void load(const float* kq, const float* vb, const float* pf, int plane) {
    q = *(const f32x4*)(kq + 16);
    lds_vals<DT>(vb + 2 * plane, d_o);
    if constexpr (VAR) lds_vals<DT>(vb + 3 * plane, d_ov);
    fn = pf[1];
  }
};

// waves per SIMD that a lane's E state entries leave registers for
constexpr int tile_waves(int E) { return E > 4 ? 2 : 3; }

template <typename TIn, int DT, int DN, int NBW, bool VAR, int SLICE>
__global__ __attribute__((amdgpu_flat_work_group_size(NBW * 64, NBW * 64), amdgpu_waves_per_eu(tile_waves(DT * DN))))
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
  constexpr bool BOTH = L.both != 0;
  float* sC = smem;
  float* sF = smem + L.oF;
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
    raw4 r1, r2, r3;
    float rdv[VAR ? 4 : 1];
    auto fetch = [&](int j) {
      int tx = tid;
      asm volatile("" : "+v"(tx));
      const int s = kG * j;
      const bool kq = offV % 64 == 0 ? w < offV / 64 : tx < offV;
      const int it = kq ? tx : tx - offV, t = it & (kG - 1), c = 4 * (it / kG);
      if (s + t < clen && c < (kq ? DNG : DS)) {
        const unsigned o = (unsigned)((s + t) * (int)(kq ? qks : vs) + (kq ? n0 : r0) + c);
        r1 = *(const raw4*)((kq ? kp : vp) + o);
        r2 = *(const raw4*)((kq ? qp : bp) + o);
        if (!kq) {
          r3 = *(const raw4*)(dop + o);
          if constexpr (VAR) {
#pragma unroll
            for (int e = 0; e < 4; ++e) rdv[e] = load_rt(A.d_o_var, tok0 * dv + o + e, a.var_bf16);
          }
        }
      }
    };
    // value rows are staged with the DT rows of a lane next to each other; tokens beyond the end are zero
    auto deposit = [&](int j) {
      int tx = tid;
      asm volatile("" : "+v"(tx));
      const int s = kG * j;
      if (offV % 64 == 0 ? w < offV / 64 : tx < offV) {
        const int t = tx & (kG - 1), c4 = tx / kG;
        const bool ok = s + t < clen;
        if (4 * c4 < DNG) {
          f32x4 x, y;
#pragma unroll
          for (int e = 0; e < 4; ++e) { x[e] = ok ? (float)r1[e] : 0.f; y[e] = ok ? (float)r2[e] : 0.f; }
          if constexpr (DN == 4) {
            float* p = smem + L.oKQ + (((j & 1) * NBW + (c4 >> 2)) * kG + t) * 32 + 4 * (c4 & 3);
            *(f32x4*)p = x;
            *(f32x4*)(p + 16) = y;
          } else {   // lane groups of three columns, four words apart
            const int wv = c4 / 3, c12 = 4 * (c4 - 3 * wv);
            float* p = smem + L.oKQ + (((j & 1) * NBW + wv) * kG + t) * 32;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int o = (c12 + e) + (((c12 + e) * 11) >> 5);   // + (c12 + e) / 3
              p[o] = x[e];
              p[o + 16] = y[e];
            }
          }
        }
      } else {
        const int it = tx - offV, t = it & (kG - 1), d = 4 * (it / kG);
        const bool ok = s + t < clen;
        float* p = smem + L.oVB + ((j & 1) * kG + t) * SV + (d & 15) * DTP + (d >> 4);
        if (d < DS) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            p[e * DTP] = ok ? (float)r1[e] : 0.f;
            p[e * DTP + plane] = ok ? (float)r2[e] : 0.f;
            p[e * DTP + 2 * plane] = ok ? scale * (float)r3[e] : 0.f;
            if constexpr (VAR) p[e * DTP + 3 * plane] = ok ? scale * rdv[e] : 0.f;
          }
        }
      }
    };
    // Transposed v, b of half hf for the matrix products, [tensor][plane][row][32 tokens]: fetched (two tokens, eight rows
    // of both tensors per item), then put into LDS.
    bf16_t* const sT = (bf16_t*)(smem + L.oT);
    constexpr int PL = F32 ? 2 : 1, groups = DS >> 3, HI = 16 * groups;   // items of a half
    struct HalfItem { Raw8<TIn> x[2][2]; };
    auto half_fetch = [&](int hf, int idx, HalfItem& y) {
      const int sp = idx / groups, c8 = idx - sp * groups;
      const int s = kHalf * hf + 2 * sp;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const unsigned o = (unsigned)((s + u < clen ? s + u : 0) * (int)vs + r0 + 8 * c8);   // (or any row that exists)
        y.x[0][u].load(vp + o);
        y.x[1][u].load(bp + o);
      }
    };
    auto half_put = [&](int hf, int idx, const HalfItem& y, bf16_t* dst) {
      const int sp = idx / groups, c8 = idx - sp * groups;
      const int s = kHalf * hf + 2 * sp;
      const bool on0 = s < clen, on1 = s + 1 < clen;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float a0 = y.x[t][0].get(e), a1 = y.x[t][1].get(e);
          a0 = on0 ? a0 : 0.f;
          a1 = on1 ? a1 : 0.f;
          bf16_t* p = dst + ((t * PL) * DS + 8 * c8 + e) * kHS + 2 * sp;
          const bf16x2 hi = pack2(a0, a1);
          *(bf16x2*)p = hi;
          if constexpr (F32) *(bf16x2*)(p + DS * kHS) = pack2(a0 - (float)hi[0], a1 - (float)hi[1]);
        }
    };
    // the wave's k in operand layout (tokens 8g + j of the half; operand row i is column i & 3 of lane group i >> 2)
    TIn kt[8];
    auto load_kt = [&](int hf) {
      int lx = lane;
      asm volatile("" : "+v"(lx));
      const int i = lx & 15, g = lx >> 4;
      const int col = nw + DN * (i >> 2) + (i & 3);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int s = kHalf * hf + 8 * g + j;
        const bool ok = (DN == 4 || (i & 3) < DN) && s < clen;
        const TIn x = kp[(int64_t)(ok ? s : 0) * qks + (ok ? col : 0)];
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
      fetch(last);
      half_fetch(0, min(tp, HI - 1), y0);
      half_fetch(two, min(tp, HI - 1), y1);
      base_fetch(bs);
      load_kt(0);
      {
      if (w == 0) {
        const float gh = a.g[h] * kLog2e;
        const float gt = (lane < clen) ? load_gate(a.gt, (int64_t)(t0 + lane) * H + h, a.gate_bf16) : 0.f;
        const float c = wave_inclusive_scan(-gt * gh, lane);
        sC[lane] = c;
        sX[lane] = 0.f;
        sF[lane] = fast_exp2(-gt * gh);
        if (lane == 63) {
          if (!PARTS || (n0 | r0) == 0) A.wFtot[(int64_t)cidx * H + h] = c;
          sF[kC] = 1.f;
        }
      }
      __syncthreads();
      // row j < kSub: weights of the tokens of the half for the state before step j; row kSub: for the state after token 31
      for (int idx = tp; idx < (kSub + 1) * kHalf; idx += NT) {
        const int j = idx / kHalf, s = idx % kHalf;
        const int hb = (j < kSub && j >= kSub / 2) ? kHalf : 0, at = j < kSub ? kG * j : kHalf;
        sW[idx] = hb + s < at ? fast_exp2(sC[at - 1] - sC[hb + s]) : 0.f;
        if (s == 0) sFB[j] = at == hb ? 1.f : fast_exp2(sC[at - 1] - (hb ? sC[hb - 1] : 0.f));
      }
      }
      for (int idx = tp; idx < HI; idx += NT) {
        if (idx >= NT) { half_fetch(0, idx, y0); half_fetch(two, idx, y1); }
        half_put(0, idx, y0, sT0);
        if (two) half_put(1, idx, y1, sT1);
      }
      base_put(bs);
      deposit(last);
      __syncthreads();
      if (two) {
        state_at(kSub, sT0);
        load_kt(1);
#pragma unroll
        for (int x = 0; x < DT; ++x) {
          *(f32x4*)(base + 256 * x) = f32x4{M[x][0], M[x][1], M[x][2], DN == 4 ? M[x][DN - 1] : 0.f};
          *(f32x4*)(base + 256 * (DT + x)) = f32x4{J[x][0], J[x][1], J[x][2], DN == 4 ? J[x][DN - 1] : 0.f};
        }
        if constexpr (!BOTH) __syncthreads();
      }
    }

    float dM[DT][DN], dJ[DT][DN];
#pragma unroll
    for (int x = 0; x < DT; ++x)
#pragma unroll
      for (int r = 0; r < DN; ++r) { dM[x][r] = 0.f; dJ[x][r] = 0.f; }
    // dq, dk: lanes with the two low bits clear store the columns oc (and, out2, oc + 1) of dq (lane bit 3 clear) or dk
    int lo = lane;
    asm volatile("" : "+v"(lo));
    const int oc = nw + DN * (lo >> 4) + 2 * ((lo >> 2) & 1), ow = (lo >> 3) & 1;
    const bool out2 = DN == 4 || (lo & 4) == 0;
    TIn* const po = (TIn*)(ow ? A.dk : A.dq) + tok0 * dk + oc;
    // bf16 rows: sums over the launches so far
    float* const pacc = PARTS ? A.pQK + ((int64_t)blockIdx.y * A.tokens * H + tok0) * (2 * dk) + ow * dk + oc
                              : A.wQK + tok0 * (2 * DNG) + ow * DNG + (oc - n0);
    const int accs = 2 * (PARTS ? dk : DNG) * H;   // per token
    const bool out_on = (lane & 3) == 0;
    // SLICE 2: what the launches over earlier value rows left for a token, requested two tokens ahead of its use
    auto acc_load = [&](int t, float* was) {
      t = t < clen ? t : 0;
      const float* acc = F32 ? (const float*)po + t * (int)dks : pacc + t * accs;
      was[0] = acc[0];
      was[1] = acc[out2 ? 1 : 0];
    };

    for (int j = last; j >= 0; --j) {
      if (j == kSub / 2 - 1 && two) {   // on to the first half
        BaseIn bs;
        base_fetch(bs);
        load_kt(0);
        if constexpr (!BOTH) {
          int it0 = tid;
          asm volatile("" : "+v"(it0));
          for (int idx = it0; idx < HI; idx += NT) {
            HalfItem y;
            half_fetch(0, idx, y);
            half_put(0, idx, y, sT);
          }
        }
        base_put(bs);
        if constexpr (!BOTH) __syncthreads();
      }
      if (j > 0) fetch(j - 1);
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
      const float* fs = sF + kG * j;
      const int o_tok = kG * j * (int)dks;   // (64 tokens of a tile stay within 32 bits)
      float sM[kG][DT][DN], sJ[kG][DT][DN];   // state after each token; in reverse mu and 1 / I in their place
      // ---- forward over the step; a token's operands are requested during the arithmetic of the token before it
      TokFwd<DT> xf[kG], xr[kG];
      TokRev<DT, VAR> yr[kG];
      xf[0].load(krow, vrow, fs, plane);
#pragma unroll
      for (int u = 0; u < kG; ++u) {
        const TokFwd<DT>& x = xf[u];
        __builtin_amdgcn_sched_barrier(0);
        if (u + 1 < kG) xf[u + 1].load(krow + (u + 1) * 32, vrow + (u + 1) * SV, fs + u + 1, plane);
        else yr[u].load(krow + u * 32, vrow + u * SV, fs + u, plane);
#pragma unroll
        for (int r = 0; r < DN; ++r) {
          const float kk = x.k[r] * x.k[r];
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            sM[u][d][r] = fmaf(x.v[d], x.k[r], (u ? sM[u ? u - 1 : 0][d][r] : M[d][r]) * x.f);
            sJ[u][d][r] = fmaf(x.b[d], kk, (u ? sJ[u ? u - 1 : 0][d][r] : J[d][r]) * x.f);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // the gate of the first token of the step after, which saw the state after this one
      float next_gate = 0.f;
#pragma unroll
      for (int r = 0; r < DN; ++r)
#pragma unroll
        for (int d = 0; d < DT; ++d) next_gate = fmaf(dM[d][r], sM[kG - 1][d][r], fmaf(dJ[d][r], sJ[kG - 1][d][r], next_gate));
      next_gate *= fs[kG];
      asm volatile("" : "+v"(next_gate));
      __builtin_amdgcn_sched_barrier(0);
      // ---- and in reverse
      float* part = smem + L.oPart + ((j & 1) * NBW + w) * (kG * 32 * DT);
      float xs[kG / 2], xo, oz[kG][2], was[kG][2], S = 0.f;
      if constexpr (SLICE == 2) acc_load(kG * j + kG - 1, was[kG - 1]);
      TokSums<DT, DN> ts[2];
      auto finish = [&](int u, TokSums<DT, DN>& z) {
        z.stage_c();
        oz[u][0] = SLICE == 2 ? z.z0 + was[u][0] : z.z0;
        oz[u][1] = SLICE == 2 ? z.z1 + was[u][1] : z.z1;
        float* pu = part + u * (32 * DT);
        if constexpr (DT >= 3) {
          if (lane < 16 * DT) {
            pu[lane] = z.p[0];
            pu[16 * DT + lane] = z.q[0];
          }
        } else {
          if (lane < 32 * DT) pu[lane] = z.p[0];
        }
        if (u & 1) xo = z.X;
        else xs[u >> 1] = pair_bit3(z.X, xo);
      };
#pragma unroll
      for (int u = kG - 1; u >= 0; --u) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (SLICE == 2) { if (u > 0) acc_load(kG * j + u - 1, was[u - 1]); }
        const TokFwd<DT>& x = u + 1 < kG ? xr[u] : xf[u];
        const TokRev<DT, VAR>& y = yr[u];
        float dq[DN], dqv[DN], dkM[DN], dkJ[DN], dvp[DT], dbp[DT], gate = 0.f;
        TokSums<DT, DN>& before = ts[(u + 1) & 1];   // of the token worked before this one
        if (u + 1 < kG) before.stage_a();
#pragma unroll
        for (int r = 0; r < DN; ++r) {
          if (r > 0) __builtin_amdgcn_sched_barrier(0);
          if (r == 1 && u + 1 < kG) before.stage_b();
          if (r == 2 && u + 1 < kG) finish(u + 1, before);
          if (r == DN - 2 && u > 0) {   // half of mu, r of this token are dead: room for the next token's operands
            xr[u - 1].load(krow + (u - 1) * 32, vrow + (u - 1) * SV, fs + u - 1, plane);
            yr[u - 1].load(krow + (u - 1) * 32, vrow + (u - 1) * SV, fs + u - 1, plane);
          }
          __builtin_amdgcn_s_setprio(3);
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            sJ[u][d][r] = fast_rcp(sJ[u][d][r] + Ip);
            asm volatile("" : "+v"(sJ[u][d][r]));
          }
          __builtin_amdgcn_s_setprio(0);
#pragma unroll
          for (int d = 0; d < DT; ++d) sM[u][d][r] *= sJ[u][d][r];
          const float kk = x.k[r] * x.k[r], q2 = y.q[r] * y.q[r];
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            const float p = y.d_o[d] * y.q[r], ri = sJ[u][d][r], m = sM[u][d][r];
            const float dl = p * ri;
            float t;
            if constexpr (VAR) {
              const float go = y.d_ov[d] * q2;
              t = fmaf(go, ri, p * m) * ri;
              dqv[r] = d ? fmaf(y.d_ov[d], ri, dqv[r]) : y.d_ov[d] * ri;
            } else {
              t = dl * m;
            }
            dM[d][r] = fmaf(dM[d][r], y.fn, dl);
            dJ[d][r] = fmaf(dJ[d][r], y.fn, -t);
            S += t;
            if (u > 0) gate = fmaf(dM[d][r], sM[u ? u - 1 : 0][d][r], fmaf(dJ[d][r], sJ[u ? u - 1 : 0][d][r], gate));
            dq[r] = d ? fmaf(m, y.d_o[d], dq[r]) : m * y.d_o[d];
            dkM[r] = d ? fmaf(dM[d][r], x.v[d], dkM[r]) : dM[d][r] * x.v[d];
            dkJ[r] = d ? fmaf(dJ[d][r], x.b[d], dkJ[r]) : dJ[d][r] * x.b[d];
            dvp[d] = r ? fmaf(dM[d][r], x.k[r], dvp[d]) : dM[d][r] * x.k[r];
            dbp[d] = r ? fmaf(dJ[d][r], kk, dbp[d]) : dJ[d][r] * kk;
          }
        }
        TokSums<DT, DN>& mine = ts[u & 1];
        mine.X = u > 0 ? x.f * gate : next_gate;
        asm volatile("" : "+v"(S), "+v"(mine.X));
#pragma unroll
        for (int r = 0; r < DN; ++r) {
          mine.o[r] = VAR ? fmaf(2.f * y.q[r], dqv[r], dq[r]) : dq[r];
          mine.o[DN + r] = fmaf(2.f * x.k[r], dkJ[r], dkM[r]);
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
      }
      __builtin_amdgcn_sched_barrier(0);
      ts[0].stage_a();
      ts[0].stage_b();
      finish(0, ts[0]);
      if (out_on) {
#pragma unroll
        for (int u = 0; u < kG; ++u) {
          if (kG * j + u < clen) {
            TIn* o = po + (o_tok + u * (int)dks);
            bool done = true;
            if constexpr (PARTS || (SLICE != 0 && !F32)) {   // the value rows of the launches add up, in fp32
              if (PARTS || (R.flags & kRectRowsAfter)) {
                float* acc = pacc + (kG * j + u) * accs;
                acc[0] = oz[u][0];
                if (out2) acc[1] = oz[u][1];
                done = false;
              }
            }
            if (done) {
              if constexpr (DN == 4) {
                store_vec<2>(o, oz[u]);
              } else {
                o[0] = from_f32<TIn>(oz[u][0]);
                if (out2) o[1] = from_f32<TIn>(oz[u][1]);
              }
            }
          }
        }
      }
      ssum += S;
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
      if (j > 0) deposit(j - 1);
      __syncthreads();
    }
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
    const float f_first = sF[0];
    int lx = lane;
    asm volatile("" : "+v"(lx));
    const int ci = lx & 15, cn = nw + DN * (lx >> 4);
#pragma unroll
    for (int x = 0; x < DT; ++x) {
      const int64_t co = tile_off + (r0 + 16 * x + ci) * dk + cn;
      float rm[DN], rj[DN];
#pragma unroll
      for (int r = 0; r < DN; ++r) { rm[r] = f_first * dM[x][r]; rj[r] = f_first * dJ[x][r]; }
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
    x = lane ? sX[lane] : sF[0] * x;
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
      rows = P.on ? P.rows : tile_rows(R.cols, dv - R.r0, sizeof(TIn) == 4);
      R.flags = P.on ? kRectParts : (R.n0 ? kRectColsBefore : 0) | (R.r0 ? kRectRowsBefore : 0) | (R.r0 + rows < dv ? kRectRowsAfter : 0);
      int rc;
      switch (rows) {
        case 16: rc = launch_tile_d<TIn, 1, VAR>(A, R, s); break;
        case 32: rc = launch_tile_d<TIn, 2, VAR>(A, R, s); break;
        case 48: rc = launch_tile_d<TIn, 3, VAR>(A, R, s); break;
        case 64: rc = launch_tile_d<TIn, 4, VAR>(A, R, s); break;
        default: rc = PAL_E_HEADDIM;
      }
      if (rc) return rc;
    }
    R.group += R.groups;
  }
  return PAL_OK;
}

}  // namespace pal
