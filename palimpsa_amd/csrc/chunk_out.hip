// Chunked Palimpsa forward, outputs: chunk_out_kernel.
//
// From the state at the start of every tile (chunk_states.hip, or the two kernels of chunk_fwd.hip) all tiles of 64
// tokens are worked in parallel (PAL_FLAG_SPARSE_STATES: walks of up to four tiles, see out_tiles_per_state).
// Inside a tile the recurrence is run token by token on the vector units in fp32,
//   M <- f_t M + v_t k_t^T,   I <- f_t I + b_t (k_t*k_t)^T + (1 - f_t) Ip,   o_t = scale (M / I) q_t
// (the naive recurrence, chunk_palimpsa_forgetting_scalar.py:712-717 of the reference; its associative scan over a
// register tile, :190-207, is what the chunked kernel of the reference does instead).
//
// Why not on the matrix cores: a state entry costs four plain fp32 instructions to advance (two per branch).  As prefix
// products it costs 12 matrix instructions of 16 cycles per 16 entries of a lane plus the operands, more issue time than
// the four, and rounds the operands.  What bounds the kernel is vector issue: per entry and token six fp32
// instructions and one reciprocal, or (scaled form) six and half a reciprocal.
//
// Scaled form (bf16 rows without the uncertainty output): with F_t the decay since the start of a group of tokens, M = F M',
// I - Ip = F J':
//   M' <- M' + (v_t / F_t) k_t^T,   J' <- J' + (b_t / F_t) (k_t*k_t)^T,   M / I = M' / (J' + Ip / F_t)
// so that the decay costs an addition per entry and token instead of two products and one addition, v / F and b / F once a
// row; two entries share a reciprocal, n1/x1 + n2/x2 = (n1 x2 + n2 x1) / (x1 x2).  A group is 64, 32, 16 or 8 tokens, the longest
// over which no group of the tile decays by more than 2^30 (a gate of 0.5 at a rate of 1: 2^-23 over 32): M', J' take the group's
// decay, and the largest precision is looked for, only at its end.  Against a float64 recurrence the outputs
// are as exact as in plain form to three digits (bf16 rounding is all of the error); in fp32 the error of the outputs would
// be up to 0.5 % larger and that of the uncertainty 15 %, so fp32 rows and the uncertainty keep the plain form.  A walk
// takes it where every eight tokens decay by less than 2^48, and is done again in plain form if a total is not finite
// or a precision over F beyond 2^61 (then a product of two may have no reciprocal).  Plain form -> groups of
// eight -> groups up to 64 and staging on all waves: 65536 tokens of 16 heads of 128x128 3060 -> 2805 -> 2750 us (2820 with
// states of segments to add up), 32768 of 16 of
// 96x96 945 -> 871 -> 857, 8 x 2048 of 12 of 64x64 without a backward 168 -> 160 (the last step), of 16 of 48x48 144 -> 140.  (Two rows a lane are held
// to four waves a SIMD: five, which 16 key columns would allow, leave some compute units 18 workgroups where an even share is 16 and the
// fifth wave without a partner: 8 x 2048, 16 heads of 16x16 40.5 -> 45.4 us.)
// (112 vector instructions a token for a lane's 16 entries at 64x64, 96 of them the entries' own; a step of eight tokens adds
// 60 for staging.  Four rows a lane halve the reads of LDS and the totals over the lanes, but leave two waves per SIMD: 193 us at 64x64.)
//
// How a SIMD of gfx950 issues these (profiles/issue_rates.txt): a lone wave issues an fp32 add, mul or fma per 5 cycles; two waves
// issue one each in the same cycles (2.4 to 2.6 per instruction), a reciprocal takes 8.2 with no other beside it, and the
// oldest wave goes first.  So (1) a wave that reaches its reciprocals is starved by the older ones' fp32 instructions, and
// those then run alone at half rate: the reciprocals of a token are issued as one burst at raised wave priority
// (s_setprio; B=8 T=2048 H=12 64x64: 185 -> 161 us); (2) fp32 instructions with a scalar-register operand do not pair
// (every operand comes from LDS into vector registers, wave-uniform ones too); (3) an odd number of waves on a
// SIMD leaves one without a partner (two or four waves, not three: at most 128 registers).
// Ideal by these rates: 6 x 2.4 + 8.2 = 22.6 cycles per entry and wave in plain form, 18.5 in scaled form; measured 27.9 and 25.3
// (profiles/bench_c1.sq_counters_pmc.txt).
// Against the earlier kernels on the matrix cores: 64x64 B=8 T=2048 H=12 250 -> 155 us, 128x128 B=2 T=4096 H=16
// 568 -> 388, 96x96 B=8 T=2048 H=16 0.287 -> 0.202 ps per entry, fp32 rows at 64x64 570 -> 160 us (they ran split operands).
//
// Layout: a wave holds a block of the state, NG lanes along the key columns x 64 / NG lanes along the value rows, DN
// columns x DD rows per lane in registers.  Blocking the registers both ways keeps the LDS traffic low (3 DN + 2 DD words
// per DN x DD entries), and the sum over the key columns is mostly in-lane.
#include <type_traits>

#include "chunk_common.h"
#include "pal_host.h"
#include "pal_profile.h"
#include "state_block.h"

namespace pal {

// Least decay over eight tokens for the scaled form, and largest precision over F: the product of two of the latter still
// has a reciprocal in fp32.  Steps that decay more are rare (gates of 0.5 at a rate of 2: 2^-12) and gain least from it.
constexpr float kMinDecay = 0x1p-48f, kMaxScaled = 0x1p61f;
// Least decay over sixteen, 32 or 64 tokens for the decay to be applied to the state only after them.
constexpr float kMinLong = 0x1p-30f;
constexpr int kOT = 8;   // tokens per staging step: two buffers of them let four workgroups of four waves share a unit's LDS

template <int DD>
__device__ __forceinline__ void lds_rows(const float* p, float* out) {
  if constexpr (DD % 4 == 0) {
#pragma unroll
    for (int x = 0; x < DD / 4; ++x) *(f32x4*)&out[4 * x] = *(const f32x4*)&p[4 * x];
  } else if constexpr (DD % 2 == 0) {
#pragma unroll
    for (int x = 0; x < DD / 2; ++x) {
      const f32x2 y = *(const f32x2*)&p[2 * x];
      out[2 * x] = y[0]; out[2 * x + 1] = y[1];
    }
  } else {
#pragma unroll
    for (int x = 0; x < DD; ++x) out[x] = p[x];
  }
}

// a lane's operands of one token
template <int NG, int DN, int DD>
struct OutRow {
  float k[DN], kk[DN], q[DN], vb[2 * DD];
  f32x2 fc;
  __device__ __forceinline__ void load(const float* row, int ng, int d0) {
    constexpr int DKP = NG * DN;
    fc = *(const f32x2*)row;
    lds_cols<NG, DN>(row + 4, ng, k);
    lds_cols<NG, DN>(row + 4 + DKP, ng, kk);
    lds_rows<2 * DD>(row + 4 + 3 * DKP + 2 * d0, vb);
    lds_cols<NG, DN>(row + 4 + 2 * DKP, ng, q);
  }
};

template <int N>
__device__ __forceinline__ float dpp_shr(float x) {   // lane i of a row of 16 takes lane i - N
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x110 + N, 0xf, 0xf, true));
}

// SEGS: the states are kept since the start of a segment (state_pass_segments; an instance of its own: the branch and its
// values took 1 to 2 % from calls that have none)
template <typename TIn, int NG, int DN, int DD, bool HAS_VAR, bool SEGS>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 512), amdgpu_waves_per_eu(HAS_VAR ? 2 : 4, !HAS_VAR && DD == 2 ? 4 : 8)))
void chunk_out_kernel(ChunkArgs a, int W) {
  extern __shared__ float smem[];
  typedef typename Raw4<TIn>::type raw4;
  constexpr int DKP = NG * DN;              // key columns of the lanes (dk, or up to 16 more that stay zero)
  constexpr int ROWS = (64 / NG) * DD;      // value rows of a wave
  constexpr int TU = 4 / DD;                // tokens per iteration
  constexpr bool kMayScale = std::is_same<TIn, bf16_t>::value && !HAS_VAR;
  const int NT = W * 64, VR = W * ROWS;     // threads and value rows of the workgroup
  constexpr int oK = 4, oKK = oK + DKP, oQ = oKK + DKP, oVB = oQ + DKP;
  const int STRIDE = oVB + 2 * VR;          // floats per staged token: f, c, -, -, k, k*k, q, (v, b) of every row
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int H = a.H, dk = a.dk, dv = a.dv;
  const int walks = a.every > 1 ? a.n_seqs * (((a.T + kC - 1) / kC + a.every - 1) / a.every) : a.total_chunks;
  int cidx, h;
  if (!tile_head(walks, H, (int)blockIdx.x, cidx, h)) return;
  const int r0 = (int)blockIdx.y * VR;
  int seq, t0, clen, cis;
  if (a.every > 1) {   // batched sequences of one length, `every` tiles from one state
    const int tiles = (a.T + kC - 1) / kC, per = (tiles + a.every - 1) / a.every;
    seq = cidx / per;
    cis = (cidx - seq * per) * a.every;
    cidx = seq * tiles + cis;
    t0 = seq * a.T + cis * kC;
    clen = min(a.every * kC, a.T - cis * kC);
  } else {
    chunk_lookup(a, cidx, seq, t0, clen, cis);
  }
  float* sFC = smem;                        // [tokens][4] f_t (scaled form: F_t), c_t, factor of v and b, f_t
  int* sForm = (int*)(sFC + 4 * kC * a.every);   // whether the tiles are worked in scaled form
  int* sLen = sForm + 1;                         // [every] scaled form: tokens after which the decay is applied
  float* sRow = sFC + 4 * kC * a.every + 8;      // [2][kOT][STRIDE]
  const float Ip = a.Ip[h];
  // every fetch of the set-up is issued before the first is used
  const float gt = 64 * w + lane < clen ? load_gate(a.gt, (int64_t)(t0 + 64 * w + lane) * H + h, a.gate_bf16) : 0.f;
  const float gh = a.g[h] * kLog2e;
  const TIn* kp = (const TIn*)a.k + qk_row(a, t0, h);
  const TIn* qp = (const TIn*)a.q + qk_row(a, t0, h);
  const TIn* vp = (const TIn*)a.v + ((int64_t)t0 * H + h) * dv + r0;
  const TIn* bp = (const TIn*)a.b + ((int64_t)t0 * H + h) * dv + r0;
  const int qs = (int)qk_stride(a), vs = H * dv;
  // staging items: (token, four columns) of k and q, (token, four rows) of v and b
  const int nk4 = dk >> 2, nv4 = min(VR, dv - r0) >> 2;
  raw4 rk, rq, rv, rb;
  // (v and b by the threads after those of k and q, where there are as many: the first waves of all workgroups share a SIMD)
  const int o_vb = kOT * (nk4 + nv4) <= NT ? kOT * nk4 : 0, i_vb = tid >= o_vb ? tid - o_vb : NT;
  const int s_kq = tid / nk4, c_kq = tid - s_kq * nk4, s_vb = i_vb / nv4, c_vb = i_vb - s_vb * nv4;
  auto fetch = [&](int s0) {
    if (s_kq < kOT && s0 + s_kq < clen) {
      rk = *(const raw4*)(kp + (int64_t)(s0 + s_kq) * qs + 4 * c_kq);
      rq = *(const raw4*)(qp + (int64_t)(s0 + s_kq) * qs + 4 * c_kq);
    }
    if (s_vb < kOT && s0 + s_vb < clen) {
      rv = *(const raw4*)(vp + (int64_t)(s0 + s_vb) * vs + 4 * c_vb);
      rb = *(const raw4*)(bp + (int64_t)(s0 + s_vb) * vs + 4 * c_vb);
    }
  };
  auto put_kq = [&](float* row, int c, raw4 k4, raw4 q4) {
    f32x4 x, xx, y;
#pragma unroll
    for (int e = 0; e < 4; ++e) { x[e] = (float)k4[e]; xx[e] = x[e] * x[e]; y[e] = (float)q4[e]; }
    *(f32x4*)&row[oK + 4 * c] = x;
    *(f32x4*)&row[oKK + 4 * c] = xx;
    *(f32x4*)&row[oQ + 4 * c] = y;
  };
  auto deposit = [&](int s0, int buf) {
    float* base = sRow + buf * kOT * STRIDE;
    if (tid < kOT) *(f32x2*)&base[tid * STRIDE] = *(const f32x2*)&sFC[4 * (s0 + tid)];   // (inside the last tile)
    if (s_kq < kOT && s0 + s_kq < clen) put_kq(base + s_kq * STRIDE, c_kq, rk, rq);
    if (s_vb < kOT && s0 + s_vb < clen) {
      float* p = &base[s_vb * STRIDE + oVB + 8 * c_vb];
      const float u = kMayScale ? sFC[4 * (s0 + s_vb) + 2] : 1.f;
      *(f32x4*)p = f32x4{u * (float)rv[0], u * (float)rb[0], u * (float)rv[1], u * (float)rb[1]};
      *(f32x4*)(p + 4) = f32x4{u * (float)rv[2], u * (float)rb[2], u * (float)rv[3], u * (float)rb[3]};
    }
    // wide keys on few waves: the items of k, q beyond the fetched ones
    for (int idx = tid + NT; idx < kOT * nk4; idx += NT) {
      const int s = idx / nk4, c = idx - s * nk4;
      if (s0 + s < clen)
        put_kq(base + s * STRIDE, c, *(const raw4*)(kp + (int64_t)(s0 + s) * qs + 4 * c),
               *(const raw4*)(qp + (int64_t)(s0 + s) * qs + 4 * c));
    }
  };
  const int ng = OutLanes<NG>::col(lane), dg = OutLanes<NG>::row(lane);
  const int d0 = w * ROWS + dg * DD;        // first value row of the lane inside the workgroup
  // The totals of DD rows x TU tokens are reduced together: four values, of which lane bits 3 and 2 select one
  const int sel = 2 * ((lane >> 3) & 1) + ((lane >> 2) & 1);
  const int dsel = sel % DD, tsel = sel / DD;
  const bool writer = OutLanes<NG>::first(lane) && r0 + d0 + dsel < dv;
  auto reduce = [&](const float* x) {
    return OutLanes<NG>::sum_other(pair_bit2(pair_bit3(x[0], x[2]), pair_bit3(x[1], x[3])));
  };
  const int64_t orow = ((int64_t)t0 * H + h) * dv + r0 + d0 + dsel;

  // fn(t, f_t) for the tokens of this thread, whole tiles; only walks of several tiles have more than the one whose gate is there
  auto tokens = [&](auto fn) {
    if (tid < a.every * kC && tid - lane < clen) fn(tid, fast_exp2(-gt * gh));
    for (int t = tid + NT; t < a.every * kC && t - lane < clen; t += NT)
      fn(t, fast_exp2(-(t < clen ? load_gate(a.gt, (int64_t)(t0 + t) * H + h, a.gate_bf16) : 0.f) * gh));
  };
  if constexpr (kMayScale) {   // each wave: the decays of its tiles
    if (tid == 0) *sForm = 1;
    __syncthreads();
    tokens([&](int t, float f) {
      // Decay since the start of a group of eight tokens (a staging step), of sixteen and so on: the product over its tokens
      // (each shift before its select: a lane that is switched off hands nothing on)
      float F = f, P = f;
      auto shift = [&](auto by) {
        constexpr int N = decltype(by)::value;
        float y = dpp_shr<N>(F);
        if constexpr (N < kOT) F = (lane & (kOT - 1)) >= N ? F * y : F;
        y = dpp_shr<N>(P);
        P = (lane & 15) >= N ? P * y : P;
      };
      shift(std::integral_constant<int, 1>{});
      shift(std::integral_constant<int, 2>{});
      shift(std::integral_constant<int, 4>{});
      shift(std::integral_constant<int, 8>{});
      if (!__all(F >= kMinDecay && F <= 1.f && Ip <= kMinDecay * kMaxScaled)) *sForm = 0;
      auto total = [&](int l) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, P), l)); };
      const float t0 = total(15), t1 = total(31), t2 = total(47);
      const int row = lane >> 4;
      const float P32 = P * (row == 1 ? t0 : row == 3 ? t2 : 1.f), P64 = P32 * (row >= 2 ? t0 * t1 : 1.f);
      int len = kOT;
      if (__all(P >= kMinLong)) { F = P; len = 16; }
      if (__all(P32 >= kMinLong)) { F = P32; len = 32; }
      if (__all(P64 >= kMinLong)) { F = P64; len = 64; }
      if (lane == 0) sLen[t / kC] = len;
      sFC[4 * t] = F;
      sFC[4 * t + 3] = f;
    });
    __syncthreads();
  }

  // The tiles in scaled or plain form (see above); whether the scaled form left its range.
  auto walk_tile = [&](auto form) -> bool {
    constexpr bool SCALED = decltype(form)::value;
    constexpr int NR = SCALED ? (DN + 1) / 2 : DN;   // reciprocals of a row and token
    fetch(0);
    float M[DD][DN], I[DD][DN];   // SCALED: M / F and (I - Ip) / F
    {
      const float* mu = a.chunk_mu + (((int64_t)cidx * H + h) * dv + r0) * dk;
      const float* Is = a.chunk_I + (((int64_t)cidx * H + h) * dv + r0) * dk;
      const int seg = SEGS ? cis / a.seg_tiles : 0;
      const int64_t before = SEGS ? seg_slot(a, seq, seg, h) + (int64_t)r0 * dk : 0;
      const SegDecay Fseg = SEGS ? seg_decays(a, seq, seg)[(cis - seg * a.seg_tiles) / a.every * H + h] : SegDecay{};
#pragma unroll
      for (int j = 0; j < DD; ++j) {
        const bool on = r0 + d0 + j < dv;
        const int64_t ro = (int64_t)(on ? d0 + j : 0) * dk;
        auto piece = [&](auto width, int i) {
          constexpr int VW = decltype(width)::value;
          const int c = col_of<NG, DN>(i, ng);
          float x[VW], y[VW];
          const bool in = DKP == 0 || c < dk;
          load_vec<VW>(mu + ro + (in ? c : 0), x);
          load_vec<VW>(Is + ro + (in ? c : 0), y);
          if constexpr (SEGS) {   // sums since the start of the segment: the state before it is added
            float m[VW], J[VW];
            load_vec<VW>(a.chunk_mu + before + ro + (in ? c : 0), m);
            load_vec<VW>(a.chunk_I + before + ro + (in ? c : 0), J);
#pragma unroll
            for (int e = 0; e < VW; ++e) {
              M[j][i + e] = on && in ? Fseg.apply(m[e], x[e]) : 0.f;
              const float J1 = Fseg.apply(J[e], y[e]);
              I[j][i + e] = on && in ? (SCALED ? J1 : J1 + Ip) : 1.f;
            }
          } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) {
              M[j][i + e] = on && in ? x[e] * y[e] : 0.f;
              I[j][i + e] = on && in ? (SCALED ? y[e] - Ip : y[e]) : 1.f;
            }
          }
        };
#pragma unroll
        for (int p = 0; p < DN / 4; ++p) piece(std::integral_constant<int, 4>{}, 4 * p);
        if constexpr ((DN & 3) >= 2) piece(std::integral_constant<int, 2>{}, 4 * (DN / 4));
        if constexpr (DN & 1) piece(std::integral_constant<int, 1>{}, DN - 1);
      }
    }
    if constexpr (kMayScale) {
      for (int t = tid; t < a.every * kC && t - lane < clen; t += NT) {   // (the thread that left f and F there)
        const float f = sFC[4 * t + 3], F = SCALED ? sFC[4 * t] : f, inv = SCALED ? fast_rcp(F) : 1.f;
        *(f32x4*)&sFC[4 * t] = f32x4{F, SCALED ? Ip * inv : (1.f - f) * Ip, inv, f};
      }
    } else {
      tokens([&](int t, float f) { *(f32x2*)&sFC[4 * t] = f32x2{f, (1.f - f) * Ip}; });
    }
    // rows and columns beyond the head dims stay zero in both buffers
    if (DKP != dk || VR > dv - r0) {
      for (int idx = tid; idx < 2 * kOT * STRIDE; idx += NT) sRow[idx] = 0.f;
    }
    __syncthreads();
    deposit(0, 0);
    __syncthreads();

    bool bad = false;
    float big = 0.f;   // SCALED: the largest |I - Ip| / F
    OutRow<NG, DN, DD> x;
    for (int s0 = 0; s0 < clen; s0 += kOT) {
      const int buf = (s0 / kOT) & 1;
      const bool more = s0 + kOT < clen;
      if (more) fetch(s0 + kOT);
      const int nt = min(kOT, clen - s0);
      const float* row = sRow + buf * kOT * STRIDE;
      const int len = SCALED ? __builtin_amdgcn_readfirstlane(sLen[s0 / kC]) : 0;
      x.load(row, ng, d0);
#pragma unroll 1
      for (int tt = 0; tt < nt; tt += TU, row += TU * STRIDE) {
        float acc[4], accv[4];
#pragma unroll
        for (int u = 0; u < TU; ++u) {
          float num[DD][NR], numv[DD][NR], den[DD][NR];
#pragma unroll
          for (int i = 0; i < DN; ++i)
#pragma unroll
            for (int j = 0; j < DD; ++j) {
              if constexpr (SCALED) {
                M[j][i] = fmaf(x.vb[2 * j], x.k[i], M[j][i]);
                I[j][i] = fmaf(x.vb[2 * j + 1], x.kk[i], I[j][i]);
                if (i & 1) {   // n1 / x1 + n2 / x2 = (n1 x2 + n2 x1) / (x1 x2)
                  const float x1 = I[j][i - 1] + x.fc[1], x2 = I[j][i] + x.fc[1];
                  num[j][i / 2] = fmaf(M[j][i] * x.q[i], x1, M[j][i - 1] * x.q[i - 1] * x2);
                  den[j][i / 2] = x1 * x2;
                } else if (i == DN - 1) {
                  num[j][i / 2] = M[j][i] * x.q[i];
                  den[j][i / 2] = I[j][i] + x.fc[1];
                }
              } else {
                M[j][i] = fmaf(x.vb[2 * j], x.k[i], M[j][i] * x.fc[0]);
                fma3(I[j][i], x.fc[0], x.fc[1]);
                I[j][i] = fmaf(x.vb[2 * j + 1], x.kk[i], I[j][i]);
                num[j][i] = x.q[i];
                if constexpr (HAS_VAR) numv[j][i] = x.q[i] * x.q[i];
                den[j][i] = I[j][i];
              }
            }
          __builtin_amdgcn_sched_barrier(0);
          // the next token's operands are requested here: the burst of reciprocals hides their latency (after the last
          // token of a step: rows of the other buffer or, at its end, not yet written; they are read again below)
          x.load(row + (u + 1) * STRIDE, ng, d0);
          __builtin_amdgcn_s_setprio(3);
#pragma unroll
          for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int j = 0; j < DD; ++j) den[j][i] = fast_rcp(den[j][i]);
          __builtin_amdgcn_s_setprio(0);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int j = 0; j < DD; ++j) { acc[u * DD + j] = 0.f; accv[u * DD + j] = 0.f; }
#pragma unroll
          for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int j = 0; j < DD; ++j) {
              float& y = acc[u * DD + j];
              if constexpr (SCALED) y = fmaf(num[j][i], den[j][i], y);
              else y = fmaf(M[j][i] * den[j][i], num[j][i], y);
              if constexpr (HAS_VAR) accv[u * DD + j] = fmaf(numv[j][i], den[j][i], accv[u * DD + j]);
            }
        }
        const int t = s0 + tt + tsel;
        const bool wr = writer && t < clen;
        const int64_t oo = orow + (int64_t)t * vs;
        const float out = reduce(acc);
        if (wr) ((TIn*)a.o)[oo] = from_f32<TIn>(out * a.scale);
        if (SCALED) bad |= wr && !(__builtin_fabsf(out) < __builtin_inff());
        if constexpr (HAS_VAR) {
          const float outv = reduce(accv);
          if (wr) store_rt(a.o_var, oo, outv * a.scale, a.var_bf16);
        }
      }
      if constexpr (SCALED) {
        if (!more || ((s0 + kOT) & (len - 1)) == 0) {
          // (b and Ip are not negative: precisions over F are largest before the decay is applied)
#pragma unroll
          for (int i = 0; i < DN; ++i)
#pragma unroll
            for (int j = 0; j < DD; ++j) big = fmaxf(big, __builtin_fabsf(I[j][i]));
          const float Fe = sFC[4 * (s0 + kOT - 1)];   // (inside the last tile)
#pragma unroll
          for (int i = 0; i < DN; ++i)
#pragma unroll
            for (int j = 0; j < DD; ++j) { M[j][i] *= Fe; I[j][i] *= Fe; }
        }
      }
      if (more) deposit(s0 + kOT, buf ^ 1);
      __syncthreads();
    }
    return bad || !(big <= kMaxScaled);
  };
  if constexpr (kMayScale) {
    if (*sForm && !__syncthreads_or(walk_tile(std::true_type{}))) return;
  }
  walk_tile(std::false_type{});
}

// Waves per workgroup for nw waves of value rows: the hardware deals the waves of a workgroup out to the four SIMDs in
// order, so four (or two) to a workgroup load them evenly and five or six do not (96x96, twelve waves: 0.202 ps per
// entry in workgroups of four, 0.225 in threes, 0.26 in sixes; 48x96, six waves: 0.207 in twos, 0.224 in threes, 0.26 in one
// six; 80x80, ten waves: 0.257 in twos, 0.35 in fives).
static int out_waves(int nw) {
  if (nw <= 4) return nw;
  if (nw % 4 == 0) return 4;
  if (nw % 2 == 0) return 2;
  return nw % 4 == 3 ? 4 : 3;
}

template <typename TIn, int NG, int DN, int DD>
static int launch_out_dd(const ChunkArgs& a, hipStream_t s) {
  constexpr int ROWS = (64 / NG) * DD;
  static_assert(ROWS <= 32, "one staging item of v, b per thread");
  const int nw = (a.dv + ROWS - 1) / ROWS;            // waves over the value rows
  const int W = out_waves(nw), slices = (nw + W - 1) / W;
  const int64_t walks = a.every > 1 ? (int64_t)a.n_seqs * (((a.T + kC - 1) / kC + a.every - 1) / a.every) : a.total_chunks;
  const int64_t blocks = tile_head_blocks(walks, a.H);
  if (blocks > 0x7fffffff) return PAL_E_DIM;
  const size_t lds = sizeof(float) * (4 * kC * a.every + 8 + (2 * kOT + 1) * (4 + 3 * NG * DN + 2 * (size_t)W * ROWS));
  if (lds > kMaxLds) return PAL_E_HEADDIM;
  auto go = [&](auto kern) -> int {
    if (int rc = allow_lds((const void*)kern, lds)) return rc;
    PAL_TIMED_LAUNCH(kKernChunkOut, s, kern, dim3((unsigned)blocks, (unsigned)slices), dim3(64 * W), lds, s, a, W);
    return 0;
  };
  const bool var = a.flags & PAL_FLAG_HAS_VAR;
  int rc;
  if (a.segs <= 1) {
    rc = var ? go(&chunk_out_kernel<TIn, NG, DN, DD, true, false>) : go(&chunk_out_kernel<TIn, NG, DN, DD, false, false>);
  } else {
    if constexpr (DD == 2 && sizeof(TIn) == 2) {
      rc = var ? go(&chunk_out_kernel<TIn, NG, DN, DD, true, true>) : go(&chunk_out_kernel<TIn, NG, DN, DD, false, true>);
    } else {
      rc = PAL_E_DIM;   // (out_takes_segments)
    }
  }
  if (rc) return rc;
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

// Two value rows per lane where that still gives every SIMD two waves; below, one row: half the work per wave and
// twice the waves (one sequence of 777 tokens, 16 heads of 64x64: 28 us with two rows, 23 with one; B=2 T=2048 H=12 64x64,
// three waves per SIMD: 49.6 against 51.0).
static int out_lane_rows(const ChunkArgs& a, int NG) {
  return (int64_t)a.total_chunks / a.every * a.H * ((a.dv * NG + 127) / 128) <= 2048 ? 1 : 2;
}

template <typename TIn, int NG, int DN>
static int launch_out_dn(const ChunkArgs& a, hipStream_t s) {
  return out_lane_rows(a, NG) == 1 ? launch_out_dd<TIn, NG, DN, 1>(a, s) : launch_out_dd<TIn, NG, DN, 2>(a, s);
}

// Whether launch_out takes states of segments: there are instances for them with two rows to a lane only (as many tiles as
// make segments fill the SIMDs; see out_tiles_per_state).
bool out_takes_segments(const ChunkArgs& a, int dtype) {
  const int NG = a.dk <= 32 ? 4 : a.dk <= 64 ? 8 : a.dk <= 128 ? 16 : 32;   // (as launch_out_t)
  return dtype == PAL_DTYPE_BF16 && out_lane_rows(a, NG) == 2;
}

template <typename TIn>
static int launch_out_t(const ChunkArgs& a, hipStream_t s) {
  switch ((a.dk + 15) / 16) {
    case 1: return launch_out_dn<TIn, 4, 4>(a, s);
    case 2: return launch_out_dn<TIn, 4, 8>(a, s);
    case 3: return launch_out_dn<TIn, 8, 6>(a, s);
    case 4: return launch_out_dn<TIn, 8, 8>(a, s);
    case 5: return launch_out_dn<TIn, 16, 5>(a, s);
    case 6: return launch_out_dn<TIn, 16, 6>(a, s);
    case 7: return launch_out_dn<TIn, 16, 7>(a, s);
    case 8: return launch_out_dn<TIn, 16, 8>(a, s);
    case 9: case 10: return launch_out_dn<TIn, 32, 5>(a, s);
    case 11: case 12: return launch_out_dn<TIn, 32, 6>(a, s);
    case 13: case 14: return launch_out_dn<TIn, 32, 7>(a, s);
    case 15: case 16: return launch_out_dn<TIn, 32, 8>(a, s);
    default: return PAL_E_HEADDIM;
  }
}

// Tiles that a walk of the output kernel takes from one state, where nothing else reads the states between: as many, up to
// four, as leave one and a half rounds of waves (four per SIMD, about 1024 state entries each).  What it saves is the state
// pass's writes and this kernel's reads; what it costs is the serial length.  States and outputs together, in us, with 1, 2, 4
// and 8 tiles to a state: 65536 tokens, 16 heads of 128x128 (65536 waves a window) 3925, 3663, 3524, 3534; 2 x 4096, 16 of
// 128x128 (32768) 478, 424, 410, 424; 8 x 2048, 12 of 64x64 (12288) 182, 177, 188, 216; 4 x 2048, 6 of 96x192 (13824) 240,
// 235, 263, 304; 16 x 512, 24 of 48x48 (6912) 137, 142, 159, 193.  A walk carries the state on unrounded where a kept one went
// through (mu, I), so how many sequences share a call would show in the last bits of all of them (a document of a large packed pass
// and the same one alone otherwise agree to 1e-6): only the windows of one sequence, which the library itself cuts, ask for walks.
int out_tiles_per_state(const ChunkArgs& a) {
  if (a.flags & PAL_FLAG_VARLEN) return 1;
  const int64_t tiles = (a.T + kC - 1) / kC;
  auto waves = [&](int every) {
    return (int64_t)a.n_seqs * ((tiles + every - 1) / every) * a.H * ((int64_t)a.dk * a.dv) / 1024;
  };
  return waves(4) >= 6144 ? 4 : waves(2) >= 6144 ? 2 : 1;
}

int launch_out(const ChunkArgs& a, int dtype, hipStream_t s) {
  return dtype == PAL_DTYPE_BF16 ? launch_out_t<bf16_t>(a, s) : launch_out_t<float>(a, s);
}

}  // namespace pal
