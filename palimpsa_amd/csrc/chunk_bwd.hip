// Chunked Palimpsa backward.
//
// Replaces chunk_palimpsa_bwd_kernel and the host-side reductions of
// ChunkPalimpsa.backward (chunk_palimpsa_forgetting_scalar.py:239-434, :519-620).
//
// With G_t = scale do_t q_t^T, the per-token local gradients are
//   dMloc_t = G_t / I_t,  dJloc_t = -G_t M_t / I_t^2 (- scale dovar_t (q_t*q_t)^T / I_t^2)
// and the state gradients obey the reverse recurrence dM_s = dMloc_s + f_{s+1} dM_{s+1}
// (:360-384).  All tiles of 64 tokens are processed in parallel; what crosses a
// tile boundary is handled by two small extra passes (scan, apply); the gate gradient is finished in the second:
//
//  local   per (tile, head): chunk_bwd_tile.h -- dq, the tile's own parts of dv, db, dk and of the gate gradient, and
//          the carry the tile hands to its predecessor, R_loc = f_first * dM^loc_first.
//          Heads above 64x64 in several pieces (chunk_bwd.h); a small pass works on them side by side and
//  sum     adds up their parts.
//  scan    per state entry: R_{c-1} = R_loc,c + F_C,c R_c backwards over the tiles
//          of a sequence (the role of curr_dM/curr_dI, :429-430); also yields the
//          gradients of the initial state.
//  apply   per (tile, head): adds the carry terms a_s R k_s etc. to dv, db, dk
//          with four small MFMA products.
//  gate    d log f_s = <dM_s, f_s M_{s-1}> + <dJ_s, f_s J_{s-1}>:
//            local part   gamma_s of the tile kernel;
//            carry part   sum_{r<s, r in tile} beta_r + F_C (<R_M, M_0> + <R_J, J_0>), with
//                         beta_r = <v_r, dv^carry_r> + <b_r, db^carry_r> from the apply pass and
//                         (M_0, J_0) the state at the start of the tile.
//          dgt = -g dlogf, dg = -sum gt dlogf, dIp = sum dJloc (- sum dJ_0 with an initial state).
//          Every term belongs to the token's own tile: the apply kernel writes dgt and the tile's share of dg,
//          a last small kernel sums the shares per head.
#include <type_traits>

#include "chunk_bwd.h"
#include "pal_host.h"
#include "pal_profile.h"

namespace pal {

void fill_chunk_args(ChunkArgs& a, const PalDims* d, const PalFwdTensors* t);

// ----------------------------------------------------------------- carry scan
// R_{c-1} = R_loc,c + F_c R_c backwards over the tiles of a sequence: one thread per four consecutive state
// entries of a (sequence, head), 1024 entries per block; the running sums stay in fp32 registers, the slot of a
// tile is read (its local carry) and overwritten (the carry coming in from the later tiles) in the row dtype.
__host__ __device__ inline int carry_scan_blocks(int64_t E) { return (int)((E + 1023) / 1024); }

template <typename TC>
__global__ __launch_bounds__(256) void chunk_bwd_carry_scan_kernel(BwdArgs A) {
  const ChunkArgs& a = A.c;
  __shared__ float sW[4];
  const int64_t E = (int64_t)a.dv * a.dk;
  const int nblk = carry_scan_blocks(E);
  const int blk = blockIdx.x % nblk;
  const int nh = blockIdx.x / nblk;
  const int h = nh % a.H, n = nh / a.H;
  const int64_t e = ((int64_t)blk * 256 + threadIdx.x) * 4;
  const bool on = e < E;
  int bos, len, cbase;
  seq_lookup(a, n, bos, len, cbase);
  const int nchunks = (len + kC - 1) / kC;
  TC* wDM = (TC*)A.wDM;
  TC* wDJ = (TC*)A.wDJ;
  float RM[4] = {0.f, 0.f, 0.f, 0.f}, RJ[4] = {0.f, 0.f, 0.f, 0.f};
  if (on) {
    auto advance = [&](int64_t off, const float* DM, const float* DJ, float Ft) {
      store_vec<4>(wDM + off, RM);
      store_vec<4>(wDJ + off, RJ);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        RM[x] = fmaf(Ft, RM[x], DM[x]);
        RJ[x] = fmaf(Ft, RJ[x], DJ[x]);
      }
    };
    int c = nchunks - 1;
    for (; c >= 3; c -= 4) {   // four tiles' loads in flight at a time
      float DM[4][4], DJ[4][4], Ft[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t off = ((int64_t)(cbase + c - u) * a.H + h) * E + e;
        load_vec<4>(wDM + off, DM[u]);
        load_vec<4>(wDJ + off, DJ[u]);
        Ft[u] = A.wFtot[(int64_t)(cbase + c - u) * a.H + h];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        advance(((int64_t)(cbase + c - u) * a.H + h) * E + e, DM[u], DJ[u], fast_exp2(Ft[u]));
    }
    for (; c >= 0; --c) {
      const int64_t off = ((int64_t)(cbase + c) * a.H + h) * E + e;
      float DM[4], DJ[4];
      load_vec<4>(wDM + off, DM);
      load_vec<4>(wDJ + off, DJ);
      advance(off, DM, DJ, fast_exp2(A.wFtot[(int64_t)(cbase + c) * a.H + h]));
    }
  }
  if (a.init_mu) {
    const int64_t so = (int64_t)nh * E + e;
    if (A.d_init_mu && on) {
      const f32x4 mu0 = *(const f32x4*)(a.init_mu + so), I0 = *(const f32x4*)(a.init_I + so);
      const f32x4 dmu = {RM[0] * I0[0], RM[1] * I0[1], RM[2] * I0[2], RM[3] * I0[3]};
      const f32x4 dI = {fmaf(RM[0], mu0[0], RJ[0]), fmaf(RM[1], mu0[1], RJ[1]), fmaf(RM[2], mu0[2], RJ[2]),
                        fmaf(RM[3], mu0[3], RJ[3])};
      *(f32x4*)(A.d_init_mu + so) = dmu;
      *(f32x4*)(A.d_init_I + so) = dI;
    }
    // J_0 = I_0 - Ip: the prior also receives -sum dJ_0
    float s = wave_sum((RJ[0] + RJ[1]) + (RJ[2] + RJ[3]));
    if ((threadIdx.x & 63) == 0) sW[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) A.wInitPart[(int64_t)nh * nblk + blk] = sW[0] + sW[1] + sW[2] + sW[3];
  }
}

// ---------------------------------------------------------------- carry apply
// dv_s += a_s R_M k_s ; db_s += a_s R_J k_s^2 ; dk_s += a_s (R_M^T v_s + 2 k_s * R_J^T b_s)
// One workgroup of 4 waves per (tile, head); wave w owns tokens [16w, 16w+16).  The four products run on the matrix cores
// (bf16 operands, fp32 accumulate) with the tokens as columns: a lane's four results are neighbours in the row of its
// token, and in every product the operand of a lane is the same four-element pieces of that token's row, so that a
// row is fetched once, serves as operand and as the factor of the results, and the sums go back to memory from the
// registers.  Bound by HBM traffic (the rows, the gradients in and out, the carries, and the states for the boundary
// term: 375 MB at 8 x 2048 tokens, 12 heads of 64x64) and by the latency that few workgroups hide: every fetch
// is issued before the first is used, and there is one barrier between them and the results.  Carries and states are gone
// through as they lie, whole kilobytes a wave instruction: in blocks of 16 rows by 32 or 64 bytes, as the products take them,
// 107 us at that size, now 96.5 (3.9 TB/s); 16 heads of 48x48 89, 83; 32768 packed tokens, 16 of 96x96 529, 459; 8 x 2048, 8 of
// 128x128 199, 175; 4 x 1531, 16 of 48x96 53.6, 50.5; fp32 rows 8 x 2048, 8 of 64x64 95.6, 93.2.
// KSMAX = operand registers per product (32 contraction indices each: head dims up to 32 KSMAX).
// PREC (fp32 rows): operands as two bf16 halves, three matrix instructions per product; the copy of the carries in LDS
// then holds a second plane with the lo halves.
// Every wave scans the gates itself (the decay a_s of its own token rows), so the operands do not wait for another wave.
// waves per SIMD: what the rows, gradients and operands leave (64x64 squeezed into 128 registers for four: 116 us)
constexpr int apply_waves(int KSMAX, bool f32) { return f32 ? (KSMAX == 1 ? 3 : 2) : KSMAX == 1 ? 4 : KSMAX <= 3 ? 3 : 2; }
template <typename TIn, int KSMAX, bool PREC>
__global__ __attribute__((amdgpu_flat_work_group_size(256, 256), amdgpu_waves_per_eu(apply_waves(KSMAX, sizeof(TIn) == 4))))
void chunk_bwd_carry_apply_kernel(BwdArgs A) {
  const ChunkArgs& a = A.c;
  extern __shared__ float smem[];
  const int H = a.H, dk = a.dk, dv = a.dv;
  float* sW4 = smem;                       // [4] shares of the boundary term
  float* sBt = smem + 4;                   // [64] beta of the carry terms
  // [2][dv][RS] R_M, R_J in bf16 as they lie in memory, operand source of all four products: the ones that contract over
  // the key columns read pieces of a row, the ones over the value rows four rows at once, transposed on their way out
  bf16_t* sR = (bf16_t*)(smem + 4 + kC);
  const int RS = A.apply_stride;
  bf16_t* sRl = sR + 2 * dv * RS;          // PREC: [2][dv][RS] lo halves
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15, g = lane >> 4;
  int cidx, h;
  if (!tile_head(a.total_chunks, H, blockIdx.x, cidx, h)) return;
  int seq, t0, clen, cis;
  chunk_lookup(a, cidx, seq, t0, clen, cis);
  int bos, len, cbase;
  seq_lookup(a, seq, bos, len, cbase);
  const bool last = cis == (len + kC - 1) / kC - 1;
  // the gates of the tile's tokens (every wave), and for wave 0 the local part of d log f
  const bool tok_ok = lane < clen;
  const int64_t tokL = (int64_t)t0 + lane;
  const float gt_l = tok_ok ? load_gate(a.gt, tokL * H + h, a.gate_bf16) : 0.f;
  float e_l = 0.f;
  if (w == 0 && tok_ok) e_l = A.wE[(int64_t)h * A.tokens + tokL];
  // Gate gradient of the tile's tokens, by wave 0 once the carry terms are known:
  //   d log f_t = (local part, from the tile kernel) + (carry terms of the earlier tokens of the tile) + (boundary term),
  //   dgt_t = -g d log f_t, and the tile's share of dg = -sum_t gt_t d log f_t.
  auto gate_grad = [&](float bc, float bnd) {
    // sum over the earlier tokens alone (the sum with this token's own term, less that term, would lose what an earlier
    // strong decay has left of the others)
    const float before = __shfl_up(bc, 1);
    const float pre = wave_inclusive_scan(lane ? before : 0.f, lane);
    const float dlogf = tok_ok ? e_l + pre + bnd : 0.f;
    if (tok_ok) A.dgt[tokL * H + h] = -a.g[h] * dlogf;
    const float share = wave_sum(-gt_l * dlogf);
    if (lane == 0) A.wDgTile[(int64_t)cidx * H + h] = share;
  };
  if (last) {  // nothing flows in from beyond the end of the sequence (uniform for the block)
    if (w == 0) gate_grad(0.f, 0.f);
    return;
  }
  const float gh = a.g[h] * kLog2e;
  const int srow = 16 * w + i;            // this lane's token
  const bool row_ok = srow < clen;
  typedef typename Raw4<TIn>::type raw4;
  constexpr int NB = 2 * KSMAX;           // blocks of 16 columns
  // where the registers are there, the gradients are fetched with everything else; where they are not even there for the
  // rows, these are fetched again
  constexpr bool AHEAD = KSMAX * sizeof(TIn) <= 8, KEEP = KSMAX * sizeof(TIn) <= 12;
  const int64_t tokA = (int64_t)(t0 + (row_ok ? srow : 0)) * H + h;
  const TIn* vp = (const TIn*)a.v + tokA * dv + 4 * g;
  const TIn* bp = (const TIn*)a.b + tokA * dv + 4 * g;
  const TIn* kp = (const TIn*)a.k + qk_row(a, t0 + (row_ok ? srow : 0), h) + 4 * g;
  TIn* dkp = (TIn*)A.dk + tokA * dk + 4 * g;
  TIn* dvp = (TIn*)A.dv + tokA * dv + 4 * g;
  TIn* dbp = (TIn*)A.db + tokA * dv + 4 * g;
  auto load = [&](const TIn* p, int nb) { return *(const raw4*)(p + 16 * nb); };
  constexpr int NK = KEEP ? NB : 1, NA = AHEAD ? NB : 1;
  raw4 vr[NK], br[NK], kr[NK], dkr[NA], dvr[NA], dbr[NA];   // columns 16 nb + 4 g .. of the token's rows
  if constexpr (KEEP) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (16 * nb < dv) {
        vr[nb] = load(vp, nb);
        br[nb] = load(bp, nb);
      }
      if (16 * nb < dk) kr[nb] = load(kp, nb);
    }
  }
  auto v_of = [&](int nb) { if constexpr (KEEP) return vr[nb]; else return load(vp, nb); };
  auto b_of = [&](int nb) { if constexpr (KEEP) return br[nb]; else return load(bp, nb); };
  auto k_of = [&](int nb) { if constexpr (KEEP) return kr[nb]; else return load(kp, nb); };
  auto fetch_grads = [&]() {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (16 * nb < dk) dkr[nb] = load(dkp, nb);
      if (16 * nb < dv) {
        dvr[nb] = load(dvp, nb);
        dbr[nb] = load(dbp, nb);
      }
    }
  };
  float as, Ftot;                         // decay from token srow to the end of the tile, and over the whole tile
  {
    const float c = wave_inclusive_scan(-gt_l * gh, lane);
    const float tot = __shfl(c, 63);
    as = row_ok ? fast_exp2(tot - __shfl(c, srow)) : 0.f;
    Ftot = fast_exp2(tot);
  }
  const int64_t E = (int64_t)dv * dk;
  const TIn* RM = (const TIn*)A.wDM + ((int64_t)cidx * H + h) * E;
  const TIn* RJ = (const TIn*)A.wDJ + ((int64_t)cidx * H + h) * E;
  {
    // F_C (<R_M, M_0> + <R_J, J_0>) with (M_0, J_0) the state at the start of this tile; the same
    // pass leaves R in LDS for the products
    const float* smu = a.chunk_mu + ((int64_t)cidx * H + h) * E;
    const float* sI = a.chunk_I + ((int64_t)cidx * H + h) * E;
    const float Ipb = a.Ip[h];
    float acc = 0.f;
    // the workgroup goes through the states as they lie in memory, 16 bytes of the carries a lane; two pieces are fetched
    // before the first is used
    constexpr int VP = 16 / sizeof(TIn), kPass = 256 * VP;
    typedef TIn piece __attribute__((ext_vector_type(VP)));
    const int n_e = (int)E, step_row = kPass / dk, step_col = kPass - step_row * dk;
    int row = VP * tid / dk, col = VP * tid - row * dk;
    for (int e0 = 0; e0 < n_e; e0 += 2 * kPass) {
      piece rm[2], rj[2];
      f32x4 mu[2][VP / 4], I[2][VP / 4];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int e = e0 + u * kPass + VP * tid;
        if (e < n_e) {
          rm[u] = *(const piece*)(RM + e);
          rj[u] = *(const piece*)(RJ + e);
#pragma unroll
          for (int x = 0; x < VP / 4; ++x) {
            mu[u][x] = *(const f32x4*)(smu + e + 4 * x);
            I[u][x] = *(const f32x4*)(sI + e + 4 * x);
          }
        }
      }
      if constexpr (AHEAD) {
        if (e0 == 0) fetch_grads();
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (e0 + u * kPass + VP * tid < n_e) {
          const int o = row * RS + col;
          typedef bf16_t half __attribute__((ext_vector_type(VP)));
          half mh, jh, ml, jl;
#pragma unroll
          for (int x = 0; x < VP; ++x) {
            const float m = (float)rm[u][x], y = (float)rj[u][x], In = I[u][x >> 2][x & 3];
            acc = fmaf(m, mu[u][x >> 2][x & 3] * In, acc);
            acc = fmaf(y, In - Ipb, acc);
            mh[x] = (bf16_t)m;
            jh[x] = (bf16_t)y;
            if constexpr (PREC) {
              ml[x] = (bf16_t)(m - (float)mh[x]);
              jl[x] = (bf16_t)(y - (float)jh[x]);
            }
          }
          *(half*)&sR[o] = mh;
          *(half*)&sR[dv * RS + o] = jh;
          if constexpr (PREC) {
            *(half*)&sRl[o] = ml;
            *(half*)&sRl[dv * RS + o] = jl;
          }
        }
        row += step_row;
        col += step_col;
        if (col >= dk) { col -= dk; ++row; }
      }
    }
    acc = wave_sum(acc);
    if (lane == 0) sW4[w] = acc;
  }
  // Operands: contraction index (g, j) -> 32 ks + 16 (j / 4) + 4 g + j % 4, rows times the decay of their token (PREC: hi, lo)
  struct Opnd { bf16x8 hi, lo; };
  auto operand = [&](const float* x) {
    Opnd y;
    if constexpr (PREC) {
      split_bf16(x, y.hi, y.lo);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) y.hi[j] = (bf16_t)x[j];
    }
    return y;
  };
  auto mac = [&](const Opnd& r, const Opnd& t, f32x4 acc) {
    if constexpr (PREC) return mfma16_split(r.hi, r.lo, t.hi, t.lo, acc);
    else return mfma16(r.hi, t.hi, acc);
  };
  const bf16x4 none = {(bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f, (bf16_t)0.f};
  Opnd X[KSMAX], Y[KSMAX];
#pragma unroll
  for (int ks = 0; ks < KSMAX; ++ks) {
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (16 * (2 * ks + q) < dv) {
        const raw4 vv = v_of(2 * ks + q), bb = b_of(2 * ks + q);
#pragma unroll
        for (int j = 0; j < 4; ++j) { x[4 * q + j] = as * (float)vv[j]; y[4 * q + j] = as * (float)bb[j]; }
      }
    }
    X[ks] = operand(x);
    Y[ks] = operand(y);
  }
  __syncthreads();
  const float bnd = Ftot * (sW4[0] + sW4[1] + sW4[2] + sW4[3]);   // every thread

  // ---- dk: out[n, s] = sum_d R_M[d, n] (a_s v_s[d]) + 2 k_s[n] sum_d R_J[d, n] (a_s b_s[d])
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    if (16 * nb < dk) {
      f32x4 accM = {0.f, 0.f, 0.f, 0.f}, accJ = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSMAX; ++ks) {
        if (32 * ks < dv) {
          // rows 32 ks + 4 g + i / 4 and 16 further on, columns 16 nb + 4 (i % 4) ..
          const int o = (32 * ks + 4 * g + (i >> 2)) * RS + 16 * nb + 4 * (i & 3);
          const bool two = 32 * ks + 16 < dv;
          auto rows = [&](int at) {
            Opnd y;
            y.hi = join(lds_read_tr(sR + at), two ? lds_read_tr(sR + at + 16 * RS) : none);
            if constexpr (PREC) y.lo = join(lds_read_tr(sRl + at), two ? lds_read_tr(sRl + at + 16 * RS) : none);
            return y;
          };
          accM = mac(rows(o), X[ks], accM);
          accJ = mac(rows(dv * RS + o), Y[ks], accJ);
        }
      }
      float y[4];
      const raw4 kk = k_of(nb), was = AHEAD ? dkr[AHEAD ? nb : 0] : load(dkp, nb);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = (float)was[r] + fmaf(2.f * (float)kk[r], accJ[r], accM[r]);
      if (row_ok) store_vec<4>(dkp + 16 * nb, y);
    }
  }
  // ---- dv, db: out[d, s] = sum_n R[d, n] (a_s k_s[n]), (a_s k_s[n]^2);  beta_s = <v_s, dv^carry_s> + <b_s, db^carry_s>
#pragma unroll
  for (int ks = 0; ks < KSMAX; ++ks) {
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, y[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (16 * (2 * ks + q) < dk) {
        const raw4 kk = k_of(2 * ks + q);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float kv = (float)kk[j];
          x[4 * q + j] = as * kv;
          y[4 * q + j] = as * kv * kv;
        }
      }
    }
    X[ks] = operand(x);
    Y[ks] = operand(y);
  }
  float beta = 0.f;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    if (16 * nb < dv) {
      f32x4 accV = {0.f, 0.f, 0.f, 0.f}, accB = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KSMAX; ++ks) {
        if (32 * ks < dk) {
          const int o = (16 * nb + i) * RS + 32 * ks + 4 * g;
          const bool two = 32 * ks + 16 < dk;
          auto row = [&](int at) {
            Opnd y;
            y.hi = join(*(const bf16x4*)(sR + at), two ? *(const bf16x4*)(sR + at + 16) : none);
            if constexpr (PREC) y.lo = join(*(const bf16x4*)(sRl + at), two ? *(const bf16x4*)(sRl + at + 16) : none);
            return y;
          };
          accV = mac(row(o), X[ks], accV);
          accB = mac(row(dv * RS + o), Y[ks], accB);
        }
      }
      float x[4], y[4];
      const raw4 vv = v_of(nb), bb = b_of(nb);
      const raw4 was_v = AHEAD ? dvr[AHEAD ? nb : 0] : load(dvp, nb), was_b = AHEAD ? dbr[AHEAD ? nb : 0] : load(dbp, nb);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        beta = fmaf((float)vv[r], accV[r], beta);
        beta = fmaf((float)bb[r], accB[r], beta);
        x[r] = (float)was_v[r] + accV[r];
        y[r] = (float)was_b[r] + accB[r];
      }
      if (row_ok) {
        store_vec<4>(dvp + 16 * nb, x);
        store_vec<4>(dbp + 16 * nb, y);
      }
    }
  }
  beta = rows4_sum(beta);
  if (g == 0) sBt[srow] = row_ok ? beta : 0.f;
  __syncthreads();
  if (w == 0) gate_grad(sBt[lane], bnd);
}

// ----------------------------------------------------------------- head sums
// dg[h] = sum over the tiles of their shares; dIp[h] = sum over the tiles of the local terms and, with an initial
// state, - sum dJ_0 (J_0 = I_0 - Ip).  One wave per head, lane-strided then over the lanes (fixed order), in double.
__global__ __launch_bounds__(64) void chunk_bwd_head_reduce_kernel(BwdArgs A) {
  const ChunkArgs& a = A.c;
  const int h = blockIdx.x, lane = threadIdx.x;
  double sg = 0.0, si = 0.0;
  for (int c = lane; c < a.total_chunks; c += 64) {
    sg += (double)A.wDgTile[(int64_t)c * a.H + h];
    si += (double)A.wSig[(int64_t)c * a.H + h];
  }
  if (a.init_mu) {
    const int nblk = carry_scan_blocks((int64_t)a.dv * a.dk);
    for (int j = lane; j < a.n_seqs * nblk; j += 64) {
      const int n = j / nblk, b2 = j - n * nblk;
      si -= (double)A.wInitPart[((int64_t)n * a.H + h) * nblk + b2];
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sg += __shfl_xor(sg, off);
    si += __shfl_xor(si, off);
  }
  if (lane == 0) {
    A.dg[h] = (float)sg;
    A.dIp[h] = (float)si;
  }
}

// A small pass: sums the rectangles' parts, slices of value rows for dq and dk, column groups for dv and db, both for the gates
// and the tiles' sums, each in one order.  A thread takes four consecutive entries of a (token, head) row, or one gate.
template <typename TIn>
__global__ __launch_bounds__(256) void chunk_bwd_parts_sum_kernel(BwdArgs A, int slices, int groups) {
  const int dk = A.c.dk, dv = A.c.dv, H = A.c.H;
  const int64_t rows = (int64_t)A.tokens * H, tiles = (int64_t)A.c.total_chunks * H;
  const int per = (dk + dv) >> 1;   // groups of four in the rows of dq, dk, dv, db
  int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx < rows * per) {
    const int64_t row = idx / per;
    const int it = (int)(idx - row * per), vb = it >= dk >> 1;
    const int len = vb ? dv : dk, e = 4 * (vb ? it - (dk >> 1) : it), second = e >= len;
    const float* p = (vb ? A.pVB : A.pQK) + row * 2 * len + e;
    f32x4 x = *(const f32x4*)p;
    for (int y = 1; y < (vb ? groups : slices); ++y) x += *(const f32x4*)(p + y * rows * 2 * len);
    TIn* o = (TIn*)(vb ? (second ? A.db : A.dv) : (second ? A.dk : A.dq)) + row * len + (second ? e - len : e);
    store_vec<4>(o, (const float*)&x);
    return;
  }
  idx -= rows * per;
  const float* p = idx < rows ? A.pE + idx : A.pSig + (idx - rows);
  if (idx >= rows + tiles) return;
  float x = 0.f;
  for (int y = 0; y < slices * groups; ++y) x += p[y * (idx < rows ? rows : tiles)];
  if (idx < rows) A.wE[idx] = x;
  else A.wSig[idx - rows] = x;
}

static int launch_parts_sum(const BwdArgs& A, const TileParts& P, bool bf16, hipStream_t s) {
  const int64_t rows = (int64_t)A.tokens * A.c.H;
  const int64_t blocks = (rows * ((A.c.dk + A.c.dv) / 2) + rows + (int64_t)A.c.total_chunks * A.c.H + 255) / 256;
  if (blocks > 0x7fffffff) return PAL_E_DIM;
  if (bf16) PAL_TIMED_LAUNCH(kKernBwdPartsSum, s, chunk_bwd_parts_sum_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, s, A, P.slices, P.groups);
  else PAL_TIMED_LAUNCH(kKernBwdPartsSum, s, chunk_bwd_parts_sum_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, s, A, P.slices, P.groups);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

struct BwdLayout {
  size_t oDM, oDJ, oFtot, oSig, oE, oInit, oDgTile, oDqFull, oDkFull, oQK, oPQK, oPVB, oPE, oPSig, total;
};

// dq, dk of a q/k head shared by `rep` value heads: the kernels leave one row per value head ([tokens, H, dk]) in the
// workspace, this adds the rows of a group in a fixed order (fp32) into the caller's [tokens, Hq, dk].
template <typename T>
__global__ __launch_bounds__(256) void group_sum_kernel(const T* src_q, const T* src_k, T* dst_q, T* dst_k, int64_t n4,
                                                        int Hq, int rep, int dk) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;   // four consecutive columns of one (token, q/k head) row
  if (idx >= n4) return;
  const int per = dk >> 2;
  const int c4 = (int)(idx % per);
  const int64_t row = idx / per;                                 // token * Hq + hq
  const int64_t tok = row / Hq;
  const int hq = (int)(row - tok * Hq);
  float aq[4] = {0.f, 0.f, 0.f, 0.f}, ak[4] = {0.f, 0.f, 0.f, 0.f};
  for (int r = 0; r < rep; ++r) {
    const int64_t so = ((tok * Hq + hq) * rep + r) * (int64_t)dk + 4 * c4;   // value head hq * rep + r
    float x[4], y[4];
    load_vec<4>(src_q + so, x);
    load_vec<4>(src_k + so, y);
#pragma unroll
    for (int e = 0; e < 4; ++e) { aq[e] += x[e]; ak[e] += y[e]; }
  }
  store_vec<4>(dst_q + row * dk + 4 * c4, aq);
  store_vec<4>(dst_k + row * dk + 4 * c4, ak);
}

// dq, dk of [tokens, Hq * rep, dk] summed over the rep value heads of each group into [tokens, Hq, dk]
int launch_group_sum(const void* src_q, const void* src_k, void* dst_q, void* dst_k, int64_t tokens, int Hq, int rep, int dk,
                     int dtype, hipStream_t s) {
  const int64_t n4 = tokens * Hq * (dk / 4);
  if ((n4 + 255) / 256 > 0x7fffffff) return PAL_E_DIM;
  const unsigned gblocks = (unsigned)((n4 + 255) / 256);
  if (dtype == PAL_DTYPE_BF16)
    hipLaunchKernelGGL(group_sum_kernel<bf16_t>, dim3(gblocks), dim3(256), 0, s, (const bf16_t*)src_q, (const bf16_t*)src_k,
                       (bf16_t*)dst_q, (bf16_t*)dst_k, n4, Hq, rep, dk);
  else
    hipLaunchKernelGGL(group_sum_kernel<float>, dim3(gblocks), dim3(256), 0, s, (const float*)src_q, (const float*)src_k,
                       (float*)dst_q, (float*)dst_k, n4, Hq, rep, dk);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static BwdLayout bwd_layout(const PalDims* d) {
  BwdLayout L;
  const size_t E = (size_t)d->dv * d->dk, row = d->dtype == PAL_DTYPE_BF16 ? 2 : 4;
  const size_t tiles = (size_t)d->total_chunks * d->n_heads;
  const size_t tokens = (size_t)d->batch * d->seq_len;
  size_t o = 0;
  L.oDM = o; o = align256(o + tiles * E * row);
  L.oDJ = o; o = align256(o + tiles * E * row);
  L.oFtot = o; o = align256(o + tiles * 4);
  L.oSig = o; o = align256(o + tiles * 4);
  L.oE = o; o = align256(o + tokens * d->n_heads * 4);
  L.oInit = o; o = align256(o + (size_t)d->n_seqs * d->n_heads * (E / 256) * 4);
  L.oDgTile = o; o = align256(o + tiles * 4);
  L.oDqFull = L.oDkFull = o;
  if (d->n_qk_heads > 0 && d->n_qk_heads != d->n_heads) {
    const size_t full = tokens * d->n_heads * d->dk * row;
    L.oDqFull = o; o = align256(o + full);
    L.oDkFull = o; o = align256(o + full);
  }
  L.oQK = o;
  const int cols = tile_piece(d->dk);   // (the first column group, the widest)
  const TileParts P = tile_parts(d->dk, d->dv, row == 4, (int64_t)tiles);
  L.oPQK = L.oPVB = L.oPE = L.oPSig = o;
  if (P.on) {
    const size_t rows = tokens * d->n_heads, rects = (size_t)P.slices * P.groups;
    L.oPQK = o; o = align256(o + P.slices * rows * 2 * d->dk * 4);
    L.oPVB = o; o = align256(o + P.groups * rows * 2 * d->dv * 4);
    L.oPE = o; o = align256(o + rects * rows * 4);
    L.oPSig = o; o = align256(o + rects * tiles * 4);
  } else if (row == 2 && tile_rows(cols, d->dv, false, P.few) < d->dv) o = align256(o + tokens * d->n_heads * cols * 2 * 4);
  L.total = o;
  return L;
}

// Launch shapes that depend on the head dims only; worked out before the first launch so that a head-dim pair the
// backward cannot serve is refused while nothing has been enqueued.
struct BwdPlan {
  size_t lds_apply;
  int apply_stride;
};

// prec: the fp32-accurate variants (fp32 rows without PAL_FLAG_FP32_FAST)
static int bwd_plan(int dk, int dv, bool prec, BwdPlan& P) {
  const int dmax = dk > dv ? dk : dv;
  if (prec && dmax > 128) return PAL_E_HEADDIM;
  // The head dims that are served: those whose carries (as columns of dv + 8 entries) fit the LDS beside a result buffer.
  const size_t planes = prec ? 2 : 1, cols = planes * 4 * (size_t)dk * (dv + 8), out = sizeof(float) * kC * (dmax + 4);
  const size_t fixed = sizeof(float) * (kC + 8 + kC * (dv >> 3)) + out;
  if (fixed + cols > kMaxLds) return PAL_E_HEADDIM;
  // row stride of the carries in LDS: an odd number of 32-byte pieces, for both kinds of reads and for the writes, where that fits
  auto lds = [&](int stride) { return sizeof(float) * (4 + kC) + planes * 4 * (size_t)dv * stride; };
  P.apply_stride = 16 * ((dk >> 4) | 1);
  if (lds(P.apply_stride) > kMaxLds) P.apply_stride = dk;
  P.lds_apply = lds(P.apply_stride);
  return P.lds_apply <= kMaxLds ? PAL_OK : PAL_E_HEADDIM;
}

template <typename TIn, int KSMAX, bool PREC>
static int launch_carry_apply_t(const BwdArgs& A, unsigned blocks, size_t lds, hipStream_t s) {
  if (int rc = allow_lds((const void*)&chunk_bwd_carry_apply_kernel<TIn, KSMAX, PREC>, lds)) return rc;
  PAL_TIMED_LAUNCH(kKernBwdCarryApply, s, (chunk_bwd_carry_apply_kernel<TIn, KSMAX, PREC>), dim3(blocks), dim3(256), lds, s, A);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}
template <typename TIn, bool PREC>
static int launch_carry_apply(const BwdArgs& A, unsigned blocks, size_t lds, hipStream_t s) {
  const int dmax = A.c.dk > A.c.dv ? A.c.dk : A.c.dv;
  if (dmax <= 32) return launch_carry_apply_t<TIn, 1, PREC>(A, blocks, lds, s);
  if (dmax <= 64) return launch_carry_apply_t<TIn, 2, PREC>(A, blocks, lds, s);
  if (dmax <= 96) return launch_carry_apply_t<TIn, 3, PREC>(A, blocks, lds, s);
  if (dmax <= 128) return launch_carry_apply_t<TIn, 4, PREC>(A, blocks, lds, s);
  if constexpr (PREC) return PAL_E_HEADDIM;   // the split operands of 256-wide heads do not fit the registers
  else return dmax <= 192 ? launch_carry_apply_t<TIn, 6, false>(A, blocks, lds, s) : launch_carry_apply_t<TIn, 8, false>(A, blocks, lds, s);
}

}  // namespace pal

extern "C" size_t pal_chunk_bwd_workspace_bytes(const PalDims* d) {
  if (pal_validate_dims(d) != PAL_OK || d->total_chunks <= 0) return 0;
  pal::BwdPlan P;
  const bool prec = d->dtype == PAL_DTYPE_F32 && !(d->flags & PAL_FLAG_FP32_FAST);
  if (pal::bwd_plan(d->dk, d->dv, prec, P) != PAL_OK) return 0;
  return pal::bwd_layout(d).total;
}

extern "C" int pal_chunk_bwd_supported(int32_t dk, int32_t dv, int32_t dtype, uint32_t flags) {
  if (dk < 16 || dk > 256 || (dk & 15) || dv < 16 || dv > 256 || (dv & 15)) return PAL_E_HEADDIM;
  if (dtype != PAL_DTYPE_F32 && dtype != PAL_DTYPE_BF16) return PAL_E_DTYPE;
  pal::BwdPlan P;
  return pal::bwd_plan(dk, dv, dtype == PAL_DTYPE_F32 && !(flags & PAL_FLAG_FP32_FAST), P);
}

extern "C" int pal_chunk_bwd(const PalDims* d, const PalFwdTensors* t, const PalBwdTensors* gr, void* workspace,
                             size_t workspace_bytes, void* stream) {
  using namespace pal;
  if (!d || !t) return PAL_E_NULL;
  // the forward-side struct is reused with o pointing at any valid buffer; final states are not needed
  PalDims dd = *d;
  dd.flags &= ~PAL_FLAG_STORE_FINAL;
  PalFwdTensors tt = *t;
  tt.final_mu = tt.final_I = nullptr;
  if (!tt.o) tt.o = gr ? (void*)gr->d_o : nullptr;
  if ((dd.flags & PAL_FLAG_HAS_VAR) && !tt.o_var) tt.o_var = gr ? (void*)gr->d_o_var : nullptr;
  int rc = check_chunk_common(&dd, &tt);
  if (rc) return rc;
  rc = check_bwd_common(&dd, gr);
  if (rc) return rc;
  BwdPlan P;
  const bool prec = dd.dtype == PAL_DTYPE_F32 && !(dd.flags & PAL_FLAG_FP32_FAST);
  rc = bwd_plan(dd.dk, dd.dv, prec, P);
  if (rc) return rc;
  if ((int64_t)dd.total_chunks * dd.n_heads > 0x7fffffff ||
      (int64_t)dd.n_seqs * dd.n_heads * carry_scan_blocks((int64_t)dd.dv * dd.dk) > 0x7fffffff)
    return PAL_E_DIM;
  const BwdLayout L = bwd_layout(&dd);
  if (!workspace || workspace_bytes < L.total || !is_aligned16(workspace)) return PAL_E_WORKSPACE;
  BwdArgs A;
  fill_chunk_args(A.c, &dd, &tt);
  A.d_o = gr->d_o;
  A.d_o_var = (dd.flags & PAL_FLAG_HAS_VAR) ? gr->d_o_var : nullptr;
  A.dq = gr->dq; A.dk = gr->dk; A.dv = gr->dv; A.db = gr->db;
  const bool grouped = A.c.Hq != A.c.H;
  if (grouped) {   // one row per value head first, summed over each group at the end
    A.dq = (char*)workspace + L.oDqFull;
    A.dk = (char*)workspace + L.oDkFull;
  }
  A.dgt = gr->dgt; A.dg = gr->dg; A.dIp = gr->dIp;
  A.d_init_mu = gr->d_init_mu; A.d_init_I = gr->d_init_I;
  char* ws = (char*)workspace;
  A.wDM = ws + L.oDM; A.wDJ = ws + L.oDJ;
  A.wFtot = (float*)(ws + L.oFtot); A.wSig = (float*)(ws + L.oSig);
  A.wE = (float*)(ws + L.oE); A.wInitPart = (float*)(ws + L.oInit);
  A.wDgTile = (float*)(ws + L.oDgTile);
  A.wQK = (float*)(ws + L.oQK);
  A.pQK = (float*)(ws + L.oPQK); A.pVB = (float*)(ws + L.oPVB);
  A.pE = (float*)(ws + L.oPE); A.pSig = (float*)(ws + L.oPSig);
  A.tokens = dd.batch * dd.seq_len;
  hipStream_t s = (hipStream_t)stream;
  const bool bf = dd.dtype == PAL_DTYPE_BF16;
  const bool var = dd.flags & PAL_FLAG_HAS_VAR;
  const TileParts parts = tile_parts(dd.dk, dd.dv, !bf, (int64_t)dd.total_chunks * dd.n_heads);
  rc = bf ? (var ? launch_tile_t<bf16_t, true>(A, parts, s) : launch_tile_t<bf16_t, false>(A, parts, s))
          : (var ? launch_tile_t<float, true>(A, parts, s) : launch_tile_t<float, false>(A, parts, s));
  if (!rc && parts.on) rc = launch_parts_sum(A, parts, bf, s);
  if (rc) return rc;
  {
    const int64_t blocks = (int64_t)dd.n_seqs * dd.n_heads * carry_scan_blocks((int64_t)dd.dv * dd.dk);
    if (blocks > 0x7fffffff) return PAL_E_DIM;
    if (bf) PAL_TIMED_LAUNCH(kKernBwdCarryScan, s, chunk_bwd_carry_scan_kernel<bf16_t>, dim3((unsigned)blocks), dim3(256), 0, s, A);
    else PAL_TIMED_LAUNCH(kKernBwdCarryScan, s, chunk_bwd_carry_scan_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, s, A);
    PAL_HIP_LAUNCH_CHECK();
  }
  {
    const unsigned blocks = (unsigned)tile_head_blocks(dd.total_chunks, dd.n_heads);
    A.apply_stride = P.apply_stride;
    rc = bf     ? launch_carry_apply<bf16_t, false>(A, blocks, P.lds_apply, s)
         : prec ? launch_carry_apply<float, true>(A, blocks, P.lds_apply, s)
                : launch_carry_apply<float, false>(A, blocks, P.lds_apply, s);
    if (rc) return rc;
    PAL_HIP_LAUNCH_CHECK();
  }
  PAL_TIMED_LAUNCH(kKernBwdHeadReduce, s, chunk_bwd_head_reduce_kernel, dim3((unsigned)dd.n_heads), dim3(64), 0, s, A);
  PAL_HIP_LAUNCH_CHECK();
  if (grouped) {
    if (int rc2 = launch_group_sum(A.dq, A.dk, gr->dq, gr->dk, A.tokens, A.c.Hq, A.c.H / A.c.Hq, dd.dk, dd.dtype, s)) return rc2;
  }
  return PAL_OK;
}
