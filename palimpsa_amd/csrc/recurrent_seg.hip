// Token-serial forward of a few sequences with many tokens each, in segments.
//
// recurrent_fwd_kernel walks a sequence with one wave per four value rows, 0.16 us a token however empty the chip is.  Here a
// workgroup of NW waves shares the walk, a segment of the tokens each.  M and I are affine in the state a segment starts from
// (S_end = F S_start + S_local), so every wave first walks its segment from zero without outputs, leaves S_local and F in LDS, folds the
// segments before its own in their order into the state it starts from, and walks again with outputs.  All in fp32.
//
// What bounds it is vector issue: a workgroup's 16 waves sit on one compute unit.  So
// * a wave stages its rows through LDS of its own (no barrier) in pieces of P tokens: 16-byte requests and one conversion per
//   element in place of 2- to 8-byte requests of every lane for itself, four lane groups over;
// * the first walk takes the tokens of a piece times their decay to its end (a scan from there over the piece's gates), so that an
//   entry costs three instructions a token, k*k included, and the decay itself two per piece;
// * outputs of four tokens are summed over the lanes together.
// Errors against float64 are those of the walk of one wave: outputs 1.0e-7 rms, precision state 3.5e-8 to 5e-8, for decay rates
// of 0.5 to 16 a token (T = 200 to 512, 32x32 to 128x128); B=2 T=256 H=4 32x32 fp32 40.4 -> 8.9 us.
#include <type_traits>

#include "chunk_common.h"
#include "pal_host.h"
#include "pal_profile.h"
#include "recurrent.h"
#include "state_block.h"

namespace pal {

template <int NPL, int NW>
struct SegShape {
  static constexpr int P = NPL <= 4 ? 16 : 8;             // tokens of a piece
  static constexpr int DK = 16 * NPL;
  static constexpr int oQ = DK, oR = 2 * DK;              // staged token: k, q, then (v, b) of four value rows, f
  static constexpr int STRIDE = oR + 12;
  static constexpr int WAVE = P * STRIDE > 2 * NPL * 64 ? P * STRIDE : 2 * NPL * 64;   // floats of a wave
  static constexpr size_t lds = sizeof(float) * (NW * WAVE + NW);
  static_assert(lds <= kMaxLds, "LDS of a compute unit");
};

template <typename TIn, int NPL, int NW, bool HAS_VAR>
__global__ __launch_bounds__(64 * NW) void recurrent_seg_kernel(RecArgs a) {
  extern __shared__ float smem[];
  typedef SegShape<NPL, NW> Sh;
  typedef typename Raw4<TIn>::type raw4;
  constexpr int P = Sh::P, DK = Sh::DK, STRIDE = Sh::STRIDE, oQ = Sh::oQ, oR = Sh::oR;
  constexpr int NI = P * NPL / 16;          // pieces of four columns per lane, of k and of q
  const int lane = threadIdx.x & 63, j = lane & 15, grp = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.H, dv = a.dv, n_dtiles = dv >> 2;
  const int tile = blockIdx.x % n_dtiles, nh = blockIdx.x / n_dtiles, h = nh % H, n = nh / H;
  float* sw = smem + w * Sh::WAVE;          // this wave's rows; after the first walk, what its segment leaves
  float* sF = smem + NW * Sh::WAVE;         // [NW] decay of the segments

  int64_t bos;
  int T;
  if (a.cu_seqlens) {
    int b0;
    packed_seq_bounds(a.cu_seqlens, n, a.T, b0, T);
    bos = b0;
  } else {
    bos = (int64_t)n * a.T;
    T = a.T;
  }
  const int len = (T + NW - 1) / NW, first = min(w * len, T);
  bos += first;
  T = min(len, T - first);                  // this wave's segment (may be empty at the end)
  const float gh = a.g[h] * kLog2e, Ip = a.Ip[h];

  const int Hq = a.Hq, hq = h / (H / Hq);
  const int64_t step_k = (int64_t)Hq * DK, step_v = (int64_t)H * dv;
  const TIn* kp = (const TIn*)a.k + (bos * Hq + hq) * DK;
  const TIn* qp = (const TIn*)a.q + (bos * Hq + hq) * DK;
  const TIn* vp = (const TIn*)a.v + (bos * H + h) * dv + 4 * tile;
  const TIn* bp = (const TIn*)a.b + (bos * H + h) * dv + 4 * tile;
  raw4 rk[NI], rq[NI], rv, rb;
  unsigned rg = 0;
  const raw4 none = {0, 0, 0, 0};
  // the rows of the P tokens from t0 on, zero beyond the segment: lane l has pieces l, l + 64, .. of k and q, v, b and the gate of
  // token l
  auto request = [&](int t0, bool with_q) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int idx = lane + 64 * u, s = idx / (4 * NPL), c = idx % (4 * NPL);
      const bool in = t0 + s < T;
      const int64_t off = in ? (t0 + s) * step_k + 4 * c : 0;
      rk[u] = in ? *(const raw4*)(kp + off) : none;
      if (with_q) rq[u] = in ? *(const raw4*)(qp + off) : none;
    }
    const bool in = lane < P && t0 + lane < T;
    const int64_t off = in ? (t0 + lane) * step_v : 0;
    rv = in ? *(const raw4*)(vp + off) : none;
    rb = in ? *(const raw4*)(bp + off) : none;
    rg = in ? load_gate_word(a.gt, (bos + t0 + lane) * H + h, a.gate_bf16) : 0u;
  };
  auto gate = [&](int t0) {   // log2 of the decay of token t0 + lane, zero beyond the segment
    const bool in = lane < P && t0 + lane < T;
    return in ? -gate_value(rg, (bos + t0 + lane) * H + h, a.gate_bf16) * gh : 0.f;
  };
  auto put = [&](bool with_q) {
#pragma unroll
    for (int u = 0; u < NI; ++u) {
      const int idx = lane + 64 * u, s = idx / (4 * NPL), c = idx % (4 * NPL);
      *(f32x4*)&sw[s * STRIDE + 4 * c] = f32x4{(float)rk[u][0], (float)rk[u][1], (float)rk[u][2], (float)rk[u][3]};
      if (with_q) *(f32x4*)&sw[s * STRIDE + oQ + 4 * c] = f32x4{(float)rq[u][0], (float)rq[u][1], (float)rq[u][2], (float)rq[u][3]};
    }
  };
  auto staged = [] {   // the rows are written by other lanes of the wave than read them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

  // ---- first walk: what the segment leaves of its own tokens
  float M[NPL], J[NPL];
#pragma unroll
  for (int e = 0; e < NPL; ++e) { M[e] = 0.f; J[e] = 0.f; }
  request(0, w == NW - 1);
  if (w < NW - 1) {
    float tot = 0.f;
    for (int t0 = 0; t0 < T; t0 += P) {
      const float c = gate(t0);
      // log2 of the decay after a token to the end of the piece: the tokens after it alone.  (As the difference of two sums from
      // the start of the piece it carried the rounding of all of them: 1e-4 of the weight behind a token of decay e^-1e4, NaN
      // behind one of zero.)
      float after = row_shl_zero<1>(c);
      after += row_shl_zero<1>(after);
      after += row_shl_zero<2>(after);
      after += row_shl_zero<4>(after);
      if constexpr (P > 8) after += row_shl_zero<8>(after);
      const float end = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, after + c)));
      tot += end;
      staged();
      put(false);
      if (lane < P) {
        const float wt = fast_exp2(after);
#pragma unroll
        for (int r = 0; r < 4; ++r) *(f32x2*)&sw[lane * STRIDE + oR + 2 * r] = f32x2{wt * (float)rv[r], wt * (float)rb[r]};
      }
      staged();
      request(t0 + P, false);
      const float F = fast_exp2(end);
#pragma unroll
      for (int e = 0; e < NPL; ++e) { M[e] *= F; J[e] *= F; }
      const int nt = min(P, T - t0);
#pragma unroll 1
      for (int s0 = 0; s0 < nt; s0 += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float* row = sw + (s0 + u) * STRIDE;
          float k[NPL];
          lds_cols<16, NPL>(row, j, k);
          const f32x2 vb = *(const f32x2*)&row[oR + 2 * grp];
#pragma unroll
          for (int e = 0; e < NPL; ++e) {
            M[e] = fmaf(vb[0], k[e], M[e]);
            J[e] = fmaf(vb[1], k[e] * k[e], J[e]);
          }
        }
      }
    }
    staged();
    float* end = sw + lane;
#pragma unroll
    for (int e = 0; e < NPL; ++e) { end[64 * e] = M[e]; end[64 * (NPL + e)] = J[e]; }
    // (a growth beyond fp32 must not turn entries that are zero into NaN; a NaN stays one)
    const float F = fast_exp2(tot);
    if (lane == 0) sF[w] = F > 3.4028235e38f ? 3.4028235e38f : F;
    request(0, true);
  }
  const int64_t so = ((int64_t)nh * dv + 4 * tile + grp) * DK;
  auto pieces = [&](auto&& f) {   // (width, first entry) of a lane's contiguous columns
#pragma unroll
    for (int p = 0; p < NPL / 4; ++p) f(std::integral_constant<int, 4>{}, 4 * p);
    if constexpr ((NPL & 3) >= 2) f(std::integral_constant<int, 2>{}, 4 * (NPL / 4));
    if constexpr (NPL & 1) f(std::integral_constant<int, 1>{}, NPL - 1);
  };
  // every wave folds from the initial state (the last one may write its final state over it: behind the barriers)
#pragma unroll
  for (int e = 0; e < NPL; ++e) { M[e] = 0.f; J[e] = 0.f; }
  if (a.init_mu) {
    pieces([&](auto width, int i) {
      constexpr int PW = decltype(width)::value;
      float x[PW], y[PW];
      load_vec<PW>(a.init_mu + so + col_of<16, NPL>(i, j), x);
      load_vec<PW>(a.init_I + so + col_of<16, NPL>(i, j), y);
#pragma unroll
      for (int e = 0; e < PW; ++e) {
        M[i + e] = x[e] * y[e];
        J[i + e] = y[e] - Ip;
        asm volatile("" : "+v"(M[i + e]), "+v"(J[i + e]));   // read before the barrier
      }
    });
  }
  __syncthreads();
#pragma unroll 4
  for (int u = 0; u < w; ++u) {
    const float* end = smem + u * Sh::WAVE + lane;
    const float F = sF[u];
#pragma unroll
    for (int e = 0; e < NPL; ++e) {
      M[e] = fmaf(F, M[e], end[64 * e]);
      J[e] = fmaf(F, J[e], end[64 * (NPL + e)]);
    }
  }
  __syncthreads();

  // ---- second walk, with outputs
  // four tokens are summed over the lanes together: lane bits 3 and 2 select one
  const int sel = 2 * ((lane >> 3) & 1) + ((lane >> 2) & 1);
  const bool writer = (lane & 3) == 0;
  auto reduce = [&](const float* y) {
    return OutLanes<16>::sum_other(pair_bit2(pair_bit3(y[0], y[2]), pair_bit3(y[1], y[3])));
  };
  TIn* op = (TIn*)a.o + (bos * H + h) * dv + 4 * tile + grp;
  const int64_t var0 = (bos * H + h) * dv + 4 * tile + grp;
  for (int t0 = 0; t0 < T; t0 += P) {
    const float f = fast_exp2(gate(t0));
    put(true);
    if (lane < P) {
#pragma unroll
      for (int r = 0; r < 4; ++r) *(f32x2*)&sw[lane * STRIDE + oR + 2 * r] = f32x2{(float)rv[r], (float)rb[r]};
      sw[lane * STRIDE + oR + 8] = f;
    }
    staged();
    request(t0 + P, true);
    const int nt = min(P, T - t0);
#pragma unroll 1
    for (int s0 = 0; s0 < nt; s0 += 4) {
      float acc[4], accv[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* row = sw + (s0 + u) * STRIDE;
        float k[NPL], q[NPL];
        lds_cols<16, NPL>(row, j, k);
        lds_cols<16, NPL>(row + oQ, j, q);
        const f32x2 vb = *(const f32x2*)&row[oR + 2 * grp];
        const float f = row[oR + 8];
        acc[u] = 0.f;
        accv[u] = 0.f;
#pragma unroll
        for (int e = 0; e < NPL; ++e) {
          M[e] = fmaf(f, M[e], vb[0] * k[e]);
          J[e] = fmaf(f, J[e], vb[1] * (k[e] * k[e]));
          const float r = fast_rcp(J[e] + Ip);
          acc[u] = fmaf(M[e] * r, q[e], acc[u]);
          if constexpr (HAS_VAR) accv[u] = fmaf(q[e] * q[e], r, accv[u]);
        }
      }
      const int t = t0 + s0 + sel;
      const float out = reduce(acc);
      if (writer && t < T) op[t * step_v] = from_f32<TIn>(out * a.scale);
      if constexpr (HAS_VAR) {
        const float outv = reduce(accv);
        if (writer && t < T) store_rt(a.o_var, var0 + t * step_v, outv * a.scale, a.var_bf16);
      }
    }
    staged();
  }
  if (a.final_mu && w == NW - 1) {
    pieces([&](auto width, int i) {
      constexpr int PW = decltype(width)::value;
      float x[PW], y[PW];
#pragma unroll
      for (int e = 0; e < PW; ++e) { y[e] = J[i + e] + Ip; x[e] = M[i + e] * fast_rcp(y[e]); }
      store_vec<PW>(a.final_mu + so + col_of<16, NPL>(i, j), x);
      store_vec<PW>(a.final_I + so + col_of<16, NPL>(i, j), y);
    });
  }
}

template <typename TIn, int NPL, int NW>
static int launch_nw(const RecArgs& a, hipStream_t s) {
  const int64_t blocks = (int64_t)a.n_seqs * a.H * (a.dv / 4);
  if (blocks > 0x7fffffff) return PAL_E_DIM;
  constexpr size_t lds = SegShape<NPL, NW>::lds;
  auto go = [&](auto kern) -> int {
    if (int rc = allow_lds((const void*)kern, lds)) return rc;
    PAL_TIMED_LAUNCH(kKernRecurrentSeg, s, kern, dim3((unsigned)blocks), dim3(64 * NW), lds, s, a);
    return 0;
  };
  const int rc = (a.flags & PAL_FLAG_HAS_VAR) ? go(&recurrent_seg_kernel<TIn, NPL, NW, true>) : go(&recurrent_seg_kernel<TIn, NPL, NW, false>);
  if (rc) return rc;
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

template <typename TIn, int NPL>
static int launch_npl(const RecArgs& a, int waves, hipStream_t s) {
  if (waves == 4) return launch_nw<TIn, NPL, 4>(a, s);
  if (waves == 8) return launch_nw<TIn, NPL, 8>(a, s);
  if constexpr (NPL <= 8) {
    if (waves == 16) return launch_nw<TIn, NPL, 16>(a, s);
  }
  return PAL_E_HEADDIM;   // (recurrent_segments asks for 16 up to 128 key columns)
}

template <typename TIn>
static int launch_dtype(const RecArgs& a, int waves, hipStream_t s) {
  switch (a.dk / 16) {
    case 1: return launch_npl<TIn, 1>(a, waves, s);
    case 2: return launch_npl<TIn, 2>(a, waves, s);
    case 3: return launch_npl<TIn, 3>(a, waves, s);
    case 4: return launch_npl<TIn, 4>(a, waves, s);
    case 6: return launch_npl<TIn, 6>(a, waves, s);
    case 8: return launch_npl<TIn, 8>(a, waves, s);
    case 12: return launch_npl<TIn, 12>(a, waves, s);
    case 16: return launch_npl<TIn, 16>(a, waves, s);
    default: return PAL_E_HEADDIM;
  }
}

int launch_recurrent_seg(const RecArgs& a, int dtype, int waves, hipStream_t s) {
  return dtype == PAL_DTYPE_BF16 ? launch_dtype<bf16_t>(a, waves, s) : launch_dtype<float>(a, waves, s);
}

// Four segments pay where the walks of one wave would be long and leave room on the chip: the two walks and the fold are work
// of 1.4 walks.  More, where a compute unit would have fewer workgroups than waves and the segments stay long enough.
// One wave against 4 / 8 / 16 (us a call; below 7 the host is the limit):
//   64 waves in all (B=2 H=4 32x32 fp32)   T=64   12.6:   6.7   6.6   6.9     T=256   40.7:  14.1  10.0   9.3
//   192 (B=1 H=16 48x48)                   T=64   16.2:   7.4   7.0   8.3     T=777  180  :  47.1  32.3  29.1
//   512 (B=1 H=16 128x128)                 T=16    8.7:   7.3   9.9  21.2     T=512  177  :  73.8  61.5  69.8
//   768 (B=4 H=16 48x48)                   T=32   10.8:   7.8  11.4  22.0     T=512  124  :  48.6  49.2  58.0
//   1536 (B=2 H=16 96x192)                 T=32   17.3:  15.5  22.3  49.8     T=256  107  :  73.0  73.9  95.3
//   2048 (B=8 H=16 64x64)                  T=32   14.5:  15.4  25.2  58.6     T=256   84.0:  63.4  68.3  95.3
//   4096 (B=16 H=16 64x64 fp32)            T=32   21.3:  30.6  55.0 129       T=256  123  : 140   150   206
// Four segments of two tokens cost more than they save, and so do segments whose workgroups (34 KB of LDS at 128 key columns, 67 at
// 256) do not all find room at once, until the walk is long: the line grows with waves times columns (us of the kernel alone).
//   784 (64 columns)                       T=8     5.6:   7.2     1024    T=13    7.0:   7.7
//   576 (B=6 H=4 256x96 fp32)              T=10    8.2:  17.9
//   576 (B=3 H=16 256x48 fp32)             T=34   22.2:  29.6
//   768 (B=4 H=12 256x64)                  T=120  73.2:  59.1
//   1920 (B=5 H=16 128x96 fp32)            T=54   31.6:  39.5
//   1920 (B=30 H=8 128x32)                 T=111  62.3:  58.4
// Over 1500 drawn calls (16 to 256 columns, 4 to 1448 tokens, up to 2048 waves) 1091 are more than a fifth faster than with one wave
// and 12 more than 5 % slower, 1.27 times at most; with a line at 8 and 48 tokens for all columns it was 124, 2.33 times at most.
int recurrent_segments(const PalDims* d) {
  const int64_t waves = (int64_t)d->n_seqs * d->n_heads * (d->dv / 4);
  const int64_t len = (d->flags & PAL_FLAG_VARLEN) ? d->seq_len / d->n_seqs : d->seq_len;   // the mean of a packed batch
  if (waves <= 256 && len >= 192 && d->dk <= 128) return 16;
  if (waves <= 512 && len >= 64) return 8;
  if (waves <= 2048 && len >= 12 && 4000 * len >= waves * d->dk) return 4;
  return 1;
}

// Whether outputs and final states of a short pass (pal_chunk_fwd) come from the walk: its three kernels take 13 us for 8 tokens and
// 25 for 64 to 256, most of it the 64 tokens of a tile one after the other, the walk costs by the token.  Both are estimated in us.
// The walk is the longer of its chain (the waves of a sequence share a compute unit's issue, so segments do not shorten it much:
// 0.5 ns a token and key column; workgroups of eight waves with 100 KB of LDS take turns beyond 256 of them) and of the chip's issue
// (33 ps a token and wave and 2 ps for each key column, more with the uncertainty output, most in the form of many rows per
// wave); the tiles are a tile's chain, the traffic of their states and their issue.
// Walk / tiles, us: H=16 48x48 T=256 12.2 / 25.6, T=777 29.1 / 32.8, T=1536 45.4 / 42.2; 128x128 T=128 19.7 / 24.4, T=256 34.8 / 31.3;
// B=8 H=16 64x64 T=64 22.0 / 25.2, T=128 36.2 / 30.9; one wave a sequence: 74 x 2 heads 16x64 fp32 T=232 60.9 / 34.1, 129 x 1 32x64 T=111
// 37.5 / 30.7, 9 x 1 256x96 fp32 T=137 30.0 / 52.7; uncertainty: 23 x 12 heads 16x128 T=21 51.1 / 24.9.
// Over 5000 drawn calls (16 to 256 key columns, 4 to 1024 tokens, 5e4 to 1e7 entries) 4120 are more than a fifth faster than by tiles
// and 38 more than 5 % slower, 1.35 times at most (by work alone, up to 1e7 entries, 299, 3.1 times at most).  Not beyond 1024 tokens and
// 1e7 entries, where nothing was measured.
bool short_pass(const PalDims* d) {
  if (!recurrent_dk_supported(d->dk) || (d->flags & PAL_FLAG_VARLEN) || d->seq_len > 1024) return false;
  const int T = d->seq_len, dk = d->dk, segments = recurrent_segments(d), tiles = (T + PAL_CHUNK - 1) / PAL_CHUNK;
  const int64_t waves = (int64_t)d->n_seqs * d->n_heads * (d->dv / 4);
  if (waves * T * dk > 10000000) return false;
  double chain = 5e-4 * T * dk + 0.03 * T / segments;
  if (segments == 8 && dk > 128 && waves > 256) chain *= 2;
  const double uncertainty = !(d->flags & PAL_FLAG_HAS_VAR) ? 0.0 : segments == 1 ? 83e-6 : 23e-6;
  const double issue = (33e-6 + 2e-6 * dk + uncertainty) * waves * T;
  const double by_tiles = 10 + 0.16 * (T < PAL_CHUNK ? T : PAL_CHUNK) + 0.4 * tiles + (0.6e-6 * T + 13e-6 * (1 + tiles)) * waves * dk;
  return 6.7 + (chain > issue ? chain : issue) <= by_tiles;
}

}  // namespace pal
