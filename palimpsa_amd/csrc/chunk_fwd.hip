// Chunked Palimpsa forward: tile-start states (two-kernel form) and the entry points.
//
//  (1) chunk_delta_kernel + chunk_scan_kernel — the state at the START of every
//      tile.  The first computes every tile's own contribution
//        Delta = (a o V)^T K                 (a_s = decay from token s to tile end)
//      with bf16 MFMA contractions, all tiles in parallel; the second runs the
//      recurrence S_c = F_C S_{c-1} + Delta_c over the tiles of a sequence as an
//      fp32 streaming scan (the only serial part of the forward) and leaves the
//      tile-start states and the final state in (mu, I) form.
//  (2) chunk_out_kernel (chunk_out.hip) — the outputs of all tiles in parallel.
#include <atomic>
#include <type_traits>

#include "chunk_common.h"
#include "pal_host.h"
#include "pal_profile.h"
#include "recurrent.h"

namespace pal {

// ------------------------------------------------------------------ kernel 1a
// Local contribution of one tile to the state: Delta = (a o V)^T K, with a_s the decay from token s
// to the end of the tile.  One workgroup of 4 waves per (tile, head), all tiles in parallel: the
// K, V, B rows of the tile are staged once through LDS (16-byte loads, stored transposed so that an
// MFMA operand is one contiguous run of tokens), then wave w produces the 16x16 blocks of the state
// whose key columns are [16w, 16w+16) (+64, ...).  The result is parked in the tile's slot of
// chunk_mu / chunk_I until the scan below replaces it.
// Row stride (elements) of the transposed staging tiles.  bf16 rows are staged as they are; fp32 rows in fp32
// tiles while those fit in LDS, else rounded to bf16 (the operands built from them are bf16 anyway).
template <typename TS>
struct StageStride { static constexpr int value = sizeof(TS) == 4 ? 68 : 72; };

template <typename TIn, typename TS>
__device__ __forceinline__ void stage_transposed(const TIn* src, int64_t row_stride, int width, int clen, TS* dst,
                                                 int tid) {
  // src: [64 tokens][width] rows -> dst[width][stride] (token index fastest), rows >= clen are zero
  constexpr int kTS = StageStride<TS>::value;
  const int groups = width >> 3;
  if constexpr (sizeof(TS) == 2) {
    // bf16 tiles: a work item is two consecutive tokens by eight columns, so that neighbouring lanes read
    // neighbouring 16-byte pieces of a row and a pair of tokens goes to LDS as one 32-bit word per column
    for (int idx = tid; idx < (kC / 2) * groups; idx += 256) {
      const int sp = idx / groups, c8 = idx - sp * groups;
      float x0[8], x1[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) { x0[e] = 0.f; x1[e] = 0.f; }
      if (2 * sp < clen) {
        load_vec<4>(src + (int64_t)(2 * sp) * row_stride + 8 * c8, x0);
        load_vec<4>(src + (int64_t)(2 * sp) * row_stride + 8 * c8 + 4, x0 + 4);
      }
      if (2 * sp + 1 < clen) {
        load_vec<4>(src + (int64_t)(2 * sp + 1) * row_stride + 8 * c8, x1);
        load_vec<4>(src + (int64_t)(2 * sp + 1) * row_stride + 8 * c8 + 4, x1 + 4);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) *(bf16x2*)&dst[(8 * c8 + e) * kTS + 2 * sp] = pack2(x0[e], x1[e]);
    }
  } else {
    for (int idx = tid; idx < kC * groups; idx += 256) {
      const int s = idx & (kC - 1), c8 = idx >> 6;
      float x[8];
      if (s < clen) {
        load_vec<4>(src + (int64_t)s * row_stride + 8 * c8, x);
        load_vec<4>(src + (int64_t)s * row_stride + 8 * c8 + 4, x + 4);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = 0.f;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[(8 * c8 + e) * kTS + s] = x[e];
    }
  }
}

// eight consecutive staged elements (16-byte aligned) as fp32
__device__ __forceinline__ void staged8(const float* p, float* out) {
  *(f32x4*)&out[0] = *(const f32x4*)p;
  *(f32x4*)&out[4] = *(const f32x4*)(p + 4);
}
__device__ __forceinline__ void staged8(const bf16_t* p, float* out) {
  const bf16x8 x = *(const bf16x8*)p;
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = (float)x[e];
}

// HAS_J = false drops the precision branch (b is not read, chunk_I is not written): the scalar-gated linear
// attention that the layer uses without its precision state.
// PREC (fp32 rows staged in fp32): operands split into two bf16 halves, three matrix instructions per product.
template <typename TIn, bool HAS_J, typename TS, bool PREC>
__global__ __launch_bounds__(256) void chunk_delta_kernel(ChunkArgs a, int dvn) {
  // blockIdx.y selects a piece of dvn value rows (dvn = dv: one piece; smaller where the staging tiles of all rows
  // would not fit the LDS)
  extern __shared__ float smem[];
  constexpr int kTS = StageStride<TS>::value;
  const int H = a.H, dk = a.dk, dv = a.dv;
  const int d0 = blockIdx.y * dvn, dn = min(dvn, dv - d0);
  float* sA = smem;                 // [64] decay from token s to the end of the tile
  TS* sKT = (TS*)(sA + kC);         // [dk][kTS]
  TS* sVT = sKT + dk * kTS;         // [dvn][kTS]
  TS* sBT = sVT + dvn * kTS;        // [dvn][kTS]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i = lane & 15, g = lane >> 4;
  const int NB = dk >> 4, ND = dn >> 4;
  const int cidx = blockIdx.x / H, h = blockIdx.x % H;
  int seq, t0, clen, cis;
  chunk_lookup(a, cidx, seq, t0, clen, cis);
  if (w == 0) {
    const float gh = a.g[h] * kLog2e;
    const float gt = (lane < clen) ? load_gate(a.gt, (int64_t)(t0 + lane) * H + h, a.gate_bf16) : 0.f;
    const float cs = wave_inclusive_scan(-gt * gh, lane);
    sA[lane] = fast_exp2((a.flags & kFlagDecayFromStart) ? cs : __shfl(cs, 63) - cs);
  }
  stage_transposed((const TIn*)a.k + qk_row(a, t0, h), qk_stride(a), dk, clen, sKT, tid);
  stage_transposed((const TIn*)a.v + ((int64_t)t0 * H + h) * dv + d0, (int64_t)H * dv, dn, clen, sVT, tid);
  if (HAS_J) stage_transposed((const TIn*)a.b + ((int64_t)t0 * H + h) * dv + d0, (int64_t)H * dv, dn, clen, sBT, tid);
  __syncthreads();
  float as[2][8];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) staged8(&sA[8 * g + 32 * ks], as[ks]);
  for (int nb = w; nb < NB; nb += 4) {
    bf16x8 BK[2], BKK[2], BKl[2], BKKl[2];   // the *l halves only exist with PREC
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      float kv[8];
      staged8(&sKT[(16 * nb + i) * kTS + 8 * g + 32 * ks], kv);
      if constexpr (PREC) {
        float kq[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) kq[j] = kv[j] * kv[j];
        split_bf16(kv, BK[ks], BKl[ks]);
        split_bf16(kq, BKK[ks], BKKl[ks]);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          BK[ks][j] = (bf16_t)kv[j];
          BKK[ks][j] = (bf16_t)(kv[j] * kv[j]);
        }
      }
    }
    for (int dt = 0; dt < ND; ++dt) {
      bf16x8 AM[2], AJ[2], AMl[2], AJl[2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        float vv[8], bb[8];
        staged8(&sVT[(16 * dt + i) * kTS + 8 * g + 32 * ks], vv);
        if (HAS_J) staged8(&sBT[(16 * dt + i) * kTS + 8 * g + 32 * ks], bb);
        if constexpr (PREC) {
#pragma unroll
          for (int j = 0; j < 8; ++j) { vv[j] *= as[ks][j]; if (HAS_J) bb[j] *= as[ks][j]; }
          split_bf16(vv, AM[ks], AMl[ks]);
          if (HAS_J) split_bf16(bb, AJ[ks], AJl[ks]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            AM[ks][j] = (bf16_t)(as[ks][j] * vv[j]);
            if (HAS_J) AJ[ks][j] = (bf16_t)(as[ks][j] * bb[j]);
          }
        }
      }
      // the products are taken transposed (K as the row operand) so that a lane ends up with four consecutive
      // key columns of one value row: rows n = 16nb + 4g + r, column d = 16dt + i, one 16-byte store per lane
      f32x4 M = {0.f, 0.f, 0.f, 0.f}, J = {0.f, 0.f, 0.f, 0.f};
      if constexpr (PREC) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          M = mfma16_split(BK[ks], BKl[ks], AM[ks], AMl[ks], M);
          if (HAS_J) J = mfma16_split(BKK[ks], BKKl[ks], AJ[ks], AJl[ks], J);
        }
      } else {
      M = mfma16(BK[0], AM[0], M);
      if (HAS_J) J = mfma16(BKK[0], AJ[0], J);
      M = mfma16(BK[1], AM[1], M);
      if (HAS_J) J = mfma16(BKK[1], AJ[1], J);
      }
      const int64_t co = (((int64_t)cidx * H + h) * dv + d0 + 16 * dt + i) * dk + 16 * nb + 4 * g;
      *(f32x4*)&a.chunk_mu[co] = M;
      if (HAS_J) *(f32x4*)&a.chunk_I[co] = J;
    }
  }
}

// ------------------------------------------------------------------ kernel 1b
// blocks of a (sequence, head) at vw entries per thread
__host__ __device__ inline int scan_blocks(int64_t E, int vw) { return (int)((E + 256 * vw - 1) / (256 * vw)); }

// Serial part of the forward: S_c = F_c S_{c-1} + Delta_c per state entry, fp32, pure streaming.
// One thread per VW consecutive state entries of a (sequence, head), 256 VW entries per block.  Each slot of
// chunk_mu / chunk_I is overwritten with the state at the START of its tile in (mu, I) form
// (what the reference stores as intermediate_*_state, chunk_palimpsa_forgetting_scalar.py:187-188);
// the state after the last tile goes to final_mu / final_I (:214-218).
template <int VW>
__global__ __launch_bounds__(256) void chunk_scan_kernel(ChunkArgs a) {
  __shared__ float sF[kScanTiles];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t E = (int64_t)a.dv * a.dk;
  const int nblk = scan_blocks(E, VW);
  const int blk = blockIdx.x % nblk;
  const int nh = blockIdx.x / nblk;
  const int h = nh % a.H, n = nh / a.H;
  const int64_t e = ((int64_t)blk * 256 + tid) * VW;
  const bool on = e < E;
  int bos, len, cbase;
  seq_lookup(a, n, bos, len, cbase);
  const int nchunks = (len + kC - 1) / kC;
  const float Ip = a.Ip[h];
  const float gh = a.g[h] * kLog2e;
  float SM[VW], SJ[VW];
#pragma unroll
  for (int x = 0; x < VW; ++x) SM[x] = SJ[x] = 0.f;
  const int64_t so = (int64_t)nh * E + e;
  if (a.init_mu && on) {
    float mu[VW], I[VW];
    load_vec<VW>(a.init_mu + so, mu);
    load_vec<VW>(a.init_I + so, I);
#pragma unroll
    for (int x = 0; x < VW; ++x) { SM[x] = mu[x] * I[x]; SJ[x] = I[x] - Ip; }
  }
  auto store_state = [&](float* dst_mu, float* dst_I) {
    float mu[VW], I[VW];
#pragma unroll
    for (int x = 0; x < VW; ++x) { I[x] = SJ[x] + Ip; mu[x] = SM[x] * fast_rcp(I[x]); }
    store_vec<VW>(dst_mu, mu);
    store_vec<VW>(dst_I, I);
  };
  // the slot of a tile: its Delta is read, the state at its start (mu, I) written if it is kept, the state advanced
  auto advance = [&](int64_t off, const float* dM, const float* dJ, float F, bool kept) {
    if (kept) store_state(a.chunk_mu + off, a.chunk_I + off);
#pragma unroll
    for (int x = 0; x < VW; ++x) {
      SM[x] = fmaf(F, SM[x], dM[x]);
      SJ[x] = fmaf(F, SJ[x], dJ[x]);
    }
  };
  constexpr int U = VW == 1 ? 8 : 4;   // tiles in flight
  for (int c0 = 0; c0 < nchunks; c0 += kScanTiles) {
    const int cn = min(kScanTiles, nchunks - c0);
    __syncthreads();
    tile_decays(a, c0, cn, bos, len, h, gh, w, lane, sF);
    __syncthreads();
    if (!on) continue;
    int c = 0;
    auto at = [&](int u) { return ((int64_t)(cbase + c0 + c + u) * a.H + h) * E + e; };
    // (a copy of the loop without conditions: with them in it a batch's loads wait for the stores of the one before, 65x31
    // 2 x 9079 tokens, 2 heads 42 -> 54 us)
    auto batches = [&](auto all) {
      for (; c + U <= cn; c += U) {
        float dM[U][VW], dJ[U][VW];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          load_vec<VW>(a.chunk_mu + at(u), dM[u]);
          load_vec<VW>(a.chunk_I + at(u), dJ[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)   // every: 1, 2 or 4
          advance(at(u), dM[u], dJ[u], sF[c + u], decltype(all)::value || u % 4 == 0 || (u % 4 == 2 && a.every == 2));
      }
    };
    if (a.every == 1) batches(std::true_type{});
    else batches(std::false_type{});
    if (const int rest = cn - c; rest > 0) {   // fetched together too
      float dM[U - 1][VW], dJ[U - 1][VW];
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (u < rest) {
          load_vec<VW>(a.chunk_mu + at(u), dM[u]);
          load_vec<VW>(a.chunk_I + at(u), dJ[u]);
        }
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (u < rest) advance(at(u), dM[u], dJ[u], sF[c + u], ((c + u) & (a.every - 1)) == 0);
    }
  }
  if (a.final_mu && on) store_state(a.final_mu + so, a.final_I + so);
}

// The same scan without the precision state: S_c = F_c S_{c-1} + Delta_c with Delta_c read from chunk_mu (fp32).
// The state at the start of every tile is written in bf16 (what its readers feed to the matrix cores) to the
// buffer handed over in the chunk_I slot; the running state stays fp32 and its last value goes to final_mu.
__global__ __launch_bounds__(256) void gla_scan_kernel(ChunkArgs a) {
  bf16_t* tile_S = (bf16_t*)a.chunk_I;
  __shared__ float sF[kScanTiles];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t E = (int64_t)a.dv * a.dk;
  const int nblk = (int)((E + 1023) / 1024);     // four consecutive entries per thread
  const int blk = blockIdx.x % nblk;
  const int nh = blockIdx.x / nblk;
  const int h = nh % a.H, n = nh / a.H;
  const int64_t e = ((int64_t)blk * 256 + tid) * 4;
  const bool on = e < E;
  int bos, len, cbase;
  seq_lookup(a, n, bos, len, cbase);
  const int nchunks = (len + kC - 1) / kC;
  const float gh = a.g[h] * kLog2e;
  const int64_t so = (int64_t)nh * E + e;
  f32x4 S = {0.f, 0.f, 0.f, 0.f};
  if (a.init_mu && on) S = *(const f32x4*)(a.init_mu + so);
  for (int c0 = 0; c0 < nchunks; c0 += kScanTiles) {
    const int cn = min(kScanTiles, nchunks - c0);
    __syncthreads();
    tile_decays(a, c0, cn, bos, len, h, gh, w, lane, sF);
    __syncthreads();
    if (!on) continue;
    int c = 0;
    for (; c + 4 <= cn; c += 4) {
      f32x4 dS[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) dS[u] = *(const f32x4*)(a.chunk_mu + ((int64_t)(cbase + c0 + c + u) * a.H + h) * E + e);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        store_vec<4>(tile_S + ((int64_t)(cbase + c0 + c + u) * a.H + h) * E + e, (const float*)&S);
        const float F = sF[c + u];
#pragma unroll
        for (int x = 0; x < 4; ++x) S[x] = fmaf(F, S[x], dS[u][x]);
      }
    }
    for (; c < cn; ++c) {
      const int64_t off = ((int64_t)(cbase + c0 + c) * a.H + h) * E + e;
      const f32x4 dS = *(const f32x4*)(a.chunk_mu + off);
      store_vec<4>(tile_S + off, (const float*)&S);
      const float F = sF[c];
#pragma unroll
      for (int x = 0; x < 4; ++x) S[x] = fmaf(F, S[x], dS[x]);
    }
  }
  if (a.final_mu && on) *(f32x4*)(a.final_mu + so) = S;
}

void fill_chunk_args(ChunkArgs& a, const PalDims* d, const PalFwdTensors* t) {
  a.q = t->q; a.k = t->k; a.v = t->v; a.b = t->b; a.gt = t->gt;
  a.g = t->g; a.Ip = t->Ip; a.o = t->o;
  a.o_var = (d->flags & PAL_FLAG_HAS_VAR) ? t->o_var : nullptr;
  a.init_mu = t->init_mu; a.init_I = t->init_I;
  a.final_mu = t->final_mu; a.final_I = t->final_I;
  a.cu_seqlens = t->cu_seqlens;
  a.chunk_table = (d->flags & PAL_FLAG_VARLEN) ? t->chunk_table : nullptr;
  a.chunk_offsets = (d->flags & PAL_FLAG_VARLEN) ? t->chunk_offsets : nullptr;
  a.chunk_mu = t->chunk_mu; a.chunk_I = t->chunk_I;
  a.T = d->seq_len; a.H = d->n_heads; a.dk = d->dk; a.dv = d->dv;
  a.Hq = d->n_qk_heads > 0 ? d->n_qk_heads : d->n_heads;
  a.n_seqs = d->n_seqs; a.total_chunks = d->total_chunks;
  a.gate_bf16 = d->gate_dtype == PAL_DTYPE_BF16;
  a.var_bf16 = d->var_dtype == PAL_DTYPE_BF16;
  a.every = 1;
  a.segs = 1;
  a.seg_tiles = 0;
  a.flags = d->flags;
  a.scale = d->scale;
}

}  // namespace pal

namespace pal {
// the outputs from the tile-start states, and how many tiles it walks from one where no one else reads them (chunk_out.hip)
int out_tiles_per_state(const ChunkArgs& a);
bool out_takes_segments(const ChunkArgs& a, int dtype);
int launch_out(const ChunkArgs& a, int dtype, hipStream_t s);
// the one-pass form of chunk_states.hip, and the segments (a.segs, a.seg_tiles) that it cuts a sequence into where few states are kept
void state_pass_segments(ChunkArgs& a);
bool state_pass_applies(const ChunkArgs& a, int dtype, bool has_j);
int launch_state_pass(const ChunkArgs& a, bool has_j, void* tiles_a, float* tiles_b, const float* init_a,
                      const float* init_b, float* fin_a, float* fin_b, bool reverse, float fin_scale, int kern_id,
                      hipStream_t s);

// Local contribution of every tile to the state, into chunk_mu (and chunk_I when has_j).
template <typename TIn, bool HAS_J, typename TS, bool PREC>
static int launch_tile_delta_t(const ChunkArgs& a, hipStream_t s) {
  const int64_t blocks = (int64_t)a.total_chunks * a.H;
  if (blocks > 0x7fffffff) return PAL_E_DIM;
  // value rows per workgroup: all of them, or the largest multiple of 16 whose staging tiles fit the LDS
  int pieces = 1, dvn = a.dv;
  size_t lds = 0;
  for (;; ++pieces) {
    dvn = ((a.dv / 16 + pieces - 1) / pieces) * 16;
    lds = sizeof(float) * kC + sizeof(TS) * (size_t)(a.dk + (HAS_J ? 2 : 1) * dvn) * StageStride<TS>::value;
    if (lds <= kMaxLds || dvn == 16) break;
  }
  if (lds > kMaxLds) return PAL_E_HEADDIM;
  pieces = (a.dv + dvn - 1) / dvn;
  if (int rc = allow_lds((const void*)&chunk_delta_kernel<TIn, HAS_J, TS, PREC>, lds)) return rc;
  PAL_TIMED_LAUNCH(kKernChunkState, s, (chunk_delta_kernel<TIn, HAS_J, TS, PREC>), dim3((unsigned)blocks, (unsigned)pieces),
                   dim3(256), lds, s, a, dvn);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

// fp32 rows take the fp32-accurate variant (fp32 staging, operands split into two bf16 halves) unless
// PAL_FLAG_FP32_FAST asks for single bf16 operands.
template <typename TIn, bool HAS_J>
static int launch_tile_delta_j(const ChunkArgs& a, hipStream_t s) {
  if constexpr (sizeof(TIn) == 4) {
    if (!(a.flags & PAL_FLAG_FP32_FAST)) return launch_tile_delta_t<TIn, HAS_J, float, true>(a, s);
    const size_t lds_f32 = sizeof(float) * (kC + (size_t)(a.dk + (HAS_J ? 2 : 1) * a.dv) * StageStride<float>::value);
    if (lds_f32 <= kMaxLds) return launch_tile_delta_t<TIn, HAS_J, float, false>(a, s);
  }
  return launch_tile_delta_t<TIn, HAS_J, bf16_t, false>(a, s);
}

int launch_tile_delta(const ChunkArgs& a, int dtype, bool has_j, hipStream_t s) {
  if (dtype == PAL_DTYPE_BF16)
    return has_j ? launch_tile_delta_j<bf16_t, true>(a, s) : launch_tile_delta_j<bf16_t, false>(a, s);
  return has_j ? launch_tile_delta_j<float, true>(a, s) : launch_tile_delta_j<float, false>(a, s);
}

// Tile-start states: local contributions, then the serial scan over the tiles of each sequence.
// has_j = false leaves the precision state out (b, Ip, chunk_I, init_I, final_I are not touched).
int launch_tile_states(const ChunkArgs& a, int dtype, bool has_j, hipStream_t s) {
  if (state_pass_applies(a, dtype, has_j))
    return launch_state_pass(a, has_j, has_j ? (void*)a.chunk_mu : (void*)a.chunk_I, has_j ? a.chunk_I : nullptr, a.init_mu,
                             a.init_I, a.final_mu, a.final_I, false, 1.f, kKernChunkStates, s);
  if (int rc = launch_tile_delta(a, dtype, has_j, s)) return rc;
  {
    const int64_t E = (int64_t)a.dv * a.dk, nh = (int64_t)a.n_seqs * a.H;
    const int64_t blocks = nh * scan_blocks(E, 4);
    if (nh * scan_blocks(E, 1) > 0x7fffffff) return PAL_E_DIM;
    // few blocks: one entry per thread spreads them over more compute units, each of which moves only so much
    // (1 x 16384 tokens, 4 heads of 48x48, 12 blocks: 59 -> 37 us; 1 x 8192, 16 of 64x64, 64 blocks: 37 -> 31)
    if (has_j && blocks < 256) PAL_TIMED_LAUNCH(kKernChunkScan, s, chunk_scan_kernel<1>, dim3((unsigned)(nh * scan_blocks(E, 1))), dim3(256), 0, s, a);
    else if (has_j) PAL_TIMED_LAUNCH(kKernChunkScan, s, chunk_scan_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, s, a);
    else PAL_TIMED_LAUNCH(kKernChunkScan, s, gla_scan_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
    PAL_HIP_LAUNCH_CHECK();
  }
  return PAL_OK;
}

}  // namespace pal

// ------------------------------------------------------------ forward on the library's own scratch
// The tile-start states of pal_chunk_fwd_static live here instead of in caller memory.  Every GPU the library runs on
// holds its own copy of this array (at its own address) until the process ends.
static __device__ __align__(256) float scratch[PAL_STATIC_SCRATCH_BYTES / sizeof(float)];

namespace pal {

// Device address of `scratch` on the current device.  In host code the array's name is only a handle of the symbol,
// not memory a kernel can touch: the address is asked for once per device (with that device current) and kept.
constexpr int kMaxDevices = 64;
static std::atomic<float*> g_scratch_ptr[kMaxDevices];

static int static_scratch(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return PAL_E_DIM;
  float* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    void* addr = nullptr;
    e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!addr) return (int)hipErrorInvalidSymbol;
    p = (float*)addr;
    g_scratch_ptr[dev].store(p, std::memory_order_release);   // two threads racing here store the same address
  }
  *out = p;
  return PAL_OK;
}

}  // namespace pal

extern "C" int pal_chunk_fwd_static(const PalDims* d, const PalFwdTensors* t, void* stream) {
  using namespace pal;
  if (!d || !t) return PAL_E_NULL;
  if (t->chunk_mu || t->chunk_I) return PAL_E_STATE;   // the states live in the library's scratch on this path
  PalFwdTensors tt = *t;
  // any aligned non-null value passes the pointer checks; the real addresses follow once the size is known to fit
  tt.chunk_mu = tt.chunk_I = (float*)(uintptr_t)256;
  int rc = check_chunk_common(d, &tt);
  if (rc) return rc;
  const uint64_t entries = (uint64_t)d->total_chunks * (uint64_t)d->n_heads * (uint64_t)d->dv * (uint64_t)d->dk;
  if (entries > PAL_STATIC_SCRATCH_BYTES / (2 * sizeof(float))) return PAL_E_SCRATCH;
  float* base = nullptr;
  rc = static_scratch(&base);
  if (rc) return rc;
  tt.chunk_mu = base;
  tt.chunk_I = base + PAL_STATIC_SCRATCH_BYTES / (2 * sizeof(float));
  ChunkArgs a;
  fill_chunk_args(a, d, &tt);
  hipStream_t s = (hipStream_t)stream;
  // every slot the output kernel reads is written by the state kernels of this call first: nothing has to start at zero
  if (int rc2 = launch_tile_states(a, d->dtype, true, s)) return rc2;
  return launch_out(a, d->dtype, s);
}

// tiles per kept state, and the segments of the pass that makes them, where the caller needs no state afterwards
static void sparse_states(pal::ChunkArgs& a, int dtype) {
  a.every = pal::out_tiles_per_state(a);
  if (pal::state_pass_applies(a, dtype, true) && pal::out_takes_segments(a, dtype)) pal::state_pass_segments(a);
}

extern "C" int pal_chunk_fwd_segments(const PalDims* d, int32_t* tiles_per_state, int32_t* tiles_per_segment) {
  if (!tiles_per_state || !tiles_per_segment) return PAL_E_NULL;
  if (int rc = pal_validate_dims(d)) return rc;
  const PalFwdTensors none = {};
  pal::ChunkArgs a;
  pal::fill_chunk_args(a, d, &none);
  if (d->flags & PAL_FLAG_SPARSE_STATES) sparse_states(a, d->dtype);
  *tiles_per_state = a.every;
  *tiles_per_segment = a.seg_tiles;
  return a.segs;
}

extern "C" int pal_chunk_fwd(const PalDims* d, const PalFwdTensors* t, void* stream) {
  using namespace pal;
  if (d && t && (d->flags & PAL_FLAG_STATES_ONLY)) {
    // tile-start states only: the outputs are not touched and need not exist
    PalDims dd = *d;
    dd.flags &= ~(uint32_t)(PAL_FLAG_STATES_ONLY | PAL_FLAG_HAS_VAR);
    PalFwdTensors tt = *t;
    tt.o = (void*)(uintptr_t)256;   // passes the pointer checks, never dereferenced
    tt.o_var = nullptr;
    int rc = check_chunk_common(&dd, &tt);
    if (rc) return rc;
    ChunkArgs a;
    fill_chunk_args(a, &dd, &tt);
    return launch_tile_states(a, dd.dtype, true, (hipStream_t)stream);
  }
  int rc = check_chunk_common(d, t);
  if (rc) return rc;
  constexpr uint32_t forms = PAL_FLAG_STATES_TWO_KERNELS | PAL_FLAG_STATES_ONE_PASS | PAL_FLAG_FP32_FAST;
  if ((d->flags & PAL_FLAG_OUTPUTS_ONLY) && !(d->flags & forms) && short_pass(d)) {
    PalDims r = *d;
    r.flags &= PAL_FLAG_HAS_INIT | PAL_FLAG_STORE_FINAL | PAL_FLAG_HAS_VAR;
    return pal_recurrent_fwd(&r, t, stream);
  }
  ChunkArgs a;
  fill_chunk_args(a, d, t);
  if (d->flags & PAL_FLAG_SPARSE_STATES) sparse_states(a, d->dtype);
  hipStream_t s = (hipStream_t)stream;
  if (int rc2 = launch_tile_states(a, d->dtype, true, s)) return rc2;
  return launch_out(a, d->dtype, s);
}
