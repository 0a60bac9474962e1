// Pieces shared by the chunked forward and backward kernels.
//
// Chunked form of the recurrence (one sequence, one head, a tile of C = 64
// tokens; c_t = running sum of log2 f inside the tile, F_t = 2^{c_t},
// L[t,s] = 2^{c_t - c_s} for s <= t, else 0):
//   M_t = sum_s L[t,s] v_s k_s^T + F_t M_0          (the associative scan of the
//   I_t = sum_s L[t,s] b_s (k_s*k_s)^T + F_t (I_0 - Ip) + Ip    reference,
//                                     chunk_palimpsa_forgetting_scalar.py:190-195)
// M_0, I_0 are the fp32 states at the start of the tile.  The kernels that carry the state from tile to tile take the
// sums over s as bf16 MFMA contractions with fp32 accumulation; those that work inside the tiles run token by token.
#pragma once
#include "pal_common.h"

namespace pal {

constexpr int kC = PAL_CHUNK;  // tokens per tile
constexpr int kScanTiles = 1024;   // per-tile decays a scan kernel keeps in LDS at a time

// internal bit of ChunkArgs::flags (above the PAL_FLAG_* bits): chunk_delta_kernel weights token s with the decay
// from the start of the tile up to s instead of from s to the end of the tile
constexpr uint32_t kFlagDecayFromStart = 1u << 30;

struct ChunkArgs {
  const void *q, *k, *v, *b, *gt;
  const float *g, *Ip;
  void *o, *o_var;
  const float *init_mu, *init_I;
  float *final_mu, *final_I;
  const int32_t *cu_seqlens, *chunk_table, *chunk_offsets;
  float *chunk_mu, *chunk_I;
  int32_t T, H, dk, dv, n_seqs, total_chunks;
  int32_t Hq;   // heads of q and k: H, or a divisor of it when a group of H / Hq value heads shares one q/k head
  int32_t gate_bf16, var_bf16;
  int32_t every;   // tiles per tile-start state that is kept: 1, or more where the output kernel walks that many from one
  int32_t segs, seg_tiles;   // segments that a sequence's state pass is cut into, tiles of one (a multiple of `every`; 1, 0: none)
  uint32_t flags;
  float scale;
};

// Segments of the state pass (chunk_states.hip): the tile states that are kept are sums since the start of their segment, M and J as
// they are, and the state before the segment is added where they are read.  Of the slots of a segment's tiles, of which only
// every fourth is kept, the second holds the segment's total, in its place then the state before it; the third and fourth of
// chunk_mu the decays since the start of the segment, [kept tile][head], and over the whole of it.
// A decay over thousands of tokens is kept as a number in [1/2, 1) and a power of two: as one fp32 number it leaves the range where
// tokens grow (f > 1) or a state is large, when the state itself, which the walk multiplies tile by tile, does not.
struct SegDecay {
  float m, e;
  __device__ __forceinline__ void times(float F) {   // (infinities, NaN and zero stay in m)
    m *= F;
    e += (float)__builtin_amdgcn_frexp_expf(m);
    m = __builtin_amdgcn_frexp_mantf(m);
  }
  // the state x after the decay, plus y: one rounding, as of a product with the number itself
  __device__ __forceinline__ float apply(float x, float y) const { return fmaf(m, __builtin_amdgcn_ldexpf(x, (int)e), y); }
};
__device__ __forceinline__ int64_t seg_slot(const ChunkArgs& a, int n, int seg, int h) {
  const int tiles = (a.T + kC - 1) / kC;
  return ((int64_t)(n * tiles + seg * a.seg_tiles + 1) * a.H + h) * a.dv * a.dk;
}
__device__ __forceinline__ SegDecay* seg_decays(const ChunkArgs& a, int n, int seg) {
  const int tiles = (a.T + kC - 1) / kC;
  return (SegDecay*)(a.chunk_mu + (int64_t)(n * tiles + seg * a.seg_tiles + 2) * a.H * a.dv * a.dk);
}

// q and k rows of value head h: element offset of token t's row, and the token stride, in a [tokens, Hq, dk] tensor
__device__ __forceinline__ int64_t qk_row(const ChunkArgs& a, int64_t t, int h) {
  return (t * a.Hq + (a.Hq == a.H ? h : h / (a.H / a.Hq))) * a.dk;   // (a division is forty instructions)
}
__device__ __forceinline__ int64_t qk_stride(const ChunkArgs& a) { return (int64_t)a.Hq * a.dk; }

// tile c -> (sequence, first token in the packed/batched token axis, tokens in tile, index in sequence)
__device__ __forceinline__ void chunk_lookup(const ChunkArgs& a, int c, int& seq, int& t0, int& clen, int& cis) {
  if (a.chunk_table) {
    const int32_t* row = a.chunk_table + 4 * (int64_t)c;
    seq = min(max(row[0], 0), a.n_seqs - 1);
    cis = row[3];
    // a tile stays inside the packed token axis whatever the table holds (its first token always exists:
    // masked lanes still address it)
    t0 = min(max(row[1], 0), a.T - 1);
    clen = min(max(row[2], 0), min(kC, a.T - t0));
  } else {
    const int per = (a.T + kC - 1) / kC;
    seq = c / per;
    cis = c - seq * per;
    t0 = seq * a.T + cis * kC;
    clen = min(kC, a.T - cis * kC);
  }
}

// sequence n -> (first token, length, index of its first tile)
__device__ __forceinline__ void seq_lookup(const ChunkArgs& a, int n, int& bos, int& len, int& cbase) {
  if (a.cu_seqlens) {
    packed_seq_bounds(a.cu_seqlens, n, a.T, bos, len);
    // the tiles of a sequence stay inside the per-tile buffers
    cbase = min(max(a.chunk_offsets[n], 0), a.total_chunks);
    len = min(len, (a.total_chunks - cbase) * kC);
  } else {
    bos = n * a.T;
    len = a.T;
    cbase = n * ((a.T + kC - 1) / kC);
  }
}

// A workgroup per (tile, head).  Consecutive workgroup ids go to different XCDs: the heads of a tile are dealt to one of them
// side by side, since rows that are no multiple of a cache line leave lines to two heads.
__host__ __device__ inline bool tiles_by_xcd(int64_t tiles) { return tiles >= 64; }
inline int64_t tile_head_blocks(int64_t tiles, int H) { return (tiles_by_xcd(tiles) ? (tiles + 7) / 8 * 8 : tiles) * H; }
__device__ __forceinline__ bool tile_head(int tiles, int H, int block, int& tile, int& h) {
  if (tiles_by_xcd(tiles)) {
    const int l = block >> 3, t = l / H;
    tile = t * 8 + (block & 7);
    h = l - t * H;
    return tile < tiles;
  }
  tile = block / H;
  h = block - tile * H;
  return true;
}

// Workgroups that walk the tiles of a sequence in order, one per (sequence, head, slice): consecutive workgroup ids go to
// different XCDs, the slices of one (sequence, head) belong on the same one (they read the same rows).
struct WalkPlan {
  int32_t n_sl, per_xcd, total;
  int32_t by_length;   // packed sequences are handed out longest first (see walk_item)
};
inline bool walk_plan(const ChunkArgs& a, int n_sl, WalkPlan& p) {
  const int64_t total = (int64_t)a.n_seqs * a.H * n_sl;
  int64_t per_xcd = (total + 7) / 8;
  per_xcd = (per_xcd + n_sl - 1) / n_sl * n_sl;
  p.by_length = (a.cu_seqlens && a.n_seqs > 1 && a.n_seqs <= 64) ? 1 : 0;
  if (p.by_length) per_xcd = (int64_t)((a.n_seqs + 7) / 8) * a.H * n_sl;   // whole sequences per XCD
  if (per_xcd * 8 > 0x7fffffff) return false;
  p.n_sl = n_sl;
  p.total = (int32_t)total;
  p.per_xcd = (int32_t)per_xcd;   // the grid is 8 per_xcd workgroups
  return true;
}
// the workgroup's sequence, head and slice; false: it has none
__device__ __forceinline__ bool walk_item(const ChunkArgs& a, const WalkPlan& p, int lane, int& n, int& h, int& sl) {
  const int xcd = (int)blockIdx.x & 7, pos = (int)blockIdx.x >> 3;
  int m;
  if (p.by_length) {
    // Packed sequences of unequal length (at most 64): the walk over a sequence's tiles is serial, so a long sequence
    // that starts late ends the kernel late.  The sequence of rank r in descending length goes to XCD r mod 8, in
    // rank order there; every wave finds the sequence of its rank with one lane per sequence.
    const int rank = (pos / (a.H * p.n_sl)) * 8 + xcd;
    if (rank >= a.n_seqs) return false;
    int b_l = 0, len_l = -1;
    if (lane < a.n_seqs) packed_seq_bounds(a.cu_seqlens, lane, a.T, b_l, len_l);
    int before = 0;   // sequences ahead of lane's own in the order (longer, or as long with a smaller index)
    for (int j = 0; j < a.n_seqs; ++j) {
      const int len_j = __builtin_amdgcn_readlane(len_l, j);
      before += (len_j > len_l || (len_j == len_l && j < lane)) ? 1 : 0;
    }
    const uint64_t hit = __ballot(lane < a.n_seqs && before == rank);
    n = hit ? (int)__builtin_ctzll(hit) : 0;
    m = n * a.H * p.n_sl + pos % (a.H * p.n_sl);
  } else {
    m = xcd * p.per_xcd + pos;
    if (m >= p.total) return false;
    n = (m / p.n_sl) / a.H;
  }
  sl = m % p.n_sl;
  h = (m / p.n_sl) % a.H;
  return true;
}

// lane l of a row of 16 gets lane l + N's value, zero from beyond the row
template <int N>
__device__ __forceinline__ float row_shl_zero(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x100 + N, 0xf, 0xf, true));
}
// inclusive prefix sum over the 64 lanes of a wave: four shifted adds inside each row of 16 lanes (DPP
// row_shr with zero fill), then the totals of the rows before (lane 15 of each, read as scalars)
template <int N>
__device__ __forceinline__ float row_shr_zero(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x110 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_inclusive_scan(float x, int lane) {
  x += row_shr_zero<1>(x);
  x += row_shr_zero<2>(x);
  x += row_shr_zero<4>(x);
  x += row_shr_zero<8>(x);
  const float t0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 15));
  const float t1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 31));
  const float t2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 47));
  const int row = lane >> 4;
  return x + (row == 0 ? 0.f : row == 1 ? t0 : row == 2 ? t0 + t1 : (t0 + t1) + t2);
}

// Decays over the tiles [c0, c0 + cn) of a sequence, by the four waves of a scan's workgroup in turn.  A wave fetches eight tiles'
// gates before the first is used: one at a time, this set-up is a chain of fetches that took longer than the scan itself (1 x 16384
// tokens, 4 heads of 48x48: 72 us, so 59).
__device__ __forceinline__ void tile_decays(const ChunkArgs& a, int c0, int cn, int bos, int len, int h, float gh, int w, int lane,
                                            float* sF) {
  constexpr int N = 8;
  for (int c = w; c < cn; c += 4 * N) {
    float gt[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int t = (c0 + c + 4 * u) * kC + lane;
      gt[u] = t < len ? load_gate(a.gt, (int64_t)(bos + t) * a.H + h, a.gate_bf16) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (c + 4 * u < cn) {
        const float tot = wave_sum(-gt[u] * gh);
        if (lane == 0) sF[c + 4 * u] = fast_exp2(tot);
      }
    }
  }
}

}  // namespace pal
