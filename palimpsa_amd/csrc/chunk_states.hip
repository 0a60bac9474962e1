// Tile-start states of the chunked algorithm in one pass (bf16 rows):
//     S_c = F_c S_{c-1} + Delta_c ,  Delta_c = sum_s a_s v_s k_s^T  (and sum_s a_s b_s (k_s*k_s)^T for the
//     precision state)
// computed by a workgroup that walks the tiles of one sequence in order with the running state in the
// accumulators of the matrix cores, so that the per-tile contributions Delta_c never go to memory (the
// two-kernel form, chunk_delta_kernel + a scan kernel, writes them in fp32 and reads them back: three times
// the bytes of the states themselves).  What the reference keeps as intermediate_*_state
// (chunk_palimpsa_forgetting_scalar.py:187-188) is written at the start of every tile, the state after
// the last tile at the end (:214-218).
//
// One workgroup of 12 waves per (sequence, head, slice of ds value rows): four hold the state (the slice times
// dk is at most 6144 entries = 24 blocks of 16x16, up to six per wave), two groups of four stage the rows for them.  The
// rows of a tile lie in LDS as they lie in memory, v and b times the weight of their token, 16 bytes a write; the matrix
// cores take the tokens as contraction index, which the transposing LDS reads turn to the front (four bf16 of a column from
// four rows at once).  The row stride is an odd number of 32-byte pieces, so neither side conflicts.  (Staged transposed, two
// tokens to a word, the 4-byte writes and their packing were what the feeding waves spent their time on: whole passes over 4 x 2048
// tokens, 6 heads of 96 x 192 with the precision state 74.6 us against 54.2, 4 x 1000, 12 of 192 x 64 51.4 against 27.3,
// 8 x 2048, 16 of 48 x 48 52.8 against 47.4; scalar-gated 2 x 2048, 16 of 128 x 128 46 against 24.)
// The serial chain over the tiles is hidden by fetching ahead: rows are fetched into registers three steps before they
// go to LDS, two LDS buffers hold the current and the next tile, one barrier per tile.
// What bounds it with the precision state, where every tile's is kept: writing mu and I (8 bytes an entry) beside reading rows that come from HBM, at
// 2.5 - 3.3 TB/s together; without the stores the walk takes half the time, and neither fetching further ahead (up to 10
// tiles), whole 128-byte lines a store nor non-temporal stores gave more than 6 % at any shape without losing as much at
// another.
// The same kernel walks a sequence backwards for the gradient of the scalar-gated path (weights from the
// start of the tile, G_{c-1} = F_c G_c + D_c, the value left after the first tile is the gradient of the
// initial state).
#include <type_traits>

#include "chunk_common.h"
#include "pal_host.h"
#include "pal_profile.h"

namespace pal {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kStMaxBlocks = 6;    // 16x16 state blocks per wave
// row stride (bf16) of a staged tile of n columns: an odd number of 32-byte pieces, so that the four rows by 32 bytes of a
// transposing read lie on different banks in every lane group
__host__ __device__ constexpr int staged_stride(int n) { return 16 * ((n >> 4) | 1); }

struct StatePassArgs {
  ChunkArgs c;
  void* tiles_a;          // scalar-gated: bf16 tile states; Palimpsa: fp32 mu at the start of every tile
  float* tiles_b;         // Palimpsa: fp32 I at the start of every tile
  const float *init_a, *init_b;
  float *fin_a, *fin_b;
  WalkPlan plan;
  int32_t ds, reverse;
  int32_t dks, ksplit;    // key columns per workgroup and slices of the key columns (dk = dks * ksplit)
  float fin_scale;
};

template <int NIK, int NIV>
struct StageRegs {
  u32x4 k[NIK], v[NIV];
  uint32_t gt;   // gate of token `lane` as loaded: fp32 bits or a bf16 in the low half (last wave)
};

// NIK: 16-byte pieces of k per feeding thread and tile (32 columns each); DSB: 16 value rows each of the slice
template <bool HAS_J, int NIK, int DSB>
__global__ __launch_bounds__(768) void chunk_states_kernel(StatePassArgs A) {
  constexpr int NIV = HAS_J ? DSB : (DSB + 1) / 2;       // pieces of v and b per feeding thread
  constexpr int NSB = (DSB * NIK + 1) / 2;               // state blocks per wave
  static_assert(NSB <= kStMaxBlocks, "state blocks of a wave");
  const ChunkArgs& a = A.c;
  extern __shared__ float smem[];
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.H, dk = a.dk, dv = a.dv, dks = A.dks;
  constexpr int ds = 16 * DSB;
  // A workgroup owns the state entries (value rows [d0, d0 + ds)) x (key columns [k0, k0 + dks)) of a (sequence, head).
  int n, h, sl;
  if (!walk_item(a, A.plan, lane, n, h, sl)) return;
  const bool segs = HAS_J && a.segs > 1;
  const int seg = segs ? n % a.segs : 0;
  if (segs) n /= a.segs;
  const int d0 = (sl / A.ksplit) * ds, k0 = (sl % A.ksplit) * dks;
  const int nh = n * H + h;
  int bos, len, cbase;
  seq_lookup(a, n, bos, len, cbase);
  if (segs) {
    const int t = seg * a.seg_tiles * kC;
    bos += t;
    len = min(len - t, a.seg_tiles * kC);
    cbase += seg * a.seg_tiles;
  }
  const int nchunks = (len + kC - 1) / kC;

  float* sA = smem;                                   // [3][64] weight of token s in its tile (ring over tiles)
  float* sF = sA + 3 * kC;                            // [3] decay over the whole tile (+1 pad)
  const int KS = staged_stride(dks);
  constexpr int VS = staged_stride(ds);
  bf16_t* sK = (bf16_t*)(sF + 4);                     // [2][64 tokens][KS]
  bf16_t* sV = sK + 2 * kC * KS;                      // [2][64][VS]: v times the weight of its token
  bf16_t* sB = sV + 2 * kC * VS;                      // [2][64][VS] (HAS_J)
  const int kbuf = kC * KS;
  constexpr int vbuf = kC * VS;

  // Waves 0-3 own the state (a 16x16 block per wave and slot), waves 4-11 feed them: a single wave issues an
  // instruction every five to eight cycles, so the kinds of work sit on different waves of each SIMD instead
  // of following one another.  The feeding waves form two groups of four, one for the even tiles (LDS buffer
  // 0) and one for the odd tiles (buffer 1): a group works out the weights of a tile and fetches ahead in one
  // step, and puts the tile's rows into its buffer in the next, while the other group does the opposite.
  // All roles pass the same barriers, one per step; steps -2 and -1 fill the pipeline.
  if (w >= 4) {
    // ---------------------------------------------------------------- staging role
    // Items of a thread: (token, 8 columns), of k, and of v followed by b (which of the two is the same for all of a wave);
    // the last wave turns the gates of a tile into its weights (in the step in which the group stages nothing).  Byte
    // offsets from the first row of a tile and places in the staging tiles do not change from tile to tile.
    const int grp = (w - 4) >> 2;           // parity of the tiles this group stages
    const int wg = (w - 4) & 3;             // wave in the group
    const int st = tid - 256 - 256 * grp;
    uint32_t koff[NIK], voff[NIV];
    int kdst[NIK], vdst[NIV], vtok[NIV];
    bool kval[NIK], vval[NIV];
#pragma unroll
    for (int j = 0; j < NIK; ++j) {
      const int per = dks >> 3, idx = st + 256 * j, s = idx / per, c8 = idx - s * per;
      kval[j] = s < kC;
      koff[j] = kval[j] ? (uint32_t)((s * a.Hq * dk + k0 + 8 * c8) * 2) : 0x80000000u;
      kdst[j] = s * KS + 8 * c8;
    }
#pragma unroll
    for (int j = 0; j < NIV; ++j) {
      const int idx = st + 256 * j, it = idx % (128 * DSB), s = it / (2 * DSB), c8 = it % (2 * DSB);
      vval[j] = idx < (HAS_J ? 2 : 1) * 128 * DSB;
      voff[j] = vval[j] ? (uint32_t)((s * H * dv + 8 * c8) * 2) : 0x80000000u;
      vdst[j] = s * VS + 8 * c8;
      vtok[j] = s;
    }
    // Rows are fetched through buffer descriptors that end with the last row of the sequence: the byte offset
    // of a row piece is a per-thread constant plus the offset of the tile, rows beyond the end of the sequence
    // (the tail of its last tile, tiles past its end) are out of range and read as zero, so no fetch needs a
    // branch or a select.  Nothing touches a fetched value before it goes to LDS: any use here would make the
    // wave wait for everything it has in flight, which is what fetching ahead is meant to avoid.
    const bf16_t* kbase = (const bf16_t*)a.k + qk_row(a, bos, h);
    const bf16_t* vbase = (const bf16_t*)a.v + ((int64_t)bos * H + h) * dv + d0;
    const int esz = a.gate_bf16 ? 2 : 4;
    const uint32_t kbytes = len > 0 ? (uint32_t)(((len - 1) * a.Hq * dk + dk) * 2) : 0u;
    const uint32_t vbytes = len > 0 ? (uint32_t)(((len - 1) * H * dv + ds) * 2) : 0u;
    const uint32_t gbytes = len > 0 ? (uint32_t)(((len - 1) * H + 1) * esz) : 0u;
    const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc((void*)kbase, 0, kbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc((void*)vbase, 0, vbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t brs = __builtin_amdgcn_make_buffer_rsrc(
        HAS_J ? (void*)((const bf16_t*)a.b + ((int64_t)bos * H + h) * dv + d0) : (void*)vbase, 0, vbytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)a.gt + ((int64_t)bos * H + h) * esz), 0, gbytes, 0x00020000);
    const uint32_t goff = (uint32_t)(lane * H * esz);
    const float gh = a.g[h] * kLog2e;
    const bool from_start = (a.flags & kFlagDecayFromStart) != 0;

    auto load_stage = [&](StageRegs<NIK, NIV>& R, int p) {
      const int c = A.reverse ? nchunks - 1 - p : p;
      const bool live = p < nchunks;
      // a tile past the end: every offset out of range
      const uint32_t tk = live ? (uint32_t)(c * kC * a.Hq * dk * 2) : 0x80000000u;
      const uint32_t tv = live ? (uint32_t)(c * kC * H * dv * 2) : 0x80000000u;
#pragma unroll
      for (int j = 0; j < NIK; ++j) R.k[j] = __builtin_amdgcn_raw_buffer_load_b128(krs, koff[j] + tk, 0, 0);
#pragma unroll
      for (int j = 0; j < NIV; ++j) {
        const bool is_b = HAS_J && 64 * wg + 256 * j >= 128 * DSB;
        R.v[j] = __builtin_amdgcn_raw_buffer_load_b128(is_b ? brs : vrs, voff[j] + tv, 0, 0);
      }
      if (wg == 3) {
        const uint32_t tg = live ? (uint32_t)(c * kC * H * esz) : 0x80000000u;
        R.gt = a.gate_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(grs, goff + tg, 0, 0)
                           : __builtin_amdgcn_raw_buffer_load_b32(grs, goff + tg, 0, 0);   // raw; widened below
      }
    };
    // v and b are staged times the weight of their token (the operand the matrix cores take is a_s v_s, rounded to bf16 once)
    auto store_stage = [&](const StageRegs<NIK, NIV>& R, int buf, int p) {
#pragma unroll
      for (int j = 0; j < NIK; ++j)
        if (kval[j]) *(u32x4*)&sK[buf * kbuf + kdst[j]] = R.k[j];
      const float* wts = sA + (p % 3) * kC;
#pragma unroll
      for (int j = 0; j < NIV; ++j) {
        if (vval[j]) {
          const float wt = wts[vtok[j]];
          u32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t word = R.v[j][e];
            const bf16x2 y = pack2(wt * __builtin_bit_cast(float, word << 16), wt * __builtin_bit_cast(float, word & 0xffff0000u));
            x[e] = __builtin_bit_cast(uint32_t, y);
          }
          const bool is_b = HAS_J && 64 * wg + 256 * j >= 128 * DSB;
          *(u32x4*)&(is_b ? sB : sV)[buf * vbuf + vdst[j]] = x;
        }
      }
    };
    // weights of the tokens of tile p and the decay over the whole tile, one step before its rows are staged
    auto scan_stage = [&](const StageRegs<NIK, NIV>& R, int p) {
      if (wg == 3) {
        const float gt = __builtin_bit_cast(float, a.gate_bf16 ? R.gt << 16 : R.gt);   // zero beyond the sequence
        const float cs = wave_inclusive_scan(-gt * gh, lane);
        const float tot = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cs), 63));
        sA[(p % 3) * kC + lane] = fast_exp2(from_start ? cs : tot - cs);
        if (lane == 0) sF[p % 3] = fast_exp2(tot);
      }
    };

    // Two register sets per group: the tile being staged and the group's next one (two tiles later), which is
    // fetched three steps before its rows go to LDS.  In step p the group of parity (p + 1) & 1 stages tile p + 1,
    // the other one handles tile p + 2: weights from its gates (set (p + 2) / 2 % 2), then the fetch of tile p + 4
    // into the set that was staged a step ago.
    // (One copy of the loop per group: with the group a compile-time constant the order of fetches and uses is
    // static, and the compiler can count how many younger fetches may still be in flight when a set is used;
    // with a run-time test it has to wait for all of them, which throws the fetching ahead away.)
    auto run = [&](auto parity) {
      constexpr int G = decltype(parity)::value;
      StageRegs<NIK, NIV> R[2];
      load_stage(R[0], G);
      for (int p0 = -2; p0 < nchunks; p0 += 4) {
#pragma unroll
        for (int ph = 0; ph < 4; ++ph) {
          const int p = p0 + ph;           // p + 2 = ph (mod 4)
          if ((ph & 1) == G) {   // folds once the loop is unrolled
            scan_stage(R[(ph >> 1) & 1], p + 2);
            load_stage(R[1 - ((ph >> 1) & 1)], p + 4);
          } else {
            if (p + 1 >= 0) store_stage(R[(((ph + 3) & 3) >> 1) & 1], G, p + 1);
          }
          __syncthreads();
        }
      }
    };
    if (grp == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    return;
  }

  // ------------------------------------------------------------------ state role
  // state blocks of this wave: block sb = w + 4 jj -> (value rows 16 db.., key columns 16 nb..)
  const int NB = dks >> 4, blocks = DSB * NB;
  int ldk[NSB], ldv[NSB], goff[NSB];   // operands in the staging tiles, entry in a state
  bool sval[NSB];
  f32x4 accM[NSB], accJ[NSB];
  const int64_t E = (int64_t)dv * dk;
  const float Ip = HAS_J ? a.Ip[h] : 0.f;
#pragma unroll
  for (int jj = 0; jj < NSB; ++jj) {
    const int sb = w + 4 * jj;
    sval[jj] = sb < blocks;
    const int db = sval[jj] ? sb / NB : 0, nb = sval[jj] ? sb - db * NB : 0;
    // rows n = 16 nb + 4 g + r (four consecutive key columns), column d = d0 + 16 db + i
    ldk[jj] = (4 * g + (i >> 2)) * KS + 16 * nb + 4 * (i & 3);
    ldv[jj] = (4 * g + (i >> 2)) * VS + 16 * db + 4 * (i & 3);
    goff[jj] = (d0 + 16 * db + i) * dk + k0 + 16 * nb + 4 * g;
    accM[jj] = f32x4{0.f, 0.f, 0.f, 0.f};
    accJ[jj] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (sval[jj] && A.init_a && seg == 0) {
      const int64_t off = (int64_t)nh * E + goff[jj];
      const f32x4 x = *(const f32x4*)(A.init_a + off);
      if (HAS_J) {
        const f32x4 I = *(const f32x4*)(A.init_b + off);
#pragma unroll
        for (int r = 0; r < 4; ++r) { accM[jj][r] = x[r] * I[r]; accJ[jj][r] = I[r] - Ip; }
      } else {
        accM[jj] = x;
      }
    }
  }
  __syncthreads();   // steps -2 and -1 of the feeding waves
  __syncthreads();
  SegDecay Fseg = {1.f, 0.f};   // decay since the start of the segment
  for (int p = 0; p < nchunks; ++p) {
    const int buf = p & 1;
    const int c = A.reverse ? nchunks - 1 - p : p;
    const int64_t slot = ((int64_t)(cbase + c) * H + h) * E;
    const float F = sF[p % 3];
    const bf16_t* kt = sK + buf * kbuf;
    const bf16_t* vt = sV + buf * vbuf;
    const bf16_t* bt = sB + buf * vbuf;
    const bool kept = !HAS_J || (c & (a.every - 1)) == 0;
    if (segs && w == 0) {
      if (lane == 0 && sl == 0 && kept) seg_decays(a, n, seg)[c / a.every * H + h] = Fseg;
      Fseg.times(F);
    }
    // operands, the tokens as contraction index (g, j) -> 32 ks + 16 (j / 4) + 4 g + j % 4; those of the next block are read
    // while a block is worked
    struct Ops { bf16x8 k[2], v[2], b[2]; } x[2];
    auto read = [&](int jj, Ops& y) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const bf16_t* pk = kt + ldk[jj] + 32 * ks * KS;
        const bf16_t* pv = vt + ldv[jj] + 32 * ks * VS;
        const bf16_t* pb = bt + ldv[jj] + 32 * ks * VS;
        y.k[ks] = join(lds_read_tr(pk), lds_read_tr(pk + 16 * KS));
        y.v[ks] = join(lds_read_tr(pv), lds_read_tr(pv + 16 * VS));
        if (HAS_J) y.b[ks] = join(lds_read_tr(pb), lds_read_tr(pb + 16 * VS));
      }
    };
    read(0, x[0]);
#pragma unroll
    for (int jj = 0; jj < NSB; ++jj) {
      if (jj > 0 && !sval[jj]) break;
      if (jj + 1 < NSB) read(jj + 1, x[(jj + 1) & 1]);   // (a block that the wave has not repeats the first one's)
      __builtin_amdgcn_sched_barrier(0);
      const Ops& y = x[jj & 1];
      const int64_t off = slot + goff[jj];
      if (sval[jj] && kept) {
        if (HAS_J) {
          f32x4 mu, I;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            I[r] = segs ? accJ[jj][r] : accJ[jj][r] + Ip;
            mu[r] = segs ? accM[jj][r] : accM[jj][r] * fast_rcp(I[r]);
          }
          *(f32x4*)((float*)A.tiles_a + off) = mu;
          *(f32x4*)(A.tiles_b + off) = I;
        } else {
          store_vec<4>((bf16_t*)A.tiles_a + off, (const float*)&accM[jj]);
        }
      }
      f32x4 M = accM[jj] * F, J = accJ[jj] * F;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        M = mfma16(y.k[ks], y.v[ks], M);
        if (HAS_J) {
          bf16x8 kk;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float kf = (float)y.k[ks][j];
            kk[j] = (bf16_t)(kf * kf);
          }
          J = mfma16(kk, y.b[ks], J);
        }
      }
      accM[jj] = M;
      accJ[jj] = J;
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  }
  // the feeding waves take their steps in groups of four, starting at -2
  for (int p = nchunks; ((p + 2) & 3) != 0; ++p) __syncthreads();

  if (segs) {
    if (w == 0 && lane == 0 && sl == 0) seg_decays(a, n, seg)[a.seg_tiles / a.every * H + h] = Fseg;
    const int64_t slot = seg_slot(a, n, seg, h);
#pragma unroll
    for (int jj = 0; jj < NSB; ++jj) {
      if (!sval[jj]) continue;
      *(f32x4*)((float*)A.tiles_a + slot + goff[jj]) = accM[jj];
      *(f32x4*)(A.tiles_b + slot + goff[jj]) = accJ[jj];
    }
    return;
  }
  if (A.fin_a) {
#pragma unroll
    for (int jj = 0; jj < NSB; ++jj) {
      if (!sval[jj]) continue;
      const int64_t off = (int64_t)nh * E + goff[jj];
      if (HAS_J) {
        f32x4 mu, I;
#pragma unroll
        for (int r = 0; r < 4; ++r) { I[r] = accJ[jj][r] + Ip; mu[r] = accM[jj][r] * fast_rcp(I[r]); }
        *(f32x4*)(A.fin_a + off) = mu;
        *(f32x4*)(A.fin_b + off) = I;
      } else {
        *(f32x4*)(A.fin_a + off) = accM[jj] * A.fin_scale;
      }
    }
  }
}

// The segments' totals become the states before them, and the last one the final state.  Four entries per thread.
__global__ __launch_bounds__(256) void chunk_segments_kernel(ChunkArgs a) {
  const int64_t E = (int64_t)a.dv * a.dk;
  const int nblk = (int)((E + 1023) / 1024), nh = blockIdx.x / nblk, n = nh / a.H, h = nh - n * a.H;
  const int64_t e = ((int64_t)(blockIdx.x % nblk) * 256 + threadIdx.x) * 4;
  if (e >= E) return;
  f32x4 M = {0.f, 0.f, 0.f, 0.f}, J = M;
  for (int s = 0; s < a.segs; ++s) {
    const int64_t slot = seg_slot(a, n, s, h) + e;
    const SegDecay F = seg_decays(a, n, s)[a.seg_tiles / a.every * a.H + h];
    const f32x4 m = *(const f32x4*)(a.chunk_mu + slot), j = *(const f32x4*)(a.chunk_I + slot);
    *(f32x4*)(a.chunk_mu + slot) = M;
    *(f32x4*)(a.chunk_I + slot) = J;
#pragma unroll
    for (int r = 0; r < 4; ++r) { M[r] = F.apply(M[r], m[r]); J[r] = F.apply(J[r], j[r]); }
  }
  if (a.final_mu) {
    const float Ip = a.Ip[h];
    f32x4 mu, I;
#pragma unroll
    for (int r = 0; r < 4; ++r) { I[r] = J[r] + Ip; mu[r] = M[r] * fast_rcp(I[r]); }
    *(f32x4*)(a.final_mu + nh * E + e) = mu;
    *(f32x4*)(a.final_I + nh * E + e) = I;
  }
}

template <bool HAS_J, int NIK, int DSB>
static int launch_state_pass_t(const StatePassArgs& A, int kern_id, unsigned grid, size_t lds, hipStream_t s) {
  if (int rc = allow_lds((const void*)&chunk_states_kernel<HAS_J, NIK, DSB>, lds)) return rc;
  PAL_TIMED_LAUNCH(kern_id, s, (chunk_states_kernel<HAS_J, NIK, DSB>), dim3(grid), dim3(768), lds, s, A);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}

template <bool HAS_J, int DSB>
static int launch_state_pass_d(const StatePassArgs& A, int kern_id, unsigned grid, size_t lds, hipStream_t s) {
  const int nik = (A.dks + 31) / 32;
  if (nik <= 2) return launch_state_pass_t<HAS_J, 2, DSB>(A, kern_id, grid, lds, s);
  if (nik == 3) return launch_state_pass_t<HAS_J, 3, DSB>(A, kern_id, grid, lds, s);
  if constexpr (DSB <= 3) {
    if (nik == 4) return launch_state_pass_t<HAS_J, 4, DSB>(A, kern_id, grid, lds, s);
  }
  if constexpr (DSB <= 2) {
    if (nik <= 6) return launch_state_pass_t<HAS_J, 6, DSB>(A, kern_id, grid, lds, s);
  }
  if constexpr (DSB == 1) return launch_state_pass_t<HAS_J, 8, DSB>(A, kern_id, grid, lds, s);
  return PAL_E_HEADDIM;   // (launch_state_pass keeps ds dks within the state waves' blocks)
}
template <bool HAS_J>
static int launch_state_pass_j(const StatePassArgs& A, int kern_id, unsigned grid, size_t lds, hipStream_t s) {
  switch (A.ds) {
    case 16: return launch_state_pass_d<HAS_J, 1>(A, kern_id, grid, lds, s);
    case 32: return launch_state_pass_d<HAS_J, 2>(A, kern_id, grid, lds, s);
    case 48: return launch_state_pass_d<HAS_J, 3>(A, kern_id, grid, lds, s);
    case 64: return launch_state_pass_d<HAS_J, 4>(A, kern_id, grid, lds, s);
    default: return PAL_E_HEADDIM;
  }
}

// key columns per workgroup of the one-pass form, see launch_state_pass
static int state_pass_key_slice(const ChunkArgs& a, int ds) {
  if (ds == 16 && a.dk % 128 == 0 && (int64_t)a.n_seqs * a.H * (a.dv / 16) < 192) return 64;
  return a.dk;
}

// Segments for a pass that keeps every fourth tile's state (the windows of one long sequence, see out_tiles_per_state).  The walk
// over the tiles is a chain of 0.7 us a tile, and 16 heads of 128x128 filled the compute units only in slices of 16 rows by 64
// columns, each of which stages rows for little state.  As segments walked side by side, in slices as wide as the registers
// hold, states that are kept since the start of the segment: the smallest number that gives three quarters of the units a workgroup.
// 65536 tokens of 16 heads of 128x128, four windows: states 731 -> 415 us (1.34 GB at 3.2 TB/s), and 20 us of output kernel for the state
// before the segment.  (Eight tiles to a kept state then: 360 us, and 100 more in the output kernel.)
void state_pass_segments(ChunkArgs& a) {
  if (a.every < 4 || a.cu_seqlens || (a.flags & PAL_FLAG_VARLEN)) return;
  const int64_t tiles = (a.T + kC - 1) / kC;
  int ds = 16;
  for (int c : {64, 48, 32})
    if (a.dv % c == 0 && c * a.dk <= 256 * 4 * kStMaxBlocks) { ds = c; break; }
  const int64_t per = (int64_t)a.n_seqs * a.H * (a.dv / ds);
  int segs = 1;
  while (segs < 16 && per * segs < 192) segs *= 2;
  const int64_t seg_tiles = (tiles + (int64_t)segs * a.every - 1) / ((int64_t)segs * a.every) * a.every;
  // (a segment needs the slots of four tiles for itself, and enough of them to be worth its own start; its decays, two numbers per
  // kept tile and head and two more, have the last two of these: sequences so long for the size of their states are walked whole)
  if (segs < 2 || seg_tiles < 16 || tiles - (segs - 1) * seg_tiles < a.every) return;
  if (2 * (seg_tiles / a.every + 1) > 2 * (int64_t)a.dv * a.dk) return;
  a.segs = segs;
  a.seg_tiles = (int32_t)seg_tiles;
}

// Whether the one-pass form serves this call: bf16 rows, and enough (sequence, head, slice) workgroups that
// the serial walk over the tiles does not leave most of the GPU idle.
bool state_pass_applies(const ChunkArgs& a, int dtype, bool has_j) {
  if (dtype != PAL_DTYPE_BF16 || (a.flags & PAL_FLAG_STATES_TWO_KERNELS)) return false;
  if (a.dk < 16 || a.dk > 256 || a.dk % 16 || a.dv % 16) return false;
  // rows are addressed with 32-bit byte offsets from the first row of a sequence
  if ((int64_t)a.T * a.H * (a.dk > a.dv ? a.dk : a.dv) * 2 >= 0x7fffffffLL) return false;
  if (a.flags & PAL_FLAG_STATES_ONE_PASS) return true;
  // The walk over the tiles is serial per workgroup (0.4-0.7 us per tile): with fewer workgroups than this the
  // two-kernel form, which spreads the tiles over the whole GPU, is faster.
  return (int64_t)a.n_seqs * a.H * (a.dv / 16) * (a.dk / state_pass_key_slice(a, 16)) >= 192;
}

// tiles_a / tiles_b, init_*, fin_*: see StatePassArgs.  reverse walks every sequence from its last tile.
int launch_state_pass(const ChunkArgs& a, bool has_j, void* tiles_a, float* tiles_b, const float* init_a,
                      const float* init_b, float* fin_a, float* fin_b, bool reverse, float fin_scale, int kern_id,
                      hipStream_t s) {
  StatePassArgs A;
  A.c = a;
  A.tiles_a = tiles_a; A.tiles_b = tiles_b;
  A.init_a = init_a; A.init_b = init_b; A.fin_a = fin_a; A.fin_b = fin_b;
  A.reverse = reverse ? 1 : 0;
  A.fin_scale = fin_scale;
  // value rows per workgroup: the largest slice that still gives three quarters of the compute units a
  // workgroup (measured: wider slices stage the key rows for more state at the same cost per tile; with
  // fewer workgroups than that the idle units cost more)
  int ds = 16;
  const int cand[3] = {64, 48, 32};
  for (int c : cand) {
    if (a.dv % c || c * a.dk > 256 * 4 * kStMaxBlocks) continue;
    if ((int64_t)a.n_seqs * a.segs * a.H * (a.dv / c) >= 192) { ds = c; break; }
  }
  // key columns per workgroup: all of them, unless even slices of 16 value rows leave the GPU short of workgroups and
  // the key columns can be halved into slices of 64 (measured at one sequence of 16 heads, 128x128: 128 workgroups
  // 102 us per 64 tiles, 256 workgroups of 16 x 64 entries 72 us, the two-kernel form 96 us; slices of 32 columns or
  // 32 x 32 entries are slower again, and with enough workgroups splitting the columns gains nothing)
  const int dks = a.segs > 1 ? a.dk : state_pass_key_slice(a, ds);
  if (ds * dks > 256 * 4 * kStMaxBlocks) return PAL_E_HEADDIM;
  A.ds = ds;
  A.dks = dks;
  A.ksplit = a.dk / dks;
  if ((int64_t)a.n_seqs * a.H <= 0) return PAL_OK;
  ChunkArgs walks = a;
  walks.n_seqs *= a.segs;
  if (!walk_plan(walks, a.dv / ds * A.ksplit, A.plan)) return PAL_E_DIM;
  const size_t lds = sizeof(float) * (3 * kC + 4) +
                     sizeof(bf16_t) * 2 * kC * (size_t)(staged_stride(dks) + staged_stride(ds) * (has_j ? 2 : 1));
  if (lds > kMaxLds) return PAL_E_HEADDIM;
  const unsigned grid = (unsigned)A.plan.per_xcd * 8;
  if (int rc = has_j ? launch_state_pass_j<true>(A, kern_id, grid, lds, s) : launch_state_pass_j<false>(A, kern_id, grid, lds, s)) return rc;
  if (a.segs > 1) {
    const int64_t blocks = (int64_t)a.n_seqs * a.H * (((int64_t)a.dv * a.dk + 1023) / 1024);
    if (blocks > 0x7fffffff) return PAL_E_DIM;
    PAL_TIMED_LAUNCH(kern_id, s, chunk_segments_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
    PAL_HIP_LAUNCH_CHECK();
  }
  return PAL_OK;
}

}  // namespace pal

extern "C" int pal_state_pass_applies(const PalDims* d, int has_precision_state) {
  if (pal_validate_dims(d) != PAL_OK) return 0;
  pal::ChunkArgs a = {};
  a.T = d->seq_len; a.H = d->n_heads; a.dk = d->dk; a.dv = d->dv; a.n_seqs = d->n_seqs;
  a.Hq = d->n_qk_heads > 0 ? d->n_qk_heads : d->n_heads;
  a.flags = d->flags;
  return pal::state_pass_applies(a, d->dtype, has_precision_state != 0) ? 1 : 0;
}
