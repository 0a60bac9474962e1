// Scalar-gated linear attention (gla.hip) as one walk over a sequence per result.
//
// Forward output and the three input gradients have one form (see gla_tile_kernel in gla.hip, whose roles these are):
//   out[x, e] = scale (w_x sum_c S[e, c] X[x, c] + sum_y (X_x . Y_y) L(x, y) Z[y, e]) ,   S <- F S + sum_y a_y Z_y Y_y^T
// over tiles of 64 tokens, from the start of the sequence (o: X = q, Y = k, Z = v; dq: dO, v, k, S transposed) or from its end
// (dv: k, q, dO; dk: v, dO, q, transposed), S in fp32.  With the tiles' states in memory this takes a pass that writes them
// and a kernel that reads them per result, 37 KB a tile and head at 96x192: 1.3 GB of a training step's 2 GB.  Here S never leaves
// the registers of the wave that uses it, the rows are read once per result, and dq needs no states kept from the forward.
// B=8 T=2048 H=16 96x192, forward and backward: 813 -> 365 us, 1.3 GB at 3.6 TB/s.  Errors against float64 are those of the
// kernels with tile states to three digits for o, dq, dk and dv, and to the scatter of a badly conditioned sum for the gate's
// gradient (96x192, 32 seeds: 1.11e-2 both; 96x96 1.04e-2 / 8.8e-3, 128x128 8.6e-3 / 9.2e-3).
//
// One workgroup per (sequence, head, slice of 16 NE columns e).  A wave holds S for 16 of the columns and all c, as the
// accumulators of 16x16 products with row c and column e: two of them, rounded, are the operand of the state term, so S takes
// no way through LDS.  From 128 columns c on, two waves share the 16 columns, half of c each (the registers of one wave
// would hold 64 columns' worth of S, a single workgroup to a compute unit): their outputs meet in LDS.  The scores are formed
// once by all waves and pass through LDS; Z and Y enter the other products transposed, by the transposing reads of gfx950, so
// every tile is staged as it is in memory.  The rows of the next tile are in flight, in registers, while a tile is worked.
//
// What bounds it: 128 heads, the memory (3.3 to 3.8 TB/s); fewer, the chain of a tile (2.1 to 2.9 us: three barriers, LDS
// latency, matrix instructions one after the other).  So the operands of a step are read while the step before is multiplied
// (the compiler left to itself waits for each read: 512 -> 446 us at the shape above), and dq and dk are one launch, one
// from each end, where each alone would leave half the compute units idle (266 -> 186 us).
#include "gla_walk.h"
#include "pal_host.h"
#include "pal_profile.h"

namespace pal {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// parts that the contraction over dc is cut into, a wave each per block of 16 output columns
constexpr int walk_parts(int KS) { return KS >= 4 ? 2 : 1; }

// waves per SIMD that the registers are cut for: two workgroups on a compute unit, where they have at most six waves
constexpr int walk_waves_per_simd(int NW) { return NW <= 4 ? 2 : NW <= 6 ? 3 : 2; }

template <int KS, int NE>
struct WalkShape {
  static constexpr int CS = walk_parts(KS), KSW = KS / CS, NW = NE * CS;
  static constexpr int NT = 64 * NW, DCP = 32 * KS, ES = 16 * NE;
  static constexpr int XS = DCP + 16;            // row strides (bf16) of the tiles: an odd number of 32-byte pieces
  static constexpr int ZS = 16 * (NE | 1);
  static constexpr int OS = ES + 8, PS = ES + 4; // row strides of the output tile (bf16) and of its second part (fp32)
  static constexpr size_t lds = sizeof(float) * (3 * kC + 4 + NW * kC) + 16 * 6 * 64 + sizeof(bf16_t) * kC * (2 * XS + ZS) +
                                (CS == 1 ? sizeof(bf16_t) * kC * OS : sizeof(float) * kC * PS);
  static_assert(lds <= kMaxLds, "LDS of a compute unit");
};

template <int KS, int NE, bool REVERSE>
__device__ __forceinline__ void gla_walk(const GlaWalkArgs& A, const GlaWalkRole& R, int n, int h, int sl) {
  typedef WalkShape<KS, NE> Sh;
  constexpr int CS = Sh::CS, KSW = Sh::KSW, NW = Sh::NW, NT = Sh::NT, DCP = Sh::DCP, ES = Sh::ES;
  constexpr int XS = Sh::XS, ZS = Sh::ZS, OS = Sh::OS, PS = Sh::PS;
  constexpr int XI = (4 * KS + NW - 1) / NW, ZI = (2 + CS - 1) / CS;   // 16-byte pieces per thread of X (and Y), of Z
  constexpr int SB = (10 + NW - 1) / NW;  // score blocks per wave
  extern __shared__ float smem[];
  const ChunkArgs& a = A.c;
  float* sC = smem;                       // [64] running log2 decay inside the tile
  float* sA = sC + kC;                    // [64] weight of a token in the state after the tile
  float* sW = sA + kC;                    // [64] weight of the state before the tile in a token's output
  float* sF = sW + kC;                    // decay over the tile (+ 3 pad)
  float* sDot = sF + 4;                   // [NW][64]
  bf16x8* sP = (bf16x8*)(sDot + NW * kC); // [6][64 lanes] scores
  bf16_t* sX = (bf16_t*)(sP + 6 * 64);
  bf16_t* sY = sX + kC * XS;
  bf16_t* sZ = sY + kC * XS;
  bf16_t* sOut = sZ + kC * ZS;            // one part: [64][OS] output rows
  float* sPart = (float*)sOut;            // two: [64][PS] the second part's share
  const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int eb = w % NE, part = w / NE, ks0 = part * KSW;   // the wave's columns, and its steps of 32 of the contraction
  const int H = a.H, dc = A.dc, de = A.de;
  // score operand of token block xb and blocks y 2 q, 2 q + 1 (the six on the causal side)
  auto p_at = [](int xb, int q) { return REVERSE ? (xb < 2 ? 2 * xb + q : 2 + xb) : (xb < 2 ? xb : 2 * xb - 2 + q); };
  int bos, len;
  if (a.cu_seqlens) {
    packed_seq_bounds(a.cu_seqlens, n, a.T, bos, len);
  } else {
    bos = n * a.T;
    len = a.T;
  }
  const int nchunks = (len + kC - 1) / kC;
  const int e0 = sl * ES;
  const int hx = h / (H / A.hX), hz = h / (H / A.hZ);

  // pieces of this thread: byte offset from the first row of a tile (out of range: reads as zero) and place in the tile
  uint32_t xoff[XI], zoff[ZI], woff[4];
  int xdst[XI], zdst[ZI];
#pragma unroll
  for (int j = 0; j < XI; ++j) {
    const int per = dc >> 3, idx = tid + NT * j, s = idx / per, c8 = idx - s * per;
    const bool on = s < kC;
    xoff[j] = on ? (uint32_t)((s * A.hX * dc + 8 * c8) * 2) : 0x80000000u;
    xdst[j] = on ? s * XS + 8 * c8 : (tid & (kC - 1)) * XS + DCP;   // (a row's padding, which nothing reads)
  }
#pragma unroll
  for (int j = 0; j < ZI; ++j) {
    const int idx = tid + NT * j, s = idx / (ES / 8), c8 = idx - s * (ES / 8);
    zoff[j] = e0 + 8 * c8 < de ? (uint32_t)((s * A.hZ * de + e0 + 8 * c8) * 2) : 0x80000000u;
    zdst[j] = s * ZS + 8 * c8;
  }
  const bool wave_on = e0 + 16 * eb < de;   // (the last slice may have fewer columns than waves)
#pragma unroll
  for (int xb = 0; xb < 4; ++xb)
    woff[xb] = wave_on ? (uint32_t)(((16 * xb + i) * A.hZ * de + e0 + 16 * eb + 4 * g) * 2) : 0x80000000u;
  const uint32_t xbytes = len > 0 ? (uint32_t)(((len - 1) * A.hX * dc + dc) * 2) : 0u;
  const uint32_t zbytes = len > 0 ? (uint32_t)(((len - 1) * A.hZ * de + de) * 2) : 0u;
  const int esz = a.gate_bf16 ? 2 : 4;
  const uint32_t gbytes = len > 0 ? (uint32_t)(((len - 1) * H + 1) * esz) : 0u;
  const int64_t xrow = ((int64_t)bos * A.hX + hx) * dc, zrow = ((int64_t)bos * A.hZ + hz) * de;
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc((void*)(R.X + xrow), 0, xbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t yrs = __builtin_amdgcn_make_buffer_rsrc((void*)(R.Y + xrow), 0, xbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t zrs = __builtin_amdgcn_make_buffer_rsrc((void*)(R.Z + zrow), 0, zbytes, 0x00020000);
  const bool has_dot = R.W != nullptr;
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc((void*)(has_dot ? R.W + zrow : R.Z + zrow), 0, zbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t grs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)a.gt + ((int64_t)bos * H + h) * esz), 0, gbytes, 0x00020000);
  const uint32_t goff = (uint32_t)(lane * H * esz);
  const float gh = a.g[h] * kLog2e;

  u32x4 RX[XI], RY[XI], RZ[ZI];
  uint32_t Rg = 0;
  auto request = [&](int p) {
    const int c = REVERSE ? nchunks - 1 - p : p;
    const bool live = p < nchunks;
    const uint32_t tx = live ? (uint32_t)(c * kC * A.hX * dc * 2) : 0x80000000u;
    const uint32_t tz = live ? (uint32_t)(c * kC * A.hZ * de * 2) : 0x80000000u;
    if (w == NW - 1) {
      const uint32_t tg = live ? (uint32_t)(c * kC * H * esz) : 0x80000000u;
      Rg = a.gate_bf16 ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(grs, goff + tg, 0, 0)
                       : __builtin_amdgcn_raw_buffer_load_b32(grs, goff + tg, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < XI; ++j) {
      RX[j] = __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[j] + tx, 0, 0);
      RY[j] = __builtin_amdgcn_raw_buffer_load_b128(yrs, xoff[j] + tx, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < ZI; ++j) RZ[j] = __builtin_amdgcn_raw_buffer_load_b128(zrs, zoff[j] + tz, 0, 0);
  };

  // The state: column e = e0 + 16 eb + i per lane, entry r of block 2 p + u is c = 32 (ks0 + p) + 8 g + 4 (u ^ (g / 2)) + r.
  // Blocks 2 p and 2 p + 1, rounded, are an operand whose contraction index is c = 32 (ks0 + p) + 8 g + j, that of a 16-byte
  // read of X (the exchange for g >= 2 spreads the transposing reads of Y over all banks).
  const bool swap = g >= 2;
  f32x4 S[2 * KSW];
  const int e = e0 + 16 * eb + i;
  const int64_t so = ((int64_t)n * H + h) * dc * de;
#pragma unroll
  for (int b = 0; b < 2 * KSW; ++b) {
    const int cc = 32 * (ks0 + (b >> 1)) + 8 * g + 4 * ((b & 1) ^ (g >> 1));
    S[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (R.init && wave_on && cc < dc) {
      if (R.init_t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[b][r] = R.init[so + (int64_t)(cc + r) * de + e];
      } else {
        S[b] = *(const f32x4*)(R.init + so + (int64_t)e * dc + cc);
      }
    }
  }
  request(0);
  // columns beyond dc and the halves of score operands that no block fills stay zero
  if (dc != DCP) {
    for (int idx = tid; idx < 2 * kC * XS / 8; idx += NT) *(u32x4*)&sX[8 * idx] = u32x4{0, 0, 0, 0};
  }
  for (int idx = tid; idx < 6 * 64; idx += NT) *(u32x4*)&sP[idx] = u32x4{0, 0, 0, 0};
  if (dc != DCP) __syncthreads();

  bf16_t* out = R.out + ((int64_t)bos * H + h) * de + e0;
  // a lane's places in the tiles (every access of the walk is one of them plus a constant, or plus a block of 16 rows)
  const bf16_t* pX = sX + i * XS + 8 * g;                                    // rows i, pieces of 8
  const bf16_t* pY = sY + i * XS + 8 * g;
  const bf16_t* pYt0 = sY + (4 * g + (i >> 2)) * XS + 32 * ks0 + 8 * (i & 3) + 4 * ((i >> 1) & 1);   // transposed, state block 2 p
  const bf16_t* pYt1 = sY + (4 * g + (i >> 2)) * XS + 32 * ks0 + 8 * (i & 3) + 4 - 4 * ((i >> 1) & 1);   // and 2 p + 1
  const bf16_t* pZt = sZ + (4 * g + (i >> 2)) * ZS + 16 * eb + 4 * (i & 3);
  bf16x8* pP = sP + lane;
  for (int p = 0; p < nchunks; ++p) {
    const int c = REVERSE ? nchunks - 1 - p : p;
    // ---- the requested tile goes to LDS (every read of the one before is behind a barrier)
    if (w == NW - 1) {
      const float gt = __builtin_bit_cast(float, a.gate_bf16 ? Rg << 16 : Rg);   // zero beyond the sequence
      const float cs = wave_inclusive_scan(-gt * gh, lane);
      const float tot = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cs), 63));
      sC[lane] = cs;
      const float from = fast_exp2(cs), to = fast_exp2(tot - cs);
      sA[lane] = REVERSE ? from : to;
      sW[lane] = REVERSE ? to : from;
      if (lane == 0) sF[0] = fast_exp2(tot);
    }
#pragma unroll
    for (int j = 0; j < XI; ++j) {
      *(u32x4*)&sX[xdst[j]] = RX[j];
      *(u32x4*)&sY[xdst[j]] = RY[j];
    }
#pragma unroll
    for (int j = 0; j < ZI; ++j) *(u32x4*)&sZ[zdst[j]] = RZ[j];
    __syncthreads();
    u32x2 RW[4];
    if (has_dot) {
      const uint32_t tw = (uint32_t)(c * kC * A.hZ * de * 2);
#pragma unroll
      for (int xb = 0; xb < 4; ++xb) RW[xb] = __builtin_amdgcn_raw_buffer_load_b64(wrs, woff[xb] + tw, 0, 0);
    }
    request(p + 1);

    // ---- scores: the ten blocks (token x, token y) on the causal side, dealt out to the waves (past the tenth: it again,
    //      not stored; a branch around single products would make each wait for its own reads)
    {
      f32x4 acc[SB];
      int xb[SB], yb[SB];
#pragma unroll
      for (int q = 0; q < SB; ++q) {
        const int b = min(w + NW * q, 9), t = b >= 6 ? 3 : b >= 3 ? 2 : b >= 1 ? 1 : 0, u = b - t * (t + 1) / 2;
        xb[q] = REVERSE ? 3 - t : t;
        yb[q] = REVERSE ? 3 - u : u;
        acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      bf16x8 fx[2][SB], fy[2][SB];
      auto operands = [&](int ks) {
#pragma unroll
        for (int q = 0; q < SB; ++q) {
          fy[ks & 1][q] = *(const bf16x8*)&pY[yb[q] * (16 * XS) + 32 * ks];
          fx[ks & 1][q] = *(const bf16x8*)&pX[xb[q] * (16 * XS) + 32 * ks];
        }
      };
      operands(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 1 < KS) operands(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < SB; ++q) acc[q] = mfma16(fy[ks & 1][q], fx[ks & 1][q], acc[q]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int q = 0; q < SB; ++q) {
        if (w + NW * q < 10) {
          const float cx = sC[16 * xb[q] + i];
          const f32x4 cy = *(const f32x4*)&sC[16 * yb[q] + 4 * g];
          float val[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const bool live = yb[q] != xb[q] || (REVERSE ? 4 * g + r >= i : 4 * g + r <= i);
            val[r] = live ? acc[q][r] * fast_exp2(REVERSE ? cy[r] - cx : cx - cy[r]) : 0.f;
          }
          store_vec<4>((bf16_t*)&pP[p_at(xb[q], yb[q] >> 1) * 64] + 4 * (yb[q] & 1), val);
        }
      }
    }
    __syncthreads();

    // ---- outputs of the wave's 16 columns, then the state after the tile
    f32x4 acc[4];
    {
#pragma unroll
      for (int xb = 0; xb < 4; ++xb) acc[xb] = f32x4{0.f, 0.f, 0.f, 0.f};
      bf16x8 fx[2][4], Za[2], P[2][2];
      const bf16_t* pX0 = pX + 32 * ks0;
      float wx[4];
      auto operands = [&](int ks) {
#pragma unroll
        for (int xb = 0; xb < 4; ++xb) fx[ks & 1][xb] = *(const bf16x8*)&pX0[xb * (16 * XS) + 32 * ks];
      };
      auto p_on = [](int xb, int q) { return REVERSE ? 2 * q + 1 >= xb : 2 * q <= xb; };
      auto scores = [&](int xb) {   // one part: both operands of a token block where they exist; two: the part's own
        if constexpr (CS == 1) {
#pragma unroll
          for (int q = 0; q < 2; ++q)
            if (p_on(xb, q)) P[xb & 1][q] = pP[p_at(xb, q) * 64];
        } else {
          P[xb & 1][0] = pP[p_at(xb, part) * 64];
        }
      };
      operands(0);
#pragma unroll
      for (int ks = 0; ks < KSW; ++ks) {
        if (ks + 1 < KSW) {
          operands(ks + 1);
        } else {
          // Z transposed: row = the wave's column i, contraction index (g, j) -> token 32 p + 16 (j / 4) + 4 g + j % 4
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            Za[q] = join(lds_read_tr(pZt + 32 * q * ZS), lds_read_tr(pZt + (32 * q + 16) * ZS));
          }
#pragma unroll
          for (int xb = 0; xb < 4; ++xb) wx[xb] = sW[16 * xb + i];
          scores(0);
        }
        const bf16x2 s0 = pack2(S[2 * ks][0], S[2 * ks][1]), s1 = pack2(S[2 * ks][2], S[2 * ks][3]);
        const bf16x2 s2 = pack2(S[2 * ks + 1][0], S[2 * ks + 1][1]), s3 = pack2(S[2 * ks + 1][2], S[2 * ks + 1][3]);
        const bf16x2 t0 = swap ? s2 : s0, t1 = swap ? s3 : s1, t2 = swap ? s0 : s2, t3 = swap ? s1 : s3;
        const bf16x8 Sa = {t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int xb = 0; xb < 4; ++xb) acc[xb] = mfma16(Sa, fx[ks & 1][xb], acc[xb]);
        __builtin_amdgcn_sched_barrier(0);
      }
      float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int xb = 0; xb < 4; ++xb) {
        if (xb < 3) scores(xb + 1);
        __builtin_amdgcn_sched_barrier(0);
        acc[xb] *= wx[xb];
        if constexpr (CS == 1) {
#pragma unroll
          for (int q = 0; q < 2; ++q)
            if (p_on(xb, q)) acc[xb] = mfma16(Za[q], P[xb & 1][q], acc[xb]);
        } else {
          const u32x4 x = __builtin_bit_cast(u32x4, P[xb & 1][0]), none = {0, 0, 0, 0};
          const bool both = xb >= 2 != REVERSE;   // (token blocks with two operands; the others have the first or the second)
          acc[xb] = mfma16(part ? Za[1] : Za[0], __builtin_bit_cast(bf16x8, both || (part == 1) == REVERSE ? x : none), acc[xb]);
        }
        acc[xb] *= a.scale;
        if (has_dot) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const uint32_t word = RW[xb][r >> 1];
            dot[xb] = fmaf(__builtin_bit_cast(float, (r & 1) ? word & 0xffff0000u : word << 16), acc[xb][r], dot[xb]);
          }
        }
        if constexpr (CS == 1) store_vec<4>(sOut + (16 * xb + i) * OS + 16 * eb + 4 * g, (const float*)&acc[xb]);
        else if (part == 1) *(f32x4*)&sPart[(16 * xb + i) * PS + 16 * eb + 4 * g] = acc[xb];
      }
      if (has_dot) sDot[w * kC + lane] = rows4_sum_x4(dot[0], dot[1], dot[2], dot[3]);   // lane = token
      __builtin_amdgcn_sched_barrier(0);
      // Y transposed: row i of the operand of a state block is the c of entry i % 4 in the lanes g = i / 4
      bf16x8 fy[2][2][2];
      auto operands_t = [&](int ks) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const bf16_t* y = (u ? pYt1 : pYt0) + 32 * ks;
            fy[ks & 1][u][q] = join(lds_read_tr(y + 32 * q * XS), lds_read_tr(y + (32 * q + 16) * XS));
          }
      };
      bf16x8 Zw[2];
      const float F = sF[0];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f32x4 w0 = *(const f32x4*)&sA[32 * q + 4 * g], w1 = *(const f32x4*)&sA[32 * q + 16 + 4 * g];
        if (q == 1) operands_t(0);
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = (j < 4 ? w0[j & 3] : w1[j & 3]) * (float)Za[q][j];
        const bf16x2 z0 = pack2(x[0], x[1]), z1 = pack2(x[2], x[3]), z2 = pack2(x[4], x[5]), z3 = pack2(x[6], x[7]);
        Zw[q] = bf16x8{z0[0], z0[1], z1[0], z1[1], z2[0], z2[1], z3[0], z3[1]};
      }
#pragma unroll
      for (int ks = 0; ks < KSW; ++ks) {
        if (ks + 1 < KSW) operands_t(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          S[2 * ks + u] *= F;
#pragma unroll
          for (int q = 0; q < 2; ++q) S[2 * ks + u] = mfma16(fy[ks & 1][u][q], Zw[q], S[2 * ks + u]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __syncthreads();
    const int clen = min(kC, len - c * kC);
    bf16_t* orow = out + (int64_t)c * kC * H * de;
    if constexpr (CS == 1) {   // rows out in 16-byte pieces
#pragma unroll
      for (int j = 0; j < ZI; ++j) {
        const int idx = tid + NT * j, s = idx / (ES / 8), c8 = idx - s * (ES / 8);
        if (s < clen && e0 + 8 * c8 < de) *(u32x4*)(orow + (int64_t)s * H * de + 8 * c8) = *(const u32x4*)&sOut[s * OS + 8 * c8];
      }
    } else if (part == 0 && wave_on) {
#pragma unroll
      for (int xb = 0; xb < 4; ++xb) {
        const f32x4 x = acc[xb] + *(const f32x4*)&sPart[(16 * xb + i) * PS + 16 * eb + 4 * g];
        if (16 * xb + i < clen) store_vec<4>(orow + (int64_t)(16 * xb + i) * H * de + 16 * eb + 4 * g, (const float*)&x);
      }
    }
    if (has_dot && w == 0 && lane < clen) {
      float tot = 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) tot += sDot[x * kC + lane];
      R.dot[((int64_t)sl * H + h) * A.n_tokens + bos + c * kC + lane] = tot;
    }
  }
  if (R.fin && wave_on) {
#pragma unroll
    for (int b = 0; b < 2 * KSW; ++b) {
      const int cc = 32 * (ks0 + (b >> 1)) + 8 * g + 4 * ((b & 1) ^ (g >> 1));
      if (cc < dc) *(f32x4*)(R.fin + so + (int64_t)e * dc + cc) = S[b] * R.fin_scale;
    }
  }
}

template <int KS, int NE>
__global__ __launch_bounds__((WalkShape<KS, NE>::NT), (walk_waves_per_simd(WalkShape<KS, NE>::NW)))
void gla_walk_kernel(GlaWalkArgs A) {
  int n, h, u;
  if (!walk_item(A.c, A.plan, threadIdx.x & 63, n, h, u)) return;
  const int r = u / A.n_sl;
  if (A.role[r].reverse) gla_walk<KS, NE, true>(A, A.role[r], n, h, u - r * A.n_sl);
  else gla_walk<KS, NE, false>(A, A.role[r], n, h, u - r * A.n_sl);
}

// Blocks of 16 output columns per workgroup, four or six.  Six share the rows and scores of a tile among more columns, but leave
// fewer workgroups: taken where four would give the GPU more than a workgroup per compute unit and the columns divide (four / six,
// us a walk, B=8 T=2048 H=16: 96x192 forward 104 / 86, dq and dk 246 / 179; with 64 heads in all 76 / 77 and 123 / 150; all
// walks of a step: 96x96 299 / 283, 192x96 450 / 428, 192x192 796 / 604, 160x192 807 / 668, 80x96 of 16 sequences 486 / 440, 96x96 of
// 32 x 512 253 / 227).  Up to 64 columns of contraction, where staging is cheap, four is never behind (48x96 with 384 heads
// 34 / 42); 97 to 128 and more than 192 columns have no instance with six.
static int walk_blocks(const PalDims* d, int dc, int de, int n_roles) {
  const int ks = (dc + 31) / 32;
  const bool six = de % 96 == 0 && (ks == 3 || ks == 5 || ks == 6) &&
                   (int64_t)d->n_seqs * d->n_heads * n_roles * ((de + 63) / 64) > 256;
  return six ? 6 : 4;
}
int gla_walk_slices(const PalDims* d, int dc, int de, int n_roles) {
  const int es = 16 * walk_blocks(d, dc, de, n_roles);
  return (de + es - 1) / es;
}

template <int KS, int NE>
static int launch_walk_t(const GlaWalkArgs& A, int kern_id, hipStream_t s) {
  typedef WalkShape<KS, NE> Sh;
  if (int rc = allow_lds((const void*)&gla_walk_kernel<KS, NE>, Sh::lds)) return rc;
  PAL_TIMED_LAUNCH(kern_id, s, (gla_walk_kernel<KS, NE>), dim3((unsigned)A.plan.per_xcd * 8), dim3(Sh::NT), Sh::lds, s, A);
  PAL_HIP_LAUNCH_CHECK();
  return PAL_OK;
}
int launch_gla_walk(GlaWalkArgs A, const PalDims* d, int kern_id, hipStream_t s) {
  const int ne = walk_blocks(d, A.dc, A.de, A.n_roles);
  A.n_sl = gla_walk_slices(d, A.dc, A.de, A.n_roles);
  if (!walk_plan(A.c, A.n_sl * A.n_roles, A.plan)) return PAL_E_DIM;
  switch ((A.dc + 31) / 32) {
    case 1: return launch_walk_t<1, 4>(A, kern_id, s);
    case 2: return launch_walk_t<2, 4>(A, kern_id, s);
    case 3: return ne == 6 ? launch_walk_t<3, 6>(A, kern_id, s) : launch_walk_t<3, 4>(A, kern_id, s);
    case 4: return launch_walk_t<4, 4>(A, kern_id, s);
    case 5: case 6: return ne == 6 ? launch_walk_t<6, 6>(A, kern_id, s) : launch_walk_t<6, 4>(A, kern_id, s);
    case 7: case 8: return launch_walk_t<8, 4>(A, kern_id, s);
    default: return PAL_E_HEADDIM;
  }
}

bool gla_walk_possible(const PalDims* d) {
  // rows and gates are addressed with 32-bit byte offsets from the first row of a sequence
  return d->dtype == PAL_DTYPE_BF16 && (int64_t)d->seq_len * d->n_heads * (d->dk > d->dv ? d->dk : d->dv) * 2 < 0x7fffffffLL;
}
// A walk takes as long as its longest sequence, 8 us a tile in forward and backward together, however few there are; the
// kernels with the tiles' states in memory take 0.55 ns a tile and head for every column of dk + dv.  The line is where the two
// meet: heads that are walked at a time, times columns.  Tiles / walks, us of kernels, T=2048 (96x192: 225 / 282 with 32 heads
// in all, 408 / 285 with 64, 827 / 365 with 128; 96x96: 261 / 258 with 64, 493 / 287 with 128; 48x96: 197 / 236, 340 / 242).
// Up to 64x64 one kernel forms the three gradients and walks are faster from 192 heads on only (194 / 224 with 128, T=512 149 / 111
// with 384): not taken.  The line would lie in the middle of ordinary batch sizes, and a large batch of such heads agrees with its
// sequences in small ones to 1e-6, which walks, whose states are rounded at other places, would end; wider heads do pay that.
bool gla_walk_applies(const PalDims* d, int64_t longest) {
  if (!gla_walk_possible(d) || (d->flags & (PAL_FLAG_STATES_TWO_KERNELS | PAL_FLAG_STATES_ONE_PASS))) return false;
  const int64_t tiles = (longest + PAL_CHUNK - 1) / PAL_CHUNK;
  if (tiles <= 0) return false;
  const int64_t at_a_time = (int64_t)d->total_chunks * d->n_heads / tiles;
  return (d->dk > 64 || d->dv > 64) && at_a_time * (d->dk + d->dv) >= 14500;
}

}  // namespace pal

extern "C" int pal_gla_walk_applies(const PalDims* d, int64_t longest) {
  return pal_validate_dims(d) == PAL_OK && pal::gla_walk_applies(d, longest) ? 1 : 0;
}
