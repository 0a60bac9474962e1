// Pieces shared by the kernels of the chunked backward (chunk_bwd.hip, chunk_bwd_tile.h).
#pragma once
#include "chunk_common.h"

namespace pal {

struct BwdArgs {
  ChunkArgs c;
  const void *d_o, *d_o_var;
  void *dq, *dk, *dv, *db;
  float *dgt, *dg, *dIp, *d_init_mu, *d_init_I;
  void *wDM, *wDJ;        // [total_chunks,H,dv,dk] local carries, then incoming carries, in the dtype of the rows
  float* wFtot;           // [total_chunks,H] log2 of the total decay of a tile
  float* wSig;            // [total_chunks,H] sum over the tile of dJloc
  float* wE;              // [H,tokens]  local part of d log f
  float* wInitPart;       // [n_seqs,H,dv*dk/256] partial sums of dJ_0
  float* wDgTile;         // [total_chunks,H] the tiles' shares of dg
  float* wQK;             // [tokens,H,2,cols] dq, dk of a column group summed so far, where a tile takes several slices of
                          // value rows (bf16 rows); the column groups follow each other, so one group's worth is kept
  // a small pass: every rectangle's parts, summed by chunk_bwd_parts_sum_kernel
  float *pQK, *pVB;       // [slices][tokens,H,2,dk] dq, dk; [column groups][tokens,H,2,dv] dv, db
  float *pE, *pSig;       // [rectangles][H,tokens], [rectangles][total_chunks,H]
  int32_t tokens;
  int32_t apply_stride;    // carry apply: row stride of the carries in LDS
};

// A launch of the tile kernel covers a rectangle of the state: `cols` key columns from n0 on, and value rows from r0 on.
// Larger heads take several: groups of 64, 48 or 32 key columns (16 for a head of 16), in each of them slices of 64, 48,
// 32 or 16 value rows.  (96 columns as 64 + 32, 80 as 48 + 32: workgroups of four or two waves, two or four of them to a
// compute unit.  One workgroup of eight waves has nothing to fill its barriers and its set-up with: 96x96, 32768 packed
// tokens, 16 heads: 5.5 ms, as rectangles 4.2.  A rectangle costs, in ps per state entry and token at B=8 T=2048 H=16, bf16
// rows, 0.63 (64x64: columns x rows), 0.71 (64x48), 0.70 (64x32), 0.80 (48x64), 0.82 (48x48), 0.89 (48x32), 0.90 (32x64), 0.78
// (32x48), 0.80 (32x32), 1.4 (16x16): hence 96 rows of bf16 as 64 + 32 where the group has 64 columns, as 48 + 48 otherwise (96x96
// B=8 T=2048 H=16, kernels of that time: 2155 us with 48 + 48 everywhere, 2055 so; 64x96 1299, 1202).)
struct TileRect {
  int n0, cols, r0, flags;
  int group, groups, slices;   // small pass: first column group, their number (grid z), slices of value rows (grid y)
};
constexpr int kRectColsBefore = 1, kRectRowsBefore = 2, kRectRowsAfter = 4, kRectParts = 8;   // launches that came before, come after; a small pass
inline int tile_piece(int n) { return n == 80 ? 48 : n >= 64 ? 64 : n; }
// fp32 rows: 64 columns by 64 rows and 48 or 32 columns by 48 or 64 take 87 KB of LDS or more than half of a unit's registers'
// worth of waves, and one or two workgroups of them run on a compute unit; slices of 32 rows, twice as many (ps per entry, when both
// were launched, 1.07 against 0.77 for 64 columns, 1.38 and 1.34 against 0.97 for 48, 1.53 and 1.35 against 1.07 for 32; us at 256 tiles
// of 8 heads, 64x64 578 -> 463, 48x48 416 -> 340, 48x96 878 -> 628, 128x64 1169 -> 882, 64x64 with the uncertainty 819 -> 497).  48 rows would
// leave a slice of 16 and stay together where a pass has `few` tiles, one workgroup to a compute unit (whole / in slices, us, by
// tiles x heads: 48x48 192 60 / 68, 256 59 / 68, 384 110 / 97, 512 113 / 110, 1024 217 / 185, with the uncertainty 256 73 / 73, 384 138 /
// 108; 32x48 256 67 / 66, 384 89 / 72, 512 90 / 94, 1024 168 / 161).
inline int tile_rows(int cols, int n, bool f32, bool few) {
  if (cols == 16) return n >= 48 ? 48 : 16;   // (one wave's staging)
  if (f32) return (cols == 64 && n % 48 == 0) || (few && n == 48) ? 48 : n < 32 ? 16 : 32;
  return n == 96 && cols < 64 ? 48 : tile_piece(n);
}

// A pass with too few tiles to fill the chip: all rectangles of a group width in one launch, side by side, each with
// outputs of its own that a last kernel adds up in a fixed order.  One after the other they cost a tile's serial latency
// each, however few workgroups there are.  The slices are small, since it is latency that counts; the group width is one
// that divides the head, if there is one, so that one launch takes them all.  Measured, in us (tile kernel and sum, one
// after the other -> side by side), bf16 rows, by tiles x heads:
//            64          256         384         512         768
//   80x80    225 -> 100  234 -> 160  288 -> 228  293 -> 280  387 -> 392
//   96x96    265 ->  69  273 -> 174  343 -> 253  349 -> 328  454 -> 488
//   96x192   472 -> 103  484 -> 326  625 -> 489  631 -> 649  843 -> 976
//   128x128  307 ->  72  314 -> 233  417 -> 338  425 -> 449  664 -> 667
//   112x112  283 -> 104  293 -> 253  382 -> 377  389 -> 477  610 -> 701
//   48x96    125 ->  55  128 -> 102  163 -> 149  165 -> 173  260 -> 255
//   128x64   148 ->  57  149 -> 122  205 -> 178  208 -> 231  316 -> 340
// fp32 rows 96x96 288 -> 70, 301 -> 184, 382 -> 266, 387 -> 355, 631 -> 528.  The line lies at one and a half workgroups per
// compute unit; at two for fp32 rows and for heads whose pieces come out small (80x80, 96x96), which are the dearest one after the other.
// It bounds the parts too: 8 bytes per token, head, slice and key column, and per group and value column (190 MB at most at 96x192).
constexpr int kPartsTiles = 384, kPartsTilesSmall = 512, kFewTiles = 256;   // tiles x heads
// The slices are of 16 rows where their waves are one to a SIMD at most (two, where there is one column group), of 32 else (16 / 32 rows, us, by tiles x heads:
// 96x96 16 43.3 / 48.8, 32 53.4 / 51.9; 128x64 32 44.3 / 50.8, 64 53.5 / 53.7; 48x96 32 42.7 / 48.9, 64 51.8 / 51.2; 96x192 16
// 55.1 / 51.8).  A head that is one piece is cut too, from 48 rows on, where the waves of its slices are two to a SIMD at most:
// half to a quarter of the tile's serial work, and the sum kernel of 6 us (whole -> slices of 16 rows or, @, 32, us, bf16 rows):
//            32            64            128            192            256
//   64x64    68.7 -> 41.5  69.8 -> 44.2  71.4 -> 54.4   72.2 -> 64.9@  72.2 -> 65.9@
//   64x48    60.0 -> 40.6  60.6 -> 42.7  62.1 -> 52.0   (63.0, 63.6)
//   48x48    52.3 -> 40.8  53.1 -> 42.2  53.8 -> 51.9   (54.8, 61)
//   32x64    69.7 -> 40.0  70.5 -> 42.0  71.7 -> 50.2   72.0 -> 52.2   72.3 -> 54.3
// and 32x32, where it gains nothing (41.1 -> 39.4, 41.2 -> 40.3, 41.9 -> 42.2), stays whole.
constexpr int kPartsWaves = 2048;
struct TileParts {
  int on, rows, slices, groups;
  bool few;   // tiles x heads at most kFewTiles
};
inline int parts_cols(int dk, int n0) { return dk % 64 == 0 ? 64 : dk % 48 == 0 ? 48 : dk % 32 == 0 ? 32 : tile_piece(dk - n0); }
inline TileParts tile_parts(int dk, int dv, bool f32, int64_t tile_heads) {
  TileParts P;
  P.groups = 0;
  P.few = tile_heads <= kFewTiles;
  int pieces = 0, waves = 0;   // one after the other; of the workgroups of a tile's slice
  for (int n0 = 0, c; n0 < dk; n0 += c, ++P.groups) {
    c = parts_cols(dk, n0);
    waves += c >= 48 ? 4 : c / 16;
  }
  for (int n0 = 0, c; n0 < dk; n0 += c) {
    c = tile_piece(dk - n0);
    for (int r0 = 0; r0 < dv; r0 += tile_rows(c, dv - r0, f32, P.few)) ++pieces;
  }
  auto fits = [&](int rows) { return tile_heads * (dv / rows) * waves <= (P.groups > 1 ? kPartsWaves / 2 : kPartsWaves); };
  const bool rows32 = dk > 16 && dv % 32 == 0;
  if (pieces > 1) {
    const bool small = f32 || dk * dv <= pieces * 48 * 48;
    P.on = tile_heads <= (small ? kPartsTilesSmall : kPartsTiles);
  } else {
    P.on = dv >= 48 && (fits(16) || (rows32 && fits(32)));
  }
  P.rows = rows32 && !fits(16) ? 32 : 16;
  P.slices = dv / P.rows;
  return P;
}

constexpr int kHalf = 32;          // tokens of a half tile: the contraction length of one matrix instruction
constexpr int kHS = kHalf + 8;     // row stride (bf16) of the transposed half tiles: 16-byte reads stay aligned

// tokens per step for DT x DN state entries per lane: mu and 1 / I of a step stay in registers
__host__ __device__ constexpr int tile_g(int DT, int DN) { return DT * DN <= 9 ? 8 : 4; }
__host__ __device__ constexpr int rows_pad(int DT) { return DT == 3 ? 4 : DT; }
__host__ __device__ constexpr int vb_stride(int DT, bool var) { return (var ? 4 : 3) * 16 * rows_pad(DT) + 4; }

// whether the tile kernel has a scaled form (chunk_bwd_tile.h), and the numbers that it keeps per token: Ip / F, 1 / F and F with it, f
__host__ __device__ constexpr bool tile_scales(bool var, bool f32) { return !var && !f32; }
__host__ __device__ constexpr int tile_decs(bool var, bool f32) { return tile_scales(var, f32) ? 4 : 1; }

// LDS (floats): running decay, decays of every token (and whether the tile is worked in plain form), decay weights of every step's
// state, their factors of the base state,
// gamma_t, its partial sums; base states; transposed v, b of both halves (of one, and the first half's in the
// partial sums' memory at the start, where that lets two workgroups share a compute unit); two buffers of staged rows
// and of partial dv, db
struct TileLds {
  int oDec, oW, oFB, oX, oXS, oBase, oT, oKQ, oVB, oPart, both, total;
};
__host__ __device__ constexpr TileLds tile_lds(int DT, int DN, int nbw, bool var, bool f32) {
  TileLds L = {};
  const int G = tile_g(DT, DN), half = (f32 ? 2 : 1) * 16 * DT * kHS;   // (two tensors of bf16)
  for (int both = 1; both >= 0; --both) {
    int o = kC;
    L.oDec = o; o += tile_decs(var, f32) * kC + (tile_scales(var, f32) ? 8 : 4);
    L.oW = o; o += (kC / G + 1) * kHalf;
    L.oFB = o; o += kC / G + 4;
    L.oX = o; o += kC + 4;
    L.oXS = o; o += 2 * nbw * G;
    o = (o + 3) & ~3;
    L.oBase = o; o += nbw * 2 * DT * 64 * 4;
    L.oT = o; o += (both ? 2 : 1) * half;
    L.oKQ = o; o += 2 * nbw * G * 32;
    L.oVB = o; o += 2 * G * vb_stride(DT, var);
    const int part = 2 * nbw * G * 32 * DT;
    L.oPart = o; o += both || part > half ? part : half;
    L.both = both;
    L.total = o;
    const int fit = 160 * 1024 / 4 / (nbw > 2 ? 2 : 4);
    if (o <= fit) break;
  }
  return L;
}

template <typename TIn, bool VAR>
int launch_tile_t(const BwdArgs& A, const TileParts& P, hipStream_t s);   // chunk_bwd_tile_*.hip

}  // namespace pal
