// Scalar-gated linear attention in one walk per result (gla_walk.hip).
#pragma once
#include "chunk_common.h"

namespace pal {

// One of the four results of a call, see gla_walk.hip.
struct GlaWalkRole {
  const bf16_t *X, *Y;         // rows [token][hX][dc]
  const bf16_t* Z;             // rows [token][hZ][de]
  const bf16_t* W;             // rows [token][hZ][de] of the dot products, or null
  bf16_t* out;                 // rows [token][H][de]
  float* dot;                  // [slices][H][tokens], written where W is given
  const float* init;           // state before the first tile: entry (e, c) at [e][c] (init_t: at [c][e]) of [N][H], or null
  float* fin;                  // state after the last tile times fin_scale, [N][H][de][dc], or null
  int32_t init_t, reverse;
  float fin_scale;
};
struct GlaWalkArgs {
  ChunkArgs c;                 // T, H, sequences, gate (gt, g), scale
  GlaWalkRole role[2];         // walks of one launch: the same dc, de, hX and hZ
  int64_t n_tokens;
  int32_t dc, de, hX, hZ, n_roles;
  int32_t n_sl;                // slices of the output columns (filled in by the launch, as the plan)
  WalkPlan plan;
};

// Whether a call can be made with PAL_FLAG_GLA_NO_TILES, and whether it should be (longest: tokens of its longest sequence).
bool gla_walk_possible(const PalDims* d);
bool gla_walk_applies(const PalDims* d, int64_t longest);
// slices of the output columns that n_roles walks over rows of width de are cut into (dot has as many parts)
int gla_walk_slices(const PalDims* d, int dc, int de, int n_roles);
int launch_gla_walk(GlaWalkArgs A, const PalDims* d, int kern_id, hipStream_t s);

}  // namespace pal
