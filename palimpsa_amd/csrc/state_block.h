// A block of the state in the registers of a wave: NG lanes along the key columns by 64 / NG along the value rows, DN columns a
// lane (chunk_out.hip, recurrent_seg.hip).
#pragma once
#include "pal_common.h"

namespace pal {

// lane -> (column group, row group) of a wave; the bits of the column group are the ones the sum over the columns
// moves along (see OutLanes::reduce)
template <int NG>
struct OutLanes {
  static constexpr int DG = 64 / NG;
  static __device__ __forceinline__ int col(int lane) {
    if constexpr (NG == 4) return (lane >> 2) & 3;
    else if constexpr (NG == 8) return ((lane >> 2) & 3) | ((lane & 1) << 2);
    else return lane & (NG - 1);
  }
  static __device__ __forceinline__ int row(int lane) {
    if constexpr (NG == 4) return (lane & 3) | ((lane >> 4) << 2);
    else if constexpr (NG == 8) return ((lane >> 1) & 1) | ((lane >> 4) << 1);
    else return lane / NG;
  }
  // the lanes that hold a copy of a total after the reduction
  static __device__ __forceinline__ bool first(int lane) {
    if constexpr (NG == 4) return true;
    else if constexpr (NG == 8) return (lane & 1) == 0;
    else if constexpr (NG == 16) return (lane & 3) == 0;
    else return (lane & 19) == 0;
  }
  // sum over lane bits 0, 1 and 4, as far as they belong to the column group; every lane gets the total
  static __device__ __forceinline__ float sum_other(float x) {
    if constexpr (NG >= 8) x += quad_move<0xB1>(x);    // quad_perm [1,0,3,2]
    if constexpr (NG >= 16) x += quad_move<0x4E>(x);   // quad_perm [2,3,0,1]
    if constexpr (NG == 32) {
      float y = x;
      swap_rows(x, y);
      x += y;
    }
    return x;
  }
};
// x <- x f + c in one instruction (the compiler would copy c first and accumulate into the copy)
__device__ __forceinline__ void fma3(float& x, float f, float c) {
  asm("v_fma_f32 %0, %0, %1, %2" : "+v"(x) : "v"(f), "v"(c));
}

// pieces of a lane's DN columns: DN / 4 pieces of four, then two, then one; every piece is contiguous over the lanes
template <int NG, int DN>
__device__ __forceinline__ void lds_cols(const float* row, int ng, float* out) {
  constexpr int N4 = DN / 4;
#pragma unroll
  for (int p = 0; p < N4; ++p) *(f32x4*)&out[4 * p] = *(const f32x4*)&row[p * NG * 4 + ng * 4];
  if constexpr ((DN & 3) >= 2) {
    const f32x2 x = *(const f32x2*)&row[N4 * 4 * NG + ng * 2];
    out[4 * N4] = x[0]; out[4 * N4 + 1] = x[1];
  }
  if constexpr (DN & 1) out[DN - 1] = row[(DN - 1) * NG + ng];
}
template <int NG, int DN>
__device__ __forceinline__ constexpr int col_of(int i, int ng) {
  constexpr int N4 = DN / 4;
  if (i < 4 * N4) return (i / 4) * NG * 4 + ng * 4 + i % 4;
  if ((DN & 3) >= 2 && i < 4 * N4 + 2) return 4 * N4 * NG + ng * 2 + (i - 4 * N4);
  return (DN - 1) * NG + ng;
}
}  // namespace pal
