// Arguments of the token-serial forward kernels (recurrent_fwd.hip, recurrent_seg.hip).
#pragma once
#include "pal_common.h"

namespace pal {

struct RecArgs {
  const void *q, *k, *v, *b, *gt;
  const float *g, *Ip;
  void *o, *o_var;
  const float *init_mu, *init_I;
  float *final_mu, *final_I;
  const int32_t* cu_seqlens;
  int32_t T, H, dk, dv, n_seqs;
  int32_t Hq;   // heads of q and k (H, or a divisor of it: a group of H / Hq value heads shares one)
  int32_t gate_bf16, var_bf16;
  uint32_t flags;
  float scale;
};

// Waves that share a sequence in segments, 1: none (recurrent_seg.hip).
int recurrent_segments(const PalDims* d);
// Whether the token-serial kernels are the faster way to the outputs of a chunked call (recurrent_seg.hip).
bool short_pass(const PalDims* d);
bool recurrent_dk_supported(int dk);
int launch_recurrent_seg(const RecArgs& a, int dtype, int waves, hipStream_t s);

}  // namespace pal
