// ConvLogicTree backward on sample-minor images (conv_sm.hip).
#pragma once

#include "slg_common.h"

namespace slg {

// Workspace floats of conv_sm_bwd, or -1 where it does not take the tree or
// the sizes (B >= 1, Ho x Wo >= 1 is the routed map); us: its estimated time
// with every gradient wanted.
int64_t conv_sm_bwd_workspace(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                              int depth, int arity, int K, int pad, bool pool, bool want_x,
                              double* us);

// Enqueue the backward on st (arguments as slg_conv_soft_bwd; raw: the pooled
// forward of these gate16 or multilinear trees runs through the caches).
int conv_sm_bwd(const float* x, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                int depth, int arity, int K, int pad, bool pool, bool raw, const float* np,
                const float* w, const int* cm, const int* ch, const int* cw, const float* gy, float* gx,
                float* gw, float* gnp, float* ws, int64_t ws_floats, hipStream_t st);

// Zero gw [N * lk] and gnp [N * np] (either may be null): a batch of no samples.
int conv_sm_zero_grads(int64_t N, int64_t lk, int64_t np, float* gw, float* gnp, hipStream_t st);

}  // namespace slg
