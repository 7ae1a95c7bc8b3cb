// ConvLogicTree backward with lanes along output positions (conv_pos.hip).
#pragma once

#include "slg_common.h"

namespace slg {

// Workspace floats of conv_pos_bwd, or -1 where it does not take the tree or
// the sizes (B >= 1, Ho x Wo >= 1 is the routed map). raw: the pooled forward
// of these sizes runs through the caches (conv_forward_on_lds). us: its
// estimated time with every gradient wanted.
int64_t conv_pos_bwd_workspace(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                               int depth, int arity, int K, int pad, bool pool, bool raw,
                               bool want_x, double* us);

// Enqueue the backward on st (arguments as slg_conv_soft_bwd).
int conv_pos_bwd(const float* x, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                 int depth, int arity, int K, int pad, bool pool, bool raw, const float* np,
                 const float* w, const int* cm, const int* ch, const int* cw, const float* gy,
                 float* gx, float* gw, float* gnp, float* ws, int64_t ws_floats, hipStream_t st);

}  // namespace slg
