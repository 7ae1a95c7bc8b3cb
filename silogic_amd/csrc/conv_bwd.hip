// Entry points of the ConvLogicTree soft backward: the sample-minor kernels
// (conv_sm.hip) for binary trees of depth 1-3 and depth-1 LUTs, the generic
// ones (conv_generic.hip) for deeper trees and for images whose chunk of 64
// samples passes 2 GB or whose rows pass LDS.
#include "conv_sm.h"
#include "conv_tree.h"

using namespace slg;

extern "C" {

int64_t slg_conv_soft_bwd_workspace(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                                    int32_t node_kind, int32_t depth, int32_t arity, int32_t K,
                                    int32_t pad, int32_t pool) {
  if (K < 1 || K > 8 || B < 0 || C <= 0 || H <= 0 || W <= 0 || N <= 0 || pad < 0 || pad > 4 ||
      B >= (1LL << 31) || N >= (1LL << 20) || C >= (1LL << 20) || H >= 4096 || W >= 4096)
    return -1;
  const int64_t Ho = pool ? H / 2 : H, Wo = pool ? W / 2 : W;
  if (Ho == 0 || Wo == 0) return 0;
  const int64_t sm = conv_sm_bwd_workspace(B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0);
  if (sm >= 0) return sm;
  return conv_generic_bwd_workspace(B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0);
}

int slg_conv_soft_bwd(const float* x, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                      int32_t node_kind, int32_t depth, int32_t arity, int32_t K,
                      const float* node_param, const float* w, const int32_t* cm,
                      const int32_t* ch, const int32_t* cw, int32_t pad, int32_t pool,
                      const float* gy, float* gx, float* gw, float* gnp, float* workspace,
                      int64_t workspace_floats, slg_stream_t stream) {
  SLG_REQUIRE(node_param && cm && ch && cw && workspace && ((x && gy) || B == 0), SLG_E_ARG,
              "conv_soft_bwd: null pointer");
  SLG_REQUIRE(node_kind == SLG_NODE_GATE16 || node_kind == SLG_NODE_WALSH ||
                  node_kind == SLG_NODE_MULTILINEAR2 || node_kind == SLG_NODE_HYBRID,
              SLG_E_ARG, "conv_soft_bwd: node_kind %d", node_kind);
  // every tree the sample-minor kernels take is one of the generic set
  SLG_REQUIRE(conv_generic_supported(node_kind, depth, arity), SLG_E_UNSUPPORTED,
              "conv_soft_bwd: node %d depth %d / arity %d", node_kind, depth, arity);
  SLG_REQUIRE(K >= 1 && K <= 8, SLG_E_SHAPE, "conv_soft_bwd: K=%d outside 1..8", K);
  SLG_REQUIRE(B >= 0 && C > 0 && H > 0 && W > 0 && N > 0 && pad >= 0 && pad <= 4 &&
                  B < (1LL << 31) && N < (1LL << 20) && C < (1LL << 20) && H < 4096 &&
                  W < 4096 && N * conv_generic_leaves(node_kind, depth, arity) * K < (1LL << 31),
              SLG_E_SHAPE, "conv_soft_bwd: bad sizes");
  const int64_t Ho = pool ? H / 2 : H, Wo = pool ? W / 2 : W;
  hipStream_t st = as_stream(stream);
  // no samples: zero weight and parameter gradients, also of an empty map
  if (B == 0)
    return conv_sm_zero_grads(N, conv_generic_leaves(node_kind, depth, arity) * (int64_t)K,
                              conv_generic_params(node_kind, depth, arity), gw, gnp, st);
  SLG_REQUIRE(Ho > 0 && Wo > 0, SLG_E_SHAPE, "conv_soft_bwd: empty output map");
  // the same choice as slg_conv_soft_bwd_workspace
  if (conv_sm_bwd_workspace(B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0) >= 0)
    return conv_sm_bwd(x, B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0, node_param, w,
                       cm, ch, cw, gy, gx, gw, gnp, workspace, workspace_floats, st);
  return conv_generic_bwd(x, B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0, node_param,
                          w, cm, ch, cw, gy, gx, gw, gnp, workspace, workspace_floats, st);
}

}  // extern "C"
