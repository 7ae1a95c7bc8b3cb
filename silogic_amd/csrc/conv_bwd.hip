// Entry points of the ConvLogicTree soft backward and the choice of its
// kernels: with lanes along samples (conv_sm.hip) or along output positions
// (conv_pos.hip), for the trees and sizes that each takes, and the generic ones
// (conv_generic.hip) for any tree.
//
// Lanes along samples do the least work, but in units of 64 samples, and few
// samples leave serial chains (an output row of a tree, the taps of a channel)
// that the chip waits for. 16 -> 32 channels, 5 x 5, 96 x 96, one pooled sample,
// along samples / positions / generic: gate16 depth 2, K = 4: 759 / 352 / 113
// us; 16 of them: 676 / 389 / 547; 64 -> 128, 3 x 3, 14 x 14, 256 samples: 114 /
// 297 / 1417. No one size divides them, so each file estimates its time from what
// it would launch, and the shortest is taken. The factors were fitted to 4700
// random shapes (1-1024 samples, 1-512 channels, maps of 4-128, kernels 1-7,
// every node kind, pooled and not, each timed on all three): the estimates
// scatter by 25-30%; the choice is 1.9% slower than the best of the three on
// average, by more than 10% for 6% of them, the worst 3.5 times (always along
// samples: 17% on average, 20 times). Not by whether the input gradient is
// wanted: the other gradients are the same bits with and without it.
#include <array>

#include "conv_pos.h"
#include "conv_sm.h"
#include "conv_tree.h"

namespace slg {

struct ConvBwdChoice {
  int path;         // SLG_CONV_BWD_*
  bool raw;         // the pooled forward of these sizes runs through the caches
  int64_t floats;   // workspace, -1: refused
};

// path: SLG_CONV_BWD_AUTO or the kernels to take, where they take the sizes.
static ConvBwdChoice conv_bwd_estimate(int path, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                                       int node, int depth, int arity, int K, int pad, bool pool,
                                       bool want_x) {
  ConvBwdChoice c{};
  c.raw = pool && (node == SLG_NODE_GATE16 || node == SLG_NODE_MULTILINEAR2) &&
          !conv_forward_on_lds(C, H, W, N, node, depth, arity, K, pad, pool);
  const auto workspace = [&](int p, bool gx, double* us) -> int64_t {
    if (p == SLG_CONV_BWD_SAMPLES)
      return conv_sm_bwd_workspace(B, C, H, W, N, node, depth, arity, K, pad, pool, gx, us);
    if (p == SLG_CONV_BWD_POSITIONS)
      return conv_pos_bwd_workspace(B, C, H, W, N, node, depth, arity, K, pad, pool, c.raw, gx, us);
    if (p == SLG_CONV_BWD_GENERIC)
      return conv_generic_bwd_workspace(B, C, H, W, N, node, depth, arity, K, pad, pool, us);
    return -1;
  };
  c.path = path;
  if (path == SLG_CONV_BWD_AUTO) {
    // past 4 GB of workspace only where no other kernels take the sizes
    constexpr int64_t kMost = int64_t(1) << 30;
    double best = 0.0;
    bool best_large = false;
    for (int p = SLG_CONV_BWD_SAMPLES; p <= SLG_CONV_BWD_GENERIC; ++p) {
      double us = 0.0;
      const int64_t floats = workspace(p, true, &us);
      const bool large = floats > kMost;
      if (floats < 0 || (c.path != SLG_CONV_BWD_AUTO && (large > best_large ||
                                                         (large == best_large && us >= best))))
        continue;
      c.path = p;
      best = us;
      best_large = large;
    }
  }
  c.floats = workspace(c.path, want_x, nullptr);
  return c;
}

// The last few choices of a thread, by everything they depend on: the workspace
// query and the call that follows it ask the same, each step again (2-3 us each).
static ConvBwdChoice conv_bwd_choose(int path, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                                     int node, int depth, int arity, int K, int pad, bool pool,
                                     bool want_x) {
  using Key = std::array<int64_t, 15>;
  struct Kept {
    Key key;
    ConvBwdChoice choice;
  };
  constexpr int kKept = 16;
  static thread_local Kept kept[kKept];  // all zero: no choice has zero channels
  static thread_local unsigned next = 0;
  const Key key{path, B, C, H, W, N, node, depth, arity, K, pad, pool, want_x, device_cus(),
                device_lds_bytes()};
  for (const Kept& k : kept)
    if (k.key == key) return k.choice;
  Kept& k = kept[next++ % kKept];
  k.choice = conv_bwd_estimate(path, B, C, H, W, N, node, depth, arity, K, pad, pool, want_x);
  k.key = key;
  return k.choice;
}

}  // namespace slg

using namespace slg;

extern "C" {

int64_t slg_conv_soft_bwd_workspace_on(int32_t path, int64_t B, int64_t C, int64_t H, int64_t W,
                                       int64_t N, int32_t node_kind, int32_t depth, int32_t arity,
                                       int32_t K, int32_t pad, int32_t pool, int32_t want_gx) {
  if (K < 1 || K > 8 || B < 0 || C <= 0 || H <= 0 || W <= 0 || N <= 0 || pad < 0 || pad > 4 ||
      B >= (1LL << 31) || N >= (1LL << 20) || C >= (1LL << 20) || H >= 4096 || W >= 4096)
    return -1;
  if (pool && (H < 2 || W < 2)) return 0;
  return conv_bwd_choose(path, std::max<int64_t>(B, 1), C, H, W, N, node_kind, depth, arity, K, pad,
                         pool != 0, want_gx != 0).floats;
}

int64_t slg_conv_soft_bwd_workspace(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                                    int32_t node_kind, int32_t depth, int32_t arity, int32_t K,
                                    int32_t pad, int32_t pool) {
  return slg_conv_soft_bwd_workspace_on(SLG_CONV_BWD_AUTO, B, C, H, W, N, node_kind, depth, arity, K,
                                        pad, pool, 1);
}

int slg_conv_soft_bwd_on(int32_t path, const float* x, int64_t B, int64_t C, int64_t H, int64_t W,
                         int64_t N, int32_t node_kind, int32_t depth, int32_t arity, int32_t K,
                         const float* node_param, const float* w, const int32_t* cm,
                         const int32_t* ch, const int32_t* cw, int32_t pad, int32_t pool,
                         const float* gy, float* gx, float* gw, float* gnp, float* workspace,
                         int64_t workspace_floats, slg_stream_t stream) {
  SLG_REQUIRE(path >= SLG_CONV_BWD_AUTO && path <= SLG_CONV_BWD_GENERIC, SLG_E_ARG,
              "conv_soft_bwd: path %d", path);
  SLG_REQUIRE(node_param && cm && ch && cw && workspace && ((x && gy) || B == 0), SLG_E_ARG,
              "conv_soft_bwd: null pointer");
  SLG_REQUIRE(node_kind == SLG_NODE_GATE16 || node_kind == SLG_NODE_WALSH ||
                  node_kind == SLG_NODE_MULTILINEAR2 || node_kind == SLG_NODE_HYBRID,
              SLG_E_ARG, "conv_soft_bwd: node_kind %d", node_kind);
  // every tree the other kernels take is one of the generic set
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
  const ConvBwdChoice c = conv_bwd_choose(path, B, C, H, W, N, node_kind, depth, arity, K, pad,
                                          pool != 0, gx != nullptr);
  SLG_REQUIRE(c.floats >= 0, SLG_E_UNSUPPORTED, "conv_soft_bwd: sizes outside the kernels");
  if (c.path == SLG_CONV_BWD_SAMPLES)
    return conv_sm_bwd(x, B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0, c.raw, node_param,
                       w, cm, ch, cw, gy, gx, gw, gnp, workspace, workspace_floats, st);
  if (c.path == SLG_CONV_BWD_POSITIONS)
    return conv_pos_bwd(x, B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0, c.raw, node_param,
                        w, cm, ch, cw, gy, gx, gw, gnp, workspace, workspace_floats, st);
  return conv_generic_bwd(x, B, C, H, W, N, node_kind, depth, arity, K, pad, pool != 0, node_param,
                          w, cm, ch, cw, gy, gx, gw, gnp, workspace, workspace_floats, st);
}

int slg_conv_soft_bwd(const float* x, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N,
                      int32_t node_kind, int32_t depth, int32_t arity, int32_t K,
                      const float* node_param, const float* w, const int32_t* cm,
                      const int32_t* ch, const int32_t* cw, int32_t pad, int32_t pool,
                      const float* gy, float* gx, float* gw, float* gnp, float* workspace,
                      int64_t workspace_floats, slg_stream_t stream) {
  return slg_conv_soft_bwd_on(SLG_CONV_BWD_AUTO, x, B, C, H, W, N, node_kind, depth, arity, K,
                              node_param, w, cm, ch, cw, pad, pool, gy, gx, gw, gnp, workspace,
                              workspace_floats, stream);
}

}  // extern "C"
