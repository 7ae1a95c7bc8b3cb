// Parameters of a layer in a training step: the connection weights
// softmax(conn) and the node parameters of every tree level from the module's
// own parameters, and the way back (the chain rule through both), one launch
// each. As torch operators they were 5-10 launches forward and as many
// backward per layer (softmax, gate softmax, basis product, sigmoid, stacks
// and concatenations of tree levels), 3-5 us each on tables of a few hundred
// KB; a walsh tree block alone took about 90. Each launch here takes 3.6-6.8 us
// at these sizes. Training steps are bound by the host there: four 2000-output
// FC layers with cross-entropy, B = 256: 1151 -> 865 us together with the FC
// kernels' changes.
//   gate16      c = softmax(logits) @ BASIS                (nodes.py:82-84)
//   walsh       (a, b)-space coefficients of z, times scale (nodes.py:138-143)
//   LUT nodes   s = sigmoid(logits)                        (nodes.py:174-178)
#include <math.h>

#include "slg_common.h"

namespace slg {

constexpr int kLpLevels = 5, kLpMaxK = 16;

struct LpArgs {
  int64_t rows;     // softmax rows of K
  int K;
  int N, NN;        // channels (FC: outputs) and nodes per channel
  int P;            // kept parameters per node
  int kind, levels;
  float scale;
  int m[kLpLevels], off[kLpLevels];  // nodes per channel of a level, first node id
  const float* raw[kLpLevels];
  float* graw[kLpLevels];
  int row_blocks;
};

// The level and row of node thread t (level by level, channels outermost in
// each): raw row n * m + j, kept row n * NN + off + j.
__device__ inline bool lp_node(const LpArgs& a, int64_t t, int& lv, int64_t& raw_row,
                               int64_t& kept_row) {
  for (lv = 0; lv < a.levels; ++lv) {
    const int64_t n = (int64_t)a.N * a.m[lv];
    if (t < n) {
      raw_row = t;
      const int64_t c = t / a.m[lv];
      kept_row = c * a.NN + a.off[lv] + (t - c * a.m[lv]);
      return true;
    }
    t -= n;
  }
  return false;
}

// gate i's value in the basis {1, a, b, ab} for table bits f(a, b) =
// bit 3 - (2a + b) of i (the DiffLogic order, functional.py:24-44).
__device__ constexpr float lp_basis(int i, int c) {
  const int f00 = (i >> 3) & 1, f01 = (i >> 2) & 1, f10 = (i >> 1) & 1, f11 = i & 1;
  return (float)(c == 0 ? f00 : c == 1 ? f10 - f00 : c == 2 ? f01 - f00 : f11 - f10 - f01 + f00);
}

// Sum of the first n of 16 values (the others 0), halves folded: the order of
// a butterfly over as many lanes as the next power of two, in which the
// framework's softmax adds, so that training's forward values (and with them
// the pooled routing at near-ties) do not depend on which of the two ran.
__device__ inline float lp_fold(const float (&e)[16], int n) {
  float s[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = e[i];
#pragma unroll
  for (int h = 8; h >= 1; h >>= 1)
    if (n > h) {
#pragma unroll
      for (int i = 0; i < h; ++i) s[i] = s[i] + s[i + h];
    }
  return s[0];
}

// softmax of 16 logits
__device__ inline void lp_gate_probs(const float* __restrict__ g, float (&p)[16]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 v = reinterpret_cast<const float4*>(g)[q];
    p[4 * q] = v.x;
    p[4 * q + 1] = v.y;
    p[4 * q + 2] = v.z;
    p[4 * q + 3] = v.w;
  }
  float m = p[0];
#pragma unroll
  for (int i = 1; i < 16; ++i) m = fmaxf(m, p[i]);
#pragma unroll
  for (int i = 0; i < 16; ++i) p[i] = expf(p[i] - m);
  const float sum = lp_fold(p, 16);
#pragma unroll
  for (int i = 0; i < 16; ++i) p[i] = p[i] / sum;
}

__global__ void __launch_bounds__(256) layer_params_kernel(LpArgs a, const float* __restrict__ conn,
                                                           float* __restrict__ w,
                                                           float* __restrict__ np,
                                                           float* __restrict__ probs) {
  if ((int)blockIdx.x < a.row_blocks) {
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= a.rows) return;
    float* o = w + r * a.K;
    if (!conn) {  // fixed wiring
      for (int k = 0; k < a.K; ++k) o[k] = 1.0f;
      return;
    }
    const float* c = conn + r * a.K;
    float e[kLpMaxK], m = c[0];
    for (int k = 1; k < a.K; ++k) m = fmaxf(m, c[k]);
#pragma unroll
    for (int k = 0; k < kLpMaxK; ++k) e[k] = k < a.K ? expf(c[k] - m) : 0.0f;
    const float sum = lp_fold(e, a.K);
#pragma unroll
    for (int k = 0; k < kLpMaxK; ++k)
      if (k < a.K) o[k] = e[k] / sum;
    return;
  }
  const int64_t t = (int64_t)((int)blockIdx.x - a.row_blocks) * 256 + threadIdx.x;
  int lv;
  int64_t rr, kr;
  const bool lut = a.kind == SLG_NODE_MULTILINEAR2 || a.kind == SLG_NODE_HYBRID;
  if (!lp_node(a, lut ? t / a.P : t, lv, rr, kr)) return;
  if (lut) {  // a thread per value
    const int e = (int)(t % a.P);
    np[kr * a.P + e] = sigmoid_exact(a.raw[lv][rr * a.P + e]);
    return;
  }
  float c[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (a.kind == SLG_NODE_GATE16) {
    float p[16];
    lp_gate_probs(a.raw[lv] + rr * 16, p);
    if (probs) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        reinterpret_cast<float4*>(probs + kr * 16)[q] =
            make_float4(p[4 * q], p[4 * q + 1], p[4 * q + 2], p[4 * q + 3]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (lp_basis(i, q) != 0.0f) c[q] = fmaf(p[i], lp_basis(i, q), c[q]);
  } else {
    const float4 v = reinterpret_cast<const float4*>(a.raw[lv])[rr];
    c[0] = (((v.x - v.y) - v.z) + v.w) * a.scale;
    c[1] = 2.0f * (v.y - v.w) * a.scale;
    c[2] = 2.0f * (v.z - v.w) * a.scale;
    c[3] = 4.0f * v.w * a.scale;
  }
  reinterpret_cast<float4*>(np)[kr] = make_float4(c[0], c[1], c[2], c[3]);
}

// From what the forward wrote: the parameters may have changed since (an
// update between a forward and its backward).
__global__ void __launch_bounds__(256)
layer_params_bwd_kernel(LpArgs a, const float* __restrict__ w, const float* __restrict__ gw,
                        const float* __restrict__ kept, float* __restrict__ gconn,
                        const float* __restrict__ gnp) {
  if ((int)blockIdx.x < a.row_blocks) {
    const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= a.rows) return;
    const float *p = w + r * a.K, *g = gw + r * a.K;
    float s = 0.0f;
    for (int k = 0; k < a.K; ++k) s = fmaf(p[k], g[k], s);
    for (int k = 0; k < a.K; ++k) gconn[r * a.K + k] = p[k] * (g[k] - s);
    return;
  }
  const int64_t t = (int64_t)((int)blockIdx.x - a.row_blocks) * 256 + threadIdx.x;
  int lv;
  int64_t rr, kr;
  const bool lut = a.kind == SLG_NODE_MULTILINEAR2 || a.kind == SLG_NODE_HYBRID;
  if (!lp_node(a, lut ? t / a.P : t, lv, rr, kr) || !a.graw[lv]) return;
  if (lut) {
    const int e = (int)(t % a.P);
    const float s = kept[kr * a.P + e];
    a.graw[lv][rr * a.P + e] = gnp[kr * a.P + e] * (s * (1.0f - s));
    return;
  }
  const float4 g = reinterpret_cast<const float4*>(gnp)[kr];
  if (a.kind == SLG_NODE_GATE16) {
    float p[16], d[16], s = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = reinterpret_cast<const float4*>(kept + kr * 16)[q];
      p[4 * q] = v.x;
      p[4 * q + 1] = v.y;
      p[4 * q + 2] = v.z;
      p[4 * q + 3] = v.w;
    }
    const float gc[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      d[i] = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (lp_basis(i, q) != 0.0f) d[i] = fmaf(lp_basis(i, q), gc[q], d[i]);
      s = fmaf(p[i], d[i], s);
    }
    float4* o = reinterpret_cast<float4*>(a.graw[lv] + rr * 16);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      o[q] = make_float4(p[4 * q] * (d[4 * q] - s), p[4 * q + 1] * (d[4 * q + 1] - s),
                         p[4 * q + 2] * (d[4 * q + 2] - s), p[4 * q + 3] * (d[4 * q + 3] - s));
  } else {
    reinterpret_cast<float4*>(a.graw[lv])[rr] =
        make_float4(g.x * a.scale, (2.0f * g.y - g.x) * a.scale, (2.0f * g.z - g.x) * a.scale,
                    (g.x + 4.0f * g.w - 2.0f * (g.y + g.z)) * a.scale);
  }
}

static bool lp_binary(int kind) { return kind == SLG_NODE_GATE16 || kind == SLG_NODE_WALSH; }

static int lp_args(LpArgs& a, int64_t rows, int32_t K, int32_t n_levels, const int32_t* nodes,
                   int64_t N, int32_t kind, int32_t arity, float scale, const char* what) {
  SLG_REQUIRE(nodes, SLG_E_ARG, "%s: null array", what);
  SLG_REQUIRE(kind >= SLG_NODE_GATE16 && kind <= SLG_NODE_HYBRID, SLG_E_ARG, "%s: node_kind %d", what,
              kind);
  SLG_REQUIRE(n_levels >= 1 && n_levels <= kLpLevels && K >= 1 && K <= kLpMaxK && arity >= 2 &&
                  arity <= 6 && N > 0 && rows >= 0 && rows < (1LL << 31) && N < (1LL << 28),
              SLG_E_SHAPE, "%s: bad sizes", what);
  a.rows = rows; a.K = K; a.N = (int)N; a.kind = kind; a.levels = n_levels; a.scale = scale;
  a.P = lp_binary(kind) ? 4 : (1 << arity);
  for (int i = 0; i < n_levels; ++i) {
    SLG_REQUIRE(nodes[i] > 0, SLG_E_ARG, "%s: level %d", what, i);
    a.m[i] = nodes[i];
    a.off[i] = a.NN;
    a.NN += nodes[i];
  }
  SLG_REQUIRE(N * a.NN * a.P < (1LL << 31), SLG_E_SHAPE, "%s: too many parameters", what);
  return 0;
}

static unsigned lp_node_blocks(const LpArgs& a) {
  return (unsigned)cdiv((int64_t)a.N * a.NN * (lp_binary(a.kind) ? 1 : a.P), 256);
}

}  // namespace slg

using namespace slg;

extern "C" {

int slg_layer_params(const float* conn, int64_t rows, int32_t K, int32_t n_levels,
                     const float* const* raw, const int32_t* nodes, int64_t N, int32_t node_kind,
                     int32_t arity, float scale, float* w, float* node_param, float* probs,
                     slg_stream_t stream) {
  LpArgs a{};
  const int rc = lp_args(a, rows, K, n_levels, nodes, N, node_kind, arity, scale, "layer_params");
  if (rc) return rc;
  SLG_REQUIRE(raw, SLG_E_ARG, "layer_params: null array");
  for (int i = 0; i < n_levels; ++i) {
    // rows of 4 and 16 values are read as quads
    SLG_REQUIRE(raw[i] && (!lp_binary(node_kind) || (uintptr_t)raw[i] % 16 == 0), SLG_E_ARG,
                "layer_params: level %d", i);
    a.raw[i] = raw[i];
  }
  SLG_REQUIRE(w && node_param && ((uintptr_t)node_param | (uintptr_t)probs) % 16 == 0, SLG_E_ARG,
              "layer_params: output");
  a.row_blocks = (int)cdiv(rows, 256);
  hipLaunchKernelGGL(layer_params_kernel, dim3(a.row_blocks + lp_node_blocks(a)), dim3(256), 0,
                     as_stream(stream), a, conn, w, node_param, probs);
  SLG_LAUNCH_CHECK("layer_params");
  return 0;
}

int slg_layer_params_bwd(const float* w, const float* gw, int64_t rows, int32_t K, int32_t n_levels,
                         const int32_t* nodes, int64_t N, int32_t node_kind, int32_t arity,
                         float scale, const float* kept, const float* gnp, float* gconn,
                         float* const* graw, slg_stream_t stream) {
  LpArgs a{};
  const int rc = lp_args(a, rows, K, n_levels, nodes, N, node_kind, arity, scale, "layer_params_bwd");
  if (rc) return rc;
  SLG_REQUIRE(!gconn || (w && gw), SLG_E_ARG, "layer_params_bwd: null weights");
  bool nodes_wanted = false;
  for (int i = 0; graw && i < n_levels; ++i) {
    SLG_REQUIRE(!graw[i] || (uintptr_t)graw[i] % 16 == 0, SLG_E_ARG, "layer_params_bwd: alignment");
    a.graw[i] = graw[i];
    nodes_wanted |= graw[i] != nullptr;
  }
  SLG_REQUIRE(!nodes_wanted || (gnp && (kept || node_kind == SLG_NODE_WALSH) &&
                                ((uintptr_t)gnp | (uintptr_t)kept) % 16 == 0),
              SLG_E_ARG, "layer_params_bwd: node gradients");
  a.row_blocks = gconn ? (int)cdiv(rows, 256) : 0;
  const unsigned blocks = a.row_blocks + (nodes_wanted ? lp_node_blocks(a) : 0);
  if (blocks == 0) return 0;
  hipLaunchKernelGGL(layer_params_bwd_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), a, w, gw,
                     kept, gconn, gnp);
  SLG_LAUNCH_CHECK("layer_params_bwd");
  return 0;
}

}  // extern "C"
