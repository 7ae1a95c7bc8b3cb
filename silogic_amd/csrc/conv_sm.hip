// ConvLogicTree soft backward for gfx950, with the fused 2x2 OR-pool (the
// gradients the reference's tree-conv ops return: kernels/conv.py:94-145,
// kernels/conv_topk.py:84-121, with F.max_pool2d's routing, layers.py:558-559).
// Given x [B,C,H,W], the trees' taps (cm, ch, cw), leaf weights w and node
// parameters, and gy [B,N,Ho,Wo] on the (pooled) output, write
//   gx  [B,C,H,W]   = sum over taps of w * (leaf gradient at the tap's output),
//   gw  [N,L,K]     = sum over samples and outputs of leaf gradient * tap value,
//   gnp             = sum over samples and outputs of dL/dparam.
// With pooling, each pooled output sends its gradient to the first window
// position (row-major) holding the window's maximum, as F.max_pool2d does.
//
// Lanes are samples. A tree's taps, weights and parameters and the position
// it is evaluated at are then the same in every lane: tap addresses are
// scalar, weights are scalar operands of the FMAs, nothing is bounds-checked
// (the images are stored with a zero border) and every global load and store
// of a wave is one contiguous 256-byte run. With lanes along positions the
// same work took 3-6 times the vector instructions (per-lane tap addresses
// and bounds, LDS broadcast of every tap) and its input-gradient gather
// visited each tap four times, once per window position.
//
// Measured (backward kernels of one block, 3 x 3, K = 4, lanes along positions
// -> here): gate16 depth 2, 64 -> 128 channels at 14 x 14, B = 1024: 950 -> 260
// us (grad 81, gx 126, images 32); LUT6, 128 -> 256 at 16 x 16, B = 512: 2900
// -> 580 us (route 106, grad 197, gx 219, images 39); walsh depth 2, 64 -> 128
// at 14 x 14, B = 256: 1470 -> 130 us. What bounds them now (counters of config 3
// and 5 training steps): sm_grad and sm_route the vector ALU (LUT6: 590 and 440
// instructions per 64 outputs, 219 us at full issue of the 288) and LDS; sm_gx
// the latency of the leaf gradients, which it reads 1.6 (gate16: 163 MB from
// HBM) and 2.8 times (LUT6: 571 MB), each being read by its tree's two channels
// and by neighbouring strips; sm_images the copy rate.
//
// Launches, per round of samples (kSmRoundFloats):
//   sm_images    x and gy to sample-minor chunks of 64 samples;
//   sm_tables    per tree: tap offsets, weights, parameters; per input
//                channel: its references (tree, leaf, tap) in ascending order;
//   sm_route     (LUTs of 5 and 6 leaves) the window position of every
//                (tree, pooled output, sample);
//   sm_grad      that of the other trees, the leaf gradients of every (tree,
//                output, sample), and the weight and parameter gradients
//                summed in registers over a job's outputs and samples;
//   sm_gx        the input gradient: a wave owns a strip of rows of one
//                channel for 64 samples in LDS and adds the channel's taps
//                to it, one read-modify-write per (tap, output);
//   sm_sum       the jobs' weight and parameter sums.
// No value is added atomically and every sum has a fixed order, so the
// gradients are the same bits on every call.
#include <math.h>

#include <type_traits>

#include "conv_sm.h"
#include "conv_tree.h"

namespace slg {

constexpr int kSmMaxK = 8;

// Trees taken: binary gate16 / walsh trees of depth 1-3, LUTs of arity 2-6.
template <int NODE, int NLEAF>
struct SmTree {
  static constexpr bool kBinary = NODE == SLG_NODE_GATE16 || NODE == SLG_NODE_WALSH;
  static constexpr int NN = kBinary ? NLEAF - 1 : 1;
  static constexpr int NP = kBinary ? 4 * NN : (1 << NLEAF);  // parameters, as the caller's
};

// A tree's record (4-byte words): tap byte offsets into the image [L*KM],
// weights [L*KM], parameters as the evaluation keeps them [NP], for a LUT its
// values as (even corner, odd - even) pairs [NP/2][2] for the backward, the
// tree's channels (two, and whether it reads more), and the taps' byte offsets
// in the window ring, one table per ring phase: A(window column 0) |
// A(window column 1) << 16.
template <int NODE, int NLEAF, int KM>
struct SmRec {
  using T = SmTree<NODE, NLEAF>;
  static constexpr int LK = NLEAF * KM;
  static constexpr int off = 0, wt = LK, par = 2 * LK, pair = par + T::NP;
  static constexpr int chan = pair + (T::kBinary ? 0 : T::NP), ring = chan + 4;
  __host__ __device__ static constexpr int words(int kernel) { return ring + (kernel + 1) / 2 * LK; }
};

struct SmArgs {
  int B, C, H, W, Hp, Wp, N, K, kernel, pad;
  int Ho, Wo, P;      // routed map
  int U, RW;          // outputs of a row per sm_gx step (and route word), steps per row
  int nc;             // 64-sample chunks of this round
  int PS, RPS;        // row splits of the map, rows per split
  int ncg;            // chunk groups: a job takes chunks cg, cg + ncg, ...
  int TH, nt;         // sm_gx: rows per strip, strips per image
  int GS;             // sm_gx: parts of a channel's taps, a wave each
  int Cz;             // channels stored: C, and a zero one for candidates past K
  int RS;             // record words
  int raw;            // the forward runs through the caches: the parameters kept as they are
  int64_t xs;         // floats per chunk of the sample-minor image
};

// ---------------------------------------------------------------------------
// sample-minor images
// ---------------------------------------------------------------------------
// dst [nc][D][64]: 64 positions x 64 samples through an LDS tile, both sides
// coalesced. x: positions of the zero-bordered image; gy: its [N*P] values as
// they lie.
__global__ void __launch_bounds__(256) sm_images_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ gy, SmArgs a,
                                                        int xt, int gt, float* __restrict__ xT,
                                                        float* __restrict__ gT) {
  __shared__ float t[64][65];
  const int per = xt + gt;  // position tiles per chunk
  const int chunk = (int)(blockIdx.x / (unsigned)per);
  const int tile = (int)(blockIdx.x - (unsigned)chunk * per);
  const bool img = tile < xt;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b0 = chunk * 64;
  const int HWp = a.Hp * a.Wp;
  const int D = img ? a.Cz * HWp : a.N * a.P;
  const int64_t S = img ? (int64_t)a.C * a.H * a.W : (int64_t)a.N * a.P;  // source sample stride
  const int d0 = (img ? tile : tile - xt) * 64;
  const int d = d0 + lane;
  int64_t si = -1;
  if (d < D) {
    if (img) {
      const int c = d / HWp, r = d - c * HWp;
      const int yp = r / a.Wp;
      const int y = yp - a.pad, xx = r - yp * a.Wp - a.pad;
      if (c < a.C && (unsigned)y < (unsigned)a.H && (unsigned)xx < (unsigned)a.W)
        si = ((int64_t)c * a.H + y) * a.W + xx;
    } else {
      si = d;
    }
  }
  const float* src = img ? x : gy;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int b = b0 + wave * 16 + i;
    v[i] = (si >= 0 && b < a.B) ? src[(int64_t)b * S + si] : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) t[lane][wave * 16 + i] = v[i];
  __syncthreads();
  float* dst = img ? xT + (int64_t)chunk * a.xs : gT + (int64_t)chunk * D * 64;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int p = wave * 16 + i;
    if (d0 + p < D) dst[(int64_t)(d0 + p) * 64 + lane] = t[p][lane];
  }
}

// ---------------------------------------------------------------------------
// tables
// ---------------------------------------------------------------------------
struct SmRef {    // one tap of a channel
  int tree;
  int next;       // index past the leaf's taps on this channel
  uint32_t d;     // dh | dw << 4 (offsets into the bordered image), the least
                  // and largest dh of the leaf's taps << 8, << 12, leaf << 16
  float w;
};

// Workgroups [0, rb): the records, one wave per tree. The others: the
// references of one input channel, in ascending order: its 16 waves count the
// references of lower channels (the channel's first slot) and their own in a
// sixteenth of the list each, then write them (a ballot per 64). One launch
// instead of a count, scan, placement and ranking over the same few thousand
// taps.
template <int NODE, int NLEAF, int KM>
__global__ void __launch_bounds__(1024)
sm_tables_kernel(SmArgs a, int rb, const float* __restrict__ np, const float* __restrict__ w,
                 const int* __restrict__ cm, const int* __restrict__ ch,
                 const int* __restrict__ cw, uint32_t* __restrict__ recs,
                 int* __restrict__ start, SmRef* __restrict__ refs) {
  using R = SmRec<NODE, NLEAF, KM>;
  using T = SmTree<NODE, NLEAF>;
  constexpr int LK = NLEAF * KM;
  static_assert(LK <= 64, "a lane per tap");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((int)blockIdx.x < rb) {
    const int n = blockIdx.x * 16 + wave;
    if (n >= a.N) return;
    uint32_t* rec = recs + (int64_t)n * a.RS;
    const int l = lane / KM, k = lane - l * KM;
    const bool tap = lane < LK && k < a.K;
    const int r = tap ? (n * NLEAF + l) * a.K + k : 0;
    const int c = min(max(cm[r], 0), a.C - 1);
    const int dh = min(max(ch[r], 0), a.kernel - 1), dw = min(max(cw[r], 0), a.kernel - 1);
    // the tree's first two channels, in tap order
    const int c0 = __builtin_amdgcn_readfirstlane(c);
    const uint64_t other = __ballot(tap && c != c0);
    const int c1 = other ? __builtin_amdgcn_readlane(c, __ffsll((unsigned long long)other) - 1) : c0;
    const bool more = __ballot(tap && c != c0 && c != c1) != 0;
    const int RC = a.kernel + 1;  // window rows and columns
    if (lane < LK) {  // candidates past K read zeros with a zero weight
      rec[R::off + lane] = (uint32_t)(tap ? (c * a.Hp + dh) * a.Wp + dw : a.C * a.Hp * a.Wp) * 256u;
      rec[R::wt + lane] = __float_as_uint(tap ? (w ? w[r] : 1.0f) : 0.0f);
      for (int ph = 0; ph < RC / 2; ++ph) {
        uint32_t A[2];
#pragma unroll
        for (int qx = 0; qx < 2; ++qx) {
          const int slot = (dw + qx + 2 * ph) % RC;
          A[qx] = (uint32_t)(tap ? (((c == c0 ? 0 : RC) + slot) * RC + dh) : 2 * RC * RC) * 256u;
        }
        rec[R::ring + ph * LK + lane] = A[0] | (A[1] << 16);
      }
    }
    if (lane < 4) rec[R::chan + lane] = lane == 0 ? (uint32_t)c0 : lane == 1 ? (uint32_t)c1 : (uint32_t)more;
    const float* p = np + (int64_t)n * T::NP;
    for (int e = lane; e < T::NP; e += 64) {
      float f = p[e];
      if constexpr (!T::kBinary) {
        const float mine = f;
        if constexpr (NODE != SLG_NODE_HYBRID) {  // the form of the forward on LDS (lut_group_coeffs)
          if (!a.raw) {
            constexpr int LG = ConvNode<NODE, NLEAF>::LG, GM = (1 << LG) - 1;
            float g[1 << LG];
#pragma unroll
            for (int u = 0; u <= GM; ++u) g[u] = p[(e & ~GM) + u];
            lut_group_coeffs<LG>(g);
            f = g[0];
#pragma unroll
            for (int u = 1; u <= GM; ++u) f = (e & GM) == u ? g[u] : f;
          }
        }
        rec[R::pair + e] = __float_as_uint((e & 1) ? mine - p[e - 1] : mine);
      }
      rec[R::par + e] = __float_as_uint(f);
    }
    return;
  }
  __shared__ int lower[16], own[16];
  const int c = (int)blockIdx.x - rb;
  const int R_ = a.N * NLEAF * a.K;
  const int seg = (R_ / 16 + 64) & ~63;
  const int r0 = min(R_, wave * seg), r1 = min(R_, r0 + seg);
  const uint64_t below = (1ull << lane) - 1ull;
  constexpr int G = 8;  // loads in flight
  int lo = 0, eq = 0;
  for (int base = r0; base < r1; base += G * 64) {
    int t[G];
#pragma unroll
    for (int i = 0; i < G; ++i) t[i] = cm[min(base + i * 64 + lane, R_ - 1)];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const bool in = base + i * 64 + lane < r1;
      const int v = min(max(t[i], 0), a.C - 1);
      lo += __popcll(__ballot(in && v < c));
      eq += __popcll(__ballot(in && v == c));
    }
  }
  if (lane == 0) {
    lower[wave] = lo;
    own[wave] = eq;
  }
  __syncthreads();
  int first = 0, at = 0, end = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    first += lower[i];
    at += i < wave ? own[i] : 0;
    end += own[i];
  }
  at += first;
  if (threadIdx.x == 0) {
    start[c] = first;
    if (c == a.C - 1) start[a.C] = first + end;
  }
  for (int base = r0; base < r1; base += G * 64) {
    int t[G];
#pragma unroll
    for (int i = 0; i < G; ++i) t[i] = cm[min(base + i * 64 + lane, R_ - 1)];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int r = base + i * 64 + lane;
      const bool mine = r < r1 && min(max(t[i], 0), a.C - 1) == c;
      const uint64_t m = __ballot(mine);
      if (mine) {
        const int j = at + __popcll(m & below);
        const int row = r / a.K;
        int dlo = 255, dhi = 0, later = 0;
        for (int k = 0; k < a.K; ++k) {  // the leaf's other taps on this channel
          const int q = row * a.K + k;
          if (min(max(cm[q], 0), a.C - 1) == c) {
            const int dh = min(max(ch[q], 0), a.kernel - 1);
            dlo = min(dlo, dh);
            dhi = max(dhi, dh);
            later += q > r;
          }
        }
        SmRef e;
        e.tree = row / NLEAF;
        e.next = j + 1 + later;
        e.d = (uint32_t)min(max(ch[r], 0), a.kernel - 1) |
              ((uint32_t)min(max(cw[r], 0), a.kernel - 1) << 4) | ((uint32_t)dlo << 8) |
              ((uint32_t)dhi << 12) | ((uint32_t)(row - e.tree * NLEAF) << 16);
        e.w = w ? w[r] : 1.0f;
        refs[j] = e;
      }
      at += __popcll(m);
    }
  }
}

// ---------------------------------------------------------------------------
// tree evaluation and gradients, one sample per lane
// ---------------------------------------------------------------------------
// Records are read as constant memory (scalar loads) through a pointer the
// compiler cannot see through, so that the loads stay where they are made: the
// tables pass the scalar registers and would otherwise be hoisted out of the
// output loop and spilled.
using SmWords = const uint32_t __attribute__((address_space(4)))*;
__device__ inline SmWords sm_words(const uint32_t* p) {
  uint64_t a = (uint64_t)p;
  asm volatile("" : "+s"(a));
  return (SmWords)a;
}

// Walsh trees have no LDS forward.
template <int NODE>
constexpr bool sm_lds_form() { return NODE != SLG_NODE_WALSH; }

// Leaf gradients of a binary tree (node ids level-major) at leaf values v
// for upstream gradient g; each node's parameter gradient U * (1, a, b, ab)
// is added to acc.
template <int NODE, int NLEAF>
__device__ inline void sm_grad_binary(const float (&v)[NLEAF], const float* par, float g,
                                      float (&gl)[NLEAF], float (&acc)[4 * (NLEAF - 1)]) {
  constexpr int NN = NLEAF - 1;
  float val[NLEAF + NN];  // leaves, then nodes
#pragma unroll
  for (int l = 0; l < NLEAF; ++l) val[l] = v[l];
#pragma unroll
  for (int i = 0; i < NN; ++i) {  // node i's children are values 2i, 2i + 1
    if constexpr (NODE == SLG_NODE_WALSH) {
      val[NLEAF + i] = gen_node<NODE, 2>(val + 2 * i, par + 4 * i);
    } else {  // the forward's on LDS
      const float* c = par + 4 * i;
      const float a = val[2 * i], b = val[2 * i + 1];
      val[NLEAF + i] = fmaf(b, fmaf(a, c[3], c[2]), fmaf(a, c[1], c[0]));
    }
  }
  float gv[NLEAF + NN];
  gv[NLEAF + NN - 1] = g;
#pragma unroll
  for (int i = NN - 1; i >= 0; --i) {
    const float a = val[2 * i], b = val[2 * i + 1];
    const float* c = par + 4 * i;
    float U = gv[NLEAF + i];
    if constexpr (NODE == SLG_NODE_WALSH) {
      const float y = val[NLEAF + i];
      U *= y * (1.0f - y);
    }
    const float Ua = U * a;
    acc[4 * i] += U;
    acc[4 * i + 1] += Ua;
    acc[4 * i + 2] = fmaf(U, b, acc[4 * i + 2]);
    acc[4 * i + 3] = fmaf(Ua, b, acc[4 * i + 3]);
    gv[2 * i] = U * fmaf(c[3], b, c[1]);
    gv[2 * i + 1] = U * fmaf(c[3], a, c[2]);
  }
#pragma unroll
  for (int l = 0; l < NLEAF; ++l) gl[l] = gv[l];
}

// Leaf gradients of a LUT node's multilinear form, by one depth-first walk of
// its lerp tree over the leaves: a node's path weight U (the upstream
// gradient times v or 1 - v of the leaves above it) goes down, its value
// comes up, and its children's difference times U is its leaf's gradient.
// Few values are live at a time (level by level, LUT6 trees spilled). `pair`
// holds the table as (even corner, odd - even); acc the corner gradients
// g * prod(v or 1 - v).
template <int A, int J, int I>
__device__ __forceinline__ float sm_lut_node(const float (&v)[A], const float (&u)[A],
                                             SmWords pair, float U,
                                             float (&gl)[A], float (&acc)[1 << A]) {
  if constexpr (J == 0) {
    const float s = __uint_as_float(pair[2 * I]), d = __uint_as_float(pair[2 * I + 1]);
    acc[2 * I] = fmaf(U, u[0], acc[2 * I]);
    acc[2 * I + 1] = fmaf(U, v[0], acc[2 * I + 1]);
    gl[0] = fmaf(U, d, gl[0]);
    return fmaf(v[0], d, s);
  } else {
    const float t0 = sm_lut_node<A, J - 1, 2 * I>(v, u, pair, U * u[J], gl, acc);
    if constexpr (J >= 3 && A >= 6) __builtin_amdgcn_sched_barrier(0);  // keep the walk's order
    const float t1 = sm_lut_node<A, J - 1, 2 * I + 1>(v, u, pair, U * v[J], gl, acc);
    const float d = t1 - t0;
    gl[J] = fmaf(U, d, gl[J]);
    return fmaf(v[J], d, t0);
  }
}

template <int A>
__device__ inline void sm_grad_lut(const float (&v)[A], SmWords pair, float g,
                                   float (&gl)[A], float (&acc)[1 << A]) {
  float u[A];
#pragma unroll
  for (int j = 0; j < A; ++j) {
    u[j] = 1.0f - v[j];
    gl[j] = 0.0f;
  }
  sm_lut_node<A, A - 1, 0>(v, u, pair, g, gl, acc);
}

// Sum over the 64 lanes, in lane 63 (a fixed order on every call).
__device__ inline float wave_sum63(float v) {
#define SLG_DPP(ctrl, rows)                                                                   \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rows, 0xf, false))
  SLG_DPP(0x111, 0xf);  // row_shr:1
  SLG_DPP(0x112, 0xf);  // row_shr:2
  SLG_DPP(0x114, 0xf);  // row_shr:4
  SLG_DPP(0x118, 0xf);  // row_shr:8
  SLG_DPP(0x142, 0xa);  // row_bcast:15
  SLG_DPP(0x143, 0xc);  // row_bcast:31
#undef SLG_DPP
  return v;
}

// The wave's job (a workgroup is one wave): (tree, row split, chunk group);
// trees innermost, so the waves of one XCD work on few chunks and rows at a
// time (their images stay in its L2).
struct SmJob {
  int n, rs, cg;
};
__device__ inline bool sm_job(const SmArgs& a, SmJob& j) {
  const unsigned l = xcd_logical_id(blockIdx.x, gridDim.x);
  const unsigned q = l / (unsigned)a.N;
  j.n = (int)(l - q * (unsigned)a.N);
  j.cg = (int)(q / (unsigned)a.PS);
  j.rs = (int)(q - (unsigned)j.cg * a.PS);
  return j.cg < a.ncg;
}

__device__ inline float sm_load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

// A tree's window in LDS: (kernel + 1) rows and columns of its (at most two)
// channels for 64 samples, [channel][column slot][row][64]; column x of the
// bordered image sits in slot x mod (kernel + 1). Stepping to the next pooled
// output replaces the two oldest columns: 16 loads of 256 bytes for a 3 x 3
// kernel, where its taps' 4 window positions are 64 loads (gate16 trees of
// depth 2) or 96 (LUT6) and the caches deliver 64 bytes a clock and CU at
// best, a quarter of what the FMAs take (half of it missed L1: 64-96 waves'
// windows of 8 KB against 32 KB). Lane = bank, so reads of a different pixel
// in every lane do not conflict either.
struct SmRing {
  float* ring;
  __amdgpu_buffer_rsrc_t xr;
  int lane, wp, row1, RC, ch0, ch1;
  bool k3;

  __device__ SmRing(const SmArgs& a, const uint32_t* chan, float* lds, int lane_)
      : ring(lds), lane(lane_), wp(a.Wp), row1(a.Wp * 256), RC(a.kernel + 1),
        ch0((int)chan[0] * a.Hp * a.Wp * 256), ch1((int)chan[1] * a.Hp * a.Wp * 256),
        k3(a.kernel == 3) {
    ring[2 * RC * RC * 64 + lane] = 0.0f;  // read by the candidates past K
    ring[2 * RC * RC * 64 + 64 + lane] = 0.0f;
  }
  // image columns [col, col + n) of window row py into slots slot..
  __device__ void fill(int py, int col, int slot, int n) {
    for (int i = 0; i < n; ++i) {
      const int so = (2 * py * wp + col + i) * 256;
      for (int r = 0; r < RC; r += 2) {
        float t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          t[u] = sm_load(xr, lane * 4, so + (r + (u & 1)) * row1 + ((u >> 1) ? ch1 : ch0));
#pragma unroll
        for (int u = 0; u < 4; ++u)
          ring[(((u >> 1) * RC + slot + i) * RC + r + (u & 1)) * 64 + lane] = t[u];
      }
    }
  }
  // two columns of a 3 x 3 kernel's window: 16 loads in flight
  __device__ void load2(int py, int col, float (&t)[16]) const {
    const int so = (2 * py * wp + col) * 256;
#pragma unroll
    for (int u = 0; u < 16; ++u)
      t[u] = sm_load(xr, lane * 4 + ((u >> 2) & 1) * 256, so + (u & 3) * row1 + ((u >> 3) ? ch1 : ch0));
  }
  __device__ void put2(int slot, const float (&t)[16]) {
#pragma unroll
    for (int u = 0; u < 16; ++u)
      ring[((u >> 3) * 4 + slot + ((u >> 2) & 1)) * 256 + (u & 3) * 64 + lane] = t[u];
  }
  __device__ void first(int py) {  // the first window of a row
    if (k3) {
      float t0[16], t1[16];
      load2(py, 0, t0);
      load2(py, 2, t1);
      put2(0, t0);
      put2(2, t1);
    } else {
      fill(py, 0, 0, RC);
    }
  }
  // the next window: issue its loads, then (after the current one's reads)
  // place them over the oldest columns, slots 2 phase and 2 phase + 1
  __device__ void ahead(int py, int px, float (&t)[16]) const {
    if (k3) load2(py, 2 * px + 4, t);
  }
  __device__ void place(int py, int px, int phase, const float (&t)[16]) {
    if (k3) put2(2 * phase, t);
    else fill(py, 2 * px + RC, 2 * phase, 2);
  }
};

// The leaf sums at the four window positions, from the ring (taps rg of the
// current phase) or through the caches: the forward's order, candidate by
// candidate.
template <int NLEAF, int KM, typename Off, typename Get>
__device__ inline void sm_window_sums(float (&v)[4][NLEAF], SmWords wt, Off off, Get get) {
#pragma unroll
  for (int k = 0; k < KM; ++k) {
#pragma unroll
    for (int l = 0; l < NLEAF; ++l) {
      const uint32_t o = off(l * KM + k);
      const float wk = __uint_as_float(wt[l * KM + k]);
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q][l] = fmaf(wk, get(o, q), k ? v[q][l] : 0.0f);
    }
  }
}

template <int NODE, int NLEAF, int KM>
__device__ inline void sm_window(float (&v)[4][NLEAF], SmWords rc, bool rings,
                                 const SmRing& rg, int phase, int base) {
  using R = SmRec<NODE, NLEAF, KM>;
  if (rings) {
    SmWords A = rc + R::ring + phase * R::LK;
    sm_window_sums<NLEAF, KM>(v, rc + R::wt, [&](int i) { return A[i]; }, [&](uint32_t o, int q) {
      return rg.ring[((q & 1) ? o >> 16 : o & 0xffffu) / 4 + (q >> 1) * 64 + rg.lane];
    });
  } else {
    sm_window_sums<NLEAF, KM>(v, rc + R::wt, [&](int i) { return rc[R::off + i]; },
                              [&](uint32_t o, int q) {
      return sm_load(rg.xr, rg.lane * 4 + (q & 1) * 256, (int)o + base + (q >> 1) * rg.row1);
    });
  }
}

// The first window position holding the maximum.
template <int NODE, int NLEAF, bool LDS = sm_lds_form<NODE>()>
__device__ inline int sm_first_max(const float (&v)[4][NLEAF], const float* par) {
  float best = tree_eval<NODE, NLEAF, LDS>(v[0], par);
  int qs = 0;
#pragma unroll
  for (int q = 1; q < 4; ++q) {
    const float val = tree_eval<NODE, NLEAF, LDS>(v[q], par);
    if (val > best) {
      best = val;
      qs = q;
    }
  }
  return qs;
}

// Trees whose evaluation and backward together pass the registers: LUTs of 5
// and 6 leaves (32-64 parameters, 56-112 sums) find their window positions
// in a launch of their own. So do gate16 trees and LUTs whose forward runs
// through the caches.
template <int NODE, int NLEAF>
constexpr bool sm_split() { return !SmTree<NODE, NLEAF>::kBinary && NLEAF >= 5; }

// Window position of every (tree, pooled output, sample): the tree evaluated
// at the four positions with the operations of the forward of its sizes
// (tree_eval), the first maximum kept. Two bits per output, the U outputs of a
// step of a row to a word, route [nc][N][Ho][RW][64].
template <int NODE, int NLEAF, int KM, bool LDS>
__global__ void __launch_bounds__(64)
sm_route_kernel(SmArgs a, const uint32_t* __restrict__ recs, const float* __restrict__ xT,
                uint32_t* __restrict__ route) {
  using R = SmRec<NODE, NLEAF, KM>;
  using T = SmTree<NODE, NLEAF>;
  extern __shared__ __align__(16) float lds[];
  SmJob job;
  if (!sm_job(a, job)) return;
  const int lane = threadIdx.x;
  const uint32_t* rec = recs + (int64_t)job.n * a.RS;
  // parameters in vector registers (a tree FMA would take two scalars); a
  // hybrid LUT is looked up in memory
  const float* pv = reinterpret_cast<const float*>(rec) + R::par;
  float par[T::NP];
  if constexpr (NODE != SLG_NODE_HYBRID) {
    int zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
#pragma unroll
    for (int i = 0; i < T::NP; ++i) par[i] = pv[zero + i];
  }
  const bool rings = rec[R::chan + 2] == 0;
  SmRing rg(a, rec + R::chan, lds, lane);
  const int y0 = job.rs * a.RPS, y1 = min(a.Ho, y0 + a.RPS);
  for (int c = job.cg; c < a.nc; c += a.ncg) {
    rg.xr = uniform_rsrc(xT + (int64_t)c * a.xs, (int)(a.xs * 4));
    uint32_t* rp = route + ((int64_t)c * a.N + job.n) * a.Ho * a.RW * 64 + lane;
    for (int py = y0; py < y1; ++py) {
      uint32_t word = 0;
      int phase = 0, u = 0, step = 0;
      if (rings) rg.first(py);
      for (int px = 0; px < a.Wo; ++px) {
        float nx[16], v[4][NLEAF];
        const bool more = rings && px + 1 < a.Wo;
        if (more) rg.ahead(py, px, nx);
        sm_window<NODE, NLEAF, KM>(v, sm_words(rec), rings, rg, phase,
                                    2 * (py * a.Wp + px) * 256);
        const int qs = sm_first_max<NODE, NLEAF, LDS>(v, NODE == SLG_NODE_HYBRID ? pv : par);
        word |= (uint32_t)qs << (2 * u);
        if (++u == a.U || px == a.Wo - 1) {
          rp[(int64_t)(py * a.RW + step++) * 64] = word;
          word = 0;
          u = 0;
        }
        if (more) rg.place(py, px, phase, nx);
        phase = phase + 1 == rg.RC / 2 ? 0 : phase + 1;
      }
    }
  }
}

// Per (tree, output, sample) the tree's backward at the routed position.
// MODE 0: no pool; 1: pooled, the window position found here and, where gl
// is wanted, written as sm_route_kernel does; 2: pooled, routes read. Writes
// leaf gradients gl [nc][N][L][P][64] (null: not wanted) and the job's
// weight and parameter gradient sums part_w [slot][N*L*K], part_np
// [slot][N*NP], slot = cg * PS + rs of this round.
template <int NODE, int NLEAF, int KM, int MODE>
__global__ void __launch_bounds__(64, 2)
sm_grad_kernel(SmArgs a, const uint32_t* __restrict__ recs, const float* __restrict__ xT,
               const float* __restrict__ gT, uint32_t* __restrict__ route,
               float* __restrict__ gl_out, float* __restrict__ part_w,
               float* __restrict__ part_np) {
  using R = SmRec<NODE, NLEAF, KM>;
  using T = SmTree<NODE, NLEAF>;
  constexpr int LK = NLEAF * KM;
  constexpr int S = MODE ? 2 : 1;
  extern __shared__ __align__(16) float lds[];
  SmJob job;
  if (!sm_job(a, job)) return;
  const int lane = threadIdx.x;
  const uint32_t* rec = recs + (int64_t)job.n * a.RS;
  // a binary tree's parameters in vector registers (its FMAs take two of them)
  float par[T::kBinary ? T::NP : 1];
  if constexpr (T::kBinary) {
    int zero;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
#pragma unroll
    for (int i = 0; i < T::NP; ++i) par[i] = reinterpret_cast<const float*>(rec)[R::par + zero + i];
  }
  float accw[LK], accn[T::NP];
#pragma unroll
  for (int i = 0; i < LK; ++i) accw[i] = 0.0f;
#pragma unroll
  for (int i = 0; i < T::NP; ++i) accn[i] = 0.0f;
  const bool rings = MODE != 0 && rec[R::chan + 2] == 0;
  SmRing rg(a, rec + R::chan, lds, lane);
  const int y0 = job.rs * a.RPS, y1 = min(a.Ho, y0 + a.RPS);
  for (int c = job.cg; c < a.nc; c += a.ncg) {
    if (lane >= a.B - c * 64) break;  // lanes past the batch (of the last chunk)
    rg.xr = uniform_rsrc(xT + (int64_t)c * a.xs, (int)(a.xs * 4));
    const float* gp = gT + ((int64_t)c * a.N + job.n) * a.P * 64 + lane;
    uint32_t* rp = route + ((int64_t)c * a.N + job.n) * a.Ho * a.RW * 64 + lane;
    float* go = gl_out ? gl_out + ((int64_t)c * a.N + job.n) * NLEAF * a.P * 64 + lane : nullptr;
    for (int py = y0; py < y1; ++py) {
      uint32_t word = 0;
      int phase = 0, u = 0, step = 0;
      if (rings) rg.first(py);
      for (int px = 0; px < a.Wo; ++px) {
        const int p = py * a.Wo + px;
        const float g = gp[(int64_t)p * 64];
        const int base = S * (py * a.Wp + px) * 256;
        float nx[16];
        const bool more = rings && px + 1 < a.Wo;
        if (more) rg.ahead(py, px, nx);
        SmWords rc = sm_words(rec);
        int qs = 0;
        if constexpr (MODE == 1) {
          float v[4][NLEAF];
          sm_window<NODE, NLEAF, KM>(v, rc, rings, rg, phase, base);
          if constexpr (T::kBinary) {
            qs = sm_first_max<NODE, NLEAF>(v, par);
          } else if constexpr (NODE == SLG_NODE_HYBRID) {  // looked up in memory
            qs = sm_first_max<NODE, NLEAF>(v, reinterpret_cast<const float*>(rec) + R::par);
          } else {
            float pr[T::NP];
#pragma unroll
            for (int i = 0; i < T::NP; ++i) pr[i] = __uint_as_float(rc[R::par + i]);
            qs = sm_first_max<NODE, NLEAF>(v, pr);
          }
          word |= (uint32_t)qs << (2 * u);
          if (++u == a.U || px == a.Wo - 1) {
            if (go) rp[(int64_t)(py * a.RW + step++) * 64] = word;
            word = 0;
            u = 0;
          }
          rc = sm_words(rec);
        } else if constexpr (MODE == 2) {
          if (u == 0) word = rp[(int64_t)(py * a.RW + step++) * 64];
          if (++u == a.U) u = 0;
          qs = (int)(word & 3u);
          word >>= 2;
        }
        // the routed position's tap values and leaf sums
        float v[NLEAF], x[LK], gl[NLEAF];
        const bool qx = qs & 1, qy = qs & 2;
        if (rings) {
          SmWords A = rc + R::ring + phase * LK;
          const int lo = lane + (qy ? 64 : 0);
#pragma unroll
          for (int i = 0; i < LK; ++i)
            x[i] = lds[(int)((qx ? A[i] >> 16 : A[i] & 0xffffu) / 4) + lo];
        } else {
          const int voff = lane * 4 + (qx ? 256 : 0) + (qy ? rg.row1 : 0);
#pragma unroll
          for (int i = 0; i < LK; ++i) x[i] = sm_load(rg.xr, voff, (int)rc[R::off + i] + base);
        }
#pragma unroll
        for (int k = 0; k < KM; ++k)
#pragma unroll
          for (int l = 0; l < NLEAF; ++l)
            v[l] = fmaf(__uint_as_float(rc[R::wt + l * KM + k]), x[l * KM + k], k ? v[l] : 0.0f);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (T::kBinary) {
          sm_grad_binary<NODE, NLEAF>(v, par, g, gl, accn);
        } else {
          sm_grad_lut<NLEAF>(v, sm_words(rec) + R::pair, g, gl, accn);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int l = 0; l < NLEAF; ++l) {
          if (go) go[((int64_t)l * a.P + p) * 64] = gl[l];
#pragma unroll
          for (int k = 0; k < KM; ++k)
            accw[l * KM + k] = fmaf(gl[l], x[l * KM + k], accw[l * KM + k]);
        }
        if (more) rg.place(py, px, phase, nx);
        phase = phase + 1 == rg.RC / 2 ? 0 : phase + 1;
      }
    }
  }
  const int64_t slot = (int64_t)job.cg * a.PS + job.rs;
  float* pw = part_w + (slot * a.N + job.n) * NLEAF * a.K;
  float* pn = part_np + (slot * a.N + job.n) * T::NP;
#pragma unroll
  for (int l = 0; l < NLEAF; ++l)
#pragma unroll
    for (int k = 0; k < KM; ++k) {
      const float s = wave_sum63(accw[l * KM + k]);
      if (k < a.K && lane == 63) pw[l * a.K + k] = s;
    }
#pragma unroll
  for (int i = 0; i < T::NP; ++i) {
    const float s = wave_sum63(accn[i]);
    if (lane == 63) pn[i] = s;
  }
}

// Input gradient: a wave owns TH image rows of one channel for 64 samples,
// [TH][Wp][64] in LDS (lane = bank, so 64 lanes at 64 different pixels do
// not conflict), and adds the channel's taps to it in table order. For one
// tap the outputs' target pixels are distinct, so a row's U outputs are
// read, added and written together; the wave's LDS operations stay in order,
// so no barrier separates the taps. Taps of one leaf share its gradients
// (NR rows x U outputs in registers); the next leaf's loads are in flight
// while this one's taps are added. Rows no tap of the leaf sends to the
// strip are not loaded (an offset past the buffer reads 0). U outputs divide
// the map's rows into equal steps; where they do not, the last step starts
// early; the outputs it repeats, and those routed to a row outside the strip,
// add to a per-lane dump slot. Few strips of long lists (few channels under
// many trees) would leave the chip idle: the list is then split over GS waves,
// part 0 into gx, the others into images that sm_gx_sum adds in order (11
// channels under 216 depth-3 trees, 12x12, 5x5, B = 126: 132 waves, 685 us
// unsplit).
template <bool POOL, int U, int NR>
__global__ void __launch_bounds__(64)
sm_gx_kernel(SmArgs a, int NLEAF, const int* __restrict__ start, const SmRef* __restrict__ refs,
             const float* __restrict__ gl, const uint32_t* __restrict__ route,
             float* __restrict__ gx, float* __restrict__ parts) {
  extern __shared__ __align__(16) float tile[];
  constexpr int S = POOL ? 2 : 1;
  const unsigned lid = xcd_logical_id(blockIdx.x, gridDim.x);
  const unsigned cs = lid / (unsigned)a.C;
  const int c = (int)(lid - cs * (unsigned)a.C);
  const unsigned cp = cs / (unsigned)a.nt;
  const int strip = (int)(cs - cp * (unsigned)a.nt);
  const int chunk = (int)(cp / (unsigned)a.GS), part = (int)(cp - (unsigned)chunk * a.GS);
  if (chunk >= a.nc) return;
  const int lane = threadIdx.x;
  const int r0 = strip * a.TH, rows = min(a.TH, a.H - r0);
  const int rw = a.Wp * 64;  // floats per tile row
  for (int i = lane * 4; i < rows * rw; i += 256)
    *reinterpret_cast<float4*>(tile + i) = make_float4(0.f, 0.f, 0.f, 0.f);
  __syncthreads();
  const int dump = a.TH * rw + lane;  // float index of the lane's dump slot
  // outputs whose window can reach rows r0 .. r0 + rows - 1: the image row of
  // output py, window row q, tap row dh is S py + q + dh - pad
  const int py_lo = max(0, (r0 + a.pad - a.kernel + 1 - (S - 1) + S * 8) / S - 8);
  const int py_hi = min(a.Ho - 1, (r0 + rows - 1 + a.pad) / S);
  const int j_first = start[c], nj = start[c + 1] - j_first, per = (nj + a.GS - 1) / a.GS;
  const int j_begin = j_first + min(part * per, nj), j_end = j_first + min((part + 1) * per, nj);
  const int leaf_bytes = a.P * 256, row_bytes = a.RW * 256;
  const auto gr = uniform_rsrc(gl + (int64_t)chunk * a.N * NLEAF * a.P * 64, a.N * NLEAF * leaf_bytes);
  const auto rr = uniform_rsrc(POOL ? (const void*)(route + (int64_t)chunk * a.N * a.Ho * a.RW * 64) : gl,
                               POOL ? a.N * a.Ho * row_bytes : 0);
  const auto ref = [&](int j) {  // scalar loads
    const SmWords w = (SmWords)(uint64_t)refs + 4 * (int64_t)j;
    SmRef e;
    e.tree = (int)w[0];
    e.next = (int)w[1];
    e.d = w[2];
    e.w = __uint_as_float(w[3]);
    return e;
  };

  struct Run {  // a leaf's taps: its loads (issued by fetch) and their use (add)
    int j0, j1;
    SmRef e;  // the first tap
    float g[NR][U];
    uint32_t word[NR];
  };
  int qo[NR][U];       // window offset of each output (floats), of tree qt
  int qt = -1;
  // branch-free, so that the waits for a run's loads count the next run's
  auto fetch = [&](Run& r, int j, int py, int p0, int px, int step) {
    const bool any = j < j_end;
    const SmRef e = ref(any ? j : 0);
    r.j0 = j;
    r.j1 = any ? min(e.next, j_end) : j;
    r.e = e;
    const int lo = (int)(e.d >> 8) & 15, hi = (int)(e.d >> 12) & 15;
    const int gbase = (e.tree * NLEAF + (int)(e.d >> 16)) * leaf_bytes + px * 256;
    const int rbase = e.tree * a.Ho * row_bytes + step * 256;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      // rows S y + [0, S) + [lo, hi] - pad against the strip
      const int y = py + i, top = S * y + lo - a.pad - r0, bot = S * y + S - 1 + hi - a.pad - r0;
      const bool need = any && y <= py_hi && bot >= 0 && top < rows;
      const int yc = min(y, a.Ho - 1), so = gbase + yc * a.Wo * 256;
      const int voff = need ? lane * 4 : 0x7fffe000;
#pragma unroll
      for (int u = 0; u < U; ++u) r.g[i][u] = sm_load(gr, voff + u * 256, so);
      if constexpr (POOL)
        r.word[i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rr, lane * 4, rbase + yc * row_bytes, 0);
    }
  };
  auto add = [&](const Run& r, int py, int p0, int px) {
    if (POOL && qt != r.e.tree) {
      qt = r.e.tree;
      const int early = 2 * (p0 - px);  // bits of the outputs a step repeats
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t q = (r.word[i] << early) >> (2 * u);
          qo[i][u] = lane + u * S * 64 + (int)((q & 1u) << 6) + ((q & 2u) ? rw : 0);
        }
    }
    SmRef e = r.e;
    for (int j = r.j0; j < r.j1; ++j) {
      const SmRef en = ref(j + 1);  // the entry past the table is there, unused
      const int dh = (int)(e.d & 15u), dw = (int)(e.d >> 4) & 15;
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        const int ly = S * (py + i) + dh - a.pad - r0;  // tile row of window row 0
        if (py + i > py_hi || ly <= -S || ly >= rows) continue;  // uniform
        const int at = ly * rw + (S * px + dw) * 64;
        int ad[U];
        float old[U];
#pragma unroll
        for (int u = 0; u < U; ++u) ad[u] = at + (POOL ? qo[i][u] : lane + u * 64);
        if (POOL && (ly < 0 || ly + S > rows)) {  // one window row in the strip: lanes routed to it
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const bool second = qo[i][u] >= lane + u * S * 64 + rw;
            ad[u] = second == (ly < 0) ? ad[u] : dump;
          }
        }
        if (px < p0) {  // outputs of the step before
#pragma unroll
          for (int u = 0; u < U; ++u) ad[u] = px + u < p0 ? dump : ad[u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) old[u] = tile[ad[u]];
#pragma unroll
        for (int u = 0; u < U; ++u) old[u] = fmaf(e.w, r.g[i][u], old[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) tile[ad[u]] = old[u];
      }
      e = en;
    }
  };
  for (int py = py_lo; py <= py_hi; py += NR) {
    for (int step = 0; step < a.RW; ++step) {
      const int p0 = step * U, px = min(p0, a.Wo - U);  // U <= Wo
      qt = -1;
      Run ra, rb;
      fetch(ra, j_begin, py, p0, px, step);
      while (ra.j0 < j_end) {
        fetch(rb, ra.j1, py, p0, px, step);
        add(ra, py, p0, px);
        if (rb.j0 >= j_end) break;
        fetch(ra, rb.j1, py, p0, px, step);
        add(rb, py, p0, px);
      }
    }
  }
  __syncthreads();
  // the strip's pixels (W of each row) to gx: 16 pixels x 16 sample quads a
  // step, four samples per lane read as one float4
  const int b0 = chunk * 64;
  const int px16 = lane & 15, quad = lane >> 4;
  const int64_t CHW = (int64_t)a.C * a.H * a.W;
  float* dst = (part ? parts + (part - 1) * (a.B * CHW) : gx) + ((int64_t)c * a.H + r0) * a.W;
  const int n = rows * a.W;
  for (int i0 = 0; i0 < n; i0 += 16) {
    const int i = i0 + px16;
    const int yy = i / a.W, xx = i - yy * a.W;
    if (i < n) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int s = (k * 4 + quad) * 4;
        const float4 v = *reinterpret_cast<const float4*>(tile + yy * rw + (xx + a.pad) * 64 + s);
        const float f[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (b0 + s + q < a.B) dst[(int64_t)(b0 + s + q) * CHW + i] = f[q];
      }
    }
  }
}

// gx[i] += the parts' images, in order.
__global__ void __launch_bounds__(256) sm_gx_sum_kernel(const float* __restrict__ parts, int n_parts,
                                                        int64_t n, float* __restrict__ gx) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = gx[i];
  for (int p = 0; p < n_parts; ++p) s += parts[p * n + i];
  gx[i] = s;
}

// gw[i] = sum over slots s of part_w[s][i], gnp likewise: a workgroup takes
// 16 columns; its 16 thread rows sum the slots s = row (mod 16) in ascending
// order, and the 16 row sums are added in row order.
__global__ void __launch_bounds__(256) sm_sum_kernel(const float* __restrict__ part_w, int64_t nw,
                                                     float* __restrict__ gw,
                                                     const float* __restrict__ part_np, int64_t nn,
                                                     float* __restrict__ gnp, int64_t slots) {
  __shared__ float rs[16][17];
  const int col = threadIdx.x & 15, row = threadIdx.x >> 4;
  const int64_t wb = gw ? (nw + 15) / 16 : 0;
  const bool first = (int64_t)blockIdx.x < wb;
  const float* part = first ? part_w : part_np;
  const int64_t n = first ? nw : nn;
  float* out = first ? gw : gnp;
  const int64_t i = ((int64_t)blockIdx.x - (first ? 0 : wb)) * 16 + col;
  float s = 0.0f;
  if (i < n)
    for (int64_t r = row; r < slots; r += 16) s += part[r * n + i];
  rs[row][col] = s;
  __syncthreads();
  if (row == 0 && i < n) {
    float t = 0.0f;
#pragma unroll
    for (int q = 0; q < 16; ++q) t += rs[q][col];
    out[i] = t;
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Dispatch over (node, leaves, candidates) with integral constants.
template <typename F>
static int sm_dispatch(int node, int depth, int arity, int K, F&& f) {
  const bool binary = node == SLG_NODE_GATE16 || node == SLG_NODE_WALSH;
  const int nleaf = binary ? (depth >= 1 && depth <= 3 ? 1 << depth : -1)
                           : (depth == 1 && arity >= 2 && arity <= 6 ? arity : -1);
  if (K < 1 || K > kSmMaxK) return SLG_E_UNSUPPORTED;
#define SLG_SM(NODE_, NL_)                                                                     \
  if (node == NODE_ && nleaf == NL_)                                                           \
    return K <= 4 ? f(std::integral_constant<int, NODE_>{}, std::integral_constant<int, NL_>{}, \
                      std::integral_constant<int, 4>{})                                        \
                  : f(std::integral_constant<int, NODE_>{}, std::integral_constant<int, NL_>{}, \
                      std::integral_constant<int, kSmMaxK>{});
  SLG_SM(SLG_NODE_GATE16, 2)
  SLG_SM(SLG_NODE_GATE16, 4)
  SLG_SM(SLG_NODE_GATE16, 8)
  SLG_SM(SLG_NODE_WALSH, 2)
  SLG_SM(SLG_NODE_WALSH, 4)
  SLG_SM(SLG_NODE_WALSH, 8)
  SLG_SM(SLG_NODE_MULTILINEAR2, 2)
  SLG_SM(SLG_NODE_MULTILINEAR2, 3)
  SLG_SM(SLG_NODE_MULTILINEAR2, 4)
  SLG_SM(SLG_NODE_MULTILINEAR2, 5)
  SLG_SM(SLG_NODE_MULTILINEAR2, 6)
  SLG_SM(SLG_NODE_HYBRID, 2)
  SLG_SM(SLG_NODE_HYBRID, 3)
  SLG_SM(SLG_NODE_HYBRID, 4)
  SLG_SM(SLG_NODE_HYBRID, 5)
  SLG_SM(SLG_NODE_HYBRID, 6)
#undef SLG_SM
  return SLG_E_UNSUPPORTED;
}

static inline int64_t sm_round(int64_t n) { return (n + 63) & ~int64_t(63); }

struct SmPlan {
  SmArgs a;
  int64_t nc_total;  // chunks over all rounds; a.nc per round
  int64_t slots;     // partial slots over all rounds
  int nleaf, nparam, rec_words;
  // workspace offsets (4-byte words, multiples of 64)
  int64_t recs, start, refs, xT, gT, route, gl, pw, pn, parts, total;
};

// A round's leaf gradients and its workspace in floats, at most, or one chunk
// of 64 samples whatever that takes.
static constexpr int64_t kSmRoundLeaves = int64_t(64) << 20, kSmRoundFloats = int64_t(96) << 20;
static constexpr int64_t kSmJobs = 4096;                      // waves that fill the chip

static bool sm_plan(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node, int depth,
                    int arity, int K, int pad, bool pool, bool want_x, SmPlan& p) {
  p = SmPlan{};
  const int rc = sm_dispatch(node, depth, arity, K, [&](auto nd, auto nl, auto km) {
    constexpr int NODE = decltype(nd)::value, NL = decltype(nl)::value, KM = decltype(km)::value;
    p.nleaf = NL;
    p.nparam = SmTree<NODE, NL>::NP;
    p.rec_words = SmRec<NODE, NL, KM>::words(2 * pad + 1);
    p.a.RS = p.rec_words;
    p.a.Cz = (int)C + (K < KM ? 1 : 0);
    return 0;
  });
  if (rc) return false;
  const int64_t Hp = H + 2 * pad, Wp = W + 2 * pad;
  const int64_t Ho = pool ? H / 2 : H, Wo = pool ? W / 2 : W, P = Ho * Wo;
  // 32-bit byte offsets into one chunk of the image, an image row in LDS
  const int64_t cap = std::min(device_lds_bytes(), 160 * 1024);
  if (P < 1 || B < 1 || (C + 1) * Hp * Wp >= (1LL << 23) || N * P >= (1LL << 30) ||
      N >= (1LL << 20) || N * p.rec_words >= (1LL << 31) || (Wp + 1) * 256 > cap ||
      N * p.nleaf * P * 256 >= (1LL << 31) - 65536)
    return false;
  SmArgs& a = p.a;
  a.B = (int)B; a.C = (int)C; a.H = (int)H; a.W = (int)W; a.Hp = (int)Hp; a.Wp = (int)Wp;
  a.N = (int)N; a.K = K; a.kernel = 2 * pad + 1; a.pad = pad;
  a.Ho = (int)Ho; a.Wo = (int)Wo; a.P = (int)P;
  a.RW = (int)cdiv(Wo, 8);
  a.U = (int)cdiv(Wo, a.RW);
  a.RW = (int)cdiv(Wo, a.U);
  a.xs = a.Cz * Hp * Wp * 64;
  p.nc_total = cdiv(B, 64);
  const int64_t gl1 = N * p.nleaf * P * 64;
  const int64_t chunk = gl1 + a.xs + N * (P + Ho * a.RW) * 64;  // with its images and routes
  a.nc = (int)std::max<int64_t>(1, std::min({p.nc_total, kSmRoundLeaves / gl1, kSmRoundFloats / chunk}));
  // rows split until the jobs fill the chip; then several chunks to a job
  a.PS = (int)std::max<int64_t>(1, std::min<int64_t>(Ho, cdiv(kSmJobs, N * a.nc)));
  a.RPS = (int)cdiv(Ho, a.PS);
  a.PS = (int)cdiv(Ho, a.RPS);
  a.ncg = (int)std::max<int64_t>(1, std::min<int64_t>(a.nc, cdiv(2 * kSmJobs, N * a.PS)));
  // strips of at most 16 KB (ten waves a CU), two rows at least
  a.TH = (int)std::max<int64_t>((2 * Wp + 1) * 256 <= cap ? 2 : 1, 16384 / (Wp * 256) & ~1LL);
  // of two where strips of more rows would leave the chip idle
  if (a.TH > 2 && C * a.nc * cdiv(H, a.TH) < kSmJobs / 2) a.TH = 2;
  a.TH = (int)std::min<int64_t>(a.TH, H);
  a.nt = (int)cdiv(H, a.TH);
  // parts of the taps while waves are missing, of 32 taps at least on average
  a.GS = (int)std::max<int64_t>(1, std::min<int64_t>({16, kSmJobs / 2 / (C * a.nc * a.nt),
                                                      N * p.nleaf * K / (32 * C)}));
  const int64_t rounds = cdiv(p.nc_total, a.nc);
  p.slots = rounds * a.ncg * a.PS;
  int64_t o = 0;
  auto take = [&](int64_t words) {
    const int64_t at = o;
    o += sm_round(words);
    return at;
  };
  // the rounds do not follow want_x: the weight sums keep their order (and bits)
  const int64_t gx = want_x;
  p.recs = take(N * p.rec_words);
  p.start = take(gx * (C + 1));
  p.refs = take(gx * (N * p.nleaf * K + 1) * 4);
  p.xT = take(a.nc * a.xs);
  p.gT = take(a.nc * N * P * 64);
  p.route = take(pool ? a.nc * N * Ho * a.RW * 64 : 0);
  p.gl = take(gx * a.nc * gl1);
  p.pw = take(p.slots * N * p.nleaf * K);
  p.pn = take(p.slots * N * p.nparam);
  p.parts = take(gx * (a.GS - 1) * std::min<int64_t>(B, a.nc * int64_t(64)) * C * H * W);
  p.total = o;
  return true;
}

// Estimated microseconds of a call that wants every gradient (conv_bwd.hip).
static double sm_us(const SmPlan& p, bool binary, bool pool) {
  const SmArgs& a = p.a;
  const int S = pool ? 2 : 1, visits = pool ? 5 : 1, L = p.nleaf;
  const double cus = device_cus(), rounds = (double)cdiv(p.nc_total, a.nc), chunks = (double)p.nc_total;
  const double taps = (double)a.N * L * a.K, refs = taps / a.C;
  // sm_grad and sm_route, per output: tap reads and evaluations at the window
  // positions and the routed one, the window ring's new columns (those of other
  // than 3 x 3 kernels four loads at a time). The outputs of a wave, one after
  // the other, and all of them on the chip's waves.
  const double tap = L * (a.K <= 4 ? 4 : kSmMaxK) * visits, eval = (binary ? 4 * (L - 1) : 1 << L) * visits;
  const double ring = pool ? a.kernel + 1 : 0, slow = a.kernel == 3 ? 0 : ring * (a.kernel + 1);
  const double own = rounds * a.RPS * a.Wo * cdiv(a.nc, a.ncg);
  const double all = (double)a.N * a.P * chunks / (8 * cus);
  const double grad = own * (0.025 * tap + 0.018 * eval + 0.26 * ring + 0.076 * slow) +
                      all * (0.0092 * eval + 0.31 * ring + 0.097 * slow);
  // sm_gx: a wave's references times its steps over the map, and all of them
  const int64_t resident = std::min<int64_t>(16, 160 * 1024 / (((int64_t)a.TH * a.Wp + 1) * 256));
  const int64_t rows = std::min<int64_t>(a.Ho, (a.TH + a.kernel + S - 2) / S + 1);
  const double steps = rounds * (refs / a.GS) * cdiv(rows, !pool || a.TH > 2 ? 4 : 3) * a.RW;
  const double waves = (double)a.C * a.nc * a.nt * a.GS / (cus * std::max<int64_t>(1, resident));
  const double gx = steps * (0.22 * (1 + 3 / sqrt(refs)) + 0.19 * waves);
  const double tables = 1e-6 * rounds * a.C * taps + 2.4e-3 * taps;
  const double memory = 64e-6 * chunks * (1.4 * ((double)a.C * a.Hp * a.Wp + (double)a.N * a.P) +
                                          1.3 * (double)a.N * L * a.P);
  return 1.5 + 2 * rounds + grad + gx + tables + memory;
}

int64_t conv_sm_bwd_workspace(int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                              int depth, int arity, int K, int pad, bool pool, bool want_x,
                              double* us) {
  SmPlan p;
  if (!sm_plan(std::max<int64_t>(B, 1), C, H, W, N, node, depth, arity, K, pad, pool, want_x, p))
    return -1;
  if (us) *us = sm_us(p, node == SLG_NODE_GATE16 || node == SLG_NODE_WALSH, pool);
  return p.total;
}

// sm_gx_kernel for rows in steps of u outputs.
using SmGxKernel = void (*)(SmArgs, int, const int*, const SmRef*, const float*, const uint32_t*,
                            float*, float*);
template <bool POOL, int NR>
static SmGxKernel sm_gx_rows(int u) {
  static const SmGxKernel k[8] = {sm_gx_kernel<POOL, 1, NR>, sm_gx_kernel<POOL, 2, NR>,
                                  sm_gx_kernel<POOL, 3, NR>, sm_gx_kernel<POOL, 4, NR>,
                                  sm_gx_kernel<POOL, 5, NR>, sm_gx_kernel<POOL, 6, NR>,
                                  sm_gx_kernel<POOL, 7, NR>, sm_gx_kernel<POOL, 8, NR>};
  return k[u - 1];
}
// Strips of two rows meet three rows of pooled outputs (3 x 3 kernels), of
// four rows four.
static SmGxKernel sm_gx_pick(bool pool, int u, int th) {
  if (!pool) return sm_gx_rows<false, 4>(u);
  return th <= 2 ? sm_gx_rows<true, 3>(u) : sm_gx_rows<true, 4>(u);
}

static int sm_sums(const float* pw, const float* pn, int64_t slots, int64_t nw, int64_t nn,
                   float* gw, float* gnp, hipStream_t st) {
  if (!gw && !gnp) return 0;
  const int64_t blocks = (gw ? cdiv(nw, 16) : 0) + (gnp ? cdiv(nn, 16) : 0);
  hipLaunchKernelGGL(sm_sum_kernel, dim3((unsigned)blocks), dim3(256), 0, st, pw, nw, gw, pn, nn, gnp,
                     slots);
  SLG_LAUNCH_CHECK("conv_soft_bwd sums");
  return 0;
}

int conv_sm_bwd(const float* x, int64_t B, int64_t C, int64_t H, int64_t W, int64_t N, int node,
                int depth, int arity, int K, int pad, bool pool, bool raw, const float* np,
                const float* w, const int* cm, const int* ch, const int* cw, const float* gy, float* gx,
                float* gw, float* gnp, float* ws, int64_t ws_floats, hipStream_t st) {
  SmPlan p;
  SLG_REQUIRE(sm_plan(B, C, H, W, N, node, depth, arity, K, pad, pool, gx != nullptr, p),
              SLG_E_UNSUPPORTED, "conv_soft_bwd: sizes outside the sample-minor kernels");
  SLG_REQUIRE(ws_floats >= p.total, SLG_E_ARG, "conv_soft_bwd: workspace of %lld floats, %lld needed",
              (long long)ws_floats, (long long)p.total);
  SmArgs a = p.a;
  a.raw = raw;
  const int64_t nw = N * p.nleaf * K, nn = N * p.nparam;
  uint32_t* recs = reinterpret_cast<uint32_t*>(ws + p.recs);
  int* start = reinterpret_cast<int*>(ws + p.start);
  SmRef* refs = reinterpret_cast<SmRef*>(ws + p.refs);
  uint32_t* route = pool ? reinterpret_cast<uint32_t*>(ws + p.route) : nullptr;
  float* gl = gx ? ws + p.gl : nullptr;
  {
    const int rc = sm_dispatch(node, depth, arity, K, [&](auto nd, auto nl, auto km) -> int {
      constexpr int NODE = decltype(nd)::value, NL = decltype(nl)::value, KM = decltype(km)::value;
      const int rb = (int)cdiv(N, 16);
      hipLaunchKernelGGL((sm_tables_kernel<NODE, NL, KM>), dim3((unsigned)(rb + (gx ? C : 0))),
                         dim3(1024), 0, st, a, rb, np, w, cm, ch, cw, recs, start, refs);
      SLG_LAUNCH_CHECK("conv_soft_bwd tables");
      for (int64_t c0 = 0, round = 0; c0 < p.nc_total; c0 += p.a.nc, ++round) {
        const int64_t b0 = c0 * 64;
        a.nc = (int)std::min<int64_t>(p.a.nc, p.nc_total - c0);
        a.B = (int)std::min<int64_t>(B - b0, (int64_t)a.nc * 64);
        const int64_t xt = cdiv((int64_t)a.Cz * a.Hp * a.Wp, 64), gt = cdiv(N * a.P, 64);
        SLG_REQUIRE(a.nc * (xt + gt) < (1LL << 31), SLG_E_SHAPE, "conv_soft_bwd: grid too large");
        hipLaunchKernelGGL(sm_images_kernel, dim3((unsigned)(a.nc * (xt + gt))), dim3(256), 0, st,
                           x + b0 * C * H * W, gy + b0 * N * a.P, a, (int)xt, (int)gt, ws + p.xT,
                           ws + p.gT);
        SLG_LAUNCH_CHECK("conv_soft_bwd images");
        const int64_t grid = cdiv(N * a.PS * a.ncg, 8) * 8;
        const int64_t s0 = round * p.a.ncg * a.PS;
        const size_t ring = (size_t)(2 * (a.kernel + 1) * (a.kernel + 1) + 2) * 256;
        constexpr bool kSplit = sm_split<NODE, NL>();
        constexpr bool kCache = NODE == SLG_NODE_GATE16 || NODE == SLG_NODE_MULTILINEAR2;
        auto grad = pool ? sm_grad_kernel<NODE, NL, KM, kSplit ? 2 : 1> : sm_grad_kernel<NODE, NL, KM, 0>;
        void (*find)(SmArgs, const uint32_t*, const float*, uint32_t*) = nullptr;
        if constexpr (kSplit) {
          if (pool) find = sm_route_kernel<NODE, NL, KM, true>;
        }
        if constexpr (kCache) {
          if (raw) {
            find = sm_route_kernel<NODE, NL, KM, false>;
            grad = sm_grad_kernel<NODE, NL, KM, 2>;
          }
        }
        if (find) {
          hipLaunchKernelGGL(find, dim3((unsigned)grid), dim3(64), ring, st, a, recs, ws + p.xT, route);
          SLG_LAUNCH_CHECK("conv_soft_bwd route");
        }
        hipLaunchKernelGGL(grad, dim3((unsigned)grid), dim3(64), ring, st, a, recs, ws + p.xT,
                           ws + p.gT, route, gl, ws + p.pw + s0 * nw, ws + p.pn + s0 * nn);
        SLG_LAUNCH_CHECK("conv_soft_bwd grad");
        if (gx) {
          const size_t lds = ((size_t)a.TH * a.Wp + 1) * 256;
          auto kern = sm_gx_pick(pool, a.U, a.TH);
          if (lds > 65536) {
            const hipError_t e = hipFuncSetAttribute(
                (const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            SLG_REQUIRE(e == hipSuccess, (int)e, "conv_soft_bwd: LDS %zu: %s", lds, hipGetErrorString(e));
          }
          const int64_t jobs = cdiv((int64_t)C * a.nc * a.nt * a.GS, 8) * 8;
          hipLaunchKernelGGL(kern, dim3((unsigned)jobs), dim3(64), lds, st, a, NL, start, refs, gl,
                             route, gx + b0 * C * H * W, ws + p.parts);
          SLG_LAUNCH_CHECK("conv_soft_bwd input gradient");
          if (a.GS > 1) {
            const int64_t n = (int64_t)a.B * C * H * W;
            hipLaunchKernelGGL(sm_gx_sum_kernel, dim3((unsigned)cdiv(n, 256)), dim3(256), 0, st,
                               ws + p.parts, a.GS - 1, n, gx + b0 * C * H * W);
            SLG_LAUNCH_CHECK("conv_soft_bwd input gradient parts");
          }
        }
      }
      return 0;
    });
    if (rc) return rc;
  }
  return sm_sums(ws + p.pw, ws + p.pn, p.slots, nw, nn, gw, gnp, st);
}

int conv_sm_zero_grads(int64_t N, int64_t lk, int64_t np, float* gw, float* gnp, hipStream_t st) {
  return sm_sums(nullptr, nullptr, 0, N * lk, N * np, gw, gnp, st);  // sums over no slots
}

}  // namespace slg
