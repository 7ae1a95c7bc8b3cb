// Input gradient of the FC soft layers (fc_bwd_input.h): the transposed
// problem of the forward, in the forward's form. The operand gradients of a
// tile of 4 samples sit in LDS (16 bytes a row, the rows of one pass at a
// time) and every input gathers its references from there: 16-byte reads at
// random rows, 76 bytes a clock and CU measured, where gathering sample-minor
// rows through L2 ran at 12 (they pass its 4 MB per XCD) and needed a
// transpose of all operand gradients before. Measured at 10000 -> 10000,
// K = 8, B = 4096: transpose and gather 474 us -> 217 us (4 tiles a CU, each
// two passes of staging 160 KB at the memory's rate, about 8 us, and of
// gathering from it at the LDS rate, about 8 us, with the whole LDS in use
// nothing of the next pass to overlap with); 4000 -> 4000 LUT4, B = 1024: 88
// -> 45 us. 512 threads of 256 registers: with 1024 of 128 the entry stream
// spilled (255-303 us).
//
// Inputs are grouped by block (the workgroup's share of the inputs) and pass
// (the rows in LDS together). Within a group they are ordered by reference
// count, so the 64 lanes of a wave have equally long lists; a chunk of 64
// inputs stores its lists side by side ([step][lane], one coalesced 512-byte
// load a step) and a wave's chunks follow each other, so that its entries are
// one stream, loaded 12 steps ahead (a chunk is about 10 steps: started
// chunk by chunk, its first loads' latency was half of the gather). An input's sum stays with a lane through a pass; between
// passes, and before the rows are written, the sums change places through
// LDS. Inputs of more than kHeavy references (narrow inputs under wide
// layers) take a wave each instead.
//
// Every sum has a fixed order: passes ascending, references ascending in a
// pass (heavy inputs: lane by lane, then over the lanes).
#include "fc_bwd_input.h"
#include "fc_soft_common.h"
#include "ref_table.h"

namespace slg {

constexpr int kIgThreads = 512;
constexpr int kIgSlots = 20;                             // inputs per thread
constexpr int kIgBlock = kIgThreads * kIgSlots;          // inputs per block, at most
constexpr int kIgRows = 10236;                           // rows per pass, at most: with a zero
                                                         // row 16 B each in 160 KB of LDS
constexpr int kIgWaves = kIgThreads / 64;
constexpr int kIgStep = 4;                               // entries a lane takes at a time
constexpr int kHeavy = 512;                              // references of a lane's list, at most

struct IgArgs {
  int B, IN, R2, OUT, NS, K;
  int NB, IB;      // input blocks, inputs per block
  int NP, RB;      // passes, rows per pass
  int64_t R;
};

// Steps of a chunk whose longest list has n entries: whole blocks of kIgStep.
__device__ inline int ig_steps(int n) { return (n + kIgStep - 1) / kIgStep * kIgStep; }
// A group's entries past its references: its longest list in the first
// chunk (lists descend, so each other chunk's padding is at most the
// references of the chunk before it) and the rounding of every chunk.
__host__ __device__ inline int ig_slack(int IB) {
  return 64 * kHeavy + 64 * kIgStep * ((IB + 63) / 64);
}

// group = pass * NB + block; key = group * IB + input within the block
__global__ void __launch_bounds__(256) ig_keys_kernel(IgArgs a, const int* __restrict__ cand,
                                                      int* __restrict__ keys) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= a.R) return;
  const int i = min(max(cand[r], 0), a.IN - 1);
  const int SK = a.NS * a.K, o = r / SK, side = (r - o * SK) / a.K;
  const int q = i / a.IB;
  keys[r] = ((side * a.OUT + o) / a.RB * a.NB + q) * a.IB + (i - q * a.IB);
}

// One workgroup per group: its inputs in descending order of their counts
// (by a counting sort; the place among equal counts does not matter to any
// sum). perm [group][IB]: each slot's input | its count << 16, and the heavy
// inputs from the end; slot [key] (heavy inputs: -1); off: the first entry of
// each chunk of 64 slots.
// s[0..IB]: where each input's references start; first: the group's first entry.
__device__ inline void ig_group_slots(const IgArgs& a, int g, const int* s, int first,
                                      int* __restrict__ perm, int* __restrict__ slot,
                                      int* __restrict__ off, int* __restrict__ heavy) {
  __shared__ int hist[kHeavy + 2], at[kHeavy + 2], part[16];
  const int n = min(a.IB, a.IN - g % a.NB * a.IB);  // inputs of the block
  const int t = threadIdx.x;
  int* pm = perm + (int64_t)g * a.IB;
  int* sl = slot + (int64_t)g * a.IB;
  for (int i = t; i < kHeavy + 2; i += 1024) hist[i] = 0;
  __syncthreads();
  for (int i = t; i < n; i += 1024) atomicAdd(&hist[min(s[i + 1] - s[i], kHeavy + 1)], 1);
  __syncthreads();
  if (t < 64) {  // at[c] = inputs of more than c references, heavy ones aside
    int run = 0;
    for (int hi = kHeavy; hi >= 0; hi -= 64) {
      const int c = hi - t;
      const int v = c >= 0 ? hist[c] : 0;
      int x = v;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (t >= d) x += y;
      }
      if (c >= 0) at[c] = run + x - v;
      run += __shfl(x, 63, 64);
    }
    if (t == 0) {
      heavy[g] = hist[kHeavy + 1];
      at[kHeavy + 1] = a.IB - hist[kHeavy + 1];
    }
  }
  __syncthreads();
  for (int i = t; i < n; i += 1024) {
    const int c = s[i + 1] - s[i];
    const int p = atomicAdd(&at[min(c, kHeavy + 1)], 1);
    pm[p] = c > kHeavy ? i : i | (c << 16);
    sl[i] = c > kHeavy ? -1 : p;
  }
  __threadfence_block();
  __syncthreads();
  // chunk offsets: a chunk is as long as its first slot's list, in whole
  // blocks; chunk w + kIgWaves j is the j-th of wave w, wave by wave
  const int m = n - hist[kHeavy + 1], nc = (m + 63) >> 6, NC = (a.IB + 63) >> 6;
  const int c = t / kIgSlots + kIgWaves * (t % kIgSlots);
  const int len = t < kIgWaves * kIgSlots && c < nc ? 64 * ig_steps(pm[64 * c] >> 16) : 0;
  int x = len;
  const int lane = t & 63, wave = t >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  if (lane == 63) part[wave] = x;
  __syncthreads();
  int base = first + g * ig_slack(a.IB);
  for (int w = 0; w < wave; ++w) base += part[w];
  if (t < kIgWaves * kIgSlots && c < NC) off[(int64_t)g * NC + c] = base + x - len;
}

__global__ void __launch_bounds__(1024) ig_slots_kernel(IgArgs a, const int* __restrict__ start,
                                                        int* __restrict__ perm,
                                                        int* __restrict__ slot,
                                                        int* __restrict__ off,
                                                        int* __restrict__ heavy) {
  const int* s = start + (int64_t)blockIdx.x * a.IB;
  ig_group_slots(a, blockIdx.x, s, s[0], perm, slot, off, heavy);
}

// Entries (LDS byte offset of the row within its pass, weight) of each
// reference: a chunk's lists [step][lane], heavy inputs' lists as they lie.
__global__ void __launch_bounds__(256) ig_entries_kernel(IgArgs a, const int* __restrict__ sorted,
                                                         const int* __restrict__ keys,
                                                         const int* __restrict__ start,
                                                         const int* __restrict__ slot,
                                                         const int* __restrict__ off,
                                                         const float* __restrict__ w,
                                                         int2* __restrict__ ent,
                                                         int2* __restrict__ ent_heavy) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= a.R) return;
  const int r = sorted[j], key = keys[r];
  const int SK = a.NS * a.K, o = r / SK, side = (r - o * SK) / a.K;
  const int row = side * a.OUT + o;
  const int2 e = make_int2((row - row / a.RB * a.RB) * 16, __float_as_int(w[r]));
  const int s = slot[key];
  if (s < 0) {
    ent_heavy[j] = e;
  } else {
    const int NC = (a.IB + 63) >> 6;
    const int64_t at = off[(int64_t)(key / a.IB) * NC + (s >> 6)] + (int64_t)(j - start[key]) * 64 + (s & 63);
    ent[at] = e;
  }
}

// The whole table in one launch, a workgroup per input block, for one pass
// (ig_small): the references that fall in the block are counted, placed and
// ranked in LDS, where the eight launches of the general way pass everything
// through memory. Each workgroup reads all candidates, twice.
__global__ void __launch_bounds__(1024)
ig_table_kernel(IgArgs a, const int* __restrict__ cand, const float* __restrict__ w,
                int* __restrict__ start, int* __restrict__ perm, int* __restrict__ slot,
                int* __restrict__ off, int* __restrict__ heavy, int2* __restrict__ ent,
                int2* __restrict__ ent_heavy) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ int part[16], before[16];
  int* cur = reinterpret_cast<int*>(smem);                              // [IB + 1]
  uint16_t* refs = reinterpret_cast<uint16_t*>(cur + a.IB + 1);         // [R]
  const int g = blockIdx.x, i0 = g * a.IB, R = (int)a.R;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int i = t; i <= a.IB; i += 1024) cur[i] = 0;
  __syncthreads();
  auto input = [&](int r) { return min(max(cand[r], 0), a.IN - 1) - i0; };  // within the block
  auto each = [&](auto&& f) {  // f(r, input) over the references, 16 loads in flight
    constexpr int U = 16;
    for (int r0 = t; r0 < R; r0 += U * 1024) {
      int i[U];
#pragma unroll
      for (int u = 0; u < U; ++u) i[u] = cand[min(r0 + u * 1024, R - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (r0 + u * 1024 < R) f(r0 + u * 1024, min(max(i[u], 0), a.IN - 1) - i0);
    }
  };
  int low = 0;  // references of earlier blocks
  each([&](int, int i) {
    low += i < 0;
    if ((unsigned)i < (unsigned)a.IB) atomicAdd(&cur[i], 1);
  });
  __syncthreads();
  // exclusive scan of the counts, a run of them per thread
  const int per = (a.IB + 1023) / 1024, c0 = min(t * per, a.IB), c1 = min(c0 + per, a.IB);
  int sum = 0;
  for (int i = c0; i < c1; ++i) sum += cur[i];
  int x = sum;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
    low += __shfl_xor(low, d, 64);
  }
  if (lane == 63) part[wave] = x;
  if (lane == 0) before[wave] = low;
  __syncthreads();
  int at = x - sum, first = 0, all = 0;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    at += v < wave ? part[v] : 0;
    all += part[v];
    first += before[v];
  }
  for (int i = c0; i < c1; ++i) {
    const int c = cur[i];
    cur[i] = at;
    start[i0 + i] = first + at;
    at += c;
  }
  if (t == 0) {
    cur[a.IB] = all;
    if (g == a.NB - 1) start[i0 + a.IB] = first + all;
  }
  __syncthreads();
  ig_group_slots(a, g, cur, first, perm, slot, off, heavy);
  __threadfence_block();
  __syncthreads();
  // place: afterwards cur[i] is the end of input i's list, cur[i - 1] its start
  each([&](int r, int i) {
    if ((unsigned)i < (unsigned)a.IB) refs[atomicAdd(&cur[i], 1)] = (uint16_t)r;
  });
  __syncthreads();
  const int SK = a.NS * a.K, NC = (a.IB + 63) >> 6;
  for (int j = t; j < all; j += 1024) {
    const int r = refs[j], i = input(r);
    const int b = i ? cur[i - 1] : 0, e = cur[i];
    int rank = 0;  // ascending references, whatever order they were placed in
    for (int k = b; k < e; ++k) rank += refs[k] < r;
    const int o = r / SK, side = (r - o * SK) / a.K;
    const int2 v = make_int2((side * a.OUT + o) * 16, __float_as_int(w[r]));
    const int sl = slot[i0 + i];
    if (sl < 0)
      ent_heavy[first + b + rank] = v;
    else
      ent[(int64_t)off[(int64_t)g * NC + (sl >> 6)] + (int64_t)rank * 64 + (sl & 63)] = v;
  }
}

__global__ void __launch_bounds__(kIgThreads)
ig_gather_kernel(IgArgs a, const float* __restrict__ gbr, const int* __restrict__ start,
                 const int* __restrict__ perm, const int* __restrict__ off,
                 const int* __restrict__ heavy, const int2* __restrict__ ent,
                 const int2* __restrict__ ent_heavy, float* __restrict__ gx) {
  extern __shared__ __align__(16) unsigned char smem[];
  f32x4* rows = reinterpret_cast<f32x4*>(smem);
  const int q = (int)(blockIdx.x % (unsigned)a.NB), tile = (int)(blockIdx.x / (unsigned)a.NB);
  const int b0 = tile * 4, nb = min(4, a.B - b0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i0 = q * a.IB, n = min(a.IB, a.IN - i0);
  const int NC = (a.IB + 63) >> 6;
  f32x4 acc[kIgSlots];
#pragma unroll
  for (int j = 0; j < kIgSlots; ++j) acc[j] = (f32x4)0.0f;
  for (int p = 0; p < a.NP; ++p) {
    const int g = p * a.NB + q;
    const int* s = start + (int64_t)g * a.IB;
    const int* pm = perm + (int64_t)g * a.IB;
    const int nh = heavy[g], m = n - nh;
    // this thread's slots (input | count << 16; past the group: count 0) and
    // the first blocks of the wave's entries
    int pv[kIgSlots];
#pragma unroll
    for (int j = 0; j < kIgSlots; ++j) {
      const int k = (wave + kIgWaves * j) * 64 + lane;
      pv[j] = k < m ? pm[k] : -1;
    }
    const int2* e = ent + __builtin_amdgcn_readfirstlane(wave < NC ? off[(int64_t)g * NC + wave] : 0);
    int2 e0[kIgStep], e1[kIgStep], e2[kIgStep];
#pragma unroll
    for (int u = 0; u < kIgStep; ++u) {
      e0[u] = e[u * 64 + lane];
      e1[u] = e[(kIgStep + u) * 64 + lane];
      e2[u] = e[(2 * kIgStep + u) * 64 + lane];
    }
    if (p) {  // the sums so far, from their inputs' places to this pass's slots
#pragma unroll
      for (int j = 0; j < kIgSlots; ++j)
        if (pv[j] >= 0) acc[j] = rows[pv[j] & 0xffff];
      for (int h = wave; h < nh; h += kIgWaves) {
        const int i = pm[a.IB - nh + h];
        if (lane < nb)
          gx[(int64_t)(b0 + lane) * a.IN + i0 + i] = reinterpret_cast<const float*>(rows + i)[lane];
      }
      __syncthreads();
    }
    // stage rows [p RB, p RB + nr) of the tile's samples, then a zero row
    const int c0 = p * a.RB, nr = min(a.RB, a.R2 - c0);
    const float* src = gbr + (int64_t)b0 * a.R2 + c0;
    if (((a.R2 | c0 | nr) & 3) == 0) {
      constexpr int NL = 3;  // 16-byte loads of a row in flight per thread, times 4 samples
      for (int k0 = tid; k0 < nr >> 2; k0 += NL * kIgThreads) {
        float4 t[NL][4];
#pragma unroll
        for (int l = 0; l < NL; ++l) {
          const int k = k0 + l * kIgThreads;
#pragma unroll
          for (int v = 0; v < 4; ++v)
            t[l][v] = v < nb && k < nr >> 2 ? ld_stream4(src + (int64_t)v * a.R2 + 4 * k)
                                            : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int l = 0; l < NL; ++l) {
          const int k = k0 + l * kIgThreads;
          if (k < nr >> 2) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
              rows[4 * k + u] = f32x4{lanev(t[l][0], u), lanev(t[l][1], u), lanev(t[l][2], u),
                                      lanev(t[l][3], u)};
          }
        }
      }
    } else {
      for (int k = tid; k < nr; k += kIgThreads) {
        f32x4 t;
#pragma unroll
        for (int v = 0; v < 4; ++v) t[v] = v < nb ? src[(int64_t)v * a.R2 + k] : 0.0f;
        rows[k] = t;
      }
    }
    if (tid == 0) rows[nr] = (f32x4)0.0f;
    __syncthreads();
    auto row = [&](int byte) { return *reinterpret_cast<const f32x4*>(smem + byte); };
#pragma unroll
    for (int j = 0; j < kIgSlots; ++j) {
      const int cnt = pv[j] >= 0 ? pv[j] >> 16 : 0;
      const int L = ig_steps(__builtin_amdgcn_readfirstlane(cnt));
      const int least = __builtin_amdgcn_readlane(cnt, 63);
      f32x4 sum = acc[j];
      for (int t0 = 0; t0 < L; t0 += kIgStep) {
        int2 cur[kIgStep];
#pragma unroll
        for (int u = 0; u < kIgStep; ++u) cur[u] = e0[u];
        e += kIgStep * 64;
#pragma unroll
        for (int u = 0; u < kIgStep; ++u) {
          e0[u] = e1[u];
          e1[u] = e2[u];
          e2[u] = e[(2 * kIgStep + u) * 64 + lane];
        }
        if (t0 + kIgStep > least) {  // past some lanes' lists: the zero row
#pragma unroll
          for (int u = 0; u < kIgStep; ++u)
            if (t0 + u >= cnt) cur[u] = make_int2(nr * 16, 0);
        }
        f32x4 v[kIgStep];
#pragma unroll
        for (int u = 0; u < kIgStep; ++u) v[u] = row(cur[u].x);
#pragma unroll
        for (int u = 0; u < kIgStep; ++u) fma_acc(sum, __int_as_float(cur[u].y), v[u]);
      }
      acc[j] = sum;
    }
    // heavy inputs, a wave each: lanes take every 64th reference; their sum
    // over the passes waits in gx
    for (int h = wave; h < nh; h += kIgWaves) {
      const int i = pm[a.IB - nh + h];
      f32x4 sum = (f32x4)0.0f;
      for (int k = s[i] + lane; k < s[i + 1]; k += 64) {
        const int2 e = ent_heavy[k];
        fma_acc(sum, __int_as_float(e.y), row(e.x));
      }
#pragma unroll
      for (int d = 32; d > 0; d >>= 1)
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[v] += __shfl_xor(sum[v], d, 64);
      if (lane < nb) {
        float f = lane == 0 ? sum[0] : lane == 1 ? sum[1] : lane == 2 ? sum[2] : sum[3];
        float* dst = gx + (int64_t)(b0 + lane) * a.IN + i0 + i;
        if (p) f += *dst;
        *dst = f;
      }
    }
    __syncthreads();  // every read of the rows is done
#pragma unroll
    for (int j = 0; j < kIgSlots; ++j)
      if (pv[j] >= 0) rows[pv[j] & 0xffff] = acc[j];
    // heavy inputs' sums too: they may not be heavy in the next pass
    for (int h = wave; h < nh; h += kIgWaves) {
      const int i = pm[a.IB - nh + h];
      if (lane < 4) {
        float f = 0.0f;
        if (lane < nb) f = gx[(int64_t)(b0 + lane) * a.IN + i0 + i];
        reinterpret_cast<float*>(rows + i)[lane] = f;
      }
    }
    __syncthreads();
  }
  for (int k = tid; k < n; k += kIgThreads) {
    const f32x4 v = rows[k];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (u < nb) gx[(int64_t)(b0 + u) * a.IN + i0 + k] = v[u];
  }
}

// ---------------------------------------------------------------------------
// Wide layers: the rows pass through memory once more, sample-minor, and every
// input gathers its references' rows through L2. Where the inputs take several
// blocks, each block stages every row again, and a (pass, block) group is left
// with few references to spread that over; here a reference costs the same at
// any width.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) iw_keys_kernel(const int* __restrict__ cand, int R,
                                                               int IN, int* __restrict__ keys) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < R) keys[r] = min(max(cand[r], 0), IN - 1);
}

__global__ void __launch_bounds__(256) iw_entries_kernel(const int* __restrict__ sorted,
                                                                  int R, int OUT, int NS, int K,
                                                                  const float* __restrict__ w,
                                                                  int2* __restrict__ ent) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= R) return;
  const int r = sorted[j], SK = NS * K;  // r = (o * NS + side) * K + k
  const int o = r / SK, side = (r - o * SK) / K;
  ent[j] = make_int2(side * OUT + o, __float_as_int(w[r]));
}

// gab [R2][LB] = transpose of gbr [B][R2] (rows b >= B of gab's columns are
// zero), through a 64 x 64 LDS tile; float4 loads along gbr rows when R2 is
// a multiple of 4, float4 stores along gab rows (LB is a multiple of 64).
__global__ void __launch_bounds__(256) iw_transpose_kernel(const float* __restrict__ gbr,
                                                                    int B, int R2, int64_t LB,
                                                                    int n_rtiles,
                                                                    float* __restrict__ gab) {
  __shared__ float t[64][65];  // [b][r]
  const int rt = blockIdx.x % n_rtiles, bt = blockIdx.x / n_rtiles;
  const int r0 = rt * 64, b0 = bt * 64;
  const int c4 = threadIdx.x & 15, q = threadIdx.x >> 4;  // 16 float4 columns x 16 rows
  if ((R2 & 3) == 0) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int bl = q + 16 * k, b = b0 + bl, r = r0 + 4 * c4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (b < B && r < R2) v = *reinterpret_cast<const float4*>(gbr + (int64_t)b * R2 + r);
      t[bl][4 * c4] = v.x;
      t[bl][4 * c4 + 1] = v.y;
      t[bl][4 * c4 + 2] = v.z;
      t[bl][4 * c4 + 3] = v.w;
    }
  } else {
    const int c = threadIdx.x & 63, qq = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const int bl = qq + 4 * k, b = b0 + bl, r = r0 + c;
      t[bl][c] = (b < B && r < R2) ? gbr[(int64_t)b * R2 + r] : 0.0f;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int rl = q + 16 * k, r = r0 + rl;
    if (r < R2) {
      const float4 v = make_float4(t[4 * c4][rl], t[4 * c4 + 1][rl], t[4 * c4 + 2][rl],
                                   t[4 * c4 + 3][rl]);
      *reinterpret_cast<float4*>(gab + (int64_t)r * LB + b0 + 4 * c4) = v;
    }
  }
}

// Input gradient from the node-gradient rows gab [2*OUT][LB] (row side*OUT+o,
// sample-minor): gx[b][i] = sum over the entries e of input i, in table
// order, of weight(e) * gab[row(e)][b]. A workgroup owns 4*IW inputs x 64*V
// samples. Each wave walks the entries of its IW consecutive inputs as one
// flat range (contiguous in the table) with its lanes along samples: the
// entries are wave-uniform (scalar loads, the next 8 prefetched), each costs
// one coalesced 64V-sample row-segment load, and 8 such loads are in flight.
// An input's sum is complete when the walk reaches the next input's start.
// The results go through LDS so gx rows are written contiguously.
template <int V, int IW>
__global__ void __launch_bounds__(256) iw_gather_kernel(const float* __restrict__ gab,
                                                                 int64_t LB, int B, int IN,
                                                                 const int* __restrict__ start,
                                                                 const int2* __restrict__ ent,
                                                                 int n_itiles, int n_blocks,
                                                                 float* __restrict__ gx) {
  using vt = typename vecf<V>::t;
  constexpr int NI = 4 * IW;       // inputs per workgroup
  constexpr int NS = 64 * V;       // samples per workgroup
  constexpr int G = 8;             // entries per step
  __shared__ float T[NI][NS + 1];  // [input][sample]
  const int L = (int)xcd_logical_id(blockIdx.x, gridDim.x);
  if (L >= n_blocks) return;
  const int it = L % n_itiles, sc = L / n_itiles;
  const int i0 = it * NI;
  const int b0 = sc * NS;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const float* col = gab + b0 + lane * V;
  const int ia = i0 + wave * IW;
  const int iend = min(ia + IW, IN);
  int cur = ia;  // input whose sum is being accumulated
  float acc[V];
#pragma unroll
  for (int v = 0; v < V; ++v) acc[v] = 0.0f;
  if (ia < iend) {
    int e = start[ia];
    const int e_end = start[iend];
    int nb = start[ia + 1];  // first entry of input cur + 1
    int2 qn[G];
#pragma unroll
    for (int u = 0; u < G; ++u) qn[u] = ent[min(e + u, max(e_end - 1, 0))];
    while (e < e_end) {
      int2 q[G];
#pragma unroll
      for (int u = 0; u < G; ++u) q[u] = qn[u];
      vt g[G];
#pragma unroll
      for (int u = 0; u < G; ++u) g[u] = *reinterpret_cast<const vt*>(col + (int64_t)q[u].x * LB);
      const int en = e + G;
#pragma unroll
      for (int u = 0; u < G; ++u) qn[u] = ent[min(en + u, e_end - 1)];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        if (e + u < e_end) {
          while (e + u == nb) {  // input cur is complete (inputs without entries: zero)
#pragma unroll
            for (int v = 0; v < V; ++v) {
              T[cur - i0][lane * V + v] = acc[v];
              acc[v] = 0.0f;
            }
            ++cur;
            nb = start[cur + 1];
          }
#pragma unroll
          for (int v = 0; v < V; ++v) acc[v] = fmaf(__int_as_float(q[u].y), lanev(g[u], v), acc[v]);
        }
      }
      e = en;
    }
  }
  for (; cur < ia + IW; ++cur) {  // the last input with entries, then empty ones
#pragma unroll
    for (int v = 0; v < V; ++v) {
      T[cur - i0][lane * V + v] = acc[v];
      acc[v] = 0.0f;
    }
  }
  __syncthreads();
  const int c = threadIdx.x % NI;
#pragma unroll 4
  for (int s = threadIdx.x / NI; s < NS; s += 256 / NI) {
    if (b0 + s < B && i0 + c < IN) gx[(int64_t)(b0 + s) * IN + i0 + c] = T[c][s];
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
static inline int64_t ig_round(int64_t n) { return (n + 3) & ~int64_t(3); }

struct IgPlan {
  IgArgs a;
  int64_t keys, table, perm, slot, off, heavy, ent, ent_heavy, total;  // offsets, 4-byte words
  int64_t groups, nkeys, tiles;
};

static IgPlan ig_plan(int64_t B, int64_t IN, int64_t OUT, int nsides, int K) {
  IgPlan p{};
  IgArgs& a = p.a;
  a.B = (int)B; a.IN = (int)IN; a.OUT = (int)OUT; a.NS = nsides; a.K = K;
  const int64_t R2 = nsides * OUT;
  a.R2 = (int)R2;
  a.R = nsides * OUT * (int64_t)K;
  p.tiles = cdiv(std::max<int64_t>(B, 1), 4);
  // a block of inputs per workgroup: all of them where the sample tiles fill
  // the chip, else enough blocks to (each stages the rows again)
  a.NB = (int)std::max<int64_t>(cdiv(IN, kIgBlock),
                                std::min<int64_t>(cdiv(device_cus(), p.tiles), cdiv(IN, 256)));
  a.IB = (int)(cdiv(cdiv(IN, a.NB), 64) * 64);
  a.NB = (int)cdiv(IN, a.IB);
  a.NP = (int)cdiv(R2, kIgRows);
  a.RB = (int)(cdiv(cdiv(R2, a.NP), 4) * 4);
  a.NP = (int)cdiv(R2, a.RB);
  p.groups = (int64_t)a.NP * a.NB;
  p.nkeys = p.groups * a.IB;
  int64_t o = 0;
  auto take = [&](int64_t n) {
    const int64_t at = o;
    o += ig_round(n);
    return at;
  };
  p.keys = take(a.R);
  p.table = take(ref_table_ints(a.R, p.nkeys));
  p.perm = take(p.nkeys);
  p.slot = take(p.nkeys);
  p.off = take(p.groups * cdiv(a.IB, 64));
  p.heavy = take(p.groups);
  p.ent = take(2 * (a.R + p.groups * ig_slack(a.IB) + 3 * kIgStep * 64));  // read ahead
  p.ent_heavy = take(2 * a.R);
  p.total = o;
  return p;
}

// Workspace of the wide way: gab [R2][LB] | keys | table | entries.
constexpr int kIwV = 4;              // samples per lane in the gather
constexpr int kIwIW = 8;             // inputs per wave
constexpr int kIwSamples = 64 * kIwV;
constexpr int kIwInputs = 4 * kIwIW;

struct IwPlan {
  int64_t LB, R, R2, gab, keys, table, ent;
  int64_t total() const { return gab + keys + table + ent; }
};

static IwPlan iw_plan(int64_t B, int64_t IN, int64_t OUT, int nsides, int K) {
  IwPlan q{};
  q.LB = cdiv(std::max<int64_t>(B, 1), kIwSamples) * kIwSamples;
  q.R2 = nsides * OUT;
  q.R = q.R2 * K;
  q.gab = q.R2 * q.LB;
  q.keys = ig_round(q.R);
  q.table = ref_table_ints(q.R, IN);
  q.ent = 2 * q.R;
  return q;
}

// Whether the wide way is the shorter, by the nanoseconds that the two differ in
// (fitted to 700 random layers of 100-400000 inputs and outputs, 1-4096 samples,
// K 1-16; the choice is within 3% of the better way for nineteen in twenty and 1%
// slower than it on average). From LDS: the key scan by one workgroup, keys per
// (pass, input), then per round of workgroups the passes, the staging of every
// row and the block's references. Wide: the transpose and the gather over 256
// samples at a time, and the list of one input, which is walked alone. FC
// backward from LDS / wide, K = 8: 10000 -> 10000, B = 1024: 186 / 273 us; 60000
// -> 60000, B = 124: 1332 / 1175; 172000 -> 172000, B = 3: 3046 / 1207.
static bool ig_small(const IgArgs& a);
static bool ig_fits(const IgPlan& p) {
  return p.a.R + p.groups * ig_slack(p.a.IB) < (1LL << 31) && p.nkeys < (1LL << 31) &&
         p.tiles * p.a.NB < (1LL << 31);
}
static bool ig_wide(const IgPlan& p) {
  if (!ig_fits(p)) return true;
  const IgArgs& a = p.a;
  const double rounds = (double)cdiv(p.tiles * a.NB, device_cus());
  const double LB = (double)cdiv(a.B, kIwSamples) * kIwSamples;
  const double table = ig_small(a) ? 0.0 : 9500.0 + 0.3 * (double)(p.nkeys - a.IN);
  const double from_lds = table + rounds * (5600.0 * a.NP + 0.49 * a.R2 + 0.14 * (double)a.R / a.NB);
  const double wide = 15000.0 + LB * (1.35e-3 * a.R2 + 3.7e-4 * (double)a.R) + 410.0 * (double)a.R / a.IN;
  return from_lds > wide;
}

int64_t fc_input_grad_floats(int64_t B, int64_t IN, int64_t OUT, int nsides, int K) {
  const IgPlan p = ig_plan(B, IN, OUT, nsides, K);
  return ig_wide(p) ? iw_plan(B, IN, OUT, nsides, K).total() : p.total;
}

static int fc_input_grad_wide(const float* gbr, int64_t B, int64_t IN, int64_t OUT, int nsides, int K,
                              const int32_t* cand, const float* w, float* ws, float* gx,
                              hipStream_t st) {
  const IwPlan q = iw_plan(B, IN, OUT, nsides, K);
  const int64_t n_rtiles = cdiv(q.R2, 64), n_tr = n_rtiles * (q.LB / 64);
  const int64_t n_itiles = cdiv(IN, kIwInputs), n_blocks = n_itiles * (q.LB / kIwSamples);
  SLG_REQUIRE(q.R < (1LL << 31) && n_tr < (1LL << 31) && n_blocks < (1LL << 31) - 8, SLG_E_SHAPE,
              "fc input gradient: too many references");
  float* gab = ws;
  int* keys = reinterpret_cast<int*>(gab + q.gab);
  int* table = keys + q.keys;
  int2* ent = reinterpret_cast<int2*>(table + q.table);  // offsets are multiples of 4
  const int R = (int)q.R, R2 = (int)q.R2;
  hipLaunchKernelGGL(iw_keys_kernel, dim3((unsigned)cdiv(R, 256)), dim3(256), 0, st, cand, R, (int)IN,
                     keys);
  RefTable tb{};
  const int rc = build_ref_table(keys, R, IN, table, st, &tb);
  if (rc) return rc;
  hipLaunchKernelGGL(iw_entries_kernel, dim3((unsigned)cdiv(R, 256)), dim3(256), 0, st, tb.sorted, R,
                     (int)OUT, nsides, K, w, ent);
  hipLaunchKernelGGL(iw_transpose_kernel, dim3((unsigned)n_tr), dim3(256), 0, st, gbr, (int)B, R2, q.LB,
                     (int)n_rtiles, gab);
  // a multiple of 8 workgroups for the XCD order
  hipLaunchKernelGGL((iw_gather_kernel<kIwV, kIwIW>), dim3((unsigned)(cdiv(n_blocks, 8) * 8)), dim3(256),
                     0, st, gab, q.LB, (int)B, (int)IN, tb.start, ent, (int)n_itiles, (int)n_blocks, gx);
  SLG_LAUNCH_CHECK("fc input gradient (wide)");
  return 0;
}

// One launch for the whole table: one pass, lists of 32 references on average
// at most (an element's rank reads its list) and at most 4096 references a
// block, 48K in all: a workgroup's scattered loads and stores bound it, so it
// follows the references of a block, and every block reads all of them. FC
// backward, K = 8, this against the general way, captured: 250 -> 250, B = 64:
// 40 / 46 us; 1000, B = 256 (4000 a block): 57 / 63; 3000, B = 64 (4000 a
// block, 48000 in all): 67 / 68; past the rule 4000, B = 64: 77 / 75; 2000,
// B = 256 (8000 a block): 81 / 73; 1000, B = 1024 (16000): 98 / 76.
static size_t ig_small_lds(const IgArgs& a) {
  return (size_t)(a.IB + 1) * 4 + (size_t)a.R * 2;
}
static bool ig_small(const IgArgs& a) {
  return a.NP == 1 && a.R <= 48 * 1024 && a.R <= 32 * (int64_t)a.IN && a.R <= 4096 * (int64_t)a.NB &&
         ig_small_lds(a) <= 150 * 1024;
}

int fc_input_grad(const float* gbr, int64_t B, int64_t IN, int64_t OUT, int nsides, int K,
                  const int32_t* cand, const float* w, float* ws, float* gx, hipStream_t st) {
  const IgPlan p = ig_plan(B, IN, OUT, nsides, K);
  if (ig_wide(p)) return fc_input_grad_wide(gbr, B, IN, OUT, nsides, K, cand, w, ws, gx, st);
  const IgArgs& a = p.a;
  int* iw = reinterpret_cast<int*>(ws);
  int *keys = iw + p.keys, *perm = iw + p.perm, *slot = iw + p.slot, *off = iw + p.off,
      *heavy = iw + p.heavy;
  int2* ent = reinterpret_cast<int2*>(iw + p.ent);
  int2* ent_heavy = reinterpret_cast<int2*>(iw + p.ent_heavy);
  RefTable tb{};
  if (ig_small(a)) {
    tb.start = iw + p.table;
    const size_t lds = ig_small_lds(a);
    if (lds > 65536 - 8192) {
      const hipError_t e = hipFuncSetAttribute((const void*)ig_table_kernel,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      SLG_REQUIRE(e == hipSuccess, (int)e, "fc input gradient: LDS %zu: %s", lds,
                  hipGetErrorString(e));
    }
    hipLaunchKernelGGL(ig_table_kernel, dim3((unsigned)a.NB), dim3(1024), lds, st, a, cand, w, tb.start,
                       perm, slot, off, heavy, ent, ent_heavy);
  } else {
    const unsigned rb = (unsigned)cdiv(a.R, 256);
    hipLaunchKernelGGL(ig_keys_kernel, dim3(rb), dim3(256), 0, st, a, cand, keys);
    const int rc = build_ref_table(keys, a.R, p.nkeys, iw + p.table, st, &tb);
    if (rc) return rc;
    hipLaunchKernelGGL(ig_slots_kernel, dim3((unsigned)p.groups), dim3(1024), 0, st, a, tb.start, perm,
                       slot, off, heavy);
    hipLaunchKernelGGL(ig_entries_kernel, dim3(rb), dim3(256), 0, st, a, tb.sorted, keys, tb.start,
                       slot, off, w, ent, ent_heavy);
  }
  SLG_LAUNCH_CHECK("fc input gradient table");
  const size_t lds = (size_t)std::max(a.RB + 1, a.IB) * 16;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute((const void*)ig_gather_kernel,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    SLG_REQUIRE(e == hipSuccess, (int)e, "fc input gradient: LDS %zu: %s", lds, hipGetErrorString(e));
  }
  hipLaunchKernelGGL(ig_gather_kernel, dim3((unsigned)(p.tiles * a.NB)), dim3(kIgThreads), lds, st, a,
                     gbr, tb.start, perm, off, heavy, ent, ent_heavy, gx);
  SLG_LAUNCH_CHECK("fc input gradient gather");
  return 0;
}

}  // namespace slg
