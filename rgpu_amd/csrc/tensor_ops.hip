// Device versions of the Tensor operations rtensor's tape calls (ops.rs,
// tensor.rs, losses.rs), so that any Sequential model -- not only the fixed
// ReLU MLP plan -- can train on the GPU.  All HBM- or latency-bound.
// Built with -ffp-contract=off and every expression in the reference's
// order, so results differ from the CPU path only where a transcendental
// (exp, log, tanh) differs in its last bits, or where a scalar reduction
// (sum_all, losses) adds in a different order.
//   unary ops and their VJPs      ops.rs:132-227
//   broadcast binary ops          tensor.rs:183-246
//   reduce_to                     tensor.rs:399-438 (per output element, source order: exact)
//   sum / mean of all elements    tensor.rs:279-286 (fixed-order two-stage tree)
//   softmax_rows and its VJP      tensor.rs:455-472, ops.rs:291-309 (row sums in column order: exact)
//   mae / softmax-xent / bce      losses.rs:46-53, 99-115, 143-162

#include <algorithm>
#include <type_traits>

#include "rt_internal.h"

namespace {

constexpr int kMaxRank = 4;

struct Shape4 {
  long long n[kMaxRank];   // output shape, right-aligned, leading 1s
  long long sa[kMaxRank];  // strides of operand a in the output index space (0 on broadcast axes)
  long long sb[kMaxRank];
};

__device__ inline float unary_fwd(int op, float k, float v) {
  switch (op) {
    case RT_U_SCALE: return v * k;
    case RT_U_OFFSET: return v + k;
    case RT_U_NEG: return v * -1.0f;
    case RT_U_SQUARE: return v * v;
    case RT_U_SQRT: return sqrtf(v);
    case RT_U_EXP: return expf(v);
    case RT_U_LN: return logf(fmaxf(v, 1e-12f));
    case RT_U_RELU: return fmaxf(v, 0.0f);
    case RT_U_LEAKY_RELU: return v > 0.0f ? v : k * v;
    case RT_U_SIGMOID: return 1.0f / (1.0f + expf(-v));
    case RT_U_TANH: return tanhf(v);
  }
  return __uint_as_float(0x7fc00000u);
}

// dx from the upstream gradient g, the input x and the output y (ops.rs VJPs).
__device__ inline float unary_vjp(int op, float k, float g, float x, float y) {
  switch (op) {
    case RT_U_SCALE: return g * k;
    case RT_U_OFFSET: return g;
    case RT_U_NEG: return g * -1.0f;
    case RT_U_SQUARE: return (g * x) * 2.0f;
    case RT_U_SQRT: return g / (y * 2.0f);
    case RT_U_EXP: return g * y;
    case RT_U_LN: return g / x;
    case RT_U_RELU: return g * (x > 0.0f ? 1.0f : 0.0f);
    case RT_U_LEAKY_RELU: return g * (x > 0.0f ? 1.0f : k);
    case RT_U_SIGMOID: return g * (y * (1.0f - y));
    case RT_U_TANH: return g * (1.0f - y * y);
  }
  return __uint_as_float(0x7fc00000u);
}

__global__ __launch_bounds__(256) void unary_kernel(int op, float k, const float* __restrict__ x, float* __restrict__ y,
                                                    long long n) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    y[i] = unary_fwd(op, k, x[i]);
}

__global__ __launch_bounds__(256) void unary_vjp_kernel(int op, float k, const float* __restrict__ g,
                                                        const float* __restrict__ x, const float* __restrict__ y,
                                                        float* __restrict__ dx, long long n) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    dx[i] = unary_vjp(op, k, g[i], x ? x[i] : 0.0f, y ? y[i] : 0.0f);
}

__device__ inline float binary_op(int op, float a, float b) {
  switch (op) {
    case RT_B_ADD: return a + b;
    case RT_B_SUB: return a - b;
    case RT_B_MUL: return a * b;
    case RT_B_DIV: return a / b;
  }
  return __uint_as_float(0x7fc00000u);
}

// R = rank after the host merged contiguous axes; I = index type (32-bit
// when the output has fewer than 2^31 elements).  R == 1 with unit strides
// is the same-shape case.
template <int R, typename I>
__global__ __launch_bounds__(256) void binary_kernel(int op, const float* __restrict__ a, const float* __restrict__ b,
                                                     float* __restrict__ out, Shape4 s, I n) {
  I nn[R], sa[R], sb[R];
#pragma unroll
  for (int ax = 0; ax < R; ++ax) {
    nn[ax] = (I)s.n[kMaxRank - R + ax];
    sa[ax] = (I)s.sa[kMaxRank - R + ax];
    sb[ax] = (I)s.sb[kMaxRank - R + ax];
  }
  for (I l = (I)blockIdx.x * 256 + (I)threadIdx.x; l < n; l += (I)gridDim.x * 256) {
    I rem = l, ia = 0, ib = 0;
#pragma unroll
    for (int ax = R - 1; ax > 0; --ax) {
      const I idx = rem % nn[ax];
      rem /= nn[ax];
      ia += idx * sa[ax];
      ib += idx * sb[ax];
    }
    ia += rem * sa[0];
    ib += rem * sb[0];
    out[l] = binary_op(op, a[ia], b[ib]);
  }
}

// reduce_to: out[t] = sum of g over the source elements that map to t, added
// in increasing source index (what every reference path does).  One thread
// per output element; the kept axes give the source base, the reduced axes
// (padded to four with extent 1) are walked by nested loops in row-major
// order.
struct ReduceArgs {
  long long keep_n[kMaxRank], keep_s[kMaxRank];  // output index -> source base
  long long red_n[kMaxRank], red_s[kMaxRank];    // reduced axes, outermost first
  int n_keep;
  long long n_out;
};

__global__ __launch_bounds__(256) void reduce_to_kernel(const float* __restrict__ g, float* __restrict__ out,
                                                        ReduceArgs r) {
  for (long long t = blockIdx.x * 256LL + threadIdx.x; t < r.n_out; t += (long long)gridDim.x * 256) {
    long long rem = t, base = 0;
    for (int ax = r.n_keep - 1; ax >= 0; --ax) {
      base += (rem % r.keep_n[ax]) * r.keep_s[ax];
      rem /= r.keep_n[ax];
    }
    // The adds form one dependent chain.  Loads go out in batches of kBatch,
    // the next batch issued before the current one is added, so the chain
    // rarely waits on memory.
    constexpr int kBatch = 32;
    const long long n3 = r.red_n[3], s3 = r.red_s[3];
    float acc = 0.0f;
    for (long long i0 = 0; i0 < r.red_n[0]; ++i0)
      for (long long i1 = 0; i1 < r.red_n[1]; ++i1)
        for (long long i2 = 0; i2 < r.red_n[2]; ++i2) {
          const float* p = g + base + i0 * r.red_s[0] + i1 * r.red_s[1] + i2 * r.red_s[2];
          long long i3 = 0;
          if (n3 >= kBatch) {
            float cur[kBatch], nxt[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) cur[u] = p[u * s3];
            for (i3 = kBatch; i3 + kBatch <= n3; i3 += kBatch) {
#pragma unroll
              for (int u = 0; u < kBatch; ++u) nxt[u] = p[(i3 + u) * s3];
#pragma unroll
              for (int u = 0; u < kBatch; ++u) acc += cur[u];
#pragma unroll
              for (int u = 0; u < kBatch; ++u) cur[u] = nxt[u];
            }
#pragma unroll
            for (int u = 0; u < kBatch; ++u) acc += cur[u];
          }
          for (; i3 < n3; ++i3) acc += p[i3 * s3];
        }
    out[t] = acc;
  }
}

// reduce_to of a row-major [rows][cols] source to one row (the bias gradient of
// a tape layer): the same chain of adds per column, so the same bits.
//
// One thread per column walking memory alone left 1024 columns on four CUs,
// each waiting for 32 loads at a time.  A block takes kColCols columns (64
// bytes of every row, enough to use a whole request) and stages kColRows rows
// at a time through LDS, transposed, so that a column's lane reads four rows
// in one access; the loads of the next rows are in flight while this one's
// are added.  What bounds it is the chain of dependent adds (7 ns each; reading
// the next 32 rows of LDS ahead of them changed nothing) or, for few rows, one
// memory round trip: 2048x1024 22.7 -> 14.9 us, 256x512 4.9 -> 3.5, 16384x64
// 170 -> 107 (from cache; 35.6 us the first in a training step).
constexpr int kColCols = 16, kColRows = 256;

__global__ __launch_bounds__(256) void reduce_columns_kernel(const float* __restrict__ g, float* __restrict__ out,
                                                             int rows, int cols) {
  constexpr int STRIDE = kColRows + 4;  // floats: b128 accesses of neighbouring columns fall into different banks
  constexpr int PASS = 64, PASSES = kColRows / PASS;
  __shared__ __attribute__((aligned(16))) float sh[2][kColCols * STRIDE];
  const int tid = threadIdx.x, c = tid % kColCols, quad = tid / kColCols;  // rows 4 quad .. + 3 of each pass
  const int col = blockIdx.x * kColCols + c;
  float4 v[PASSES];
  auto load = [&](int row0) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
      const int row = row0 + PASS * i + 4 * quad;
      const float* p = g + (long long)row * cols + col;
      auto at = [&](int e) { return row + e < rows && col < cols ? p[(long long)e * cols] : 0.0f; };
      v[i] = make_float4(at(0), at(1), at(2), at(3));
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PASSES; ++i) *reinterpret_cast<float4*>(&sh[buf][c * STRIDE + PASS * i + 4 * quad]) = v[i];
  };
  float acc = 0.0f;
  load(0);
  store(0);
  __syncthreads();
  for (int row0 = 0, buf = 0; row0 < rows; row0 += kColRows, buf ^= 1) {
    const bool more = rows - row0 > kColRows;
    if (more) load(row0 + kColRows);
    if (tid < kColCols) {
      const float* x = &sh[buf][c * STRIDE];
      const int n = min(rows - row0, kColRows);
      int k = 0;
      for (; k + 32 <= n; k += 32) {
        float4 t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = *reinterpret_cast<const float4*>(x + k + 4 * j);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          acc += t[j].x;
          acc += t[j].y;
          acc += t[j].z;
          acc += t[j].w;
        }
      }
      for (; k < n; ++k) acc += x[k];
    }
    if (more) {
      store(buf ^ 1);
      __syncthreads();
    }
  }
  if (tid < kColCols && col < cols) out[col] = acc;
}

// Fixed-order two-stage sum of n floats: block b adds its 256 x chunk
// elements (each thread strided, then a shared-memory tree); stage 2 adds
// the block sums in order and divides by `div`.
// With a single block (n <= 65536) stage 1 also finishes the sum: out[0] =
// (0 + block sum) / div, the value stage 2 would produce from one part.
__global__ __launch_bounds__(256) void sum_stage1(const float* __restrict__ x, long long n, long long chunk,
                                                  float* __restrict__ part, float div, float* __restrict__ out) {
  __shared__ float sh[256];
  const long long b0 = blockIdx.x * chunk, b1 = min(n, b0 + chunk);
  float acc = 0.0f;
  for (long long i = b0 + threadIdx.x; i < b1; i += 256) acc += x[i];
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (gridDim.x == 1) out[0] = (0.0f + sh[0]) / div;
    else part[blockIdx.x] = sh[0];
  }
}

// out[0] = (the parts added) / div: thread t adds parts t, t + 256, ... in
// order, then a shared-memory tree over as many threads as there are parts.  One thread walking the parts alone was a
// chain of dependent loads (512 parts: the whole sum 90 us, 69 us this way).
__global__ __launch_bounds__(256) void sum_stage2(const float* __restrict__ part, int parts, float div,
                                                  float* __restrict__ out) {
  __shared__ float sh[256];
  float acc = 0.0f;
  for (int i = threadIdx.x; i < parts; i += 256) acc += part[i];
  sh[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (w >= parts) continue;  // the upper half is zeros
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = sh[0] / div;
}

// out[i] = (s[0] / div) * (x ? x[i] : 1): the VJPs of sum / mean (Tensor::full)
// and the "scale by g / n" of the losses.
__global__ __launch_bounds__(256) void scalar_fill_kernel(const float* __restrict__ s, float div,
                                                          const float* __restrict__ x, float* __restrict__ out,
                                                          long long n) {
  const float v = s[0] / div;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    out[i] = x ? x[i] * v : v;
}

// Row kernels (softmax, its VJP, softmax cross-entropy from the logits).  A
// block takes a band of G·NR rows, G = T / L groups of L lanes with NR rows
// each, a lane holding columns l, l + L, ... of its rows in R registers: rows
// are read once, in whole cache lines, and written once.  The sums over a
// row (Σ exp, Σ g·s) keep the reference's left-to-right order, hence its
// bits: the terms go to LDS and one lane per row adds that row, all rows of
// the band side by side.  What bounds them is that chain (about 6 us per
// 1000 columns), then HBM.  One thread per row, each walking its row in memory
// alone, read a cache line per lane and step: 4096 x 1000 softmax and VJP
// 864 + 901 us, 14.2 + 11.9 us this way (a tree over the lanes: 8.7 + 7.6 us,
// but then the result is not the reference's sum).
typedef float f4t __attribute__((ext_vector_type(4)));

template <int L_, int R_, int NR_, int T_>
struct Band {
  static constexpr int L = L_, R = R_, NR = NR_, T = T_, G = T / L, ROWS = G * NR;
  // Row pitch in LDS (floats): 16-byte rows an odd number of 16 bytes apart,
  // so the adding lanes' b128 reads fall into different banks.
  static constexpr int PITCH = (L * R / 8) * 8 + 4;
  static constexpr int SMEM = ROWS * PITCH;
  static_assert(ROWS <= T, "one adding lane per row");

  float v[NR][R];

  // This lane's columns of the band's rows from row0, all loads issued
  // together.  Past the last row or column they repeat it (rows, cols >= 1).
  __device__ inline void load(const float* m, long long row0, long long rows, int cols) {
    const int lane = threadIdx.x % L;
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      const float* row = m + min(row0 + group_row(n), rows - 1) * cols;
#pragma unroll
      for (int q = 0; q < R; ++q) v[n][q] = row[min(lane + L * q, cols - 1)];
    }
  }
  __device__ static inline int group_row(int n) { return threadIdx.x / L + G * n; }
  // f(n, q, column) for this lane's columns.
  template <class F>
  __device__ static inline void each(int cols, F&& f) {
    const int lane = threadIdx.x % L;
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + L * q < cols) f(n, q, lane + L * q);
  }
  // v = exp(v - row max).
  __device__ inline void exponentials(int cols) {
    const int lane = threadIdx.x % L;
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      float mx = -INFINITY;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + L * q < cols) mx = fmaxf(mx, v[n][q]);
#pragma unroll
      for (int off = L / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + L * q < cols) v[n][q] = expf(v[n][q] - mx);
    }
  }
  // sums[r] = the terms of row r added in column order; put(n, q) is the term.
  template <class F>
  __device__ inline void add_rows(int cols, float* sh, float* sums, F&& put) const;
};

// acc + p[0] + p[1] + ... + p[n - 1], one add after another; p is 16-byte
// aligned.  Two batches of 32 terms take turns: one is on its way from LDS
// while the other is added, so the chain waits on its own adds only.
__device__ inline float add_in_order(float acc, const float* p, int n) {
  const f4t* q = reinterpret_cast<const f4t*>(p);
  auto fetch = [&](f4t (&t)[8], int j) {
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = q[j / 4 + u];
  };
  auto add = [&](const f4t (&t)[8]) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc += t[u][e];
  };
  const int whole = n & ~31;
  if (whole > 0) {
    // Fetches past the end repeat the last batch: a branch there would make
    // the compiler wait for both batches.
    f4t a[8], b[8];
    fetch(a, 0);
    int j = 0;
    for (; j + 64 <= whole; j += 64) {
      fetch(b, j + 32);
      add(a);
      fetch(a, min(j + 64, whole - 32));
      add(b);
    }
    if (j < whole) add(a);
  }
  for (int j = whole; j < n; ++j) acc += p[j];
  return acc;
}

template <int L_, int R_, int NR_, int T_>
template <class F>
__device__ inline void Band<L_, R_, NR_, T_>::add_rows(int cols, float* sh, float* sums, F&& put) const {
  each(cols, [&](int n, int q, int col) { sh[group_row(n) * PITCH + col] = put(n, q); });
  __syncthreads();
  if (threadIdx.x < ROWS) sums[threadIdx.x] = add_in_order(0.0f, sh + threadIdx.x * PITCH, cols);
  __syncthreads();
}

// The row kernels for rows too long for a lane group's registers (3000 x 4000
// softmax and VJP 87 + 63 us; one row per block of 256 lanes x 16 registers
// took 96 + 92 us): a block of
// four waves takes four rows, one per wave, in chunks of kLongChunk columns
// through LDS; z (or s and g) is read again for the results.
constexpr int kRowThreads = 256, kLossThreads = 1024, kLongChunk = 2048;
constexpr int kLongPitch = kLongChunk + 4, kLongRows = kRowThreads / 64;

__device__ inline float wave_max_row(const float* row, long long cols) {
  float mx = -INFINITY;
  for (long long j = threadIdx.x & 63; j < cols; j += 64) mx = fmaxf(mx, row[j]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
  return mx;
}

// The in-order sum of term(j), j < cols, of this wave's row.  Every thread of
// the block takes part; `in`: the wave has a row.
template <class F>
__device__ inline float long_row_sum(long long cols, bool in, float* sh, F&& term) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  __shared__ float sums[kLongRows];
  float acc = 0.0f;
  for (long long c0 = 0; c0 < cols; c0 += kLongChunk) {
    const int n = (int)min((long long)kLongChunk, cols - c0);
    if (in)
      for (int j = lane; j < n; j += 64) sh[wave * kLongPitch + j] = term(c0 + j);
    __syncthreads();
    if (threadIdx.x < kLongRows) acc = add_in_order(acc, sh + threadIdx.x * kLongPitch, n);
    __syncthreads();
  }
  if (threadIdx.x < kLongRows) sums[threadIdx.x] = acc;
  __syncthreads();
  const float v = sums[wave];
  __syncthreads();
  return v;
}

// tensor.rs:455-472: max, exp, sum, then divide.  y may be z.
template <class B>
__global__ __launch_bounds__(B::T) void softmax_rows_kernel(const float* z, float* y, long long rows, int cols) {
  __shared__ __attribute__((aligned(16))) float sh[B::SMEM];
  __shared__ float sums[B::ROWS];
  const long long row0 = (long long)blockIdx.x * B::ROWS;
  B b;
  b.load(z, row0, rows, cols);
  b.exponentials(cols);
  b.add_rows(cols, sh, sums, [&](int n, int q) { return b.v[n][q]; });
  B::each(cols, [&](int n, int q, int col) {
    const int r = B::group_row(n);
    if (row0 + r < rows) y[(row0 + r) * cols + col] = b.v[n][q] / sums[r];
  });
}

__global__ __launch_bounds__(kRowThreads) void softmax_long_rows_kernel(const float* z, float* y, long long rows,
                                                                        long long cols) {
  __shared__ __attribute__((aligned(16))) float sh[kLongRows * kLongPitch];
  const long long i = (long long)blockIdx.x * kLongRows + (threadIdx.x >> 6);
  const bool in = i < rows;
  const float* row = z + min(i, rows - 1) * cols;
  const float mx = wave_max_row(row, cols);
  const float sum = long_row_sum(cols, in, sh, [&](long long j) { return expf(row[j] - mx); });
  if (in)
    for (long long j = threadIdx.x & 63; j < cols; j += 64) y[i * cols + j] = expf(row[j] - mx) / sum;
}

// ops.rs:291-309: dx = s ⊙ (g − Σ_j g_j s_j), per row.  dx may be s or g.
template <class B>
__global__ __launch_bounds__(B::T) void softmax_rows_vjp_kernel(const float* s, const float* g, float* dx,
                                                                long long rows, int cols) {
  __shared__ __attribute__((aligned(16))) float sh[B::SMEM];
  __shared__ float sums[B::ROWS];
  const long long row0 = (long long)blockIdx.x * B::ROWS;
  B sb, gb;
  sb.load(s, row0, rows, cols);
  gb.load(g, row0, rows, cols);
  sb.add_rows(cols, sh, sums, [&](int n, int q) { return gb.v[n][q] * sb.v[n][q]; });
  B::each(cols, [&](int n, int q, int col) {
    const int r = B::group_row(n);
    if (row0 + r < rows) dx[(row0 + r) * cols + col] = sb.v[n][q] * (gb.v[n][q] - sums[r]);
  });
}

__global__ __launch_bounds__(kRowThreads) void softmax_long_rows_vjp_kernel(const float* s, const float* g, float* dx,
                                                                            long long rows, long long cols) {
  __shared__ __attribute__((aligned(16))) float sh[kLongRows * kLongPitch];
  const long long i = (long long)blockIdx.x * kLongRows + (threadIdx.x >> 6);
  const bool in = i < rows;
  const float* sr = s + min(i, rows - 1) * cols;
  const float* gr = g + min(i, rows - 1) * cols;
  const float dot = long_row_sum(cols, in, sh, [&](long long j) { return gr[j] * sr[j]; });
  if (in)
    for (long long j = threadIdx.x & 63; j < cols; j += 64) dx[i * cols + j] = sr[j] * (gr[j] - dot);
}

// Per-element loss terms (summed by the two-stage sum) and the unscaled
// gradient directions (scaled by g / n with scalar_fill_kernel).
__global__ __launch_bounds__(256) void loss_terms_kernel(int kind, const float* __restrict__ p,
                                                         const float* __restrict__ y, float* __restrict__ term,
                                                         float* __restrict__ dir, long long n) {
  const float lo = 1e-7f, hi = 1.0f - 1e-7f;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
    const float pi = p[i], yi = y[i];
    switch (kind) {
      case RT_LOSS_MAE: {  // losses.rs:46-53 (p = pred - target already)
        term[i] = fabsf(pi);
        if (dir) dir[i] = pi >= 0.0f ? 1.0f : -1.0f;
        break;
      }
      case RT_LOSS_SOFTMAX_XENT: {  // losses.rs:99-115 (p = softmax(pred))
        term[i] = yi != 0.0f ? -(yi * logf(fmaxf(pi, 1e-12f))) : 0.0f;
        if (dir) dir[i] = pi - yi;
        break;
      }
      case RT_LOSS_BCE: {  // losses.rs:143-162
        const float c = pi < lo ? lo : (pi > hi ? hi : pi);  // f32::clamp: NaN stays NaN
        term[i] = -(yi * logf(c) + (1.0f - yi) * logf(1.0f - c));
        if (dir) dir[i] = (c - yi) / (c * (1.0f - c));
        break;
      }
    }
  }
}

// losses.rs:99-115 from the logits in one pass per row: the softmax of
// softmax_rows_kernel (the same bits), then dir = p − y and the row's loss
// terms −y·ln(max(p, 1e-12)) (y ≠ 0).  Each thread adds its terms, a block
// tree adds the threads; without `part` (one block) the launch also writes value
// = (0 + total) / div, else each block writes its part for sum_stage2.  dir may
// be z.
template <int T>
__device__ inline void loss_block_sum(float terms, float* __restrict__ part, float div, float* __restrict__ out) {
  __shared__ float red[T];
  red[threadIdx.x] = terms;
  __syncthreads();
  for (int w = T / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (part == nullptr) out[0] = (0.0f + red[0]) / div;
    else part[blockIdx.x] = red[0];
  }
}

// dir_scale 1 leaves P − Y exactly as it is.
__device__ inline float xent_element(float p, float y, float dir_scale, float& terms) {
  if (y != 0.0f) terms += -(y * logf(fmaxf(p, 1e-12f)));
  return (p - y) * dir_scale;
}

template <class B>
__global__ __launch_bounds__(B::T) void xent_logits_kernel(const float* z, const float* __restrict__ y, float* dir,
                                                           long long rows, int cols, float* __restrict__ part,
                                                           float div, float* __restrict__ out, float dir_scale) {
  __shared__ __attribute__((aligned(16))) float sh[B::SMEM];
  __shared__ float sums[B::ROWS];
  const long long row0 = (long long)blockIdx.x * B::ROWS;
  B zb, yb;
  zb.load(z, row0, rows, cols);
  yb.load(y, row0, rows, cols);
  zb.exponentials(cols);
  zb.add_rows(cols, sh, sums, [&](int n, int q) { return zb.v[n][q]; });
  float terms = 0.0f;
  B::each(cols, [&](int n, int q, int col) {
    const int r = B::group_row(n);
    if (row0 + r < rows)
      dir[(row0 + r) * cols + col] = xent_element(zb.v[n][q] / sums[r], yb.v[n][q], dir_scale, terms);
  });
  loss_block_sum<B::T>(terms, part, div, out);
}

// Also the form for no rows or no columns (nothing to load): value = 0 / div.
__global__ __launch_bounds__(kRowThreads) void xent_logits_long_kernel(const float* z, const float* __restrict__ y,
                                                                       float* dir, long long rows, long long cols,
                                                                       float* __restrict__ part, float div,
                                                                       float* __restrict__ out, float dir_scale) {
  __shared__ __attribute__((aligned(16))) float sh[kLongRows * kLongPitch];
  const long long i = (long long)blockIdx.x * kLongRows + (threadIdx.x >> 6);
  const bool in = i < rows;
  const float* row = z + (in ? i : 0) * cols;
  const float mx = in ? wave_max_row(row, cols) : 0.0f;
  const float sum = long_row_sum(cols, in, sh, [&](long long j) { return expf(row[j] - mx); });
  float terms = 0.0f;
  if (in)
    for (long long j = threadIdx.x & 63; j < cols; j += 64) {
      const long long e = i * cols + j;
      dir[e] = xent_element(expf(row[j] - mx) / sum, y[e], dir_scale, terms);
    }
  loss_block_sum<kRowThreads>(terms, part, div, out);
}

// f(Band) for rows of 1 <= cols <= 1024: the fewest lanes that hold the row
// in one register each up to 64 columns (narrow rows fill the lanes with
// rows), else a wave with 4 or 16 registers.  One row per group: the blocks of
// a CU then add, load and store beside each other (four rows per group, in a
// quarter of the blocks, took 18.7 + 15.3 us at 4096 x 1000 against 15.7 +
// 14.0).
template <class F>
hipError_t by_row_length(long long cols, F&& f) {
#define RT_BAND(l, r) return f(Band<l, r, 1, kRowThreads>{})
  if (cols <= 4) RT_BAND(4, 1);
  if (cols <= 8) RT_BAND(8, 1);
  if (cols <= 16) RT_BAND(16, 1);
  if (cols <= 32) RT_BAND(32, 1);
  if (cols <= 64) RT_BAND(64, 1);
  if (cols <= 256) RT_BAND(64, 4);
  RT_BAND(64, 16);
#undef RT_BAND
}
constexpr long long kBandCols = 1024;

unsigned grid_for(long long n) { return (unsigned)std::max<long long>(1, std::min<long long>((n + 255) / 256, 8192)); }

}  // namespace

namespace rt {

hipError_t unary_launch(hipStream_t s, int op, float k, const float* x, float* y, long long n) {
  if (n <= 0) return hipSuccess;
  rt::launch(unary_kernel, dim3(grid_for(n)), dim3(256), 0, s, op, k, x, y, n);
  return hipGetLastError();
}

hipError_t unary_vjp_launch(hipStream_t s, int op, float k, const float* g, const float* x, const float* y, float* dx,
                            long long n) {
  if (n <= 0) return hipSuccess;
  rt::launch(unary_vjp_kernel, dim3(grid_for(n)), dim3(256), 0, s, op, k, g, x, y, dx, n);
  return hipGetLastError();
}

template <int R>
hipError_t binary_launch_r(hipStream_t s, int op, const float* a, const float* b, float* out, const Shape4& sh,
                           long long n) {
  const dim3 grid(grid_for(n)), block(256);
  // 32-bit indices only where the grid-stride index cannot pass INT32_MAX
  // (its last step goes up to n - 1 + the grid's threads).
  if (n <= (1LL << 31) - 1 - (long long)grid.x * 256)
    rt::launch((binary_kernel<R, int>), grid, block, 0, s, op, a, b, out, sh, (int)n);
  else
    rt::launch((binary_kernel<R, long long>), grid, block, 0, s, op, a, b, out, sh, n);
  return hipGetLastError();
}

hipError_t binary_launch(hipStream_t s, int op, const float* a, const long long* sa, const float* b,
                         const long long* sb, float* out, const long long* shape, int rank) {
  if (rank < 1 || rank > kMaxRank) return hipErrorInvalidValue;
  // Merge axis i into i + 1 where both operands step contiguously across the
  // boundary (a broadcast axis next to a broadcast axis also merges), so a
  // same-shape zip is rank 1 and a bias broadcast rank 2.
  long long n_[kMaxRank], a_[kMaxRank], b_[kMaxRank];
  int r = 0;
  long long n = 1;
  for (int i = 0; i < rank; ++i) {
    n *= shape[i];
    if (shape[i] == 1) continue;  // extent-1 axes contribute nothing
    if (r > 0 && a_[r - 1] == sa[i] * shape[i] && b_[r - 1] == sb[i] * shape[i]) {
      n_[r - 1] *= shape[i];
      a_[r - 1] = sa[i];
      b_[r - 1] = sb[i];
    } else {
      n_[r] = shape[i];
      a_[r] = sa[i];
      b_[r] = sb[i];
      ++r;
    }
  }
  if (n <= 0) return hipSuccess;
  if (r == 0) {  // every axis has extent 1: one element
    n_[0] = 1;
    a_[0] = b_[0] = 0;
    r = 1;
  }
  Shape4 sh{};
  for (int i = 0; i < kMaxRank; ++i) {
    const int src = i - (kMaxRank - r);
    sh.n[i] = src >= 0 ? n_[src] : 1;
    sh.sa[i] = src >= 0 ? a_[src] : 0;
    sh.sb[i] = src >= 0 ? b_[src] : 0;
  }
  switch (r) {
    case 1: return binary_launch_r<1>(s, op, a, b, out, sh, n);
    case 2: return binary_launch_r<2>(s, op, a, b, out, sh, n);
    case 3: return binary_launch_r<3>(s, op, a, b, out, sh, n);
    default: return binary_launch_r<4>(s, op, a, b, out, sh, n);
  }
}

hipError_t reduce_to_launch(hipStream_t s, const float* g, const long long* gshape, int grank, float* out,
                            const long long* tshape) {
  // tshape is aligned with gshape (same rank, 1 on the reduced axes).
  if (grank < 1 || grank > kMaxRank) return hipErrorInvalidValue;
  ReduceArgs r{};
  long long gstride[kMaxRank];
  long long stride = 1;
  for (int ax = grank - 1; ax >= 0; --ax) {
    gstride[ax] = stride;
    stride *= gshape[ax];
  }
  long long red_n[kMaxRank], red_s[kMaxRank];
  int n_red = 0;
  r.n_out = 1;
  for (int ax = 0; ax < grank; ++ax) {
    if (gshape[ax] == 1) continue;
    if (tshape[ax] == gshape[ax]) {
      r.keep_n[r.n_keep] = gshape[ax];
      r.keep_s[r.n_keep] = gstride[ax];
      ++r.n_keep;
      r.n_out *= gshape[ax];
    } else {
      if (tshape[ax] != 1) return hipErrorInvalidValue;
      red_n[n_red] = gshape[ax];
      red_s[n_red] = gstride[ax];
      ++n_red;
    }
  }
  for (int i = 0; i < kMaxRank; ++i) {  // pad the reduced axes in front with extent 1
    const int src = i - (kMaxRank - n_red);
    r.red_n[i] = src >= 0 ? red_n[src] : 1;
    r.red_s[i] = src >= 0 ? red_s[src] : 0;
  }
  if (r.n_out <= 0) return hipSuccess;
  // One reduced axis over one contiguous kept axis: columns of a matrix.  Up to
  // 4096 of them, a block per CU; more fill the chip with one thread each
  // (2048x16384 34.3 us, 43.2 in columns), and fewer than 32 rows are one batch
  // of loads there.
  constexpr long long kMax = 1LL << 30;  // row counts stay in int with a stage added
  if (n_red == 1 && r.n_keep == 1 && r.keep_s[0] == 1 && red_n[0] >= 32 && red_n[0] <= kMax && r.n_out <= 4096) {
    rt::launch(reduce_columns_kernel, dim3((unsigned)((r.n_out + kColCols - 1) / kColCols)), dim3(256), 0, s, g, out,
               (int)red_n[0], (int)r.n_out);
    return hipGetLastError();
  }
  rt::launch(reduce_to_kernel, dim3(grid_for(r.n_out)), dim3(256), 0, s, g, out, r);
  return hipGetLastError();
}

size_t sum_scratch_elems(long long n) { return (size_t)std::max<long long>(1, std::min<long long>((n + 65535) / 65536, 4096)); }

hipError_t sum_all_launch(hipStream_t s, const float* x, long long n, float div, float* out, float* scratch) {
  const long long parts = (long long)sum_scratch_elems(n);
  const long long chunk = std::max<long long>(1, (n + parts - 1) / parts);
  rt::launch(sum_stage1, dim3((unsigned)parts), dim3(256), 0, s, x, n, chunk, scratch, div, out);
  if (parts > 1) rt::launch(sum_stage2, dim3(1), dim3(256), 0, s, scratch, (int)parts, div, out);
  return hipGetLastError();
}

hipError_t scalar_fill_launch(hipStream_t s, const float* scalar, float div, const float* x, float* out, long long n) {
  if (n <= 0) return hipSuccess;
  rt::launch(scalar_fill_kernel, dim3(grid_for(n)), dim3(256), 0, s, scalar, div, x, out, n);
  return hipGetLastError();
}

static long long band_blocks(long long rows, int per) { return (rows + per - 1) / per; }

// f(first row, rows, grid, first block) per launch: a grid holds fewer than
// 2^32 threads (HIP takes a larger one and runs what is left of its size
// modulo 2^32), so 2^26 rows of 33 columns and more go in parts.
template <class F>
static hipError_t by_grid(long long rows, int per, int threads, F&& f) {
  const long long most = 0xffffffffLL / threads;
  for (long long b = 0, n = band_blocks(rows, per); b < n; b += most)
    f(b * per, std::min(rows - b * per, most * per), dim3((unsigned)std::min(n - b, most)), b);
  return hipGetLastError();
}

hipError_t softmax_rows_launch(hipStream_t s, const float* z, float* y, long long rows, long long cols) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (cols > kBandCols)
    return by_grid(rows, kLongRows, kRowThreads, [&](long long r0, long long n, dim3 grid, long long) {
      rt::launch(softmax_long_rows_kernel, grid, dim3(kRowThreads), 0, s, z + r0 * cols, y + r0 * cols, n, cols);
    });
  return by_row_length(cols, [&](auto band) {
    using B = decltype(band);
    return by_grid(rows, B::ROWS, B::T, [&](long long r0, long long n, dim3 grid, long long) {
      rt::launch(softmax_rows_kernel<B>, grid, dim3(B::T), 0, s, z + r0 * cols, y + r0 * cols, n, (int)cols);
    });
  });
}

hipError_t softmax_rows_vjp_launch(hipStream_t s, const float* sm, const float* g, float* dx, long long rows,
                                   long long cols) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  if (cols > kBandCols)
    return by_grid(rows, kLongRows, kRowThreads, [&](long long r0, long long n, dim3 grid, long long) {
      rt::launch(softmax_long_rows_vjp_kernel, grid, dim3(kRowThreads), 0, s, sm + r0 * cols, g + r0 * cols,
                 dx + r0 * cols, n, cols);
    });
  return by_row_length(cols, [&](auto band) {
    using B = decltype(band);
    return by_grid(rows, B::ROWS, B::T, [&](long long r0, long long n, dim3 grid, long long) {
      rt::launch(softmax_rows_vjp_kernel<B>, grid, dim3(B::T), 0, s, sm + r0 * cols, g + r0 * cols, dx + r0 * cols, n,
                 (int)cols);
    });
  });
}

// f(Band or void*) as the loss launch takes it: a thread per row of at most 7
// columns (256 x 2 3.5 us, 4.6 on kLossThreads; 256 x 5 4.0 and 4.6; 300000 x 5
// 10.5, 21.6 on lane groups; at 8 columns 18.9 and 22.2, but 256 x 8 5.1 and
// 4.7), one block of kLossThreads for a batch of narrow rows that fits it (a
// second launch, for the parts, costs more: 256 x 10 takes 4.8 us, 257 x 10
// 6.8), long or empty rows as null.
template <class F>
static hipError_t by_loss_shape(long long rows, long long cols, F&& f) {
  if (rows <= 0 || cols <= 0 || cols > kBandCols) return f(static_cast<void*>(nullptr));
  if (cols <= 4) return f(Band<1, 4, 1, kRowThreads>{});
  if (cols <= 7) return f(Band<1, 8, 1, kRowThreads>{});
  if (cols <= 16 && rows <= 256) return f(Band<16, 1, 4, kLossThreads>{});
  return by_row_length(cols, f);
}

size_t xent_logits_parts(long long rows, long long cols) {
  size_t n = 1;
  (void)by_loss_shape(rows, cols, [&](auto band) {
    using B = decltype(band);
    if constexpr (std::is_pointer_v<B>) n = (size_t)std::max<long long>(1, band_blocks(rows, kLongRows));
    else n = (size_t)band_blocks(rows, B::ROWS);
    return hipSuccess;
  });
  return n;
}

hipError_t xent_logits_launch(hipStream_t s, const float* z, const float* y, float* dir, long long rows,
                              long long cols, float div, float* out, float* scratch, size_t scratch_elems,
                              float dir_scale) {
  const size_t blocks = xent_logits_parts(rows, cols);
  if (blocks > 1 && blocks > scratch_elems) return hipErrorInvalidValue;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  float* const part = blocks > 1 ? scratch : nullptr;
  hipError_t e = by_loss_shape(rows, cols, [&](auto band) {
    using B = decltype(band);
    if constexpr (std::is_pointer_v<B>)
      // One block where there is nothing to load.
      return by_grid(std::max(rows, 1LL), kLongRows, kRowThreads, [&](long long r0, long long n, dim3 grid, long long b) {
        rt::launch(xent_logits_long_kernel, grid, dim3(kRowThreads), 0, s, z + r0 * cols, y + r0 * cols, dir + r0 * cols,
                   std::min(n, rows), cols, part ? part + b : part, div, out, dir_scale);
      });
    else
      return by_grid(rows, B::ROWS, B::T, [&](long long r0, long long n, dim3 grid, long long b) {
        rt::launch(xent_logits_kernel<B>, grid, dim3(B::T), 0, s, z + r0 * cols, y + r0 * cols, dir + r0 * cols, n,
                   (int)cols, part ? part + b : part, div, out, dir_scale);
      });
  });
  if (e == hipSuccess && blocks > 1) {
    rt::launch(sum_stage2, dim3(1), dim3(256), 0, s, scratch, (int)blocks, div, out);
    e = hipGetLastError();
  }
  return e;
}

hipError_t loss_terms_launch(hipStream_t s, int kind, const float* p, const float* y, float* term, float* dir,
                             long long n) {
  if (n <= 0) return hipSuccess;
  rt::launch(loss_terms_kernel, dim3(grid_for(n)), dim3(256), 0, s, kind, p, y, term, dir, n);
  return hipGetLastError();
}

}  // namespace rt

// ------------------------------------------------------------------ C ABI
using namespace rt;

namespace {

bool is_f32(const rt_buf* b) { return b && b->dtype == RT_F32; }

// Shape of b right-aligned to rank r with leading 1s.
void aligned_shape(const rt_buf* b, int r, long long* out) {
  for (int i = 0; i < r; ++i) {
    const int src = i - (r - b->rank);
    out[i] = src >= 0 ? (long long)b->shape[src] : 1;
  }
}

// Strides of b in the index space of an output of rank r and shape `shape`
// (0 on axes where b has extent 1 and the output does not).
void broadcast_strides(const rt_buf* b, int r, const long long* shape, long long* out) {
  long long bs[kMaxRank];
  aligned_shape(b, r, bs);
  long long acc = 1;
  for (int i = r - 1; i >= 0; --i) {
    out[i] = (bs[i] == shape[i]) ? acc : 0;
    acc *= bs[i];
  }
}

bool needs_x(int op) {
  return op == RT_U_SQUARE || op == RT_U_LN || op == RT_U_RELU || op == RT_U_LEAKY_RELU;
}
bool needs_y(int op) { return op == RT_U_SQRT || op == RT_U_EXP || op == RT_U_SIGMOID || op == RT_U_TANH; }

const char* kUnaryNames[] = {"map_scale", "map_offset", "map_neg",  "map_square", "map_sqrt", "map_exp",
                             "map_ln",    "map_relu",   "map_leaky", "map_sigmoid", "map_tanh"};

}  // namespace

extern "C" {

int rt_map(rt_ctx* c, rt_unary_op op, float k, const rt_buf* x, rt_buf* y) {
  CHECK_CTX(c);
  if (!x || !y) return fail(c, RT_ERR_INVALID, "null buffer");
  if (op < RT_U_SCALE || op > RT_U_TANH) return fail(c, RT_ERR_INVALID, "unknown unary op %d", (int)op);
  if (!is_f32(x) || !is_f32(y)) return fail(c, RT_ERR_DTYPE, "map takes f32");
  if (x->n != y->n) return fail(c, RT_ERR_SHAPE, "map: %zu elements into %zu", x->n, y->n);
  Launch L(c, kUnaryNames[op]);
  HIP_TRY(c, unary_launch(c->stream, op, k, static_cast<const float*>(x->ptr), static_cast<float*>(y->ptr), x->n),
          "map");
  return RT_OK;
}

int rt_map_vjp(rt_ctx* c, rt_unary_op op, float k, const rt_buf* g, const rt_buf* x, const rt_buf* y, rt_buf* dx) {
  CHECK_CTX(c);
  if (!g || !dx) return fail(c, RT_ERR_INVALID, "null buffer");
  if (op < RT_U_SCALE || op > RT_U_TANH) return fail(c, RT_ERR_INVALID, "unknown unary op %d", (int)op);
  if (needs_x(op) && !x) return fail(c, RT_ERR_INVALID, "this VJP needs the op's input");
  if (needs_y(op) && !y) return fail(c, RT_ERR_INVALID, "this VJP needs the op's output");
  if (!is_f32(g) || !is_f32(dx) || (x && !is_f32(x)) || (y && !is_f32(y))) return fail(c, RT_ERR_DTYPE, "f32 only");
  if (g->n != dx->n || (x && x->n != g->n) || (y && y->n != g->n))
    return fail(c, RT_ERR_SHAPE, "map_vjp: operands differ in size");
  Launch L(c, "map_vjp");
  HIP_TRY(c,
          unary_vjp_launch(c->stream, op, k, static_cast<const float*>(g->ptr),
                           needs_x(op) ? static_cast<const float*>(x->ptr) : nullptr,
                           needs_y(op) ? static_cast<const float*>(y->ptr) : nullptr, static_cast<float*>(dx->ptr),
                           g->n),
          "map_vjp");
  return RT_OK;
}

int rt_zip(rt_ctx* c, rt_binary_op op, const rt_buf* a, const rt_buf* b, rt_buf* out) {
  CHECK_CTX(c);
  if (!a || !b || !out) return fail(c, RT_ERR_INVALID, "null buffer");
  if (op < RT_B_ADD || op > RT_B_DIV) return fail(c, RT_ERR_INVALID, "unknown binary op %d", (int)op);
  if (!is_f32(a) || !is_f32(b) || !is_f32(out)) return fail(c, RT_ERR_DTYPE, "zip takes f32");
  const int r = std::max(std::max(a->rank, b->rank), 1);
  long long sa_shape[kMaxRank], sb_shape[kMaxRank], shape[kMaxRank];
  aligned_shape(a, r, sa_shape);
  aligned_shape(b, r, sb_shape);
  for (int i = 0; i < r; ++i) {
    if (sa_shape[i] == sb_shape[i] || sb_shape[i] == 1) shape[i] = sa_shape[i];
    else if (sa_shape[i] == 1) shape[i] = sb_shape[i];
    else return fail(c, RT_ERR_SHAPE, "shapes do not broadcast (axis %d: %lld vs %lld)", i, sa_shape[i], sb_shape[i]);
  }
  // out must have exactly the broadcast shape (leading 1s may be dropped).
  long long os[kMaxRank];
  if (out->rank > r) return fail(c, RT_ERR_SHAPE, "zip output rank too large");
  aligned_shape(out, r, os);
  for (int i = 0; i < r; ++i)
    if (os[i] != shape[i]) return fail(c, RT_ERR_SHAPE, "zip output does not have the broadcast shape");
  // Aliasing is allowed only between same-shaped tensors (elementwise in place).
  if ((out->ptr == a->ptr && a->n != out->n) || (out->ptr == b->ptr && b->n != out->n))
    return fail(c, RT_ERR_INVALID, "zip output aliases a broadcast operand");
  if (out->n == 0) return RT_OK;
  long long sa[kMaxRank], sb[kMaxRank];
  broadcast_strides(a, r, shape, sa);
  broadcast_strides(b, r, shape, sb);
  Launch L(c, "zip");
  HIP_TRY(c,
          binary_launch(c->stream, op, static_cast<const float*>(a->ptr), sa, static_cast<const float*>(b->ptr), sb,
                        static_cast<float*>(out->ptr), shape, r),
          "zip");
  return RT_OK;
}

int rt_sum_all(rt_ctx* c, const rt_buf* x, float div, rt_buf* out) {
  CHECK_CTX(c);
  if (!x || !out) return fail(c, RT_ERR_INVALID, "null buffer");
  if (!is_f32(x) || !is_f32(out)) return fail(c, RT_ERR_DTYPE, "sum_all takes f32");
  if (out->n != 1) return fail(c, RT_ERR_SHAPE, "sum_all writes one element");
  int rc = ensure_scratch(c, sum_scratch_elems((long long)x->n));
  if (rc) return rc;
  Launch L(c, "sum_all");
  HIP_TRY(c,
          sum_all_launch(c->stream, static_cast<const float*>(x->ptr), (long long)x->n, div,
                         static_cast<float*>(out->ptr), c->scratch),
          "sum_all");
  return RT_OK;
}

int rt_reduce_to(rt_ctx* c, const rt_buf* g, rt_buf* out) {
  CHECK_CTX(c);
  if (!g || !out) return fail(c, RT_ERR_INVALID, "null buffer");
  if (!is_f32(g) || !is_f32(out)) return fail(c, RT_ERR_DTYPE, "reduce_to takes f32");
  const int r = std::max(g->rank, 1);
  if (out->rank > r) return fail(c, RT_ERR_SHAPE, "reduce_to target has a larger rank than the source");
  long long gs[kMaxRank], ts[kMaxRank];
  aligned_shape(g, r, gs);
  aligned_shape(out, r, ts);
  for (int i = 0; i < r; ++i)
    if (ts[i] != gs[i] && ts[i] != 1)
      return fail(c, RT_ERR_SHAPE, "reduce_to: target axis %d is %lld, source %lld", i, ts[i], gs[i]);
  if (out->n == g->n) {
    // Same shape: the reference returns a copy (tensor.rs:400-402).
    if (out->ptr != g->ptr && g->n > 0)
      HIP_TRY(c, hipMemcpyAsync(out->ptr, g->ptr, g->bytes, hipMemcpyDeviceToDevice, c->stream), "reduce_to copy");
    return RT_OK;
  }
  if (out->n == 1) return rt_sum_all(c, g, 1.0f, out);  // tensor.rs:406-409
  Launch L(c, "reduce_to");
  HIP_TRY(c, reduce_to_launch(c->stream, static_cast<const float*>(g->ptr), gs, r, static_cast<float*>(out->ptr), ts),
          "reduce_to");
  return RT_OK;
}

int rt_fill_scaled(rt_ctx* c, const rt_buf* s, float div, const rt_buf* x, rt_buf* out) {
  CHECK_CTX(c);
  if (!s || !out) return fail(c, RT_ERR_INVALID, "null buffer");
  if (!is_f32(s) || !is_f32(out) || (x && !is_f32(x))) return fail(c, RT_ERR_DTYPE, "fill_scaled takes f32");
  if (s->n != 1) return fail(c, RT_ERR_SHAPE, "the scale must have one element");
  if (x && x->n != out->n) return fail(c, RT_ERR_SHAPE, "fill_scaled: x and out differ in size");
  Launch L(c, "fill_scaled");
  HIP_TRY(c,
          scalar_fill_launch(c->stream, static_cast<const float*>(s->ptr), div,
                             x ? static_cast<const float*>(x->ptr) : nullptr, static_cast<float*>(out->ptr),
                             (long long)out->n),
          "fill_scaled");
  return RT_OK;
}

int rt_softmax_rows(rt_ctx* c, const rt_buf* z, rt_buf* y) {
  CHECK_CTX(c);
  if (!z || !y) return fail(c, RT_ERR_INVALID, "null buffer");
  if (!is_f32(z) || !is_f32(y)) return fail(c, RT_ERR_DTYPE, "softmax_rows takes f32");
  if (z->rank != 2) return fail(c, RT_ERR_SHAPE, "softmax_rows needs rank 2");
  if (y->n != z->n) return fail(c, RT_ERR_SHAPE, "softmax_rows: output size");
  Launch L(c, "softmax_rows");
  HIP_TRY(c,
          softmax_rows_launch(c->stream, static_cast<const float*>(z->ptr), static_cast<float*>(y->ptr),
                              (long long)z->shape[0], (long long)z->shape[1]),
          "softmax_rows");
  return RT_OK;
}

int rt_softmax_rows_vjp(rt_ctx* c, const rt_buf* s, const rt_buf* g, rt_buf* dx) {
  CHECK_CTX(c);
  if (!s || !g || !dx) return fail(c, RT_ERR_INVALID, "null buffer");
  if (!is_f32(s) || !is_f32(g) || !is_f32(dx)) return fail(c, RT_ERR_DTYPE, "f32 only");
  if (s->rank != 2) return fail(c, RT_ERR_SHAPE, "softmax VJP needs rank 2");
  if (g->n != s->n || dx->n != s->n) return fail(c, RT_ERR_SHAPE, "softmax VJP: operands differ in size");
  Launch L(c, "softmax_rows_vjp");
  HIP_TRY(c,
          softmax_rows_vjp_launch(c->stream, static_cast<const float*>(s->ptr), static_cast<const float*>(g->ptr),
                                  static_cast<float*>(dx->ptr), (long long)s->shape[0], (long long)s->shape[1]),
          "softmax_rows_vjp");
  return RT_OK;
}

int rt_loss(rt_ctx* c, rt_loss_kind kind, const rt_buf* p, const rt_buf* y, rt_buf* value, rt_buf* dir) {
  CHECK_CTX(c);
  if (!p || !value) return fail(c, RT_ERR_INVALID, "null buffer");
  if (kind != RT_LOSS_MAE && kind != RT_LOSS_SOFTMAX_XENT && kind != RT_LOSS_BCE &&
      kind != RT_LOSS_SOFTMAX_XENT_LOGITS && kind != RT_LOSS_SOFTMAX_XENT_LOGITS_MEAN)
    return fail(c, RT_ERR_INVALID, "unknown loss kind %d", (int)kind);
  if (kind != RT_LOSS_MAE && !y) return fail(c, RT_ERR_INVALID, "this loss needs targets");
  if (!is_f32(p) || !is_f32(value) || (y && !is_f32(y)) || (dir && !is_f32(dir)))
    return fail(c, RT_ERR_DTYPE, "losses take f32");
  if (value->n != 1) return fail(c, RT_ERR_SHAPE, "the loss value has one element");
  if (y && y->n != p->n) return fail(c, RT_ERR_SHAPE, "predictions and targets differ in size");
  if (dir && dir->n != p->n) return fail(c, RT_ERR_SHAPE, "dir must match the predictions");
  float batch = (float)p->n;
  if (kind == RT_LOSS_SOFTMAX_XENT_LOGITS || kind == RT_LOSS_SOFTMAX_XENT_LOGITS_MEAN) {
    if (p->rank != 2 || y->rank != 2 || y->shape[0] != p->shape[0] || y->shape[1] != p->shape[1])
      return fail(c, RT_ERR_SHAPE, "logits and targets differ in shape");  // losses.rs:100
    if (!dir) return fail(c, RT_ERR_INVALID, "the logits form writes dir (it holds the softmax on the way)");
    const long long rows = (long long)p->shape[0], cols = (long long)p->shape[1];
    int rc = ensure_scratch(c, xent_logits_parts(rows, cols));
    if (rc) return rc;
    Launch L(c, "loss");
    HIP_TRY(c,
            xent_logits_launch(c->stream, static_cast<const float*>(p->ptr), static_cast<const float*>(y->ptr),
                               static_cast<float*>(dir->ptr), rows, cols, (float)rows, static_cast<float*>(value->ptr),
                               c->scratch, c->scratch_elems,
                               kind == RT_LOSS_SOFTMAX_XENT_LOGITS_MEAN ? 1.0f / (float)rows : 1.0f),
            "softmax-xent");
    return RT_OK;
  }
  if (kind == RT_LOSS_SOFTMAX_XENT) {
    if (p->rank != 2) return fail(c, RT_ERR_SHAPE, "softmax cross-entropy takes [batch, classes]");
    if (y->rank != 2 || y->shape[0] != p->shape[0] || y->shape[1] != p->shape[1])
      return fail(c, RT_ERR_SHAPE, "logits and targets differ in shape");  // losses.rs:100
    batch = (float)p->shape[0];
  }
  const long long n = (long long)p->n;
  const size_t parts = sum_scratch_elems(n);
  int rc = ensure_scratch(c, (size_t)n + parts);
  if (rc) return rc;
  float* term = c->scratch + parts;
  Launch L(c, "loss");
  HIP_TRY(c,
          loss_terms_launch(c->stream, kind, static_cast<const float*>(p->ptr),
                            y ? static_cast<const float*>(y->ptr) : nullptr, term,
                            dir ? static_cast<float*>(dir->ptr) : nullptr, n),
          "loss terms");
  HIP_TRY(c, sum_all_launch(c->stream, term, n, batch, static_cast<float*>(value->ptr), c->scratch), "loss sum");
  return RT_OK;
}

}  // extern "C"
