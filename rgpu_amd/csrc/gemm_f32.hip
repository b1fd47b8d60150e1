// f32 GEMM on CDNA4 matrix cores.
//
// Replaces rtensor's MM_FAST / MM_EPILOGO / MM_SPLITK WGSL kernels
// (crates/rtensor/src/gpu/gemm.rs:65-494, splitk.rs:33-237) for the three
// operand layouts of the training step:
//   NN  C = A·B      A [M,K] (K contiguous),  B [K,N] (N contiguous)  forward
//   TN  C = Aᵀ·B     A [K,M] (M contiguous),  B [K,N] (N contiguous)  dW = Xᵀ·δ
//   NT  C = A·Bᵀ     A [M,K] (K contiguous),  B [N,K] (K contiguous)  dX = δ·Wᵀ
//
// Five kernels share the work (dispatch_tile):
//   F32Split    f32 by exact splits on the bf16 matrix units: most products
//   F32Dma      v_mfma_f32_16x16x4_f32 fed by direct-to-LDS loads: whole 64x64
//               tiles over a short K (dma_better)
//   F32Tile     the same MFMA, register-staged, any shape: weight gradients
//               over few rows (row_order_tn), short products (short_k)
//   F32RankK    dX of a narrow layer (K <= 16)
//   gemm_f32_skinny_kernel   at most 64 rows of output
//
// Epilogues run on the accumulators in registers: bias, bias+ReLU (forward,
// mm_bias in gemm.rs:452-493) and the ReLU mask (δ ← acc ⊙ 1[A>0], fusing
// RELU_BWD, kernels.rs:119-131).  For TN with a colsum target the blocks of
// the first M tile also sum the B values they stage over K: that is
// db = 1ᵀ·δ (COLSUM, kernels.rs:182-199) at no extra HBM traffic.
// With more than one K slice, each slice writes a raw f32 partial plane and
// splitk_reduce sums the planes in slice order (REDUZ, splitk.rs:240-256):
// deterministic, no float atomics.

#include "device_util.h"
#include "optim_dev.h"
#include "rt_internal.h"

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

struct F32Args {
  const float* A;
  const float* B;
  float* C;
  int M, N, K, lda, ldb, ldc;
  int epi;
  const float* bias;
  const float* mask;
  float* colsum;  // [N], or [splits, N] partial rows when splits > 1
  int k_per_split;
  long long split_stride;
  int tiles_m, tiles_n, splits;
  int vec_a, vec_b, vec_c;
};

// Consecutive workgroups go to different XCDs (round robin over 8), each
// with its own L2.  Renumber so that every XCD gets a contiguous run of
// tile indices; the grouped raster below then keeps the tiles resident on
// one XCD sharing A rows and B columns.
__device__ inline int xcd_local(int bid, int nb) { return (nb & 7) == 0 ? (bid & 7) * (nb >> 3) + (bid >> 3) : bid; }

// Loads `cnt` consecutive floats (cnt = 1, 2 or 4) from LDS as one access.
template <int CNT>
__device__ inline void lds_read(const float* p, float* out) {
  if constexpr (CNT == 4) {
    f4 v = *reinterpret_cast<const f4*>(p);
    out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; out[3] = v[3];
  } else if constexpr (CNT == 2) {
    f2 v = *reinterpret_cast<const f2*>(p);
    out[0] = v[0]; out[1] = v[1];
  } else {
    out[0] = p[0];
  }
}

// Global -> register load of one float4 of an operand tile.  `row`/`col`
// index the stored matrix (row-major, leading dimension ld); the 4 elements
// run along the contiguous dimension.  Out-of-range elements read as 0.
__device__ inline f4 load4(const float* base, int ld, int row, int col, int rows, int cols, int vec) {
  const float* src = base + (long long)row * ld + col;
  if (vec && row < rows && col + 3 < cols) return *reinterpret_cast<const f4*>(src);
  f4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (row < rows && col + e < cols) ? src[e] : 0.0f;
  return v;
}

// One block's work: tile `bid` (already XCD-renumbered, in [0, tiles)) of
// K slice `split`, with v_mfma_f32_16x16x4_f32, every access bounds-checked:
// short weight gradients (row_order_tn), other short products (short_k) and
// operands whose rows are too long for the tiles below.
//
// Four wave64s in a 2x2 arrangement, K staged through LDS 32 at a time,
// double-buffered with register staging (one barrier per K step).  A 16x16x4
// MFMA takes, in lane l = 16g + r, the A value (row r, k g) and the B value
// (k g, col r), and returns D(4g+q, r) in accumulator register q.  Rows,
// columns and k inside a wave tile may be permuted freely as long as A and B
// agree on k, so MFMA row r of row-tile t is wave row TM*r + t (likewise the
// columns), and within a 16-wide k chunk MFMA step s of lane group g uses k =
// 4g + s: one LDS vector read serves a lane's tiles or steps.
template <bool A_KC, bool B_KC, int BN_ = 64>
struct F32Tile {
  static constexpr int THREADS = 256, BM = 64, BN = BN_, BK = 32;
  static constexpr int PAD = 4;
  static constexpr int TM = BM / 32, TN = BN / 32;  // MFMA tiles per wave (2x2 waves of BM/2 x BN/2)
  static constexpr int A_STRIDE = A_KC ? (BK + PAD) : (BM + PAD);
  static constexpr int B_STRIDE = B_KC ? (BK + PAD) : (BN + PAD);
  static constexpr int A_ELEMS = A_KC ? BM * A_STRIDE : BK * A_STRIDE;
  static constexpr int B_ELEMS = B_KC ? BN * B_STRIDE : BK * B_STRIDE;
  static constexpr int SMEM = 2 * (A_ELEMS + B_ELEMS);  // floats: two stages of both operands
  static constexpr int A_LD = BM * BK / 4 / THREADS;    // float4 loads per thread per K step
  static constexpr int B_LD = BN * BK / 4 / THREADS;
  static constexpr int SUB = BK / 16;

  __device__ static void run(const F32Args& p, int bid, int split, float* smem);
};

template <bool A_KC, bool B_KC, int BN_>
__device__ void F32Tile<A_KC, B_KC, BN_>::run(const F32Args& p, int bid, int split, float* smem) {
  float* const sA0 = smem;
  float* const sB0 = smem + 2 * A_ELEMS;
  auto sA = [&](int buf) { return sA0 + buf * A_ELEMS; };
  auto sB = [&](int buf) { return sB0 + buf * B_ELEMS; };

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);

  constexpr int GROUP = 8;
  const int per_group = GROUP * p.tiles_n;
  const int grp = bid / per_group;
  const int first_m = grp * GROUP;
  const int gsize = min(p.tiles_m - first_m, GROUP);
  const int in_grp = bid - grp * per_group;
  const int tile_m = first_m + in_grp % gsize;
  const int tile_n = in_grp / gsize;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int kb = split * p.k_per_split;
  const int ke = min(p.K, kb + p.k_per_split);
  const int nk = ke > kb ? (ke - kb + BK - 1) / BK : 0;

  auto load_tiles = [&](f4 (&ra)[A_LD], f4 (&rb)[B_LD], int k0) {
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      const int idx = tid + THREADS * i;
      if constexpr (A_KC) {
        const int rr = idx / (BK / 4), kq = idx % (BK / 4);
        ra[i] = load4(p.A, p.lda, m0 + rr, k0 + 4 * kq, p.M, ke, p.vec_a);
      } else {
        constexpr int Q = BM / 4;
        const int kk = idx / Q, mq = idx % Q;
        ra[i] = load4(p.A, p.lda, k0 + kk, m0 + 4 * mq, ke, p.M, p.vec_a);
      }
    }
#pragma unroll
    for (int i = 0; i < B_LD; ++i) {
      const int idx = tid + THREADS * i;
      if constexpr (B_KC) {
        const int rr = idx / (BK / 4), kq = idx % (BK / 4);
        rb[i] = load4(p.B, p.ldb, n0 + rr, k0 + 4 * kq, p.N, ke, p.vec_b);
      } else {
        constexpr int Q = BN / 4;
        const int kk = idx / Q, nq = idx % Q;
        rb[i] = load4(p.B, p.ldb, k0 + kk, n0 + 4 * nq, ke, p.N, p.vec_b);
      }
    }
  };
  auto store_tiles = [&](const f4 (&ra)[A_LD], const f4 (&rb)[B_LD], int buf) {
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      const int idx = tid + THREADS * i;
      if constexpr (A_KC) {
        *reinterpret_cast<f4*>(&sA(buf)[(idx / (BK / 4)) * A_STRIDE + 4 * (idx % (BK / 4))]) = ra[i];
      } else {
        constexpr int Q = BM / 4;
        *reinterpret_cast<f4*>(&sA(buf)[(idx / Q) * A_STRIDE + 4 * (idx % Q)]) = ra[i];
      }
    }
#pragma unroll
    for (int i = 0; i < B_LD; ++i) {
      const int idx = tid + THREADS * i;
      if constexpr (B_KC) {
        *reinterpret_cast<f4*>(&sB(buf)[(idx / (BK / 4)) * B_STRIDE + 4 * (idx % (BK / 4))]) = rb[i];
      } else {
        constexpr int Q = BN / 4;
        *reinterpret_cast<f4*>(&sB(buf)[(idx / Q) * B_STRIDE + 4 * (idx % Q)]) = rb[i];
      }
    }
  };

  f4 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < TN; ++u) acc[t][u] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  auto compute = [&](int buf) {
    const float* as = sA(buf);
    const float* bs = sB(buf);
#pragma unroll
    for (int ss = 0; ss < SUB; ++ss) {
      float af[TM][4], bf[TN][4];
      if constexpr (A_KC) {
#pragma unroll
        for (int t = 0; t < TM; ++t) lds_read<4>(&as[(wm + TM * r + t) * A_STRIDE + ss * 16 + 4 * g], af[t]);
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float tmp[TM];
          lds_read<TM>(&as[(ss * 16 + 4 * g + s) * A_STRIDE + wm + TM * r], tmp);
#pragma unroll
          for (int t = 0; t < TM; ++t) af[t][s] = tmp[t];
        }
      }
      if constexpr (B_KC) {
#pragma unroll
        for (int u = 0; u < TN; ++u) lds_read<4>(&bs[(wn + TN * r + u) * B_STRIDE + ss * 16 + 4 * g], bf[u]);
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          float tmp[TN];
          lds_read<TN>(&bs[(ss * 16 + 4 * g + s) * B_STRIDE + wn + TN * r], tmp);
#pragma unroll
          for (int u = 0; u < TN; ++u) bf[u][s] = tmp[u];
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
          for (int u = 0; u < TN; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[t][s], bf[u][s], acc[t][u], 0, 0, 0);
    }
  };

  // Column sums of B (the bias gradient when B = δ), from the LDS tiles of
  // the first M tile's blocks, summed over k in increasing order.
  const bool do_cs = !B_KC && p.colsum != nullptr && tile_m == 0 && tid < BN;
  float cs = 0.0f;
  auto colsum = [&](int buf) {
    if constexpr (!B_KC) {
      if (do_cs) {
        const float* bs = sB(buf);
#pragma unroll 8
        for (int kk = 0; kk < BK; ++kk) cs += bs[kk * B_STRIDE + tid];
      }
    }
  };

  if (nk > 0) {
    f4 ra[A_LD], rb[B_LD];
    load_tiles(ra, rb, kb);
    store_tiles(ra, rb, 0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
      if (kt + 1 < nk) load_tiles(ra, rb, kb + (kt + 1) * BK);
      compute(cur);
      colsum(cur);
      if (kt + 1 < nk) store_tiles(ra, rb, cur ^ 1);
      __syncthreads();
    }
  }

  if (do_cs && n0 + tid < p.N) p.colsum[(long long)split * p.N + n0 + tid] = cs;

  // Epilogue.  Lane owns rows m0+wm+TM*(4g+q)+t and columns n0+wn+TN*r+u.
  const bool partial = p.splits > 1;
  float* Cout = p.C + (long long)split * p.split_stride;
  const int col0 = n0 + wn + TN * r;
  float bias_v[TN];
#pragma unroll
  for (int u = 0; u < TN; ++u)
    bias_v[u] = (!partial && p.bias != nullptr && col0 + u < p.N) ? p.bias[col0 + u] : 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      const int row = m0 + wm + TM * (4 * g + q) + t;
      if (row >= p.M) continue;
      float v[TN];
#pragma unroll
      for (int u = 0; u < TN; ++u) v[u] = acc[t][u][q];
      if (!partial) {
        if (p.epi == RT_EPI_BIAS || p.epi == RT_EPI_BIAS_RELU) {
#pragma unroll
          for (int u = 0; u < TN; ++u) v[u] = v[u] + bias_v[u];
          if (p.epi == RT_EPI_BIAS_RELU) {
#pragma unroll
            for (int u = 0; u < TN; ++u) v[u] = fmaxf(v[u], 0.0f);
          }
        } else if (p.epi == RT_EPI_RELU_MASK) {
          const float* mrow = p.mask + (long long)row * p.ldc;
#pragma unroll
          for (int u = 0; u < TN; ++u)
            if (col0 + u < p.N && !(mrow[col0 + u] > 0.0f)) v[u] = 0.0f;
        }
      }
      float* dst = Cout + (long long)row * p.ldc + col0;
#pragma unroll
      for (int u = 0; u < TN; ++u)
        if (col0 + u < p.N) dst[u] = v[u];
    }
  }
}

// ---------------------------------------------------------------- f32 tile on the bf16 matrix units
// An f32 value is the exact sum of three bf16 values: hi = bf16(x), mid =
// bf16(x - hi), lo = bf16(x - hi - mid), each remainder exact in f32 (8 + 8 +
// 8 significant bits).  A product of two f32 values is then nine bf16
// products, each exact in the MFMA's f32 accumulator; the three smallest (mid
// lo, lo mid, lo lo: below 2^-26 of the product, against the 2^-24 that each
// f32 sum rounds by) are left out, and six v_mfma_f32_16x16x32_bf16 replace
// eight v_mfma_f32_16x16x4_f32 at 16 times their rate.
//
// Operands are split after a multiplication by 2^16: the smallest bit of an
// f32, 2^-149, is then 2^-133, that of a bf16, so the split is exact down to
// the last subnormal (the conversions, the remainders and the MFMA keep
// subnormals); unscaled, an operand below 2^-109 lost its last part and one
// below 2^-134 was taken as zero.  The sums are scaled back at the end.  What
// the scale costs at the other end is left to the f32 MFMA: operands of 2^111
// and sums of 2^96 (8e28) or more become infinities here.
//
// Block: 256 threads, 4 waves stacked along M, each 16 TM rows by all BN =
// 16 TN columns.  A wave loads its own A rows straight into registers in
// fragment order (nothing shares them) and splits them there; B, which all
// four waves read, is loaded by the block, split once and put into LDS as
// three bf16 planes [col][64 k] (16-byte granule j of column c at j ^ ((c >>
// 1) & 7), for the fragment reads; 18 to 25% of the LDS cycles are conflicts,
// of an LDS that is active 5% of the time).  Stages are 64 k: the global loads
// of a stage go out one stage ahead, its split runs between the MFMAs of the
// stage before it, one barrier per stage.  MFMAs take the operands swapped, so
// lane (g, r) ends with C(row 16t + r, columns 16u + 4g .. + 3): float4 stores.
//
// An operand that is not finite has hi = itself, so the hi hi products alone
// give what f32 arithmetic gives (the small ones hold inf - inf and inf times a
// zero part, and are left out).  A sum or an operand that left the scaled range
// looks the same: a block that finds a result that is not finite reads its
// operands once more, and unless their size rules that out its waves compute
// their tiles again with the f32 MFMA.  2048^3 NN, 98 us: with an infinity or a
// NaN 187 us, all of a row 209 (recomputed 345 and 490, on the f32 MFMA alone
// 125), with sums beyond 2^96 377; looking costs 0.1 us where nothing is found.
constexpr float kSplitScale = 65536.0f, kUnsplit = 1.0f / kSplitScale;
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));

// The two selectors of split8's remainders: dot2(hi pair, {-1, 0}) + x0.
// Held in registers: as literals they were encoded into the instruction with
// the halves exchanged.
struct SplitSel {
  b2 first, second;
  __device__ inline SplitSel() {
    first = b2{(__bf16)-1.0f, (__bf16)0.0f};
    second = b2{(__bf16)0.0f, (__bf16)-1.0f};
    asm volatile("" : "+v"(first), "+v"(second));
  }
};

// Eight f32 values times kSplitScale into their three bf16 planes, 9 VALU
// instructions a pair, in 18 steps of two: step Q of the eight values x
// (overwritten by their remainders).  Breadth first, so that no step needs the
// result of the one before it.
constexpr int kScaleSteps = 4, kSplitSteps = kScaleSteps + 14;
// The plane that step Q completes, -1 if none.
constexpr int plane_done(int Q) {
  return Q == kScaleSteps + 1 ? 0 : Q == kScaleSteps + 7 ? 1 : Q == kScaleSteps + 13 ? 2 : -1;
}
template <int Q>
__device__ __forceinline__ void split_step(float (&x)[8], const SplitSel& sel, u4 (&out)[3]) {
  constexpr int s = Q - kScaleSteps, plane = s < 6 ? 0 : s < 12 ? 1 : 2, q = s % 6;
  if constexpr (s < 0) {
    x[2 * Q] *= kSplitScale;
    x[2 * Q + 1] *= kSplitScale;
  } else if constexpr (q < 2) {
#pragma unroll
    for (int i = 2 * q; i < 2 * q + 2; ++i)
      out[plane][i] = __builtin_bit_cast(unsigned, __builtin_convertvector((f2{x[2 * i], x[2 * i + 1]}), b2));
  } else {
    constexpr int i = q - 2;
    const b2 h = __builtin_bit_cast(b2, (unsigned)out[plane][i]);
    x[2 * i] = __builtin_amdgcn_fdot2_f32_bf16(h, sel.first, x[2 * i], false);
    x[2 * i + 1] = __builtin_amdgcn_fdot2_f32_bf16(h, sel.second, x[2 * i + 1], false);
  }
}

// A tile's plain stores (F32Split::run's default epilogue).
struct NoEpi {
  static constexpr bool kOn = false;
};

template <int TM_, int TN_, bool A_KC, bool B_KC>
struct F32Split {
  static constexpr int TM = TM_, TN = TN_;
  static constexpr int THREADS = 256, BM = 64 * TM, BN = 16 * TN, BK = 64, KK = BK / 32;
  static constexpr int PLANE = BN * BK;             // halves
  static constexpr int SMEM = 2 * 3 * PLANE / 2;    // floats: two stages of three planes
  static constexpr int UNITS = BN * BK / 8;         // (column, 8-k granule) units of B per stage
  static constexpr int UPT = UNITS / THREADS;
  static constexpr bool CS = !A_KC && !B_KC;  // column sums of B: TN only
  static_assert(TN % 2 == 0 && UNITS % THREADS == 0, "tile");

  template <class Epi = NoEpi>
  __device__ static void run(const F32Args& p, int bid, int split, float* smem, const Epi& e = Epi{});
  __device__ static bool may_overflow(const F32Args& p, int m0, int n0, int kb, int ke, float* smem, int tid);
  __device__ static void plain_f32(const F32Args& p, f4 (&acc)[TM][TN], int row0, int n0, int kb, int ke, int g,
                                   int r);
  // The k that element e of granule j stands for within a stage.  An MFMA may
  // take its 32 k in any order as long as A and B agree; this one makes the
  // 16-byte loads of four neighbouring granules of a row contiguous.
  __device__ static constexpr int k_of(int j, int e) { return 32 * (j / 4) + 4 * (j % 4) + (e < 4 ? e : 12 + e); }
  // Place of granule j (8 k) of column c in an LDS plane (halves).
  __device__ static inline int place(int c, int j) { return c * BK + 8 * (j ^ ((c >> 1) & 7)); }
};

__device__ inline bool finite4(const f4& v) {
  return fabsf(v[0]) <= 3.402823466e38f && fabsf(v[1]) <= 3.402823466e38f && fabsf(v[2]) <= 3.402823466e38f &&
         fabsf(v[3]) <= 3.402823466e38f;
}

// 16 k of T row (or column) tiles of an operand from k0: lane (g, r) gets rows
// row0 + 16t + r (past the last one, that one again), k0 + 4g .. + 3; unless
// WHOLE, zero from ke on.
template <bool KC, bool WHOLE, int T>
__device__ __forceinline__ void load_16k(const float* base, int ld, int row0, int rows, int k0, int ke, int g, int r,
                                         float (&x)[T][4]) {
  const int k = k0 + 4 * g;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int row = min(row0 + 16 * t + r, rows - 1);
    const float* src = KC ? base + (long long)row * ld + k : base + (long long)k * ld + row;
    if constexpr (KC && WHOLE) {
      __builtin_memcpy(x[t], src, 16);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) x[t][j] = WHOLE || k + j < ke ? src[KC ? j : (long long)j * ld] : 0.0f;
    }
  }
}

// The largest finite |x| of R rows (or columns) from row0 of an operand over
// [kb, ke), thread tid's share of the block's (256 threads).
template <bool KC, int R>
__device__ __forceinline__ float most_of(const float* base, int ld, int row0, int rows, int kb, int ke, int tid) {
  constexpr int waves = 4;
  const int lane = tid & 63, wave = tid >> 6, n = ke - kb;
  float most = 0.0f;
  auto take = [&](float x) { most = fabsf(x) <= 3.402823466e38f ? fmaxf(most, fabsf(x)) : most; };
  if constexpr (KC) {
    for (int i = wave; i < R; i += waves) {
      const float* src = base + (long long)min(row0 + i, rows - 1) * ld + kb;
#pragma unroll 4
      for (int k = 4 * lane; k + 4 <= n; k += 256) {
        f4 v;
        __builtin_memcpy(&v, src + k, 16);
#pragma unroll
        for (int j = 0; j < 4; ++j) take(v[j]);
      }
      if (lane < n % 4) take(src[n - n % 4 + lane]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; i += 64) {
      const float* src = base + (long long)kb * ld + min(row0 + i + lane % R, rows - 1);
#pragma unroll 8
      for (int k = wave; k < n; k += waves) take(src[(long long)k * ld]);
    }
  }
  return most;
}

// Whether a sum or an operand of the block's tile may have left the range of
// the scaled products.  If not, a result that is not finite comes from an
// operand that is not, and is what f32 arithmetic gives.  All threads take part.
template <int TM, int TN, bool A_KC, bool B_KC>
__device__ __forceinline__ bool F32Split<TM, TN, A_KC, B_KC>::may_overflow(const F32Args& p, int m0, int n0, int kb,
                                                                           int ke, float* smem, int tid) {
  float a = most_of<A_KC, BM>(p.A, p.lda, m0, p.M, kb, ke, tid);
  float b = most_of<B_KC, BN>(p.B, p.ldb, n0, p.N, kb, ke, tid);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a = fmaxf(a, __shfl_xor(a, off, 64));
    b = fmaxf(b, __shfl_xor(b, off, 64));
  }
  smem[tid] = a;
  smem[THREADS + tid] = b;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < THREADS; w += 64) {
    a = fmaxf(a, smem[w]);
    b = fmaxf(b, smem[THREADS + w]);
  }
  constexpr float kMost = 1.7014118e38f * kUnsplit;  // 2^127, of a scaled operand
  return !(a < kMost && b < kMost && (a * kSplitScale) * (b * kSplitScale) * (float)(ke - kb) < 1.7014118e38f);
}

// The wave's tile with v_mfma_f32_16x16x4_f32, operands straight from memory
// into registers: only for tiles whose sums may have left the range of the
// scaled products.  MFMA step j of a chunk takes k = 4g + j in lane group g.
template <int TM, int TN, bool A_KC, bool B_KC>
__device__ __forceinline__ void F32Split<TM, TN, A_KC, B_KC>::plain_f32(const F32Args& p, f4 (&acc)[TM][TN], int row0,
                                                                        int n0, int kb, int ke, int g, int r) {
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < TN; ++u) acc[t][u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  auto chunk = [&](int k0, auto whole) {
    constexpr bool W = decltype(whole)::value;
    float a[TM][4], b[TN][4];
    load_16k<A_KC, W>(p.A, p.lda, row0, p.M, k0, ke, g, r, a);
    load_16k<B_KC, W>(p.B, p.ldb, n0, p.N, k0, ke, g, r, b);
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[u][j], a[t][j], acc[t][u], 0, 0, 0);
  };
  int k0 = kb;
  for (; k0 + 16 <= ke; k0 += 16) chunk(k0, std::integral_constant<bool, true>{});
  if (k0 < ke) chunk(k0, std::integral_constant<bool, false>{});
}

// Stores of a wave tile: lane (g, r) holds rows row0 + 16t + r, columns n0 +
// 16u + 4g .. + 3.  WHOLE: the tile lies inside C, whose rows are 16-byte
// aligned (with the checks in the way the bias loads of a 64x64 tile wait for
// one another: 64x320, K 64 4.27 us, 4.0 without).
template <int EPI, bool WHOLE, int TM, int TN>
__device__ __forceinline__ void store_rows(const F32Args& p, const f4 (&acc)[TM][TN], int row0, int n0, int g, int r,
                                            int split) {
  float* C = p.C + (p.splits > 1 ? (long long)split * p.split_stride : 0);
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int row = row0 + 16 * t + r;
    if (!WHOLE && row >= p.M) continue;
    const long long row_off = (long long)row * p.ldc;
#pragma unroll
    for (int u = 0; u < TN; ++u) {
      const int col = n0 + 16 * u + 4 * g;
      f4 v = acc[t][u];
      if (WHOLE || (p.vec_c && col + 4 <= p.N)) {
        if constexpr (EPI == RT_EPI_BIAS || EPI == RT_EPI_BIAS_RELU) {
          const f4 b = *reinterpret_cast<const f4*>(p.bias + col);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = v[e] + b[e];
            if constexpr (EPI == RT_EPI_BIAS_RELU) v[e] = fmaxf(v[e], 0.0f);
          }
        } else if constexpr (EPI == RT_EPI_RELU_MASK) {
          const f4 mk = *reinterpret_cast<const f4*>(p.mask + row_off + col);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (!(mk[e] > 0.0f)) v[e] = 0.0f;
        }
        *reinterpret_cast<f4*>(C + row_off + col) = v;
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (col + e >= p.N) break;
        float x = v[e];
        if constexpr (EPI == RT_EPI_BIAS || EPI == RT_EPI_BIAS_RELU) {
          x = x + p.bias[col + e];
          if constexpr (EPI == RT_EPI_BIAS_RELU) x = fmaxf(x, 0.0f);
        } else if constexpr (EPI == RT_EPI_RELU_MASK) {
          if (!(p.mask[row_off + col + e] > 0.0f)) x = 0.0f;
        }
        C[row_off + col + e] = x;
      }
    }
  }
}

template <bool WHOLE, int TM, int TN, class Epi>
__device__ __forceinline__ void store_tile(const F32Args& p, const f4 (&acc)[TM][TN], int row0, int n0, int g, int r,
                                           int split, const Epi& e) {
  if constexpr (Epi::kOn) return e.tile(p, acc, row0, n0, g, r);
  if (p.splits > 1) return store_rows<RT_EPI_NONE, WHOLE>(p, acc, row0, n0, g, r, split);
  switch (p.epi) {
    case RT_EPI_BIAS: return store_rows<RT_EPI_BIAS, WHOLE>(p, acc, row0, n0, g, r, split);
    case RT_EPI_BIAS_RELU: return store_rows<RT_EPI_BIAS_RELU, WHOLE>(p, acc, row0, n0, g, r, split);
    case RT_EPI_RELU_MASK: return store_rows<RT_EPI_RELU_MASK, WHOLE>(p, acc, row0, n0, g, r, split);
    default: return store_rows<RT_EPI_NONE, WHOLE>(p, acc, row0, n0, g, r, split);
  }
}

template <int TM, int TN, bool A_KC, bool B_KC>
template <class Epi>
__device__ void F32Split<TM, TN, A_KC, B_KC>::run(const F32Args& p, int bid, int split, float* smem, const Epi& e) {
  unsigned short* const lds = reinterpret_cast<unsigned short*>(smem);
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15;

  constexpr int GROUP = 8;
  const int per_group = GROUP * p.tiles_n;
  const int grp = bid / per_group;
  const int first_m = grp * GROUP;
  const int gsize = min(p.tiles_m - first_m, GROUP);
  const int in_grp = bid - grp * per_group;
  const int tile_m = first_m + in_grp % gsize;
  const int tile_n = in_grp / gsize;
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  const int row0 = m0 + 16 * TM * wave;

  const int kb = split * p.k_per_split;
  const int ke = min(p.K, kb + p.k_per_split);
  const int nk = ke > kb ? (ke - kb + BK - 1) / BK : 0;

  // Byte offsets of this lane's loads from the stage's origin (below 2^31,
  // checked by the host).  Rows and columns past the edge read the last one;
  // what they give is not stored.
  int va[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const int m = min(row0 + 16 * t + r, p.M - 1) - m0;
    va[t] = A_KC ? 4 * (m * p.lda + 4 * g) : 4 * (4 * g * p.lda + m);
  }
  const int a_kk = A_KC ? 4 * 32 : 4 * 32 * p.lda;  // bytes between the two 32-k steps
  int vb[UPT], lb[UPT];                             // ... and the unit's place in an LDS plane
#pragma unroll
  for (int i = 0; i < UPT; ++i) {
    const int q = tid + THREADS * i;
    const int col = B_KC ? q / (BK / 8) : q % BN, j = B_KC ? q % (BK / 8) : q / BN;
    const int n = min(n0 + col, p.N - 1) - n0;
    vb[i] = B_KC ? 4 * (n * p.ldb + k_of(j, 0)) : 4 * (k_of(j, 0) * p.ldb + n);
    lb[i] = place(col, j);
  }

  // K runs over the stages 0 .. nk - 1; when K is not a multiple of 64 the
  // remainder is stage 0, so that every load inside the loop is a whole one
  // (a branch there would make the compiler wait for loads still in flight).
  const int rest = (ke - kb) % BK;
  float fa[TM][KK][8], fb[UPT][8];
  auto rsrcs = [&](int k0, __amdgpu_buffer_rsrc_t& ra, __amdgpu_buffer_rsrc_t& rb) {
    ra = rt_dev::raw_rsrc(A_KC ? p.A + (long long)m0 * p.lda + k0 : p.A + (long long)k0 * p.lda + m0);
    rb = rt_dev::raw_rsrc(B_KC ? p.B + (long long)n0 * p.ldb + k0 : p.B + (long long)k0 * p.ldb + n0);
  };
  // The f32 values of whole stage s: B's units and the A rows of its first
  // 32 k (part 0), the A rows of its second 32 k (part 1).
  auto load_op = [&](const __amdgpu_buffer_rsrc_t& rs, int vo, int so, int ld, auto kc, float (&x)[8]) {
    if constexpr (decltype(kc)::value) {
      const u4 lo = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so, 0);
      const u4 hi = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, so + 64, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        x[j] = __uint_as_float(lo[j]);
        x[4 + j] = __uint_as_float(hi[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        x[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, vo, so + 4 * k_of(0, j) * ld, 0));
    }
  };
  auto load = [&](int s, auto part) {
    constexpr int kk = decltype(part)::value;
    __amdgpu_buffer_rsrc_t ra, rb;
    rsrcs(kb + s * BK - (rest ? BK - rest : 0), ra, rb);
    if constexpr (kk == 0) {
#pragma unroll
      for (int i = 0; i < UPT; ++i) load_op(rb, vb[i], 0, p.ldb, std::integral_constant<bool, B_KC>{}, fb[i]);
    }
#pragma unroll
    for (int t = 0; t < TM; ++t)
      load_op(ra, va[t], kk * a_kk, p.lda, std::integral_constant<bool, A_KC>{}, fa[t][kk]);
  };
  // The remainder's first k is kb: granules inside it whole, the one it ends in
  // element by element, zero past it.
  auto load_rest = [&]() {
    __amdgpu_buffer_rsrc_t ra, rb;
    rsrcs(kb, ra, rb);
    auto granule = [&](const __amdgpu_buffer_rsrc_t& rs, int vo, int ld, auto kc, int j, float (&x)[8]) {
      if (k_of(j, 7) < rest) return load_op(rs, vo, 0, ld, kc, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int off = vo + 4 * k_of(0, e) * (decltype(kc)::value ? 1 : ld);
        x[e] = k_of(j, e) < rest ? __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0)) : 0.0f;
      }
    };
#pragma unroll
    for (int i = 0; i < UPT; ++i) {
      const int q = tid + THREADS * i;
      granule(rb, vb[i], p.ldb, std::integral_constant<bool, B_KC>{}, B_KC ? q % (BK / 8) : q / BN, fb[i]);
    }
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int kk = 0; kk < KK; ++kk)
        granule(ra, va[t] + kk * a_kk, p.lda, std::integral_constant<bool, A_KC>{}, 4 * kk + g, fa[t][kk]);
  };

  // Bias gradient (TN with a colsum target, first M tile): a unit's values are
  // 8 k rows of one column; they are added in f32, and the column's units in
  // order at the end.
  const bool do_cs = CS && p.colsum != nullptr && tile_m == 0;  // uniform over the block
  float cs[UPT];
#pragma unroll
  for (int i = 0; i < UPT; ++i) cs[i] = 0.0f;

  const SplitSel sel;
  u4 ap[KK][TM][3], bq[3];
  // Step w of the split of B's units (w / 14), whose planes go to LDS buffer
  // `buf` as they are complete; likewise of the A rows of one 32-k step.
  auto split_b = [&](int buf, auto wc) {
    constexpr int i = decltype(wc)::value / kSplitSteps, q = decltype(wc)::value % kSplitSteps;
    if constexpr (CS && q == 0) {  // every M tile adds (a branch would part the schedule); the first one stores
#pragma unroll
      for (int j = 0; j < 8; ++j) cs[i] += fb[i][j];
    }
    split_step<q>(fb[i], sel, bq);
    constexpr int pl = plane_done(q);
    if constexpr (pl >= 0) {
      *reinterpret_cast<u4*>(&lds[(buf * 3 + pl) * PLANE + lb[i]]) = bq[pl];
    }
  };
  auto split_a = [&](auto kkc, auto wc) {
    constexpr int kk = decltype(kkc)::value, t = decltype(wc)::value / kSplitSteps;
    split_step<decltype(wc)::value % kSplitSteps>(fa[t][kk], sel, ap[kk][t]);
  };

  // The hi·hi products have an accumulator of their own: the small ones, added
  // into it one MFMA after another, would round it six times per 32 k (which
  // measured 15% more error than the f32 MFMA on operands after a ReLU).
  f4 acc[TM][TN], small[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < TN; ++u) acc[t][u] = small[t][u] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  // (B plane, A plane) of the six products, smallest first.
  constexpr int PB[6] = {2, 0, 1, 1, 0, 0}, PA[6] = {0, 2, 1, 0, 1, 0};
  // A stage's MFMAs run over P column pairs (kk, u0); the B fragments of a
  // pair are read while the pair before it computes.
  constexpr int P = KK * TN / 2;
  u4 bp[2][2][3];
  auto read_pair = [&](int buf, auto ic) {
    constexpr int i = decltype(ic)::value, kk = i / (TN / 2), u0 = 2 * (i % (TN / 2));
#pragma unroll
    for (int uu = 0; uu < 2; ++uu)
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        bp[i & 1][uu][pl] = *reinterpret_cast<const u4*>(
            &lds[(buf * 3 + pl) * PLANE + place(16 * (u0 + uu) + r, 4 * kk + g)]);
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  // The MFMAs of one 32-k step (half a stage), one by one: behind each comes
  // its share of the `steps` split steps, step(w), and in the middle of a pair
  // the LDS reads of the next one.  The schedule is fixed here
  // (sched_barrier): left to itself the compiler puts the splits after the
  // MFMAs, and with one wave per SIMD nothing else would fill the matrix
  // unit meanwhile.
  auto half = [&](int buf, auto hc, auto steps_c, auto&& step) {
    constexpr int kk = decltype(hc)::value, PH = TN / 2, MF = 12 * TM, SLOTS = PH * MF;
    constexpr int STEPS = decltype(steps_c)::value;
    rt_dev::static_for<0, SLOTS>([&](auto sc) {
      constexpr int slot = decltype(sc)::value, i = kk * PH + slot / MF, m = slot % MF;
      constexpr int c = m / (2 * TM), uu = m / TM % 2, t = m % TM, u = 2 * (i % PH) + uu;
      if constexpr (m == MF / 2 && i + 1 < P) read_pair(buf, std::integral_constant<int, i + 1>{});
      f4& d = c == 5 ? acc[t][u] : small[t][u];
      d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, bp[i & 1][uu][PB[c]]),
                                                  __builtin_bit_cast(b8, ap[kk][t][PA[c]]), d, 0, 0, 0);
      rt_dev::static_for<slot * STEPS / SLOTS, (slot + 1) * STEPS / SLOTS>([&](auto wc) { step(wc); });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  constexpr int NA = kSplitSteps * TM, NB = kSplitSteps * UPT;

  if (nk > 0) {
    if (rest) {
      load_rest();
    } else {
      load(0, H0{});
      load(0, H1{});
    }
    rt_dev::static_for<0, NB>([&](auto wc) { split_b(0, wc); });
    rt_dev::static_for<0, NA>([&](auto wc) { split_a(H0{}, wc); });
    rt_dev::barrier_lds();
    // Stage s: its B planes are in LDS buffer s % 2, the A planes of its
    // first 32 k in ap[0], the f32 values of its second in fa.  Under the
    // first half's MFMAs those are split, under the second half's the first
    // 32 k and B of stage s + 1, fetched at the start of stage s.
    for (int s = 0; s + 1 < nk; ++s) {
      const int buf = s & 1;
      load(s + 1, H0{});
      read_pair(buf, H0{});
      __builtin_amdgcn_sched_barrier(0);
      half(buf, H0{}, std::integral_constant<int, NA>{}, [&](auto wc) { split_a(H1{}, wc); });
      load(s + 1, H1{});
      __builtin_amdgcn_sched_barrier(0);
      half(buf, H1{}, std::integral_constant<int, NA + NB>{}, [&](auto wc) {
        constexpr int w = decltype(wc)::value;
        if constexpr (w < NB) split_b(buf ^ 1, wc);
        else split_a(H0{}, std::integral_constant<int, w - NB>{});
      });
      rt_dev::barrier_lds();
    }
    const int buf = (nk - 1) & 1;
    read_pair(buf, H0{});
    half(buf, H0{}, std::integral_constant<int, NA>{}, [&](auto wc) { split_a(H1{}, wc); });
    half(buf, H1{}, std::integral_constant<int, 0>{}, [&](auto) {});
  }

  if (do_cs) {
    __syncthreads();
    float* red = smem;  // [granule of 8 k][BN]: the same sums whatever the tile
#pragma unroll
    for (int i = 0; i < UPT; ++i) red[tid + THREADS * i] = cs[i];
    __syncthreads();
    if (tid < BN && n0 + tid < p.N) {
      float v = red[tid];
#pragma unroll
      for (int j = 1; j < BK / 8; ++j) v += red[j * BN + tid];
      if constexpr (Epi::kOn)
        e.bias(p, n0 + tid, v);
      else
        p.colsum[(long long)split * p.N + n0 + tid] = v;
    }
  }

  bool fine = true;
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < TN; ++u) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = acc[t][u][e];
        acc[t][u][e] = (fabsf(x) <= 3.402823466e38f ? x + small[t][u][e] : x) * (kUnsplit * kUnsplit);
      }
      fine = fine && finite4(acc[t][u]);
    }
  // The block's waves look for the cause together: all of them read B.  (The
  // thread's index from what the epilogue holds anyway: threadIdx.x, kept for
  // this alone, cost a spill and the 64x64 TN tile its third wave per SIMD.)
  __shared__ int bad[THREADS / 64];
  const int mine = __any(!fine);
  if (lane == 0) bad[wave] = mine;
  __syncthreads();
  if (__builtin_expect(bad[0] | bad[1] | bad[2] | bad[3], 0)) {
    if (may_overflow(p, m0, n0, kb, ke, smem, 64 * wave + 16 * g + r) && mine) plain_f32(p, acc, row0, n0, kb, ke, g, r);
  }

  store_tile<false>(p, acc, row0, n0, g, r, split, e);
}

// ---------------------------------------------------------------- f32 MFMA tile fed by DMA
// For whole 64x64 tiles over a short K (dma_better) with 16-byte aligned
// operands the tiles go from
// global memory straight into LDS (buffer_load ... lds: lane l's 16 bytes
// land at the instruction's LDS base + 16 l), two stages of BK = 32 k.
// Within a stage the two 16-k halves are pipelined around one barrier:
//   A: read (k, half 1) fragments     | MFMAs of (k, half 0)
//   B: wait for stage k+1, barrier, DMA stage k+2 into stage k's buffer,
//      read (k+1, half 0) fragments   | MFMAs of (k, half 1)
// MFMAs take the operands swapped (D = op(B)·op(A)), so lane (g, r) ends with
// C(m0+wm+16t+r, n0+wn+16u+4g+q), q = 0..3: one float4 store per 16x16 tile.
//
// LDS layouts (unpadded, bank-conflict-free for the fragment reads):
//   K-contiguous [row][32]: 16-byte granule j of row r at j ^ ((r >> 1) & 7);
//     a fragment is one b128 read of row 16t + r at granule 4 half + g (the
//     four k of the lane's four MFMA steps);
//   M/N-contiguous [k][64]: 64-byte chunk c of row k at c ^ ((k >> 2) & 3); a
//     fragment is four b32 reads (k = 16 half + 4g + s, column 16u + r).
struct F32Dma {
  static constexpr int BM = 64, BN = 64, BK = 32, THREADS = 256, WAVES = 4;
  static constexpr int TM = 2, TN = 2;                 // 16x16 MFMA tiles per wave (32x32 wave tile)
  static constexpr int ELEMS = 64 * BK;                // floats per operand per stage
  static constexpr int PER_WAVE = ELEMS / 256 / WAVES; // 1 KB DMA instructions per operand per wave
  static constexpr int STAGE = 2 * ELEMS;
  static constexpr int SMEM = 2 * STAGE;               // floats: two stages of both operands
  static constexpr int PER_STAGE = 2 * PER_WAVE;

  template <bool KC>
  struct Op {
    __amdgpu_buffer_rsrc_t rsrc;
    int voff;       // this lane's byte offset from the tile origin (first instruction)
    int istep;      // bytes between a lane's consecutive instructions (uniform)
    // Wave w's i-th instruction fills LDS floats [256 (4 i + w), +256); with
    // that spacing the lane's swizzle term is the same for every instruction.
    __device__ inline void init(const float* tile, int ld, int wave, int lane) {
      rsrc = rt_dev::raw_rsrc(tile);
      if constexpr (KC) {
        const int row = 8 * wave + (lane >> 3), slot = lane & 7;  // 8 rows of 128 B per instruction
        voff = 4 * (row * ld + 4 * (slot ^ ((row >> 1) & 7)));
        istep = 4 * 32 * ld;                                        // 32 rows
      } else {
        const int k = 4 * wave + (lane >> 4), s = lane & 15;        // 4 rows of 256 B per instruction
        voff = 4 * (k * ld + 16 * ((s >> 2) ^ ((k >> 2) & 3)) + 4 * (s & 3));
        istep = 4 * 16 * ld;                                        // 16 rows
      }
    }
    __device__ inline void issue(int stage_bytes, float* lds, int wave) const {
#pragma unroll
      for (int i = 0; i < PER_WAVE; ++i) rt_dev::dma16(rsrc, lds + 256 * (4 * i + wave), voff, stage_bytes + i * istep);
    }
    // Fragment of MFMA tile `base` (16 rows / columns) for k-half h: the
    // lane's four k values 16 h + 4 g + s, s = 0..3.
    __device__ static inline f4 frag(const float* lds, int h, int base, int g, int r) {
      if constexpr (KC) {
        const int row = base + r;
        return *reinterpret_cast<const f4*>(&lds[row * BK + 4 * ((4 * h + g) ^ ((row >> 1) & 7))]);
      } else {
        const int col = base + r;
        f4 v;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int k = 16 * h + 4 * g + s;  // (k >> 2) & 3 == g
          v[s] = lds[k * BM + 16 * ((col >> 4) ^ g) + (col & 15)];
        }
        return v;
      }
    }
    // Element (k, col) of an M/N-contiguous stage.
    __device__ static inline float at(const float* lds, int k, int col) {
      return lds[k * BM + 16 * ((col >> 4) ^ ((k >> 2) & 3)) + (col & 15)];
    }
  };

  template <bool A_KC, bool B_KC, class Epi = NoEpi>
  __device__ static void run(const F32Args& p, int bid, int split, float* smem, const Epi& e = Epi{});
};

template <bool A_KC, bool B_KC, class Epi>
__device__ void F32Dma::run(const F32Args& p, int bid, int split, float* smem, const Epi& e) {
  using OpA = Op<A_KC>;
  using OpB = Op<B_KC>;
  auto sA = [&](int buf) { return smem + buf * STAGE; };
  auto sB = [&](int buf) { return smem + buf * STAGE + ELEMS; };

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;

  constexpr int GROUP = 8;
  const int per_group = GROUP * p.tiles_n;
  const int grp = bid / per_group;
  const int first_m = grp * GROUP;
  const int gsize = min(p.tiles_m - first_m, GROUP);
  const int in_grp = bid - grp * per_group;
  const int tile_m = first_m + in_grp % gsize;
  const int tile_n = in_grp / gsize;
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int kb = split * p.k_per_split;
  const int nk = (min(p.K, kb + p.k_per_split) - kb) / BK;  // whole stages (checked by the host)

  OpA oa;
  OpB ob;
  oa.init(A_KC ? p.A + (long long)m0 * p.lda + kb : p.A + (long long)kb * p.lda + m0, p.lda, wave, lane);
  ob.init(B_KC ? p.B + (long long)n0 * p.ldb + kb : p.B + (long long)kb * p.ldb + n0, p.ldb, wave, lane);
  const int a_step = 4 * (A_KC ? BK : BK * p.lda);  // bytes per stage
  const int b_step = 4 * (B_KC ? BK : BK * p.ldb);
  auto issue = [&](int stage, int buf) {
    oa.issue(stage * a_step, sA(buf), wave);
    ob.issue(stage * b_step, sB(buf), wave);
  };

  f4 acc[TM][TN];
#pragma unroll
  for (int t = 0; t < TM; ++t)
#pragma unroll
    for (int u = 0; u < TN; ++u) acc[t][u] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  auto read_frags = [&](int buf, int h, f4 (&fa)[TM], f4 (&fb)[TN]) {
#pragma unroll
    for (int u = 0; u < TN; ++u) fb[u] = OpB::frag(sB(buf), h, wn + 16 * u, g, r);
#pragma unroll
    for (int t = 0; t < TM; ++t) fa[t] = OpA::frag(sA(buf), h, wm + 16 * t, g, r);
  };
  auto mfmas = [&](const f4 (&fa)[TM], const f4 (&fb)[TN]) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[u][s], fa[t][s], acc[t][u], 0, 0, 0);
  };

  // Bias gradient (TN with a colsum target, first M tile): thread t sums
  // column t % 64 over the k rows 8 (t / 64) .. +7 of every stage; the four
  // partial rows are added in order at the end.
  const bool do_cs = !B_KC && p.colsum != nullptr && tile_m == 0;  // uniform over the block
  float cs = 0.0f;
  auto colsum = [&](int buf) {
    if constexpr (!B_KC) {
      if (do_cs) {
        const int col = tid & 63, k0 = 8 * (tid >> 6);
#pragma unroll
        for (int k = 0; k < 8; ++k) cs += OpB::at(sB(buf), k0 + k, col);
      }
    }
  };

  if (nk > 0) {
    f4 fa0[TM], fb0[TN], fa1[TM], fb1[TN];
    // Every B step waits for everything and issues one stage (past the last
    // stage it re-fetches stage nk-1 into a buffer nothing reads), so the
    // bookkeeping is the same in every stage.
    issue(0, 0);
    issue(min(1, nk - 1), 1);
    rt_dev::wait_vm<PER_STAGE>();
    rt_dev::barrier_lds();
    read_frags(0, 0, fa0, fb0);
    auto stage = [&](int k, auto bc) {
      constexpr int BUF = decltype(bc)::value;  // k % 2
      read_frags(BUF, 1, fa1, fb1);
      mfmas(fa0, fb0);
      colsum(BUF);
      rt_dev::wait_vm<0>();
      rt_dev::barrier_lds();  // stage k+1 everywhere; stage k no longer read
      issue(min(k + 2, nk - 1), BUF);
      read_frags(BUF ^ 1, 0, fa0, fb0);  // (k+1, half 0); discarded after the last stage
      mfmas(fa1, fb1);
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    for (int k = 0; k < nk; k += 2) {
      stage(k, B0{});
      if (k + 1 < nk) stage(k + 1, B1{});
    }
  }

  if (do_cs) {
    __syncthreads();  // main-loop LDS reads are finished
    float* red = smem;  // [4][64]
    red[tid] = cs;
    __syncthreads();
    if (tid < 64) {
      const float v = ((red[tid] + red[64 + tid]) + red[128 + tid]) + red[192 + tid];
      if constexpr (Epi::kOn)
        e.bias(p, n0 + tid, v);
      else
        p.colsum[(long long)split * p.N + n0 + tid] = v;
    }
  }

  store_tile<true>(p, acc, m0 + wm, n0 + wn, g, r, split, e);
}

// Adapter so the single and pair kernels can run an F32Dma layout like an
// F32Tile.
template <bool A_KC, bool B_KC>
struct F32DmaTile {
  static constexpr int THREADS = F32Dma::THREADS, SMEM = F32Dma::SMEM, BM = F32Dma::BM, BN = F32Dma::BN;
  template <class Epi = NoEpi>
  __device__ static void run(const F32Args& p, int bid, int split, float* smem, const Epi& e = Epi{}) {
    F32Dma::run<A_KC, B_KC>(p, bid, split, smem, e);
  }
};

// Two waves per SIMD: the compiler would otherwise spread a 128x64 tile over
// more than half of the registers (4096^3 NN 724 -> 917 us).
template <class T>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_f32_kernel(F32Args p) {
  __shared__ __attribute__((aligned(16))) float smem[T::SMEM];
  T::run(p, xcd_local(blockIdx.x, gridDim.x), blockIdx.z, smem);
}

// C = A·Bᵀ (NT) for K <= 16, one 64x64 block of C per workgroup: the
// block's 64 rows of A and 64 rows of B go to LDS, and thread t computes
// rows 4(t/16) .. +3, columns 4(t%16) .. +3 with K multiply-adds each, in k
// order, then applies the epilogue.  A rank-K update is a stream of C (and
// of the mask): the MFMA tile's K pipeline padded to 32 only adds latency.
struct F32RankK {
  static constexpr int THREADS = 256, BM = 64, BN = 64;
  static constexpr int KMAX = 16;
  static constexpr int LD = KMAX + 1;  // LDS row stride (floats)
  static constexpr int SMEM = 2 * 64 * LD;
  __device__ static void run(const F32Args& p, int bid, int, float* smem) {
    float* sa = smem;
    float* sb = smem + 64 * LD;
    const int tile_m = bid / p.tiles_n, tile_n = bid - tile_m * p.tiles_n;
    const int m0 = 64 * tile_m, n0 = 64 * tile_n, K = p.K, tid = threadIdx.x;
    const int r0 = 4 * (tid / 16), c0 = 4 * (tid % 16);
    const int col = n0 + c0;
    // The ReLU mask of this thread's outputs, loaded first so that its
    // latency runs under the operand staging and the multiply-adds.
    const bool vec_mask = p.epi == RT_EPI_RELU_MASK && p.vec_c && col + 4 <= p.N;
    f4 mkv[4];
    if (vec_mask) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mkv[i] = m0 + r0 + i < p.M ? *reinterpret_cast<const f4*>(p.mask + (long long)(m0 + r0 + i) * p.ldc + col)
                                   : f4{0, 0, 0, 0};
    }
    for (int i = tid; i < 64 * K; i += THREADS) {
      const int r = i / K, k = i - r * K;
      sa[r * LD + k] = m0 + r < p.M ? p.A[(long long)(m0 + r) * p.lda + k] : 0.0f;
      sb[r * LD + k] = n0 + r < p.N ? p.B[(long long)(n0 + r) * p.ldb + k] : 0.0f;
    }
    __syncthreads();
    f4 acc[4] = {f4{0, 0, 0, 0}, f4{0, 0, 0, 0}, f4{0, 0, 0, 0}, f4{0, 0, 0, 0}};
    for (int k = 0; k < K; ++k) {
      const f4 b = f4{sb[c0 * LD + k], sb[(c0 + 1) * LD + k], sb[(c0 + 2) * LD + k], sb[(c0 + 3) * LD + k]};
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += sa[(r0 + i) * LD + k] * b;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = m0 + r0 + i;
      if (row >= p.M) break;
      f4 v = acc[i];
      float* c = p.C + (long long)row * p.ldc + col;
      const float* mk = p.mask + (long long)row * p.ldc + col;
      if (p.vec_c && col + 4 <= p.N) {
        if (p.epi == RT_EPI_BIAS || p.epi == RT_EPI_BIAS_RELU) {
          v += *reinterpret_cast<const f4*>(p.bias + col);
          if (p.epi == RT_EPI_BIAS_RELU)
            for (int q = 0; q < 4; ++q) v[q] = fmaxf(v[q], 0.0f);
        } else if (vec_mask) {
          for (int q = 0; q < 4; ++q)
            if (!(mkv[i][q] > 0.0f)) v[q] = 0.0f;
        }
        *reinterpret_cast<f4*>(c) = v;
      } else {
        for (int q = 0; q < 4 && col + q < p.N; ++q) {
          float x = v[q];
          if (p.epi == RT_EPI_BIAS || p.epi == RT_EPI_BIAS_RELU) {
            x = x + p.bias[col + q];
            if (p.epi == RT_EPI_BIAS_RELU) x = fmaxf(x, 0.0f);
          } else if (p.epi == RT_EPI_RELU_MASK && !(mk[q] > 0.0f)) {
            x = 0.0f;
          }
          c[q] = x;
        }
      }
    }
  }
};

// Two independent GEMMs in one launch (horizontal fusion): blocks
// [0, n0) run problem 0, the rest problem 1, each problem's split index
// folded into its block range.  n0 is a multiple of 8 so both problems are
// spread evenly over the XCDs; problem 0 is dispatched first.
template <class T0, class T1>
__global__ __launch_bounds__(T0::THREADS, 2) void gemm_f32_pair_kernel(F32Args p0, F32Args p1, int n0) {
  static_assert(T0::THREADS == T1::THREADS, "one block size");
  constexpr int S = T0::SMEM > T1::SMEM ? T0::SMEM : T1::SMEM;
  __shared__ __attribute__((aligned(16))) float smem[S];
  const int b = blockIdx.x;
  if (b < n0) {
    const int tiles = p0.tiles_m * p0.tiles_n;
    const int nb = tiles * p0.splits;
    if (b >= nb) return;  // padding up to a multiple of 8
    const int loc = xcd_local(b, nb);
    T0::run(p0, loc % tiles, loc / tiles, smem);
  } else {
    const int tiles = p1.tiles_m * p1.tiles_n;
    const int nb = tiles * p1.splits;
    const int loc = xcd_local(b - n0, nb);
    T1::run(p1, loc % tiles, loc / tiles, smem);
  }
}

// A GEMM and an optimizer update that does not touch its operands in one
// launch: blocks [0, n_gemm) run the GEMM's (tile, K slice) items, the rest
// the optimizer blocks of b.  The GEMM is dispatched first; the update, which
// is HBM-bound, runs on the CUs next to its MFMA-bound tiles.
template <class T>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_f32_opt_kernel(F32Args p, rt_opt::OptBatch b, int n_gemm) {
  static_assert(T::THREADS == rt_opt::kThreads, "one block size");
  __shared__ __attribute__((aligned(16))) float smem[T::SMEM];
  const int blk = blockIdx.x;
  if (blk < n_gemm) {
    const int tiles = p.tiles_m * p.tiles_n;
    const int loc = xcd_local(blk, n_gemm);
    T::run(p, loc % tiles, loc / tiles, smem);
  } else {
    rt_opt::optimizer_block<false>(b, blk - n_gemm);
  }
}

// The update of the layer whose dW this unsplit TN launch computes, done by
// the tiles themselves: an element's gradient is final in the tile that
// computed it, so the tile stores it and updates the parameter and its
// optimizer state there, with the optimizer's per-element arithmetic (same
// bits as the separate update); the first row of tiles does the same for the
// bias from its column sums.  w / b index like dW / db (w.n = M·N, ldc = N).
struct UpdEpi {
  static constexpr bool kOn = true;
  rt::OptTensor w, b;
  rt::OptParams P;
  template <int TM, int TN>
  __device__ void tile(const F32Args& p, const f4 (&acc)[TM][TN], int row0, int n0, int g, int r) const {
    const bool skip = rt_opt::skipped(P);
    const rt_opt::Coef c = rt_opt::coef(P);
    const bool adam = P.kind == 0, has_m = w.m != nullptr;
    // Whole tiles only (gemm_opt_update_ok).
    const long long i0 = (long long)(row0 + r) * p.ldc + n0 + 4 * g;
    // Every load of θ and the state first, so that they go out together
    // (the stores below could alias them as far as the compiler knows).
    f4 th[TM][TN], m[TM][TN], v[TM][TN];
    if (!skip) {
#pragma unroll
      for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u) {
          const long long i = i0 + (long long)16 * t * p.ldc + 16 * u;
          th[t][u] = *reinterpret_cast<const f4*>(w.theta + i);
          m[t][u] = has_m ? *reinterpret_cast<const f4*>(w.m + i) : f4{0, 0, 0, 0};
          v[t][u] = adam ? *reinterpret_cast<const f4*>(w.v + i) : f4{0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
      for (int u = 0; u < TN; ++u) {
        const long long i = i0 + (long long)16 * t * p.ldc + 16 * u;
        const f4 gv = acc[t][u];
        *reinterpret_cast<f4*>(p.C + i) = gv;
        if (skip) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float te = th[t][u][q], me = m[t][u][q], ve = v[t][u][q];
          rt_opt::update(P, c, gv[q], te, &me, &ve);
          th[t][u][q] = te;
          m[t][u][q] = me;
          v[t][u][q] = ve;
        }
        *reinterpret_cast<f4*>(w.theta + i) = th[t][u];
        if (has_m) *reinterpret_cast<f4*>(w.m + i) = m[t][u];
        if (adam) *reinterpret_cast<f4*>(w.v + i) = v[t][u];
      }
  }
  __device__ void bias(const F32Args& p, int col, float gv) const {
    p.colsum[col] = gv;
    if (rt_opt::skipped(P)) return;
    const bool adam = P.kind == 0, has_m = b.m != nullptr;
    float th = b.theta[col], m = has_m ? b.m[col] : 0.0f, v = adam ? b.v[col] : 0.0f;
    rt_opt::update(P, rt_opt::coef(P), gv, th, &m, &v);
    b.theta[col] = th;
    if (has_m) b.m[col] = m;
    if (adam) b.v[col] = v;
  }
};

// gemm_f32_opt_kernel on whole 64x64 tiles of an unsplit TN product whose
// tiles also update their own layer (UpdEpi).
template <class T>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_f32_opt_upd_kernel(F32Args p, rt_opt::OptBatch b, int n_gemm,
                                                                        UpdEpi u) {
  static_assert(T::THREADS == rt_opt::kThreads && T::BM == 64 && T::BN == 64, "one block size, 64x64 tiles");
  __shared__ __attribute__((aligned(16))) float smem[T::SMEM];
  const int blk = blockIdx.x;
  if (blk < n_gemm) {
    T::run(p, xcd_local(blk, n_gemm), 0, smem, u);
  } else {
    rt_opt::optimizer_block<false>(b, blk - n_gemm);
  }
}

// Two such products (two layers' dW, each updating its own layer) and the
// optimizer blocks of b in one launch: blocks [0, n0) problem 0 (n0 a
// multiple of 8, the padding idle), [n0, n1) problem 1, the rest the update.
template <class T>
__global__ __launch_bounds__(T::THREADS, 2) void gemm_f32_opt_upd2_kernel(F32Args p0, F32Args p1, rt_opt::OptBatch b,
                                                                         int n0, int n1, UpdEpi u0, UpdEpi u1) {
  static_assert(T::THREADS == rt_opt::kThreads && T::BM == 64 && T::BN == 64, "one block size, 64x64 tiles");
  __shared__ __attribute__((aligned(16))) float smem[T::SMEM];
  const int blk = blockIdx.x;
  if (blk < n0) {
    const int nb = p0.tiles_m * p0.tiles_n;
    if (blk >= nb) return;  // padding up to a multiple of 8
    T::run(p0, xcd_local(blk, nb), 0, smem, u0);
  } else if (blk < n1) {
    T::run(p1, xcd_local(blk - n0, n1 - n0), 0, smem, u1);
  } else {
    rt_opt::optimizer_block<false>(b, blk - n1);
  }
}

// The first cs_blocks blocks each take 256 columns of the column sums: they
// start first, so their chains of loads run under the plane sums; the rest
// sum the planes (grid-stride over M*N).  A result that is not finite sets
// *nf_flag, where one is given: the bf16 plan's overflow check without a pass
// of its own over the gradients.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S, long long stride,
                                                             int M, int N, float* C, int ldc, int epi,
                                                             const float* bias, const float* mask,
                                                             const float* __restrict__ cs_part, int cs_rows,
                                                             float* cs, int cs_blocks, int vec4, int* nf_flag) {
  if ((int)blockIdx.x < cs_blocks) {
    const long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= N) return;
    // Slice s's column sum: cs_part[s, j], or with shares the cs_rows rows
    // cs_part[s, t, j] added in order from zero; then the slices in order.
    // Element e = s * rows + t of that sequence is at cs_part[e * N + j]; the
    // loads go out 16 at a time and the adds follow in sequence order.
    const int rows = cs_rows > 0 ? cs_rows : 1;
    const long long n = (long long)S * rows;
    float v = 0.0f, w = 0.0f;
    int t = 0;          // row of element e within its slice
    bool first = true;  // e lies in slice 0
    for (long long e0 = 0; e0 < n; e0 += 16) {
      float x[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) x[u] = e0 + u < n ? cs_part[(e0 + u) * N + j] : 0.0f;
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        if (e0 + u >= n) break;
        w = cs_rows > 0 ? (t == 0 ? 0.0f : w) + x[u] : x[u];
        if (++t == rows) {
          v = first ? w : v + w;
          first = false;
          t = 0;
        }
      }
    }
    cs[j] = v;
    if (nf_flag != nullptr && !(fabsf(v) <= 3.402823466e38f)) *nf_flag = 1;
    return;
  }
  const int plane_blocks = (int)gridDim.x - cs_blocks;
  const long long total = (long long)M * N;
  const long long first = (blockIdx.x - cs_blocks) * (long long)blockDim.x + threadIdx.x;
  const long long step = (long long)plane_blocks * blockDim.x;
  if (vec4) {
    // Four consecutive elements of one row per thread (N, ldc, stride and
    // every pointer 16-byte aligned); each element's sum is the scalar one.
    const f4* P = reinterpret_cast<const f4*>(part);
    const long long s4 = stride / 4, total4 = total / 4;
    for (long long i = first; i < total4; i += step) {
      f4 v = P[i];
      int s = 1;
      for (; s + 8 <= S; s += 8) {
        f4 t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) t[j] = P[(long long)(s + j) * s4 + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) v += t[j];
      }
      f4 t[7];
#pragma unroll
      for (int j = 0; j < 7; ++j) t[j] = s + j < S ? P[(long long)(s + j) * s4 + i] : f4{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 7; ++j)
        if (s + j < S) v += t[j];
      const long long e = 4 * i, row = e / N;
      const int col = (int)(e - row * N);
      if (epi == RT_EPI_BIAS || epi == RT_EPI_BIAS_RELU) {
        const f4 b = *reinterpret_cast<const f4*>(bias + col);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[q] = v[q] + b[q];
          if (epi == RT_EPI_BIAS_RELU) v[q] = fmaxf(v[q], 0.0f);
        }
      } else if (epi == RT_EPI_RELU_MASK) {
        const f4 mk = *reinterpret_cast<const f4*>(mask + row * ldc + col);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (!(mk[q] > 0.0f)) v[q] = 0.0f;
      }
      *reinterpret_cast<f4*>(C + row * ldc + col) = v;
      if (nf_flag != nullptr && !finite4(v)) *nf_flag = 1;
    }
    return;
  }
  for (long long i = first; i < total; i += step) {
    // v = plane 0 + plane 1 + ... in slice order; the loads go out 8 at a
    // time (the last S - 1 mod 8 together) so the chain of adds does not
    // wait on one load after another.
    float v = part[i];
    int s = 1;
    for (; s + 8 <= S; s += 8) {
      float t[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] = part[(long long)(s + j) * stride + i];
#pragma unroll
      for (int j = 0; j < 8; ++j) v += t[j];
    }
    float t[7];
#pragma unroll
    for (int j = 0; j < 7; ++j) t[j] = s + j < S ? part[(long long)(s + j) * stride + i] : 0.0f;
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (s + j < S) v += t[j];
    long long o = i;  // offset in C
    if (epi != RT_EPI_NONE || ldc != N) {
      const long long row = i / N;
      const int col = (int)(i - row * N);
      o = row * ldc + col;
      if (epi == RT_EPI_BIAS || epi == RT_EPI_BIAS_RELU) {
        v = v + bias[col];
        if (epi == RT_EPI_BIAS_RELU) v = fmaxf(v, 0.0f);
      } else if (epi == RT_EPI_RELU_MASK) {
        if (!(mask[o] > 0.0f)) v = 0.0f;
      }
    }
    C[o] = v;
    if (nf_flag != nullptr && !(fabsf(v) <= 3.402823466e38f)) *nf_flag = 1;
  }
}

// Tile of a product: the largest of 128x64, 64x64 and 64x32 that still gives
// every CU a block (a smaller one splits and reads its operands more often:
// 4096^3 NN 724 / 821 / 1069 us; too few blocks leave CUs idle: 512x1024, K
// 2048 in two slices 35.1 / 25.3 / 24.5 us, 300x200, K 500 18.4 / 12.4 / 8.7).
enum TileCfg { kT128x64, kT64x64, kT64x32 };
TileCfg pick_tile(const F32Args& a) {
  const long long n64 = (a.N + 63) / 64, t128 = (long long)((a.M + 127) / 128) * n64 * a.splits;
  if (a.N <= 32) return kT64x32;
  if (t128 >= 256) return kT128x64;
  return (long long)((a.M + 63) / 64) * n64 * a.splits >= 256 ? kT64x64 : kT64x32;
}

// The split tiles address a stage by 32-bit byte offsets: at most 128 rows or
// 64 k of either operand.  Longer rows go to the f32 MFMA tile.
bool split_ok(const F32Args& a) { return a.lda <= (1 << 21) && a.ldb <= (1 << 21); }

// Products that stay on the f32 MFMA tile: whole 64x64 tiles, every K slice
// (the last included) a multiple of 32 and at most 512 long, too few tiles for
// larger ones, 16-byte aligned rows and pointers, and operands addressable
// with 32-bit byte offsets.  Over so short a K the split tile's longer
// prologue costs what its matrix rate gains: 2048x1024, K 512 takes 20.6 us
// here and 20.3 split (K 1024: 36.4 and 32.5), the batch-32 step's update
// launch (K 32) 11.6 and 12.4.
template <bool A_KC, bool B_KC>
bool dma_better(const F32Args& a) {
  const int last = a.K - (a.splits - 1) * a.k_per_split;
  const long long lim = 1LL << 31, t128 = (long long)((a.M + 127) / 128) * ((a.N + 127) / 128) * a.splits;
  return a.M % 64 == 0 && a.N % 64 == 0 && a.k_per_split <= 512 && a.k_per_split % 32 == 0 && last > 0 &&
         last % 32 == 0 && t128 < 512 && a.vec_a && a.vec_b && a.vec_c &&
         (long long)(A_KC ? a.M : a.K) * a.lda * 4 < lim && (long long)(B_KC ? a.N : a.K) * a.ldb * 4 < lim;
}

// TN products (weight gradients) over at most 128 rows, or 256 where N is at
// most 32 columns, that dma_better leaves out stay on the plain f32 tile, whose
// column sums are added row by row: the bias gradient of a small batch then has
// the bits of the reference's left-to-right sum, as it had before the split
// tile.  That is what the limits are for; it costs the narrow layer's launch
// some time near them (512x10: K 128 6.2 us, K 256 9.8, K 257 6.5 on the split
// tile, 11.5 on this one).
bool row_order_tn(const F32Args& a) {
  return a.splits <= 1 && a.K <= (a.N <= 32 ? 256 : 128) && !dma_better<false, false>(a);
}

// Products with so short a K that the split tile's prologue (operands split
// before the first MFMA) costs more than its matrix rate gains, on grids that
// give every CU a 64x64 block: 640x2033 NN, K 64 7.4 us on the plain f32 tile,
// 8.6 split, K 96 8.9 and 9.8, K 128 10.4 and 9.8; with twice the blocks up to
// K 128 (1856x2450 NN 22.8 and 24.1, K 192 30.5 and 28.5), K 192 where both
// operands lie along K (25.7 and 27.8); K slices of 32 (500x500 in slices of 64
// 27.4 and 25.3).  Smaller grids take less split at any K (300x200, K 20 4.1
// and 3.7).  And K of 1 and 2, where the terms the split leaves out are not
// small against the rounding of the sum: 1.5 and 2.6 units of 2^-24 |A||B| at
// most, 1.0 and 1.9 here.
template <bool A_KC, bool B_KC>
bool short_k(const F32Args& a) {
  const long long n64 = (a.N + 63) / 64, t64 = (a.M + 63) / 64 * n64 * a.splits;
  const long long t128 = (a.M + 127) / 128 * n64 * a.splits;
  const int k = std::min(a.k_per_split, a.K);
  if (k <= 2) return true;
  if (t64 < 256 || a.N <= 32) return false;
  if (a.splits > 1) return k <= 32;
  return k <= (t128 < 256 ? 96 : A_KC && B_KC ? 192 : 128);
}

// Products on the plain f32 tile.
template <bool A_KC, bool B_KC>
bool plain_tile(const F32Args& a) {
  return !split_ok(a) || (!A_KC && row_order_tn(a)) || short_k<A_KC, B_KC>(a);
}

template <class T>
hipError_t launch_tile(hipStream_t s, F32Args a) {
  a.tiles_m = (a.M + T::BM - 1) / T::BM;
  a.tiles_n = (a.N + T::BN - 1) / T::BN;
  dim3 grid(a.tiles_m * a.tiles_n, 1, a.splits);
  rt::launch((gemm_f32_kernel<T>), grid, dim3(T::THREADS), 0, s, a);
  return hipGetLastError();
}

// Skinny products: at most 64 rows of output, A K-contiguous (the NN
// forward and the NT dX of a small batch).  A block owns 16 output columns
// over the whole K; its 8 waves take consecutive runs of 16-k sub-blocks and
// issue the loads of up to 8 sub-blocks together ahead of their MFMAs, so
// the K loop is a few memory round trips instead of one per step.  The
// waves' partial tiles are added in LDS in wave order, then the epilogue.
// One launch and no partial planes, where split-K needs a reduction launch.
//
// Within a sub-block at k0, lane (g, r) feeds MFMA step q the element
// k0 + 4g + q of its A row and B column (one float4 of A per sub-block); the
// accumulator of row block rb holds C[16 rb + 4g + q][n0 + r].
constexpr int kSkinnyWaves = 8, kSkinnyChunk = 8;

template <int RB, bool B_KC>
__global__ __launch_bounds__(64 * kSkinnyWaves) void gemm_f32_skinny_kernel(F32Args p) {
  __shared__ float red[kSkinnyWaves * RB * 16 * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, r = lane & 15;
  const int n0 = blockIdx.x * 16;
  const int nsub = p.K / 16;  // K % 16 == 0 (checked by the host)
  const int per = (nsub + kSkinnyWaves - 1) / kSkinnyWaves;
  const int s_end = min(nsub, (wave + 1) * per);

  f4 acc[RB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int sb = wave * per; sb < s_end; sb += kSkinnyChunk) {
    f4 a[kSkinnyChunk][RB], b[kSkinnyChunk];
#pragma unroll
    for (int c = 0; c < kSkinnyChunk; ++c) {
      const int k = 16 * (sb + c) + 4 * g;
      const bool in = sb + c < s_end;
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int row = 16 * rb + r;
        a[c][rb] = (in && row < p.M) ? *reinterpret_cast<const f4*>(p.A + (long long)row * p.lda + k)
                                     : f4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      if (!in) {
        b[c] = f4{0.0f, 0.0f, 0.0f, 0.0f};
      } else if constexpr (B_KC) {
        b[c] = *reinterpret_cast<const f4*>(p.B + (long long)(n0 + r) * p.ldb + k);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) b[c][q] = p.B[(long long)(k + q) * p.ldb + n0 + r];
      }
    }
#pragma unroll
    for (int c = 0; c < kSkinnyChunk; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) acc[rb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][rb][q], b[c][q], acc[rb], 0, 0, 0);
  }

  // red[w][row][col]: wave w's partial C[row][n0 + col].
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[(wave * RB * 16 + 16 * rb + 4 * g + q) * 16 + r] = acc[rb][q];
  __syncthreads();
  for (int e = tid; e < RB * 16 * 16; e += 64 * kSkinnyWaves) {
    const int row = e >> 4, col = n0 + (e & 15);
    if (row >= p.M) continue;
    float v = red[e];
#pragma unroll
    for (int w = 1; w < kSkinnyWaves; ++w) v += red[w * RB * 16 * 16 + e];
    if (p.epi == RT_EPI_BIAS || p.epi == RT_EPI_BIAS_RELU) {
      v = v + p.bias[col];
      if (p.epi == RT_EPI_BIAS_RELU) v = fmaxf(v, 0.0f);
    } else if (p.epi == RT_EPI_RELU_MASK) {
      if (!(p.mask[(long long)row * p.ldc + col] > 0.0f)) v = 0.0f;
    }
    p.C[(long long)row * p.ldc + col] = v;
  }
}

// The skinny kernel takes a product when it has at most 64 rows, too few
// 64x64 tiles to fill the chip, whole 16-column and 16-k blocks, a
// K-contiguous A (NN or NT) with float4-loadable rows, and no K slices or
// column sums.
template <bool A_KC, bool B_KC>
bool skinny_ok(const F32Args& a) {
  auto al = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  const long long tiles = (long long)((a.M + 63) / 64) * ((a.N + 63) / 64);
  return A_KC && a.splits == 1 && a.colsum == nullptr && rt::gemm_f32_skinny_shape(a.M, a.N, a.K) && tiles < 256 &&
         a.lda % 4 == 0 && al(a.A) && (!B_KC || (a.ldb % 4 == 0 && al(a.B)));
}

template <bool B_KC>
hipError_t launch_skinny(hipStream_t s, const F32Args& a) {
  const dim3 grid(a.N / 16), block(64 * kSkinnyWaves);
  if (a.M <= 32)
    rt::launch((gemm_f32_skinny_kernel<2, B_KC>), grid, block, 0, s, a);
  else
    rt::launch((gemm_f32_skinny_kernel<4, B_KC>), grid, block, 0, s, a);
  return hipGetLastError();
}

// dX of a narrow layer (K = that layer's outputs <= 16): the rank-K block.
bool rank_k_ok(const F32Args& a) {
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool epi_ok = (a.epi != RT_EPI_RELU_MASK || al16(a.mask)) &&
                      ((a.epi != RT_EPI_BIAS && a.epi != RT_EPI_BIAS_RELU) || al16(a.bias));
  return a.K >= 1 && a.K <= F32RankK::KMAX && a.splits <= 1 && epi_ok;
}

hipError_t launch_rank_k(hipStream_t s, F32Args a) {
  a.tiles_m = (a.M + 63) / 64;
  a.tiles_n = (a.N + 63) / 64;
  rt::launch((gemm_f32_kernel<F32RankK>), dim3(a.tiles_m * a.tiles_n), dim3(F32RankK::THREADS), 0, s, a);
  return hipGetLastError();
}

// Rows that one launch of any tile takes: a grid holds fewer than 2^32 threads
// (HIP runs a larger one modulo 2^32), 2^24 blocks of at least 64 rows.
constexpr int kMostRows = 1 << 29;

template <bool A_KC, bool B_KC>
hipError_t dispatch_tile(hipStream_t s, F32Args a) {
  if (a.M > kMostRows) {
    F32Args rest = a;
    a.M = kMostRows;
    if (hipError_t e = dispatch_tile<A_KC, B_KC>(s, a); e != hipSuccess) return e;
    rest.M -= kMostRows;
    rest.A += A_KC ? (long long)kMostRows * a.lda : (long long)kMostRows;
    rest.C += (long long)kMostRows * a.ldc;
    if (rest.mask != nullptr) rest.mask += (long long)kMostRows * a.ldc;
    rest.colsum = nullptr;  // the first part's
    return dispatch_tile<A_KC, B_KC>(s, rest);
  }
  if constexpr (A_KC) {
    if (skinny_ok<A_KC, B_KC>(a)) return launch_skinny<B_KC>(s, a);
  }
  if constexpr (A_KC && B_KC) {
    if (rank_k_ok(a)) return launch_rank_k(s, a);
  }
  if (dma_better<A_KC, B_KC>(a)) return launch_tile<F32DmaTile<A_KC, B_KC>>(s, a);
  if constexpr (!A_KC) {
    if (row_order_tn(a) && a.N <= 32) return launch_tile<F32Tile<A_KC, B_KC, 32>>(s, a);
  }
  if (plain_tile<A_KC, B_KC>(a)) return launch_tile<F32Tile<A_KC, B_KC>>(s, a);
  switch (pick_tile(a)) {
    case kT128x64: return launch_tile<F32Split<2, 4, A_KC, B_KC>>(s, a);
    case kT64x64: return launch_tile<F32Split<1, 4, A_KC, B_KC>>(s, a);
    default: return launch_tile<F32Split<1, 2, A_KC, B_KC>>(s, a);
  }
}

F32Args make_args(const rt::GemmDesc& d) {
  F32Args a{};
  a.A = static_cast<const float*>(d.A);
  a.B = static_cast<const float*>(d.B);
  a.C = static_cast<float*>(d.C);
  a.M = d.M;
  a.N = d.N;
  a.K = d.K;
  a.lda = d.lda;
  a.ldb = d.ldb;
  a.ldc = d.ldc;
  a.epi = d.epi;
  a.bias = d.bias;
  a.mask = static_cast<const float*>(d.mask);
  a.colsum = d.splits > 1 ? d.colsum_partials : d.colsum;
  a.splits = d.splits < 1 ? 1 : d.splits;
  // Slices are whole multiples of the 32-wide K step.
  int kps = (d.K + a.splits - 1) / a.splits;
  kps = ((kps + 31) / 32) * 32;
  a.k_per_split = a.splits > 1 ? kps : (d.K > 0 ? d.K : 1);
  a.split_stride = d.split_stride;
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  a.vec_a = (d.lda % 4 == 0) && al16(d.A);
  a.vec_b = (d.ldb % 4 == 0) && al16(d.B);
  a.vec_c = (d.ldc % 4 == 0) && al16(d.C) && (d.bias == nullptr || al16(d.bias)) &&
            (d.epi != RT_EPI_RELU_MASK || al16(d.mask)) && (d.splits <= 1 || d.split_stride % 4 == 0);
  return a;
}

// The backward pair of a hidden layer: dW = Aᵀ·δ (TN, any number of K
// slices) and dX = (δ·Wᵀ) ⊙ mask (NT, whole K).
template <class T0, class T1>
hipError_t launch_pair_tn_nt(hipStream_t s, F32Args a0, F32Args a1) {
  a0.tiles_m = (a0.M + T0::BM - 1) / T0::BM;
  a0.tiles_n = (a0.N + T0::BN - 1) / T0::BN;
  a1.tiles_m = (a1.M + T1::BM - 1) / T1::BM;
  a1.tiles_n = (a1.N + T1::BN - 1) / T1::BN;
  const long long nb0 = (long long)a0.tiles_m * a0.tiles_n * a0.splits;
  const long long nb1 = (long long)a1.tiles_m * a1.tiles_n * a1.splits;
  const long long n0 = (nb0 + 7) / 8 * 8;
  if (n0 + nb1 > 0x7fffffffLL) return hipErrorInvalidValue;
  rt::launch((gemm_f32_pair_kernel<T0, T1>), dim3((unsigned)(n0 + nb1)), dim3(T0::THREADS), 0, s, a0,
                     a1, (int)n0);
  return hipGetLastError();
}

// f(tile) for the dW of an update launch: the tile of its own launch.
template <class F>
hipError_t by_tn_tile(const F32Args& a, F&& f) {
  if (dma_better<false, false>(a)) return f(F32DmaTile<false, false>{});
  if (row_order_tn(a) && a.N <= 32) return f(F32Tile<false, false, 32>{});
  if (plain_tile<false, false>(a)) return f(F32Tile<false, false>{});
  switch (pick_tile(a)) {
    case kT128x64: return f(F32Split<2, 4, false, false>{});
    case kT64x64: return f(F32Split<1, 4, false, false>{});
    default: return f(F32Split<1, 2, false, false>{});
  }
}

// f(64x64 tile) for a dW whose tiles update their layer.
template <class F>
hipError_t by_update_tile(const F32Args& a, F&& f) {  // whole 64x64 tiles (gemm_opt_update_ok)
  return dma_better<false, false>(a) ? f(F32DmaTile<false, false>{}) : f(F32Split<1, 4, false, false>{});
}

}  // namespace

namespace rt {

bool gemm_f32_skinny_shape(int M, int N, int K) {
  return M >= 1 && M <= 64 && N >= 16 && N % 16 == 0 && K >= 128 && K % 16 == 0;
}

hipError_t gemm_f32_launch(hipStream_t s, const GemmDesc& d) {
  const F32Args a = make_args(d);
  switch (d.layout) {
    case RT_NN: return dispatch_tile<true, false>(s, a);
    case RT_TN: return dispatch_tile<false, false>(s, a);
    case RT_NT: return dispatch_tile<true, true>(s, a);
  }
  return hipErrorInvalidValue;
}

template <class T>
hipError_t launch_gemm_opt(hipStream_t s, F32Args a, const rt_opt::OptBatch& b, long long opt_blocks) {
  a.tiles_m = (a.M + T::BM - 1) / T::BM;
  a.tiles_n = (a.N + T::BN - 1) / T::BN;
  const long long n_gemm = (long long)a.tiles_m * a.tiles_n * a.splits;
  if (n_gemm + opt_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  rt::launch((gemm_f32_opt_kernel<T>), dim3((unsigned)(n_gemm + opt_blocks)), dim3(T::THREADS), 0, s, a, b,
             (int)n_gemm);
  return hipGetLastError();
}

bool gemm_opt_supported(const GemmDesc& d, const OptTensor* ts, int nt, const OptParams& P) {
  if (d.in_dtype != RT_F32 || d.layout != RT_TN || d.M <= 0 || d.N <= 0 || d.K <= 0) return false;
  if (d.M > kMostRows) return false;
  return nt > 0 && (split_ok(make_args(d)) || row_order_tn(make_args(d))) && optimizer_fits_cache(ts, nt, P);
}

bool gemm_opt_update_ok(const GemmDesc& d, const OptTensor* wb, const OptParams& P) {
  if (d.in_dtype != RT_F32 || d.layout != RT_TN || d.splits > 1 || d.epi != RT_EPI_NONE || d.colsum == nullptr ||
      d.ldc != d.N || d.M <= 0 || d.N <= 0 || d.K <= 0)
    return false;
  // Whole 64x64 tiles with float4 stores; a product of 512 128x128 tiles or
  // more is left to its own, larger tiles (and its update to the optimizer).
  const F32Args a = make_args(d);
  if (a.M % 64 != 0 || a.N % 64 != 0 || !a.vec_c || !split_ok(a) || row_order_tn(a) ||
      (long long)((a.M + 127) / 128) * ((a.N + 127) / 128) >= 512)
    return false;
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  const OptTensor &W = wb[0], &Bt = wb[1];
  const bool adam = P.kind == 0, need_m = adam || P.momentum != 0.0f;
  for (const OptTensor* T : {&W, &Bt}) {
    if (T->theta == nullptr || T->parts != nullptr || T->half_copy != nullptr) return false;
    if (need_m != (T->m != nullptr) || (adam && T->v == nullptr)) return false;
  }
  return W.n == (size_t)d.M * d.N && Bt.n == (size_t)d.N && W.grad == d.C && Bt.grad == d.colsum &&
         al16(W.theta) && (W.m == nullptr || al16(W.m)) && (!adam || al16(W.v));
}

hipError_t gemm_opt_launch(hipStream_t s, const GemmDesc& d, const OptTensor* ts, int nt, const OptParams& P,
                           const OptTensor* upd) {
  if (!gemm_opt_supported(d, ts, nt, P)) return hipErrorInvalidValue;
  if (upd != nullptr && !gemm_opt_update_ok(d, upd, P)) return hipErrorInvalidValue;
  rt_opt::OptBatch b{};
  long long opt_blocks = 0;
  double bytes = 0.0;
  hipError_t e = rt_opt::make_batch(ts, nt, P, b, &opt_blocks, &bytes);
  if (e != hipSuccess) return e;
  // The tile the TN GEMM's own launch would take (same bits).
  F32Args a = make_args(d);
  if (upd != nullptr) {
    a.tiles_m = a.M / 64;
    a.tiles_n = a.N / 64;
    const long long n_gemm = (long long)a.tiles_m * a.tiles_n;
    if (n_gemm + opt_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    UpdEpi u{upd[0], upd[1], P};
    u.P.skip_count = nullptr;  // counted by the optimizer blocks of the launch
    return by_update_tile(a, [&](auto t) {
      using T = decltype(t);
      rt::launch(gemm_f32_opt_upd_kernel<T>, dim3((unsigned)(n_gemm + opt_blocks)), dim3(T::THREADS), 0, s, a, b,
                 (int)n_gemm, u);
      return hipGetLastError();
    });
  }
  return by_tn_tile(a, [&](auto t) { return launch_gemm_opt<decltype(t)>(s, a, b, opt_blocks); });
}

hipError_t gemm_opt_update2_launch(hipStream_t s, const GemmDesc& d0, const OptTensor* upd0, const GemmDesc& d1,
                                   const OptTensor* upd1, const OptTensor* ts, int nt, const OptParams& P) {
  if (!gemm_opt_supported(d0, ts, nt, P) || !gemm_opt_update_ok(d0, upd0, P) || !gemm_opt_update_ok(d1, upd1, P))
    return hipErrorInvalidValue;
  rt_opt::OptBatch b{};
  long long opt_blocks = 0;
  double bytes = 0.0;
  hipError_t e = rt_opt::make_batch(ts, nt, P, b, &opt_blocks, &bytes);
  if (e != hipSuccess) return e;
  F32Args a0 = make_args(d0), a1 = make_args(d1);
  for (F32Args* a : {&a0, &a1}) {
    a->tiles_m = a->M / 64;
    a->tiles_n = a->N / 64;
  }
  const long long n0 = ((long long)a0.tiles_m * a0.tiles_n + 7) / 8 * 8;
  const long long n1 = n0 + (long long)a1.tiles_m * a1.tiles_n;
  if (n1 + opt_blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  UpdEpi u0{upd0[0], upd0[1], P}, u1{upd1[0], upd1[1], P};
  u0.P.skip_count = u1.P.skip_count = nullptr;  // counted by the optimizer blocks of the launch
  if (dma_better<false, false>(a0) != dma_better<false, false>(a1)) return hipErrorInvalidValue;  // one batch, one K
  return by_update_tile(a0, [&](auto t) {
    using T = decltype(t);
    rt::launch(gemm_f32_opt_upd2_kernel<T>, dim3((unsigned)(n1 + opt_blocks)), dim3(T::THREADS), 0, s, a0, a1, b,
               (int)n0, (int)n1, u0, u1);
    return hipGetLastError();
  });
}

bool gemm_pair_supported(const GemmDesc& d0, const GemmDesc& d1) {
  if (d0.in_dtype != RT_F32 || d1.in_dtype != RT_F32) return false;
  if (d0.layout != RT_TN || d1.layout != RT_NT || d1.splits > 1) return false;
  if (d0.M > kMostRows || d1.M > kMostRows) return false;
  // Where the dW alone does not fill the chip with the largest tile.
  const F32Args a0 = make_args(d0), a1 = make_args(d1);
  return (split_ok(a0) || row_order_tn(a0)) && split_ok(a1) && pick_tile(a0) != kT128x64;
}

hipError_t gemm_pair_launch(hipStream_t s, const GemmDesc& d0, const GemmDesc& d1) {
  if (!gemm_pair_supported(d0, d1)) return hipErrorInvalidValue;
  const F32Args a0 = make_args(d0), a1 = make_args(d1);
  // dX takes the rank-K block for K <= 16, else the tile of its own launch;
  // a dW next to it 64x64 tiles (the launch has blocks enough) unless it is
  // narrow.  Each product is computed as in its own launch (same bits).
  auto with_dx = [&](auto t0) {
    using T0 = decltype(t0);
    if (rank_k_ok(a1)) return launch_pair_tn_nt<T0, F32RankK>(s, a0, a1);
    if (dma_better<true, true>(a1)) return launch_pair_tn_nt<T0, F32DmaTile<true, true>>(s, a0, a1);
    if (plain_tile<true, true>(a1)) return launch_pair_tn_nt<T0, F32Tile<true, true>>(s, a0, a1);
    return pick_tile(a1) == kT128x64 ? launch_pair_tn_nt<T0, F32Split<2, 4, true, true>>(s, a0, a1)
                                     : launch_pair_tn_nt<T0, F32Split<1, 4, true, true>>(s, a0, a1);
  };
  if (dma_better<false, false>(a0)) return with_dx(F32DmaTile<false, false>{});
  if (row_order_tn(a0) && a0.N <= 32) return with_dx(F32Tile<false, false, 32>{});
  if (plain_tile<false, false>(a0)) return with_dx(F32Tile<false, false>{});
  return a0.N <= 32 ? with_dx(F32Split<1, 2, false, false>{}) : with_dx(F32Split<1, 4, false, false>{});
}

hipError_t splitk_reduce_launch(hipStream_t s, const float* partials, int splits, long long stride, int M, int N,
                                void* C, int out_dtype, int ldc, int epi, const float* bias, const void* mask,
                                int mask_dtype, const float* colsum_partials, float* colsum, int cs_rows,
                                int* nf_flag) {
  if (out_dtype != RT_F32 || mask_dtype != RT_F32) return hipErrorInvalidValue;
  const long long total = (long long)M * N;
  auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec4 = N % 4 == 0 && ldc % 4 == 0 && stride % 4 == 0 && al16(partials) && al16(C) &&
                    (bias == nullptr || al16(bias)) && (mask == nullptr || al16(mask));
  const long long items = vec4 ? total / 4 : total;
  int blocks = (int)std::min<long long>((items + 255) / 256, 4096);
  if (blocks < 1) blocks = 1;
  const int cs_blocks = colsum != nullptr ? (N + 255) / 256 : 0;
  rt::launch(splitk_reduce_kernel, dim3(blocks + cs_blocks), dim3(256), 0, s, partials, splits, stride, M, N,
             static_cast<float*>(C), ldc, epi, bias, static_cast<const float*>(mask), colsum_partials, cs_rows, colsum,
             cs_blocks, vec4 ? 1 : 0, nf_flag);
  return hipGetLastError();
}

}  // namespace rt
