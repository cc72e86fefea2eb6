// fp32 MFMA GEMM for the rank-space contractions of the VAMP / CD path.
//
//   P[s] = A[:, Ks] * op(B)[Ks, :]        (split-K partials, s = 0..splits-1)
//   C    = alpha * sum_s P[s] + beta * C  (deterministic split order)
//
// A is M x K row-major (lda).  op(B)(k, n) is B[k*ldb + n] (trans_b = 0),
// B[n*ldb + k] (trans_b = 1, e.g. V^T from V), or B[rows[k]*ldb + n] (row gather,
// used by the CD Schur update H[order[window], :]).
//
// Tiling for gfx950: 256 threads = 4 wave64s; work-group tile BM x BN, wave tile
// WM x WN built from v_mfma_f32_32x32x2_f32 (full fp32 precision).  Tiles are
// staged through LDS as [k][m] / [k][n] (each MFMA operand read is 32 consecutive
// floats), double-buffered.  Interior tiles (the rank-space products always are) run
// gemm_f32_full_kernel: no bounds checks and two K slabs of global loads in flight;
// ragged or gathered products run gemm_f32_kernel with one slab of register prefetch.
#include "gemm.h"
#include "f16_pair.h"

namespace mpq {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kBK = 16;  // K slab of the default configurations (k_per_split is a multiple of 32)
constexpr int kThreads = 256;

template <int BM, int BN, int WM, int WN, bool TRANS_B, bool GATHER_B, int kBK = 16, bool PRE_C = false>
__global__ __launch_bounds__(kThreads) void gemm_f32_kernel(GemmParams p) {
  constexpr int WAVES_N = BN / WN;
  constexpr int MI = WM / 32;
  constexpr int NI = WN / 32;
  constexpr int PAD = 4;
  constexpr int LDA_S = BM + PAD;
  constexpr int LDB_S = BN + PAD;
  // per-thread loads per K slab
  constexpr int A_F4 = BM * kBK / 4 / kThreads;
  constexpr int B_F4 = BN * kBK / 4 / kThreads;
  static_assert(A_F4 >= 1 && B_F4 >= 1, "tile too small for 256 threads");

  __shared__ float As[2][kBK][LDA_S];
  __shared__ float Bs[2][kBK][LDB_S];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WM;
  const int wn0 = (wave % WAVES_N) * WN;

  const int64_t m0 = (int64_t)blockIdx.y * BM;
  const int64_t n0 = (int64_t)blockIdx.x * BN;
  if (p.lower_only && n0 >= m0 + BM + p.upper_band) return;  // uniform, before any barrier
  const int split = blockIdx.z;
  const int32_t* b_rows = p.b_rows;
  if (GATHER_B && p.b_rows_group > 0) b_rows += (m0 / p.b_rows_group) * p.b_rows_group_stride;
  const int64_t kbeg = (int64_t)split * p.k_per_split;
  int64_t kend = kbeg + p.k_per_split;
  if (kend > p.K) kend = p.K;

  floatx16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // PRE_C (axpby epilogue with beta != 0): this lane's C entries are loaded before the K loop, so
  // their latency overlaps the MFMAs instead of stalling the epilogue.  Rows/columns outside C
  // read a clamped in-range entry (never used) so the loads need no branches.
  float cpre[PRE_C ? MI : 1][PRE_C ? NI : 1][PRE_C ? 16 : 1];
  if constexpr (PRE_C) {
    const int col = lane & 31;
    const int rbase = (lane >> 5) * 4;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int64_t gn = min(n0 + wn0 + j * 32 + col, p.N - 1);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int64_t gm = min(m0 + wm0 + i * 32 + (v >> 2) * 8 + rbase + (v & 3), p.M - 1);
          cpre[i][j][v] = p.C[gm * p.ldc + gn];
        }
      }
  }

  float4 ra[A_F4];
  float4 rb[B_F4];

  // A slab: element (m, k) = A[(m0+m)*lda + k0 + k]; thread t loads float4 along k.
  auto load_a = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < A_F4; ++i) {
      const int t = tid + i * kThreads;
      const int m = t / (kBK / 4);
      const int kq = (t % (kBK / 4)) * 4;
      const int64_t gm = m0 + m;
      const int64_t gk = k0 + kq;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (gm < p.M) {
        const float* src = p.A + gm * p.lda + gk;
        if (gk + 3 < kend && p.a_vec4) {
          v = *reinterpret_cast<const float4*>(src);
        } else {
          if (gk + 0 < kend) v.x = src[0];
          if (gk + 1 < kend) v.y = src[1];
          if (gk + 2 < kend) v.z = src[2];
          if (gk + 3 < kend) v.w = src[3];
        }
      }
      ra[i] = v;
    }
  };
  auto store_a = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_F4; ++i) {
      const int t = tid + i * kThreads;
      const int m = t / (kBK / 4);
      const int kq = (t % (kBK / 4)) * 4;
      As[buf][kq + 0][m] = ra[i].x;
      As[buf][kq + 1][m] = ra[i].y;
      As[buf][kq + 2][m] = ra[i].z;
      As[buf][kq + 3][m] = ra[i].w;
    }
  };
  auto load_b = [&](int64_t k0) {
#pragma unroll
    for (int i = 0; i < B_F4; ++i) {
      const int t = tid + i * kThreads;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if constexpr (!TRANS_B) {
        const int k = t / (BN / 4);
        const int nq = (t % (BN / 4)) * 4;
        const int64_t gk = k0 + k;
        const int64_t gn = n0 + nq;
        if (gk < kend) {
          int64_t row = gk;
          if constexpr (GATHER_B) row = b_rows[gk];
          const float* src = p.B + row * p.ldb + gn;
          if (gn + 3 < p.N && p.b_vec4) {
            v = *reinterpret_cast<const float4*>(src);
          } else {
            if (gn + 0 < p.N) v.x = src[0];
            if (gn + 1 < p.N) v.y = src[1];
            if (gn + 2 < p.N) v.z = src[2];
            if (gn + 3 < p.N) v.w = src[3];
          }
        }
      } else {
        const int n = t / (kBK / 4);
        const int kq = (t % (kBK / 4)) * 4;
        const int64_t gn = n0 + n;
        const int64_t gk = k0 + kq;
        if (gn < p.N) {
          const float* src = p.B + gn * p.ldb + gk;
          if (gk + 3 < kend && p.b_vec4) {
            v = *reinterpret_cast<const float4*>(src);
          } else {
            if (gk + 0 < kend) v.x = src[0];
            if (gk + 1 < kend) v.y = src[1];
            if (gk + 2 < kend) v.z = src[2];
            if (gk + 3 < kend) v.w = src[3];
          }
        }
      }
      rb[i] = v;
    }
  };
  auto store_b = [&](int buf) {
#pragma unroll
    for (int i = 0; i < B_F4; ++i) {
      const int t = tid + i * kThreads;
      if constexpr (!TRANS_B) {
        const int k = t / (BN / 4);
        const int nq = (t % (BN / 4)) * 4;
        *reinterpret_cast<float4*>(&Bs[buf][k][nq]) = rb[i];
      } else {
        const int n = t / (kBK / 4);
        const int kq = (t % (kBK / 4)) * 4;
        Bs[buf][kq + 0][n] = rb[i].x;
        Bs[buf][kq + 1][n] = rb[i].y;
        Bs[buf][kq + 2][n] = rb[i].z;
        Bs[buf][kq + 3][n] = rb[i].w;
      }
    }
  };

  const int64_t nslab = (kend - kbeg + kBK - 1) / kBK;
  if (nslab > 0) {
    load_a(kbeg);
    load_b(kbeg);
    store_a(0);
    store_b(0);
    __syncthreads();
    for (int64_t s = 0; s < nslab; ++s) {
      const int buf = (int)(s & 1);
      if (s + 1 < nslab) {
        load_a(kbeg + (s + 1) * kBK);
        load_b(kbeg + (s + 1) * kBK);
      }
      const int kl = lane >> 5;  // operand k row within a 2-step
      const int ml = lane & 31;
#pragma unroll
      for (int kk = 0; kk < kBK; kk += 2) {
        float a[MI], b[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) a[i] = As[buf][kk + kl][wm0 + i * 32 + ml];
#pragma unroll
        for (int j = 0; j < NI; ++j) b[j] = Bs[buf][kk + kl][wn0 + j * 32 + ml];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      if (s + 1 < nslab) {
        store_a(buf ^ 1);
        store_b(buf ^ 1);
      }
      __syncthreads();
    }
  }

  // Epilogue: lane l, accumulator v -> row 8*(v/4) + 4*(l/32) + v%4, col l%32.
  const int col = lane & 31;
  const int rbase = (lane >> 5) * 4;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int64_t gn = n0 + wn0 + j * 32 + col;
      if (gn >= p.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t gm = m0 + wm0 + i * 32 + (v >> 2) * 8 + rbase + (v & 3);
        if (gm >= p.M) continue;
        const float val = acc[i][j][v];
        if (p.mode == kGemmPartials) {
          p.C[(int64_t)split * p.split_stride + gm * p.ldc + gn] = val;
        } else {  // kGemmAxpby, single split: C = alpha*acc + beta*C
          float* dst = p.C + gm * p.ldc + gn;
          if constexpr (PRE_C) {
            *dst = p.alpha * val + p.beta * cpre[i][j][v];
          } else {
            *dst = p.beta == 0.f ? p.alpha * val : p.alpha * val + p.beta * *dst;
          }
        }
      }
    }
  }
}

// Deterministic split-K reduction: C = alpha * sum_s P[s] + beta * C.
__global__ void splitk_reduce_kernel(const float* __restrict__ P, int splits, int64_t split_stride,
                                     int64_t M, int64_t N, float* __restrict__ C, int64_t ldc,
                                     float alpha, float beta) {
  const int64_t total = M * N;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t m = e / N, n = e % N;
    const float acc = sum_splits(P, splits, split_stride, m * N + n);
    float* dst = C + m * ldc + n;
    *dst = beta == 0.f ? alpha * acc : alpha * acc + beta * *dst;
  }
}

// Interior-tile variant: every M/N tile and K slab is in range and 16-byte aligned (checked by
// the host), no row gather.  Two K slabs of global loads are kept in flight (register sets R0/R1,
// the loop is unrolled by two so both sets are static), and a slab's LDS operands are all read
// before its MFMA chain, so each slab waits once for LDS and once for global memory.
template <int BM, int BN, int WM, int WN, bool TRANS_B, int HOIST = 8, bool PRE_C = false, bool GATHER_B = false>
__global__ __launch_bounds__(kThreads) void gemm_f32_full_kernel(GemmParams p) {
  static_assert(!(GATHER_B && TRANS_B), "row gather needs a row-major K x N B");
  constexpr int BK = 16;
  constexpr int WAVES_N = BN / WN;
  constexpr int MI = WM / 32;
  constexpr int NI = WN / 32;
  constexpr int LDA_S = BM + 4;
  constexpr int LDB_S = BN + 4;
  constexpr int A_F4 = BM * BK / 4 / kThreads;
  constexpr int B_F4 = BN * BK / 4 / kThreads;
  static_assert(A_F4 >= 1 && B_F4 >= 1, "tile too small for 256 threads");

  __shared__ float As[2][BK][LDA_S];
  __shared__ float Bs[2][BK][LDB_S];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm0 = (wave / WAVES_N) * WM;
  const int wn0 = (wave % WAVES_N) * WN;
  const int64_t m0 = (int64_t)blockIdx.y * BM;
  const int64_t n0 = (int64_t)blockIdx.x * BN;
  if (p.lower_only && n0 >= m0 + BM + p.upper_band) return;  // uniform, before any barrier
  const int split = blockIdx.z;
  const int64_t kbeg = (int64_t)split * p.k_per_split;
  const int64_t nslab = p.k_per_split / BK;

  // per-thread global source pointers of the first slab (advanced by BK per slab)
  const float* asrc[A_F4];
  const float* bsrc[B_F4];
#pragma unroll
  for (int i = 0; i < A_F4; ++i) {
    const int t = tid + i * kThreads;
    asrc[i] = p.A + (m0 + t / (BK / 4)) * p.lda + kbeg + (t % (BK / 4)) * 4;
  }
#pragma unroll
  for (int i = 0; i < B_F4; ++i) {
    const int t = tid + i * kThreads;
    if constexpr (!TRANS_B) {
      bsrc[i] = p.B + (kbeg + t / (BN / 4)) * p.ldb + n0 + (t % (BN / 4)) * 4;
    } else {
      bsrc[i] = p.B + (n0 + t / (BK / 4)) * p.ldb + kbeg + (t % (BK / 4)) * 4;
    }
  }
  const int64_t b_step = TRANS_B ? BK : BK * p.ldb;
  // GATHER_B: K row k of B is B[b_rows[k]] (per M tile group as in gemm_f32_kernel); each thread
  // reads its slab row index in the same two-slabs-ahead prefetch as the data
  const int32_t* b_rows = p.b_rows;
  if (GATHER_B && p.b_rows_group > 0) b_rows += (m0 / p.b_rows_group) * p.b_rows_group_stride;

  float4 ra0[A_F4], rb0[B_F4], ra1[A_F4], rb1[B_F4];
  auto gload = [&](float4 (&ra)[A_F4], float4 (&rb)[B_F4], int64_t s) {
#pragma unroll
    for (int i = 0; i < A_F4; ++i) ra[i] = *reinterpret_cast<const float4*>(asrc[i] + s * BK);
#pragma unroll
    for (int i = 0; i < B_F4; ++i) {
      if constexpr (GATHER_B) {
        const int t = tid + i * kThreads;
        const int64_t row = b_rows[kbeg + s * BK + t / (BN / 4)];
        rb[i] = *reinterpret_cast<const float4*>(p.B + row * p.ldb + n0 + (t % (BN / 4)) * 4);
      } else {
        rb[i] = *reinterpret_cast<const float4*>(bsrc[i] + s * b_step);
      }
    }
  };
  auto lstore = [&](const float4 (&ra)[A_F4], const float4 (&rb)[B_F4], int buf) {
#pragma unroll
    for (int i = 0; i < A_F4; ++i) {
      const int t = tid + i * kThreads;
      const int m = t / (BK / 4);
      const int kq = (t % (BK / 4)) * 4;
      As[buf][kq + 0][m] = ra[i].x;
      As[buf][kq + 1][m] = ra[i].y;
      As[buf][kq + 2][m] = ra[i].z;
      As[buf][kq + 3][m] = ra[i].w;
    }
#pragma unroll
    for (int i = 0; i < B_F4; ++i) {
      const int t = tid + i * kThreads;
      if constexpr (!TRANS_B) {
        *reinterpret_cast<float4*>(&Bs[buf][t / (BN / 4)][(t % (BN / 4)) * 4]) = rb[i];
      } else {
        const int n = t / (BK / 4);
        const int kq = (t % (BK / 4)) * 4;
        Bs[buf][kq + 0][n] = rb[i].x;
        Bs[buf][kq + 1][n] = rb[i].y;
        Bs[buf][kq + 2][n] = rb[i].z;
        Bs[buf][kq + 3][n] = rb[i].w;
      }
    }
  };

  floatx16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // PRE_C: this lane's C entries of an axpby epilogue with beta != 0, loaded before the K loop
  float cpre[PRE_C ? MI : 1][PRE_C ? NI : 1][PRE_C ? 16 : 1];
  if constexpr (PRE_C) {
    const int col = lane & 31;
    const int rbase = (lane >> 5) * 4;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const int64_t gn = n0 + wn0 + j * 32 + col;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int64_t gm = m0 + wm0 + i * 32 + (v >> 2) * 8 + rbase + (v & 3);
          cpre[i][j][v] = p.C[gm * p.ldc + gn];
        }
      }
  }

  const int kl = lane >> 5;
  const int ml = lane & 31;
  auto compute = [&](int buf) {
#pragma unroll
    for (int k0 = 0; k0 < BK / 2; k0 += HOIST) {
      float a[HOIST][MI], b[HOIST][NI];
#pragma unroll
      for (int kk = 0; kk < HOIST; ++kk) {
#pragma unroll
        for (int i = 0; i < MI; ++i) a[kk][i] = As[buf][2 * (k0 + kk) + kl][wm0 + i * 32 + ml];
#pragma unroll
        for (int j = 0; j < NI; ++j) b[kk][j] = Bs[buf][2 * (k0 + kk) + kl][wn0 + j * 32 + ml];
      }
#pragma unroll
      for (int kk = 0; kk < HOIST; ++kk)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[kk][i], b[kk][j], acc[i][j], 0, 0, 0);
    }
  };

  // prologue: slab 0 -> LDS buffer 0, slab 1 in flight in R1 (nslab is even)
  gload(ra0, rb0, 0);
  gload(ra1, rb1, 1);
  lstore(ra0, rb0, 0);
  __syncthreads();
  // slab s is in LDS buffer s&1; slab s+1 is in flight in R((s+1)&1).  The body covers two slabs
  // with no early exit: an exit between the halves leaves the accumulators in different registers
  // on the two paths, and the compiler then copies all of them through VGPRs every iteration,
  // which drains the MFMA pipeline (measured 88 -> 121 TFLOP/s at 128 x 14336 x 14336).
  for (int64_t s = 0; s < nslab; s += 2) {
    if (s + 2 < nslab) gload(ra0, rb0, s + 2);
    compute(0);
    lstore(ra1, rb1, 1);
    __syncthreads();
    if (s + 3 < nslab) gload(ra1, rb1, s + 3);
    compute(1);
    if (s + 2 < nslab) lstore(ra0, rb0, 0);
    __syncthreads();
  }

  const int col = lane & 31;
  const int rbase = (lane >> 5) * 4;
#pragma unroll
  for (int i = 0; i < MI; ++i) {
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const int64_t gn = n0 + wn0 + j * 32 + col;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int64_t gm = m0 + wm0 + i * 32 + (v >> 2) * 8 + rbase + (v & 3);
        const float val = acc[i][j][v];
        if (p.mode == kGemmPartials) {
          p.C[(int64_t)split * p.split_stride + gm * p.ldc + gn] = val;
        } else {
          float* dst = p.C + gm * p.ldc + gn;
          if constexpr (PRE_C) {
            *dst = p.alpha * val + p.beta * cpre[i][j][v];
          } else {
            *dst = p.beta == 0.f ? p.alpha * val : p.alpha * val + p.beta * *dst;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// fp32 product on the 16-bit matrix cores (the "x6" entry points; the name is older than the split).
// Both operands are held as pairs of f16 planes of scaled values (f16_pair.h), x s = x0 + x1 to about
// 2^-23 |x s|, and the product keeps three of the four plane products,
//   a b s = a0 b0 + (a0 b1 + a1 b0) + e,   |e| = |a1 b1| <= 2^-22 |a0 b0|,
// each exact in the fp32 accumulator of v_mfma_f32_32x32x16_f16.  That is half the products of a split
// into three bf16 planes (six), with about the same representation error as one fp32 rounding per operand
// and a third of the roundings into the accumulator.  f16 has five exponent bits, so the planes are scaled by
// powers of two: A's by the largest magnitude of (row, 1024 columns of K), found where A is packed; B's by a
// running scale per column that its wave finds as it goes.  A's scale changes along K, so each chunk's sum
// is added, unscaled, to a second set of accumulators, which also shortens the chains of roundings.
//
// Operands are packed into 128-row x 16-k tiles in MFMA fragment order: chunk c = (blk*2 + h)*32 + r
// of a tile holds row blk*32 + r at k = 16 ks + 8 h + (0..7).  B (the large, reused operand) is
// packed once as fp32 [N/128][K/16][2][256 chunks][4] (first and second four k of every chunk in two
// 4 KB halves, so a fragment is two conflict-free 16-byte LDS reads); as f16 pairs it would take the same
// bytes but need its column scales at hand.  A (small, re-formed per product) is packed as planes
// [ceil(M/128)][K/16][2][256][8] and its reciprocal scales.  A work-group (128 x 128 tile, one K slice, four
// waves of 128 x 32) reads each K slab as contiguous 8 KB (A, L2-resident) + 8 KB (B); every wave splits only
// its own 32 columns of B and runs 12 MFMAs per slab.  Split s of tile t is block t * splits + s, so with
// 8 or 16 splits every XCD (blocks are dispatched round-robin over 8) works on one or two K slices
// and its L2 holds those slices of A.
//
// Bound at 128 rows: reading B.  128 x 14336 x 14336 (4 splits): 278 -> 206 us (4.0 TB/s of B; the
// card copies at 4.7), 128 x 8192 x 8192 95 -> 74, 128 x 4096 x 4096 26.7 -> 23.4, against the six bf16 products of
// the same tiling, with a relative error of 3.6e-7 against 9.9e-7 at 14336 (fp32 MFMA 7.6e-7).  At 4096 rows, bound
// by the matrix cores: 4096 x 14336 x 14336 7.99 -> 5.56 ms.
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));


// B tiles: thread per chunk (8 floats).  trans_b: op(B)(k, n) = B[n*ldb + k] (32 contiguous bytes
// per thread), else B[k*ldb + n] (lanes along n).
template <bool TRANS_B>
__global__ void x6_pack_b_kernel(const float* __restrict__ B, int64_t ldb, int64_t K, int64_t N, float* __restrict__ Bt) {
  const int64_t KS = K / 16;
  const int64_t nchunks = (N / 128) * KS * 256;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nchunks; q += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(q & 255);
    const int64_t tk = q >> 8;  // nt * KS + ks
    const int64_t nt = tk / KS, ks = tk - nt * KS;
    const int64_t n = nt * 128 + (c >> 6) * 32 + (c & 31), k0 = ks * 16 + ((c >> 5) & 1) * 8;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = TRANS_B ? B[n * ldb + k0 + e] : B[(k0 + e) * ldb + n];
    float4* d = reinterpret_cast<float4*>(Bt) + tk * 512 + c;
    d[0] = make_float4(v[0], v[1], v[2], v[3]);
    d[256] = make_float4(v[4], v[5], v[6], v[7]);
  }
}

// A pairs (of A diag(colscale) when colscale is given): work-group per (row, 1024 columns); rows >= M
// are zero.
__global__ __launch_bounds__(kThreads) void x6_pack_a_kernel(const float* __restrict__ A, int64_t lda, int64_t M,
                                                             int64_t K, uint4* __restrict__ At,
                                                             const float* __restrict__ colscale, int chunks,
                                                             bool vec4) {
  __shared__ float red[4];
  const int64_t b = blockIdx.x / chunks;
  const int64_t chunk = blockIdx.x - b * chunks;
  const int64_t j0 = chunk * kPairChunk + 4 * (int64_t)threadIdx.x;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (b < M && j0 < K) {
    const float* src = A + b * lda + j0;
    if (vec4) v = *reinterpret_cast<const float4*>(src);
    else v = make_float4(src[0], src[1], src[2], src[3]);
    if (colscale) {
      v.x *= colscale[j0];
      v.y *= colscale[j0 + 1];
      v.z *= colscale[j0 + 2];
      v.w *= colscale[j0 + 3];
    }
  }
  pack_pair_chunk(At, M, K, b, chunk, v, red);
}

// s_waitcnt immediate that waits for vmcnt <= n only (gfx9 encoding: vmcnt bits 3:0 and 15:14).
constexpr int vmcnt_imm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

// C[split] (rows < M) = A[:, K slice] * op(B)[K slice, :] from the packed operands, the slabs moved by
// global_load_lds into a ring of four LDS
// stages (three slabs in flight, no register staging).  Each stage is its own __shared__ array and
// the loops are unrolled by four, so every stage index is a constant: the compiler then tells the
// stages apart and waits only where this code waits (s_waitcnt vmcnt(n) before each barrier: all
// but the n most recent loads of this wave done, i.e. the slab about to be read).  The barrier is
// s_barrier without a fence (the fence of __syncthreads would wait for every load in flight).
// kRagged: K slices of any number of slabs; otherwise every slice is a positive multiple of four.
// kStream: B is read with the non-temporal hint (it does not fit the caches anyway).
template <bool kRagged, bool kStream>
__global__ __launch_bounds__(kThreads, 2) void gemm_x6_kernel(int64_t M, int64_t N, int64_t K,
                                                              const uint4* __restrict__ At,
                                                              const float* __restrict__ Bt, float* __restrict__ C,
                                                              int64_t ldc, int64_t split_stride,
                                                              int64_t k_per_split, int splits) {
  constexpr int S = 4;
  constexpr int STAGE = 512 + 512;  // 16-byte slots: A planes, then the two halves of B
  constexpr int LOADS = 4;          // global_load_lds per wave per slab: 2 (A) + 2 (B)
  constexpr int RT = 4;             // 32-row tiles of a wave (128 x 32)
  constexpr int FAC = 16;           // chunks of A's scales kept in LDS
  __shared__ uint4 st0[STAGE];
  __shared__ uint4 st1[STAGE];
  __shared__ uint4 st2[STAGE];
  __shared__ uint4 st3[STAGE];
  __shared__ float fac[FAC][128];
  auto stage = [&](int slot) -> uint4* { return slot == 0 ? st0 : slot == 1 ? st1 : slot == 2 ? st2 : st3; };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const unsigned utile = blockIdx.x / (unsigned)splits, ntn = (unsigned)(N / 128);  // 32-bit divisions: short
  const int split = (int)(blockIdx.x - utile * (unsigned)splits);
  const int64_t mt = utile / ntn, nt = utile % ntn;
  const int64_t KS = K / 16;
  const int nslab = (int)(k_per_split / 16);
  const int64_t ks0 = (int64_t)split * nslab;
  // wave w moves A slots w*128 + 64 q and B slots w*128 + 64 q (q < 2); lane l adds 16 l bytes
  const uint4* asrc = At + (mt * KS + ks0) * 512 + wave * 128 + lane;
  const uint4* bsrc = reinterpret_cast<const uint4*>(Bt) + (nt * KS + ks0) * 512 + wave * 128 + lane;
  auto issue = [&](int s, int slot) {
    uint4* d = stage(slot);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_global_load_lds(asrc + (int64_t)s * 512 + q * 64, d + wave * 128 + q * 64, 16, 0, 0);
#pragma unroll
    for (int q = 0; q < 2; ++q)
      __builtin_amdgcn_global_load_lds(bsrc + (int64_t)s * 512 + q * 64, d + 512 + wave * 128 + q * 64, 16, 0,
                                       kStream ? 2 : 0);
  };
  // slabs past the end of the slice are the last one again (never multiplied), so every step issues the
  // same number of loads and waits for the same count
  auto clamp_slab = [&](int t) { return t < nslab ? t : nslab - 1; };
  // reciprocal scales of A's rows in the chunks of this slice: loaded before the first slabs, in LDS
  // some barriers before they are read
  const int64_t Mp = (M + 127) / 128 * 128;
  const float* inv = reinterpret_cast<const float*>(At + Mp * K / 4) + mt * 128;
  const int c0 = (int)(ks0 >> 6), nch = (int)((ks0 + nslab - 1) >> 6) - c0 + 1;  // kPairChunk = 64 slabs
  float fq[FAC / 2];
#pragma unroll
  for (int q = 0; q < FAC / 2; ++q) {
    const int c = 2 * q + (tid >> 7);
    fq[q] = inv[(c0 + (c < nch ? c : nch - 1)) * Mp + (tid & 127)];
  }
#pragma unroll
  for (int t = 0; t < S - 1; ++t) issue(clamp_slab(t), t);
#pragma unroll
  for (int q = 0; q < FAC / 2; ++q) fac[2 * q + (tid >> 7)][tid & 127] = fq[q];

  floatx16 acc[RT], total[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = total[i][v] = 0.f;
  // this lane's column of B (shared with lane ^ 32): scale, and the magnitude it holds up to.  The first
  // nonzero slab sets the scale, with three bits to spare for larger values in later slabs.
  float bs = 0x1p120f, blim = 60000.f * 0x1p-120f;
  const int rbase = (lane >> 5) * 4;

  // total += acc / (scales), for the chunk c of this slice
  auto flush = [&](int c) {
    const float binv = 1.f / bs;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = i * 32 + q * 8 + rbase;
        const float4 f = nch <= FAC ? *reinterpret_cast<const float4*>(&fac[c][r])
                                    : *reinterpret_cast<const float4*>(inv + (int64_t)(c0 + c) * Mp + r);
        const float fv[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          total[i][4 * q + v] += acc[i][4 * q + v] * fv[v] * binv;
          acc[i][4 * q + v] = 0.f;
        }
      }
  };

  auto compute = [&](int slot) {
    const uint4* d = stage(slot);
    f16x8 a[2][RT];
#pragma unroll
    for (int pl = 0; pl < 2; ++pl)
#pragma unroll
      for (int i = 0; i < RT; ++i) a[pl][i] = __builtin_bit_cast(f16x8, d[pl * 256 + i * 64 + lane]);
    const float4 x = __builtin_bit_cast(float4, d[512 + wave * 64 + lane]);
    const float4 y = __builtin_bit_cast(float4, d[512 + 256 + wave * 64 + lane]);
    const float m = fmaxf(fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fmaxf(fabsf(x.z), fabsf(x.w))),
                          fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
    if (__builtin_amdgcn_ballot_w64(m > blim)) {  // rare: a column outgrew its scale
      const float mc = fmaxf(m, __shfl_xor(m, 32));
      if (mc > blim && mc < INFINITY) {
        const float ns = pair_scale(mc, 12);
        const float f = ns / bs;
        bs = ns;
        blim = 60000.f / ns;
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][v] *= f;
      }
    }
    uint4 h, l;
    split2(x.x, x.y, bs, h.x, l.x);
    split2(x.z, x.w, bs, h.y, l.y);
    split2(y.x, y.y, bs, h.z, l.z);
    split2(y.z, y.w, bs, h.w, l.w);
    const f16x8 b0 = __builtin_bit_cast(f16x8, h), b1 = __builtin_bit_cast(f16x8, l);
    // smallest terms first; the row tiles innermost keep four independent accumulator chains
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[1][i], b0, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][i], b1, acc[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][i], b0, acc[i], 0, 0, 0);
  };
  auto sync = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // slab t is the last of its chunk of A's scales, or of the slice
  auto chunk_ends = [&](int t) { return t + 1 == nslab || ((ks0 + t) & 63) == 63; };
  // Slab t lives in stage t % 4.  Step t: wait for slab t (loads of slabs t+1, t+2 may stay in
  // flight), barrier (slab t visible; every wave is done with stage (t-1) % 4), issue slab t+3 into
  // that stage, compute slab t.  One copy of the body, also for the last slabs: the code is fetched once
  // per launch, and a short product spends a good part of its time on that.
  for (int t0 = 0; t0 < nslab; t0 += S) {
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const int t = t0 + u;
      if (kRagged && t >= nslab) break;
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(LOADS * (S - 2)));
      sync();
      issue(clamp_slab(t + S - 1), (u + S - 1) % S);
      compute(u);
      if ((kRagged || u == S - 1) && chunk_ends(t)) flush((int)((ks0 + t) >> 6) - c0);  // slices start at
      // multiples of four slabs, so without kRagged chunks end with the last step
    }
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // no load may land in LDS after the work-group ends

  const int col = lane & 31;
  float* Cs = C + (int64_t)split * split_stride;
  const int64_t gn = nt * 128 + wave * 32 + col;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t gm = mt * 128 + i * 32 + (v >> 2) * 8 + rbase + (v & 3);
      if (gm < M) Cs[gm * ldc + gn] = total[i][v];
    }
}

template <int BM, int BN, int WM, int WN>
hipError_t launch_cfg(const GemmParams& p, dim3 grid, hipStream_t stream) {
  // interior-tile kernel: whole tiles, an even number of 16-wide K slabs per split; a row gather
  // also needs its groups aligned to the 128-row M tile
  const bool gather_ok = !p.b_rows || (!p.trans_b && (p.b_rows_group == 0 || p.b_rows_group % BM == 0));
  const bool full = gather_ok && p.a_vec4 && p.b_vec4 && p.M % BM == 0 && p.N % BN == 0 &&
                    p.k_per_split % 32 == 0 && (int64_t)grid.z * p.k_per_split == p.K;
  const bool pre_c = p.mode == kGemmAxpby && p.beta != 0.f;
  if (full && p.b_rows) {
    if (pre_c) hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, false, 8, true, true>), grid, dim3(kThreads), 0, stream, p);
    else hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, false, 8, false, true>), grid, dim3(kThreads), 0, stream, p);
    return hipGetLastError();
  }
  if (full) {
    if (p.trans_b) {
      if (pre_c) hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, true, 8, true>), grid, dim3(kThreads), 0, stream, p);
      else hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, true>), grid, dim3(kThreads), 0, stream, p);
    } else {
      if (pre_c) hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, false, 8, true>), grid, dim3(kThreads), 0, stream, p);
      else hipLaunchKernelGGL((gemm_f32_full_kernel<BM, BN, WM, WN, false>), grid, dim3(kThreads), 0, stream, p);
    }
    return hipGetLastError();
  }
  // (the general kernel does not prefetch C: that costs it 96 VGPRs, occupancy 6 -> 2, and measured
  // slower on the CD Schur update)
  if (p.trans_b) {
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WM, WN, true, false>), grid, dim3(kThreads), 0, stream, p);
  } else if (p.b_rows) {
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WM, WN, false, true>), grid, dim3(kThreads), 0, stream, p);
  } else {
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WM, WN, false, false>), grid, dim3(kThreads), 0, stream, p);
  }
  return hipGetLastError();
}

}  // namespace

int choose_splits(int64_t M, int64_t N, int64_t K, int64_t workspace_floats, int* bn_out) {
  // 128x64 tiles: the 128x128 variant needs 154 VGPRs + 128 AGPRs (one work-group per SIMD set),
  // which measured slower on every shape tried.
  const int64_t tiles_m = (M + 127) / 128;
  const int bn = 64;
  const int64_t tiles = tiles_m * ((N + bn - 1) / bn);
  int splits = 1;
  const int64_t target = 2048;  // ~8 work-groups per CU on 256 CUs (latency hiding at small M)
  while (splits < 32 && tiles * splits * 2 <= target && K / (splits * 2) >= 256 &&
         (int64_t)(splits * 2) * M * N <= workspace_floats)
    splits *= 2;
  *bn_out = bn;
  return splits;
}

hipError_t gemm_partials(GemmParams p, int splits, int bn, hipStream_t stream) {
  p.mode = splits > 1 ? kGemmPartials : p.mode;
  const int64_t kps = ((p.K + splits - 1) / splits + 31) / 32 * 32;
  p.k_per_split = kps > 0 ? kps : kBK;
  p.a_vec4 = ((reinterpret_cast<uintptr_t>(p.A) & 15u) == 0) && (p.lda % 4 == 0);
  p.b_vec4 = ((reinterpret_cast<uintptr_t>(p.B) & 15u) == 0) && (p.ldb % 4 == 0);
  (void)bn;  // one tile shape: 128 x 64 (4 waves of 64 x 32)
  dim3 grid((unsigned)((p.N + 63) / 64), (unsigned)((p.M + 127) / 128), (unsigned)splits);
  return launch_cfg<128, 64, 64, 32>(p, grid, stream);
}

hipError_t splitk_reduce(const float* P, int splits, int64_t split_stride, int64_t M, int64_t N, float* C,
                         int64_t ldc, float alpha, float beta, hipStream_t stream) {
  const int64_t total = M * N;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, P, splits,
                     split_stride, M, N, C, ldc, alpha, beta);
  return hipGetLastError();
}

bool x6_shape_ok(int64_t N, int64_t K) { return N > 0 && K > 0 && N % 128 == 0 && K % 32 == 0; }

// Split K until the grid holds about two work-groups per CU (512) or a K slice would fall below
// 32 slabs (512): more splits do not speed the product up and every split is one more partial the
// epilogues read.  128 x 14336 x 14336: 4 splits, 0.292 ms per product and 8.7 us to read the
// partials back, against 0.298 ms and 20.7 us with 16 (the down_proj layer: 2 splits 1085 ms, 4
// splits 1053-1062 ms).  128 x 4096 x 4096: 8 splits; a 14336 x 4096 gate_proj layer takes 391 ms
// against 414 ms with 16 splits, 451 ms with 4 and 619 ms with 2.
int x6_choose_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 127) / 128) * (N / 128);
  int splits = 1;
  while (splits < 16 && tiles * splits * 2 <= 512 && K % (splits * 2 * 32) == 0 && K / (splits * 2) >= 512)
    splits *= 2;
  return splits;
}

int64_t x6_packed_a_bytes(int64_t M, int64_t K) { return ((M + 127) / 128) * 128 * K * 6; }

static unsigned grid_for(int64_t items) {
  int64_t b = (items + 255) / 256;
  return (unsigned)(b < 1 ? 1 : b > 16384 ? 16384 : b);
}

hipError_t x6_pack_b(const float* B, int64_t ldb, bool trans_b, int64_t K, int64_t N, float* Bt, hipStream_t stream) {
  const unsigned g = grid_for((N / 128) * (K / 16) * 256);
  if (trans_b) hipLaunchKernelGGL(x6_pack_b_kernel<true>, dim3(g), dim3(256), 0, stream, B, ldb, K, N, Bt);
  else hipLaunchKernelGGL(x6_pack_b_kernel<false>, dim3(g), dim3(256), 0, stream, B, ldb, K, N, Bt);
  return hipGetLastError();
}

hipError_t x6_pack_a(const float* A, int64_t lda, int64_t M, int64_t K, void* At, hipStream_t stream,
                     const float* colscale) {
  const int64_t chunks = (K + kPairChunk - 1) / kPairChunk, blocks = (M + 127) / 128 * 128 * chunks;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  const bool vec4 = (reinterpret_cast<uintptr_t>(A) & 15u) == 0 && lda % 4 == 0;
  hipLaunchKernelGGL(x6_pack_a_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, stream, A, lda, M, K,
                     static_cast<uint4*>(At), colscale, (int)chunks, vec4);
  return hipGetLastError();
}

hipError_t x6_gemm_partials(const void* At, const float* Bt, int64_t M, int64_t N, int64_t K, float* C, int64_t ldc,
                            int64_t split_stride, int splits, hipStream_t stream) {
  const int64_t kps = K / splits;
  if (!x6_shape_ok(N, K) || splits < 1 || K % splits != 0 || kps % 32 != 0) return hipErrorInvalidValue;
  const int64_t blocks = ((M + 127) / 128) * (N / 128) * splits;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  // An operator larger than the 256 MB last-level cache is gone before the next product reads it, and only
  // pushes the other operands out: 128 x 14336 x 14336 takes 199 us with the hint and 210 without; 4096 x 4096
  // (64 MB, which stays cached between products) 31.1 with and 28.2 without.
  const bool ragged = (kps / 16) % 4 != 0, big = K * N * 4 >= ((int64_t)256 << 20);
  const auto kernel = ragged ? (big ? gemm_x6_kernel<true, true> : gemm_x6_kernel<true, false>)
                             : (big ? gemm_x6_kernel<false, true> : gemm_x6_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), 0, stream, M, N, K, static_cast<const uint4*>(At),
                     Bt, C, ldc, split_stride, kps, splits);
  return hipGetLastError();
}

hipError_t gemm_lower(const float* A, int64_t lda, const float* B, int64_t ldb, bool trans_b, float* C,
                      int64_t ldc, int64_t M, int64_t K, float alpha, float beta, int upper_band,
                      hipStream_t stream) {
  GemmParams p{};
  p.M = M; p.N = M; p.K = K;
  p.A = A; p.lda = lda; p.B = B; p.ldb = ldb; p.trans_b = trans_b;
  p.alpha = alpha; p.beta = beta;
  p.mode = kGemmAxpby;
  p.C = C; p.ldc = ldc;
  p.lower_only = true;
  p.upper_band = upper_band;
  return gemm_partials(p, 1, 64, stream);
}

hipError_t gemm(const float* A, int64_t lda, const float* B, int64_t ldb, bool trans_b,
                const int32_t* b_rows, float* C, int64_t ldc, int64_t M, int64_t N, int64_t K,
                float alpha, float beta, float* workspace, int64_t workspace_floats,
                hipStream_t stream) {
  int bn = 128;
  int splits = choose_splits(M, N, K, workspace ? workspace_floats : 0, &bn);
  // whole 32-k slices per split let interior tiles run gemm_f32_full_kernel
  if (K % 32 == 0)
    while (splits > 1 && K % (splits * 32) != 0) splits /= 2;
  GemmParams p{};
  p.M = M; p.N = N; p.K = K;
  p.A = A; p.lda = lda; p.B = B; p.ldb = ldb; p.trans_b = trans_b; p.b_rows = b_rows;
  p.alpha = alpha; p.beta = beta;
  if (splits == 1) {
    p.mode = kGemmAxpby;
    p.C = C; p.ldc = ldc;
    return gemm_partials(p, 1, bn, stream);
  }
  p.mode = kGemmPartials;
  p.C = workspace; p.ldc = N; p.split_stride = M * N;
  hipError_t e = gemm_partials(p, splits, bn, stream);
  if (e != hipSuccess) return e;
  return splitk_reduce(workspace, splits, M * N, M, N, C, ldc, alpha, beta, stream);
}

}  // namespace mpq

extern "C" int mpq_gemm_f32(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                            const float* B, int64_t ldb, int trans_b, const int32_t* b_rows,
                            float* C, int64_t ldc, float alpha, float beta, float* workspace,
                            int64_t workspace_floats, hipStream_t stream) {
  MPQ_CHECK_ARG(M >= 0 && N >= 0 && K >= 0, "mpq_gemm_f32: negative extent");
  if (M == 0 || N == 0) return mpq::kOk;
  MPQ_CHECK_ARG(A && B && C, "mpq_gemm_f32: null operand");
  MPQ_CHECK_ARG(lda >= K && ldc >= N, "mpq_gemm_f32: leading dimension too small");
  MPQ_CHECK_ARG(trans_b ? ldb >= K : ldb >= N, "mpq_gemm_f32: ldb too small");
  MPQ_CHECK_ARG(!(trans_b && b_rows), "mpq_gemm_f32: row gather needs trans_b = 0");
  MPQ_CHECK_ARG(M <= (int64_t)65535 * 128 && N <= (int64_t)0x7fffffff * 64,
                "mpq_gemm_f32: extent too large");
  MPQ_HIP_TRY(mpq::gemm(A, lda, B, ldb, trans_b != 0, b_rows, C, ldc, M, N, K, alpha, beta,
                        workspace, workspace_floats, stream));
  return mpq::kOk;
}

extern "C" int mpq_gemm_f32_split_count(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 1;
  int bn = 128;
  return mpq::choose_splits(M, N, K, (int64_t)1 << 62, &bn);
}

extern "C" int mpq_gemm_f32_splitk(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B,
                                   int64_t ldb, int trans_b, float* partials, int splits, hipStream_t stream) {
  MPQ_CHECK_ARG(M > 0 && N > 0 && K > 0, "mpq_gemm_f32_splitk: empty product");
  MPQ_CHECK_ARG(splits >= 1 && splits <= 32, "mpq_gemm_f32_splitk: splits must be in [1, 32]");
  MPQ_CHECK_ARG(A && B && partials, "mpq_gemm_f32_splitk: null operand");
  MPQ_CHECK_ARG(lda >= K && (trans_b ? ldb >= K : ldb >= N), "mpq_gemm_f32_splitk: leading dimension too small");
  MPQ_CHECK_ARG(M <= (int64_t)65535 * 128, "mpq_gemm_f32_splitk: M too large");
  int bn = 128;
  mpq::choose_splits(M, N, K, (int64_t)1 << 62, &bn);
  mpq::GemmParams p{};
  p.M = M; p.N = N; p.K = K;
  p.A = A; p.lda = lda; p.B = B; p.ldb = ldb; p.trans_b = trans_b != 0;
  p.C = partials; p.ldc = N; p.split_stride = M * N;
  p.alpha = 1.f; p.beta = 0.f; p.mode = mpq::kGemmPartials;
  MPQ_HIP_TRY(mpq::gemm_partials(p, splits, bn, stream));
  return mpq::kOk;
}

extern "C" int mpq_gemm_x6_pack_b(int64_t K, int64_t N, const float* B, int64_t ldb, int trans_b, float* packed,
                                  hipStream_t stream) {
  MPQ_CHECK_ARG(mpq::x6_shape_ok(N, K), "mpq_gemm_x6_pack_b: needs N %% 128 == 0 and K %% 32 == 0 (N=%lld K=%lld)",
                (long long)N, (long long)K);
  MPQ_CHECK_ARG(B && packed, "mpq_gemm_x6_pack_b: null operand");
  MPQ_CHECK_ARG(trans_b ? ldb >= K : ldb >= N, "mpq_gemm_x6_pack_b: ldb too small");
  MPQ_HIP_TRY(mpq::x6_pack_b(B, ldb, trans_b != 0, K, N, packed, stream));
  return mpq::kOk;
}

extern "C" int64_t mpq_gemm_x6_workspace_size(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || !mpq::x6_shape_ok(N, K)) return 0;
  const int splits = mpq::x6_choose_splits(M, N, K);
  return (mpq::x6_packed_a_bytes(M, K) + 255) / 256 * 256 + (int64_t)splits * M * N * 4;
}

extern "C" int mpq_gemm_x6(int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, const float* B_packed,
                           float* C, int64_t ldc, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  MPQ_CHECK_ARG(M >= 0, "mpq_gemm_x6: negative M");
  if (M == 0) return mpq::kOk;
  MPQ_CHECK_ARG(mpq::x6_shape_ok(N, K), "mpq_gemm_x6: needs N %% 128 == 0 and K %% 32 == 0 (N=%lld K=%lld)",
                (long long)N, (long long)K);
  MPQ_CHECK_ARG(A && B_packed && C && workspace, "mpq_gemm_x6: null operand");
  MPQ_CHECK_ARG(lda >= K && ldc >= N, "mpq_gemm_x6: leading dimension too small");
  MPQ_CHECK_ARG((reinterpret_cast<uintptr_t>(workspace) & 255u) == 0, "mpq_gemm_x6: workspace must be 256-byte aligned");
  const int64_t need = mpq_gemm_x6_workspace_size(M, N, K);
  MPQ_CHECK_ARG(workspace_bytes >= need, "mpq_gemm_x6: workspace too small (%lld < %lld bytes)",
                (long long)workspace_bytes, (long long)need);
  const int splits = mpq::x6_choose_splits(M, N, K);
  char* ws = static_cast<char*>(workspace);
  float* P = reinterpret_cast<float*>(ws + (mpq::x6_packed_a_bytes(M, K) + 255) / 256 * 256);
  MPQ_HIP_TRY(mpq::x6_pack_a(A, lda, M, K, ws, stream));
  MPQ_HIP_TRY(mpq::x6_gemm_partials(ws, B_packed, M, N, K, P, N, M * N, splits, stream));
  MPQ_HIP_TRY(mpq::splitk_reduce(P, splits, M * N, M, N, C, ldc, 1.f, 0.f, stream));
  return mpq::kOk;
}

extern "C" int64_t mpq_rankspace_pack_floats(int64_t n) {
  return (n > 0 && mpq::x6_shape_ok(n, n)) ? 3 * n * n : 0;
}

extern "C" int mpq_rankspace_pack(int64_t n, const float* V, const float* Vs, float* packed, hipStream_t stream) {
  MPQ_CHECK_ARG(n > 0 && mpq::x6_shape_ok(n, n), "mpq_rankspace_pack: n must be a positive multiple of 128 (n=%lld)",
                (long long)n);
  MPQ_CHECK_ARG(V && Vs && packed, "mpq_rankspace_pack: null operand");
  MPQ_HIP_TRY(mpq::x6_pack_b(V, n, false, n, n, packed, stream));
  MPQ_HIP_TRY(mpq::x6_pack_b(V, n, true, n, n, packed + n * n, stream));
  MPQ_HIP_TRY(mpq::x6_pack_b(Vs, n, false, n, n, packed + 2 * n * n, stream));
  return mpq::kOk;
}

extern "C" int mpq_gemm_x6_split_count(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || !mpq::x6_shape_ok(N, K)) return 0;
  return mpq::x6_choose_splits(M, N, K);
}

extern "C" int64_t mpq_gemm_x6_packed_a_size(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0 || K % 32 != 0) return 0;
  return mpq::x6_packed_a_bytes(M, K);
}

extern "C" int mpq_gemm_x6_pack_a(int64_t M, int64_t K, const float* A, int64_t lda, void* packed, hipStream_t stream) {
  MPQ_CHECK_ARG(M > 0 && K > 0 && K % 32 == 0, "mpq_gemm_x6_pack_a: needs M > 0 and K %% 32 == 0");
  MPQ_CHECK_ARG(A && packed && lda >= K, "mpq_gemm_x6_pack_a: null operand or lda < K");
  MPQ_CHECK_ARG((reinterpret_cast<uintptr_t>(packed) & 15u) == 0, "mpq_gemm_x6_pack_a: packed must be 16-byte aligned");
  MPQ_HIP_TRY(mpq::x6_pack_a(A, lda, M, K, packed, stream));
  return mpq::kOk;
}

extern "C" int mpq_gemm_x6_splitk(int64_t M, int64_t N, int64_t K, const void* A_packed, const float* B_packed,
                                  float* partials, int splits, hipStream_t stream) {
  MPQ_CHECK_ARG(M > 0 && mpq::x6_shape_ok(N, K), "mpq_gemm_x6_splitk: needs M > 0, N %% 128 == 0, K %% 32 == 0");
  MPQ_CHECK_ARG(splits >= 1 && K % splits == 0 && (K / splits) % 32 == 0,
                "mpq_gemm_x6_splitk: K / splits must be a whole multiple of 32");
  MPQ_CHECK_ARG(A_packed && B_packed && partials, "mpq_gemm_x6_splitk: null operand");
  MPQ_HIP_TRY(mpq::x6_gemm_partials(A_packed, B_packed, M, N, K, partials, N, M * N, splits, stream));
  return mpq::kOk;
}
