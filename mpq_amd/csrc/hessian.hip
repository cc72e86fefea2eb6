// Per-linear Hessian accumulation H = beta H + alpha X^T X (gfx950).
//
// The step before the per-linear solve: GPTQModel's add_batch keeps H = 2/m sum_t x_t x_t^T
// (mpq/adapters/gptqmodel.py:39 states the convention) and QUIP#'s hooks accumulate
// H = sum_t x_t x_t^T plus the column sums mu for the mean correction
// (mpq/quip_generic.py:823-921, H / ct - mu mu^T).  Both are one symmetric rank-T update per
// batch of T activations X (T x n, fp32 or bf16).
//
// SYRK on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16, fp32 accumulation).  bf16 activations are
// their own plane, and every product of two bf16 values is exact in the fp32 accumulator.  fp32
// activations are split exactly into three bf16 planes (x6_split.h) and the six plane products of
// order >= 2^-16 |a||b| are kept, the accuracy of an fp32 product.  The accumulator is rounded once per
// 16 tokens, where v_mfma_f32_32x32x2_f32 rounds once per 2.
#include <hip/hip_bf16.h>

#include <type_traits>

#include "common.h"
#include "x6_split.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;

// H tile (TS x TS, on or above the diagonal) = beta H + alpha X^T X, mirrored to the transposed tile,
// so H stays exactly symmetric.  Four waves of TS/2 x TS/2.
//
// Both operands are column panels of X (token-major), but an MFMA operand wants 8 consecutive tokens
// of one column per lane.  A thread loads R tokens x 4 columns, transposes them in registers and writes
// one 2R-byte piece per column to LDS: [plane][8-token group][slot], 16 bytes per slot, with column m at
// slot (m % 4) * TS/4 + m / 4, so a wave's writes and its fragment reads are both contiguous.  Two LDS
// buffers, D slabs of loads in flight in registers, one barrier per slab.
//
// Bound: bf16, the LDS fragment reads (1 KB per MFMA and wave with 64 x 64 wave tiles: the LDS rate);
// fp32, the matrix cores (six products per fragment pair).  4096 columns x 16384 tokens
// bf16: 4780 -> 523 us (525 TFLOP/s of n^2 T); 14336 x 8192 bf16: 18.9 -> 2.57 ms (656 TFLOP/s); 2048 x 3001
// fp32: 228 -> 140 us, all against one fp32 MFMA kernel for either type (repeated calls on one input).
template <bool kBf16, int TS>
__global__ __launch_bounds__(kThreads, 2) void syrk_kernel(const void* __restrict__ X, int64_t T, int64_t n,
                                                        int64_t ldx, float alpha, float beta,
                                                        float* __restrict__ H, int64_t ldh) {
  constexpr int NP = kBf16 ? 1 : 3;
  constexpr int NQ = TS / 4;                    // column quads of a tile
  constexpr int R = kBf16 && TS == 128 ? 8 : 4;  // tokens per thread and slab
  constexpr int KS = R * 128 / NQ;              // tokens per slab: 32 (16: fp32, TS = 128)
  constexpr int NB = TS / 64;                   // 32 x 32 blocks per wave and dimension
  constexpr int D = !kBf16 && TS == 128 ? 2 : 4;  // slabs of loads in flight (even)
  union Lds {
    uint4 op[2][2][NP][KS / 8][TS];
    float out[TS / NB][TS];
  };
  __shared__ Lds lds;
  auto& As = lds.op[0];
  auto& Bs = lds.op[1];

  // upper-triangular tile index -> (ti, tj), ti <= tj: tj (tj + 1) / 2 tiles precede column tj
  const int t = (int)blockIdx.x;
  int tj = (int)((sqrtf(8.f * (float)t + 1.f) - 1.f) * 0.5f);
  while ((tj + 1) * (tj + 2) / 2 <= t) ++tj;
  while (tj * (tj + 1) / 2 > t) --tj;
  const int ti = t - tj * (tj + 1) / 2;
  const int64_t m0 = (int64_t)ti * TS, n0 = (int64_t)tj * TS;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int op = tid >> 7, c = (tid & 127) % NQ, kg = (tid & 127) / NQ;
  typedef typename std::conditional<kBf16, uint2, float4>::type Quad;  // four columns of one token
  const char* mine = static_cast<const char*>(X) + (kg * R * ldx + (op ? n0 : m0) + 4 * c) * (kBf16 ? 2 : 4);
  const int64_t nslab = (T + KS - 1) / KS;

  Quad r[D][R];
  auto gload = [&](int64_t s, int set) {
    const int64_t left = T - s * KS - kg * R;  // tokens from this thread's first one on
#pragma unroll
    for (int e = 0; e < R; ++e) {
      r[set][e] = Quad{};
      if (e < left) r[set][e] = *reinterpret_cast<const Quad*>(mine + (s * KS + e) * ldx * (kBf16 ? 2 : 4));
    }
  };
  auto put = [&](int buf, int pl, int j, const uint32_t (&w)[R / 2]) {
    uint4* slot = op ? &Bs[buf][pl][kg * R / 8][j * NQ + c] : &As[buf][pl][kg * R / 8][j * NQ + c];
    if constexpr (R == 8)
      *slot = make_uint4(w[0], w[1], w[2], w[3]);
    else
      reinterpret_cast<uint2*>(slot)[kg & 1] = make_uint2(w[0], w[1]);
  };
  auto lstore = [&](int set, int buf) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t w[NP][R / 2];
#pragma unroll
      for (int d = 0; d < R / 2; ++d) {
        if constexpr (kBf16) {
          const uint2 p = r[set][2 * d], q = r[set][2 * d + 1];
          const uint32_t lo = j < 2 ? p.x : p.y, hi = j < 2 ? q.x : q.y;
          w[0][d] = __builtin_amdgcn_perm(hi, lo, j & 1 ? 0x07060302u : 0x05040100u);
        } else {
          const float4 a = r[set][2 * d], b = r[set][2 * d + 1];
          const float x = j == 0 ? a.x : j == 1 ? a.y : j == 2 ? a.z : a.w;
          const float y = j == 0 ? b.x : j == 1 ? b.y : j == 2 ? b.z : b.w;
          mpq::split3(x, y, w[0][d], w[1][d], w[2][d]);
        }
      }
#pragma unroll
      for (int pl = 0; pl < NP; ++pl) put(buf, pl, j, w[pl]);
    }
  };

  // the small plane products have accumulators of their own: every sum into the large one costs half an
  // ulp of it whatever is added (one accumulator for all six: relative error 3.0e-6 instead of 6.5e-7 at
  // 4096 x 16384; fp32 MFMA 2.0e-6)
  floatx16 acc[NB][NB], low[NP == 3 ? NB : 1][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.f;
        if constexpr (NP == 3) low[i][j][v] = 0.f;
      }
  const int sm = (wave >> 1) * (TS / 2) + (lane & 31), sn = (wave & 1) * (TS / 2) + (lane & 31);
  auto compute = [&](int buf) {
#pragma unroll
    for (int k = 0; k < KS / 16; ++k) {
      bf16x8 a[NP][NB], b[NP][NB];
#pragma unroll
      for (int pl = 0; pl < NP; ++pl)
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          a[pl][i] = __builtin_bit_cast(bf16x8, As[buf][pl][2 * k + (lane >> 5)][sm + 32 * i]);
          b[pl][i] = __builtin_bit_cast(bf16x8, Bs[buf][pl][2 * k + (lane >> 5)][sn + 32 * i]);
        }
      if constexpr (NP == 3) {  // smallest terms first
        constexpr int pa[5] = {2, 1, 0, 1, 0};
        constexpr int pb[5] = {0, 1, 2, 0, 1};
#pragma unroll
        for (int q = 0; q < 5; ++q)
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[q]][i], b[pb[q]][j], low[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0][i], b[0][j], acc[i][j], 0, 0, 0);
    }
  };

  // Slab s is in LDS buffer s & 1, slabs s + 1 .. s + D - 1 are in flight in the register sets s % D.
  // Rounds of D slabs with no exit inside; the slabs past the last token load nothing and multiply zeros.
  // The barrier waits for this wave's LDS accesses only: __syncthreads would also wait for the loads in
  // flight.
  auto barrier = []() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
#pragma unroll
  for (int u = 0; u < D; ++u) gload(u, u);
  lstore(0, 0);
  barrier();
  for (int64_t s0 = 0; s0 < nslab; s0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      gload(s0 + u + D, u);
      compute(u & 1);
      lstore((u + 1) % D, (u + 1) & 1);
      barrier();
    }
  }

  // slot s of an operand is column 4 (s % NQ) + s / NQ of its panel
  auto col_of = [](int s) { return 4 * (s % NQ) + s / NQ; };
  if constexpr (!kBf16) {
    bool redo = false;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          acc[i][j][v] += low[i][j][v];
          redo |= isnan(acc[i][j][v]);
        }
    // The planes of an infinity (or of a value that rounds to one in bf16) are not finite.  A wave with such a
    // sum forms its block again as fp32 products, two tokens at a time from L2, and takes its NaN entries from
    // there, so they overflow as fp32 products do.  (4096 columns x 4096 tokens, every activation infinite:
    // 150 ms with one serial dot product per entry, 2.6 with this, 0.6 for finite ones.)
    if (__any(redo)) {
      const float* xm = static_cast<const float*>(X) + m0;
      const float* xn = static_cast<const float*>(X) + n0;
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) low[i][j][v] = 0.f;
#pragma unroll 4
      for (int64_t tk = lane >> 5; tk - (lane >> 5) < T; tk += 2) {
        float a[NB], b[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          a[i] = tk < T ? xm[tk * ldx + col_of(sm + 32 * i)] : 0.f;
          b[i] = tk < T ? xn[tk * ldx + col_of(sn + 32 * i)] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            low[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], low[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (isnan(acc[i][j][v])) acc[i][j][v] = low[i][j][v];
    }
  }

  // Elements on or above the diagonal are written to (m, n) and (n, m), by way of LDS so that both are
  // written along rows of H: straight from the accumulators they went out 16 bytes and, for (n, m), four rows
  // apart (16 tokens, both with 128 x 128 tiles: 4096 bf16 88 -> 57 us, 8192 fp32 248 -> 161).  Chunk i holds the
  // tile's rows NB lr + i; entry (lr, cn) is kept at column (cn + lr) % TS, so reads along either index spread over
  // the banks.
  constexpr int kBatch = 8;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if (i) __syncthreads();
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int cn = col_of(sn + 32 * j);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int lr = col_of((wave >> 1) * (TS / 2) + 32 * i + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3)) / NB;
        lds.out[lr][(cn + lr) % TS] = alpha * acc[i][j][v];
      }
    }
    __syncthreads();
    for (int q0 = tid; q0 < TS / NB * TS; q0 += kBatch * kThreads) {
      float old[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int q = q0 + u * kThreads, lr = q / TS, cn = q % TS;
        const int64_t gm = m0 + NB * lr + i, gn = n0 + cn;
        old[u] = beta != 0.f && gn >= gm ? H[gm * ldh + gn] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int q = q0 + u * kThreads, lr = q / TS, cn = q % TS;
        const int64_t gm = m0 + NB * lr + i, gn = n0 + cn;
        if (gn < gm) continue;
        float val = lds.out[lr][(cn + lr) % TS];
        if (beta != 0.f) lds.out[lr][(cn + lr) % TS] = val = val + beta * old[u];
        H[gm * ldh + gn] = val;
      }
    }
    __syncthreads();
#pragma unroll 8
    for (int q = tid; q < TS / NB * TS; q += kThreads) {
      const int cn = q / (TS / NB), lr = q % (TS / NB);
      const int64_t gm = m0 + NB * lr + i, gn = n0 + cn;
      if (gn > gm) H[gn * ldh + gm] = lds.out[lr][(cn + lr) % TS];
    }
  }
}

// colsum[j] += sum_t X[t][j], in a fixed order: a work-group owns 16 columns, thread (g, j) adds the
// tokens g, g + 64, ... of column j, and the 64 sums of a column are added pairwise in LDS.  One work-group
// per 16 columns with 64 token streams keeps enough loads in flight (2048 columns x 3001 tokens fp32:
// 10 us; one thread per column took 691 us, a chain of 3001 loads in 8 work-groups).
template <bool kBf16>
__global__ __launch_bounds__(1024) void colsum_kernel(const void* __restrict__ X, int64_t T, int64_t n, int64_t ldx,
                                                      float* __restrict__ colsum) {
  __shared__ float red[64][17];
  const int j = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int64_t col = (int64_t)blockIdx.x * 16 + j;  // n % 128 == 0: every column exists
  float acc = 0.f;
#pragma unroll 4
  for (int64_t t = g; t < T; t += 64) {
    if constexpr (kBf16) {
      acc += __bfloat162float(static_cast<const __hip_bfloat16*>(X)[t * ldx + col]);
    } else {
      acc += static_cast<const float*>(X)[t * ldx + col];
    }
  }
  red[g][j] = acc;
  __syncthreads();
  for (int w = 32; w > 0; w >>= 1) {
    if (g < w) red[g][j] += red[g + w][j];
    __syncthreads();
  }
  if (g == 0) colsum[col] += red[0][j];
}

template <bool kBf16>
void launch(const void* X, int64_t T, int64_t n, int64_t ldx, float alpha, float beta, float* H, int64_t ldh,
            float* colsum, hipStream_t stream) {
  // 128 x 128 tiles read half as much LDS per product, but well below one tile per CU the chip idles:
  // there 64 x 64 tiles (four times as many).  8192 tokens, 128 / 64 tiles, us: n = 1024 bf16 171 / 113,
  // fp32 482 / 208; 2304 (171 tiles) 175 / 153, 488 / 395; 2432 (190) 172 / 148, 478 / 396; 2560 (210) 176 / 173,
  // 475 / 521; 2816 (253) 169 / 176, 481 / 532; 4096 286 / 361, 1105 / 1099; 8192 913 / 1322, 3453 / 4145.
  // Up to 256 tokens the time is that of reading and writing H, and smaller tiles spread it over more
  // work-groups: 32 tokens, 128 / 64 tiles, us: 2560 bf16 43 / 30, fp32 43 / 39; 4096 55 / 42, 71 / 57; 8192
  // 133 / 100, 158 / 153; 256 tokens: 2560 47 / 34, 56 / 51; 3584 53 / 45, 66 / 67; 8192 166 / 130, 242 / 226.  At
  // 512 tokens 3584 59 / 52, 86 / 92; 8192 184 / 161, 331 / 352.
  const int64_t nt = n / 128, tiles = nt * (nt + 1) / 2;
  if (tiles >= 200 && T > 256) {
    hipLaunchKernelGGL((syrk_kernel<kBf16, 128>), dim3((unsigned)tiles), dim3(kThreads), 0, stream, X, T, n, ldx,
                       alpha, beta, H, ldh);
  } else {
    hipLaunchKernelGGL((syrk_kernel<kBf16, 64>), dim3((unsigned)(nt * (2 * nt + 1))), dim3(kThreads), 0, stream, X, T,
                       n, ldx, alpha, beta, H, ldh);
  }
  if (colsum)
    hipLaunchKernelGGL(colsum_kernel<kBf16>, dim3((unsigned)(n / 16)), dim3(1024), 0, stream, X, T, n, ldx, colsum);
}

}  // namespace

extern "C" int mpq_hessian_accumulate(const void* X, int x_bf16, int64_t T, int64_t n, int64_t ldx, float alpha,
                                      float beta, float* H, int64_t ldh, float* colsum, hipStream_t stream) {
  using namespace mpq;
  MPQ_CHECK_ARG(T >= 0 && n > 0, "mpq_hessian_accumulate: bad shape");
  MPQ_CHECK_ARG(H && (X || T == 0), "mpq_hessian_accumulate: null pointer");
  MPQ_CHECK_ARG(n % 128 == 0, "mpq_hessian_accumulate: n must be a multiple of 128; got %lld", (long long)n);
  MPQ_CHECK_ARG(ldx >= n && ldx % 4 == 0 && ldh >= n, "mpq_hessian_accumulate: bad leading dimension");
  MPQ_CHECK_ARG(T == 0 || (reinterpret_cast<uintptr_t>(X) & (x_bf16 ? 7u : 15u)) == 0,
                "mpq_hessian_accumulate: X must be 16-byte (fp32) / 8-byte (bf16) aligned");
  MPQ_CHECK_ARG(n / 64 <= 65535, "mpq_hessian_accumulate: n too large");
  if (x_bf16) launch<true>(X, T, n, ldx, alpha, beta, H, ldh, colsum, stream);
  else launch<false>(X, T, n, ldx, alpha, beta, H, ldh, colsum, stream);
  MPQ_LAUNCH_CHECK();
  return kOk;
}
