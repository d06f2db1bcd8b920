// C = A W^T for any M, N, K, in true 32-bit arithmetic: the matrix product of
// the float32 path, and the fallback of the bfloat16 path for shapes its fast
// kernels refuse (operands are widened to float, exactly).  A is [M, K], W is
// [N, K], both row-major in T.
//
// Every output element sums its K products in an order that K alone decides,
// so a token's result does not depend on what else is in the batch.
//
//   gemm_f32_kernel      float32 with rows of whole, aligned float4s: the 32-bit
//                        matrix instructions (fused multiply-adds of full
//                        precision, twice the rate of the vector unit's)
//   gemm_generic_kernel  everything else: one fused multiply-add at a time, in
//                        ascending k
#include "common.h"
#include "tinyinfer_kernels.h"

TI_ERROR_API

#define GT 64   // tile of C: GT x GT
#define GK 16   // depth of one LDS stage

template <typename T, int EPI>
__global__ void __launch_bounds__(256)
gemm_generic_kernel(const T* __restrict__ A, const T* __restrict__ W, void* __restrict__ out_,
                    int M, int N, int K, long lda) {
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  __shared__ float As[GK][GT + 4];
  __shared__ float Ws[GK][GT + 4];
  __shared__ float Us[SW ? GK : 1][GT + 4];   // the up rows, for SwiGLU
  const int m0 = blockIdx.y * GT, n0 = blockIdx.x * GT;
  const int tid = threadIdx.x;
  const int ty = tid / 16, tx = tid % 16;
  const int lrow = tid / 4, lk = (tid % 4) * 4;
  float acc[4][4] = {};
  float accu[SW ? 4 : 1][4] = {};
  for (int k0 = 0; k0 < K; k0 += GK) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      const int am = m0 + lrow, wn = n0 + lrow;
      As[lk + j][lrow] = (am < M && k < K) ? ld<T>(A + (size_t)am * lda + k) : 0.f;
      Ws[lk + j][lrow] = (wn < N && k < K) ? ld<T>(W + (size_t)wn * K + k) : 0.f;
      if (SW) Us[lk + j][lrow] = (wn < N && k < K) ? ld<T>(W + (size_t)(wn + N) * K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
      if (SW) {
        float u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j] = Us[kk][tx * 4 + j];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) accu[i][j] = fmaf(a[i], u[j], accu[i][j]);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      const size_t o = (size_t)m * N + n;
      if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = acc[i][j];
      if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] += acc[i][j];
      if (TI_EPI_ACT(EPI)) st<T>((T*)out_ + o, epi_act<EPI>(acc[i][j]));
      if (EPI == TI_EPI_SWIGLU) {
        const float g = acc[i][j];
        st<T>((T*)out_ + o, g / (1.0f + expf(-g)) * accu[SW ? i : 0][j]);
      }
    }
  }
}

template <typename T>
static int launch(const void* A, const void* W, void* out, int M, int N, int K, long lda, int epi,
                  hipStream_t stream) {
  dim3 grid((N + GT - 1) / GT, (M + GT - 1) / GT);
  switch (epi) {
    case TI_EPI_STORE_F32:
      gemm_generic_kernel<T, TI_EPI_STORE_F32><<<grid, 256, 0, stream>>>((const T*)A, (const T*)W, out, M, N, K, lda);
      break;
    case TI_EPI_ADD_F32:
      gemm_generic_kernel<T, TI_EPI_ADD_F32><<<grid, 256, 0, stream>>>((const T*)A, (const T*)W, out, M, N, K, lda);
      break;
    case TI_EPI_STORE_ACT:
      gemm_generic_kernel<T, TI_EPI_STORE_ACT><<<grid, 256, 0, stream>>>((const T*)A, (const T*)W, out, M, N, K, lda);
      break;
    case TI_EPI_SWIGLU:
      gemm_generic_kernel<T, TI_EPI_SWIGLU><<<grid, 256, 0, stream>>>((const T*)A, (const T*)W, out, M, N, K, lda);
      break;
    case TI_EPI_RELU2:
      gemm_generic_kernel<T, TI_EPI_RELU2><<<grid, 256, 0, stream>>>((const T*)A, (const T*)W, out, M, N, K, lda);
      break;
    default:
      ti_set_error("gemm_generic: unknown epilogue %d", epi);
      return 1;
  }
  return 0;
}

// ------------------------------------------------------------------------------------------------ float32, matrix cores
// A workgroup of eight wavefronts owns 16 RB weight rows x 16 NB tokens and cuts K into eight runs of whole 16s (the
// same runs whatever M, N and the tile are), one a wavefront.  A wavefront walks its run in steps of 16: each lane
// loads four consecutive k of one weight row and of one token straight from memory, and four v_mfma_f32_16x16x4_f32
// take one of the four each (both operands are permuted alike, so every k meets itself).  The runs' sums meet in LDS
// and are added in ascending order.
//
// Few tokens: the weights' bytes bound it, each is read once, and eight runs keep eight wavefronts loading per tile.
// Many: a 16x16x4 lasts 32 cycles, so 32-bit products are bound by the matrix cores' 157 TFLOP/s long before L1 or
// LDS; operands need no staging, and what counts is that the tiles fill whole rounds of the compute units.
// Measured inside a prompt of 300 tokens of Qwen3-0.6B's sizes, us (the generic kernel): 4096 x 1024 37.1 (157), [gate; up]
// 6144 x 1024 47.8 (273), 1024 x 2048 and 1024 x 3072 29.4 on average (294), 151936 x 1024 1,055 (2,984); its products
// together 5.1 ms (31.5).
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf4;
#define GF_RUNS 8

template <int RB, int NB, bool SW>
__global__ void __launch_bounds__(64 * GF_RUNS)
gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ out, int M, int N, int K,
                long lda, int run, int m_tiles, int n_tiles, int epi, int wide_out) {
  constexpr int PL = SW ? 2 : 1;                    // planes of weight rows: gate and up
  constexpr int TR = 16 * RB, TM = 16 * NB;
  constexpr int LD = TR + 4;                        // floats between tokens of a tile in LDS
  __shared__ __attribute__((aligned(16))) float s_tile[GF_RUNS][PL][TM][LD];
  // the dies take workgroups in turn: a die gets all token tiles of a set of weight rows, one after the other, so
  // that the rows come from memory once
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int nt = m_tiles == 1 ? (int)blockIdx.x : (local / m_tiles) * 8 + die;
  const int mt = m_tiles == 1 ? 0 : local % m_tiles;
  if (nt >= n_tiles) return;
  const int n0 = nt * TR, m0 = mt * TM;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;

  // rows past the end repeat the last one; their sums are not stored
  const float* wp[PL][RB];
  const float* ap[NB];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r) wp[p][r] = W + (size_t)(min(n0 + r * 16 + r16, N - 1) + p * N) * K + quad * 4;
#pragma unroll
  for (int b = 0; b < NB; ++b) ap[b] = A + (size_t)min(m0 + b * 16 + r16, M - 1) * lda + quad * 4;

  gf4 acc[PL][RB][NB];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[p][r][b] = gf4{0.f, 0.f, 0.f, 0.f};

  struct Step { gf4 w[PL][RB], a[NB]; };
  auto load = [&](Step& s, int k) {
#pragma unroll
    for (int p = 0; p < PL; ++p)
#pragma unroll
      for (int r = 0; r < RB; ++r) s.w[p][r] = *reinterpret_cast<const gf4*>(wp[p][r] + k);
#pragma unroll
    for (int b = 0; b < NB; ++b) s.a[b] = *reinterpret_cast<const gf4*>(ap[b] + k);
  };
  auto multiply = [&](const Step& s) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int p = 0; p < PL; ++p)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            acc[p][r][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(s.w[p][r][j], s.a[b][j], acc[p][r][b], 0, 0, 0);
  };
  const int k0 = wave * run, k1 = min(K, k0 + run);
  const int steps = k1 > k0 ? (k1 - k0) / 16 : 0;   // whole steps; K's last 4, 8 or 12 are a step of their own
  // loads run DEPTH steps ahead; past the run's end they repeat its last step
  constexpr int DEPTH = (PL * RB + NB <= 3) ? 8 : (PL * RB + NB <= 6) ? 4 : 2;
  if (steps > 0) {
    Step s[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(s[d], k0 + 16 * min(d, steps - 1));
    int i = 0;
    for (; i + DEPTH <= steps; i += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        multiply(s[d]);
        load(s[d], k0 + 16 * min(i + DEPTH + d, steps - 1));
        __builtin_amdgcn_sched_barrier(0);          // the loads leave here, not where the next product needs them
      }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (i + d < steps) multiply(s[d]);
  }
  if (k1 > k0 && (k1 - k0) % 16) {
    const int k = k0 + steps * 16;
    Step s;
    if (k + quad * 4 < K) {                         // K is a multiple of 4: a lane's four are there or not
      load(s, k);
    } else {
#pragma unroll
      for (int p = 0; p < PL; ++p)
#pragma unroll
        for (int r = 0; r < RB; ++r) s.w[p][r] = gf4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NB; ++b) s.a[b] = gf4{0.f, 0.f, 0.f, 0.f};
    }
    multiply(s);
  }
  // a lane holds four weight rows of one token
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b)
        *reinterpret_cast<gf4*>(&s_tile[wave][p][b * 16 + r16][r * 16 + quad * 4]) = acc[p][r][b];
  __syncthreads();
  const int runs = (K + run - 1) / run;
  for (int e = threadIdx.x; e < TM * (TR / 4); e += 64 * GF_RUNS) {
    const int t = e / (TR / 4), c = (e % (TR / 4)) * 4;
    const int m = m0 + t, n = n0 + c;
    if (m >= M || n >= N) continue;
    gf4 v = *reinterpret_cast<const gf4*>(&s_tile[0][0][t][c]);
    for (int w = 1; w < runs; ++w) v += *reinterpret_cast<const gf4*>(&s_tile[w][0][t][c]);
    if (SW) {
      gf4 u = *reinterpret_cast<const gf4*>(&s_tile[0][PL - 1][t][c]);
      for (int w = 1; w < runs; ++w) u += *reinterpret_cast<const gf4*>(&s_tile[w][PL - 1][t][c]);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
    }
    if (epi == TI_EPI_RELU2) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = epi_act<TI_EPI_RELU2>(v[i]);
    }
    float* o = out + (size_t)m * N + n;
    if (wide_out) {
      if (epi == TI_EPI_ADD_F32) v += *reinterpret_cast<const gf4*>(o);
      *reinterpret_cast<gf4*>(o) = v;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N) o[i] = epi == TI_EPI_ADD_F32 ? o[i] + v[i] : v[i];
    }
  }
}

static int compute_units() {
  static int n = 0;
  if (!n) {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) n = prop.multiProcessorCount;
    if (n <= 0) n = 256;
  }
  return n;
}

// The tile: of those that are built, the one whose rounds of the compute units take the least time in all.  A round costs a
// start, its products (RB NB) and its operands' loads (RB + NB, four times a product's weight each: sixteen lines a load).
// Fitted to 1 to 1,000 rows times the weights of Qwen3-0.6B's sizes: the tile it picks is on average 0.9 % slower than the
// fastest (300 x 1024 x 3072: 32 x 48 35.7 us, 16 x 80 40.8).
static long f32_tile_cost(int rb, int nb, bool sw, int M, int N, int units) {
  const long tiles = (long)((M + 16 * nb - 1) / (16 * nb)) * ((N + 16 * rb - 1) / (16 * rb));
  const int pl = sw ? 2 : 1;
  const long rounds = (tiles + units - 1) / units;
  return rounds * (2 + pl * rb * nb + 4 * (pl * rb + nb));
}

static int launch_f32(const float* A, const float* W, float* out, int M, int N, int K, long lda, int epi, hipStream_t stream) {
  static const int TILES[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 2}, {2, 3}, {2, 4}, {2, 5}, {4, 2}, {4, 4}};
  const bool sw = epi == TI_EPI_SWIGLU;
  int rb = 1, nb = 1;
  long best = -1;
  for (const auto& t : TILES) {
    if (sw && t[0] * t[1] > 8) continue;           // two planes of it would not fit in LDS
    const long cost = f32_tile_cost(t[0], t[1], sw, M, N, compute_units());
    if (best < 0 || cost < best) {
      best = cost;
      rb = t[0];
      nb = t[1];
    }
  }
  const int wide_out = N % 4 == 0 && ((uintptr_t)out & 15) == 0;
  const int run = ((K + GF_RUNS - 1) / GF_RUNS + 15) / 16 * 16;
  const int m_tiles = (M + 16 * nb - 1) / (16 * nb), n_tiles = (N + 16 * rb - 1) / (16 * rb);
  const long grid = m_tiles == 1 ? n_tiles : (long)((n_tiles + 7) / 8) * 8 * m_tiles;
#define GF_CASE(R, B)                                                                                                     \
  if (rb == R && nb == B) {                                                                                               \
    if (sw) {                                                                                                             \
      if constexpr (R * B <= 8)                                                                                          \
        gemm_f32_kernel<R, B, true><<<(unsigned)grid, 64 * GF_RUNS, 0, stream>>>(A, W, out, M, N, K, lda, run, m_tiles, n_tiles, epi, wide_out); \
    } else {                                                                                                              \
      gemm_f32_kernel<R, B, false><<<(unsigned)grid, 64 * GF_RUNS, 0, stream>>>(A, W, out, M, N, K, lda, run, m_tiles, n_tiles, epi, wide_out); \
    }                                                                                                                     \
    return 0;                                                                                                             \
  }
  GF_CASE(1, 1) GF_CASE(1, 2) GF_CASE(1, 3) GF_CASE(1, 4) GF_CASE(1, 5) GF_CASE(2, 2) GF_CASE(2, 3) GF_CASE(2, 4) GF_CASE(2, 5)
  GF_CASE(4, 2) GF_CASE(4, 4)
#undef GF_CASE
  return 1;
}

// N is the number of output columns (for SwiGLU: F, with W holding 2F rows).
extern "C" int ti_gemm_generic(int dtype, const void* A, const void* W, void* out, int M, int N, int K,
                               long lda, int epi, hipStream_t stream) {
  TI_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm_generic: bad sizes M=%d N=%d K=%d lda=%ld", M, N, K, lda);
  TI_REQUIRE((M + GT - 1) / GT <= 65535, "gemm_generic: M=%d too large for one launch", M);
  if (M == 0) return 0;
  int rc;
  // rows of whole float4s on 16-byte boundaries (what K, lda and the addresses say, never M: a token's sum keeps its order)
  const bool f4 = dtype == TI_F32 && K % 4 == 0 && lda % 4 == 0 &&
                  (((uintptr_t)A | (uintptr_t)W) & 15) == 0;
  if (f4 && epi >= TI_EPI_STORE_F32 && epi <= TI_EPI_RELU2 && epi != TI_EPI_QKV_PREP)
    rc = launch_f32((const float*)A, (const float*)W, (float*)out, M, N, K, lda, epi, stream);
  else if (dtype == TI_F32)
    rc = launch<float>(A, W, out, M, N, K, lda, epi, stream);
  else if (dtype == TI_BF16)
    rc = launch<bf16_t>(A, W, out, M, N, K, lda, epi, stream);
  else {
    ti_set_error("gemm_generic: unknown dtype %d", dtype);
    return 1;
  }
  if (rc) return rc;
  TI_LAUNCH_CHECK();
  return 0;
}
