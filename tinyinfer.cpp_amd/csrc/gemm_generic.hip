// C = A W^T for any M, N, K, in true 32-bit arithmetic: the matrix product of
// the float32 path, and the fallback of the bfloat16 path for shapes its fast
// kernels refuse (operands are widened to float, exactly).  A is [M, K], W is
// [N, K], both row-major in T.
//
// Every output element sums its K products in an order that K alone decides,
// so a token's result does not depend on what else is in the batch.
//
//   gemm_f32_kernel      float32 with rows of whole, aligned float4s: matrix
//                        instructions on the floats cut into three bfloat16
//   gemm_generic_kernel  everything else: one fused multiply-add at a time, in
//                        ascending k
#include <float.h>
#include <type_traits>
#include "common.h"
#include "tinyinfer_kernels.h"
#include "staged_rows.h"

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
// A workgroup of eight wavefronts owns 16 RB weight rows x 16 NB tokens and cuts K into eight runs of whole 32s (the
// same runs whatever M, N and the tile are), one a wavefront.  The runs' sums meet in LDS and are added in ascending order.
//
// A float is the sum of three bfloat16 (8 + 8 + 8 bits: the nearest, what is left cut to eight bits, and the rest, without a remainder),
// so a product of floats is nine products of bfloat16, which v_mfma_f32_16x16x32_bf16 multiplies exactly and adds in 32 bits.  Six of them
// are taken, the smallest first; the three left out are below 2^-22 of the product, where each addition already rounds at 2^-24 of the
// sum, and 32 products share a rounding in place of one each.  Six of these take 96 cycles where the 32-bit instructions take 256.  Error
// against 64 bits, 2-norm over 2-norm, with N(0, 1) tokens and N(0, 0.02) weights (by 32-bit instructions): K = 1024 1.6e-7 (2.1e-7),
// 3072 3.0e-7 (3.6e-7), 12288 6.4e-7 (7.1e-7), 36 4.7e-8 (8.0e-8).
// The matrix unit cuts what it adds downwards, which leaves every sum too low by some 5e-8 of the outputs' size: small, but the same way
// in every layer (a prompt's logits 9.2e-7 off, by 32-bit instructions 8.1e-7).  The odd runs therefore take the tokens' negatives
// and their sums are subtracted: the mean error is then 1e-9.
// What the three pieces cannot hold (infinite, not a number, above the largest bfloat16) leaves a sum that is not finite; such an element
// is computed again by fused multiply-adds.  (Below 2^-110 the last piece may lie below the normal numbers, 2^-133 at least.)
//
// A wavefront's rows come through its own part of LDS by direct loads (staged_rows.h; loaded as operands straight into registers they were
// all that bounded these products).  What bounds them now is the splitting (52 instructions a block of 16 rows
// and step beside 16 cycles each of six matrix instructions a pair of blocks), and for 1,024 columns the ends: the first loads and the
// sums' way through LDS are a third of the 13 us.
// us a call, before (32-bit instructions, operands straight from memory) and now: 300 rows x 4096 x 1024 36.9 -> 25.7, [gate; up]
// 6144 x 1024 47.9 -> 31.9, 1024 x 2048 24.3 -> 13.3, 1024 x 3072 33.6 -> 19.5, 151936 x 1024 1,040 -> 697; 53 rows 14.0 -> 9.2,
// 20.6 -> 12.6, 13.1 -> 7.7, 16.9 -> 10.2, 242 -> 186; one row 8.4 -> 6.9, 12.7 -> 9.3, 11.5 -> 9.0 (1024 x 3072), 171 -> 127.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf4;
#define GF_RUNS 8
#define GF_STEP 32
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 gbf8;

// Eight floats, times `sign` (1 or -1), as three bfloat16 each, the sum of which they are: the nearest, and twice the upper half of what
// is left.
struct Planes {
  gbf8 p[3];
};
__device__ __forceinline__ Planes split_planes(const gf4& x, const gf4& y, float sign) {
  const uint32_t flip = __float_as_uint(sign) & 0x80000000u;
  uint32_t u[3][4];
  float r[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[i] = x[i];
    r[4 + i] = y[i];
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      h[i] = j == 0 ? (__float_as_uint(r[i]) ^ flip) + 0x8000u : __float_as_uint(r[i]);
      if (j == 0) r[i] = fmaf(r[i], sign, -__uint_as_float(h[i] & 0xffff0000u));
      if (j == 1) r[i] -= __uint_as_float(h[i] & 0xffff0000u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) u[j][i] = __builtin_amdgcn_perm(h[2 * i + 1], h[2 * i], 0x07060302u);
  }
  Planes s;
#pragma unroll
  for (int j = 0; j < 3; ++j) s.p[j] = __builtin_bit_cast(gbf8, make_uint4(u[j][0], u[j][1], u[j][2], u[j][3]));
  return s;
}

// One element by fused multiply-adds, in the same runs: where the three pieces do not hold an operand.
__device__ __forceinline__ float dot_by_fma(const float* __restrict__ a, const float* __restrict__ w, int K, int run) {
  float total = 0.f;
  for (int k0 = 0; k0 < K; k0 += run) {
    float s = 0.f;
    for (int k = k0; k < min(K, k0 + run); ++k) s = fmaf(a[k], w[k], s);
    total = k0 ? total + s : s;
  }
  return total;
}

struct Eight { gf4 x, y; };      // eight consecutive k of one row

template <int RB, int NB, bool SW> struct F32Tile {
  static constexpr int PL = SW ? 2 : 1;               // planes of weight rows: gate and up
  static constexpr int TR = 16 * RB, TM = 16 * NB;
  static constexpr int LD = TR + 4;                   // floats between tokens of a tile in LDS
  static constexpr int BLOCKS = PL * RB + NB;         // of 16 rows: what a step of a wavefront reads
  static constexpr int STEP_BYTES = BLOCKS * 2048;
  static constexpr int STAGES = BLOCKS <= 2 ? 4 : BLOCKS <= 3 ? 3 : BLOCKS <= 4 ? 2 : 1;
  static constexpr int SUMS = GF_RUNS * PL * TM * LD * 4, STAGED = GF_RUNS * STAGES * STEP_BYTES;
  static constexpr int LDS = SUMS > STAGED ? SUMS : STAGED;
};

template <int RB, int NB, bool SW>
__global__ void __launch_bounds__(64 * GF_RUNS)
gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ out, int M, int N, int K,
                long lda, int run, int m_tiles, int n_tiles, int epi, int wide_out) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  using T = F32Tile<RB, NB, SW>;
  constexpr int PL = T::PL, TR = T::TR, TM = T::TM, LD = T::LD, BLOCKS = T::BLOCKS, STAGES = T::STAGES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float (*s_tile)[PL][TM][LD] = reinterpret_cast<float (*)[PL][TM][LD]>(smem);
  // the dies take workgroups in turn: a die gets all token tiles of a set of weight rows, one after the other, so
  // that the rows come from memory once
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int nt = m_tiles == 1 ? (int)blockIdx.x : (local / m_tiles) * 8 + die;
  const int mt = m_tiles == 1 ? 0 : local % m_tiles;
  if (nt >= n_tiles) return;
  const int n0 = nt * TR, m0 = mt * TM;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;

  gf4 acc[PL][RB][NB];
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[p][r][b] = gf4{0.f, 0.f, 0.f, 0.f};

  const float sign = wave & 1 ? -1.f : 1.f;
  // one step's products: blocks of weight rows (gate, then up), then blocks of tokens
  const auto multiply = [&](const Eight* e) {
    Planes w[PL * RB];
#pragma unroll
    for (int r = 0; r < PL * RB; ++r) w[r] = split_planes(e[r].x, e[r].y, 1.f);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const Planes a = split_planes(e[PL * RB + b].x, e[PL * RB + b].y, sign);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        constexpr int WJ[6] = {2, 0, 1, 1, 0, 0}, AJ[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int r = 0; r < PL * RB; ++r)
          acc[r / RB][r % RB][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[r].p[WJ[j]], a.p[AJ[j]], acc[r / RB][r % RB][b], 0, 0, 0);
      }
    }
  };
  const int k0 = wave * run, k1 = min(K, k0 + run);
  const int steps = k1 > k0 ? (k1 - k0) / GF_STEP : 0;   // whole steps; what is left of K is a step of its own
  if (steps > 0) {
    // Rows past the end repeat the last one; their sums are not stored.
    unsigned voff[BLOCKS][2];
    const int lr = lane >> 3, piece = (lane & 7) ^ lr;
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        voff[i][h] = (i < PL * RB ? (unsigned)min((i % RB) * 16 + h * 8 + lr, N - 1 - n0) * (unsigned)(K * 4)
                                  : (unsigned)min((i - PL * RB) * 16 + h * 8 + lr, M - 1 - m0) * (unsigned)(lda * 4)) + piece * 16;
    const auto rows_at = [](const float* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
    const auto rsW = rows_at(W + (size_t)n0 * K + k0), rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K + k0);
    const auto rsA = rows_at(A + (size_t)m0 * lda + k0);
    unsigned char* mine = smem + wave * STAGES * T::STEP_BYTES;
    const auto load = [&](int step, unsigned stage) {
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto* dst = (__attribute__((address_space(3))) void*)(mine + stage + i * 2048 + h * 1024);      // the same in every lane
          if (i < RB) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, dst, 16, voff[i][h], step * GF_STEP * 4, 0, 0);
          else if (i < PL * RB) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsU, dst, 16, voff[i][h], step * GF_STEP * 4, 0, 0);
          else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, dst, 16, voff[i][h], step * GF_STEP * 4, 0, 0);
        }
    };
    const unsigned at = (unsigned)(size_t)mine + r16 * 128, x = at + (((2 * quad) ^ (r16 & 7)) << 4), y = at + (((2 * quad + 1) ^ (r16 & 7)) << 4);
    staged_steps<BLOCKS, STAGES, Eight>(steps, x, y, load, multiply);
  }
  if (k1 > k0 && (k1 - k0) % GF_STEP) {
    const int k = k0 + steps * GF_STEP + quad * 8;
    const auto part = [&](const float* p) {                // K is a multiple of 4: a lane's fours are there or not
      Eight e = {gf4{0.f, 0.f, 0.f, 0.f}, gf4{0.f, 0.f, 0.f, 0.f}};
      if (k < K) e.x = *reinterpret_cast<const gf4*>(p + k);
      if (k + 4 < K) e.y = *reinterpret_cast<const gf4*>(p + k + 4);
      return e;
    };
    Eight e[BLOCKS];
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
      e[i] = part(i < PL * RB ? W + (size_t)(min(n0 + (i % RB) * 16 + r16, N - 1) + (i / RB) * N) * K
                              : A + (size_t)min(m0 + (i - PL * RB) * 16 + r16, M - 1) * lda);
    multiply(e);
  }
  __syncthreads();                                         // the stages are free
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
    for (int w = 1; w < runs; ++w) {
      const gf4 x = *reinterpret_cast<const gf4*>(&s_tile[w][0][t][c]);
      v = w & 1 ? v - x : v + x;
    }
    const auto settle = [&](gf4& x, size_t row0) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(fabsf(x[i]) <= FLT_MAX) && n + i < N) x[i] = dot_by_fma(A + (size_t)m * lda, W + (row0 + n + i) * K, K, run);
    };
    settle(v, 0);
    if (SW) {
      gf4 u = *reinterpret_cast<const gf4*>(&s_tile[0][PL - 1][t][c]);
      for (int w = 1; w < runs; ++w) {
        const gf4 x = *reinterpret_cast<const gf4*>(&s_tile[w][PL - 1][t][c]);
        u = w & 1 ? u - x : u + x;
      }
      settle(u, N);
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
#endif
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
// start, its products (RB NB) and its operands (RB + NB blocks to split, four times a product's weight each).
// Fitted to 1 to 1,000 rows times the weights of Qwen3-0.6B's sizes: the tile it picks is on average 0.9 % slower than the
// fastest (300 x 1024 x 3072: 32 x 48 20.2 us, 16 x 80 22.4), and 0.3 % over those and the 1.7B to 4B sizes with the present kernel.
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
  const int run = ((K + GF_RUNS - 1) / GF_RUNS + GF_STEP - 1) / GF_STEP * GF_STEP;
  const int m_tiles = (M + 16 * nb - 1) / (16 * nb), n_tiles = (N + 16 * rb - 1) / (16 * rb);
  const long grid = m_tiles == 1 ? n_tiles : (long)((n_tiles + 7) / 8) * 8 * m_tiles;
#define GF_LAUNCH(R, B, S)                                                                                                \
  do {                                                                                                                    \
    constexpr int lds = F32Tile<R, B, S>::LDS;                                                                            \
    static const hipError_t room = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_kernel<R, B, S>),           \
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, lds);                  \
    TI_REQUIRE(room == hipSuccess, "gemm_generic: %d bytes of LDS: %s", lds, hipGetErrorString(room));                    \
    gemm_f32_kernel<R, B, S><<<(unsigned)grid, 64 * GF_RUNS, lds, stream>>>(A, W, out, M, N, K, lda, run, m_tiles, n_tiles, epi, wide_out); \
  } while (0)
#define GF_CASE(R, B)                                                                                                     \
  if (rb == R && nb == B) {                                                                                               \
    if (sw) {                                                                                                             \
      if constexpr (R * B <= 8) GF_LAUNCH(R, B, true);                                                                    \
    } else {                                                                                                              \
      GF_LAUNCH(R, B, false);                                                                                             \
    }                                                                                                                     \
    return 0;                                                                                                             \
  }
  GF_CASE(1, 1) GF_CASE(1, 2) GF_CASE(1, 3) GF_CASE(1, 4) GF_CASE(1, 5) GF_CASE(2, 2) GF_CASE(2, 3) GF_CASE(2, 4) GF_CASE(2, 5)
  GF_CASE(4, 2) GF_CASE(4, 4)
#undef GF_CASE
#undef GF_LAUNCH
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
  // (and a tile's rows within 2 GiB, which is what a buffer's descriptor spans)
  const bool f4 = dtype == TI_F32 && K % 4 == 0 && lda % 4 == 0 && lda < (1 << 22) &&
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
