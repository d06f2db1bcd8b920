// C = A W^T for any M, N, K, to the precision of 32-bit arithmetic: the matrix product of
// the float32 path, and the fallback of the bfloat16 path for shapes its fast
// kernels refuse (operands are widened to float, exactly).  A is [M, K], W is
// [N, K], both row-major in T.
//
// Every output element sums its K products in an order that K alone decides,
// so a token's result does not depend on what else is in the batch.
//
//   gemm_f32_kernel      float32 with rows of whole, aligned float4s: matrix
//                        instructions on the floats cut into three bfloat16
//   gemm_f32_shared_kernel  the same bits, cut once a workgroup: many tiles
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
// A float is the sum of three bfloat16 (8 + 8 + 8 bits: the nearest, the nearest to what is left, and the rest, without a remainder; the
// method of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations",
// ARITH 2019), so a product of floats is nine products of bfloat16, which v_mfma_f32_16x16x32_bf16 multiplies exactly and adds in 32 bits.
// Six of them are taken; the three left out are at most 2^-24 of the product together.  The leading pieces' products have a sum of their
// own, and the five others, each at most 2^-8 of them, one that is added at the end: what the matrix unit cuts off there is below the
// leading sum's last place, so a single product comes out rounded once.  Six of these take 96 cycles where the 32-bit instructions take 256.
// Operands are multiplied by 2^16 first, so that subnormal floats too have three pieces, and sums divided by 2^32.
// Error against 64 bits, 2-norm over 2-norm, with N(0, 1) tokens and N(0, 0.02) weights (by 32-bit instructions): K = 8 2.8e-8 (5.4e-8), 36
// 4.6e-8 (8.0e-8), 1024 8.6e-8 (2.1e-7), 3072 1.2e-7 (3.6e-7), 12288 2.4e-7 (7.0e-7); tokens of 1e-36 and of 1e-39 the same; one
// element that is not zero 2.6e-8 (2.5e-8), at most 8.8e-8 of a product.  (All in one sum, with the second piece cut and no factors: 1024
// 1.6e-7, one element 3.8e-8 and at most 2.0e-7, tokens of 1e-36 5e-5 and of 1e-39 3e-2; eight products make one element's error
// 2.5e-8 and calls of 300 rows 10 % longer.)
// The matrix unit cuts what it adds downwards, which leaves every sum too low: small, but the same way in every layer.  The odd runs
// therefore take the tokens' negatives and their sums are subtracted: the mean error is then 1e-11.
// What the three pieces cannot hold (infinite, not a number, above 2^111, sums above 2^95) leaves a sum that is not finite; such an element
// is computed again by fused multiply-adds.
//
// A wavefront's rows come through its own part of LDS by direct loads (staged_rows.h; loaded as operands straight into registers they were
// all that bounded these products).  What bounds them now is the splitting (52 instructions a block of 16 rows
// and step beside 16 cycles each of six matrix instructions a pair of blocks), and for 1,024 columns the ends: the first loads and the
// sums' way through LDS are a third of the 15 us.
// us a call, by 32-bit instructions with operands straight from memory, and now: 300 rows x 4096 x 1024 35.6 -> 26.2, [gate; up]
// 6144 x 1024 46.7 -> 33.4, 1024 x 2048 23.8 -> 15.2, 1024 x 3072 32.7 -> 21.4, 151936 x 1024 1,043 -> 832; 53 rows 12.7 -> 8.7,
// 17.8 -> 12.5, 16.2 -> 10.2 (1024 x 3072); one row 6.5 -> 5.1, 9.6 -> 7.1, 10.8 -> 9.6, 172 -> 132.  (In one sum 26.1, 32.4, 13.9, 20.2, 762.)
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float gf4;
#define GF_RUNS 8
#define GF_STEP 32
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 gbf8;

// Eight floats, times `factor`, as three bfloat16 each, the sum of which they are: the nearest, the nearest to what is left, and the rest.
struct Planes {
  gbf8 p[3];
};
#define GF_SCALE 65536.f         // 2^16: multiples of 2^-149 become multiples of 2^-133, the last place of a bfloat16
__device__ __forceinline__ Planes split_planes(const gf4& x, const gf4& y, float factor) {
  uint32_t u[3][4];
  float r[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[i] = x[i] * factor;
    r[4 + i] = y[i] * factor;
  }
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u[j][i] = pack_bf16x2(r[2 * i], r[2 * i + 1]);
      if (j < 2) {
        r[2 * i] -= __uint_as_float(u[j][i] << 16);
        r[2 * i + 1] -= __uint_as_float(u[j][i] & 0xffff0000u);
      }
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

// Four neighbouring results of one token, from the sums of all runs to `o`: what is not finite is computed again, SwiGLU, the store.
template <bool SW>
__device__ __forceinline__ void f32_finish(gf4 v, gf4 u, const float* __restrict__ a, const float* __restrict__ W, float* __restrict__ o,
                                           int n, int N, int K, int run, int epi, int wide_out) {
  const auto settle = [&](gf4& x, size_t row0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (fabsf(x[i]) <= FLT_MAX) x[i] *= 1.f / (GF_SCALE * GF_SCALE);
      else if (n + i < N) x[i] = dot_by_fma(a, W + (row0 + n + i) * K, K, run);
  };
  settle(v, 0);
  if (SW) {
    settle(u, N);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.0f + expf(-v[i])) * u[i];
  }
  if (epi == TI_EPI_RELU2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = epi_act<TI_EPI_RELU2>(v[i]);
  }
  if (wide_out) {
    if (epi == TI_EPI_ADD_F32) v += *reinterpret_cast<const gf4*>(o);
    *reinterpret_cast<gf4*>(o) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) o[i] = epi == TI_EPI_ADD_F32 ? o[i] + v[i] : v[i];
  }
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

  gf4 acc[PL][RB][NB], fine[PL][RB][NB];           // the leading products, the others
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[p][r][b] = fine[p][r][b] = gf4{0.f, 0.f, 0.f, 0.f};

  const float turned = wave & 1 ? -GF_SCALE : GF_SCALE;
  // one step's products: blocks of weight rows (gate, then up), then blocks of tokens; the pieces of the fewer are kept
  const auto multiply = [&](const Eight* e) {
    constexpr int NW = PL * RB, KEEP = NW <= NB ? NW : NB, TURN = NW <= NB ? NB : NW;
    const auto split = [&](int block) { return split_planes(e[block].x, e[block].y, block < NW ? GF_SCALE : turned); };
    Planes kept[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) kept[i] = split(NW <= NB ? i : NW + i);
#pragma unroll
    for (int t = 0; t < TURN; ++t) {
      const Planes one = split(NW <= NB ? NW + t : t);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        constexpr int WJ[6] = {2, 0, 1, 1, 0, 0}, AJ[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int i = 0; i < KEEP; ++i) {
          const int r = NW <= NB ? i : t, b = NW <= NB ? t : i;
          gf4& sum = j < 5 ? fine[r / RB][r % RB][b] : acc[r / RB][r % RB][b];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16((NW <= NB ? kept[i] : one).p[WJ[j]], (NW <= NB ? one : kept[i]).p[AJ[j]], sum, 0, 0, 0);
        }
      }
    }
  };
  const int k0 = wave * run, k1 = min(K, k0 + run);
  const int steps = k1 > k0 ? (k1 - k0) / GF_STEP : 0;   // whole steps; what is left of K is a step of its own
  if (steps > 0) {
    // Rows past the end repeat the last one; their sums are not stored.
    unsigned voff[BLOCKS][2];
    const int lr = lane >> 3, piece = piece_of((lane & 7) ^ lr);
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
    const unsigned at = (unsigned)(size_t)mine + r16 * 128, x = at + ((quad ^ (r16 & 7)) << 4), y = at + (((quad + 4) ^ (r16 & 7)) << 4);
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
        *reinterpret_cast<gf4*>(&s_tile[wave][p][b * 16 + r16][r * 16 + quad * 4]) = acc[p][r][b] + fine[p][r][b];
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
    gf4 u = v;
    if (SW) {
      u = *reinterpret_cast<const gf4*>(&s_tile[0][PL - 1][t][c]);
      for (int w = 1; w < runs; ++w) {
        const gf4 x = *reinterpret_cast<const gf4*>(&s_tile[w][PL - 1][t][c]);
        u = w & 1 ? u - x : u + x;
      }
    }
    f32_finish<SW>(v, u, A + (size_t)m * lda, W, out + (size_t)m * N + n, n, N, K, run, epi, wide_out);
  }
#endif
}

// ---------------------------------------------------------------------------------- float32, more tokens: shared splits
// In gemm_f32_kernel every wavefront splits what it multiplies, 52 vector instructions a block, twice the time of its matrix instructions.
// Here WR x WT wavefronts own a tile together, each RB blocks of weight rows (SwiGLU: of gates and of their ups) x NB of tokens: a
// k-step's floats come into registers eight lanes to a row's 128 bytes, are split once for the workgroup and go as pieces into one of
// two stages of LDS, in the order in which a matrix instruction takes them.  While one stage is multiplied the next is split, and the
// loads of the two after that are out; a step has one barrier.  A wavefront alone on its SIMD issues a vector instruction every 8
// cycles, two one every 4.7: two workgroups of four wavefronts to a unit, or eight wavefronts.
// The runs of K are those of gemm_f32_kernel, one after the other in the same wavefront, each with sums of its own that are
// added to (or subtracted from) the total at its end: the same bits, whichever kernel takes a product.
// Piece (k / 8, row) of a block's plane lies in place (k / 8) * 16 + (row ^ 2 (k / 8)).  A wavefront's read of a plane takes 1.8 ns a unit so, as
// in a row, and its write of 512 bytes 3.0; exchanged by 4 (k / 8) 3.5 and 3.4, not exchanged 1.9 and 6.8.
// What bounds it: vector and matrix instructions of a step hardly overlap (tiles of 64 x 128, two to a unit: 1.83 us a step of both, of which
// matrix instructions alone take 0.7 and vector instructions 0.8; in which order they stand changes nothing).
// us a call, there and here: 300 rows x 151936 x 1024 868 -> 680, [gate; up] 6144 x 1024 37.4 -> 31.7; 64 rows x 151936 x 1024 208 -> 178;
// 1,000 rows x 4096 x 1024 79 -> 62, x 151936 x 1024 2,490 -> 2,080.
template <int WR, int WT, int RB, int NB, bool SW> struct F32Shared {
  static constexpr int WAVES = WR * WT, PL = SW ? 2 : 1, ROWS = WR * RB, TOKENS = WT * NB;      // blocks of 16: weight rows of a plane, tokens
  static constexpr int BLOCKS = PL * ROWS + TOKENS, LOADS = 2 * BLOCKS / WAVES;      // half blocks of 8 rows a wavefront asks for
  static constexpr int STAGE = BLOCKS * 3072, LDS = 2 * STAGE;
  static_assert(ROWS % (WAVES / 2) == 0 && TOKENS % (WAVES / 2) == 0, "a load of all wavefronts is rows of one kind");
};

// Four floats, times `factor`, as three bfloat16 each: split_planes for half an operand.
struct HalfPlanes {
  uint2 p[3];
};
__device__ __forceinline__ HalfPlanes split_half(const gf4& x, float factor) {
  HalfPlanes s;
  float r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = x[i] * factor;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    s.p[j] = make_uint2(pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3]));
    if (j < 2) {
      r[0] -= __uint_as_float(s.p[j].x << 16);
      r[1] -= __uint_as_float(s.p[j].x & 0xffff0000u);
      r[2] -= __uint_as_float(s.p[j].y << 16);
      r[3] -= __uint_as_float(s.p[j].y & 0xffff0000u);
    }
  }
  return s;
}

template <int WR, int WT, int RB, int NB, bool SW>
__global__ void __launch_bounds__(64 * WR * WT, 2)
gemm_f32_shared_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ out, int M, int N, int K,
                       long lda, int run, int m_tiles, int n_tiles, int epi, int wide_out) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  using T = F32Shared<WR, WT, RB, NB, SW>;
  constexpr int WAVES = T::WAVES, PL = T::PL, ROWS = T::ROWS, LOADS = T::LOADS, STAGE = T::STAGE;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;      // (as in gemm_f32_kernel)
  const int nt = m_tiles == 1 ? (int)blockIdx.x : (local / m_tiles) * 8 + die;
  const int mt = m_tiles == 1 ? 0 : local % m_tiles;
  if (nt >= n_tiles) return;
  const int n0 = nt * 16 * ROWS, m0 = mt * 16 * T::TOKENS;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;
  const int wr = wave % WR, wt = wave / WR;                      // this wavefront's part of the rows, of the tokens

  // what this wavefront brings: half blocks WAVES i + wave.  Rows past the end repeat the last one; their sums are not stored.
  unsigned voff[LOADS], put[LOADS];
  const int lr = lane >> 3, c = lane & 7;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int hb = WAVES * i + wave, block = hb >> 1, row8 = (hb & 1) * 8 + lr;
    const bool tokens = block >= PL * ROWS;
    const int row = (tokens ? block - PL * ROWS : block % ROWS) * 16 + row8;
    voff[i] = (tokens ? (unsigned)min(row, M - 1 - m0) * (unsigned)(lda * 4) : (unsigned)min(row, N - 1 - n0) * (unsigned)(K * 4)) + c * 16;
    put[i] = block * 3072 + (c >> 1) * 256 + (row8 ^ ((c >> 1) * 2)) * 16 + (c & 1) * 8;
  }
  const auto rows_at = [](const float* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
  const auto rsW = rows_at(W + (size_t)n0 * K), rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K), rsA = rows_at(A + (size_t)m0 * lda);
  const auto load = [&](gf4* g, int step) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const auto& rs = WAVES / 2 * i >= PL * ROWS ? rsA : WAVES / 2 * i >= ROWS ? rsU : rsW;
      g[i] = __builtin_bit_cast(gf4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff[i], step * GF_STEP * 4, 0));
    }
  };
  const auto split = [&](const gf4* g, unsigned stage, float turned) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const HalfPlanes h = split_half(g[i], WAVES / 2 * i >= PL * ROWS ? turned : GF_SCALE);
#pragma unroll
      for (int j = 0; j < 3; ++j) *reinterpret_cast<uint2*>(smem + stage + put[i] + j * 1024) = h.p[j];
    }
  };

  gf4 acc[PL][RB][NB], fine[PL][RB][NB], total[PL][RB][NB];       // the leading products, the others, the runs before
#pragma unroll
  for (int p = 0; p < PL; ++p)
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[p][r][b] = fine[p][r][b] = total[p][r][b] = gf4{0.f, 0.f, 0.f, 0.f};
  const unsigned read_at = quad * 256 + (r16 ^ (quad * 2)) * 16;
  struct Pieces {
    gbf8 w[PL][RB][3], t[NB][3];
  };
  const auto read = [&](Pieces& f, unsigned stage) {
    const auto piece = [&](int block, int j) { return *reinterpret_cast<const gbf8*>(smem + stage + read_at + block * 3072 + j * 1024); };
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
      for (int b = 0; b < NB; ++b) f.t[b][j] = piece(PL * ROWS + wt * NB + b, j);
#pragma unroll
      for (int p = 0; p < PL; ++p)
#pragma unroll
        for (int r = 0; r < RB; ++r) f.w[p][r][j] = piece(p * ROWS + wr * RB + r, j);
    }
  };
  const auto multiply = [&](const Pieces& f) {
    constexpr int WJ[6] = {2, 0, 1, 1, 0, 0}, AJ[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int j = 0; j < 6; ++j)
#pragma unroll
      for (int p = 0; p < PL; ++p)
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
          for (int b = 0; b < NB; ++b) {
            gf4& sum = j < 5 ? fine[p][r][b] : acc[p][r][b];
            sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[p][r][WJ[j]], f.t[b][AJ[j]], sum, 0, 0, 0);
          }
  };
  const int steps = K / GF_STEP, run_steps = run / GF_STEP, end = steps - 1;
  int left = run_steps, split_left = run_steps;                   // steps of the run that is multiplied, of the run that is split
  float sign = 1.f, turned = GF_SCALE;
  const auto split_next = [&](const gf4* g, unsigned stage) {
    split(g, stage, turned);
    if (--split_left == 0) split_left = run_steps, turned = -turned;
  };
  const auto end_of_run = [&]() {
#pragma unroll
    for (int p = 0; p < PL; ++p)
#pragma unroll
      for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
          for (int i = 0; i < 4; ++i) total[p][r][b][i] = fmaf(acc[p][r][b][i] + fine[p][r][b][i], sign, total[p][r][b][i]);
          acc[p][r][b] = fine[p][r][b] = gf4{0.f, 0.f, 0.f, 0.f};
        }
    left = run_steps;
    sign = -sign;
  };
  // One step: `g`, the step behind it, is split into the other stage and asked for anew two steps further on.  (Past the end the last step is
  // loaded and split again, into a stage that nothing multiplies.)
  Pieces pieces;
  const auto step = [&](int s, gf4* g, unsigned stage) {
    __syncthreads();
    read(pieces, stage);
    __builtin_amdgcn_sched_barrier(0);
    split_next(g, STAGE - stage);
    load(g, min(s + 3, end));
    multiply(pieces);
    __builtin_amdgcn_sched_barrier(0);
    if (--left == 0 || s == end) end_of_run();
  };
  gf4 g0[LOADS], g1[LOADS];                                       // steps of even and of odd number
  load(g0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load(g1, min(1, end));
  __builtin_amdgcn_sched_barrier(0);
  split_next(g0, 0);
  load(g0, min(2, end));
  __builtin_amdgcn_sched_barrier(0);
  int s = 0;
  for (; s + 2 <= steps; s += 2) {
    step(s, g1, 0);
    step(s + 1, g0, STAGE);
  }
  if (s < steps) step(s, g1, 0);

  // a lane holds four weight rows of one token
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int m = m0 + (wt * NB + b) * 16 + r16;
    if (m >= M) continue;
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      const int n = n0 + (wr * RB + r) * 16 + quad * 4;
      if (n >= N) continue;
      f32_finish<SW>(total[0][r][b], total[PL - 1][r][b], A + (size_t)m * lda, W, out + (size_t)m * N + n, n, N, K, run, epi, wide_out);
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

template <int WR, int WT, int RB, int NB, bool SW>
static int launch_f32_shared(const float* A, const float* W, float* out, int M, int N, int K, long lda, int run, int epi, int wide_out,
                             hipStream_t stream) {
  using T = F32Shared<WR, WT, RB, NB, SW>;
  static const hipError_t room = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_shared_kernel<WR, WT, RB, NB, SW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS);
  TI_REQUIRE(room == hipSuccess, "gemm_generic: %d bytes of LDS: %s", T::LDS, hipGetErrorString(room));
  const int m_tiles = (M + 16 * T::TOKENS - 1) / (16 * T::TOKENS), n_tiles = (N + 16 * T::ROWS - 1) / (16 * T::ROWS);
  const long grid = m_tiles == 1 ? n_tiles : (long)((n_tiles + 7) / 8) * 8 * m_tiles;
  gemm_f32_shared_kernel<WR, WT, RB, NB, SW><<<(unsigned)grid, 64 * T::WAVES, T::LDS, stream>>>(A, W, out, M, N, K, lda, run, m_tiles, n_tiles, epi, wide_out);
  return 0;
}

// The tile: of those that are built, the one whose rounds of the compute units take the least time in all.  A round costs a
// start, its products (RB NB) and its operands (RB + NB blocks to split, four times a product's weight each).
// Fitted to 1 to 1,000 rows times the weights of Qwen3-0.6B's sizes: the tile it picks is on average 0.9 % slower than the
// fastest (300 x 1024 x 3072: 32 x 48 20.2 us, 16 x 80 22.4), and 0.3 % over those and the 1.7B to 4B sizes with the present kernel.
// dies = 8: by the rounds of the die that has the most columns of tiles.
static long f32_tile_cost(int rb, int nb, bool sw, int M, int N, int units, int dies = 1) {
  const long columns = (N + 16 * rb - 1) / (16 * rb), tiles = (long)((M + 16 * nb - 1) / (16 * nb)) * ((columns + dies - 1) / dies);
  const int pl = sw ? 2 : 1;
  units = (units + dies - 1) / dies;
  const long rounds = (tiles + units - 1) / units;
  return rounds * (2 + pl * rb * nb + 4 * (pl * rb + nb));
}

// Whether the tiles with shared splits take it, 64 tokens x 128 weight rows (SwiGLU: 64 gates and their ups).  The dies take columns of tiles in turn, so
// what counts is the rounds of the die that has the most.  A unit holds two workgroups of the former (four wavefronts of 242 registers): a round is 4 us
// and 1.55 a k-step of both, 1.05 where there is one each.  Of the latter (eight wavefronts of 145) it holds one: 2.5 us and 0.86 a k-step a round.
// The other kernel's cost, counted so, is worth 0.075 us and 0.256 a thousand of K (95 of 100 within 13 %).  Over 307 products, thirteen weights under 40
// to 3,000 rows and 60 of random sizes, what this chooses is on average 0.13 % slower than the faster of the two, at worst 9 % (rounds of all units at one
// rate, a tenth in favour of the other: 1.1 and 52 %).
// us, the other and this: 64 rows of 151936 x 1024 214 172, 300 790 654; [gate; up] 6144 x 1024 under 200 rows 30.4 31.0, 256 34.6 29.9, 512 51 58, 1,000
// 104 90, 9728 x 896 under 600 92 102, 384 64 52, 19456 x 2560 under 64 79 67, 512 365 342; 4096 x 1024 under 512 37.1 38.5, 1,000 73 60, 2,000 153 114;
// 6144 x 4096 under 300 108 135, 2,048 699 665.
static bool f32_shared_serves(int rb, int nb, bool sw, int M, int N, int K, long lda) {
  // whole k-steps, and a tile's rows within what a buffer's descriptor spans
  if (K % GF_STEP || K >= (1 << 20) || lda >= (1 << 20)) return false;
  const long columns = (N + (sw ? 63 : 127)) / (sw ? 64 : 128), tiles = (long)((M + 63) / 64) * ((columns + 7) / 8), units = (compute_units() + 7) / 8;      // of a die
  const double steps = K / GF_STEP;
  double us = 1.0;
  if (sw) us += (double)((tiles + units - 1) / units) * (2.5 + 0.86 * steps);
  else {
    const long rest = tiles % (2 * units);
    us += (double)(tiles / (2 * units) + (rest > units)) * (4.0 + 1.55 * steps) + (rest > 0 && rest <= units ? 4.0 + 1.05 * steps : 0.0);
  }
  return us < 2.7 + f32_tile_cost(rb, nb, sw, M, N, compute_units(), 8) * (0.075 + 0.256 * K / 1024);
}

// the tile of gemm_f32_kernel that costs the least
static void f32_best_tile(bool sw, int M, int N, int& rb, int& nb) {
  static const int TILES[][2] = {{1, 1}, {1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 2}, {2, 3}, {2, 4}, {2, 5}, {4, 2}, {4, 4}};
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
}

// What is chosen, for tests: 1: the tiles with shared splits.
extern "C" int ti_gemm_generic_f32_choice(int swiglu, int M, int N, int K, long lda) {
  int rb, nb;
  f32_best_tile(swiglu != 0, M, N, rb, nb);
  return f32_shared_serves(rb, nb, swiglu != 0, M, N, K, lda) ? 1 : 0;
}

static int launch_f32(const float* A, const float* W, float* out, int M, int N, int K, long lda, int epi, hipStream_t stream) {
  const bool sw = epi == TI_EPI_SWIGLU;
  int rb, nb;
  f32_best_tile(sw, M, N, rb, nb);
  const int wide_out = N % 4 == 0 && ((uintptr_t)out & 15) == 0;
  const int run = ((K + GF_RUNS - 1) / GF_RUNS + GF_STEP - 1) / GF_STEP * GF_STEP;
  if (f32_shared_serves(rb, nb, sw, M, N, K, lda))
    return sw ? launch_f32_shared<4, 2, 1, 2, true>(A, W, out, M, N, K, lda, run, epi, wide_out, stream)
              : launch_f32_shared<2, 2, 4, 2, false>(A, W, out, M, N, K, lda, run, epi, wide_out, stream);
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
