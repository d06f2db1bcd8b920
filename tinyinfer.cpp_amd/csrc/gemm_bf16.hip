// bfloat16 matrix products C = A W^T on the matrix cores of gfx950, 32-bit
// accumulation.  A is [M, K] (row stride lda), W is [N, K], both bfloat16 with K
// contiguous, which is the natural operand layout of MFMA for both sides.
//
// Two kernels:
//  * skinny (M <= 64, decode and small portions): every weight element is read
//    from memory exactly once per call.  A workgroup of four wavefronts owns 16
//    weight rows; the wavefronts split K between them in interleaved 128-byte
//    pieces and reduce through LDS in a fixed order.  The weights are the "A"
//    operand of v_mfma_f32_16x16x32_bf16, the tokens are the 16 columns.
//  * tiled (M > 64, prefill): tiles of 64 x 64 to 256 x 256, k-tiles of 64 through two to
//    five stages of LDS, wavefronts' shares out of v_mfma_f32_32x32x16_bf16.  K that is
//    no multiple of 64: 128 x 128 x 32 through double-buffered LDS.
//
// Epilogues: store float, add into a float residual, store bfloat16, or SwiGLU
// over a stacked [gate; up] weight.  The reduction order of an output element
// never depends on M within one kernel.  (The reference's two products are
// src/cuda/gemm.cu:37-85 and 152-261; it reads the weights once
// per row of A for M <= 32.)
#include <algorithm>
#include <string>
#include <type_traits>
#include <utility>
#include "common.h"
#include "tinyinfer_kernels.h"
#include "tinyinfer_kernels_tuning.h"
#include "qk_prep.h"
#include "staged_rows.h"

TI_ERROR_API

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

typedef unsigned v4u __attribute__((ext_vector_type(4)));

union Frag {
  uint4 u;
  bf16x8 v;
};

__device__ __forceinline__ uint4 ld16(const bf16_t* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.0f + __expf(-g)) * u; }

// ============================================================== skinny kernel
// grid.x = ceil(N / 16) (SwiGLU: ceil(F / 8): 8 gate rows and their 8 up rows).
// NW wavefronts split K between them.
// UN: 64-element chunks of K a wavefront has in flight at a time.  All loads of a pass are
// issued before the first product: out-of-range pieces read a valid address (piece 0 of the
// row) and get a zeroed weight instead of a branch, so that nothing waits in between.
// STAGES > 0 (K of whole chunks; up to 16 tokens where staged_16_serves says so): the rows come through LDS (staged_rows.h), a chunk a step; the same sums in the
// same order.  G: groups of 16 weight rows a workgroup then takes (skinny_groups_for).  Every workgroup pulls in all token rows, which as operands from memory was most of its time.  us, before and now, at 17,
// 32, 48 and 64 rows: 4096 x 1024 4.3 4.9 5.9 6.9 -> 3.9 4.0 3.9 4.6; [gate; up] 6144 x 1024 6.7 7.8 9.8 10.0 -> 5.3 5.8 6.9 7.9 (the
// latter two were tiles; G = 2: 4.9 5.1 5.7 6.4); 4096 x 2048 8.7 9.3 10.9 11.9 -> 6.0 6.4 7.2 8.3; 12288 x 2048 16.1 17.0 17.8 18.4 -> 11.5 13.5 16.3 18.6.
struct RowPieces { v4u x, y; };
template <int MT, int EPI, int NW = 4, int UN = 4, int STAGES = 0, int G = 1>
__global__ void __launch_bounds__(NW * 64)
gemm_skinny_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_,
                   int M, int N, int K, long lda) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  constexpr int BLOCKS = MT + G, STAGED = STAGES * BLOCKS * 2048;      // a wavefront's stages, where its sums lie afterwards
  static_assert(STAGES == 0 || STAGED >= G * MT * 16 * 17 * 4, "a wavefront's sums fit into its stages");
  static_assert(G == 1 || STAGES > 0, "several groups of weight rows: through LDS");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  __shared__ float s_red[STAGES ? 1 : NW][MT][16][17];
  const auto red = [&](int w, int g, int t, int a, int b) -> float& {
    if constexpr (STAGES) return reinterpret_cast<float (*)[16][17]>(smem + w * STAGED)[g * MT + t][a][b];
    else return s_red[w][t][a][b];
  };
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, j = lane >> 4;   // MFMA row / column, and k group
  // the weight row this lane feeds
  int wrow;
  if (SW) {
    const int n = blockIdx.x * 8 + (r & 7);
    wrow = (r < 8 ? 0 : N) + (n < N ? n : N - 1);
  } else {
    const int n = blockIdx.x * 16 + r;
    wrow = n < N ? n : N - 1;
  }
  const bf16_t* wp = W + (size_t)wrow * K;
  const bf16_t* ap[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + r;
    ap[t] = A + (size_t)(m < M ? m : 0) * lda;   // columns beyond M are computed from row 0 and never stored
  }
  // the residual this thread will add to, asked for before the product
  const int tok = threadIdx.x >> 4, row = threadIdx.x & 15;
  float prev[G][MT];
  if (EPI == TI_EPI_ADD_F32) {   // threads without an output element read a valid one: no branch
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int m = t * 16 + (tok & 15), n = blockIdx.x * 16 * G + g * 16 + row;
        prev[g][t] = ((const float*)out_)[(size_t)(m < M ? m : 0) * N + (n < N ? n : N - 1)];
      }
  }
  floatx4 acc[G][MT];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[g][t] = floatx4{0.f, 0.f, 0.f, 0.f};

  const uint4 zero = make_uint4(0, 0, 0, 0);
  // chunk c covers k in [64 c, 64 c + 64); lane group j takes [64 c + 16 j, +16)
  const int chunks = (K + 63) / 64;
  if constexpr (STAGES > 0) {
    const int lr = lane >> 3, piece = piece_of((lane & 7) ^ lr) * 16;
    const int n0 = blockIdx.x * G * (SW ? 8 : 16);
    unsigned voff[BLOCKS][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int g = 0; g < G; ++g) voff[g][h] = (unsigned)min((SW ? 8 * g : 16 * g + 8 * h) + lr, N - 1 - n0) * (unsigned)(K * 2) + piece;
#pragma unroll
      for (int t = 0; t < MT; ++t) voff[G + t][h] = (unsigned)min(16 * t + 8 * h + lr, M - 1) * (unsigned)(lda * 2) + piece;
    }
    const auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
    const auto rsW = rows_at(W + (size_t)n0 * K + wave * 64), rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K + wave * 64);
    const auto rsA = rows_at(A + wave * 64);
    unsigned char* mine = smem + wave * STAGED;
    const auto load = [&](int step, unsigned stage) {
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto* dst = (__attribute__((address_space(3))) void*)(mine + stage + i * 2048 + h * 1024);      // the same in every lane
          if (i >= G) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, dst, 16, voff[i][h], step * NW * 128, 0, 0);
          else if (SW && h == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsU, dst, 16, voff[i][h], step * NW * 128, 0, 0);
          else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, dst, 16, voff[i][h], step * NW * 128, 0, 0);
        }
    };
    const unsigned at = (unsigned)(size_t)mine + r * 128;
    const int steps = wave < chunks ? (chunks - wave + NW - 1) / NW : 0;
    staged_steps<BLOCKS, STAGES, RowPieces>(steps, at + ((j ^ (r & 7)) << 4), at + (((j + 4) ^ (r & 7)) << 4), load,
                                            [&](const RowPieces* e) {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, e[g].x), __builtin_bit_cast(bf16x8, e[G + t].x), acc[g][t], 0, 0, 0);
          acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, e[g].y), __builtin_bit_cast(bf16x8, e[G + t].y), acc[g][t], 0, 0, 0);
        }
    });
  }
  if constexpr (STAGES == 0)
  for (int c0 = wave; c0 < chunks; c0 += NW * UN) {
    Frag w0[UN], w1[UN], a0[UN][MT], a1[UN][MT];
    bool ok0[UN], ok1[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int k = (c0 + NW * u) * 64 + j * 16;
      ok0[u] = k + 8 <= K;    // false too for chunks beyond the last
      ok1[u] = k + 16 <= K;
      w0[u].u = ld16(wp + (ok0[u] ? k : 0));
      w1[u].u = ld16(wp + (ok1[u] ? k + 8 : 0));
    }
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int k = (c0 + NW * u) * 64 + j * 16;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        a0[u][t].u = ld16(ap[t] + (ok0[u] ? k : 0));
        a1[u][t].u = ld16(ap[t] + (ok1[u] ? k + 8 : 0));
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // every load above is issued before the first product waits
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (!ok0[u]) w0[u].u = zero;
      if (!ok1[u]) w1[u].u = zero;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[u].v, a0[u][t].v, acc[0][t], 0, 0, 0);
        acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[u].v, a1[u][t].v, acc[0][t], 0, 0, 0);
      }
    }
  }
  // acc[g][t][i]: row 4 j + i of weight group g, token 16 t + r
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red(wave, g, t, r, 4 * j + i) = acc[g][t][i];
  __syncthreads();
  // thread -> (token = tid / 16, row = tid % 16): consecutive threads, consecutive columns
  if (NW > 4 && threadIdx.x >= 256) return;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = t * 16 + tok;
    if (m >= M) continue;
    if (SW) {
      static_assert(G <= 2, "a thread a column");
      if (row >= 8 * G) continue;
      const int n = blockIdx.x * 8 * G + row, at = G > 1 ? row >> 3 : 0;
      if (n >= N) continue;
      float g = 0.f, u = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        g += red(w, at, t, tok, row & 7);
        u += red(w, at, t, tok, (row & 7) + 8);
      }
      ((bf16_t*)out_)[(size_t)m * N + n] = f2bf(silu_mul(g, u));
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int n = blockIdx.x * 16 * G + g * 16 + row;
        if (n >= N) continue;
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += red(w, g, t, tok, row);
        const size_t o = (size_t)m * N + n;
        if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = s;
        if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev[g][t] + s;
        if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(s));
      }
    }
  }
#endif
}

// ================================== skinny kernel with the token rows in LDS
// A producer has `template <int NW> __device__ void fill(bf16_t* sA, int lda, int M, int K)`,
// called by all NW * 64 threads, writing sA[m * lda + k]; the kernel synchronizes after it.

// Rows that do exist in memory (bfloat16 [M, K], row stride lda): copied into LDS once per
// workgroup, 16 bytes per thread and load, instead of every wavefront fetching its token
// fragments from memory with one load instruction per fragment (for one token fifteen of
// sixteen lanes of such a load repeat a row): a compute unit takes a load instruction of 64
// lanes every 16 cycles or so, and the kernel for few tokens is bound by that.
struct CopyProducer {
  const bf16_t* A;
  long lda;
  template <int NW, class IssueWeights>
  __device__ __forceinline__ void fill(bf16_t* sA, int lds_stride, int M, int K, IssueWeights issue_weights) const {
    constexpr int NT = NW * 64, PB = 8;
    const int kp = K >> 3, pieces = M * kp;
    bool first = true;
    for (int p0 = threadIdx.x; first || p0 < pieces; p0 += NT * PB) {
      uint4 v[PB];
      int dst[PB];
      bool ok[PB];
#pragma unroll
      for (int b = 0; b < PB; ++b) {
        const int p = p0 + NT * b;
        ok[b] = p < pieces;
        const int pc = ok[b] ? p : 0;
        const int m = pc / kp, k8 = pc - m * kp;
        v[b] = ld16(A + (size_t)m * lda + k8 * 8);
        dst[b] = m * lds_stride + k8 * 8;
      }
      if (first) {
        __builtin_amdgcn_sched_barrier(0);
        issue_weights();
        __builtin_amdgcn_sched_barrier(0);
        first = false;
      }
#pragma unroll
      for (int b = 0; b < PB; ++b)
        if (ok[b]) *reinterpret_cast<uint4*>(sA + dst[b]) = v[b];
    }
  }
};

template <class Producer, int EPI, int NW, int UN = 4>
__global__ void __launch_bounds__(NW * 64)
gemm_skinny_staged_kernel(Producer producer, const bf16_t* __restrict__ W, void* __restrict__ out_, int M, int N,
                          int K) {
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
  bf16_t* sA = reinterpret_cast<bf16_t*>(dyn_smem);          // [M][K + 8]
  __shared__ float red[NW][16][17];
  const int lda = K + 8;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, j = lane >> 4;
  int wrow;
  if (SW) {
    const int n = blockIdx.x * 8 + (r & 7);
    wrow = (r < 8 ? 0 : N) + (n < N ? n : N - 1);
  } else {
    const int n = blockIdx.x * 16 + r;
    wrow = n < N ? n : N - 1;
  }
  const bf16_t* wp = W + (size_t)wrow * K + j * 16;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  const int chunks = K / 64;

  // the residual this thread will add to
  const int tok = threadIdx.x >> 4, row = threadIdx.x & 15;   // tok >= 16 for the wavefronts beyond four
  float prev = 0.f;
  if (EPI == TI_EPI_ADD_F32) {   // threads without an output element read a valid one: no branch
    const int n = blockIdx.x * 16 + row;
    prev = ((const float*)out_)[(size_t)(tok < M ? tok : 0) * N + (n < N ? n : N - 1)];
  }

  // the first weights of this wavefront: the producer asks for them right after its own first
  // loads, so that they are on their way while the rows are made.  A chunk beyond the last
  // reads chunk 0 and is zeroed afterwards: no branch between the loads.
  Frag w0[UN], w1[UN];
  auto issue_weights = [&]() {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int c = wave + NW * u < chunks ? wave + NW * u : 0;
      w0[u].u = ld16(wp + (size_t)c * 64);
      w1[u].u = ld16(wp + (size_t)c * 64 + 8);
    }
  };
  producer.template fill<NW>(sA, lda, M, K, issue_weights);
  __syncthreads();

  // ---- the product, as in the plain skinny kernel with the token fragments from LDS
  const bf16_t* ap = sA + (size_t)(r < M ? r : 0) * lda + j * 16;
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = wave; c0 < chunks; c0 += NW * UN) {
    if (c0 != wave) {
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        const int c = c0 + NW * u < chunks ? c0 + NW * u : 0;
        w0[u].u = ld16(wp + (size_t)c * 64);
        w1[u].u = ld16(wp + (size_t)c * 64 + 8);
      }
    }
    Frag a0[UN], a1[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int c = c0 + NW * u < chunks ? c0 + NW * u : 0;
      a0[u].u = ld16(ap + (size_t)c * 64);
      a1[u].u = ld16(ap + (size_t)c * 64 + 8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      if (c0 + NW * u >= chunks) w0[u].u = w1[u].u = zero;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[u].v, a0[u].v, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[u].v, a1[u].v, acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][r][4 * j + i] = acc[i];
  __syncthreads();
  if (tok >= M) return;
  if (SW) {
    if (row >= 8) return;
    const int n = blockIdx.x * 8 + row;
    if (n >= N) return;
    float gt = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      gt += red[w][tok][row];
      up += red[w][tok][row + 8];
    }
    ((bf16_t*)out_)[(size_t)tok * N + n] = f2bf(silu_mul(gt, up));
  } else {
    const int n = blockIdx.x * 16 + row;
    if (n >= N) return;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += red[w][tok][row];
    const size_t o = (size_t)tok * N + n;
    if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = sum;
    if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev + sum;
    if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(sum));
  }
}

// ================================== the norm inside the product
// out (op)= rmsnorm(X; Gw, eps) W^T for M <= 16.  Every workgroup norms all rows for itself into LDS (bfloat16, the bits of the norm's own
// kernel: lane l of a wavefront holds the float4 pieces l, l + 64, ... of a row) while its weights are on their way into LDS stages of each
// wavefront's own (staged_rows.h).  G groups of KW wavefronts, a tile of 16 weight rows (SwiGLU: 8 gate and 8 up rows) each, so that a unit
// norms the rows once for all tiles it has; KW wavefronts split K as the plain kernels do: the same bits as norm and product.
// KC: float4 pieces of a row a lane holds (K <= 256 KC).  ST: chunks of 64 columns a wavefront has under way.
// What bounds it: the chain of loads, norm and products of one launch, then the weights' bytes.  A load of 1 KiB keeps the unit that takes
// addresses for 16 cycles (64 for weights as operands), so rows are asked for only by the wavefronts that norm them, and nothing waits for
// more than it uses.  Weights as operands straight from memory, norm in front, in a chain of launches with weights from memory, us before
// and now at 1, 8 and 16 rows: 4096 x 1024 4.0 4.0 5.2 -> 3.2 3.5 4.7, [gate; up] 6144 x 1024 5.6 5.9 7.3 -> 4.2 4.7 5.3, 4096 x 2048 7.5 7.6
// 9.6 -> 5.3 6.7 8.2, [gate; up] 12288 x 2048 13.6 15.1 18.1 -> 11.7 12.8 16.6, 6144 x 2560 11.7 14.3 20.1 -> 7.4 9.3 11.3, 6144 x 4096
// at 1 and 8 14.0 16.5 -> 11.3 16.0 (the plain product alone, at 1 row: 3.2, 4.4, 5.6, 10.9, 7.4, 11.3).
template <int KC, int EPI, int KW, int G, int ST>
__global__ void __launch_bounds__(64 * KW * G)
gemm_normed_kernel(const float* __restrict__ X, const bf16_t* __restrict__ W, int M, int N, int K, float eps, const float* __restrict__ Gw,
                   void* __restrict__ out_) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  constexpr int NW = KW * G;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];      // the stages, then the rows [M][K + 8]
  constexpr unsigned ROWS_AT = NW * ST * 2048;
  static_assert(ST == 4 || ST == 8, "four chunks' operands at a time");
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int kw = wave % KW, group = wave / KW;
  const int r = lane & 15, j = lane >> 4;
  const int per = SW ? 8 : 16, tiles = (N + per - 1) / per;
  const int tile = blockIdx.x * G + group, n0 = min(tile, tiles - 1) * per;      // (a group beyond the last works, and stores nothing)
  const int chunks = K / 64, steps = (chunks - kw + KW - 1) / KW;

  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  asm volatile("" : "+v"(acc));        // (in registers of its own from here: in some that loads went to it would wait for everything under way)
  // the rows' and the norm's loads, then the weights': they come back in that order.  (As buffer loads whose descriptor ends with the row:
  // one address for all pieces, and zeros beyond K.)
  constexpr int RB = KC <= 8 ? 2 : 1;
  typedef float v4f __attribute__((ext_vector_type(4)));
  v4f g[KC], v[RB][KC];
  auto row_at = [&](const float* p) __attribute__((always_inline)) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, K * 4, 0x00020000); };
  auto load_row = [&](const float* p, v4f (&to)[KC]) __attribute__((always_inline)) {
    const auto rs = row_at(p);
#pragma unroll
    for (int c = 0; c < KC; ++c) to[c] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16 + c * 1024, 0, 0));
  };
  auto load_rows = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
      if (r0 + NW * b < M) load_row(X + (size_t)(r0 + NW * b) * K, v[b]);
  };
  // (only what is needed: a load of 1 KiB keeps the unit that takes addresses for 16 cycles, and twelve of every wavefront were 0.6 us)
  if (wave < M) {
    load_rows(wave);
    load_row(Gw, g);
  }
  const int tok = (threadIdx.x % (64 * KW)) >> 4, row = threadIdx.x & 15;
  const int n = (SW ? n0 + (row & 7) : n0 + row);
  float prev = 0.f;
  if (EPI == TI_EPI_ADD_F32) prev = ((const float*)out_)[(size_t)(tok < M ? tok : 0) * N + (n < N ? n : N - 1)];
  __builtin_amdgcn_sched_barrier(0);
  const int lr = lane >> 3, piece = piece_of((lane & 7) ^ lr) * 16;
  const unsigned v0 = (unsigned)min(lr, N - 1 - n0) * (unsigned)(K * 2) + piece;
  const unsigned v1 = SW ? v0 : (unsigned)min(8 + lr, N - 1 - n0) * (unsigned)(K * 2) + piece;
  const auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
  const auto rsW = rows_at(W + (size_t)n0 * K), rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K);
  unsigned char* mine = smem + wave * (ST * 2048);
  auto load = [&](int step, unsigned stage) __attribute__((always_inline)) {
    const int at = max(kw + KW * step, 0) * 128;         // (a wavefront without a chunk asks for the first)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, (__attribute__((address_space(3))) void*)(mine + stage), 16, v0, at, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsU, (__attribute__((address_space(3))) void*)(mine + stage + 1024), 16, v1, at, 0, 0);
  };
  // (without a condition, the last one again where there are fewer: the compiler counts these loads where the rows are waited for)
#pragma unroll
  for (int d = 0; d < ST; ++d) load(min(d, steps - 1), d * 2048);
  __builtin_amdgcn_sched_barrier(0);

  // the norm; written as instructions, or the compiler would have the writes wait for the weights
  const unsigned rows_lds = (unsigned)(size_t)smem + ROWS_AT, row_bytes = (K + 8) * 2;
  const bool full = K == 256 * KC;
  auto norm_rows = [&](int r0) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int m = r0 + NW * b;
      if (b > 0 && m >= M) continue;
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < KC; ++c) ss = rms_accumulate(ss, make_float4(v[b][c].x, v[b][c].y, v[b][c].z, v[b][c].w));
      const float scale = rms_scale(ss, K, eps);
      if (m < M) {
        const unsigned to = rows_lds + m * row_bytes + lane * 8;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          typedef unsigned v2u __attribute__((ext_vector_type(2)));
          const v2u h = {pack_bf16x2(v[b][c].x * scale * g[c].x, v[b][c].y * scale * g[c].y),
                         pack_bf16x2(v[b][c].z * scale * g[c].z, v[b][c].w * scale * g[c].w)};
          if (full || lane * 4 + 256 * c < K) asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(to), "v"(h), "n"(c * 512) : "memory");
        }
      }
    }
  };
  if (wave < M) norm_rows(wave);      // (not in the loop, where the compiler would wait for the weights too)
#pragma clang loop unroll(disable)
  for (int r0 = wave + NW * RB; r0 < M; r0 += NW * RB) {
    load_rows(r0);
    norm_rows(r0);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();

  // ---- the product: chunks kw, kw + KW, ...
  const unsigned a_at = rows_lds + (r < M ? r : 0) * row_bytes + j * 32 + kw * 128;
  const unsigned w_x = (unsigned)(size_t)mine + r * 128 + ((j ^ (r & 7)) << 4);
  const unsigned w_y = (unsigned)(size_t)mine + r * 128 + (((j + 4) ^ (r & 7)) << 4);
  unsigned stage = 0;
  int i = 0;
  auto multiply = [&](const RowPieces& w, const v4u& x, const v4u& y) __attribute__((always_inline)) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w.x), __builtin_bit_cast(bf16x8, x), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w.y), __builtin_bit_cast(bf16x8, y), acc, 0, 0, 0);
  };
  for (; i + ST < steps; ++i) {
    wait_vmcnt<2 * (ST - 1)>();
    RowPieces w, a;
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %6 offset:16\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(w.x), "=&v"(w.y), "=&v"(a.x), "=&v"(a.y) : "v"(w_x + stage), "v"(w_y + stage), "v"(a_at + i * (KW * 128)) : "memory");
    load(i + ST, stage);
    multiply(w, a.x, a.y);
    stage = stage == (ST - 1) * 2048 ? 0 : stage + 2048;
  }
  // the last ST: the rows' operands first, which are there
  v4u a[2 * ST];
#pragma unroll
  for (int u = 0; u < ST; u += 4) {
    const unsigned a0 = a_at + min(i + u, max(steps - 1, 0)) * (KW * 128), a1 = a_at + min(i + u + 1, max(steps - 1, 0)) * (KW * 128),
                   a2 = a_at + min(i + u + 2, max(steps - 1, 0)) * (KW * 128), a3 = a_at + min(i + u + 3, max(steps - 1, 0)) * (KW * 128);
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:16\n\tds_read_b128 %2, %9\n\tds_read_b128 %3, %9 offset:16\n\t"
                 "ds_read_b128 %4, %10\n\tds_read_b128 %5, %10 offset:16\n\tds_read_b128 %6, %11\n\tds_read_b128 %7, %11 offset:16\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(a[2 * u]), "=&v"(a[2 * u + 1]), "=&v"(a[2 * u + 2]), "=&v"(a[2 * u + 3]), "=&v"(a[2 * u + 4]), "=&v"(a[2 * u + 5]),
                   "=&v"(a[2 * u + 6]), "=&v"(a[2 * u + 7])
                 : "v"(a0), "v"(a1), "v"(a2), "v"(a3) : "memory");
  }
  auto last = [&](auto tag) __attribute__((always_inline)) {
    constexpr int u = decltype(tag)::value;
    if (i + u >= steps) return false;
    wait_vmcnt<2 * (ST - 1 - u)>();
    RowPieces w;
    read_some_blocks<1>(&w, w_x + stage, w_y + stage);
    multiply(w, a[2 * u], a[2 * u + 1]);
    stage = stage == (ST - 1) * 2048 ? 0 : stage + 2048;
    return true;
  };
  auto all = [&](auto... tags) __attribute__((always_inline)) { return (last(tags) && ...); };
  using std::integral_constant;
  if (all(integral_constant<int, 0>{}, integral_constant<int, 1>{}, integral_constant<int, 2>{}, integral_constant<int, 3>{}))
    if constexpr (ST == 8)
      (void)all(integral_constant<int, 4>{}, integral_constant<int, 5>{}, integral_constant<int, 6>{}, integral_constant<int, 7>{});
  wait_vmcnt<0>();      // (stages filled and never read: the sums come after the loads)
  // acc[i]: weight row 4 j + i, token r
  auto red = [&](int w) -> float (*)[17] { return reinterpret_cast<float (*)[17]>(smem + w * (ST * 2048)); };
#pragma unroll
  for (int i = 0; i < 4; ++i) red(wave)[r][4 * j + i] = acc[i];
  __syncthreads();
  if (tok >= M || tile >= tiles || n >= N || (SW && row >= 8)) return;
  if (SW) {
    float gt = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < KW; ++w) {
      gt += red(group * KW + w)[tok][row];
      up += red(group * KW + w)[tok][row + 8];
    }
    ((bf16_t*)out_)[(size_t)tok * N + n] = f2bf(silu_mul(gt, up));
  } else {
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < KW; ++w) sum += red(group * KW + w)[tok][row];
    const size_t o = (size_t)tok * N + n;
    if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = sum;
    if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev + sum;
    if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(sum));
  }
#endif
}

// ================================== few tokens, any K: the token rows in pieces, loads never at rest
// out (op)= A W^T for M <= 16, K a multiple of 64.  As in the kernels above a workgroup of four
// wavefronts owns 16 weight rows, wavefront w takes the 64-wide chunks w, w + 4, ... of K, and the
// four sums meet in LDS in the order 0..3: with one workgroup per 16 rows the bits are those of
// the kernels above.  Two things differ.
//  * The token rows go through LDS in pieces of SP_PIECE columns, two buffers in turn: any K fits,
//    and any M <= 16 leaves room for two workgroups or more on a compute unit.
//  * While a piece is multiplied, the weights and the token rows of the next one are already on
//    their way: a wavefront always has 8 to 16 KB of weights in flight, where the kernels above
//    ask for a batch, wait for all of it, multiply, and only then ask again.  On weights of tens
//    to hundreds of megabytes that is the difference between ~3.5 and ~5.5 TB/s.
// grid (ceil(N / 16), KS) (SwiGLU: ceil(F / 8)).  KS > 1 (adding epilogue only): workgroup
// (., s) takes the pieces s, s + KS, ... and leaves its sums in partial [KS][M][N]; they are
// added to the residual in the order 0..KS-1 by whoever reads it next.
#define SP_PIECE 1024              // 16 chunks: four per wavefront, one batch of loads
#define SP_LD (SP_PIECE + 8)       // LDS row stride in bfloat16
// AV: 16-byte pieces of the token rows per thread and piece (M <= 2 AV)
template <int EPI, int AV, bool SPLIT>
__global__ void __launch_bounds__(256)
gemm_skinny_pieces_kernel(const bf16_t* __restrict__ A, long lda, const bf16_t* __restrict__ W, void* __restrict__ out_,
                          float* __restrict__ partial, int M, int N, int K) {
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
  bf16_t* sA = reinterpret_cast<bf16_t*>(dyn_smem);          // [2][M][SP_LD]
  __shared__ float red[4][16][17];
  constexpr int NT = 256;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, j = lane >> 4;
  const int tile = blockIdx.x;               // 16 rows (SwiGLU: 8 gate and 8 up rows)
  int wrow;
  if (SW) {
    const int n = tile * 8 + (r & 7);
    wrow = (r < 8 ? 0 : N) + (n < N ? n : N - 1);
  } else {
    const int n = tile * 16 + r;
    wrow = n < N ? n : N - 1;
  }
  const bf16_t* wp = W + (size_t)wrow * K + j * 16;
  const int chunks = K / 64;
  const int n_pieces = (K + SP_PIECE - 1) / SP_PIECE;
  const int KS = SPLIT ? gridDim.y : 1, split = SPLIT ? blockIdx.y : 0;

  const int tok = threadIdx.x >> 4, row = threadIdx.x & 15;
  float prev = 0.f;
  if (EPI == TI_EPI_ADD_F32 && !SPLIT) {   // threads without an output element read a valid one: no branch
    const int n = tile * 16 + row;
    prev = ((const float*)out_)[(size_t)(tok < M ? tok : 0) * N + (n < N ? n : N - 1)];
  }

  // piece p: thread t copies the 16-byte pieces t, t + NT, ... of [M][SP_PIECE / 8]
  uint4 av[AV];
  auto ask_rows = [&](int p) {
#pragma unroll
    for (int b = 0; b < AV; ++b) {
      const int v = threadIdx.x + NT * b;
      const int m = v / (SP_PIECE / 8), k = p * SP_PIECE + (v % (SP_PIECE / 8)) * 8;
      const bool ok = m < M && k < K;
      av[b] = ld16(A + (ok ? (size_t)m * lda + k : 0));
    }
  };
  auto keep_rows = [&](int buf) {
#pragma unroll
    for (int b = 0; b < AV; ++b) {
      const int v = threadIdx.x + NT * b;
      const int m = v / (SP_PIECE / 8);
      if (m < M) *reinterpret_cast<uint4*>(sA + ((size_t)buf * M + m) * SP_LD + (v % (SP_PIECE / 8)) * 8) = av[b];
    }
  };
  // a chunk beyond the last reads chunk 0 and counts for nothing: no branch between the loads
  auto ask_weights = [&](int p, Frag (&w0)[4], Frag (&w1)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = p * (SP_PIECE / 64) + wave + 4 * u;
      const size_t at = (size_t)(c < chunks ? c : 0) * 64;
      w0[u].u = ld16(wp + at);
      w1[u].u = ld16(wp + at + 8);
    }
  };
  floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
  const uint4 zero = make_uint4(0, 0, 0, 0);
  auto multiply = [&](int p, int buf, Frag (&w0)[4], Frag (&w1)[4]) {
    const bf16_t* ap = sA + ((size_t)buf * M + (r < M ? r : 0)) * SP_LD + j * 16;
    Frag a0[4], a1[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a0[u].u = *reinterpret_cast<const uint4*>(ap + (wave + 4 * u) * 64);
      a1[u].u = *reinterpret_cast<const uint4*>(ap + (wave + 4 * u) * 64 + 8);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (p * (SP_PIECE / 64) + wave + 4 * u >= chunks) w0[u].u = w1[u].u = zero;
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[u].v, a0[u].v, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[u].v, a1[u].v, acc, 0, 0, 0);
    }
  };
  // one turn: piece p is multiplied out of `buf` and (w0, w1) while piece p + KS arrives in the
  // other buffer and (n0, n1).  Loads return in the order they were asked for: the rows of the
  // next piece are asked for before its weights, so that keeping them waits for nothing else.
  auto turn = [&](int p, int buf, Frag (&w0)[4], Frag (&w1)[4], Frag (&n0)[4], Frag (&n1)[4]) {
    const bool more = p + KS < n_pieces;
    if (more) {
      ask_rows(p + KS);
      __builtin_amdgcn_sched_barrier(0);
      ask_weights(p + KS, n0, n1);
      __builtin_amdgcn_sched_barrier(0);
    }
    multiply(p, buf, w0, w1);
    if (more) keep_rows(buf ^ 1);
    __syncthreads();
  };
  Frag wa0[4], wa1[4], wb0[4], wb1[4];
  int p = split;
  if (p < n_pieces) {
    ask_rows(p);
    __builtin_amdgcn_sched_barrier(0);
    ask_weights(p, wa0, wa1);
    __builtin_amdgcn_sched_barrier(0);
    keep_rows(0);
  }
  __syncthreads();
  while (p < n_pieces) {
    turn(p, 0, wa0, wa1, wb0, wb1);
    p += KS;
    if (p >= n_pieces) break;
    turn(p, 1, wb0, wb1, wa0, wa1);
    p += KS;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][r][4 * j + i] = acc[i];
  __syncthreads();
  if (tok >= M) return;
  if (SW) {
    if (row >= 8) return;
    const int n = tile * 8 + row;
    if (n >= N) return;
    float gt = 0.f, up = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      gt += red[w][tok][row];
      up += red[w][tok][row + 8];
    }
    ((bf16_t*)out_)[(size_t)tok * N + n] = f2bf(silu_mul(gt, up));
  } else {
    const int n = tile * 16 + row;
    if (n >= N) return;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) sum += red[w][tok][row];
    const size_t o = (size_t)tok * N + n;
    if (SPLIT) partial[(size_t)split * M * N + o] = sum;
    else if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = sum;
    else if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev + sum;
    else if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(sum));
  }
}

// ================================== few tokens, a weight of few rows: a row per wavefront
// out (op)= A W^T for M <= MMAX tokens and a weight with so few rows that the kernels above,
// whose workgroups own 16 rows each, would leave most compute units idle (N = 1024: 64
// workgroups), while each busy unit would have hundreds of load instructions to get through
// (a unit takes one 64-lane load every ~25 cycles: measured 2.7 us to issue 256 of them).
// Here a wavefront owns one weight row: lane l holds the 8-element pieces l, l + 64, ... of
// it (every load instruction fetches 1 KiB that nobody else fetches), the token rows are
// copied into LDS once per workgroup, the products are v_dot2c_f32_bf16 (two multiply-adds
// on packed bfloat16, accumulated in 32-bit), and the lanes' partial sums meet in a
// butterfly.  N / 4 workgroups of four wavefronts.  A row's bits do not depend on the rows
// beside it.  K a multiple of 8, up to 512 NL (NL: pieces of the weight row per lane); MMAX: the
// most tokens.  Both are template parameters so that every load is unconditional and counted.
#define GR_LOADS 8
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dot2_bf16(unsigned a, unsigned b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}

// The token rows come by direct loads into LDS, each once a workgroup, and a lane reads back the pieces that go with its own.
// (Every wavefront asking for them itself, MMAX NL loads of 1 KiB at 16 cycles each of the unit that takes addresses, was what 3 to 8
// tokens waited for, and the residual, which the compiler asked for at the end.  us in a chain of launches with weights from memory, before and
// now, at 4 and 8 tokens: 1,024 x 2,048 3.52 4.17 -> 3.16 3.83, 1,024 x 3,072 4.03 4.98 -> 3.59 4.34, 1,024 x 4,096 4.66 6.79 -> 4.04 4.88, 2,048 x
// 2,048 at 4 4.46 -> 3.98.  Up to two tokens ask for them themselves: the next kernel.)
template <int EPI, int MMAX, int NL>
__global__ void __launch_bounds__(256)
gemv_rows_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_, int M, int N,
                 int K, long lda) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  static_assert(EPI != TI_EPI_SWIGLU, "no SwiGLU here");
  static_assert(MMAX % 4 == 0, "the wavefronts take the token rows in turn");
  extern __shared__ __attribute__((aligned(1024))) unsigned char dyn_smem[];     // pieces of 1 KiB: [MMAX][NL], then each wavefront's [NL]
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + wave;
  // the residual lane m will add to (row m of the tokens)
  float prev = 0.f;
  if (EPI == TI_EPI_ADD_F32) prev = ((const float*)out_)[(size_t)(lane < M ? lane : 0) * N + (n < N ? n : N - 1)];
  // The token rows wave, wave + 4, ... (a row beyond M is row 0: read and dropped, so that every load is counted), then the weight row.
  // All of them direct loads: the waits below count these alone, and whatever else is on its way makes them wait for more, not for less.
  const auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
#pragma unroll
  for (int t = 0; t < MMAX / 4; ++t) {
    const int m = wave + 4 * t;
    const auto rs = rows_at(A + (size_t)(m < M ? m : 0) * lda);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int kk = (i * 64 + lane) * 8;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(dyn_smem + (m * NL + i) * 1024), 16,
                                               (kk < K ? kk : 0) * 2, 0, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  const auto rsW = rows_at(W + (size_t)(n < N ? n : N - 1) * K);
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int kk = (i * 64 + lane) * 8;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, (__attribute__((address_space(3))) void*)(dyn_smem + (MMAX * NL + wave * NL + i) * 1024), 16,
                                             (kk < K ? kk : 0) * 2, 0, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  wait_vmcnt<NL>();      // the rows have landed; the weights may be on their way
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);

  float acc[MMAX];
#pragma unroll
  for (int m = 0; m < MMAX; ++m) acc[m] = 0.f;
  const unsigned at = (unsigned)(size_t)dyn_smem + lane * 16, w_at = at + (MMAX + wave) * NL * 1024;
  auto piece = [&](auto tag) __attribute__((always_inline)) {
    constexpr int i = decltype(tag)::value;
    const int kk = (i * 64 + lane) * 8;
    // (read as instructions, or the compiler would have them wait for everything under way)
    v4u a[MMAX], w;
#pragma unroll
    for (int m = 0; m < MMAX; m += 4)
      asm volatile("ds_read_b128 %0, %4 offset:%5\n\tds_read_b128 %1, %4 offset:%6\n\tds_read_b128 %2, %4 offset:%7\n\t"
                   "ds_read_b128 %3, %4 offset:%8\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(a[m]), "=&v"(a[m + 1]), "=&v"(a[m + 2]), "=&v"(a[m + 3])
                   : "v"(at), "n"((m * NL + i) * 1024), "n"(((m + 1) * NL + i) * 1024), "n"(((m + 2) * NL + i) * 1024),
                     "n"(((m + 3) * NL + i) * 1024)
                   : "memory");
    wait_vmcnt<NL - 1 - i>();
    asm volatile("ds_read_b128 %0, %1 offset:%2\n\ts_waitcnt lgkmcnt(0)" : "=&v"(w) : "v"(w_at), "n"(i * 1024) : "memory");
    if (kk >= K) w = v4u{0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < MMAX; ++m) {
      acc[m] = dot2_bf16(w.x, a[m].x, acc[m]);
      acc[m] = dot2_bf16(w.y, a[m].y, acc[m]);
      acc[m] = dot2_bf16(w.z, a[m].z, acc[m]);
      acc[m] = dot2_bf16(w.w, a[m].w, acc[m]);
    }
  };
  static_assert(NL == 2 || NL == 4 || NL == 6 || NL == 8, "pieces of a row");
  piece(std::integral_constant<int, 0>{}), piece(std::integral_constant<int, 1>{});
  if constexpr (NL > 2) piece(std::integral_constant<int, 2>{}), piece(std::integral_constant<int, 3>{});
  if constexpr (NL > 4) piece(std::integral_constant<int, 4>{}), piece(std::integral_constant<int, 5>{});
  if constexpr (NL > 6) piece(std::integral_constant<int, 6>{}), piece(std::integral_constant<int, 7>{});
  if (EPI == TI_EPI_ADD_F32) asm volatile("" : "+v"(prev));      // (or the load would move behind the condition below)
  float mine = 0.f;
#pragma unroll
  for (int m = 0; m < MMAX; ++m) {
    const float t = group_sum<TI_WAVE>(acc[m]);
    if (lane == m) mine = t;
  }
  if (lane < M && n < N) {
    const size_t o = (size_t)lane * N + n;
    if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = mine;
    if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev + mine;
    if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(mine));
  }
#endif
}

// The same product for one or two tokens, their rows straight from memory into registers: lane l fetches, for every
// token, the pieces of the row that go with its pieces of the weight row (all workgroups read the same few
// KB: they come from the caches), after its weights have been asked for.  Nothing is waited for at a barrier and read back between
// the arrival of the weights and the products.  The same order of sums, the same bits.  (With the residual asked for in front, one token:
// 1,024 x 2,048 3.14 -> 2.83, 1,024 x 3,072 3.38 -> 3.16.)
template <int EPI, int MMAX, int NL>
__global__ void __launch_bounds__(256)
gemv_rows_direct_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_, int M,
                        int N, int K, long lda) {
  static_assert(EPI != TI_EPI_SWIGLU, "no SwiGLU here");
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = blockIdx.x * 4 + wave;
  const bf16_t* wp = W + (size_t)(n < N ? n : N - 1) * K;
  const uint4 zero = make_uint4(0, 0, 0, 0);
  float prev = 0.f;
  if (EPI == TI_EPI_ADD_F32) prev = ((const float*)out_)[(size_t)(lane < M ? lane : 0) * N + (n < N ? n : N - 1)];
  uint4 wv[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int kk = (i * 64 + lane) * 8;
    wv[i] = ld16(wp + (kk < K ? kk : 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  uint4 a[NL][MMAX];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int kk = (i * 64 + lane) * 8;
#pragma unroll
    for (int m = 0; m < MMAX; ++m) a[i][m] = ld16(A + (size_t)(m < M ? m : 0) * lda + (kk < K ? kk : 0));
  }
  __builtin_amdgcn_sched_barrier(0);
  float acc[MMAX];
#pragma unroll
  for (int m = 0; m < MMAX; ++m) acc[m] = 0.f;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int kk = (i * 64 + lane) * 8;
    const uint4 w = kk < K ? wv[i] : zero;
#pragma unroll
    for (int m = 0; m < MMAX; ++m) {
      acc[m] = dot2_bf16(w.x, a[i][m].x, acc[m]);
      acc[m] = dot2_bf16(w.y, a[i][m].y, acc[m]);
      acc[m] = dot2_bf16(w.z, a[i][m].z, acc[m]);
      acc[m] = dot2_bf16(w.w, a[i][m].w, acc[m]);
    }
  }
  if (EPI == TI_EPI_ADD_F32) asm volatile("" : "+v"(prev));      // (or the load would move behind the condition below)
  float mine = 0.f;
#pragma unroll
  for (int m = 0; m < MMAX; ++m) {
    const float t = group_sum<TI_WAVE>(acc[m]);
    if (lane == m) mine = t;
  }
  if (lane < M && n < N) {
    const size_t o = (size_t)lane * N + n;
    if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = mine;
    if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = prev + mine;
    if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(mine));
  }
}

// =============================================================== tiled kernel
#define TBM 128
#define TBN 128
#define TBK 32
#define TLD (TBK + 8)   // LDS row stride in bfloat16: 80 bytes, keeps 16-byte reads off the same banks
#define TPIECES (TBM * TBK / 8 / 256)   // 16-byte pieces per thread and operand tile
#define TKP (TBK / 8)                   // pieces per row

// SwiGLU: the workgroup covers 64 output columns; LDS row b of the weight tile is
// global row (b & 32 ? F : 0) + n0 + (b >> 6) * 32 + (b & 31), so that in every
// wavefront MFMA tile 0 holds gate columns and tile 1 the matching up columns.
template <int EPI>
__global__ void __launch_bounds__(256)
gemm_tiled_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_,
                  int M, int N, int K, long lda) {
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  __shared__ __attribute__((aligned(16))) bf16_t sA[2][TBM * TLD];
  __shared__ __attribute__((aligned(16))) bf16_t sB[2][TBN * TLD];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * TBM;
  const int n0 = blockIdx.x * (SW ? TBN / 2 : TBN);
  const int w_rows = SW ? 2 * N : N;

  // global -> LDS in pieces of 16 bytes, TPIECES per thread and operand tile
  constexpr int RSTEP = 256 / TKP;   // rows covered by one round of the workgroup
  const int lrow = tid / TKP, lkc = (tid % TKP) * 8;
  const bf16_t* gA[TPIECES];
  const bf16_t* gB[TPIECES];
  bool okA[TPIECES], okB[TPIECES];
#pragma unroll
  for (int i = 0; i < TPIECES; ++i) {
    const int row = lrow + RSTEP * i;
    const int am = m0 + row;
    okA[i] = am < M;
    gA[i] = A + (size_t)(okA[i] ? am : 0) * lda + lkc;
    int wr;
    if (SW) {
      const int n = n0 + (row >> 6) * 32 + (row & 31);
      okB[i] = n < N;
      wr = ((row & 32) ? N : 0) + (okB[i] ? n : 0);
    } else {
      wr = n0 + row;
      okB[i] = wr < N;
      if (!okB[i]) wr = 0;
    }
    (void)w_rows;
    gB[i] = W + (size_t)wr * K + lkc;
  }
  const uint4 zero = make_uint4(0, 0, 0, 0);
  uint4 ra[TPIECES], rb[TPIECES];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < TPIECES; ++i) {
      const bool kin = k0 + lkc + 8 <= K;
      ra[i] = (okA[i] && kin) ? ld16(gA[i] + k0) : zero;
      rb[i] = (okB[i] && kin) ? ld16(gB[i] + k0) : zero;
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < TPIECES; ++i) {
      *reinterpret_cast<uint4*>(&sA[buf][(lrow + RSTEP * i) * TLD + lkc]) = ra[i];
      *reinterpret_cast<uint4*>(&sB[buf][(lrow + RSTEP * i) * TLD + lkc]) = rb[i];
    }
  };

  floatx16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  const int fr = lane & 31, fk = (lane >> 5) * 8;
  const int n_k = (K + TBK - 1) / TBK;
  fetch(0);
  stash(0);
  __syncthreads();
  for (int kt = 0; kt < n_k; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < n_k) fetch((kt + 1) * TBK);
#pragma unroll
    for (int ks = 0; ks < TBK; ks += 16) {
      Frag fa[2], fb[2];
#pragma unroll
      for (int a = 0; a < 2; ++a)
        fa[a].u = *reinterpret_cast<const uint4*>(&sA[buf][(wm * 64 + a * 32 + fr) * TLD + ks + fk]);
#pragma unroll
      for (int b = 0; b < 2; ++b)
        fb[b].u = *reinterpret_cast<const uint4*>(&sB[buf][(wn * 64 + b * 32 + fr) * TLD + ks + fk]);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a].v, fb[b].v, acc[a][b], 0, 0, 0);
    }
    if (kt + 1 < n_k) stash(buf ^ 1);
    __syncthreads();
  }

  // acc[a][b][i]: row wm*64 + a*32 + 8*(i/4) + 4*(lane/32) + i%4, column wn*64 + b*32 + lane%32
  const int ccol = lane & 31, crow = (lane >> 5) * 4;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + wm * 64 + a * 32 + (i >> 2) * 8 + crow + (i & 3);
      if (m >= M) continue;
      if (SW) {
        const int n = n0 + wn * 32 + ccol;
        if (n < N) ((bf16_t*)out_)[(size_t)m * N + n] = f2bf(silu_mul(acc[a][0][i], acc[a][1][i]));
      } else {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int n = n0 + wn * 64 + b * 32 + ccol;
          if (n >= N) continue;
          const size_t o = (size_t)m * N + n;
          const float s = acc[a][b][i];
          if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = s;
          if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] += s;
          if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(s));
        }
      }
    }
  }
}

// ====================================================== tiled kernel, pipelined
// The same product with the tiles brought in by direct memory-to-LDS loads
// (buffer_load_dwordx4 ... lds: each lane fetches 16 bytes, the wavefront's 64 pieces
// land in 1 KiB of LDS in lane order), STAGES - 1 k-tiles ahead of the one that is
// multiplied (K must be a multiple of 64; other K take the plain tiled kernel).
// BK = 64: a tile row is 128 bytes = 8 pieces, one line of the caches (k-tiles of 32,
// half a line a row, take a third longer from memory).  Rows are stored unpadded, and
// piece c of row r sits in slot c ^ ((r >> 1) & 7): the 16 rows that one phase of a
// 16-byte LDS read touches then fall on all 64 banks once.  The lane that fills slot
// (r, c) simply fetches piece c ^ ((r >> 1) & 7) of row r.
//
// WG tile BM x BN, four or eight wavefronts as WAVES_M x WAVES_N, each (BM / WAVES_M) x
// (BN / WAVES_N) out of 32 x 32 x 16 MFMAs.  SwiGLU needs two 32-column tiles per
// wavefront: the first half holds gate columns, the second the matching up columns.
#define PBK 64
#define PSTAGES 3

// What the epilogue TI_EPI_QKV_PREP needs: the product is the fused q/k/v projection of a step's
// rows, and instead of storing it the kernel finishes each head of each row: per-head norm and
// rotation for q heads (to q_out, T [M, n_head hd]) and k heads (into the cache page of the row's
// position), v heads copied into the cache transposed.  A workgroup's BN columns are whole heads.
struct QKVEpilogue {
  const float* q_w;          // per-head norm weights or nullptr
  const float* k_w;
  float eps;
  const float* inv_freq;     // nullptr: no rotation
  const float2* rope_table;  // (cos, sin) [table_len][hd / 2] or nullptr
  int table_len;
  const int* pos;            // position of each row
  const int* slot;           // block-table row of each row
  const int* table;
  int table_stride;
  bf16_t* pool;              // [pages][2][n_kv][P * hd]
  bf16_t* q_out;
  int n_head, n_kv, hd, P;
};

// A q or k head (unit u of the fused projection, head hh of the tile) of all BM rows of a tile that
// lies in LDS in 32-bit (row stride FS): eight lanes a row, 8 NWV rows a pass.  The angles of the
// next pass are asked for before a pass is finished; a lane reads its HD / 16 pairs from LDS as runs of
// 16 bytes and writes its finished elements to memory as two runs of HD / 8 bytes, the eight lanes
// together the row's 2 HD consecutive bytes.
template <int HD, int BM, int NWV, int FS, bool NORMED, bool ROTATE>
__device__ __forceinline__ void qkv_rows_by_lanes(const QKVEpilogue& ep, float* ft, const int* s_pos,
                                                  const int* s_page, const int* s_prow, const int* s_live, int hh,
                                                  int u, int m0) {
  constexpr int NP = HD / 16, PASSES = BM / (NWV * 8);
  const int tid = threadIdx.x;
  const bool is_q = u < ep.n_head;
  float wlo[NP], whi[NP];
  qk_lanes_weights<HD>(wlo, whi, NORMED ? (is_q ? ep.q_w : ep.k_w) : nullptr);
  float2 cs[NP], next[NP];
#pragma unroll 1
  for (int ps = -1; ps < PASSES; ++ps) {
    if (ROTATE && ps + 1 < PASSES)
      qk_lanes_angles<HD>(next, s_pos[(ps + 1) * NWV * 8 + tid / 8], ep.inv_freq, ep.rope_table, ep.table_len);
    if (ps >= 0) {
      const int r = ps * NWV * 8 + tid / 8;
      unsigned lo[NP / 2], hi[NP / 2];
      qk_head_lanes<HD, NORMED, ROTATE>(ft + r * FS + hh * HD, wlo, whi, ep.eps, cs, lo, hi);
      bf16_t* dst = nullptr;
      if (is_q) {
        if (s_live[r] >= 0) dst = ep.q_out + ((size_t)(m0 + r) * ep.n_head + u) * HD;
      } else if (s_page[r] >= 0) {
        dst = kv_page_slot<bf16_t>(ep.pool, s_page[r], 0, u - ep.n_head, s_prow[r], ep.n_kv, ep.P, HD);
      }
      if (dst) {
        bf16_t* mine = dst + NP * (tid & 7);
        if constexpr (NP == 8) {
          *reinterpret_cast<uint4*>(mine) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
          *reinterpret_cast<uint4*>(mine + HD / 2) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        } else {
          *reinterpret_cast<uint2*>(mine) = make_uint2(lo[0], lo[1]);
          *reinterpret_cast<uint2*>(mine + HD / 2) = make_uint2(hi[0], hi[1]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) cs[k] = next[k];
  }
}

template <int HD, int BM, int NWV, int FS>
__device__ __forceinline__ void qkv_rows_by_lanes(const QKVEpilogue& ep, float* ft, const int* s_pos,
                                                  const int* s_page, const int* s_prow, const int* s_live, int hh,
                                                  int u, int m0) {
  const bool normed = (u < ep.n_head ? ep.q_w : ep.k_w) != nullptr, rotate = ep.inv_freq != nullptr;
  if (normed && rotate)
    qkv_rows_by_lanes<HD, BM, NWV, FS, true, true>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
  else if (normed)
    qkv_rows_by_lanes<HD, BM, NWV, FS, true, false>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
  else if (rotate)
    qkv_rows_by_lanes<HD, BM, NWV, FS, false, true>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
  else
    qkv_rows_by_lanes<HD, BM, NWV, FS, false, false>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
}

// LDS of that epilogue: 128 columns of a tile of bm rows in 32-bit, and four words a row.
constexpr int qkv_prep_lds(int bm, int bn) { return bm * ((bn < 128 ? bn : 128) + 8) * 4 + 4 * bm * 4; }

// tile(n_k - LEFT, LEFT) for LEFT = STAGES - 2, ..., 0, as far as there are tiles
template <class Tile, int... I>
__device__ __forceinline__ void last_tiles(int n_k, Tile&& tile, std::integer_sequence<int, I...>) {
  constexpr int N = (int)sizeof...(I);
  ((n_k >= N - I ? (tile(n_k - (N - I), std::integral_constant<int, N - 1 - I>{}), 0) : 0), ...);
}

// PHASED: the multiply loop goes by quarters of a wavefront's tile, for tiles of 256 x 256 (see the loop).
template <int BM, int BN, int WAVES_M, int WAVES_N, int EPI, int STAGES = PSTAGES, bool PHASED = false>
__global__ void __launch_bounds__(WAVES_M * WAVES_N * 64)
gemm_pipelined_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_arg,
                      int M, int N, int K, long lda, int n_first, int xcd_rows, int die_rows, QKVEpilogue ep = QKVEpilogue{}) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  // n_first: the output column the grid's first workgroup starts at (a launch may cover a range of columns)
  // xcd_rows > 0: which tile a workgroup takes follows the eight dies.  Workgroups go to the dies in turn, so die c has
  // numbers c, c + 8, ...; it takes one block of the tiles (the rows cut in die_rows, the columns in 8 / die_rows, both
  // dividing the grid), in groups of xcd_rows row tiles, down the rows of a column first: the workgroups of a die then read
  // only the block's rows of A and W into the die's own L2, and those that run together share them.
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd_rows > 0) {
    const int die_cols = 8 / die_rows, nx = gridDim.x, cx = nx / die_cols, cy = gridDim.y / die_rows;
    const int id = bx + nx * by, die = id & 7, local = id >> 3;
    const int full = cy / xcd_rows, per = xcd_rows * cx;
    int rb = local / per, rem = local - rb * per, rows = xcd_rows;
    if (rb >= full) {
      rb = full;
      rem = local - full * per;
      rows = cy - full * xcd_rows;
    }
    by = (die / die_cols) * cy + rb * xcd_rows + rem % rows;
    bx = (die % die_cols) * cx + rem / rows;
  }
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  constexpr int TM = BM / WAVES_M / 32, TN = BN / WAVES_N / 32;
  constexpr int NWV = WAVES_M * WAVES_N;                     // wavefronts: 4 or 8
  static_assert(NWV == 4 || NWV == 8, "four or eight wavefronts");
  static_assert(!SW || TN % 2 == 0, "SwiGLU pairs the column tiles of a wavefront: the first half gate, the second half up");
  static_assert(STAGES >= 2, "one stage is multiplied, the others are on their way");
  // a row of a stage is KT bfloat16 (CPR pieces of 16 bytes); a wavefront's load of 1 KiB covers RPL rows
  constexpr int KT = PBK, CPR = KT / 8, RPL = 64 / CPR, ROWB = KT * 2, KSTEPS = KT / 16;
  auto swz = [](int r) { return (r >> 1) & 7; };

  constexpr int STAGE_BYTES = (BM + BN) * ROWB;
  constexpr int GROUPS_A = BM / RPL, GROUPS_B = BN / RPL;    // RPL rows = 1 KiB = one wavefront load
  static_assert((GROUPS_A + GROUPS_B) % NWV == 0, "every wavefront issues the same number of loads");
  constexpr int LOADS = (GROUPS_A + GROUPS_B) / NWV;         // per wavefront and k-tile
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  // gridDim.z > 1 (storing epilogue only): K is split; workgroup z takes its share of the k-tiles and
  // stores its sums into the z-th [M, N] of out
  const int kt0 = (int)((long)(K / KT) * blockIdx.z / gridDim.z);
  const int n_k = (int)((long)(K / KT) * (blockIdx.z + 1) / gridDim.z) - kt0;
  void* __restrict__ out_ = (EPI == TI_EPI_STORE_F32) ? (void*)((float*)out_arg + (size_t)blockIdx.z * M * N) : out_arg;
  // the wavefront's number in a scalar register: where its loads go in LDS is scalar arithmetic then
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;
  const int m0 = by * BM;
  const int n0 = n_first + bx * (SW ? BN / 2 : BN);
  const int lr = lane / CPR, lc = lane % CPR;                // row within a load's group of rows, slot within the row

  // Which group of RPL rows this wavefront's load i brings: 0 .. GROUPS_A - 1 of A, then of B, the weight's rows or, SwiGLU, its up rows.
  // PHASED: the first half of the loads brings the first halves of every wavefront's rows of A and of B, the second half the others.
  constexpr int span = BN / WAVES_N, half = span / 2;        // SwiGLU: a wavefront's columns are gate rows, then up rows
  constexpr int HA = GROUPS_A / 2 / NWV, HB = GROUPS_B / 2 / NWV;
  auto half_group = [](int rows, int second, int x) { return x / (rows / 2 / RPL) * (rows / RPL) + second * (rows / 2 / RPL) + x % (rows / 2 / RPL); };
  auto group_of = [&](int i) {
    if constexpr (!PHASED) return wave + NWV * i;
    else if (i < HA) return half_group(BM / WAVES_M, 0, wave + NWV * i);
    else if (i < HA + 2 * HB) return GROUPS_A + half_group(span, i < HA + HB ? 0 : 1, wave + NWV * ((i - HA) % HB));
    else return half_group(BM / WAVES_M, 1, wave + NWV * (i - HA - 2 * HB));
  };
  auto of_a = [&](int i, int g) { return PHASED ? i < HA || i >= HA + 2 * HB : g < GROUPS_A; };
  auto of_up = [&](int i, int g) { return SW && (PHASED ? i >= HA + HB : ((g - GROUPS_A) * RPL) % span >= half); };      // (of B's)
  // A load's rows lie behind one of three descriptors (tokens, weight rows, up rows), which are scalar, as is where a k-tile
  // starts; a lane's own offset stays the same from tile to tile, so that a load costs no vector arithmetic.  Rows beyond
  // the matrix are clamped into it: they are computed and thrown away.
  unsigned voff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int g = group_of(i);
    if (of_a(i, g)) {
      const int row = g * RPL + lr;
      voff[i] = (unsigned)min(row, M - 1 - m0) * (unsigned)(lda * 2) + (lc ^ swz(row)) * 16;
    } else {
      const int row = (g - GROUPS_A) * RPL + lr;
      const int n = SW ? (row / span) * half + (row % half) : row;
      voff[i] = (unsigned)min(n, N - 1 - n0) * (unsigned)(K * 2) + (lc ^ swz(row)) * 16;
    }
  }
  auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
  const auto rsA = rows_at(A + (size_t)m0 * lda + (size_t)kt0 * KT);
  const auto rsW = rows_at(W + (size_t)n0 * K + (size_t)kt0 * KT);
  const auto rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K + (size_t)kt0 * KT);
  // load i of this wavefront's LOADS loads of k-tile kt, into the stage at that byte
  auto issue_one = [&](int kt, unsigned stage, int i) {
    const int g = group_of(i);
    auto* dst = (__attribute__((address_space(3))) void*)(smem + stage + g * 1024);      // the same in every lane
    if (of_a(i, g)) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, dst, 16, voff[i], kt * KT * 2, 0, 0);
    else if (of_up(i, g)) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsU, dst, 16, voff[i], kt * KT * 2, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, dst, 16, voff[i], kt * KT * 2, 0, 0);
  };

  floatx16 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f;

  // The multiply loop is scheduled by hand.  The compiler does not know which LDS
  // bytes a direct load will write, so before any LDS read it can see, and at every
  // fence, it waits for all of them, the k-tiles in flight included; that would
  // undo the pipeline.  So LDS is read with ds_read_b128 in inline assembly, the
  // barrier is the bare instruction, and the waits are written out.
  //
  // A k-step's matrix instructions stand one by one, and between them what the steps ahead need: the
  // next step's fragments from LDS, and the loads of k-tile kt + STAGES - 1 (the unit that takes their
  // addresses handles 64 bytes a cycle for the whole compute unit: asked for at once they would queue
  // there with nothing on the matrix cores).  The last k-step's fragments are in registers before any
  // of its matrix instructions, so the workgroup meets behind number GB of that step: then the tile's
  // stage is free, tile kt + 1 has landed for every wavefront, and its first fragments are read behind
  // the remaining instructions; no k-tile begins with a wait for LDS.  Whole tiles run without a branch,
  // the last STAGES - 1 by themselves.
  // (Against a loop that met in front of each k-tile, read its first fragments there and asked by lane
  // addresses, us alone: 2048 x 24576 x 4096 with SwiGLU 382 -> 328, 2048 x 4096 x 12288 193 -> 167,
  // 2048 x 4096 x 4096 70 -> 61, 2048 x 4096 x 1024 24 -> 22.  Inside a prompt, where the chip is warmer, the first
  // takes 340.)
  const int fr = lane & 31, fh = lane >> 5;                  // fragment row, and which half of a 16-wide k-step
  const unsigned lds0 = (unsigned)(size_t)smem;              // LDS byte address of the first stage
  const unsigned rowA = lds0 + (wm * (BM / WAVES_M) + fr) * ROWB;
  const unsigned rowB = lds0 + BM * ROWB + (wn * (BN / WAVES_N) + fr) * ROWB;
  unsigned xo[KSTEPS];                                       // swizzled byte offset of this lane's piece, per k-step
#pragma unroll
  for (int ks = 0; ks < KSTEPS; ++ks) xo[ks] = ((ks * 2 + fh) ^ swz(fr)) << 4;

  // the residual an adding epilogue adds to: asked for while the last k-tile is multiplied
  // (elements outside the matrix read a valid one and are not stored)
  // (a tile of many accumulators has no registers for it and reads the residual in the epilogue)
  constexpr bool PREV = !PHASED && EPI == TI_EPI_ADD_F32 && (NWV == 4 || TM * TN <= 4);
  float prev[PREV ? TM : 1][PREV ? TN : 1][16];
  if constexpr (PHASED) {
    // By quarters: a phase multiplies half of the wavefront's rows of A with half of its rows of B over the whole k-tile, and the fragments of
    // a half stay in registers as long as they are used, so that a half's bytes of LDS are free again when they have been read once:
    //   lo x lo (reads B hi)   lo x hi (reads A hi)   hi x lo (reads the next k-tile's A lo)   hi x hi (reads its B lo)
    // The workgroup meets twice a k-tile.  In the first phase A lo and B lo are free, and B hi and A hi have landed; in the third the other
    // way round, of the next k-tile.  What is freed is asked for again at once: with two stages, which are all that LDS holds
    // of this tile, a load has a k-tile and a half to arrive in.  (In the loop below it has three quarters of one, and a k-tile of 256 x 256 takes
    // as long as memory does: 1.60 us on all units, 1.09 on eight, matrix instructions alone 1.17 and 0.87; by quarters 1.54 and 0.95 by
    // eight wavefronts, 1.45 and 0.92 by four, which read LDS the least.  Tiles of 256 x 128 and 128 x 128, whose three
    // and four stages are as deep as that, gain nothing.)  The sums are taken in the same order: the same bits.
    constexpr int HM = TM / 2, HN = TN / 2, G = HA + HB;     // blocks of a half; loads of half a stage
    constexpr int NP = KSTEPS * HM * HN;                     // matrix instructions of a phase
    constexpr int AR = KSTEPS * HM, BR = KSTEPS * HN;        // reads of a half
    constexpr int GB = 1;                                    // matrix instructions in front of a meeting
    static_assert(GROUPS_A % (2 * NWV) == 0 && GROUPS_B % (2 * NWV) == 0 && TM % 2 == 0 && TN % 2 == 0, "halves of whole loads and blocks");
    static_assert(LOADS == 2 * G && NP > GB, "two groups of loads a k-tile");
    v4u fa[2][HM][KSTEPS], fb[2][HN][KSTEPS];
    auto read_a = [&](unsigned st, int h, int j) {
      const int ks = j / HM, a = j % HM;
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[h][a][ks]) : "v"(rowA + st + xo[ks]), "n"((h * HM + a) * 32 * ROWB));
    };
    auto read_b = [&](unsigned st, int h, int j) {
      const int ks = j / HN, b = j % HN;
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[h][b][ks]) : "v"(rowB + st + xo[ks]), "n"((h * HN + b) * 32 * ROWB));
    };
    // all reads asked for have arrived; tied to the wait, so that no matrix instruction is moved above it
    auto arrived = [&](int a_half, int b_half) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (a_half >= 0) {
#pragma unroll
        for (int j = 0; j < AR; ++j) asm volatile("" : "+v"(fa[a_half][j % HM][j / HM]));
      }
      if (b_half >= 0) {
#pragma unroll
        for (int j = 0; j < BR; ++j) asm volatile("" : "+v"(fb[b_half][j % HN][j / HN]));
      }
    };
    auto meet = [&]() {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    auto phase = [&](int ah, int bh, auto behind) {          // behind(g): what follows matrix instruction g
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks)
#pragma unroll
        for (int a = 0; a < HM; ++a)
#pragma unroll
          for (int b = 0; b < HN; ++b) {
            floatx16& c = acc[ah * HM + a][bh * HN + b];
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[ah][a][ks]), __builtin_bit_cast(bf16x8, fb[bh][b][ks]), c, 0, 0, 0);
            behind((ks * HM + a) * HN + b);
            __builtin_amdgcn_sched_barrier(0);
          }
    };
#pragma unroll
    for (int t = 0; t < STAGES; ++t)
      if (t < n_k) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue_one(t, t * STAGE_BYTES, i);
      }
    if (n_k >= STAGES) wait_vmcnt<(2 * STAGES - 1) * G>();
    else wait_vmcnt<0>();
    meet();
    if (n_k > 0) {
#pragma unroll
      for (int j = 0; j < AR; ++j) read_a(0, 0, j);
#pragma unroll
      for (int j = 0; j < BR; ++j) read_b(0, 0, j);
      arrived(0, 0);
    }
    unsigned st = 0;                                         // where tile kt lies
    // LEFT: how many tiles follow tile kt (STAGES: at least STAGES)
    auto tile = [&](int kt, auto left) {
      constexpr int LEFT = decltype(left)::value;
      constexpr bool MORE = LEFT >= STAGES, AFTER = LEFT >= 1;
      const unsigned st_next = st == (STAGES - 1) * STAGE_BYTES ? 0 : st + STAGE_BYTES;
      // what has been asked for behind this tile's second group of loads, and behind the next tile's first
      constexpr int BEHIND_2 = 2 * (LEFT < STAGES - 1 ? LEFT : STAGES - 1) * G;
      constexpr int BEHIND_1 = AFTER ? (1 + 2 * (LEFT - 1 < STAGES - 2 ? LEFT - 1 : STAGES - 2) + (MORE ? 1 : 0)) * G : 0;
      auto at = [](int j, int count, int from) { return from + j * (NP / 2) / count; };      // reads behind the first half of a phase
      phase(0, 0, [&](int g) {
        if (g == GB) {
          __builtin_amdgcn_sched_barrier(0);
          wait_vmcnt<BEHIND_2>();
          meet();
        }
#pragma unroll
        for (int j = 0; j < BR; ++j)
          if (at(j, BR, GB) == g) read_b(st, 1, j);
        if (MORE) {
#pragma unroll
          for (int i = 0; i < G; ++i)
            if (GB + i * (NP - GB) / G == g) issue_one(kt + STAGES, st, i);
        }
      });
      arrived(-1, 1);
      phase(0, 1, [&](int g) {
#pragma unroll
        for (int j = 0; j < AR; ++j)
          if (at(j, AR, 0) == g) read_a(st, 1, j);
      });
      arrived(1, -1);
      phase(1, 0, [&](int g) {
        if (AFTER) {
          if (g == GB) {
            __builtin_amdgcn_sched_barrier(0);
            wait_vmcnt<BEHIND_1>();
            meet();
          }
#pragma unroll
          for (int j = 0; j < AR; ++j)
            if (at(j, AR, GB) == g) read_a(st_next, 0, j);
        }
        if (MORE) {
#pragma unroll
          for (int i = 0; i < G; ++i)
            if (GB + i * (NP - GB) / G == g) issue_one(kt + STAGES, st, G + i);
        }
      });
      phase(1, 1, [&](int g) {
        if (AFTER) {
#pragma unroll
          for (int j = 0; j < BR; ++j)
            if (at(j, BR, 0) == g) read_b(st_next, 0, j);
        }
      });
      if (AFTER) arrived(0, 0);
      st = st_next;
    };
    for (int kt = 0; kt + STAGES < n_k; ++kt) tile(kt, std::integral_constant<int, STAGES>{});
    last_tiles(n_k, tile, std::make_integer_sequence<int, STAGES>{});
  } else {
    constexpr int NR = TM + TN, NM = TM * TN;                  // fragment reads and matrix instructions of a k-step
    constexpr int GB = NM >= 8 ? 2 : 0;
    // matrix instructions of a k-tile that its loads are spread over: up to the barrier; where only one k-tile is ahead the
    // first quarter, so that the loads have the rest of the tile to arrive in
    constexpr int SPAN = STAGES == 2 ? NM : (KSTEPS - 1) * NM + GB + 1;
    v4u fa[2][TM], fb[2][TN];
    // fragment j of k-step ks of the stage at byte st
    auto read_one = [&](unsigned st, int ks, int set, int j) {
      const unsigned pa = rowA + st + xo[ks], pb = rowB + st + xo[ks];
#pragma unroll
      for (int a = 0; a < TM; ++a)
        if (a == j) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[set][a]) : "v"(pa), "n"(a * 32 * ROWB));
#pragma unroll
      for (int b = 0; b < TN; ++b)
        if (b == j - TM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[set][b]) : "v"(pb), "n"(b * 32 * ROWB));
    };
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
      if (t < n_k) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue_one(t, t * STAGE_BYTES, i);
      }
    if (n_k >= STAGES - 1) wait_vmcnt<(STAGES - 2) * LOADS>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    if (n_k > 0) {
#pragma unroll
      for (int j = 0; j < NR; ++j) read_one(0, 0, 0, j);
    }
    unsigned st = 0, st_new = (STAGES - 1) * STAGE_BYTES;      // where tile kt lies, where tile kt + STAGES - 1 goes
    // LEFT: how many tiles follow tile kt (STAGES: at least STAGES - 1)
    auto tile = [&](int kt, auto left) {
      constexpr int LEFT = decltype(left)::value;
      constexpr bool MORE = LEFT >= STAGES - 1, NEXT = LEFT >= 1;
      const unsigned st_next = st == (STAGES - 1) * STAGE_BYTES ? 0 : st + STAGE_BYTES;
      if constexpr (PREV && LEFT == 0) {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const int m = m0 + wm * (BM / WAVES_M) + a * 32 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3);
              const int n = n0 + wn * (BN / WAVES_N) + b * 32 + (lane & 31);
              prev[a][b][i] = ((const float*)out_)[(size_t)min(m, M - 1) * N + min(n, N - 1)];
            }
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ++ks) {
        const int set = ks & 1;
        constexpr int LAST = KSTEPS - 1;
        // this step's fragments have arrived (the next step's are asked for below); tied to the wait, so that no
        // matrix instruction is moved above it
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int a = 0; a < TM; ++a) asm volatile("" : "+v"(fa[set][a]));
#pragma unroll
        for (int b = 0; b < TN; ++b) asm volatile("" : "+v"(fb[set][b]));
#pragma unroll
        for (int g = 0; g < NM; ++g) {
          const int a = g / TN, b = g % TN;
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[set][a]),
                                                              __builtin_bit_cast(bf16x8, fb[set][b]), acc[a][b], 0, 0, 0);
          if (MORE) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
              if ((2 * i + 1) * SPAN / (2 * LOADS) == ks * NM + g) issue_one(kt + STAGES - 1, st_new, i);
          }
          if (ks < LAST) {
#pragma unroll
            for (int j = 0; j < NR; ++j)
              if (j * (NM - 1) / NR == g) read_one(st, ks + 1, set ^ 1, j);
          } else if (NEXT) {
            if (g == GB) {
              // the loads of the tiles behind kt + 1 may still be out
              __builtin_amdgcn_sched_barrier(0);
              wait_vmcnt<(MORE ? STAGES - 2 : LEFT >= 1 ? LEFT - 1 : 0) * LOADS>();
              __builtin_amdgcn_s_barrier();
              __builtin_amdgcn_sched_barrier(0);
            }
            if (g >= GB) {
#pragma unroll
              for (int j = 0; j < NR; ++j)
                if (GB + j * (NM - 1 - GB) / NR == g) read_one(st_next, 0, set ^ 1, j);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      st_new = st;
      st = st_next;
    };
    for (int kt = 0; kt + STAGES - 1 < n_k; ++kt) tile(kt, std::integral_constant<int, STAGES>{});
    last_tiles(n_k, tile, std::make_integer_sequence<int, STAGES - 1>{});
  }

  // acc[a][b][i]: row wm*(BM/WAVES_M) + a*32 + 8*(i/4) + 4*(lane/32) + i%4, column wn*(BN/WAVES_N) + b*32 + lane%32
  const int ccol = lane & 31, crow = (lane >> 5) * 4;
  if constexpr (EPI == TI_EPI_QKV_PREP) {
    // The tile goes to LDS in 32-bit (the stages are free now); then, head by head of the tile, eight
    // lanes finish a row of a q or k head (the arithmetic of the kernel that prepares whole steps; a
    // row's eight lanes read its angles and write its result as runs of consecutive bytes), and a
    // thread a dim of a v head.
    // (A tile of 256 columns goes in two ranges of 128, which is what LDS holds in 32-bit.)
    static_assert(BM % 64 == 0 && BM <= 256 && NWV == 8, "the first wavefronts look up a row each; 64 rows per pass of all eight");
    constexpr int COLS = BN < 128 ? BN : 128, RANGES = BN / COLS, WN = BN / WAVES_N;
    static_assert(BN % COLS == 0 && COLS % WN == 0, "a range is whole wavefronts' columns");
    constexpr int FS = COLS + 8;                            // row stride: the eight rows x eight lanes of a wavefront
                                                            // read 64 different banks
    static_assert(qkv_prep_lds(BM, BN) <= (160 << 10), "the 32-bit tile fits into LDS");
    float* ft = reinterpret_cast<float*>(smem);
#pragma unroll 1
    for (int range = 0; range < RANGES; ++range) {
    __syncthreads();
    if (RANGES == 1 || wn * WN / COLS == range) {
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int b = 0; b < TN; ++b)
            ft[(wm * (BM / WAVES_M) + a * 32 + (i >> 2) * 8 + crow + (i & 3)) * FS + wn * WN % COLS + b * 32 + ccol] = acc[a][b][i];
    }
    // each row's position, and where its key and value go
    int* s_page = reinterpret_cast<int*>(ft + BM * FS);     // [BM] page of the row's position, -1: none
    int* s_prow = s_page + BM;                              // [BM] row of the position in that page
    int* s_live = s_prow + BM;                              // [BM] block-table row (request) of the row, -1: none
    int* s_pos = s_live + BM;                               // [BM] position of the row
    const int hd = ep.hd, units = ep.n_head + 2 * ep.n_kv;
    if (tid < BM) {
      const int m = m0 + tid;
      const bool live = m < M;
      const int p = live ? ep.pos[m] : 0;
      // the host reserves pages first; a row without one (-1) writes nothing
      s_page[tid] = (live && ep.n_kv > 0) ? ep.table[(size_t)ep.slot[m] * ep.table_stride + p / ep.P] : -1;
      s_prow[tid] = p % ep.P;
      s_live[tid] = live ? ep.slot[m] : -1;
      s_pos[tid] = p;
    }
    __syncthreads();
    for (int hh = 0; hh < COLS / hd; ++hh) {
      const int u = (n0 + range * COLS) / hd + hh;           // the same in every thread
      if (u >= units) break;
      const bool is_q = u < ep.n_head, is_v = u >= ep.n_head + ep.n_kv;
      if (is_v) {
        // values go in transposed, [dim][row of the page]: thread -> one dim, for runs of 16 rows of
        // the tile; a run that is 16 consecutive rows of one page leaves as 32 contiguous bytes
        const int kvh = u - ep.n_head - ep.n_kv;
        const int d = tid % hd;
        for (int r0 = (tid / hd) * 16; r0 < BM; r0 += (NWV * 64 / hd) * 16) {
          const int pg = s_page[r0], pr = s_prow[r0];
          // rows of a run are consecutive positions of one request: its first and last row tell
          bool run = (pg >= 0) & (pr % 16 == 0) & (s_page[r0 + 15] == pg) & (s_prow[r0 + 15] == pr + 15) &
                     (s_live[r0] == s_live[r0 + 15]);
          const float* col = ft + r0 * FS + hh * hd + d;
          if (run) {
            float v[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = col[j * FS];
            bf16_t* dst = kv_page_slot<bf16_t>(ep.pool, pg, 1, kvh, pr, ep.n_kv, ep.P, hd) + (size_t)d * ep.P;
            *reinterpret_cast<uint4*>(dst) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                                        pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
            *reinterpret_cast<uint4*>(dst + 8) = make_uint4(pack_bf16x2(v[8], v[9]), pack_bf16x2(v[10], v[11]),
                                                            pack_bf16x2(v[12], v[13]), pack_bf16x2(v[14], v[15]));
          } else {
            for (int j = 0; j < 16; ++j) {
              const int pj = s_page[r0 + j];
              if (pj >= 0)
                kv_page_slot<bf16_t>(ep.pool, pj, 1, kvh, s_prow[r0 + j], ep.n_kv, ep.P, hd)[(size_t)d * ep.P] =
                    f2bf(col[j * FS]);
            }
          }
        }
        continue;
      }
      if (hd == 128)
        qkv_rows_by_lanes<128, BM, NWV, FS>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
      else
        qkv_rows_by_lanes<64, BM, NWV, FS>(ep, ft, s_pos, s_page, s_prow, s_live, hh, u, m0);
    }
    }
    return;
  }
  if constexpr (SW) {
    // Whole pieces of 16 bytes: a wavefront's results through LDS (the stages are free now), and out as runs of its columns.  (Two bytes a lane: 2,048
    // rows of 6144 x 1024 in tiles of 256 x 256 29.5 us, so 28.2; of 24576 x 4096 by four wavefronts 316 and 305; 512 rows in tiles of 128 x 128
    // 12.0 and 11.7.)
    if (N % 8 == 0 && ((uintptr_t)out_ & 15) == 0) {
      constexpr int ROWS = BM / WAVES_M, COLS = half, LDB = COLS * 2 + 16;      // a wavefront's part, and the bytes from row to row
      static_assert(NWV * ROWS * LDB <= STAGES * STAGE_BYTES && COLS % 8 == 0 && 64 % (COLS / 8) == 0, "it fits into the stages, rows of whole pieces");
      __syncthreads();
      unsigned char* mine = smem + wave * (ROWS * LDB);
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int b = 0; b < TN / 2; ++b)
            *reinterpret_cast<bf16_t*>(mine + (a * 32 + (i >> 2) * 8 + crow + (i & 3)) * LDB + (b * 32 + ccol) * 2) =
                f2bf(silu_mul(acc[a][b][i], acc[a][b + TN / 2][i]));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      constexpr int EACH = COLS / 8, PASS = 64 / EACH;       // lanes a row, rows a pass
      const int col = (lane % EACH) * 8, n = n0 + wn * COLS + col;
#pragma unroll
      for (int r0 = 0; r0 < ROWS; r0 += PASS) {
        const int r = r0 + lane / EACH, m = m0 + wm * ROWS + r;
        const uint4 v = *reinterpret_cast<const uint4*>(mine + r * LDB + col * 2);
        if (r < ROWS && m < M && n < N) *reinterpret_cast<uint4*>((bf16_t*)out_ + (size_t)m * N + n) = v;
      }
      return;
    }
  }
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int m = m0 + wm * (BM / WAVES_M) + a * 32 + (i >> 2) * 8 + crow + (i & 3);
      if (m >= M) continue;
      if (SW) {
#pragma unroll
        for (int b = 0; b < TN / 2; ++b) {
          const int n = n0 + wn * (BN / WAVES_N / 2) + b * 32 + ccol;
          if (n < N) ((bf16_t*)out_)[(size_t)m * N + n] = f2bf(silu_mul(acc[a][b][i], acc[a][b + TN / 2][i]));
        }
      } else {
#pragma unroll
        for (int b = 0; b < TN; ++b) {
          const int n = n0 + wn * (BN / WAVES_N) + b * 32 + ccol;
          if (n >= N) continue;
          const size_t o = (size_t)m * N + n;
          const float v = acc[a][b][i];
          if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = v;
          if constexpr (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] = (PREV ? prev[a][b][i] : ((const float*)out_)[o]) + v;
          if (TI_EPI_ACT(EPI)) ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(v));
        }
      }
    }
  }
#endif
}

// The order in which the dies take a product's tiles (see the kernel): rows = 0 is the grid's own, which deals the columns
// out to the dies where 8 divides them and mixes everything where not.
struct DieOrder {
  int rows = 0, die_rows = 1;
};
static int g_xcd_rows = 0;       // a hook for measurements: > 0 forces the group's rows (all rows to a die), -1 the grid's order
static int g_die_order = 1;      // a hook for measurements: 0: no blocks of rows
// A: bytes of the token rows, W: of the weight rows.  Large weights: an eighth of the columns to a die, in groups of eight row
// tiles.  In the grid's order every row tile pulls the whole weight from memory again once it is larger than the cache
// in front of the memory holds (256 MB; Qwen3-32B's gate/up and down over 2,048 rows, 524 and 262 MB: a prompt of 2,048
// tokens 9.6 % faster).  Otherwise the cut that brings the fewest bytes into the eight L2s, A / die_rows + W / die_cols each.
static DieOrder die_order(const dim3& grid, long A, long W) {
  DieOrder o;
  if (g_xcd_rows < 0) return o;
  if (g_xcd_rows > 0 || W >= (192L << 20)) {
    if (grid.x % 8 == 0) o.rows = g_xcd_rows > 0 ? g_xcd_rows : 8;
    return o;
  }
  if (!g_die_order) return o;
  long least = grid.x % 8 == 0 ? A + W / 8 : A + W;
  for (int r = 1; r <= 8; r *= 2) {
    if (grid.y % r || grid.x % (8 / r)) continue;
    const long bytes = A / r + W / (8 / r);
    if (bytes * 10 < least * 9) {
      least = bytes;
      o.rows = 8;
      o.die_rows = r;
    }
  }
  return o;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int EPI, int STAGES = PSTAGES, bool PHASED = false>
static int launch_pipelined(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda,
                            hipStream_t s, int ksplit = 1, int n_first = 0, int n_end = -1) {
  constexpr int bytes = STAGES * (BM + BN) * PBK * 2;
  auto kernel = gemm_pipelined_kernel<BM, BN, WAVES_M, WAVES_N, EPI, STAGES, PHASED>;
  static bool ready = false;          // per instantiation: allow more than 64 KiB of dynamic LDS
  if (!ready) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
      ti_set_error("gemm_bf16: cannot reserve %d bytes of LDS", bytes);
      return 2;
    }
    ready = true;
  }
  const int bn = (EPI == TI_EPI_SWIGLU) ? BN / 2 : BN;
  // columns [n_first, n_end) of the output (all of them by default); n_end short of N is a multiple of the tile
  if (n_end < 0) n_end = N;
  dim3 grid((n_end - n_first + bn - 1) / bn, (M + BM - 1) / BM, (EPI == TI_EPI_STORE_F32) ? ksplit : 1);
  const DieOrder o = die_order(grid, (long)M * K * 2, (EPI == TI_EPI_SWIGLU ? 2L : 1L) * N * K * 2);
  kernel<<<grid, WAVES_M * WAVES_N * 64, bytes, s>>>(A, W, out, M, N, K, lda, n_first, o.rows, o.die_rows, QKVEpilogue{});
  return 0;
}

static int g_tiles_160 = 1;      // a hook for measurements: 0 = no tiles of 160 columns
static int g_tiles_256 = 1;      // a hook for measurements: 0 = no tiles of 256 x 256
static int g_two_ranges = 1;     // a hook for measurements: 0 = never split the columns between two tile shapes
static int g_qkv_rows = 0;       // hooks for measurements: 64, 128 or 256 forces the tile's rows, 512 tiles of 256 x 256;
static int g_qkv_min_rows = 17;  // the fewest rows served (fewer take the kernels with the norm in front)

// What the pipelined kernel takes: k-tiles of 64, and rows whose offsets inside a tile fit its 32-bit load offsets.
static bool pipelined_serves(int K, long lda) { return K % PBK == 0 && K < (1 << 21) && lda < (1 << 21); }

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

template <int BM, int WAVES_M, int WAVES_N, int STAGES, int BN = 128, bool PHASED = false>
static int launch_qkv_prep(const void* A, const void* W, int M, int N, int K, long lda, const QKVEpilogue& ep,
                           hipStream_t stream, int n_first = 0, int n_end = -1) {
  constexpr int stages = STAGES * (BM + BN) * PBK * 2, bytes = stages > qkv_prep_lds(BM, BN) ? stages : qkv_prep_lds(BM, BN);
  auto kernel = gemm_pipelined_kernel<BM, BN, WAVES_M, WAVES_N, TI_EPI_QKV_PREP, STAGES, PHASED>;
  static bool ready = false;
  if (!ready) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
      ti_set_error("gemm_bf16_qkv_prep: cannot reserve %d bytes of LDS", bytes);
      return 2;
    }
    ready = true;
  }
  if (n_end < 0) n_end = N;               // columns [n_first, n_end): whole heads
  dim3 grid((n_end - n_first + BN - 1) / BN, (M + BM - 1) / BM);
  const DieOrder o = die_order(grid, (long)M * K * 2, (long)N * K * 2);
  kernel<<<grid, 512, bytes, stream>>>((const bf16_t*)A, (const bf16_t*)W, nullptr, M, N, K, lda, n_first, o.rows, o.die_rows, ep);
  return 0;
}

// for measurements: 0 = choose the tile by the shape, else a tile's id below
static int g_force_tile = 0;

// The tiles, and what one costs.  A launch is rounds of workgroups; a round lasts start + k-tiles x (each + fill x the share
// of the compute units that is busy), for workgroups alone on a unit and, where two fit in its LDS, for two.  The numbers
// (us, k-tiles of 64) are fitted to 300 products: 65 to 6,000 rows times the four weights of a layer of Qwen3-0.6B's, 1.7B's,
// 4B's and 8B's sizes, weights not in the caches, K also cut in two, four and eight.  The median error is 3 to 9 %, and the
// tile that is the cheapest by them is on average 0.8 % slower than the fastest (with K split 1.8 %, SwiGLU 0.9 %).
// Beyond what it was fitted to, 17 to 2,048 rows times the weights of Qwen3-14B's and 32B's sizes against the rules measured
// before it: 0 to 49 % faster (5120 x 25600 under 264 rows 206 -> 124 us), but for 200 rows times 32B's gate/up, 2 % slower,
// and for the runs of K under up to 64 rows, which ti_gemm_bf16_add_split therefore counts itself.  Inside the fit the worst
// seen against them is 2560 x 4096 under 264 to 300 rows, 21.7 -> 23.9 us.
// Fewer rows of A than a tile has cost what the whole tile costs.
struct TileRate {
  int id, bm, bn;
  float start1, each1, fill1;        // one workgroup to a unit
  float start2, each2, fill2;        // two (0: they do not fit)
};
static const TileRate TILES_PLAIN[] = {
    {1, 256, 128, 4.96f, 0.54f, 0.35f, 0.f, 0.f, 0.f},     {11, 256, 128, 6.58f, 0.55f, 0.30f, 0.f, 0.f, 0.f},
    {2, 128, 128, 3.25f, 0.39f, 0.16f, 0.f, 0.f, 0.f},     {4, 128, 64, 2.46f, 0.28f, 0.05f, 0.f, 0.f, 0.f},
    {3, 128, 64, 2.17f, 0.38f, 0.06f, 3.48f, 0.26f, 0.39f}, {6, 64, 64, 1.27f, 0.20f, 0.05f, 1.96f, 0.19f, 0.22f},
    {8, 128, 160, 4.98f, 0.51f, 0.13f, 0.f, 0.f, 0.f},     {9, 256, 160, 8.03f, 0.63f, 0.35f, 0.f, 0.f, 0.f}};
static const TileRate TILES_SWIGLU[] = {
    {1, 256, 128, 3.08f, 0.56f, 0.28f, 0.f, 0.f, 0.f},
    {2, 128, 128, 0.f, 0.54f, 0.05f, 0.f, 0.f, 0.f},       {7, 64, 128, 0.f, 0.40f, 0.03f, 0.f, 0.f, 0.f},
    {5, 64, 128, 0.f, 0.45f, 0.09f, 0.f, 0.55f, 0.20f},
    // by quarters, eight wavefronts and four
    {10, 256, 256, 5.76f, 0.93f, 0.60f, 0.f, 0.f, 0.f},    {12, 256, 256, 8.00f, 0.93f, 0.55f, 0.f, 0.f, 0.f}};
// Two SwiGLU ranges, of which the first goes by quarters as a rule, take more than their launches' costs by this share and this time.  Over 122 products, 200
// to 6,000 rows times the four sizes' gate/up, up to nine plans each in turns, what the costs choose is on average 0.5 % slower than the fastest, 1.6 % faster than
// the better of no tiles by quarters and only whole launches of them, and never slower than either beyond noise (without this share and time 0.65 % slower than
// so, 2048-wide gate/up under 1,650 to 1,792 and 3,000 to 3,300 rows by 2 to 5 %).  us, 256 x 256 in the older loop, quarters as whole launches alone, and
// so: 4B's gate/up under 800 and 1,000 rows 100 102 93, 106 110 99, under 1,650 176 176 165; 1.7B's under 1,300 77 79 74; 8B's under 650, 1,000, 1,300 and
// 2,304 rows 149 147 136, 179 177 168, 266 263 246, 395 396 373.
static const double RANGES_SHARE = 1.04, RANGES_US = 3.0;
static const double LAUNCH_US = 2.0;

static double tile_us(const TileRate& t, long workgroups, int k_tiles) {
  const long units = compute_units();
  const long round = t.each2 > 0.f ? 2 * units : units;
  const long full = workgroups / round, rest = workgroups % round;
  auto one = [&](double share) { return t.start1 + k_tiles * (t.each1 + t.fill1 * share); };
  auto two = [&](double share) { return t.start2 + k_tiles * (t.each2 + t.fill2 * share); };
  double us = full * (t.each2 > 0.f ? two(1.0) : one(1.0));
  if (rest) us += rest <= units ? one((double)rest / units) : two((double)rest / round);
  return us;
}

struct TileChoice {
  int id = 0;
  double us = 0.0;
  int n_big = 0;            // > 0: only that many rows of W, the others by tile `rest`
  int rest = 0;
};
// The cheapest tile for M rows times `rows` rows of W (for SwiGLU both halves), k_tiles deep, the launch `copies` times as
// large (K split).  two_ranges: also two launches, whole rounds of one tile and the columns left over in another.  quarters: SwiGLU by
// quarters as well, whole or for either range.
static TileChoice choose_tile(bool swiglu, int M, int rows, int k_tiles, int copies, bool two_ranges, bool quarters = false) {
  const TileRate* tiles = swiglu ? TILES_SWIGLU : TILES_PLAIN;
  const int n = swiglu ? (int)(sizeof(TILES_SWIGLU) / sizeof(TileRate)) : (int)(sizeof(TILES_PLAIN) / sizeof(TileRate));
  auto allowed = [&](const TileRate& t) { return t.bn == 160 ? g_tiles_160 != 0 : t.bn != 256 || (quarters && g_tiles_256); };
  auto row_tiles = [&](const TileRate& t) { return (long)((M + t.bm - 1) / t.bm); };
  auto us = [&](const TileRate& t, int r) { return LAUNCH_US + tile_us(t, row_tiles(t) * ((r + t.bn - 1) / t.bn) * copies, k_tiles); };
  TileChoice best;
  for (int i = 0; i < n; ++i) {
    if (!allowed(tiles[i])) continue;
    const double c = us(tiles[i], rows);
    if (!best.id || c < best.us) best = {tiles[i].id, c, 0, 0};
  }
  if (!two_ranges || !g_two_ranges || copies != 1) return best;
  for (int i = 0; i < n; ++i) {
    const TileRate& t = tiles[i];
    const long units = compute_units(), rt = row_tiles(t), all = rt * ((rows + t.bn - 1) / t.bn);
    if (!allowed(t) || t.each2 > 0.f || all < units || all % units == 0) continue;
    const int n_big = (int)(all / units * units / rt) * t.bn;
    if (n_big <= 0 || n_big >= rows) continue;
    const double first = us(t, n_big);
    for (int j = 0; j < n; ++j) {
      if (!allowed(tiles[j])) continue;
      double c = first + us(tiles[j], rows - n_big);
      if (quarters) c = c * RANGES_SHARE + RANGES_US;
      if (c < best.us) best = {t.id, c, n_big, tiles[j].id};
    }
  }
  return best;
}

// The tile of the q/k/v product that finishes its heads: of 64, 128 or 256 rows the one whose launch costs the least,
// 256-row tiles also as whole rounds of the units with the heads left over in 128-row tiles behind them (Qwen3-8B's 48 heads
// over 2,048 rows), beside the plain product in its own best tile followed by the kernel that prepares whole steps, which
// reads the product's 32-bit sums again.  Finishing the heads costs a tile about 3 us (512 rows of Qwen3-0.6B's sizes in
// tiles of 128 x 128: 18.9 us; of 64 x 128, on all units: 12).  Steps of up to 64 rows whose tiles leave most units idle
// always go to the product.
struct QKVChoice {
  int rows = 0;             // of a tile; 512: tiles of 256 x 256; 0: left to the product and the preparation kernel
  int n_big = 0;            // > 0: that many columns in 256-row tiles, the others in 128-row tiles
};
// Tiles of 256 x 256 read A and W the least, but every round of them ends with two ranges of heads, some 10 us: its start here.  Fitted to 128 products, 200 to
// 6,000 rows times q/k/v of 4096 to 10240 rows at K of 1,024 to 5,120 (median error 0.7 %); what is chosen is on average 0.1 % slower than the faster of
// this tile and the others' best, at worst 8 %.  us, the others and this tile: 6144 x 2560 under 2,048 rows 78 72, 3,000 117 134, 6,000 203 214; 6144 x 4096
// under 1,300 (product and preparation apart; this tile 97), 2,048 106 104, 6,000 288 313; 4096 x 2048 under 2,048 rows 38 57, 3,000 68 61, 6,000 106 121;
// 5120 x 2048 under 3,000 71 67; 4096 x 1024 under 4,096 48 44, 7168 x 5120 under 2,048 144 133, 10240 x 5120 under 3,500 360 374.
static const TileRate TILE_QKV_256 = {512, 256, 256, 16.1f, 0.91f, 0.61f, 0.f, 0.f, 0.f};
static QKVChoice qkv_choice(int M, int N, int K, bool wide_tiles) {
  QKVChoice c{g_qkv_rows, 0};
  if (c.rows) return c;                             // (a test asks for a tile)
  const long units = compute_units();
  const int k_tiles = K / PBK, col_tiles = (N + 127) / 128;
  auto us = [&](int rows, int cols) {               // (a tile of 64 x 128 does what one of 128 x 64 does)
    const int id = rows == 256 ? 1 : rows == 128 ? 2 : 4;
    const TileRate* t = TILES_PLAIN;
    while (t->id != id) ++t;
    return LAUNCH_US + 3.0 + tile_us(*t, (long)((M + rows - 1) / rows) * cols, k_tiles);
  };
  double least = us(64, col_tiles);
  c.rows = 64;
  for (int r = 128; r <= 256; r *= 2)
    if (us(r, col_tiles) < least) {
      least = us(r, col_tiles);
      c.rows = r;
    }
  const long row_tiles = (M + 255) / 256, big = row_tiles * col_tiles;
  if (g_two_ranges && big > units && big % units != 0) {
    const int cols = (int)(big / units * units / row_tiles);
    if (cols >= 1 && us(256, cols) + us(128, col_tiles - cols) < least) {
      least = us(256, cols) + us(128, col_tiles - cols);
      c = {256, cols * 128};
    }
  }
  // (the others' is the least of several costs, which is on average a fiftieth too low)
  if (wide_tiles && g_tiles_256) {
    const double wide = (LAUNCH_US + tile_us(TILE_QKV_256, row_tiles * ((N + 255) / 256), k_tiles)) / 1.02;
    if (wide < least) {
      least = wide;
      c = {512, 0};
    }
  }
  const double apart = choose_tile(false, M, N, k_tiles, 1, true).us + LAUNCH_US + 2.0 + 2.0 * M * N * 4 / 4.0e6;
  if (M <= 64 ? (long)((M + 127) / 128) * col_tiles * 2 < units : apart < least) c = {0, 0};
  return c;
}

// What the two rules choose, for tests: the tile of a product of N output columns (and, where the columns are split, the
// second tile and the column it begins at), the rows of the q/k/v product's tile (0: left to the product, and likewise).
extern "C" int ti_gemm_bf16_tile_choice(int swiglu, int M, int N, int K, int* rest, int* n_big) {
  const TileChoice c = choose_tile(swiglu != 0, M, swiglu ? 2 * N : N, K / PBK, 1, true);
  *rest = c.rest;
  *n_big = swiglu ? c.n_big / 2 : c.n_big;
  return c.id;
}
// ... where SwiGLU goes by quarters in its place, whole or in a range: likewise, 0 where it does not.
extern "C" int ti_gemm_bf16_quarters_ranges(int M, int N, int K, int* rest, int* n_big) {
  const TileChoice c = choose_tile(true, M, 2 * N, K / PBK, 1, true, true);
  *rest = c.rest;
  *n_big = c.n_big / 2;
  return c.id >= 10 || c.rest >= 10 ? c.id : 0;
}
extern "C" int ti_gemm_bf16_quarters_choice(int M, int N, int K) {
  int rest, n_big;
  return ti_gemm_bf16_quarters_ranges(M, N, K, &rest, &n_big);
}
extern "C" int ti_gemm_bf16_qkv_choice(int M, int N, int K, int* n_big) {
  const QKVChoice c = qkv_choice(M, N, K, false);
  *n_big = c.n_big;
  return c.rows;
}
// ... 1: tiles of 256 x 256 in its place.
extern "C" int ti_gemm_bf16_qkv_wide(int M, int N, int K) { return qkv_choice(M, N, K, true).rows == 512; }

// The fused q/k/v projection of a step's rows with the per-head work in its epilogue (see
// QKVEpilogue): A [M, K] bf16, W [(n_head + 2 n_kv) hd, K] bf16 (n_kv = 0: q heads only, nothing is
// written to the cache).  Returns 3 for what it does not serve: M <= 16, K not a multiple of 64,
// head sizes other than 64 and 128, and sizes at which the product and the preparation kernel cost
// less (qkv_choice).
extern "C" int ti_gemm_bf16_qkv_prep(const void* A, const void* W, int M, int K, long lda, const float* q_w,
                                     const float* k_w, float eps, const float* inv_freq, const float* rope_table,
                                     int table_len, const int* pos, const int* slot, const int* table,
                                     int table_stride, void* pool, void* q_out, int n_head, int n_kv, int hd,
                                     int page_size, hipStream_t stream) {
  TI_REQUIRE(M >= 0 && K > 0 && lda >= K && n_head > 0 && n_kv >= 0 && hd > 0 && page_size > 0 && table_stride > 0,
             "gemm_bf16_qkv_prep: bad sizes");
  if (M < g_qkv_min_rows || !pipelined_serves(K, lda) || lda % 8 != 0 || !(hd == 64 || hd == 128) || ((uintptr_t)A & 15) ||
      ((uintptr_t)W & 15) || ((uintptr_t)q_out & 15) || ((uintptr_t)pool & 15) || ((uintptr_t)rope_table & 15)) {
    ti_set_error("gemm_bf16_qkv_prep: M=%d K=%d head_dim=%d is not served (M > 16, K %% 64 == 0, head_dim 64 or 128)",
                 M, K, hd);
    return 3;
  }
  TI_REQUIRE(pos && slot && q_out && (n_kv == 0 || (table && pool)), "gemm_bf16_qkv_prep: a buffer is missing");
  TI_REQUIRE(inv_freq || !rope_table, "gemm_bf16_qkv_prep: a sin/cos table without inv_freq");
  QKVEpilogue ep{q_w, k_w, eps, inv_freq, (const float2*)rope_table, table_len, pos, slot, table, table_stride,
                 (bf16_t*)pool, (bf16_t*)q_out, n_head, n_kv, hd, page_size};
  const int N = (n_head + 2 * n_kv) * hd;
  const QKVChoice c = qkv_choice(M, N, K, true);
  if (!c.rows) {
    ti_set_error("gemm_bf16_qkv_prep: %d rows are left to the product and the preparation kernel", M);
    return 3;
  }
  int rc_;
  if (c.n_big) {
    rc_ = launch_qkv_prep<256, 4, 2, 3>(A, W, M, N, K, lda, ep, stream, 0, c.n_big);
    if (!rc_) rc_ = launch_qkv_prep<128, 4, 2, 4>(A, W, M, N, K, lda, ep, stream, c.n_big, N);
  } else if (c.rows == 512) {      // (256 x 256)
    rc_ = launch_qkv_prep<256, 2, 4, 2, 256, true>(A, W, M, N, K, lda, ep, stream);
  } else if (c.rows == 64) {
    rc_ = launch_qkv_prep<64, 2, 4, 4>(A, W, M, N, K, lda, ep, stream);
  } else if (c.rows == 128) {
    rc_ = launch_qkv_prep<128, 4, 2, 4>(A, W, M, N, K, lda, ep, stream);
  } else {
    rc_ = launch_qkv_prep<256, 4, 2, 3>(A, W, M, N, K, lda, ep, stream);
  }
  if (rc_) return rc_;
  TI_LAUNCH_CHECK();
  return 0;
}

template <int EPI>
static int launch_tile(int id, const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda, hipStream_t s,
                       int ksplit = 1, int n_first = 0, int n_end = -1) {
  constexpr bool SW = EPI == TI_EPI_SWIGLU;          // a SwiGLU wavefront needs two column tiles
  switch (id) {
    case 1: return launch_pipelined<256, 128, 4, 2, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
    case 2: return launch_pipelined<128, 128, 4, 2, EPI, 4>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
  }
  if constexpr (SW) {
    switch (id) {
      case 5: return launch_pipelined<64, 128, 2, 2, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 7: return launch_pipelined<64, 128, 2, 2, EPI, 4>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 10: return launch_pipelined<256, 256, 2, 4, EPI, 2, true>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 12: return launch_pipelined<256, 256, 2, 2, EPI, 2, true>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);     // for a long K
    }
    // (a forced tile that it does not have)
    return launch_pipelined<128, 128, 4, 2, EPI, 4>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
  } else {
    switch (id) {
      case 4: return launch_pipelined<128, 64, 2, 2, EPI, 4>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 6: return launch_pipelined<64, 64, 2, 2, EPI, 5>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 8: return launch_pipelined<128, 160, 4, 1, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 9: return launch_pipelined<256, 160, 4, 1, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
      case 11: return launch_pipelined<256, 128, 4, 1, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);      // for a long K
    }
    return launch_pipelined<128, 64, 2, 2, EPI>(A, W, out, M, N, K, lda, s, ksplit, n_first, n_end);
  }
}

template <int EPI>
static int launch_tiled_best(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda,
                             hipStream_t s) {
  constexpr bool SW = EPI == TI_EPI_SWIGLU;
  if (g_force_tile) return launch_tile<EPI>(g_force_tile, A, W, out, M, N, K, lda, s);
  const TileChoice c = choose_tile(SW, M, SW ? 2 * N : N, K / PBK, 1, true, SW);
  if (!c.n_big) return launch_tile<EPI>(c.id, A, W, out, M, N, K, lda, s);
  const int n_big = SW ? c.n_big / 2 : c.n_big;
  if (int rc = launch_tile<EPI>(c.id, A, W, out, M, N, K, lda, s, 1, 0, n_big)) return rc;
  return launch_tile<EPI>(c.rest, A, W, out, M, N, K, lda, s, 1, n_big, N);
}

// ------------------------------------------------------------------- dispatch
// Wavefronts per workgroup of the skinny kernel (4 or 8).  A product with few output columns
// has few workgroups (one per 16 columns); more wavefronts in each, splitting K further, keep
// more loads in flight.  0 = choose by the shape.
static int g_skinny_waves = 0;
// 1 (default): eight chunks of K in flight per wavefront where its share of K is more than four
static int g_skinny_deep = 1;

// rows within 2 GiB, which is what a buffer's descriptor spans
static bool staged_fits(int K, long lda) { return K % 64 == 0 && lda < (1L << 24) && K < (1 << 24); }
// Up to 16 rows of it as well (us, by rows in pieces, rows copied to LDS or a weight row a wavefront, and this; the same bits as the
// former two): 6144 x 4096 under 1 and 8 rows 12.5 13.9 -> 10.5 10.7, [gate; up] 24576 x 4096 34.1 37.5 -> 32.6 33.2, 4096 x 4096 8.9 9.9 ->
// 7.7 7.9, 4096 x 12288 20.7 22.0 -> 17.5 17.4, 2560 x 9728 14.8 17.0 -> 10.6 12.0, [gate; up] 6144 x 1024 5.2 5.3 -> 4.2 4.3,
// 151936 x 1024 52.8 61.0 -> 49.0 53.8.  But a weight of 288 Mi elements (576 MiB) and more keeps the pieces under up to
// 8 rows (151936 x 2048 104 and 117, here 112 and 122; 151936 x 4096 195 and 207, here 203 and 207).
static int g_rows_staged = 1;      // a hook for measurements: 0: up to 16 rows take the other kernels
static bool staged_16_serves(int M, int N, int K, long lda, int epi) {
  const long elements = (epi == TI_EPI_SWIGLU ? 2L * N : (long)N) * K;
  return g_rows_staged && M <= 16 && staged_fits(K, lda) && (M > 8 || elements < (288L << 20));
}
// Stages where a workgroup has four wavefronts, MT blocks of token rows and G of weight rows: as many as fit, up to all of 1,024 columns, where a workgroup
// has its compute unit for itself; two where that leaves room for a second workgroup and there is one.
constexpr int skinny_stages(int MT, int G, bool alone) {
  const int step = 4 * (MT + G) * 2048, most = 160 * 1024 / step;
  return !alone && 4 * step <= 160 * 1024 ? 2 : most < 4 ? most : 4;
}
template <int MT, int EPI, int NW, int STAGES, int G = 1>
static int launch_skinny_staged(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda, int grid, hipStream_t s) {
  constexpr int lds = NW * STAGES * (MT + G) * 2048;
  auto kernel = gemm_skinny_kernel<MT, EPI, NW, 4, STAGES, G>;
  static const hipError_t room = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  TI_REQUIRE(room == hipSuccess, "gemm_bf16: %d bytes of LDS: %s", lds, hipGetErrorString(room));
  kernel<<<(grid + G - 1) / G, NW * 64, lds, s>>>(A, W, out, M, N, K, lda);
  return 0;
}

// Groups of 16 weight rows a workgroup of the staged kernel takes: two where the busiest compute unit then pulls in clearly less (its
// workgroups' weight rows and, with each workgroup, all token rows).
// Bound by what a unit pulls in, about 50 bytes a nanosecond.  us, one group and two, weights not in the caches: [gate; up] 6144 x 1024
// at 17, 32, 48 and 64 rows 5.4 5.9 7.1 8.1 and 4.8 5.2 6.0 6.5 (three at 64 7.6); 6144 x 2560 at 20 and 64 10.6 16.9 and 9.2 13.0; [gate;
// up] 24576 x 4096 at 20 and 48 41.8 56.9 and 37.5 43.6.  Equal where the loads are no less: 4096 x 2048, a workgroup a unit either way, 6.3
// 8.5 and 6.7 9.5; up to 16 rows [gate; up] 24576 x 4096 34.1 and 37.6.
// Where sums are stored as they are, a short K is starts and ends: two groups only where fewer workgroups then follow one another on a unit (6144 x
// 256 at 17 and 64 rows, a turn either way, 2.80 3.76 and 3.07 3.77, 8192 x 64 2.23 2.71 and 2.41 3.12; 12288 x 256 at 48, two turns and one, 5.4 and
// 4.4, at 64, two either way, 6.3 and 6.5); from K = 640 on, 384 from 33 rows on, the bytes decide (6144 x 640 at 17 and 64 4.0 6.2 and 3.9 5.4).
// Row strides of 4 KiB and more that are powers of two cost two groups up to a fifth, and up to 32 rows they lose by it where they
// leave nearly every unit a workgroup: 8192 x 4096 at 17, 32 and 48 15.4 17.2 20.1 and 16.5 16.9 18.1, 8192 x 8192 28.3 32.6 37.8 and 34.1 34.5 36.0,
// [gate; up] 8192 x 2048 9.0 10.4 12.2 and 9.3 9.7 11.0.  Strides of 12, 20 and 24 KiB do not: no rule here.
static int g_skinny_groups = 0;      // a hook for measurements: 1 or 2 forces them
static int skinny_rounds(long groups, int G) { return (int)(((groups + G - 1) / G + compute_units() - 1) / compute_units()); }
// how many workgroups of G groups follow one another in a unit's place, as many side by side as its LDS holds
static int skinny_turns(int mt, long groups, int G) {
  const long n = (groups + G - 1) / G, units = compute_units();
  if (n <= units) return 1;
  const long beside = units * (160 * 1024 / (skinny_stages(mt, G, false) * 4 * (mt + G) * 2048));
  return (int)((n + beside - 1) / beside);
}
static int skinny_groups_for(int M, long groups, int K, bool swiglu) {
  const int mt = (M + 15) / 16;
  if (mt == 1) return 1;
  if (g_skinny_groups) return g_skinny_groups;
  if (!swiglu && K < (mt == 2 ? 640 : 384)) return skinny_turns(mt, groups, 2) < skinny_turns(mt, groups, 1) ? 2 : 1;
  return 20 * skinny_rounds(groups, 2) * (mt + 2) <= 17 * skinny_rounds(groups, 1) * (mt + 1) ? 2 : 1;
}
static int skinny_waves_for(int grid, int K);
template <int EPI>
static int launch_skinny(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda,
                          hipStream_t s) {
  const int grid = (EPI == TI_EPI_SWIGLU) ? (N + 7) / 8 : (N + 15) / 16;
  const int mt = (M + 15) / 16;
  int waves = g_skinny_waves;
  // by the weight's shape only, so that a row's bits do not depend on the rows beside it (up to 64 of them: above, where the tiles had
  // them and a row's bits changed too, four wavefronts are what LDS has room for); up to K = 4,096 and 16 rows as many as the
  // kernels with the norm in front take, so that those give the same bits
  if (waves == 0) waves = mt == 1 && K <= 4096 ? skinny_waves_for(grid, K) : (grid <= 128 && K >= 1024) ? 8 : 4;
  if (mt > 4) waves = 4;
  const bool staged = (mt > 1 && staged_fits(K, lda)) || staged_16_serves(M, N, K, lda, EPI);
  const int groups = waves == 4 ? skinny_groups_for(M, grid, K, EPI == TI_EPI_SWIGLU) : 1;
  const bool alone = (grid + groups - 1) / groups <= compute_units();
#define TI_GO(MTV, GV, ALONE) launch_skinny_staged<MTV, EPI, 4, skinny_stages(MTV, GV, ALONE), GV>(A, W, out, M, N, K, lda, grid, s)
#define TI_STAGED(MTV)                                                                             \
  if (mt == MTV && staged) {                                                                       \
    if (waves == 8) return launch_skinny_staged<MTV, EPI, 8, 2>(A, W, out, M, N, K, lda, grid, s); \
    if (MTV > 1 && groups == 2) return alone ? TI_GO((MTV > 1 ? MTV : 2), 2, true) : TI_GO((MTV > 1 ? MTV : 2), 2, false); \
    return alone ? TI_GO(MTV, 1, true) : TI_GO(MTV, 1, false);                                     \
  }
  TI_STAGED(1)
  TI_STAGED(2)
  TI_STAGED(3)
  TI_STAGED(4)
#undef TI_STAGED
  if constexpr (EPI != TI_EPI_ADD_F32) {
    constexpr int MORE = EPI == TI_EPI_SWIGLU ? 2 : 1;      // more than a round of single groups: [gate; up] alone (staged_112_serves)
#define TI_MORE(MTV) \
  if (mt == MTV) return groups == 2 ? TI_GO(MTV, MORE, true) : TI_GO(MTV, 1, true);
    TI_MORE(5)
    TI_MORE(6)
    TI_MORE(7)
#undef TI_MORE
  }
#undef TI_GO
#define TI_SKINNY(MTV)                                                               \
  if (mt == MTV) {                                                                   \
    if (waves == 8)                                                                  \
      gemm_skinny_kernel<MTV, EPI, 8><<<grid, 512, 0, s>>>(A, W, out, M, N, K, lda); \
    else                                                                             \
      gemm_skinny_kernel<MTV, EPI, 4><<<grid, 256, 0, s>>>(A, W, out, M, N, K, lda); \
  }
  // up to 16 tokens: a wavefront whose share of K is more than four chunks takes eight at a
  // time, so that one round trip to memory serves K up to 512 per wavefront
  if (mt == 1 && (K + 63) / 64 > 4 * waves && g_skinny_deep) {
    if (waves == 8)
      gemm_skinny_kernel<1, EPI, 8, 8><<<grid, 512, 0, s>>>(A, W, out, M, N, K, lda);
    else
      gemm_skinny_kernel<1, EPI, 4, 8><<<grid, 256, 0, s>>>(A, W, out, M, N, K, lda);
    return 0;
  }
  TI_SKINNY(1)
  TI_SKINNY(2)
  TI_SKINNY(3)
  TI_SKINNY(4)
#undef TI_SKINNY
  return 0;
}

template <int EPI>
static void launch_tiled(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda,
                         hipStream_t s) {
  const int bn = (EPI == TI_EPI_SWIGLU) ? TBN / 2 : TBN;
  dim3 grid((N + bn - 1) / bn, (M + TBM - 1) / TBM);
  gemm_tiled_kernel<EPI><<<grid, 256, 0, s>>>(A, W, out, M, N, K, lda);
}

// 1: the pipelined tiled kernel for M > 64 (default); 0: the plain tiled kernel (for comparison)
static int g_use_pipelined = 1;

// 17..64 rows: the kernels whose workgroups own 16 weight rows pull all token rows in once per 16
// rows, (1 + M / 16) times the weight's bytes through the caches.  Under a small weight that hides
// behind the launch; under a large one it is what the product waits for (Qwen3-8B's gate/up at 64
// rows: 110 us, 1.8 TB/s of weights), and the tiled kernels, which read the token rows once per
// 64 rows of the weight and take about the same time for 17 rows as for 64, are faster although
// their tile is partly empty (50 us).  Measured at the widths of Qwen3-0.6B to 8B: the tiled
// kernels win from about rows x weight elements = 280 Mi on.  13..16 rows: the 16-row kernels
// multiply without the matrix cores and under a large weight that is what they wait for (8B's
// gate/up at 16 rows: 72 us with the norm inside, 62 us as norm + tiled product; Qwen3-4B's: 50
// against 37 us); from rows x weight elements = 600 Mi on these take the tiled kernels too, and
// the norm a kernel of its own.  (At 9 to 12 rows that was measured as well, and loses.)
// With the rows through LDS the 16-row workgroups hold out longer where the product stores and is not cut over K (which it is into
// the residual, and from K = 4096 on): to 1000 Mi (us, tiles and 16-row workgroups: 6144 x 2560 at 64 rows, 960 Mi, 16.7 and 16.5, at 32
// 14.7 and 12.0; [gate; up] 12288 x 2048 at 48 rows, 1152 Mi, 17.8 and 16.3, at 64, 1536 Mi, 18.4 and 18.6; 19456 x 2560 at 17 rows,
// 807 Mi, 24.7 and 23.9, at 32, 1520 Mi, 26.4 and 28.7).  But every workgroup pulls in all token rows, and beyond one round of them (two to a
// unit at 64 rows) the tiles win again from 280 Mi on (weights that are not in the cache; 8192 x 2048 at 48 rows 12.3 and 11.9, 10240 x
// 2048 12.7 and 15.9, 12288 x 2048 at 24 12.7 and 14.2, 16000 x 1024 at 48 8.7 and 12.3).  [gate; up] tiles cost more, and lose up to three
// to a unit, up to 32 rows and from K above 2048 on (12288 x 1024 at 48 rows 10.5 and 10.2; 16000 x 1024 at 32 10.7 and 10.2, at 48 10.9 and 12.8).
static long g_tiled_from = 280L << 20;           // 17..64 rows x weight elements from which steps take the tiled kernels
static long g_tiled_from_16 = 600L << 20;        // the same for 13..16 rows
#define TILED_FROM_STORED (1000L << 20)
static long g_tiled_from_stored = TILED_FROM_STORED;      // the same for 17..64 rows whose product stores, K below 4096
static void set_tiled_from(long rows_times_elems) {
  g_tiled_from = g_tiled_from_stored = rows_times_elems;
  g_tiled_from_16 = rows_times_elems >= (280L << 20) && rows_times_elems < (1L << 59) ? rows_times_elems / 280 * 600
                                                                                     : rows_times_elems;
}
// 17..64 rows, a product that stores: whether the 16-row workgroups hold out to g_tiled_from_stored
static bool holds_out(int M, long rows, int K, int epi) {
  if (epi == TI_EPI_ADD_F32 || K >= 4096) return false;
  const long groups = (rows + 15) / 16;
  return epi == TI_EPI_SWIGLU ? groups <= 3L * compute_units() || M <= 32 || K > 2048 : groups <= 2L * compute_units();
}
static bool large_weight(int M, int N, int K, int epi) {
  const long rows = (epi == TI_EPI_SWIGLU) ? 2L * N : (long)N;
  if (M <= 12 || M > 64 || K % PBK != 0) return false;
  return rows * K * M >= (M <= 16 ? g_tiled_from_16 : holds_out(M, rows, K, epi) ? g_tiled_from_stored : g_tiled_from);
}
// 17 to 112 rows, a product that stores: whether the kernel with its rows through LDS takes it where the line above, or that of 64 rows,
// gave it to the tiles.  Up to 64 rows as long as two groups of weight rows a workgroup are one round of them (up to K = 4,095 the line
// above let one group have most of these; us, tiles and this: 2048 x 4096 at 48 and 64 rows 18.7 20.5 and 10.5 12.2, [gate; up] 4096 x 4096 at 40 and 64
// 27.9 30.4 and 12.1 14.7, 8192 x 4096 at 17, 32 and 64, stored in 16 bits, 18.9 19.8 23.3 and 16.5 16.9 19.4); beyond a round only [gate; up], whose tiles
// cost more (24576 x 4096 at 20, 40 and 64 44.1
// 44.5 45.6 and 37.5 42.0 49.8; 34816 x 5120 at 20, 40 and 64 89 93 100 and 71 85 106; 19456 x 2560 at 20, 32 and 40 25.7 27.1 27.5 and 24.1 25.8 27.9;
// 51200 x 5120, seven rounds, at 20 101.5 and 100.4; 12288 x 2048 without [gate; up] at 40 14.1 and 15.6).  32-bit sums of large weights from K =
// 4,096 on seldom come here up to 64 rows: a caller with a workspace asks ti_gemm_bf16_store_split first, which takes them in tiles that share K (with the
// adding kernel, and here, at 17, 33, 48 and 64 rows: 6144 x 4096 14.9 15.8 16.7 17.7 and 14.1 15.3 16.3 17.7, 8192 x 4096 16.5 17.2 18.0 19.2 and 16.7
// 17.5 18.3 19.4, 7168 x 5120 18.8 19.9 21.7 22.8 and 16.1 18.7 20.8 24.0, 4096 x 4096 from 33 on 11.3 11.5 11.9 and 10.5 12.0 13.7, 4096 x 12288 24.1
// 24.8 26.0 27.9 and 22.3 28.2 32.0 36.9: the tiles' cuts are ahead where it matters, and which shapes gain a tenth by leaving them is left).
// 65 to 112 rows, five to seven blocks of
// them beside the tiles' two row tiles: a round of workgroups of one group (4096 x 1024 at 65, 77 and 112 6.8 6.8 7.2 and 5.4 5.5 6.7; 4096 x
// 4096 17.6 17.9 19.6 and 14.2 14.7 18.3; 1024 x 1024 6.7 at 65, 6.9 at 112 and 5.1, 6.3) or, for [gate; up], two (6144 x 1024 9.1 9.2 10.0 and 6.9 7.0
// 8.7; 8192 x 2560 22.0 at 77, 23.8 at 100 and 15.6, 18.6); without [gate; up] two groups lose from 77 on (6144 x 2560 13.9
// and 14.5).  Measured at 256 to 8192 weight rows and K up to 32,768, where it stays ahead (4096 x 12288 at 65 and 112 46.6 57.7 and 39.6 52.2, 256 x 24576
// 83 100 and 64 91).  K of 256 and more, so that each of the four wavefronts has a chunk (1024 x 256 at 77 rows 3.6 and 2.7, 4096 x 256 4.1 and 3.3).
// The sums of four wavefronts, added in their order, are not the tiles' bits, which take K in ascending order in one; relative error of 32-bit results
// against 64 bits, tiles and this: 1024 x 1024 1.8e-7 and 0.95e-7, 4096 x 4096 4.0e-7 and 1.9e-7, 4096 x 12288 7.1e-7 and 3.4e-7.
static int g_rows_112 = 1;      // a hook for measurements: 0: only the line above
static bool staged_112_serves(int M, int N, int K, long lda, int epi) {
  if (!g_rows_112 || !g_use_pipelined || g_force_tile || g_tiled_from_stored != TILED_FROM_STORED || M <= 16 || M > 112 || epi == TI_EPI_ADD_F32 ||
      !staged_fits(K, lda) || (M > 64 && lda >= (1L << 23)))      // (112 rows within 2 GiB)
    return false;
  const long units = compute_units(), groups = epi == TI_EPI_SWIGLU ? (N + 7) / 8 : (N + 15) / 16;
  if (M > 64) return K >= 256 && groups <= (epi == TI_EPI_SWIGLU ? 2 : 1) * units;
  if (groups <= 2 * units) return true;
  const int rounds = skinny_rounds(groups, 2);
  return epi == TI_EPI_SWIGLU && rounds <= 5 && M <= (K >= 4096 || rounds == 2 ? 48 : 32);
}

// 1 (default): up to GR_MMAX tokens and a weight of fewer than GR_ROWS_BELOW rows take the kernel
// with a weight row per wavefront; 0: they take the kernels whose workgroups own 16 rows
#define GR_MMAX 8
#define GR_ROWS_BELOW 4096
static int g_row_per_wave = 1;
// Every workgroup (four weight rows) copies all M token rows into LDS: M / 4 times the bytes of its
// weight rows.  Up to four tokens that is no more than the weight itself; beyond, the kernel is taken
// only while its workgroups are no more than the compute units (Qwen3-0.6B's o and down, 1,024 rows: 4.7
// against 7.5 us at 8 tokens), not for more rows (Qwen3-4B's o, 2,560 x 4,096: 10.8 us here, 6.1 in
// workgroups of 16 rows; 1.7B's, 2,048 x 2,048: 3.9 against 3.0).
static bool row_per_wave_serves(int M, int N, int K, int epi) {
  // A weight of more than 8 Mi elements streams better with its rows through LDS stages (2048 x 6144 under 1 and 8 rows 9.4 and 11.0 us here,
  // 7.1 and 8.2 there); a smaller one is a matter of the chain of launches (o and down of 0.6B: a step of 1 request 775 us, there 829).
  if (g_rows_staged && K % 64 == 0 && (long)N * K > (8L << 20)) return false;
  return g_row_per_wave && M <= GR_MMAX && N < GR_ROWS_BELOW && (M <= 4 || N <= 4 * compute_units()) && K % 8 == 0 &&
         K <= 64 * 8 * GR_LOADS && (epi == TI_EPI_STORE_F32 || epi == TI_EPI_ADD_F32 || epi == TI_EPI_RELU2);
}

static int g_rows_direct = 1;     // a hook for measurements: 0: the rows of one and two tokens go through LDS too
template <int EPI, int MMAX, int NL>
static int launch_rows_mk(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda, hipStream_t s) {
  if constexpr (MMAX <= 2) {
    gemv_rows_direct_kernel<EPI, MMAX, NL><<<(N + 3) / 4, 256, 0, s>>>(A, W, out, M, N, K, lda);
  } else {
    constexpr int lds = (MMAX + 4) * NL * 1024;
    auto kern = gemv_rows_kernel<EPI, MMAX, NL>;
    static const hipError_t room = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TI_REQUIRE(room == hipSuccess, "gemm_bf16: %d bytes of LDS: %s", lds, hipGetErrorString(room));
    kern<<<(N + 3) / 4, 256, lds, s>>>(A, W, out, M, N, K, lda);
  }
  return 0;
}
template <int EPI, int MMAX>
static int launch_rows_m(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda, hipStream_t s) {
  if (K <= 1024) return launch_rows_mk<EPI, MMAX, 2>(A, W, out, M, N, K, lda, s);
  if (K <= 2048) return launch_rows_mk<EPI, MMAX, 4>(A, W, out, M, N, K, lda, s);
  if (K <= 3072) return launch_rows_mk<EPI, MMAX, 6>(A, W, out, M, N, K, lda, s);
  return launch_rows_mk<EPI, MMAX, GR_LOADS>(A, W, out, M, N, K, lda, s);
}
// the kernel is compiled for 1, 2, 4 and GR_MMAX tokens and four lengths of K; a row's bits are
// the same in all of them
template <int EPI>
static int launch_rows(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda, hipStream_t s) {
  if (M <= 1 && g_rows_direct) return launch_rows_m<EPI, 1>(A, W, out, M, N, K, lda, s);
  if (M <= 2 && g_rows_direct) return launch_rows_m<EPI, 2>(A, W, out, M, N, K, lda, s);
  if (M <= 4) return launch_rows_m<EPI, 4>(A, W, out, M, N, K, lda, s);
  return launch_rows_m<EPI, GR_MMAX>(A, W, out, M, N, K, lda, s);
}

template <class Producer, int EPI, int NW, int UN = 4>
static int launch_staged(const char* what, Producer producer, const bf16_t* w, void* out, int M, int N, int K,
                         int grid, hipStream_t stream) {
  const size_t lds = (size_t)M * (K + 8) * 2;
  auto kern = gemm_skinny_staged_kernel<Producer, EPI, NW, UN>;
  static size_t allowed = 48 * 1024;   // per instantiation: the largest size asked for so far
  if (lds > allowed) {
    TI_REQUIRE(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) ==
                   hipSuccess, "%s: LDS size refused", what);
    allowed = lds;
  }
  kern<<<grid, NW * 64, lds, stream>>>(producer, w, out, M, N, K);
  TI_LAUNCH_CHECK();
  return 0;
}

// The number of wavefronts the plain skinny kernel takes for this weight: the kernels that
// make their rows themselves take the same, so that they give the same bits.
// (not under a weight of 8 Mi elements or more: there the kernel that takes the token rows in pieces, four
// wavefronts, is faster: Qwen3-1.7B's down projection, 2,048 x 6,144, at 8 tokens 12.2 -> 9.2 us)
static int skinny_waves_for(int grid, int K) {
  return g_skinny_waves ? g_skinny_waves : ((grid <= 128 && K >= 1024 && (long)grid * K < (512L << 10)) ? 8 : 4);
}

static size_t normed_lds(int M, int K, int waves, int stages) { return (size_t)waves * stages * 2048 + (size_t)M * (K + 8) * 2; }
#define NORMED_LDS (160 << 10)
template <int KC, int EPI, int KW, int G, int ST>
static int launch_normed(const float* x, const float* nw, float eps, const bf16_t* w, void* out, int M, int N, int K, int tiles,
                         hipStream_t stream) {
  auto kernel = gemm_normed_kernel<KC, EPI, KW, G, ST>;
  static const hipError_t room = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, NORMED_LDS);
  TI_REQUIRE(room == hipSuccess, "gemm_bf16_normed: LDS size refused: %s", hipGetErrorString(room));
  kernel<<<(tiles + G - 1) / G, 64 * KW * G, normed_lds(M, K, KW * G, ST), stream>>>(x, w, M, N, K, eps, nw, out);
  TI_LAUNCH_CHECK();
  return 0;
}
static int g_normed_groups = 0;    // a hook for measurements: 1 to 3 groups of wavefronts in the product with the norm inside, 0: by the tiles
// Groups of four wavefronts: as many as a unit has tiles, three at most; with more two (us at 1, 4 and 8 rows of K = 1024, two and three groups:
// 16384 weight rows, four tiles a unit, 6.9 7.3 8.5 and 8.2 8.5 9.1).  Two workgroups of two groups share a unit only where their rows leave room, 16 KiB of
// them and less (at K = 1024 up to 7 rows, at 2048 up to 3); beyond four tiles a unit three groups would be ahead where they do not (20000 x 1024
// at 1, 4, 8 and 16 rows 8.8 9.2 11.3 13.0 and 9.1 9.4 9.8 11.3, [gate; up] 17920 x 1536 11.7 12.4 15.7 18.1 and 12.1 12.8 14.0 15.7), which is left.  A long K under two
// tiles a unit has three as well, for 96 KiB of weights under way instead of 64 (6144 x 4096 at 1 and 4 rows 12.2 13.0 with two, 11.3 12.0).
template <int KC, int EPI>
static int launch_normed_groups(const float* x, const float* nw, float eps, const bf16_t* w, void* out, int M, int N, int K, int tiles,
                                hipStream_t stream) {
  const int each = (tiles + compute_units() - 1) / compute_units();
  int groups = g_normed_groups ? g_normed_groups : each <= 1 ? 1 : each == 3 || (each == 2 && K > 3072) ? 3 : 2;
  if (groups == 3 && normed_lds(M, K, 12, 4) > NORMED_LDS) groups = 2;
  if (groups == 3) return launch_normed<KC, EPI, 4, 3, 4>(x, nw, eps, w, out, M, N, K, tiles, stream);
  if (groups == 2) return launch_normed<KC, EPI, 4, 2, 4>(x, nw, eps, w, out, M, N, K, tiles, stream);
  return launch_normed<KC, EPI, 4, 1, KC == 4 ? 4 : 8>(x, nw, eps, w, out, M, N, K, tiles, stream);
}

static bool pieces_serves(int M, int N, int K, int epi);
#define NORMED_WEIGHT_BELOW (40L << 20)   // weight elements from which the norm stays a kernel of its own
static long g_normed_weight_below = NORMED_WEIGHT_BELOW;
// out = rmsnorm(x; nw, eps) W^T for M <= 16 (see gemm_normed_kernel).  Returns 3 for what it leaves to the norm's kernel and the product's: M > 16,
// K not a multiple of 64 or above 4096, operands not 16-byte aligned, rows that do not fit into LDS beside 64 KiB of weights (M (K + 8) above
// 48 Ki: 16 rows of more than 3,064 columns, 12 of more than 4,088; 6144 x 4096 at 12 and 16 rows 15.5 16.5 us that way, 21.9 24.2 in the kernel
// that took them before this one), squared relu, and the weights that the rules below name.
extern "C" int ti_gemm_bf16_normed(const float* x, const float* nw, float eps, const void* W, void* out,
                                   int M, int N, int K, int epi, hipStream_t stream) {
  TI_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm_bf16_normed: bad sizes M=%d N=%d K=%d", M, N, K);
  if (M > 16 || K % 64 != 0 || K > 4096 || ((uintptr_t)W & 15) || ((uintptr_t)x & 15) || ((uintptr_t)nw & 15)) {
    ti_set_error("gemm_bf16_normed: M=%d K=%d is not served (M <= 16, K %% 64 == 0, K <= 4096)", M, K);
    return 3;
  }
  if (epi == TI_EPI_RELU2) {
    ti_set_error("gemm_bf16_normed: this epilogue is left to the norm's kernel and the product's");
    return 3;
  }
  if (normed_lds(M, K, 8, 4) > NORMED_LDS) {
    ti_set_error("gemm_bf16_normed: %d rows of %d columns do not fit beside the weights", M, K);
    return 3;
  }
  if (row_per_wave_serves(M, N, K, epi)) {
    // the plain product of these sizes takes another kernel, with another order of summation: the
    // caller norms first and takes that one too, so that the norm in front changes no bit
    ti_set_error("gemm_bf16_normed: M=%d N=%d is left to the kernel with a weight row per wavefront", M, N);
    return 3;
  }
  if (large_weight(M, N, K, epi) && g_use_pipelined) {
    ti_set_error("gemm_bf16_normed: M=%d times a weight of %d x %d is left to the tiled kernels", M, N, K);
    return 3;
  }
  // Every workgroup here norms all M rows for itself, which pulls as many bytes through the caches as
  // its share of the weight has.  Under a large weight the product alone gains more than the norm's own launch
  // costs (us at 1, 2, 4 and 8 rows, here and as norm and product: Qwen3-4B's gate/up, 50 M elements, 20.7 21.4 22.9 26.0 and 21.6 21.9
  // 22.2 22.5; 8B's, 100 M, 35.8 36.9 38.4 41.1 and 36.3 36.6 37.2 38.0; below the line [gate; up] 8192 x 4096, 34 M, 13.4 13.9 14.2 15.5 and 15.8
  // 16.0 16.6 16.8, Qwen3-1.7B's, 25 M, 12.0 12.1 12.3 12.8 and 13.1 13.3 13.4 13.4).
  if ((long)(epi == TI_EPI_SWIGLU ? 2 : 1) * N * K >= g_normed_weight_below && pieces_serves(M, N, K, epi)) {
    ti_set_error("gemm_bf16_normed: a weight of %d x %d is left to the norm's kernel and the product's", N, K);
    return 3;
  }
  if (M == 0) return 0;
  const bf16_t* w = (const bf16_t*)W;
  const int grid = (epi == TI_EPI_SWIGLU) ? (N + 7) / 8 : (N + 15) / 16;
  const int kc = (K + 255) / 256;
  const int waves = skinny_waves_for(grid, K);
#define TI_GNK(E, KCV)                                                                                                      \
  return waves == 8 ? launch_normed<KCV, E, 8, 1, 4>(x, nw, eps, w, out, M, N, K, grid, stream)                             \
                    : launch_normed_groups<KCV, E>(x, nw, eps, w, out, M, N, K, grid, stream);
#define TI_GN(E)                        \
  case E:                               \
    if (kc <= 4) TI_GNK(E, 4)           \
    else if (kc <= 8) TI_GNK(E, 8)      \
    else TI_GNK(E, 16)
  switch (epi) {
    TI_GN(TI_EPI_STORE_F32)
    TI_GN(TI_EPI_ADD_F32)
    TI_GN(TI_EPI_STORE_ACT)
    TI_GN(TI_EPI_SWIGLU)
    default:
      TI_REQUIRE(false, "gemm_bf16_normed: unknown epilogue %d", epi);
  }
#undef TI_GN
#undef TI_GNK
  return 0;
}

// 1 (default): up to 16 tokens with K a multiple of 64 up to 4096, the token rows are copied into
// LDS once per workgroup (see CopyProducer); 0: every wavefront fetches its fragments from memory
static int g_skinny_copy = 1;

template <int EPI>
static int launch_skinny_copied(const bf16_t* A, const bf16_t* W, void* out, int M, int N, int K, long lda,
                                hipStream_t s) {
  const int grid = (EPI == TI_EPI_SWIGLU) ? (N + 7) / 8 : (N + 15) / 16;
  int waves = g_skinny_waves;
  if (waves == 0) waves = (grid <= 128 && K >= 1024) ? 8 : 4;         // as the plain kernel: same bits
  const bool deep = K / 64 > 4 * waves && g_skinny_deep;
  CopyProducer pr{A, lda};
  if (waves == 8)
    return deep ? launch_staged<CopyProducer, EPI, 8, 8>("gemm_bf16", pr, W, out, M, N, K, grid, s)
                : launch_staged<CopyProducer, EPI, 8, 4>("gemm_bf16", pr, W, out, M, N, K, grid, s);
  return deep ? launch_staged<CopyProducer, EPI, 4, 8>("gemm_bf16", pr, W, out, M, N, K, grid, s)
              : launch_staged<CopyProducer, EPI, 4, 4>("gemm_bf16", pr, W, out, M, N, K, grid, s);
}

// ---------------------------------------------------------------------------------------------
// 17 to 64 rows: 16x16x32 MFMAs fed through LDS (staged_rows.h).  A workgroup takes 16 rows of W (16
// output columns; SwiGLU: 8 gate and 8 up rows) and a range of K; its four wavefronts take the
// 64-wide k-blocks of that range in turn, each block as MB + 1 blocks of rows (a lane's two pieces: 8 k at 8 (lane / 16) in the first
// and in the second half) and 2 MB MFMAs over all 16 MB rows of A.  (Operands straight from memory: 1024 x 3072 at 64 rows 6.0 us, now
// 4.5; 1024 x 2048 4.9, now 4.6; 2048 x 2048 7.1, now 5.3; up to 32 rows the same.)  The four wavefronts' sums meet in LDS, in the order 0..3.
// With a weight of few rows the launch would fill a fraction of the compute units and every
// workgroup would pull in all of A: then K is split over KS workgroups, which leave their sums
// in `partial` [KS][M][N], and gemm_partials_add_kernel adds them to the residual in the order
// 0..KS-1.  A row's bits do not depend on the other rows.
#define MBK_STAGES 2
#define MBK_STRIDE 20   // floats per row of the LDS tile: the 4 x 16 lanes of a store hit 64 banks

template <int MB, int EPI>
__global__ void __launch_bounds__(256)
gemm_mblocks_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ out_,
                    float* __restrict__ partial, int M, int N, int K, long lda) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  constexpr bool SW = (EPI == TI_EPI_SWIGLU);
  constexpr int TILE = SW ? 8 : 16;                          // output columns of a workgroup
  constexpr int BLOCKS = MB + 1, STAGES = MBK_STAGES, STAGED = STAGES * BLOCKS * 2048;
  static_assert(4 * STAGED >= 4 * MB * 16 * MBK_STRIDE * 4, "the sums fit into the stages");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float (*red)[MB * 16][MBK_STRIDE] = reinterpret_cast<float (*)[MB * 16][MBK_STRIDE]>(smem);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TILE;
  const int KS = gridDim.y, split = blockIdx.y;
  const int nb = K / 64;
  const int kb0 = (int)((long)nb * split / KS), kb1 = (int)((long)nb * (split + 1) / KS);

  // rows outside the matrices read a valid row; what they give is not stored
  unsigned voff[BLOCKS][2];
  const int lr = lane >> 3, piece = ((lane & 7) ^ lr) * 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    voff[0][h] = (unsigned)min((SW ? 0 : 8 * h) + lr, N - 1 - n0) * (unsigned)(K * 2) + piece;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) voff[1 + mb][h] = (unsigned)min(mb * 16 + 8 * h + lr, M - 1) * (unsigned)(lda * 2) + piece;
  }
  const auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
  const size_t k0 = (size_t)(kb0 + wave) * 64;
  const auto rsW = rows_at(W + (size_t)n0 * K + k0), rsU = rows_at(W + (size_t)(n0 + (SW ? N : 0)) * K + k0), rsA = rows_at(A + k0);
  unsigned char* mine = smem + wave * STAGED;
  const auto load = [&](int step, unsigned stage) {
#pragma unroll
    for (int i = 0; i < BLOCKS; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        auto* dst = (__attribute__((address_space(3))) void*)(mine + stage + i * 2048 + h * 1024);      // the same in every lane
        if (i > 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsA, dst, 16, voff[i][h], step * 4 * 128, 0, 0);
        else if (SW && h == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(rsU, dst, 16, voff[i][h], step * 4 * 128, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rsW, dst, 16, voff[i][h], step * 4 * 128, 0, 0);
      }
  };
  floatx4 acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = floatx4{0.f, 0.f, 0.f, 0.f};
  const unsigned at = (unsigned)(size_t)mine + r * 128;
  const int steps = kb0 + wave < kb1 ? (kb1 - kb0 - wave + 3) / 4 : 0;
  staged_steps<BLOCKS, STAGES, RowPieces>(steps, at + ((g ^ (r & 7)) << 4), at + (((g + 4) ^ (r & 7)) << 4), load, [&](const RowPieces* e) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, e[1 + mb].x), __builtin_bit_cast(bf16x8, e[0].x), acc[mb], 0, 0, 0);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, e[1 + mb].y), __builtin_bit_cast(bf16x8, e[0].y), acc[mb], 0, 0, 0);
  });
  __syncthreads();                                           // the stages are free
  // acc[mb][q]: row 16 mb + 4 g + q, column r
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int q = 0; q < 4; ++q) red[wave][mb * 16 + 4 * g + q][r] = acc[mb][q];
  __syncthreads();
  if (SW) {
    // thread -> a row and 4 of the 8 columns: gate in columns 0..7 of the tile, up in 8..15
    const int row = tid >> 1, c = (tid & 1) * 4;
    if (row >= MB * 16 || row >= M) return;
    float gt[4] = {0.f, 0.f, 0.f, 0.f}, up[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        gt[i] += red[w][row][c + i];
        up[i] += red[w][row][8 + c + i];
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n0 + c + i < N) ((bf16_t*)out_)[(size_t)row * N + n0 + c + i] = f2bf(silu_mul(gt[i], up[i]));
    return;
  }
  const int row = tid >> 2, c = (tid & 3) * 4;
  if (row >= MB * 16 || row >= M) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 4; ++w)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += red[w][row][c + i];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + c + i;
    if (n >= N) continue;
    const size_t o = (size_t)row * N + n;
    if (EPI == TI_EPI_ADD_F32 && KS > 1) partial[(size_t)split * M * N + o] = v[i];
    else if (EPI == TI_EPI_ADD_F32) ((float*)out_)[o] += v[i];
    else if (EPI == TI_EPI_STORE_F32) ((float*)out_)[o] = v[i];
    else ((bf16_t*)out_)[o] = f2bf(epi_act<EPI>(v[i]));
  }
#endif
}

// out[i] += partial[0][i] + ... + partial[KS - 1][i], in that order
__global__ void __launch_bounds__(256)
gemm_partials_add_kernel(float* __restrict__ out, const float* __restrict__ partial, int KS, size_t count) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float v = out[i];
  for (int s = 0; s < KS; ++s) v += partial[(size_t)s * count + i];
  out[i] = v;
}

// 17 to 64 rows times a weight of very many rows (the head: 151,936): the same MFMAs, but a
// workgroup keeps its share of A in registers (wavefront w of NW the k-blocks w, w + NW, ..., at
// most four) and walks over tiles of 16 weight rows, blockIdx.x, blockIdx.x + gridDim.x, ...: the
// weight streams through once, and A is read once per workgroup instead of once per tile (with a
// workgroup per tile the 9,496 tiles of the head pulled 1.2 GB of A through the caches: 170 us at
// 64 rows, against ~60 us for the weight alone).  The next tile's weight fragments are asked for
// before this tile is multiplied.  Stores 32-bit results; a row's bits do not depend on the others.
template <int MB, int NW>
__global__ void __launch_bounds__(64 * NW)
gemm_wide_rows_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, float* __restrict__ out, int M,
                      int N, int K, long lda) {
  constexpr int BPW = 4;                                     // k-blocks of 64 per wavefront at most
  __shared__ __attribute__((aligned(16))) float red[2][NW][MB * 16][MBK_STRIDE];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int r = lane & 15, g = lane >> 4;
  const int nb = K / 64, tiles = (N + 15) / 16;
  // this wavefront's k-blocks: block j is k-block wave + NW j (one past the end repeats the last
  // and is not multiplied)
  int kof[BPW];
  bool live[BPW];
#pragma unroll
  for (int j = 0; j < BPW; ++j) {
    live[j] = wave + NW * j < nb;
    kof[j] = min(wave + NW * j, nb - 1) * 64 + g * 8;
  }
  uint4 a[BPW][MB][2];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const bf16_t* arow = A + (size_t)min(mb * 16 + r, M - 1) * lda;
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      a[j][mb][0] = *reinterpret_cast<const uint4*>(arow + kof[j]);
      a[j][mb][1] = *reinterpret_cast<const uint4*>(arow + kof[j] + 32);
    }
  }
  auto load_w = [&](uint4 (&b)[BPW][2], int tile) {
    const bf16_t* wrow = W + (size_t)min(tile * 16 + r, N - 1) * K;
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      b[j][0] = *reinterpret_cast<const uint4*>(wrow + kof[j]);
      b[j][1] = *reinterpret_cast<const uint4*>(wrow + kof[j] + 32);
    }
  };
  int tile = blockIdx.x;
  if (tile >= tiles) return;
  uint4 cur[BPW][2];
  load_w(cur, tile);
  for (int it = 0; tile < tiles; ++it, tile += gridDim.x) {
    uint4 next[BPW][2];
    load_w(next, min(tile + (int)gridDim.x, tiles - 1));
    floatx4 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < BPW; ++j)
      if (live[j]) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[j][mb][h]),
                                                              __builtin_bit_cast(bf16x8, cur[j][h]), acc[mb], 0, 0, 0);
      }
    // the wavefronts' sums meet in LDS, in the order 0..NW-1; two buffers take turns, so that one
    // barrier a tile is enough (a wavefront two tiles ahead would have to pass the barrier between)
    float (*rd)[MB * 16][MBK_STRIDE] = red[it & 1];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int q = 0; q < 4; ++q) rd[wave][mb * 16 + 4 * g + q][r] = acc[mb][q];
    __syncthreads();
    for (int e = tid; e < MB * 16 * 4; e += 64 * NW) {
      const int row = e >> 2, c = (e & 3) * 4;
      if (row >= M) continue;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] += rd[w][row][c + i];
      const int n = tile * 16 + c;
      float* dst = out + (size_t)row * N + n;
      if (n + 3 < N && (N & 3) == 0) {
        *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) dst[i] = v[i];
      }
    }
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      cur[j][0] = next[j][0];
      cur[j][1] = next[j][1];
    }
  }
}

static int g_wide_rows = 1;      // a hook for measurements: 0: the kernel above serves nothing
#define WIDE_ROWS_MIN_N 16384

// whether gemm_wide_rows_kernel takes the product (storing 32-bit results)
static int g_wide_rows_min_n = WIDE_ROWS_MIN_N, g_wide_rows_grid = 0;     // hooks for measurements
static bool wide_rows_serves(int M, int N, int K, int epi) {
  return g_wide_rows && epi == TI_EPI_STORE_F32 && M > 16 && M <= 64 && N >= g_wide_rows_min_n && K % 64 == 0 &&
         K / 64 <= 4 * 8;
}

static void launch_wide_rows(const bf16_t* a, const bf16_t* w, float* out, int M, int N, int K, long lda,
                             hipStream_t s) {
  const int mb = (M + 15) / 16, tiles = (N + 15) / 16;
  const bool eight = K / 64 > 4 * 4;                         // more than 16 k-blocks: eight wavefronts
  int dev = 0, units = 256;
  hipDeviceProp_t prop;
  static int cached_units = 0;
  if (!cached_units) {
    if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) units = prop.multiProcessorCount;
    cached_units = units > 0 ? units : 256;
  }
  const int grid = g_wide_rows_grid > 0 ? min(tiles, g_wide_rows_grid) : min(tiles, cached_units);
#define TI_GO(MBV)                                                                                   \
  if (eight) gemm_wide_rows_kernel<MBV, 8><<<grid, 512, 0, s>>>(a, w, out, M, N, K, lda);            \
  else gemm_wide_rows_kernel<MBV, 4><<<grid, 256, 0, s>>>(a, w, out, M, N, K, lda)
  if (mb == 2) { TI_GO(2); }
  else if (mb == 3) { TI_GO(3); }
  else { TI_GO(4); }
#undef TI_GO
}

template <int EPI, int AV, bool SPLIT>
static int launch_pieces_av(const bf16_t* a, long lda, const bf16_t* w, void* out, float* partial, int M, int N, int K,
                            int KS, hipStream_t s) {
  const size_t lds = (size_t)2 * M * SP_LD * 2;
  auto kern = gemm_skinny_pieces_kernel<EPI, AV, SPLIT>;
  static size_t allowed = 48 * 1024;
  if (lds > allowed) {
    TI_REQUIRE(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess,
               "gemm_bf16: LDS size refused");
    allowed = lds;
  }
  const int tile = (EPI == TI_EPI_SWIGLU) ? 8 : 16;
  kern<<<dim3((N + tile - 1) / tile, KS), 256, lds, s>>>(a, lda, w, out, partial, M, N, K);
  return 0;
}
template <int EPI, bool SPLIT>
static int launch_pieces(const bf16_t* a, long lda, const bf16_t* w, void* out, float* partial, int M, int N, int K, int KS,
                         hipStream_t s) {
  if (M <= 2) return launch_pieces_av<EPI, 1, SPLIT>(a, lda, w, out, partial, M, N, K, KS, s);
  if (M <= 4) return launch_pieces_av<EPI, 2, SPLIT>(a, lda, w, out, partial, M, N, K, KS, s);
  if (M <= 8) return launch_pieces_av<EPI, 4, SPLIT>(a, lda, w, out, partial, M, N, K, KS, s);
  return launch_pieces_av<EPI, 8, SPLIT>(a, lda, w, out, partial, M, N, K, KS, s);
}

// 1 (default): up to 16 rows times a weight whose K is a multiple of 64 and at least two pieces long
// take the kernel with the token rows in pieces; 0: the kernels above it (for comparison)
static int g_pieces = 1;
static bool pieces_serves(int M, int N, int K, int epi) {
  if (!g_pieces || M > 16 || K % 64 != 0 || K < 2 * SP_PIECE) return false;
  if ((epi < TI_EPI_STORE_F32 || epi > TI_EPI_SWIGLU) && epi != TI_EPI_RELU2) return false;
  // few tokens times a weight of few rows: a row per wavefront wins (and fills the compute units)
  if (row_per_wave_serves(M, N, K, epi)) return false;
  // where the kernels with the norm in front (K up to 4,096) take eight wavefronts, this one would give other bits
  const int grid = (epi == TI_EPI_SWIGLU) ? (N + 7) / 8 : (N + 15) / 16;
  return K > 4096 || skinny_waves_for(grid, K) == 4;
}
// Into how many workgroups the pieces of K go when the product adds into the residual: a long K under
// few rows of weight leaves a launch of few workgroups that each walk a long way (Qwen3-32B's down
// projection: 320 workgroups, 25 pieces each, 3.1 TB/s; split four ways 4.8 TB/s).  By the weight's
// shape alone, so that a row's bits do not depend on the rows beside it.
static int pieces_splits(int N, int K, long partial_bytes) {
  const int n_pieces = (K + SP_PIECE - 1) / SP_PIECE;
  if (n_pieces < 16) return 1;      // (from 8 pieces on: Qwen3-4B's and 8B's down projections lose 1-3 % of the step)
  const int grid = (N + 15) / 16;
  int ks = std::min(n_pieces / 4, (4 * compute_units() + grid - 1) / grid);
  while (ks > 1 && (long)ks * 16 * N * 4 > partial_bytes) --ks;
  return ks < 1 ? 1 : ks;
}

static int g_add_split = 1;        // a hook for measurements: 0: ti_gemm_bf16_add_split serves nothing

// Elements from which up to 64 rows times a weight cut K by the weight's bytes and not by the tiles' cost.  Below it the cost
// is right or better (4096 x 4096 at 24 rows: 12.3 us in four runs, 14.0 in eight), from here on it is slower or the same.
#define STREAMED_WEIGHT (24L << 20)

template <int EPI>
static int launch_mblocks(const bf16_t* a, const bf16_t* w, void* out, float* partial, int M, int N, int K,
                           long lda, int KS, hipStream_t s) {
  const int tile = (EPI == TI_EPI_SWIGLU) ? 8 : 16;
  dim3 grid((N + tile - 1) / tile, KS);
  const int mb = (M + 15) / 16;
  const int lds = 4 * MBK_STAGES * (mb + 1) * 2048;
  if (mb == 1) gemm_mblocks_kernel<1, EPI><<<grid, 256, lds, s>>>(a, w, out, partial, M, N, K, lda);
  else if (mb == 2) gemm_mblocks_kernel<2, EPI><<<grid, 256, lds, s>>>(a, w, out, partial, M, N, K, lda);
  else if (mb == 3) gemm_mblocks_kernel<3, EPI><<<grid, 256, lds, s>>>(a, w, out, partial, M, N, K, lda);
  else {
    static const hipError_t room = hipFuncSetAttribute((const void*)gemm_mblocks_kernel<4, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    TI_REQUIRE(room == hipSuccess, "gemm_bf16: %d bytes of LDS: %s", lds, hipGetErrorString(room));
    gemm_mblocks_kernel<4, EPI><<<grid, 256, lds, s>>>(a, w, out, partial, M, N, K, lda);
  }
  return 0;
}

// out[i] += partial[0][i] + ... + partial[KS - 1][i] for count elements: what a product with a split
// K leaves to do (see ti_gemm_bf16_add_split)
extern "C" int ti_gemm_bf16_partials_add(float* out, const float* partial, int KS, long count, hipStream_t stream) {
  TI_REQUIRE(KS >= 1 && count >= 0, "gemm_bf16_partials_add: bad sizes KS=%d count=%ld", KS, count);
  if (count == 0) return 0;
  gemm_partials_add_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>(out, partial, KS, (size_t)count);
  TI_LAUNCH_CHECK();
  return 0;
}

// The product that adds into the 32-bit residual, for steps of more than 16 rows whose launch would
// leave most compute units idle (few rows times a weight of few rows): K is split over workgroups,
// which leave their sums in `partial` [KS][M][N] (workspace of partial_bytes).  17..64 rows:
// gemm_mblocks_kernel (measured against the kernels without MFMA at 64 rows: 1024 x 3072 19.7 ->
// 9.7 us with the addition of the partial sums as a kernel of its own, ~6 us without).  More rows, and
// 17..64 under a large weight: the pipelined kernel, storing, in the tile that costs the least.
// Up to 16 rows: the kernel with the token rows in pieces, where pieces_splits says so.
// defer = 0: the partial sums are added to `out` here, and only what gains even so is served.
// defer = 1: they are left in `partial`, *splits gets their number, and the caller sees to the
// addition (ti_gemm_bf16_partials_add, or a kernel that reads the residual next and adds them on
// the way).  defer = 2: what defer = 1 serves, added here (the same bits).  Returns 3 for what
// it does not serve.
extern "C" int ti_gemm_bf16_add_split(const void* A, const void* W, void* out, int M, int N, int K, long lda, int epi,
                                    void* partial, long partial_bytes, int defer, int* splits, hipStream_t stream) {
  TI_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm_bf16_add_split: bad sizes M=%d N=%d K=%d lda=%ld", M, N, K, lda);
  TI_REQUIRE(splits != nullptr, "gemm_bf16_add_split: splits must point to an int");
  *splits = 0;
  if (M <= 16 && M > 0 && g_add_split && epi == TI_EPI_ADD_F32 && partial && lda % 8 == 0 && !((uintptr_t)A & 15) &&
      !((uintptr_t)W & 15) && !((uintptr_t)partial & 15) && pieces_serves(M, N, K, epi)) {
    const int ks = pieces_splits(N, K, partial_bytes);
    if (ks > 1) {
      int rc_ = launch_pieces<TI_EPI_ADD_F32, true>((const bf16_t*)A, lda, (const bf16_t*)W, out, (float*)partial, M, N, K, ks,
                                                    stream);
      if (rc_) return rc_;
      if (defer == 1) {
        *splits = ks;
      } else {
        const size_t count = (size_t)M * N;
        gemm_partials_add_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>((float*)out, (const float*)partial,
                                                                                    ks, count);
      }
      TI_LAUNCH_CHECK();
      return 0;
    }
  }
  int KS = 1, tile = 0;      // (tile: of the pipelined kernel, 0: not taken)
  const bool small = M <= 64 && lda < (1L << 24) && !(large_weight(M, N, K, epi) && g_use_pipelined);
  if (g_add_split && epi == TI_EPI_ADD_F32 && partial && M > 16 && K % 64 == 0 && lda % 8 == 0 &&
      !((uintptr_t)A & 15) && !((uintptr_t)W & 15) && !((uintptr_t)partial & 15) && (small || g_use_pipelined)) {
    const int nb = K / 64;
    if (small) {
      // split K until the launch has about a workgroup per compute unit
      const long tiles = (N + 15) / 16;
      while (KS < 8 && tiles * KS * 2 <= compute_units() && nb / (KS * 2) >= 4) KS *= 2;
      while (KS > 1 && (long)KS * M * N * 4 > partial_bytes) KS /= 2;
      // with the addition as a kernel of its own, only large products gain
      if (!defer && !((long)M * K >= 128 * 1024 || (K >= 3072 && (long)M * K >= 96 * 1024))) KS = 1;
    } else if (pipelined_serves(K, lda) && M <= 64 && (long)N * K >= STREAMED_WEIGHT) {
      // Up to 64 rows times a weight that is waited for from memory: about four workgroups of 64 x 64 per unit, so that
      // enough of it is on its way at any time, as long as the sums stay a small part of its bytes.  The costs below know
      // nothing of a weight's bytes and cut such a K in four (us at 32 rows, eight runs and four: 5120 x 25600 56.6 and
      // 65.4, 5120 x 17408 40.3 and 45.9, 5120 x 8192 26.3 and 27.8).
      const long tiles = (N + 63) / 64;
      while (KS < 8 && tiles * KS * 2 <= 4L * compute_units() && nb / (KS * 2) >= 4 && (long)KS * 2 * M * 16 <= K) KS *= 2;
      while (KS > 1 && (long)KS * M * N * 4 > partial_bytes) KS /= 2;
      if (!defer && KS < 4) KS = 1;
      if (KS > 1) tile = choose_tile(false, M, N, nb / KS, KS, false).id;
    } else if (pipelined_serves(K, lda)) {
      // A product of few tiles, a short loop each, leaves units idle: K split between workgroups fills them, and the sums
      // cost their bytes once more where they are added (by the norm behind, or a kernel of its own).  Split as many
      // ways as tile and sums together are the cheapest (512 x 1024 x 3072: 13 us whole, 9.5 in two; the norm 0.6 more).
      // One way means that the sums of whole tiles are left to the norm, which spares the product the wait for the
      // residual behind its last k-tile; only where few tiles of many rows leave it short of other work (o and down of a
      // whole prompt at small widths).
      const double sums = (double)M * N * 4 / 10e6;      // us: the norm reads them at about 10 TB/s, out of the caches
      const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
      const bool few = defer && M >= 256 && tiles128 * 2 <= compute_units();
      double least = choose_tile(false, M, N, nb, 1, true).us + 1.5;
      for (int ks = few ? 1 : 2; ks <= 8; ks *= 2) {
        if (nb / ks < 4 || (long)ks * M * N * 4 > partial_bytes) break;
        const TileChoice c = choose_tile(false, M, N, nb / ks, ks, false);
        const double us = c.us + ks * sums + (defer ? 1.0 : 4.0 + 2 * sums);
        if (us < least || (few && !tile)) {
          least = us;
          KS = ks;
          tile = c.id;
        }
      }
    }
  }
  if (KS == 1 && !tile) {
    ti_set_error("gemm_bf16_add_split: serves more than 16 rows added into a product of few tiles, K a multiple of 64");
    return 3;
  }
  if (small) {
    int rc_ = launch_mblocks<TI_EPI_ADD_F32>((const bf16_t*)A, (const bf16_t*)W, out, (float*)partial, M, N, K, lda, KS, stream);
    if (rc_) return rc_;
  } else {
    int rc_ = launch_tile<TI_EPI_STORE_F32>(tile, (const bf16_t*)A, (const bf16_t*)W, partial, M, N, K, lda, stream, KS);
    if (rc_) return rc_;
  }
  if (defer == 1) {
    *splits = KS;
  } else {
    const size_t count = (size_t)M * N;
    gemm_partials_add_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>((float*)out, (const float*)partial,
                                                                                KS, count);
  }
  TI_LAUNCH_CHECK();
  return 0;
}

// the kernel with the token rows in pieces alone, for tests and measurements: any epilogue, 1..16
// rows, K a multiple of 64 split ks ways (1: not split; partial sums are added here)
extern "C" int ti_gemm_bf16_pieces_any(const void* A, const void* W, void* out, int M, int N, int K, long lda, int epi,
                                       void* partial, int ks, hipStream_t stream) {
  TI_REQUIRE(M > 0 && M <= 16 && N > 0 && K > 0 && K % 64 == 0 && lda >= K && lda % 8 == 0 && ks >= 1 &&
                 ks <= (K + SP_PIECE - 1) / SP_PIECE,
             "gemm_bf16_pieces_any: bad sizes M=%d N=%d K=%d lda=%ld ks=%d", M, N, K, lda, ks);
  TI_REQUIRE(ks == 1 || (epi == TI_EPI_ADD_F32 && partial), "gemm_bf16_pieces_any: a split K needs the adding epilogue");
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  int rc = 0;
  switch (epi) {
    case TI_EPI_STORE_F32: rc = launch_pieces<TI_EPI_STORE_F32, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
    case TI_EPI_STORE_ACT: rc = launch_pieces<TI_EPI_STORE_ACT, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
    case TI_EPI_RELU2: rc = launch_pieces<TI_EPI_RELU2, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
    case TI_EPI_SWIGLU: rc = launch_pieces<TI_EPI_SWIGLU, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
    case TI_EPI_ADD_F32:
      if (ks == 1) {
        rc = launch_pieces<TI_EPI_ADD_F32, false>(a, lda, w, out, nullptr, M, N, K, 1, stream);
      } else {
        rc = launch_pieces<TI_EPI_ADD_F32, true>(a, lda, w, out, (float*)partial, M, N, K, ks, stream);
        const size_t count = (size_t)M * N;
        gemm_partials_add_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>((float*)out, (const float*)partial,
                                                                                    ks, count);
      }
      break;
    default:
      TI_REQUIRE(false, "gemm_bf16_pieces_any: unknown epilogue %d", epi);
  }
  if (rc) return rc;
  TI_LAUNCH_CHECK();
  return 0;
}

// out[i] = partial[0][i] + ... + partial[KS - 1][i], in that order
__global__ void __launch_bounds__(256)
gemm_partials_sum_kernel(float* __restrict__ out, const float* __restrict__ partial, int KS, size_t count) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float v = partial[i];
  for (int s = 1; s < KS; ++s) v += partial[(size_t)s * count + i];
  out[i] = v;
}

// The product that stores 32-bit results, for 17 to 64 rows times a large weight whose 64 x 64 tiles
// are few (the q/k/v projection of a decode step of many requests with a large model: 96 to 160
// workgroups that wait for the weight from memory with too little of it under way).  K is split over
// four or eight workgroups a tile, which store their sums into `partial` [KS][M][N]; a kernel of its
// own adds them up into `out` (Qwen3-8B's q/k/v at 64 rows: 27 -> 17 us).  The number of shares
// depends on the weight's shape alone.  Returns 3 for what it does not serve.
extern "C" int ti_gemm_bf16_store_split(const void* A, const void* W, void* out, int M, int N, int K, long lda,
                                        void* partial, long partial_bytes, hipStream_t stream) {
  TI_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm_bf16_store_split: bad sizes M=%d N=%d K=%d lda=%ld", M, N, K, lda);
  int KS = 1;
  if (g_add_split && g_use_pipelined && partial && M > 16 && M <= 64 && pipelined_serves(K, lda) && lda % 8 == 0 &&
      !((uintptr_t)A & 15) && !((uintptr_t)W & 15) && !((uintptr_t)partial & 15) &&
      large_weight(M, N, K, TI_EPI_STORE_F32) && !wide_rows_serves(M, N, K, TI_EPI_STORE_F32)) {
    const long tiles = (N + 63) / 64;
    const int nb = K / 64;
    while (KS < 8 && tiles * KS * 2 <= 4L * compute_units() && nb / (KS * 2) >= 4 && (long)KS * 2 * 64 * 16 <= K) KS *= 2;
    while (KS > 1 && (long)KS * M * N * 4 > partial_bytes) KS /= 2;
  }
  if (KS < 4) {
    ti_set_error("gemm_bf16_store_split: serves 17 to 64 rows times a large weight of few tiles, K a multiple of 64");
    return 3;
  }
  int rc_ = launch_tile<TI_EPI_STORE_F32>(6, (const bf16_t*)A, (const bf16_t*)W, partial, M, N, K, lda, stream, KS);
  if (rc_) return rc_;
  const size_t count = (size_t)M * N;
  gemm_partials_sum_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>((float*)out, (const float*)partial, KS, count);
  TI_LAUNCH_CHECK();
  return 0;
}

// hooks for tests of the kernel alone: any epilogue, K split `ks` ways (1: not split; partial sums
// are added here)
extern "C" int ti_gemm_bf16_mblocks_any(const void* A, const void* W, void* out, int M, int N, int K, long lda,
                                        int epi, void* partial, int ks, hipStream_t stream) {
  TI_REQUIRE(M > 0 && M <= 64 && N > 0 && K > 0 && K % 64 == 0 && lda >= K && lda % 8 == 0 && ks >= 1 && ks <= K / 64,
             "gemm_bf16_mblocks_any: bad sizes M=%d N=%d K=%d lda=%ld ks=%d", M, N, K, lda, ks);
  TI_REQUIRE(ks == 1 || (epi == TI_EPI_ADD_F32 && partial), "gemm_bf16_mblocks_any: a split K needs the adding epilogue");
  if (lda >= (1L << 24) && M > 1) {      // 64 rows lie further apart than a buffer's descriptor spans: one at a time (the same bits)
    const size_t row = (size_t)N * (epi == TI_EPI_STORE_F32 || epi == TI_EPI_ADD_F32 ? 4 : 2);
    for (int m = 0; m < M; ++m) {
      int rc_ = ti_gemm_bf16_mblocks_any((const bf16_t*)A + (size_t)m * lda, W, (char*)out + m * row, 1, N, K, K, epi, partial, ks, stream);
      if (rc_) return rc_;
    }
    return 0;
  }
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  int rc_ = 0;
  switch (epi) {
    case TI_EPI_STORE_F32: rc_ = launch_mblocks<TI_EPI_STORE_F32>(a, w, out, nullptr, M, N, K, lda, 1, stream); break;
    case TI_EPI_STORE_ACT: rc_ = launch_mblocks<TI_EPI_STORE_ACT>(a, w, out, nullptr, M, N, K, lda, 1, stream); break;
    case TI_EPI_RELU2: rc_ = launch_mblocks<TI_EPI_RELU2>(a, w, out, nullptr, M, N, K, lda, 1, stream); break;
    case TI_EPI_SWIGLU: rc_ = launch_mblocks<TI_EPI_SWIGLU>(a, w, out, nullptr, M, N, K, lda, 1, stream); break;
    case TI_EPI_ADD_F32:
      rc_ = launch_mblocks<TI_EPI_ADD_F32>(a, w, out, (float*)partial, M, N, K, lda, ks, stream);
      if (rc_ == 0 && ks > 1) {
        const size_t count = (size_t)M * N;
        gemm_partials_add_kernel<<<(unsigned)((count + 255) / 256), 256, 0, stream>>>((float*)out, (const float*)partial,
                                                                                    ks, count);
      }
      break;
    default:
      TI_REQUIRE(false, "gemm_bf16_mblocks_any: unknown epilogue %d", epi);
  }
  if (rc_) return rc_;
  TI_LAUNCH_CHECK();
  return 0;
}


// N: output columns (SwiGLU: F, with W holding 2F rows).  Returns 3 for a shape
// these kernels do not serve (the caller takes the generic kernel then).
extern "C" int ti_gemm_bf16(const void* A, const void* W, void* out, int M, int N, int K, long lda, int epi,
                            hipStream_t stream) {
  TI_REQUIRE(M >= 0 && N > 0 && K > 0 && lda >= K, "gemm_bf16: bad sizes M=%d N=%d K=%d lda=%ld", M, N, K, lda);
  if (K % 8 != 0 || lda % 8 != 0 || ((uintptr_t)A & 15) || ((uintptr_t)W & 15)) {
    ti_set_error("gemm_bf16: K=%d / lda=%ld not multiples of 8 or operands not 16-byte aligned", K, lda);
    return 3;
  }
  if ((M + TBM - 1) / TBM > 65535) {
    ti_set_error("gemm_bf16: M=%d too large for one launch", M);
    return 3;
  }
  if (M == 0) return 0;
  const bf16_t* a = (const bf16_t*)A;
  const bf16_t* w = (const bf16_t*)W;
  const bool skinny = (M <= 64 && !(large_weight(M, N, K, epi) && g_use_pipelined)) || staged_112_serves(M, N, K, lda, epi);
  const bool staged = staged_16_serves(M, N, K, lda, epi) && (skinny || pieces_serves(M, N, K, epi));
  const bool copied = !staged && g_skinny_copy && M <= 16 && K % 64 == 0 && K <= 4096 && skinny;
  if (!staged && pieces_serves(M, N, K, epi)) {
    int rc_ = 0;
    switch (epi) {
      case TI_EPI_STORE_F32: rc_ = launch_pieces<TI_EPI_STORE_F32, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
      case TI_EPI_ADD_F32: rc_ = launch_pieces<TI_EPI_ADD_F32, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
      case TI_EPI_STORE_ACT: rc_ = launch_pieces<TI_EPI_STORE_ACT, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
      case TI_EPI_RELU2: rc_ = launch_pieces<TI_EPI_RELU2, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
      default: rc_ = launch_pieces<TI_EPI_SWIGLU, false>(a, lda, w, out, nullptr, M, N, K, 1, stream); break;
    }
    if (rc_) return rc_;
    TI_LAUNCH_CHECK();
    return 0;
  }
  if (wide_rows_serves(M, N, K, epi)) {
    launch_wide_rows(a, w, (float*)out, M, N, K, lda, stream);
    TI_LAUNCH_CHECK();
    return 0;
  }
  if (row_per_wave_serves(M, N, K, epi)) {
    int rc_ = 0;
    if (epi == TI_EPI_STORE_F32) rc_ = launch_rows<TI_EPI_STORE_F32>(a, w, out, M, N, K, lda, stream);
    else if (epi == TI_EPI_RELU2) rc_ = launch_rows<TI_EPI_RELU2>(a, w, out, M, N, K, lda, stream);
    else rc_ = launch_rows<TI_EPI_ADD_F32>(a, w, out, M, N, K, lda, stream);
    if (rc_) return rc_;
    TI_LAUNCH_CHECK();
    return 0;
  }
#define TI_GO(E)                                                  \
  case E:                                                         \
    if (copied) {                                                 \
      int rc_ = launch_skinny_copied<E>(a, w, out, M, N, K, lda, stream); \
      if (rc_) return rc_;                                        \
    } else if (skinny || staged) {                                \
      int rc_ = launch_skinny<E>(a, w, out, M, N, K, lda, stream); \
      if (rc_) return rc_;                                        \
    } else if (g_use_pipelined && pipelined_serves(K, lda)) {    \
      int rc_ = launch_tiled_best<E>(a, w, out, M, N, K, lda, stream); \
      if (rc_) return rc_;                                        \
    } else                                                        \
      launch_tiled<E>(a, w, out, M, N, K, lda, stream);           \
    break;
  switch (epi) {
    TI_GO(TI_EPI_STORE_F32)
    TI_GO(TI_EPI_ADD_F32)
    TI_GO(TI_EPI_STORE_ACT)
    TI_GO(TI_EPI_SWIGLU)
    TI_GO(TI_EPI_RELU2)
    default:
      TI_REQUIRE(false, "gemm_bf16: unknown epilogue %d", epi);
  }
#undef TI_GO
  TI_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------- tests and measurements
// One entry for every shape rule above that a test or a measurement may want to force: `name` as in
// tinyinfer_kernels_tuning.h, value 0 (or what the table says) restores the rule's own choice.
// The rules are the library's, process-wide; the host library's Ops applies an object's own
// overrides around its calls and resets them afterwards.  Returns 0, or 1 for an unknown name.
extern "C" void ti_tuning_reset() {
  g_xcd_rows = 0; g_die_order = 1; g_tiles_160 = 1; g_tiles_256 = 1; g_two_ranges = 1; g_qkv_rows = 0; g_qkv_min_rows = 17; g_force_tile = 0; g_skinny_waves = 0;
  g_skinny_deep = 1; g_use_pipelined = 1; set_tiled_from(280L << 20); g_tiled_from_stored = TILED_FROM_STORED; g_row_per_wave = 1; g_rows_staged = 1;
  g_normed_weight_below = NORMED_WEIGHT_BELOW; g_normed_groups = 0; g_skinny_groups = 0; g_rows_112 = 1; g_skinny_copy = 1; g_wide_rows = 1; g_pieces = 1; g_add_split = 1;
  g_rows_direct = 1;
  g_wide_rows_min_n = WIDE_ROWS_MIN_N;
  g_wide_rows_grid = 0;
}
extern "C" int ti_tuning_set(const char* name, long value) {
  const std::string n = name ? name : "";
  if (n == "force_tile") g_force_tile = (int)value;
  else if (n == "normed_groups") g_normed_groups = (int)value;
  else if (n == "normed_weight_below") g_normed_weight_below = value > 0 ? value : NORMED_WEIGHT_BELOW;
  else if (n == "skinny_groups") g_skinny_groups = (int)value;
  else if (n == "rows_112") g_rows_112 = (int)value;
  else if (n == "tiles_160") g_tiles_160 = (int)value;
  else if (n == "tiles_256") g_tiles_256 = (int)value;
  else if (n == "two_ranges") g_two_ranges = (int)value;
  else if (n == "xcd_rows") g_xcd_rows = (int)value;
  else if (n == "die_order") g_die_order = (int)value;
  else if (n == "skinny_waves") g_skinny_waves = (int)value;
  else if (n == "qkv_prep_min_rows") g_qkv_min_rows = (int)value;
  else if (n == "qkv_prep_rows") g_qkv_rows = (int)value;
  else if (n == "rows_staged") g_rows_staged = (int)value;
  else if (n == "wide_rows") g_wide_rows = (int)value;
  else if (n == "tiled_from") set_tiled_from(value);
  else if (n == "add_split") g_add_split = (int)value;
  else if (n == "use_pipelined") g_use_pipelined = (int)value;
  else if (n == "row_per_wave") g_row_per_wave = (int)value;
  else if (n == "skinny_copy") g_skinny_copy = (int)value;
  else if (n == "pieces") g_pieces = (int)value;
  else if (n == "skinny_deep") g_skinny_deep = (int)value;
  else if (n == "rows_direct") g_rows_direct = (int)value;
  else if (n == "wide_rows_min_n") g_wide_rows_min_n = value > 0 ? (int)value : WIDE_ROWS_MIN_N;
  else if (n == "wide_rows_grid") g_wide_rows_grid = (int)value;
  else return 1;
  return 0;
}
