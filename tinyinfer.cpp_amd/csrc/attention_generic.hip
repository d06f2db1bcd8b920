// Paged causal grouped-query attention for any head size that is a multiple of
// 16 up to 256, any number of heads and groups, any page size, with an optional
// window.
//
//   attention_f32_kernel   the float32 path: a step's portions and single tokens
//                          on the 32-bit matrix instructions, pages of whole 4s
//   attention_rows_kernel  one workgroup per (token row, q head): float32 in
//                          other pages or without a step's lists, and the
//                          bfloat16 path for head sizes its fast kernels refuse
//
// In attention_rows_kernel a workgroup is 16 groups of 16 lanes.  Lane j of a group owns dims j, j+16, ...
// Group g walks keys lo+g, lo+g+16, ... with an online softmax; the 16 partial
// results are merged in LDS with the usual rescaling.  Scores, softmax statistics
// and the output accumulate in 32-bit.
#include "common.h"
#include "tinyinfer_kernels.h"
#include "staged_rows.h"

TI_ERROR_API

#define AG_GROUPS 16
#define AG_LANES 16

template <typename T, int DPL>
__global__ void __launch_bounds__(256)
attention_rows_kernel(const T* __restrict__ q, const T* __restrict__ pool, const int* __restrict__ table,
                      int table_stride, const int* __restrict__ pos, const int* __restrict__ slot,
                      T* __restrict__ out, int n_head, int n_kv, int P, float scale, int window) {
  constexpr int HD = DPL * AG_LANES;
  __shared__ float s_o[AG_GROUPS][HD];
  __shared__ float s_m[AG_GROUPS], s_l[AG_GROUPS];
  const int m = blockIdx.x, h = blockIdx.y;
  const int g = threadIdx.x / AG_LANES, lane = threadIdx.x % AG_LANES;
  const int kvh = h / (n_head / n_kv);
  const int p_q = pos[m];
  const int lo = (window > 0 && p_q - window + 1 > 0) ? p_q - window + 1 : 0;
  const int* tab = table + (size_t)slot[m] * table_stride;
  const size_t page_elems = (size_t)2 * n_kv * P * HD;
  const size_t k_off = (size_t)kvh * P * HD;
  const size_t v_off = ((size_t)n_kv + kvh) * P * HD;

  float qv[DPL], o[DPL];
  const T* qh = q + ((size_t)m * n_head + h) * HD;
#pragma unroll
  for (int i = 0; i < DPL; ++i) {
    qv[i] = ld<T>(qh + lane + i * AG_LANES) * scale;
    o[i] = 0.f;
  }
  float mx = -INFINITY, l = 0.f;
  for (int p = lo + g; p <= p_q; p += AG_GROUPS) {
    const int page = tab[p / P];
    if (page < 0) continue;   // never happens for a reserved request; never read astray
    const T* kp = pool + (size_t)page * page_elems + k_off + (size_t)(p % P) * HD;
    const T* vp = pool + (size_t)page * page_elems + v_off + (p % P);   // values lie transposed: [d][row]
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < DPL; ++i) s = fmaf(qv[i], ld<T>(kp + lane + i * AG_LANES), s);
    s = group_sum<AG_LANES>(s);
    const float m_new = fmaxf(mx, s);
    const float alpha = expf(mx - m_new);   // exp(-inf) = 0 on the first key
    const float w = expf(s - m_new);
    l = l * alpha + w;
#pragma unroll
    for (int i = 0; i < DPL; ++i) o[i] = o[i] * alpha + w * ld<T>(vp + (size_t)(lane + i * AG_LANES) * P);
    mx = m_new;
  }
#pragma unroll
  for (int i = 0; i < DPL; ++i) s_o[g][lane + i * AG_LANES] = o[i];
  if (lane == 0) {
    s_m[g] = mx;
    s_l[g] = l;
  }
  __syncthreads();
  // merge: every thread takes dims tid, tid+256, ... (HD <= 256: at most one)
  for (int d = threadIdx.x; d < HD; d += 256) {
    float mm = -INFINITY;
#pragma unroll
    for (int j = 0; j < AG_GROUPS; ++j) mm = fmaxf(mm, s_m[j]);
    float lt = 0.f, acc = 0.f;
#pragma unroll
    for (int j = 0; j < AG_GROUPS; ++j) {
      const float w = (s_m[j] == -INFINITY) ? 0.f : expf(s_m[j] - mm);
      lt += s_l[j] * w;
      acc += s_o[j][d] * w;
    }
    st<T>(out + ((size_t)m * n_head + h) * HD + d, acc / lt);
  }
}

template <typename T>
static int launch_rows(int dpl, dim3 grid, const void* q, const void* pool, const int* table, int table_stride,
                       const int* pos, const int* slot, void* out, int n_head, int n_kv, int P, float scale,
                       int window, hipStream_t stream) {
#define AG_CASE(D)                                                                                     \
  case D:                                                                                              \
    attention_rows_kernel<T, D><<<grid, 256, 0, stream>>>((const T*)q, (const T*)pool, table,           \
                                                          table_stride, pos, slot, (T*)out, n_head,    \
                                                          n_kv, P, scale, window);                     \
    break;
  switch (dpl) {
    AG_CASE(1) AG_CASE(2) AG_CASE(3) AG_CASE(4) AG_CASE(5) AG_CASE(6) AG_CASE(7) AG_CASE(8)
    AG_CASE(9) AG_CASE(10) AG_CASE(11) AG_CASE(12) AG_CASE(13) AG_CASE(14) AG_CASE(15) AG_CASE(16)
    default:
      return 1;
  }
#undef AG_CASE
  return 0;
}

// q, out: [M, n_head, hd] in T; pool: [pages][K: [n_kv][P][hd] | V: [n_kv][hd][P]] in T;
// table: [slots][table_stride];
// pos, slot: [M].  window <= 0: all keys up to the row's own position.
extern "C" int ti_attention_rows(int dtype, const void* q, const void* pool, const int* table, int table_stride,
                                 const int* pos, const int* slot, void* out, int M, int n_head, int n_kv,
                                 int hd, int page_size, float scale, int window, hipStream_t stream) {
  TI_REQUIRE(hd >= 16 && hd <= 256 && hd % 16 == 0,
             "attention: head_dim %d is not served (multiples of 16 up to 256)", hd);
  TI_REQUIRE(n_head > 0 && n_kv > 0 && n_head % n_kv == 0, "attention: heads %d / kv_heads %d", n_head, n_kv);
  TI_REQUIRE(n_head <= 65535, "attention: too many heads (%d)", n_head);
  TI_REQUIRE(page_size > 0 && table_stride > 0, "attention: bad page_size %d / table_stride %d", page_size, table_stride);
  if (M == 0) return 0;
  dim3 grid(M, n_head);
  int rc;
  if (dtype == TI_F32)
    rc = launch_rows<float>(hd / 16, grid, q, pool, table, table_stride, pos, slot, out, n_head, n_kv, page_size, scale, window, stream);
  else if (dtype == TI_BF16)
    rc = launch_rows<bf16_t>(hd / 16, grid, q, pool, table, table_stride, pos, slot, out, n_head, n_kv, page_size, scale, window, stream);
  else
    TI_REQUIRE(false, "attention: unknown dtype %d", dtype);
  TI_REQUIRE(rc == 0, "attention: no kernel for head_dim %d", hd);
  TI_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------------------
// float32 on the matrix cores.  A workgroup's eight wavefronts hold 16 columns: 16 consecutive tokens of one q head
// (a portion; four workgroups a tile of 64 rows), or the q heads of one token that share a kv head (single tokens).
// They walk the keys in blocks of 16:
//   S^T (16 keys x 16 columns) = K (16 x hd) . Q^T      O^T (hd x 16) += V^T (hd x 16 keys) . P^T
// both by v_mfma_f32_16x16x4_f32 with four consecutive entries a lane (loaded as one float4; both operands of a product
// are permuted alike), so that the scores' layout is the second product's operand.  Block b belongs to wavefront
// b mod 8 whatever the tile, and a key that a column may not see leaves it bit by bit as it was, whatever the key and its
// value hold: a token's result depends on its keys alone, however a step is cut.  Keys and values come through LDS or straight from memory (below),
// the next block's while one is multiplied; short contexts are bounded by the start and the merge.  (With the rows kernel below, one workgroup
// per row and head, lane sums and one value a load, a portion of 300 tokens with 16 heads of 128 on 8 kv heads took
// 201 us a layer, 5.6 ms of a prompt of Qwen3-0.6B's sizes.)
#define AF_WAVES 8
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float af4;

// N slices of 1 KiB of LDS, this lane's 16 bytes of each (`at`: of the first), have arrived in registers when this returns.
template <int N> __device__ __forceinline__ void read_some_slices(af4* e, unsigned at) {
  if constexpr (N == 1) asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(e[0]) : "v"(at) : "memory");
  if constexpr (N == 2)
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:1024\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0]), "=&v"(e[1]) : "v"(at) : "memory");
  if constexpr (N == 4)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:1024\n\tds_read_b128 %2, %4 offset:2048\n\t"
                 "ds_read_b128 %3, %4 offset:3072\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(e[0]), "=&v"(e[1]), "=&v"(e[2]), "=&v"(e[3]) : "v"(at) : "memory");
}
template <int DB> __device__ __forceinline__ void read_slices(af4* e, unsigned at) {
#pragma unroll
  for (int d = 0; d + 4 <= DB; d += 4) read_some_slices<4>(e + d, at + d * 1024);
  if constexpr (DB & 2) read_some_slices<2>(e + (DB & ~3), at + (DB & ~3) * 1024);
  if constexpr (DB & 1) read_some_slices<1>(e + (DB & ~1), at + (DB & ~1) * 1024);
}

// STAGED (heads of up to 128, pages of whole blocks): the blocks come by direct loads through LDS of each wavefront's own, DB slices of 16
// rows x 64 bytes for the keys and as many for the values.  As operands straight from memory, neighbouring lanes in different rows, a load
// takes the unit that takes addresses 64 cycles, and a compute unit's eight wavefronts share it: some 3.4 us a round of eight blocks of
// heads of 128; four lanes to a row's 64 bytes take 16.  A slice is asked for again, for the wavefront's next block, as soon as it has been
// read.  Piece c (16 bytes) of row r lies in place 4 r + (c ^ (-(r / 4) % 4)): the sixteen lanes that LDS serves together are rows 0 to 3 and 12 to 15 of
// one quarter and 4 to 11 of the next, and read from different banks so (from places c ^ (r / 4) a read takes twice as long).  The
// arithmetic is the same, and so are the bits.  us, straight from memory, so, and with the order of tiles below: a portion
// of 300 tokens, 16 heads of 128 on 8, 27.7, 20.8, 15.9; 512 tokens behind 300 63.5, 46.9, 43.3; 300 tokens with 32 heads of 64 23.8, 19.8,
// 17.7; 8 single tokens of 900 31.6 -> 25.7.  Left: 304 workgroups on 256 units, one a unit, and each one's start and merge.
template <int DB, bool SINGLE, bool STAGED>
__global__ void __launch_bounds__(64 * AF_WAVES)
attention_f32_kernel(const float* __restrict__ q, const float* __restrict__ pool, const int* __restrict__ table,
                     int table_stride, const int* __restrict__ pos, const int* __restrict__ slot,
                     const int* __restrict__ rows, const int* __restrict__ tiles, const int* __restrict__ entries,
                     float* __restrict__ out, int n_head, int n_kv, int P, float scale, int window) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
  constexpr int HD = DB * 16, STAGE = 2 * DB * 1024;       // bytes of a wavefront's stage, where its sums lie afterwards
  static_assert(STAGE >= 16 * (HD + 4) * 4, "a wavefront's sums fit into its stage");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  __shared__ __attribute__((aligned(16))) float s_sums[STAGED ? 1 : AF_WAVES][16][HD + 4];
  const auto s_o = [&](int w, int c) -> float* {
    if constexpr (STAGED) return reinterpret_cast<float*>(smem + w * STAGE) + c * (HD + 4);
    else return s_sums[w][c];
  };
  __shared__ float s_m[AF_WAVES][16], s_l[AF_WAVES][16];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;
  const int G = n_head / n_kv;
  // the workgroup's columns: rows m_row .. of head `head0`, or heads head0 .. of row m_row
  int m_row, head0, n_cols, kvh, p_first, p_last;
  const int* tab;
  if constexpr (SINGLE) {
    const int parts = (G + 15) / 16;
    m_row = rows ? rows[blockIdx.x] : blockIdx.x;
    kvh = blockIdx.y / parts;
    head0 = kvh * G + (blockIdx.y % parts) * 16;
    n_cols = min(16, (kvh + 1) * G - head0);
    p_first = p_last = pos[m_row];
    tab = table + (size_t)slot[m_row] * table_stride;
  } else {
    // the list's first tiles, which see the most keys, first and in all heads: what is left for a second round is short
    const unsigned at = blockIdx.y * gridDim.x + blockIdx.x, part = at / n_head;
    const int entry = tiles[(part >> 2) * 2], row0 = entries[entry * 4];
    m_row = tiles[(part >> 2) * 2 + 1] + (3 - (part & 3)) * 16;
    head0 = at % n_head;
    kvh = head0 / G;
    n_cols = min(16, row0 + entries[entry * 4 + 1] - m_row);
    if (n_cols <= 0) return;
    p_first = entries[entry * 4 + 2] + m_row - row0;
    p_last = p_first + n_cols - 1;
    tab = table + (size_t)entry * table_stride;
  }
  const int col = min(r16, n_cols - 1);             // columns past the end repeat the last one and are not stored
  const size_t q_row = SINGLE ? (size_t)m_row * n_head + head0 + col : (size_t)(m_row + col) * n_head + head0;
  const int hi = SINGLE ? p_last : p_first + col;
  const int lo = (window > 0 && hi - window + 1 > 0) ? hi - window + 1 : 0;
  const int lo_min = (window > 0 && p_first - window + 1 > 0) ? p_first - window + 1 : 0;
  const int lo_max = (window > 0 && p_last - window + 1 > 0) ? p_last - window + 1 : 0;

  const size_t page_elems = (size_t)2 * n_kv * P * HD;
  const float* k_head = pool + (size_t)kvh * P * HD;
  const float* v_head = pool + ((size_t)n_kv + kvh) * P * HD;
  af4 qf[DB], o[DB];
#pragma unroll
  for (int s = 0; s < DB; ++s) {
    qf[s] = *reinterpret_cast<const af4*>(q + q_row * HD + s * 16 + quad * 4);
    o[s] = af4{0.f, 0.f, 0.f, 0.f};
  }
  struct Block { af4 k[DB], v[DB]; int key0; bool have; };
  auto load = [&](Block& f, int b) {                // keys past the last one repeat it, whatever their place holds
    f.key0 = b * 16;
    const int key = min(b * 16 + r16, p_last), v4 = min(b * 16 + quad * 4, p_last & ~3);
    const int pk = tab[key / P], pv = tab[v4 / P];
    f.have = pv >= 0;                               // a page given back behind the window holds nothing that is seen
    const float* kp = k_head + (size_t)max(pk, 0) * page_elems + (size_t)(key % P) * HD + quad * 4;
    const float* vp = v_head + (size_t)max(pv, 0) * page_elems + (size_t)r16 * P + (v4 % P);
#pragma unroll
    for (int s = 0; s < DB; ++s) f.k[s] = *reinterpret_cast<const af4*>(kp + s * 16);
#pragma unroll
    for (int d = 0; d < DB; ++d) f.v[d] = *reinterpret_cast<const af4*>(vp + (size_t)d * 16 * P);
  };
  float mx = -INFINITY, l = 0.f;
  auto attend = [&](Block& f, auto values) {         // values(): f.v are there when it returns
    af4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DB; ++s) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (s % 2 == 0) s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(f.k[s][j], qf[s][j], s0, 0, 0, 0);
        else s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(f.k[s][j], qf[s][j], s1, 0, 0, 0);
      }
    }
    values();
    float sc[4], bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = f.key0 + quad * 4 + i;
      sc[i] = (f.have && key >= lo && key <= hi) ? (s0[i] + s1[i]) * scale : -INFINITY;
      bm = fmaxf(bm, sc[i]);
      if (!f.have || key > p_last || key < lo_min) {  // seen by no column: any bits, and 0 times NaN is NaN
#pragma unroll
        for (int d = 0; d < DB; ++d) f.v[d][i] = 0.f;
      }
    }
    bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float m_new = fmaxf(mx, bm);
    const float m_safe = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = expf(mx - m_safe);          // 1 where nothing new is seen; 0 in front of the first key
    float w[4];
    l *= alpha;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      w[i] = expf(sc[i] - m_safe);
      l += w[i];
    }
    mx = m_new;
#pragma unroll
    for (int d = 0; d < DB; ++d) o[d] *= alpha;
    // A key that some columns see and others do not: a weight of 0 leaves those out unless the value is infinite or not a
    // number.  Such values are taken out of the product and given to the columns that see them one by one.
    if (!SINGLE && (f.key0 + 15 > p_first || f.key0 < lo_max)) {
      float nil = 0.f;
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) nil = fmaf(f.v[d][j], 0.f, nil);
      if (__any(nil != 0.f)) {
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int key = f.key0 + g * 4 + j;
            const float weight = __shfl(w[j], g * 16 + r16, 64);
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                const float v = __shfl(f.v[d][j], g * 16 + quad * 4 + i, 64);
                if (v * 0.f != 0.f && key >= lo && key <= hi) o[d][i] = fmaf(v, weight, o[d][i]);
              }
          }
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int j = 0; j < 4; ++j) f.v[d][j] = f.v[d][j] * 0.f != 0.f ? 0.f : f.v[d][j];
      }
    }
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.v[d][j], w[j], o[d], 0, 0, 0);
  };
  const int b_last = p_last / 16;
  int b = lo_min / 16;
  b += (wave - b % AF_WAVES + AF_WAVES) % AF_WAVES;
  const auto there = [] {};
  if (b <= b_last) {
    Block f0;
    if constexpr (STAGED) {
      const int row = lane >> 2, piece = (lane & 3) ^ (-(row >> 2) & 3);
      const unsigned k_off = (unsigned)row * (HD * 4) + piece * 16, v_off = (unsigned)row * (unsigned)(P * 4) + piece * 16;
      unsigned char* mine = smem + wave * STAGE;
      const unsigned at = (unsigned)(size_t)mine + r16 * 64 + ((quad ^ (-(r16 >> 2) & 3)) << 4);
      const auto rows_at = [](const float* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
      const auto page_of = [&](int block) { return __builtin_amdgcn_readfirstlane(tab[block * 16 / P]); };
      const auto ask_keys = [&](int page, int block) {
        const auto rs = rows_at(k_head + (size_t)max(page, 0) * page_elems + (size_t)(block * 16 % P) * HD);
#pragma unroll
        for (int s = 0; s < DB; ++s)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(mine + s * 1024), 16, k_off, s * 64, 0, 0);
      };
      const auto ask_values = [&](int page, int block) {
        const auto rs = rows_at(v_head + (size_t)max(page, 0) * page_elems + block * 16 % P);
#pragma unroll
        for (int d = 0; d < DB; ++d)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(mine + (DB + d) * 1024), 16, v_off, d * 64 * P, 0, 0);
      };
      int page = page_of(b);
      ask_keys(page, b);
      ask_values(page, b);
      for (;;) {
        const int next = b + AF_WAVES;
        const bool more = next <= b_last;           // the same in every lane
        const int next_page = more ? page_of(next) : 0;
        f0.key0 = b * 16;
        f0.have = page >= 0;
        wait_vmcnt<DB>();                           // the keys are there; their values may still be out
        read_slices<DB>(f0.k, at);
        if (more) ask_keys(next_page, next);
        __builtin_amdgcn_sched_barrier(0);
        attend(f0, [&] {
          if (more) wait_vmcnt<DB>();               // the next keys may still be out
          else wait_vmcnt<0>();
          read_slices<DB>(f0.v, at + DB * 1024);
          if (more) ask_values(next_page, next);
          __builtin_amdgcn_sched_barrier(0);
        });
        if (!more) break;
        b = next;
        page = next_page;
      }
    } else if constexpr (DB > 8) {                         // two blocks of such heads do not fit in the registers
      for (; b <= b_last; b += AF_WAVES) {
        load(f0, b);
        attend(f0, there);
      }
    } else {
    Block f1;
    load(f0, b);
    for (;;) {
      load(f1, min(b + AF_WAVES, b_last));
      __builtin_amdgcn_sched_barrier(0);
      attend(f0, there);
      if ((b += AF_WAVES) > b_last) break;
      load(f0, min(b + AF_WAVES, b_last));
      __builtin_amdgcn_sched_barrier(0);
      attend(f1, there);
      if ((b += AF_WAVES) > b_last) break;
    }
    }
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
#pragma unroll
  for (int d = 0; d < DB; ++d) *reinterpret_cast<af4*>(s_o(wave, r16) + d * 16 + quad * 4) = o[d];
  if (quad == 0) {
    s_m[wave][r16] = mx;
    s_l[wave][r16] = l;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_cols * HD; e += 64 * AF_WAVES) {
    const int c = e / HD, d = e % HD;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) mm = fmaxf(mm, s_m[w][c]);
    float lt = 0.f, acc = 0.f;
#pragma unroll
    for (int w = 0; w < AF_WAVES; ++w) {
      const float f = (s_m[w][c] == -INFINITY) ? 0.f : expf(s_m[w][c] - mm);
      lt += s_l[w][c] * f;
      acc += s_o(w, c)[d] * f;
    }
    const size_t row = SINGLE ? (size_t)m_row * n_head + head0 + c : (size_t)(m_row + c) * n_head + head0;
    out[row * HD + d] = acc / lt;
  }
#endif
}

// the stages' LDS; pages of whole blocks whose values lie within what a buffer's offset spans
template <int DB, bool SINGLE>
static int launch_attention_f32(dim3 grid, const float* q, const float* pool, const int* table, int table_stride, const int* pos,
                                const int* slot, const int* rows, const int* tiles, const int* entries, float* out, int n_head, int n_kv,
                                int P, float scale, int window, hipStream_t stream) {
  if constexpr (DB <= 8) {
    if (P % 16 == 0 && P <= 65536) {
      constexpr int lds = AF_WAVES * 2 * DB * 1024;
      auto kernel = attention_f32_kernel<DB, SINGLE, true>;
      static const hipError_t room = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      TI_REQUIRE(room == hipSuccess, "attention: %d bytes of LDS: %s", lds, hipGetErrorString(room));
      kernel<<<grid, 64 * AF_WAVES, lds, stream>>>(q, pool, table, table_stride, pos, slot, rows, tiles, entries, out, n_head, n_kv, P, scale, window);
      return 0;
    }
  }
  attention_f32_kernel<DB, SINGLE, false><<<grid, 64 * AF_WAVES, 0, stream>>>(q, pool, table, table_stride, pos, slot, rows, tiles, entries, out,
                                                                             n_head, n_kv, P, scale, window);
  return 0;
}

// A step's attention in float32: n_tiles tiles of up to 64 rows of portions (tiles int32 [n_tiles][2] = (entry, first
// row), entries int32 [.][4] = (row0, tokens, first position, .), an entry being its own row of the block table) and
// n_single rows of single tokens (row numbers in `rows`, or 0 .. n_single - 1).  3: sizes not served (what the head
// and page sizes say, never the step: one kernel serves all steps of a model).
extern "C" int ti_attention_f32(const void* q, const void* pool, const int* table, int table_stride, const int* pos, const int* slot,
                                const int* rows, int n_single, const int* tiles, const int* entries, int n_tiles, void* out,
                                int n_head, int n_kv, int hd, int page_size, float scale, int window, hipStream_t stream) {
  TI_REQUIRE(n_head > 0 && n_kv > 0 && n_head % n_kv == 0, "attention: heads %d / kv_heads %d", n_head, n_kv);
  TI_REQUIRE(n_head <= 65535, "attention: too many heads (%d)", n_head);
  TI_REQUIRE(page_size > 0 && table_stride > 0, "attention: bad page_size %d / table_stride %d", page_size, table_stride);
  TI_REQUIRE(n_tiles >= 0 && n_single >= 0 && (n_tiles == 0 || (tiles && entries)), "attention: %d tiles without their lists", n_tiles);
  if (hd < 16 || hd > 256 || hd % 16 != 0 || page_size % 4 != 0) return 3;
  const int parts = (n_head / n_kv + 15) / 16;
  int rc_ = 0;
#define AF_CASE(D)                                                                                                            \
  case D:                                                                                                                     \
    if (n_tiles)                                                                                                              \
      rc_ = launch_attention_f32<D, false>(dim3(n_tiles * 4, n_head), (const float*)q, (const float*)pool, table, table_stride, pos,\
                                           slot, rows, tiles, entries, (float*)out, n_head, n_kv, page_size, scale, window, stream);\
    if (rc_ == 0 && n_single)                                                                                                 \
      rc_ = launch_attention_f32<D, true>(dim3(n_single, n_kv * parts), (const float*)q, (const float*)pool, table, table_stride, pos,\
                                          slot, rows, tiles, entries, (float*)out, n_head, n_kv, page_size, scale, window, stream);\
    break;
  switch (hd / 16) {
    AF_CASE(1) AF_CASE(2) AF_CASE(3) AF_CASE(4) AF_CASE(5) AF_CASE(6) AF_CASE(7) AF_CASE(8)
    AF_CASE(9) AF_CASE(10) AF_CASE(11) AF_CASE(12) AF_CASE(13) AF_CASE(14) AF_CASE(15) AF_CASE(16)
    default:
      return 3;
  }
#undef AF_CASE
  if (rc_) return rc_;
  TI_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------------------------------------------
// The same walk (a workgroup per row and head) for attention whose keys and values differ in size and whose scores are soft-capped:
//   s = (q . k) * scale;  s <- softcap * tanh(s / softcap)  (softcap <= 0: none);  softmax over the
// visible keys.  Any key size dk and value size dv up to 256 (lanes beyond a size idle).  A page is
// K [n_kv][P][dk] | V [n_kv][dv][P]; with dk == dv that is the layout above.
template <typename T, int DPL>
__global__ void __launch_bounds__(256)
attention_capped_kernel(const T* __restrict__ q, const T* __restrict__ pool, const int* __restrict__ table,
                        int table_stride, const int* __restrict__ pos, const int* __restrict__ slot,
                        T* __restrict__ out, int n_head, int n_kv, int dk, int dv, int P, float scale, float softcap,
                        int window) {
  constexpr int HD = DPL * AG_LANES;
  __shared__ float s_o[AG_GROUPS][HD];
  __shared__ float s_m[AG_GROUPS], s_l[AG_GROUPS];
  const int m = blockIdx.x, h = blockIdx.y;
  const int g = threadIdx.x / AG_LANES, lane = threadIdx.x % AG_LANES;
  const int kvh = h / (n_head / n_kv);
  const int p_q = pos[m];
  const int lo = (window > 0 && p_q - window + 1 > 0) ? p_q - window + 1 : 0;
  const int* tab = table + (size_t)slot[m] * table_stride;
  const size_t page_elems = (size_t)n_kv * P * (dk + dv);
  const size_t k_off = (size_t)kvh * P * dk;
  const size_t v_off = (size_t)n_kv * P * dk + (size_t)kvh * dv * P;
  const float inv_cap = softcap > 0.f ? 1.f / softcap : 0.f;

  float qv[DPL], o[DPL];
  const T* qh = q + ((size_t)m * n_head + h) * dk;
#pragma unroll
  for (int i = 0; i < DPL; ++i) {
    const int d = lane + i * AG_LANES;
    qv[i] = d < dk ? ld<T>(qh + d) : 0.f;
    o[i] = 0.f;
  }
  float mx = -INFINITY, l = 0.f;
  for (int p = lo + g; p <= p_q; p += AG_GROUPS) {
    const int page = tab[p / P];
    if (page < 0) continue;
    const T* kp = pool + (size_t)page * page_elems + k_off + (size_t)(p % P) * dk;
    const T* vp = pool + (size_t)page * page_elems + v_off + (p % P);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      const int d = lane + i * AG_LANES;
      if (d < dk) s = fmaf(qv[i], ld<T>(kp + d), s);
    }
    s = group_sum<AG_LANES>(s) * scale;
    if (softcap > 0.f) s = softcap * tanhf(s * inv_cap);
    const float m_new = fmaxf(mx, s);
    const float alpha = expf(mx - m_new);
    const float w = expf(s - m_new);
    l = l * alpha + w;
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      const int d = lane + i * AG_LANES;
      if (d < dv) o[i] = o[i] * alpha + w * ld<T>(vp + (size_t)d * P);
    }
    mx = m_new;
  }
#pragma unroll
  for (int i = 0; i < DPL; ++i) s_o[g][lane + i * AG_LANES] = o[i];
  if (lane == 0) {
    s_m[g] = mx;
    s_l[g] = l;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < dv; d += 256) {
    float mm = -INFINITY;
#pragma unroll
    for (int j = 0; j < AG_GROUPS; ++j) mm = fmaxf(mm, s_m[j]);
    float lt = 0.f, acc = 0.f;
#pragma unroll
    for (int j = 0; j < AG_GROUPS; ++j) {
      const float w = (s_m[j] == -INFINITY) ? 0.f : expf(s_m[j] - mm);
      lt += s_l[j] * w;
      acc += s_o[j][d] * w;
    }
    st<T>(out + ((size_t)m * n_head + h) * dv + d, acc / lt);
  }
}

template <typename T>
static int launch_capped(int dpl, dim3 grid, const void* q, const void* pool, const int* table, int table_stride,
                         const int* pos, const int* slot, void* out, int n_head, int n_kv, int dk, int dv, int P,
                         float scale, float softcap, int window, hipStream_t stream) {
#define AG_CASE(D)                                                                                              \
  case D:                                                                                                       \
    attention_capped_kernel<T, D><<<grid, 256, 0, stream>>>((const T*)q, (const T*)pool, table, table_stride, pos, \
                                                            slot, (T*)out, n_head, n_kv, dk, dv, P, scale, softcap, \
                                                            window);                                            \
    break;
  switch (dpl) {
    AG_CASE(1) AG_CASE(2) AG_CASE(3) AG_CASE(4) AG_CASE(5) AG_CASE(6) AG_CASE(7) AG_CASE(8)
    AG_CASE(9) AG_CASE(10) AG_CASE(11) AG_CASE(12) AG_CASE(13) AG_CASE(14) AG_CASE(15) AG_CASE(16)
    default:
      return 1;
  }
#undef AG_CASE
  return 0;
}

// q: [M, n_head, dk], out: [M, n_head, dv] in T; pool: [pages][K: [n_kv][P][dk] | V: [n_kv][dv][P]] in T
extern "C" int ti_attention_capped_rows(int dtype, const void* q, const void* pool, const int* table, int table_stride,
                                        const int* pos, const int* slot, void* out, int M, int n_head, int n_kv, int dk,
                                        int dv, int page_size, float scale, float softcap, int window,
                                        hipStream_t stream) {
  TI_REQUIRE(dk >= 1 && dk <= 256 && dv >= 1 && dv <= 256, "attention: key size %d / value size %d are not served (up to 256)",
             dk, dv);
  TI_REQUIRE(n_head > 0 && n_kv > 0 && n_head % n_kv == 0, "attention: heads %d / kv_heads %d", n_head, n_kv);
  TI_REQUIRE(n_head <= 65535, "attention: too many heads (%d)", n_head);
  TI_REQUIRE(page_size > 0 && table_stride > 0, "attention: bad page_size %d / table_stride %d", page_size, table_stride);
  if (M == 0) return 0;
  dim3 grid(M, n_head);
  const int big = dk > dv ? dk : dv;
  const int dpl = (big + AG_LANES - 1) / AG_LANES;
  int rc;
  if (dtype == TI_F32)
    rc = launch_capped<float>(dpl, grid, q, pool, table, table_stride, pos, slot, out, n_head, n_kv, dk, dv, page_size, scale,
                              softcap, window, stream);
  else if (dtype == TI_BF16)
    rc = launch_capped<bf16_t>(dpl, grid, q, pool, table, table_stride, pos, slot, out, n_head, n_kv, dk, dv, page_size, scale,
                               softcap, window, stream);
  else
    TI_REQUIRE(false, "attention: unknown dtype %d", dtype);
  TI_REQUIRE(rc == 0, "attention: no kernel for sizes %d / %d", dk, dv);
  TI_LAUNCH_CHECK();
  return 0;
}
