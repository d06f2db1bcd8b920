// Paged causal grouped-query attention in bfloat16 on the matrix cores of gfx950,
// for decode rows (flash decoding: the context of a row is split over several
// workgroups and merged) and for portions of prompts (flash attention over the
// pages, earlier portions included).
//
// Both walk the cache in blocks of 16 positions.  A page holds keys as
// [row][head_dim] and values transposed as [head_dim][row], so both products
// read their operands along the dimension they reduce over.  Launches by records (what an
// engine's decode steps take) and the prompt kernel for head sizes 64 and 128, which works on
// tiles of 32 x 32, bring them through LDS by direct loads; decode by equal runs and the
// prompt kernel for head size 32 read them straight from memory.  A tile of 16 columns:
//   S^T (16 keys x 16 columns)  = K (16 x hd) . Q^T          v_mfma_f32_16x16x32_bf16
//   O^T (hd x 16 columns)      += V^T (hd x 16 keys) . P^T   v_mfma_f32_16x16x16_bf16
// The transposed score tile leaves each lane with four keys of one column, which
// is exactly the operand layout the second product wants for P^T: no shuffles and
// no LDS between the two products.  The softmax statistics of a column are one scalar per
// lane; scores, statistics and outputs are 32-bit.
//
// What the 16 columns are differs:
//   decode   the q heads that share one kv head, for one token: the kv head's
//            keys and values are read once for all of them.  Four wavefronts take
//            the blocks of the split in turn and merge through LDS.
//   prefill  16 consecutive tokens of one q head; a workgroup's four wavefronts
//            take four such tiles of the same head, so they walk the same pages
//            together and share them in the cache.
// (The reference scans positions with 16-lane groups and FMA for both cases:
// src/cuda/attention.cu:107-198.)
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
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short short4v;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

#define TI_LOG2E 1.4426950408889634f

union Frag8 {
  uint4 u;
  bf16x8 v;
};
union Frag4 {
  uint2 u;
  short4v v;
  bf16_t h[4];
};

struct PagedKV {
  const bf16_t* pool;   // [pages][2][n_kv][P * hd]
  const int* table;     // block-table row of the request
  int P;                // rows per page (multiple of 16)
  int n_kv;
  int kvh;
};

// The fragments of two blocks of 16 keys each, [keyA, keyA + 16) and [keyB, keyB + 16),
// for the two products.  The pair is what one turn of the walk handles: one softmax
// update and one rescaling of the output for 32 keys, and the second product as
// v_mfma_f32_16x16x32_bf16 over both blocks at once.
template <int HD>
struct KVPair {
  // Of the pair's 32 keys (block A's, then block B's) a lane's eight scores are those of keys 8 (lane / 16) .. + 7, so that the
  // values they weigh lie in one run of 16 bytes: half as many loads as with four keys of either block.
  Frag8 k[2][HD / 32];   // K:   k[j]: key 8 (row / 4) + row % 4 + 4 j of the pair, row = lane % 16; dims 32 s + 8 (lane / 16) .. + 7
  Frag8 v[HD / 16];      // V^T: row (dim) 16 d + lane % 16; keys 8 (lane / 16) .. + 7
};

// Issue the loads of a pair.  They are unconditional (the caller passes pages that
// exist, whatever they hold) so that the compiler can count them and let the
// arithmetic of the pair before run while they are in flight.
template <int HD>
__device__ __forceinline__ void load_pair(const PagedKV& kv, int pageA, int keyA, int pageB, int keyB,
                                          KVPair<HD>& f) {
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;
  // where a block's keys and values start is the same in every lane (scalar registers)
  const size_t page_elems = (size_t)2 * kv.n_kv * kv.P * HD, head_elems = (size_t)kv.P * HD;
  const bf16_t* ka = kv.pool + (size_t)pageA * page_elems + kv.kvh * head_elems;
  const bf16_t* kb = kv.pool + (size_t)pageB * page_elems + kv.kvh * head_elems;
  const bf16_t* va = ka + kv.n_kv * head_elems;
  const bf16_t* vb = kb + kv.n_kv * head_elems;
  if (kv.P != 16) {      // blocks that start inside their page
    const int rowA = keyA % kv.P, rowB = keyB % kv.P;
    ka += (size_t)rowA * HD;
    kb += (size_t)rowB * HD;
    va += rowA;
    vb += rowB;
  }
  const bf16_t* k = (r16 < 8 ? ka : kb) + (((r16 >> 2) & 1) * 8 + (r16 & 3)) * HD + quad * 8;
  const bf16_t* v = (quad < 2 ? va : vb) + r16 * kv.P + (quad & 1) * 8;
#pragma unroll
  for (int s = 0; s < HD / 32; ++s) {
    f.k[0][s].u = *reinterpret_cast<const uint4*>(k + s * 32);
    f.k[1][s].u = *reinterpret_cast<const uint4*>(k + 4 * HD + s * 32);
  }
  const unsigned v_step = 16u * kv.P;                                // elements between blocks of 16 dims
#pragma unroll
  for (int d = 0; d < HD / 16; ++d) f.v[d].u = *reinterpret_cast<const uint4*>(v + d * v_step);
}

// What the walk knows of one block.
struct BlockInfo {
  int key0;     // first key
  bool valid;   // false: the block does not count (a stand-in loaded to keep the loads
                // unconditional, or a page that was given back)
  bool check;   // true: some key of it may be hidden from some column, or not written yet
};

// tanh from one exponential and one reciprocal: 1 - 2 / (1 + e^(2x)); exact at both ends (e^(2x) = 0 or infinite), within
// 2e-7 elsewhere, which a soft cap multiplies by the cap: far below a score's own rounding
__device__ __forceinline__ float tanh_fast(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * 2.8853900817779268f));
}

// One pair of blocks for this wavefront's 16 columns.
//   qf       Q^T fragments: column lane % 16, dims 32 * step + 8 * (lane / 16) .. + 7
//   scale    softmax scale times log2(e): scores, maxima and partial maxima are in units of log 2,
//            so that the weights are bare exp2
//   lo, hi   the keys this lane's column may see: lo <= key <= hi
//   kv_last  last position of the request that has been written (rows after it hold rubbish)
//   cap2     > 0: scores are soft-capped, s <- cap tanh(s / cap), cap2 being the cap in units of log 2 like `scale`
template <int HD>
__device__ __forceinline__ void attend_pair(KVPair<HD>& f, const Frag8* qf, BlockInfo A, BlockInfo B, int lo,
                                            int hi, int kv_last, float scale, float& m, float& l, floatx4* o,
                                            float cap2 = 0.f) {
  const int lane = threadIdx.x & 63;
  const int quad = lane >> 4;
  // S^T = K . Q^T, both blocks
  floatx4 sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < HD / 32; ++s) {
    sa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.k[0][s].v, qf[s].v, sa, 0, 0, 0);
    sb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.k[1][s].v, qf[s].v, sb, 0, 0, 0);
  }
  if (cap2 > 0.f) {      // the same in every lane; before the masks, which put -inf where a key is hidden
    const float r = scale / cap2, back = cap2 / scale;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sa[i] = tanh_fast(sa[i] * r) * back;
      sb[i] = tanh_fast(sb[i] * r) * back;
    }
  }
  // this lane: eight keys in a row of one block
  float sv[8];
  const bool plain = A.valid && B.valid && !A.check && !B.check;   // the same in every lane
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    sv[i] = sa[i] * scale;
    sv[4 + i] = sb[i] * scale;
  }
  if (!plain) {
    const int key0 = (quad < 2 ? A.key0 : B.key0) + (quad & 1) * 8;
    const bool valid = quad < 2 ? A.valid : B.valid, check = quad < 2 ? A.check : B.check;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      unsigned keep = 0xFFFFFFFFu;
#pragma unroll
      for (int i = 2 * w; i < 2 * w + 2; ++i) {
        const int key = key0 + i;
        const bool see = valid & (!check | ((key >= lo) & (key <= hi)));   // bitwise: selects, no branches
        sv[i] = see ? sv[i] : -INFINITY;
        // rows never written may hold anything, NaN included, and 0 * NaN is NaN
        const bool zero = !valid | (key > kv_last);
        keep &= zero ? ((i & 1) ? 0x0000FFFFu : 0xFFFF0000u) : 0xFFFFFFFFu;
      }
#pragma unroll
      for (int d = 0; d < HD / 16; ++d) reinterpret_cast<unsigned*>(&f.v[d].u)[w] &= keep;
    }
  }
  float bm = sv[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) bm = fmaxf(bm, sv[i]);
  {
    const LanePair p = lane_pair<32>(bm);
    bm = fmaxf(p.a, p.b);
  }
  {
    const LanePair p = lane_pair<16>(bm);
    bm = fmaxf(p.a, p.b);
  }
  const float m_new = fmaxf(m, bm);
  const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
  Frag8 pf;
  float pv[8], ps = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    pv[i] = __builtin_amdgcn_exp2f(sv[i] - m_safe);      // scores are in units of log 2
    ps += pv[i];
  }
  pf.u = make_uint4(pack_bf16x2(pv[0], pv[1]), pack_bf16x2(pv[2], pv[3]), pack_bf16x2(pv[4], pv[5]),
                    pack_bf16x2(pv[6], pv[7]));
  // the running maximum settles after a few blocks; then nothing needs rescaling
  if (__builtin_amdgcn_ballot_w64(m_new != m) != 0) {
    const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
    l *= alpha;
#pragma unroll
    for (int d = 0; d < HD / 16; ++d)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[d][i] *= alpha;
    m = m_new;
  }
  l += ps;
#pragma unroll
  for (int d = 0; d < HD / 16; ++d)
    o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.v[d].v, pf.v, o[d], 0, 0, 0);
}

// Walk blocks first, first + stride, ... (n of them) of one request, two at a time.
// The page ids of 64 blocks are fetched at once, one per lane, so that the walk waits
// for the block table once per 1024 positions and not once per block; within such a
// run the loads of the next pairs are in flight while a pair is computed (two fragment
// sets take turns; loads past the end repeat the last block and are not used).
// `check(block)` tells whether a block needs masks.
struct NoHook {
  __device__ __forceinline__ void operator()() const {}
};

// `after_table` runs once, right after the first load of page ids has been issued, and
// `before_attend` once, after the loads of the first pair have been issued, `after_second` once, after those of
// the second, and before the first pair is computed (all also when there is no block to walk; every wavefront of a
// workgroup runs each exactly once, so they may hold a barrier).  Loads come back in the
// order they were issued: what a caller asks for in `after_table` arrives before the keys
// and values, and what it computes in `before_attend` runs while those are in flight.
template <int HD, typename Check, typename AfterTable = NoHook, typename BeforeAttend = NoHook,
          typename AfterSecond = NoHook>
__device__ __forceinline__ void walk_blocks(const PagedKV& kv, const Frag8* qf, int first, int stride, int n,
                                            int lo, int hi, int kv_last, float scale, Check check, float& m,
                                            float& l, floatx4* o, AfterTable after_table = NoHook{},
                                            BeforeAttend before_attend = NoHook{}, float cap2 = 0.f,
                                            AfterSecond after_second = NoHook{}) {
  const int lane = threadIdx.x & 63;
  bool hooks_due = true;
  for (int c0 = 0; c0 == 0 || c0 < n; c0 += 64) {      // (once at least: the hooks)
    const int nc = max(0, min(64, n - c0));
    int mine = -1;
    if (lane < nc) mine = kv.table[((first + (c0 + lane) * stride) * 16) / kv.P];
    if (hooks_due) {
      __builtin_amdgcn_sched_barrier(0);
      after_table();
      __builtin_amdgcn_sched_barrier(0);
    }
    KVPair<HD> f0, f1;
    BlockInfo a0, b0, a1, b1;
    // block j of this run, clamped to the run's last block
    auto info = [&](int j, int& page) {
      const int jc = max(0, min(j, nc - 1));
      const int blk = first + (c0 + jc) * stride;
      page = __builtin_amdgcn_readlane(mine, jc);
      return BlockInfo{blk * 16, j < nc && page >= 0, check(blk)};
    };
    auto issue = [&](int j, KVPair<HD>& f, BlockInfo& A, BlockInfo& B) {
      int pa, pb;
      A = info(j, pa);
      B = info(j + 1, pb);
      load_pair<HD>(kv, max(pa, 0), A.key0, max(pb, 0), B.key0, f);
    };
    issue(0, f0, a0, b0);
    if (hooks_due) {
      __builtin_amdgcn_sched_barrier(0);
      before_attend();
      __builtin_amdgcn_sched_barrier(0);
    }
    issue(2, f1, a1, b1);
    if (hooks_due) {
      __builtin_amdgcn_sched_barrier(0);
      after_second();
      hooks_due = false;
    }
    for (int i = 0; i < nc; i += 4) {
      attend_pair<HD>(f0, qf, a0, b0, lo, hi, kv_last, scale, m, l, o, cap2);
      if (i + 2 >= nc) break;
      issue(i + 4, f0, a0, b0);
      attend_pair<HD>(f1, qf, a1, b1, lo, hi, kv_last, scale, m, l, o, cap2);
      issue(i + 6, f1, a1, b1);
    }
  }
}

// f(integral_constant<int, 0>), f(<1>), ... f(<N - 1>), until one returns false
template <typename F, int... Is>
__device__ __forceinline__ void unrolled_while_impl(F&& f, std::integer_sequence<int, Is...>) {
  (void)(f(std::integral_constant<int, Is>{}) && ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled_while(F&& f) {
  unrolled_while_impl(f, std::make_integer_sequence<int, N>{});
}

// ---- the same walk with the operands through LDS
// As operands straight from memory a pair's keys lie with a row in every lane, and a load of 1 KiB takes the unit that takes addresses 64
// cycles; direct loads of four whole rows each take 16.
// A wavefront has ST stages of its own, of a pair each, and meets no barrier; a stage is asked for again as soon as it lies in registers.
// With it, the arguments asked for beside the record, and the merge of the columns in use alone, a launch at 16 heads, 8 for keys, in a
// chain of 28 (us, straight from memory before): 1 row of 200 7.6 -> 5.7, 8 of 2,048 in four runs with their merge 19.7 -> 17.9, 2 of
// 16,000 in sixteen 30.0 -> 27.7, 23 of 900 in two 27.9 -> 22.9, 64 of 200 17.6 -> 14.6, 64 of 2,048 99.5 -> 98.4 (5.5 TB/s).  What is left
// of the shortest: 1.5 until its loads are out, 2.5 until they are back (a unit takes about 50 bytes a ns), 1.3 for two pairs, 0.7 the merge.
//
// Row R of a pair's keys (block A's 16, then block B's) lies at R HD 2 bytes with piece c (16 bytes) in place c ^ f(R),
// f(R) = R % 4 + 4 ((R / 8) % 4): the rows that sixteen lanes read together differ in it.  The values of a block lie as in a page of 16
// rows, 32 bytes a dim: LDS serves lanes 0 to 3, 12 to 15 and 20 to 27 together, which are dims 0 to 3 and 12 to 15 of one half and 4 to 11 of
// the other, sixteen different places (1.8 ns a read of a unit; with the halves of some dims exchanged 3.4).
typedef unsigned v4u __attribute__((ext_vector_type(4)));

template <int HD> struct StagedPairs {
  static constexpr int NP = HD / 8;                      // pieces of a key row
  static constexpr int ROWS = 64 / NP;                   // key rows a load
  static constexpr int K_LOADS = 32 / ROWS, V_LOADS = HD / 32;   // of a pair's keys, of one block's values
  static constexpr int LOADS = K_LOADS + 2 * V_LOADS;
  static constexpr unsigned K_BYTES = 32 * HD * 2, V_BYTES = 16 * HD * 2, BYTES = K_BYTES + 2 * V_BYTES;
  static_assert(2 * LOADS <= 63, "vmcnt counts to 63");

  unsigned k_at[HD / 32], v_at;       // LDS: this lane's pieces of the operands in stage 0
  unsigned k_lane, v_lane;            // memory: this lane's piece of a load, in bytes
  unsigned lds;                       // stage 0 of this wavefront

  __device__ __forceinline__ StagedPairs(unsigned lds_, int P) : lds(lds_) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, quad = lane >> 4;
    const int R = ((r16 >> 2) << 3) | (r16 & 3);
    const int f = r16 & (NP - 1);                        // f(R): bits 0, 1 and 3, 4 of R
#pragma unroll
    for (int s = 0; s < HD / 32; ++s) k_at[s] = lds + R * (HD * 2) + (((s * 4 + quad) ^ f) << 4);
    v_at = lds + K_BYTES + (quad >> 1) * V_BYTES + r16 * 32 + ((quad & 1) << 4);
    const int row = lane / NP, c = lane % NP;            // of a load's rows; bits 2 of R and above come with the load's number
    k_lane = (unsigned)(row * HD * 2 + ((c ^ (row & 3)) << 4));
    v_lane = (unsigned)((lane >> 1) * P * 2 + ((lane & 1) << 4));
  }
  // the loads of a pair into the stage at `stage` (bytes); pages that exist, as for load_pair
  __device__ __forceinline__ void ask(const PagedKV& kv, int pageA, int keyA, int pageB, int keyB, unsigned stage) const {
    const size_t page_elems = (size_t)2 * kv.n_kv * kv.P * HD, head_elems = (size_t)kv.P * HD;
    const bf16_t* ka = kv.pool + (size_t)pageA * page_elems + kv.kvh * head_elems;
    const bf16_t* kb = kv.pool + (size_t)pageB * page_elems + kv.kvh * head_elems;
    const bf16_t* va = ka + kv.n_kv * head_elems;
    const bf16_t* vb = kb + kv.n_kv * head_elems;
    if (kv.P != 16) {
      const int rowA = keyA % kv.P, rowB = keyB % kv.P;
      ka += (size_t)rowA * HD;
      kb += (size_t)rowB * HD;
      va += rowA;
      vb += rowB;
    }
    const unsigned to = lds + stage;
    constexpr int HALF = K_LOADS / 2;                    // a block's
    // (as buffer loads: the compiler waits for everything under way where one of the others' kind is)
    const auto rows_at = [](const bf16_t* p) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000); };
    const auto rs_ka = rows_at(ka), rs_kb = rows_at(kb), rs_va = rows_at(va), rs_vb = rows_at(vb);
    unrolled_while<K_LOADS>([&](auto tag) __attribute__((always_inline)) {
      constexpr int g = decltype(tag)::value;
      constexpr unsigned flip = (unsigned)((((g * ROWS) >> 3) << 2) & (NP - 1)) << 4;      // of the load's first row, the same in every lane
      // (what is constant is added to both addresses)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(g < HALF ? rs_ka : rs_kb, (__attribute__((address_space(3))) void*)(size_t)(to + (g / HALF) * HALF * 1024),
                                               16, k_lane ^ flip, 0, (g % HALF) * 1024, 0);
      return true;
    });
#pragma unroll
    for (int g = 0; g < V_LOADS; ++g) {
      const unsigned v_to = to + K_BYTES + g * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_va, (__attribute__((address_space(3))) void*)(size_t)v_to, 16, v_lane, g * 64 * kv.P, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_vb, (__attribute__((address_space(3))) void*)(size_t)(v_to + V_BYTES), 16, v_lane, g * 64 * kv.P, 0, 0);
    }
  }
  // the operands of the pair in stage number S, in registers when this returns (they have landed in LDS before)
  template <int S> __device__ __forceinline__ void read(KVPair<HD>& f) const {
    constexpr int OFF = S * (int)BYTES;
    v4u k[2][HD / 32], v[HD / 16];
    if constexpr (HD == 128)
      asm volatile("ds_read_b128 %0, %16 offset:%21\n\tds_read_b128 %1, %17 offset:%21\n\tds_read_b128 %2, %18 offset:%21\n\t"
                   "ds_read_b128 %3, %19 offset:%21\n\tds_read_b128 %4, %16 offset:%21+1024\n\tds_read_b128 %5, %17 offset:%21+1024\n\t"
                   "ds_read_b128 %6, %18 offset:%21+1024\n\tds_read_b128 %7, %19 offset:%21+1024\n\t"
                   "ds_read_b128 %8, %20 offset:%21\n\tds_read_b128 %9, %20 offset:%21+512\n\tds_read_b128 %10, %20 offset:%21+1024\n\t"
                   "ds_read_b128 %11, %20 offset:%21+1536\n\tds_read_b128 %12, %20 offset:%21+2048\n\tds_read_b128 %13, %20 offset:%21+2560\n\t"
                   "ds_read_b128 %14, %20 offset:%21+3072\n\tds_read_b128 %15, %20 offset:%21+3584\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]), "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2]),
                     "=&v"(k[1][3]), "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]), "=&v"(v[6]), "=&v"(v[7])
                   : "v"(k_at[0]), "v"(k_at[1]), "v"(k_at[2]), "v"(k_at[3]), "v"(v_at), "n"(OFF)
                   : "memory");
    else
      asm volatile("ds_read_b128 %0, %8 offset:%11\n\tds_read_b128 %1, %9 offset:%11\n\tds_read_b128 %2, %8 offset:%11+512\n\t"
                   "ds_read_b128 %3, %9 offset:%11+512\n\tds_read_b128 %4, %10 offset:%11\n\tds_read_b128 %5, %10 offset:%11+512\n\t"
                   "ds_read_b128 %6, %10 offset:%11+1024\n\tds_read_b128 %7, %10 offset:%11+1536\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                   : "v"(k_at[0]), "v"(k_at[1]), "v"(v_at), "n"(OFF)
                   : "memory");
#pragma unroll
    for (int s = 0; s < HD / 32; ++s) {
      f.k[0][s].v = __builtin_bit_cast(bf16x8, k[0][s]);
      f.k[1][s].v = __builtin_bit_cast(bf16x8, k[1][s]);
    }
#pragma unroll
    for (int d = 0; d < HD / 16; ++d) f.v[d].v = __builtin_bit_cast(bf16x8, v[d]);
  }
};

// walk_blocks through ST stages (launches by records: the ids of the first four blocks are given, whatever the run's length).  The hooks
// come as there, none of them may touch LDS but by instructions of its own (the compiler would wait for every load that is under way).
// Behind the first pair nothing is asked for beyond the run's end.
template <int HD, int ST, typename Check, typename AfterTable = NoHook, typename BeforeAttend = NoHook, typename AfterSecond = NoHook>
__device__ __forceinline__ void walk_staged(const StagedPairs<HD>& st, const PagedKV& kv, const Frag8* qf, int first, int stride, int n,
                                            int lo, int hi, int kv_last, float scale, Check check, float& m, float& l, floatx4* o,
                                            AfterTable after_table, BeforeAttend before_attend, float cap2, int held, int held_id,
                                            const int* first4, AfterSecond after_second) {
  static_assert(ST == 1 || ST == 2, "a pair, or two");
  const int lane = threadIdx.x & 63;
  int c0 = 0, nc = min(64, n);               // the run of up to 64 blocks whose page ids the lanes hold, as in walk_blocks
  int mine = -1;
  auto ids = [&](int have) __attribute__((always_inline)) {
    const auto table = (const __attribute__((address_space(1))) int*)kv.table;      // (in memory, here)
    if (nc > have && lane >= have && lane < nc) mine = table[((first + (c0 + lane) * stride) * 16) / kv.P];
  };
  BlockInfo a[ST], b[ST];
  // the loads of blocks j and j + 1 of the run, on pages pa and pb
  auto issue = [&](int j, auto stage_tag, int pa, int pb) __attribute__((always_inline)) {
    constexpr int S = decltype(stage_tag)::value;
    const int blk_a = first + (c0 + j) * stride, blk_b = first + (c0 + min(j + 1, max(nc - 1, 0))) * stride;
    a[S] = BlockInfo{blk_a * 16, j < nc && pa >= 0, check(blk_a)};
    b[S] = BlockInfo{blk_b * 16, j + 1 < nc && pb >= 0, check(blk_b)};
    st.ask(kv, max(pa, 0), a[S].key0, max(pb, 0), b[S].key0, S * StagedPairs<HD>::BYTES);
  };
  auto issue_held = [&](int j, auto stage_tag) __attribute__((always_inline)) {
    issue(j, stage_tag, __builtin_amdgcn_readlane(mine, j), __builtin_amdgcn_readlane(mine, min(j + 1, nc - 1)));
  };
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, ST - 1>;
  ids(held);               // (those that the record does not hold)
  __builtin_amdgcn_sched_barrier(0);
  after_table();
  __builtin_amdgcn_sched_barrier(0);
  // (without a condition, whatever there is to walk: the compiler counts these loads where `before_attend` waits for what
  // `after_table` asked for)
  issue(0, S0{}, first4[0], first4[1]);
  __builtin_amdgcn_sched_barrier(0);
  before_attend();
  __builtin_amdgcn_sched_barrier(0);
  if (ST > 1 && nc > 2) issue(2, S1{}, first4[2], first4[3]);
  __builtin_amdgcn_sched_barrier(0);
  after_second();
  if (lane < min(nc, held)) mine = held_id;
  auto turn = [&](int i, auto stage_tag) __attribute__((always_inline)) {
    constexpr int S = decltype(stage_tag)::value;
    KVPair<HD> f;
    if (ST > 1 && i + 2 < nc) wait_vmcnt<StagedPairs<HD>::LOADS>();
    else wait_vmcnt<0>();
    st.template read<S>(f);
    const BlockInfo A = a[S], B = b[S];
    if (i + 2 * ST < nc) issue_held(i + 2 * ST, stage_tag);
    attend_pair<HD>(f, qf, A, B, lo, hi, kv_last, scale, m, l, o, cap2);
  };
  while (true) {
    for (int i = 0; i < nc; i += 2 * ST) {
      turn(i, S0{});
      if (ST > 1 && i + 2 < nc) turn(i + 2, S1{});
    }
    c0 += 64;
    if (c0 >= n) break;
    nc = min(64, n - c0);
    ids(0);
    issue_held(0, S0{});
    if (ST > 1 && nc > 2) issue_held(2, S1{});
  }
  wait_vmcnt<0>();      // (a wavefront without blocks: what it leaves in its stage comes after the loads)
}

// ------------------------------------------- queries and the new key prepared in place
// What the decode kernel needs to start from the 32-bit projections instead of prepared
// queries: it norms and rotates its own query heads, and the workgroup whose blocks hold the
// row's own position writes that position's key and value into the cache before it walks.
struct QKPrep {
  const float* qkv;          // [rows, row_width]: q heads, then (if keys are written) k heads, v heads
  int row_width;
  const float* q_w;          // per-head norm weights or nullptr
  const float* k_w;
  float eps;
  const float* inv_freq;     // nullptr: no rotation
  const float2* rope_table;  // (cos, sin) [table_len][hd / 2] or nullptr
  int table_len;
  bf16_t* pool_w;            // the cache to write the new key and value into; nullptr: nothing is written
};

// One head of the row by one wavefront, in two steps, so that the loads of keys and values can go out between them: lane i
// holds pair i.  The arithmetic is qk_head_wave's (the same bits); w null: a value head, rounded alone.
template <int HD>
struct HeadJob {
  static_assert(HD == 64 || HD == 128, "a lane holds one rotation pair at most");
  static constexpr int HALF = HD / 2;
  float lo, hi, wl, wh;
  float2 cs;
  bool from_table;
  __device__ __forceinline__ void load(const QKPrep& pr, const float* __restrict__ src, const float* __restrict__ w, int p) {
    const int i = (threadIdx.x & 63) & (HALF - 1);
    lo = src[i];
    hi = src[i + HALF];
    wl = wh = 1.f;
    if (w) {
      wl = w[i];
      wh = w[i + HALF];
    }
    from_table = pr.inv_freq && pr.rope_table && p < pr.table_len;   // the same in every lane
    if (from_table) cs = pr.rope_table[(size_t)p * HALF + i];
  }
  // the pair, finished
  __device__ __forceinline__ void pair(const QKPrep& pr, const float* w, bool value, int p, bf16_t& first, bf16_t& second) {
    const int lane = threadIdx.x & 63;
    float a = lo, b = hi;
    if (!value) {
      if (w) {
        const float scale = qk_norm_scale(group_sum<TI_WAVE>(lane < HALF ? qk_pair_square(lo, hi) : 0.f), HD, pr.eps);
        a *= scale;
        b *= scale;
        a *= wl;
        b *= wh;
      }
      if (pr.inv_freq) {
        if (!from_table) cs = qk_cos_sin(lane & (HALF - 1), HALF, p, pr.inv_freq, nullptr, 0);
        qk_rotate(a, b, cs);
      }
    }
    first = f2bf(a);
    second = f2bf(b);
  }
  // `dst`: HD consecutive elements
  __device__ __forceinline__ void finish(const QKPrep& pr, const float* w, bool value, int p, bf16_t* dst) {
    const int lane = threadIdx.x & 63;
    bf16_t a, b;
    pair(pr, w, value, p, a, b);
    if (lane < HALF) {
      dst[lane] = a;
      dst[lane + HALF] = b;
    }
  }
  // the same into LDS (its byte address) while direct loads into other parts of it are under way: written as an instruction, or the
  // compiler would have it wait for them
  __device__ __forceinline__ void finish_lds(const QKPrep& pr, const float* w, bool value, int p, unsigned dst) {
    const int lane = threadIdx.x & 63;
    bf16_t a, b;
    pair(pr, w, value, p, a, b);
    if (lane < HALF)
      asm volatile("ds_write_b16 %0, %1\n\tds_write_b16 %0, %2 offset:%3" ::"v"(dst + lane * 2), "v"((unsigned)a), "v"((unsigned)b), "n"(HALF * 2)
                   : "memory");
  }
};

// =================================================================== decode
// grid (rows, n_kv * head_parts, splits), 256 threads.  Partials (splits > 1):
//   part_o [row][head][split][hd], part_ml [row][head][split][2] = (max, sum)
// PREP: the queries come from the 32-bit projections (see QKPrep); needs parts == 1.  The row's query heads, and its own
// key and value where a workgroup walks their block, are prepared a head a wavefront and shared through LDS while the first
// keys and values are on their way.  (A lane that prepared its column's head by itself asked for 64 to 112 bytes in 28 loads
// in front of its keys, and kept 100 registers for them: 8 requests of 2,048 tokens at 0.6B 21.8 us a layer, now 17.5.)
// A learned sink in the softmax's denominator: exp(sink[head]) joins the sum where a column is finished (no key, no value,
// not scaled).  m, lt: the column's maximum (in units of log 2) and the sum of its weights; lt becomes the new denominator
// and the factor on the column's unscaled outputs comes back.  sink null: nothing changes.
__device__ __forceinline__ float sink_join(const float* __restrict__ sink, int head, float m, float& lt) {
  if (!sink) return 1.f;
  const float s = sink[head] * TI_LOG2E;
  const float m_new = fmaxf(m, s);
  const float f = (m == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(m - m_new);
  lt = fmaf(lt, f, __builtin_amdgcn_exp2f(s - m_new));
  return f;
}

#define DEC_TABLE_LDS 1024     // entries of a block-table row that the decode kernel can hold in LDS
// The workgroup's LDS: what its NW wavefronts leave for the merge (a column's HD values in a row of HD + 4: sixteen lanes write 16 bytes of as
// many columns at once, and rows of HD floats would put them all into the same banks), and their maxima and sums.
template <int HD, int NW>
struct DecodeMerge {
  float o[NW][16][HD + 4];
  float2 ml[NW][16];
};
// The same where the operands come through LDS stages: a wavefront leaves its outputs in its own first stage.
template <int HD, int NW, int ST>
struct StagedMerge {
  union {
    unsigned char stages[ST][StagedPairs<HD>::BYTES];
    float o[16][HD + 4];
  } w[NW];
  float2 ml[NW][16];
  bf16_t q[16][HD], kv[2][HD];      // the query heads, the row's own key and value (16-byte aligned)
};
// A launch by records (TI_RUN_* in tinyinfer_kernels.h): the host cuts every row's context into runs of its own choice and says what each
// workgroup walks.  Record i, of a launch's `run_stride` ints: the header below, then for each of the workgroup's
// NW wavefronts (run_stride - TI_RUN_HEAD) / NW page ids, at least four: those of the first blocks that it walks (-1: given back;
// beyond the run's end any page of the pool, or a number below 0: loaded, as every loop's last loads are, and not used; asking for
// the run's end first took up to 0.2 us a layer).  A workgroup's first loads are then its header and its page ids, side by side, and its
// keys' are the next.  Runs of no blocks are nobody's:
// their workgroups end at once (a captured graph launches as many records for every step).
struct DecodeRuns {
  const int* runs;      // null: no records, `split` of n_splits equal runs of every row
  int run_stride;
};
// A kernel argument that is to have arrived here.  (Pointers as ones to memory: an asm statement makes others point to anything, and flat
// loads wait for everything under way.)
template <class T> __device__ __forceinline__ void arrived(T& v) { asm volatile("" : "+s"(v)); }
template <class T> __device__ __forceinline__ void arrived(T*& p) {
  auto g = (__attribute__((address_space(1))) T*)p;
  asm volatile("" : "+s"(g));
  p = (T*)g;
}
// One workgroup of NW wavefronts: row `ridx` of the launch, kv head and set of q heads `y`, run `split` of n_splits; or record `ridx`.
// ST: stages of LDS a wavefront takes its operands through, by records; 0: straight from memory, by equal runs
template <int HD, bool PREP, int NW, int ST, class Shared>
__device__ __forceinline__ void
decode_run(Shared& sm, int ridx, int y, int split, const bf16_t* __restrict__ q, const bf16_t* __restrict__ pool,
           const int* __restrict__ table, int table_stride, const int* __restrict__ pos, const int* __restrict__ slot,
           const int* __restrict__ rows, bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
           int n_head, int n_kv, int P, float scale, int window, int n_splits, QKPrep prep, float softcap,
           const float* __restrict__ sink, DecodeRuns by = DecodeRuns{nullptr, 0}, int group = 0) {
  static_assert(!PREP || NW == 4, "the preparation is written for four wavefronts");
  constexpr bool RUNS = ST > 0;
  auto s_o = [&](int w) -> float(&)[16][HD + 4] {
    if constexpr (ST > 0) return sm.w[w].o;
    else return sm.o[w];
  };
  // the wavefront's number in scalar registers, and with it what it walks
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int held = RUNS ? (by.run_stride - TI_RUN_HEAD) / NW : 0;      // lanes whose first block's page id comes with the record
  int held_id = -1, first4[4] = {};
  int rh[TI_RUN_HEAD] = {};
  if constexpr (RUNS) {
    const int* rec = by.runs + (size_t)ridx * by.run_stride;
    const int* ids = rec + TI_RUN_HEAD + wave * held;
    if (lane < held) held_id = ids[lane];
#pragma unroll
    for (int i = 0; i < TI_RUN_HEAD; ++i) rh[i] = rec[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) first4[i] = ids[i];
#pragma unroll
    for (int i = 0; i < TI_RUN_HEAD; ++i) asm volatile("" : "+s"(rh[i]));      // all of it at once
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+s"(first4[i]));
    // so do the arguments that did not come with the wavefront: fetched where they are first needed they are round trips one behind another
    if constexpr (PREP) {
      arrived(prep.q_w), arrived(prep.k_w), arrived(table), arrived(table_stride), arrived(window), arrived(prep.inv_freq);
      arrived(prep.pool_w), arrived(prep.eps), arrived(scale), arrived(out), arrived(part_o), arrived(part_ml);
    }
    if (rh[TI_RUN_BLOCKS] == 0) return;
  }
  const int m_row = RUNS ? rh[TI_RUN_ROW] : rows ? rows[ridx] : ridx;
  const int G = group ? group : n_head / n_kv;       // (a division in the kernel takes longer than an argument)
  const int parts = PREP ? 1 : (G + 15) / 16;        // q heads per kv head, in sets of up to 16 columns
  const int kvh = y / parts, part = y % parts;
  const int r16 = lane & 15, quad = lane >> 4;
  const int n_cols = min(16, G - part * 16);
  const int head = kvh * G + part * 16 + r16;   // valid if r16 < n_cols

  // (By equal runs, for callers of Ops that plan no records and for steps of more rows than a launch has records.)
  // slot == nullptr: row m of the step is row m of the block tables (a step of single tokens, where the
  // host knows it), and a table row has at most DEC_TABLE_LDS entries.  The row's page ids are then asked
  // for at once, all of them, beside the position instead of behind it (which pages the workgroup walks
  // depends on the position), and looked up in LDS afterwards: one round trip to memory less before the
  // first keys can be asked for (0.15 us of the kernel's 19 at batch 8 of Qwen3-0.6B's sizes).
  constexpr bool CAN_EARLY = NW == 4 && !RUNS;
  constexpr int EARLY = CAN_EARLY ? DEC_TABLE_LDS : 1;
  __shared__ int s_table[EARLY];
  const bool early = CAN_EARLY && slot == nullptr;
  int ids[DEC_TABLE_LDS / 256];
  if (early) {
    const int* table_row = table + (size_t)m_row * table_stride;
#pragma unroll
    for (int j = 0; j < DEC_TABLE_LDS / 256; ++j) {
      const int i = threadIdx.x + 256 * j;
      ids[j] = i < table_stride ? table_row[i] : -1;
    }
  }
  const int p_q = RUNS ? rh[TI_RUN_POS] : pos[m_row];
  const int lo = (window > 0 && p_q - window + 1 > 0) ? p_q - window + 1 : 0;
  const int blk_lo = lo / 16, blk_hi = p_q / 16;
  const int n_blk = blk_hi - blk_lo + 1;
  const int per = (n_blk + n_splits - 1) / n_splits;
  const int b0 = RUNS ? rh[TI_RUN_FIRST] : blk_lo + split * per;
  const int b1 = RUNS ? b0 + rh[TI_RUN_BLOCKS] : min(blk_hi + 1, b0 + per);
  // where the results go: straight out, or to place part_at + part_step * head of the partial results
  const bool whole = RUNS ? rh[TI_RUN_PART] < 0 : n_splits == 1;
  const size_t part_at = RUNS ? (size_t)rh[TI_RUN_PART] * n_head : (size_t)ridx * n_head * n_splits + split;
  const int part_step = RUNS ? 1 : n_splits;
  if (early) {
#pragma unroll
    for (int j = 0; j < DEC_TABLE_LDS / 256; ++j)
      if constexpr (CAN_EARLY) s_table[threadIdx.x + 256 * j] = ids[j];
    __syncthreads();
  }

  PagedKV kv{pool, early ? s_table : table + (size_t)(RUNS ? rh[TI_RUN_TABLE_ROW] : slot[m_row]) * table_stride, P, n_kv, kvh};
  Frag8 qf[HD / 32];
  float mx = -INFINITY, l = 0.f;
  floatx4 o[HD / 16];
#pragma unroll
  for (int d = 0; d < HD / 16; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int mine = (b1 - (b0 + wave) + NW - 1) / NW;   // blocks b0 + wave, + NW, ... below b1
  auto edge = [=](int b) { return (lo > 0 && b == blk_lo) || b == blk_hi; };
  bool own_key = false;
  if constexpr (PREP) {
    const float* row = prep.qkv + (size_t)m_row * prep.row_width;
    // The workgroup that walks the block of the row's own position prepares the position's key and value as well: from LDS
    // they go into the cache for later steps, and into this step's attention as a block of their own, so nothing waits for
    // the cache to hold them.
    own_key = prep.pool_w && blk_hi >= b0 && blk_hi < b1;
    const int last = own_key ? p_q - 1 : p_q;      // what the cache holds for this workgroup
    const int n_jobs = n_cols + (own_key ? 2 : 0);
    HeadJob<HD> job;
    auto job_load = [&](int j) {
      const int h = j < n_cols ? kvh * G + j : j == n_cols ? n_head + kvh : n_head + n_kv + kvh;
      job.load(prep, row + (size_t)h * HD, j < n_cols ? prep.q_w : j == n_cols ? prep.k_w : nullptr, p_q);
    };
    if constexpr (ST > 0) {
      const unsigned q_lds = (unsigned)(size_t)&sm.q[0][0], kv_lds = (unsigned)(size_t)&sm.kv[0][0];
      auto finish = [&](int j) {
        job.finish_lds(prep, j < n_cols ? prep.q_w : prep.k_w, j > n_cols, p_q,
                       j < n_cols ? q_lds + j * (HD * 2) : kv_lds + (j - n_cols) * (HD * 2));
      };
      // HD / 32 operands of 16 bytes, 64 bytes apart
      auto operands = [&](unsigned at, Frag8* f) {
        v4u e[HD / 32];
        if constexpr (HD == 128)
          asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:64\n\tds_read_b128 %2, %4 offset:128\n\t"
                       "ds_read_b128 %3, %4 offset:192\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(e[0]), "=&v"(e[1]), "=&v"(e[2]), "=&v"(e[3]) : "v"(at) : "memory");
        else
          asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:64\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(e[0]), "=&v"(e[1]) : "v"(at) : "memory");
#pragma unroll
        for (int s = 0; s < HD / 32; ++s) f[s].v = __builtin_bit_cast(bf16x8, e[s]);
      };
      const StagedPairs<HD> st((unsigned)(size_t)&sm.w[wave], P);
      walk_staged<HD, ST>(
          st, kv, qf, b0 + wave, NW, mine, lo, last, last, scale * TI_LOG2E, edge, mx, l, o,
          [&]() {
            if (wave < n_jobs) job_load(wave);
          },
          [&]() {
            for (int j = wave; j < n_jobs; j += NW) {
              if (j != wave) job_load(j);
              finish(j);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            operands(q_lds + min(r16, n_cols - 1) * (HD * 2) + quad * 16, qf);
#pragma unroll
            for (int s = 0; s < HD / 32; ++s)
              if (r16 >= n_cols) qf[s].u = make_uint4(0, 0, 0, 0);
          },
          0.f, held, held_id, first4,
          [&]() {
            if (!own_key || wave != 0) return;
            // the row's own key and value come first: their score is the maximum, their weight 1
            floatx4 sc = {0.f, 0.f, 0.f, 0.f};
            Frag8 k[HD / 32];
            operands(kv_lds + quad * 16, k);
#pragma unroll
            for (int s = 0; s < HD / 32; ++s) {
              if (r16 != 0) k[s].u = make_uint4(0, 0, 0, 0);
              sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[s].v, qf[s].v, sc, 0, 0, 0);
            }
            mx = __shfl(sc[0], r16, 64) * (scale * TI_LOG2E);      // row 0 of the tile lies in the first sixteen lanes
            l = quad == 0 ? 1.f : 0.f;                             // the lanes of a column are added at the end
            // dims 16 d + 4 quad .. + 3, eight bytes of every 32
            typedef unsigned v2u __attribute__((ext_vector_type(2)));
            v2u e[HD / 16];
            const unsigned at = kv_lds + HD * 2 + quad * 8;
            asm volatile("ds_read_b64 %0, %4\n\tds_read_b64 %1, %4 offset:32\n\tds_read_b64 %2, %4 offset:64\n\t"
                         "ds_read_b64 %3, %4 offset:96\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(e[0]), "=&v"(e[1]), "=&v"(e[2]), "=&v"(e[3]) : "v"(at) : "memory");
            if constexpr (HD == 128)
              asm volatile("ds_read_b64 %0, %4 offset:128\n\tds_read_b64 %1, %4 offset:160\n\tds_read_b64 %2, %4 offset:192\n\t"
                           "ds_read_b64 %3, %4 offset:224\n\ts_waitcnt lgkmcnt(0)"
                           : "=&v"(e[HD / 16 - 4]), "=&v"(e[HD / 16 - 3]), "=&v"(e[HD / 16 - 2]), "=&v"(e[HD / 16 - 1]) : "v"(at) : "memory");
#pragma unroll
            for (int d = 0; d < HD / 16; ++d)
#pragma unroll
              for (int i = 0; i < 4; ++i) o[d][i] = __uint_as_float((i & 1) ? e[d][i >> 1] & 0xffff0000u : e[d][i >> 1] << 16);
          });
    } else {
      __shared__ __attribute__((aligned(16))) bf16_t s_q[16][HD];       // the query heads
      __shared__ __attribute__((aligned(16))) bf16_t s_kv[2][HD];       // the row's own key, then its value
      auto job_finish = [&](int j) {
        job.finish(prep, j < n_cols ? prep.q_w : prep.k_w, j > n_cols, p_q, j < n_cols ? s_q[j] : s_kv[j - n_cols]);
      };
      walk_blocks<HD>(
          kv, qf, b0 + wave, NW, mine, lo, last, last, scale * TI_LOG2E, edge, mx, l, o,
          [&]() {
            if (wave < n_jobs) job_load(wave);
          },
          [&]() {
            for (int j = wave; j < n_jobs; j += NW) {
              if (j != wave) job_load(j);
              job_finish(j);
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < HD / 32; ++s)
              qf[s].u = r16 < n_cols ? *reinterpret_cast<const uint4*>(&s_q[r16][s * 32 + quad * 8]) : make_uint4(0, 0, 0, 0);
          },
          0.f,
          [&]() {
            if (!own_key) return;
            if (wave == 0) {
              // the row's own key and value come first: their score is the maximum, their weight 1
              floatx4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int s = 0; s < HD / 32; ++s) {
                Frag8 k;
                k.u = (r16 == 0) ? *reinterpret_cast<const uint4*>(&s_kv[0][s * 32 + quad * 8]) : make_uint4(0, 0, 0, 0);
                sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k.v, qf[s].v, sc, 0, 0, 0);
              }
              mx = __shfl(sc[0], r16, 64) * (scale * TI_LOG2E);      // row 0 of the tile lies in the first sixteen lanes
              l = quad == 0 ? 1.f : 0.f;                             // the lanes of a column are added at the end
#pragma unroll
              for (int d = 0; d < HD / 16; ++d)
#pragma unroll
                for (int i = 0; i < 4; ++i) o[d][i] = bf2f(s_kv[1][d * 16 + quad * 4 + i]);
            } else if (wave == NW - 1) {
              const int page = kv.table[p_q / P];
              if (page >= 0) {    // the host reserves pages first; never write astray
                bf16_t* kd = kv_page_slot<bf16_t>(prep.pool_w, page, 0, kvh, p_q % P, n_kv, P, HD);
                bf16_t* vd = kv_page_slot<bf16_t>(prep.pool_w, page, 1, kvh, p_q % P, n_kv, P, HD);
                for (int i = lane; i < HD; i += 64) {
                  kd[i] = s_kv[0][i];
                  vd[(size_t)i * P] = s_kv[1][i];
                }
              }
            }
          });
    }
  } else {
#pragma unroll
    for (int s = 0; s < HD / 32; ++s) {
      qf[s].u = make_uint4(0, 0, 0, 0);
      if (r16 < n_cols)
        qf[s].u = *reinterpret_cast<const uint4*>(q + ((size_t)m_row * n_head + head) * HD + s * 32 + quad * 8);
    }
    if constexpr (ST > 0)
      walk_staged<HD, ST>(StagedPairs<HD>((unsigned)(size_t)&sm.w[wave], P), kv, qf, b0 + wave, NW, mine, lo, p_q, p_q,
                          scale * TI_LOG2E, edge, mx, l, o, NoHook{}, NoHook{}, softcap * TI_LOG2E, held, held_id, first4, NoHook{});
    else
      walk_blocks<HD>(kv, qf, b0 + wave, NW, mine, lo, p_q, p_q, scale * TI_LOG2E, edge, mx, l, o, NoHook{}, NoHook{},
                      softcap * TI_LOG2E);
  }
  if constexpr (ST > 0) {
    const LanePair near = lane_pair<16>(l);
    l = near.a + near.b;
    const LanePair far = lane_pair<32>(l);
    l = far.a + far.b;
  } else {      // (with the lanes swapped as above the compiler takes 19 to 34 registers more: at a head size of 64 three wavefronts a SIMD, not four)
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
  }

  // merge the wavefronts: what the columns in use hold, four values of a column a thread.  (A wavefront's dims of all sixteen columns,
  // eight of its lanes at work, took 0.95 us from the barrier to the end where this takes 0.45.)
  if (r16 < n_cols) {
#pragma unroll
    for (int d = 0; d < HD / 16; ++d) *reinterpret_cast<floatx4*>(&s_o(wave)[r16][d * 16 + quad * 4]) = o[d];
    if (quad == 0) sm.ml[wave][r16] = make_float2(mx, l);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n_cols * (HD / 4); i += 64 * NW) {
    const int col = i / (HD / 4), dim = i % (HD / 4) * 4, at = kvh * G + part * 16 + col;
    floatx4 v[NW];
    float2 ml[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      ml[w] = sm.ml[w][col];
      v[w] = *reinterpret_cast<const floatx4*>(&s_o(w)[col][dim]);
    }
    float mm = -INFINITY, lt = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) mm = fmaxf(mm, ml[w].x);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float wgt = (ml[w].x == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(ml[w].x - mm);
      lt += ml[w].y * wgt;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += v[w][e] * wgt;
    }
    if (whole) {
      float den = lt;
      const float inv = sink_join(sink, at, mm, den) / den;
      *reinterpret_cast<uint2*>(out + ((size_t)m_row * n_head + at) * HD + dim) =
          make_uint2(pack_bf16x2(acc[0] * inv, acc[1] * inv), pack_bf16x2(acc[2] * inv, acc[3] * inv));
    } else {
      const size_t place = part_at + (size_t)part_step * at;
      *reinterpret_cast<float4*>(part_o + place * HD + dim) = make_float4(acc[0], acc[1], acc[2], acc[3]);
      if (dim == 0) reinterpret_cast<float2*>(part_ml)[place] = make_float2(mm, lt);
    }
  }
  // the row's own key and value, for later steps: nobody waits for these stores
  if constexpr (PREP && ST > 0) {
    if (own_key && wave == NW - 1 && rh[TI_RUN_OWN_PAGE] >= 0) {    // the host reserves pages first; never write astray
      const int page = rh[TI_RUN_OWN_PAGE];
      bf16_t* kd = kv_page_slot<bf16_t>(prep.pool_w, page, 0, kvh, p_q % P, n_kv, P, HD);
      bf16_t* vd = kv_page_slot<bf16_t>(prep.pool_w, page, 1, kvh, p_q % P, n_kv, P, HD);
      for (int i = lane; i < HD; i += 64) {
        kd[i] = sm.kv[0][i];
        vd[(size_t)i * P] = sm.kv[1][i];
      }
    }
  }
}

template <int HD, bool PREP>
__global__ void __launch_bounds__(256, 2)
attn_decode_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ pool, const int* __restrict__ table,
                   int table_stride, const int* __restrict__ pos, const int* __restrict__ slot,
                   const int* __restrict__ rows, bf16_t* __restrict__ out, float* __restrict__ part_o,
                   float* __restrict__ part_ml, int n_head, int n_kv, int P, float scale, int window,
                   int n_splits, QKPrep prep, float softcap = 0.f, const float* __restrict__ sink = nullptr) {
  __shared__ DecodeMerge<HD, 4> sm;
  decode_run<HD, PREP, 4, 0>(sm, blockIdx.x, blockIdx.y, blockIdx.z, q, pool, table, table_stride, pos, slot, rows,
                                         out, part_o, part_ml, n_head, n_kv, P, scale, window, n_splits, prep, softcap, sink);
}

// The same from the projections, by records: grid (n_kv, records).  A launch's workgroups differ by what the host gave them:
// with every row in as many runs a launch lasted as long as the longest row asks.
// (The arguments that the first loads need come first: they arrive in scalar registers with the wavefront.)
template <int HD, int ST>
__global__ void __launch_bounds__(256, 2)
attn_decode_runs_kernel(const int* __restrict__ runs, int run_stride, int group, const float* __restrict__ qkv, int row_width,
                        int n_kv, const float2* __restrict__ rope_table, const bf16_t* __restrict__ pool, int P, int table_len,
                        const float* __restrict__ q_w, const float* __restrict__ k_w, const int* __restrict__ table,
                        int table_stride, int window, const float* __restrict__ inv_freq, bf16_t* __restrict__ pool_w, float eps, float scale,
                        bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const QKPrep prep{qkv, row_width, q_w, k_w, eps, inv_freq, rope_table, table_len, pool_w};
  decode_run<HD, true, 4, ST>(*reinterpret_cast<StagedMerge<HD, 4, ST>*>(smem), blockIdx.y, blockIdx.x, 0, nullptr, pool, table, table_stride, nullptr, nullptr, nullptr,
                                out, part_o, part_ml, group * n_kv, n_kv, P, scale, window, 1, prep, 0.f, nullptr,
                                DecodeRuns{runs, run_stride}, group);
}

// grid (rows, n_head), max(HD, 64) threads: out = sum_s w_s o_s / sum_s w_s l_s, w_s = 2^(m_s - max m).
// The partial outputs are fetched in batches of eight independent loads: the kernel waits for
// memory a few times, not once per split.
#define MERGE_MAX_SPLITS 64
// RECORDS: `rows` holds (row, first run's place, runs, -) of every row, whose run s lies at [first + s][head]; a row of one
// run has its result already.
template <int HD, bool RECORDS = false>
__global__ void __launch_bounds__(HD < 64 ? 64 : HD)
attn_merge_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                  const int* __restrict__ rows, bf16_t* __restrict__ out, int n_head, int n_splits,
                  const float* __restrict__ sink = nullptr) {
  const int ridx = blockIdx.x, head = blockIdx.y, d = threadIdx.x;
  if (d >= HD) return;
  int m_row;
  size_t at, step;                    // the runs' places: at, at + step, ...
  if constexpr (RECORDS) {
    n_splits = rows[4 * ridx + 2];
    if (n_splits < 2) return;
    m_row = rows[4 * ridx];
    at = (size_t)rows[4 * ridx + 1] * n_head + head;
    step = n_head;
  } else {
    m_row = rows ? rows[ridx] : ridx;
    at = ((size_t)ridx * n_head + head) * n_splits;
    step = 1;
  }
  const float2* pm = reinterpret_cast<const float2*>(part_ml) + at;
  const float* po = part_o + at * HD + d;
  // every thread works the weights of the splits out for itself: they are few, and no thread waits
  // for another.  Up to 32 splits: everything asked for at once, one round trip to memory (splits
  // beyond the last repeat it and count for nothing).
  auto at_once = [&](auto cap_tag) {
    constexpr int CAP = decltype(cap_tag)::value;
    float v[CAP];
    float2 ml[CAP];
#pragma unroll
    for (int j = 0; j < CAP; ++j) {
      const int sj = j < n_splits ? j : n_splits - 1;
      ml[j] = pm[sj * step];
      v[j] = po[sj * step * HD];
    }
    float mm = -INFINITY;
#pragma unroll
    for (int j = 0; j < CAP; ++j)
      if (j < n_splits) mm = fmaxf(mm, ml[j].x);
    float acc = 0.f, lt = 0.f;
#pragma unroll
    for (int j = 0; j < CAP; ++j)
      if (j < n_splits) {
        const float w = split_weight(ml[j].x, mm);
        lt = fmaf(ml[j].y, w, lt);
        acc = split_accumulate(acc, v[j], w);
      }
    const float f = sink_join(sink, head, mm, lt);
    out[((size_t)m_row * n_head + head) * HD + d] = f2bf(acc * (f / lt));
  };
  if (n_splits <= 8) {
    at_once(std::integral_constant<int, 8>{});
    return;
  }
  if (n_splits <= 16) {
    at_once(std::integral_constant<int, 16>{});
    return;
  }
  if (n_splits <= 32) {      // (run by run 17 took 6 us longer than 16)
    at_once(std::integral_constant<int, 32>{});
    return;
  }
  float mm = -INFINITY;
  for (int s = 0; s < n_splits; ++s) mm = fmaxf(mm, pm[s * step].x);
  float acc = 0.f, lt = 0.f;
  int s = 0;
  for (; s + 8 <= n_splits; s += 8) {
    float v[8];
    float2 ml[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = po[(s + j) * step * HD];
      ml[j] = pm[(s + j) * step];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float w = split_weight(ml[j].x, mm);
      lt = fmaf(ml[j].y, w, lt);
      acc = split_accumulate(acc, v[j], w);
    }
  }
  for (; s < n_splits; ++s) {
    const float2 ml = pm[s * step];
    const float w = split_weight(ml.x, mm);
    lt = fmaf(ml.y, w, lt);
    acc = split_accumulate(acc, po[s * step * HD], w);
  }
  const float f = sink_join(sink, head, mm, lt);
  out[((size_t)m_row * n_head + head) * HD + d] = f2bf(acc * (f / lt));
}

// ================================================================== prefill
// grid (tiles, n_head), 512 threads.  tiles[t] = (entry, first row); entries[e] =
// (row0, n_tokens, start_pos, -).  A tile is 128 rows; wavefront w takes rows
// first + 16 w .. + 15 as its columns.
template <int HD>
__global__ void __launch_bounds__(512)
attn_prefill_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ pool, const int* __restrict__ table,
                    int table_stride, const int* __restrict__ tiles, const int* __restrict__ entries,
                    bf16_t* __restrict__ out, int n_head, int n_kv, int P, float scale, int window, float softcap = 0.f,
                    const float* __restrict__ sink = nullptr) {
  const int entry = tiles[2 * blockIdx.x], first = tiles[2 * blockIdx.x + 1];
  const int row0 = entries[4 * entry], n_tok = entries[4 * entry + 1], start = entries[4 * entry + 2];
  const int head = blockIdx.y;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r16 = lane & 15, quad = lane >> 4;
  const int w_first = first + wave * 16;            // first row of this wavefront's tile
  const int row_end = row0 + n_tok;
  if (w_first >= row_end) return;
  const int w_rows = min(16, row_end - w_first);
  const int my_row = w_first + r16;
  const bool col_ok = r16 < w_rows;
  const int my_pos = start + (my_row - row0);       // position of this lane's column
  const int kv_last = start + n_tok - 1;
  const int pos_first = start + (w_first - row0), pos_last = pos_first + w_rows - 1;
  const int my_lo = (window > 0 && my_pos - window + 1 > 0) ? my_pos - window + 1 : 0;
  const int tile_lo = (window > 0 && pos_first - window + 1 > 0) ? pos_first - window + 1 : 0;

  PagedKV kv{pool, table + (size_t)entry * table_stride, P, n_kv, head / (n_head / n_kv)};
  Frag8 qf[HD / 32];
#pragma unroll
  for (int s = 0; s < HD / 32; ++s) {
    qf[s].u = make_uint4(0, 0, 0, 0);
    if (col_ok) qf[s].u = *reinterpret_cast<const uint4*>(q + ((size_t)my_row * n_head + head) * HD + s * 32 + quad * 8);
  }
  float mx = -INFINITY, l = 0.f;
  floatx4 o[HD / 16];
#pragma unroll
  for (int d = 0; d < HD / 16; ++d) o[d] = floatx4{0.f, 0.f, 0.f, 0.f};

  const int blk_lo = tile_lo / 16, blk_hi = pos_last / 16;
  // a block is free of checks if every column sees all of it: it ends at or before the
  // tile's first position and (with a window) starts inside the last column's window
  const int hi_col = col_ok ? my_pos : -1;          // columns beyond the portion see nothing
  walk_blocks<HD>(kv, qf, blk_lo, 1, blk_hi - blk_lo + 1, my_lo, hi_col, kv_last, scale * TI_LOG2E,
                  [=](int b) {
                    const int key0 = b * 16;
                    const bool inside = (key0 + 15 <= pos_first) && (w_rows == 16) &&
                                        (window <= 0 || key0 >= pos_last - window + 1) && (key0 >= tile_lo);
                    return !inside;
                  },
                  mx, l, o, NoHook{}, NoHook{}, softcap * TI_LOG2E);
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!col_ok) return;
  const float inv = sink_join(sink, head, mx, l) / l;
#pragma unroll
  for (int d = 0; d < HD / 16; ++d) {
    Frag4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.h[i] = f2bf(o[d][i] * inv);
    *reinterpret_cast<uint2*>(out + ((size_t)my_row * n_head + head) * HD + d * 16 + quad * 4) = r.u;
  }
}

// ======================================================= prefill, through LDS
// The prefill kernel for head sizes 64 and 128.  A workgroup takes 128 consecutive
// tokens of one q head; a wavefront's tokens are column blocks of 32 of
// v_mfma_f32_32x32x16_bf16 (one block each for four wavefronts, or two each for two).  Keys and values come in turns of 32 keys by direct
// global-to-LDS loads, several turns deep, and are shared by the wavefronts.
//
//   S^T (32 keys x 32 tokens) = K (32 x hd) . Q^T          8 (hd=128) MFMAs per column block
//   O^T (hd x 32 tokens)     += V^T (hd x 32 keys) . P^T   hd/32 x 2 MFMAs per column block
//
// LDS rows of K are not in key order: row r of a 16-row group holds the key whose
// bits 2 and 3 are those of r swapped.  The score tile then leaves a lane with eight
// keys that are contiguous in memory (8h .. 8h+7 of each 16), so that the matching
// V^T fragment is one 16-byte read.  Pieces are XOR-swizzled against bank conflicts.
#define PF_ROWS 128
#define PF_KEYS 32
#define PF_STAGES 4      // LDS stages: PF_STAGES - 1 turns are in flight while one is computed

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float floatx16;

__device__ __forceinline__ void lgkm_wait(int n) {
  switch (n) {
#define TI_LGKM(N) case N: asm volatile("s_waitcnt lgkmcnt(" #N ")" ::: "memory"); break;
    TI_LGKM(1) TI_LGKM(2) TI_LGKM(3) TI_LGKM(4) TI_LGKM(5) TI_LGKM(6) TI_LGKM(7) TI_LGKM(8)
    TI_LGKM(9) TI_LGKM(10) TI_LGKM(11) TI_LGKM(12) TI_LGKM(13) TI_LGKM(14) TI_LGKM(15)
#undef TI_LGKM
    default: asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); break;
  }
}
// wait until at most k * LOADS vector-memory operations are outstanding
// (s_waitcnt with only vmcnt set: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14)
template <int LOADS, int STAGES>
__device__ __forceinline__ void vm_wait_turns(int k) {
#define TI_VM(N) __builtin_amdgcn_s_waitcnt(0x0F70 | ((N) & 15) | ((((N) >> 4) & 3) << 14))
  static_assert(LOADS * (STAGES - 2) <= 63, "vmcnt has six bits");
  switch (k) {
    case 0: TI_VM(0); break;
    case 1: TI_VM(LOADS); break;
    case 2: TI_VM(2 * LOADS); break;
    case 3: TI_VM(3 * LOADS); break;
    case 4: TI_VM(4 * LOADS); break;
    case 5: TI_VM(5 * LOADS); break;
    case 6: TI_VM(6 * LOADS); break;
    default: TI_VM(0); break;
  }
#undef TI_VM
}

// LDS of a workgroup: every stage of keys of all groups, behind them every stage of values (so that the stage is a constant in a read), and the
// queries where many groups take the same ones.  The groups' partial results take the stages' place.
template <int HD, int NG, int NW, int ST>
struct PrefillLds {
  static constexpr int TURN = PF_KEYS * HD * 2;                            // a stage: a turn's keys, or its values
  static constexpr int VALUES = ST * NG * TURN, QUERIES = 2 * VALUES;
  static constexpr int BYTES = QUERIES + (NG >= 4 ? NW * 32 * HD * 2 : 0);
};

// NG groups of NW wavefronts in the workgroup.  A tile is 32 NW rows: a column block of 32
// tokens per wavefront of a group, and every group takes all of the tile's rows.  With more
// than one group the turns (32 keys) go to the groups in rotation (each group loads and walks
// its own turns through its own ST LDS stages) and their partial results are merged through
// LDS at the end.  More groups put two wavefronts on every SIMD when a launch has only one
// workgroup per compute unit, so that one's loads, LDS reads and vector work hide behind the
// other's matrix products.
// CB: column blocks of 32 tokens per wavefront.  (Two, for groups of one wavefront that need no barrier
// and read every K fragment once for 64 tokens, do not fit the registers: the accumulators and the
// queries alone are 192, and the compiler moves them through the other register file all the time.)
// PAIRED: a workgroup takes two tiles, one after the other: tiles[blockIdx.x] and
// tiles[n_tiles - 1 - blockIdx.x] of a list ordered from the most keys to the fewest, so that
// under a causal mask every workgroup of a launch has about the same work.
// Workgroup (bx, by) of a grid of gx x n_head.
//   n_splits > 1: the keys a tile sees are cut into n_splits runs of whole turns, the workgroup takes
//   run `split` and leaves its maxima, sums and unscaled outputs in part_ml [row][head][split] = (m, l) and
//   part_o [row][head][split][HD] for the kernel that merges them
template <int HD, int NG, int NW, int ST, bool PAIRED, int CB, bool TOGETHER>
__device__ __forceinline__ void
prefill_tiles(unsigned char* smem, int bx, int by, int gx, int n_splits, int split, const bf16_t* __restrict__ q,
              const bf16_t* __restrict__ pool, const int* __restrict__ table, int table_stride,
              const int* __restrict__ tiles, int n_tiles, const int* __restrict__ entries, bf16_t* __restrict__ out,
              int n_head, int n_kv, int P, float scale, int window, float* __restrict__ part_o,
              float* __restrict__ part_ml, float softcap, const float* __restrict__ sink) {
  constexpr int WROWS = 32 * CB;                      // tokens per wavefront
  constexpr int TROWS = NW * WROWS;                   // tokens per tile
  constexpr int NP = HD / 8;                          // 16-byte pieces per K row
  typedef PrefillLds<HD, NG, NW, ST> Lds;
  constexpr int NEXT = NG * Lds::TURN;                // from a stage to the next
  constexpr int K_ROWS = 1024 / (HD * 2);             // K rows per wavefront load
  constexpr int K_LOADS = PF_KEYS / K_ROWS;
  constexpr int V_LOADS = HD / 16, V_BLOCK = HD / 32;   // 32 dims (the 32 bytes of a block's 16 keys each) per wavefront load
  static_assert(K_LOADS % NW == 0 && V_LOADS % NW == 0, "every wavefront takes the same kinds of loads");
  constexpr int MY_K = K_LOADS / NW, MY_LOADS = (K_LOADS + V_LOADS) / NW;   // per wavefront and turn
  constexpr int QL = NG >= 4 ? TROWS * HD * 2 / 1024 / (NG * NW) : 0;      // loads of queries a wavefront, 0: as operands from memory
  constexpr int KS = HD / 16;                         // k-steps of the first product
  constexpr int DB = HD / 32;                         // 32-dim blocks of the output

  // Which (tile, head) this workgroup takes: the tiles with the most keys come first in all heads, so that what starts behind the first round
  // of the units is ever smaller and the units end together.  (With a head's tiles behind one another the last heads' largest tiles started
  // last.  us, tiles of 64 rows, heads first and tiles first: 32 heads of 700 tokens 21.9 and 16.9, of 1,500 47.6 and 42.8; 16 of 2,048
  // 37.4 and 35.3.)  Workgroups go to the eight XCDs in turn (linear id mod 8) and each XCD has an L2 of its own: with a multiple of
  // eight kv heads, an XCD is given whole kv heads, so that the keys and values of a head are read into one L2 only.  With others a tile's heads
  // are dealt out one by one and every L2 reads all kv heads, which costs nothing while they fit; TOGETHER: the heads that read a tile's keys
  // stand behind one another on one XCD, and what is no multiple of eight such groups comes last.
  int head;
  {
    const int id = by * gx + bx, group = n_head / n_kv;
    if (n_kv % 8 == 0) {
      const int xcd = id & 7, local = id >> 3, heads = n_head / 8, nth = local % heads;      // heads: an XCD's
      bx = local / heads;
      head = (xcd + 8 * (nth / group)) * group + nth % group;
    } else if (TOGETHER) {
      const int spread = (gx * n_kv) & ~7, rest = id - spread * group, local = rest < 0 ? id >> 3 : rest;
      const int unit = rest < 0 ? (local / group) * 8 + (id & 7) : spread + local / group;
      bx = unit / n_kv;
      head = (unit % n_kv) * group + local % group;
    } else {
      bx = id / n_head;
      head = id % n_head;
    }
  }
  // the wavefront's number in scalar registers: what follows from it (which turns it loads, where they
  // go, which rows are its own) is then worked out once per wavefront, not once per lane
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wid / NW, wave = wid % NW, lane = threadIdx.x & 63;
  const int r32 = lane & 31, h = lane >> 5;
  const int kvh = head / (n_head / n_kv);
  const size_t page_elems = (size_t)2 * n_kv * P * HD;
  const bf16_t* kpool = pool + (size_t)kvh * P * HD;

  // scores are kept in units of log 2: softmax weights are then bare exp2
  const float scale2 = scale * 1.4426950408889634f;

  // what this lane fetches in each of its loads of a turn
  //  K load g: LDS rows K_ROWS g .. + K_ROWS - 1; lane i -> row r = K_ROWS g + i / NP, slot c = i % NP,
  //            holds piece c ^ (r & (NP - 1)) of key 16 (r / 16) + swap23(r % 16)
  //  V load g of a block: dims 32 g .. 32 g + 31; lane i -> dim 32 g + i / 2, keys 8 ((i + i / 32) % 2) .. + 7: in pages of 16 rows 1 KiB of
  //            consecutive bytes, and in LDS what an operand reads is 1 KiB of consecutive bytes too, dims 16 to 31 with their halves exchanged:
  //            of the lanes that LDS serves together, 0 to 3 and 12 to 15 with 20 to 27, no two meet in a bank so (1.8 ns a read of a unit, 3.5 without)
  // K load g starts for lane i (lr = i / NP < K_ROWS, c = i % NP) from its block's first K row at
  //   (k_lane ^ X(g)) + C(g),  k_lane = swap23(lr) * HD * 2 + (c ^ lr) * 16,
  //   X(g) = ((K_ROWS g) & (NP - 1)) * 16,  C(g) = swap23((K_ROWS g) & 15) * HD * 2
  // (the row number K_ROWS g + lr has g's bits and the lane's bits apart, and so have its pieces), of the turn's first block if
  // (K_ROWS g) & 16 is clear, else of the second; V load g at v_lane + 64 g P from the V^T row of the block's first key.  A block has one
  // descriptor, C(g) and 64 g P go into the scalar offset: a load is one scalar addition, the step of m0, and itself.  (As flat
  // addresses, two blocks' values in a load, a turn's loads took 75 instructions, most of them scalar ones behind one another, now 35; us a
  // launch at 16 heads, 8 for keys: 2,048 tokens 33.5 -> 32.6, 6,000 238 -> 229, 77 7.05 -> 6.95.)
  static_assert(K_ROWS <= 16 && (K_ROWS & (K_ROWS - 1)) == 0, "rows of a K load lie in one block of 16");
  auto swap23 = [](int r16) __attribute__((always_inline)) { return ((r16 & 4) << 1) | ((r16 & 8) >> 1) | (r16 & 3); };
  const unsigned k_lane = (unsigned)(swap23(lane / NP) * HD * 2 + (((lane % NP) ^ (lane / NP)) << 4));
  const unsigned v_lane = (unsigned)((lane >> 1) * P * 2 + ((lane ^ (lane >> 5)) & 1) * 16);

  const unsigned lds_k = (unsigned)(size_t)smem + grp * Lds::TURN, lds_v = lds_k + Lds::VALUES;      // this group's first stages
  // the wavefronts of a group wait for each other at the workgroup's barrier (a handshake of a group's
  // two wavefronts through a word of LDS, which lets the groups drift apart, was slower: 4.72 ms against
  // 4.59 ms for a prompt of 2,048 tokens at Qwen3-0.6B's sizes)
  auto group_sync = [&]() __attribute__((always_inline)) {
    if constexpr (NW > 1) __builtin_amdgcn_s_barrier();
  };
  // LDS addresses of this lane's fragments; the stage, and the dims and the block of a V^T fragment, are
  // constants in the read instructions
  unsigned k_addr[KS];
  const unsigned v_addr = lds_v + r32 * 32 + ((h ^ (r32 >> 4)) & 1) * 16;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_addr[ks] = lds_k + r32 * (HD * 2) + (((ks * 2 + h) ^ (r32 & (NP - 1))) << 4);

  for (int slot = 0; slot < (PAIRED ? 2 : 1); ++slot) {
  // ---- this slot's tile
  const int tile = (slot == 0) ? bx : n_tiles - 1 - bx;
  if (PAIRED && slot == 1 && tile <= bx) break;                     // an odd count: the middle tile came first
  const int entry = tiles[2 * tile], first = tiles[2 * tile + 1];
  const int row0 = entries[4 * entry], n_tok = entries[4 * entry + 1], start = entries[4 * entry + 2];
  const int row_end = row0 + n_tok;
  const int kv_last = start + n_tok - 1;
  const int* tab = table + (size_t)entry * table_stride;

  // this wavefront: rows w_first .. w_first + WROWS - 1, in column blocks of 32
  const int w_first = first + wave * WROWS;
  const int w_rows = max(0, min(WROWS, row_end - w_first));
  const int w_pos_first = start + (w_first - row0), w_pos_last = w_pos_first + w_rows - 1;
  const int w_lo = (window > 0 && w_pos_first - window + 1 > 0) ? w_pos_first - window + 1 : 0;
  // the workgroup: rows first .. first + TROWS - 1
  const int g_rows = min(TROWS, row_end - first);
  const int g_pos_first = start + (first - row0), g_pos_last = g_pos_first + g_rows - 1;
  const int g_lo = (window > 0 && g_pos_first - window + 1 > 0) ? g_pos_first - window + 1 : 0;

  int blk_lo = (g_lo / PF_KEYS) * 2, blk_hi = g_pos_last / 16;         // 16-key blocks, starting on a turn
  const int v_limit = min(kv_last, blk_hi * 16 + 15);               // last key whose value row is real
  if (n_splits > 1) {
    const int per = (((blk_hi + 1 - blk_lo) + n_splits - 1) / n_splits + 1) & ~1;   // whole turns
    blk_lo += split * per;
    blk_hi = min(blk_hi, blk_lo + per - 1);                         // a run past the end is empty
  }

  // A run is 64 blocks.  Lane i keeps where block i of a run starts in the pool (the bytes of its page's first K row of this kv head) and the
  // row of its first key in that page, for the run that loads are asked from and the next, so that the walk divides by the page size once a
  // run and waits for the block table once a tile.  Blocks past the end stand on page 0, and so do blocks whose page was given back
  // (all their keys are masked).
  unsigned run_lo[2] = {0, 0}, run_hi[2] = {0, 0};
  int run_row[2] = {0, 0}, asked = 0;
  const int n_blk = blk_hi + 1 - blk_lo;
  auto ask_run = [&](int r) __attribute__((always_inline)) {
    const int b = 64 * r + lane;
    asked = b < n_blk ? tab[(blk_lo + b) * 16 / P] : 0;
  };
  auto place_run = [&](int r) __attribute__((always_inline)) {
    const unsigned long at = (unsigned long)kpool + (unsigned long)max(asked, 0) * (page_elems * 2);
    const int row = (blk_lo + 64 * r + lane) * 16 % P;
    if (r & 1) run_lo[1] = (unsigned)at, run_hi[1] = (unsigned)(at >> 32), run_row[1] = row;
    else run_lo[0] = (unsigned)at, run_hi[0] = (unsigned)(at >> 32), run_row[0] = row;
  };
  // The loads of this group's turn i: where its two blocks lie, then one load after another (n < MY_K: keys).  What is the same in every lane
  // is worked out in scalar registers.
  unsigned at_lo[2], at_hi[2];
  int at_row[2];
  auto find_turn = [&](int i) __attribute__((always_inline)) {
    const int t = i * NG + grp, j = (2 * t) & 63;
    if ((t >> 5) & 1) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        at_lo[x] = __builtin_amdgcn_readlane(run_lo[1], j + x);
        at_hi[x] = __builtin_amdgcn_readlane(run_hi[1], j + x);
        at_row[x] = __builtin_amdgcn_readlane(run_row[1], j + x);
      }
    } else {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        at_lo[x] = __builtin_amdgcn_readlane(run_lo[0], j + x);
        at_hi[x] = __builtin_amdgcn_readlane(run_hi[0], j + x);
        at_row[x] = __builtin_amdgcn_readlane(run_row[0], j + x);
      }
    }
  };
  const unsigned v_from = (unsigned)(n_kv * P * HD * 2);             // a page's values behind its keys
  auto load_one = [&](unsigned stage_off, int n) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)      // (the host's pass has no buffer descriptors)
    const bool keys = n < MY_K;
    const int g = wave + NW * (keys ? n : n - MY_K);                 // the same in every lane
    const int rows = K_ROWS * g;
    // which of the turn's blocks: known where it is compiled unless a wavefront's loads of a kind are fewer than the blocks
    const int x = keys ? (K_ROWS * NW <= 16 ? (K_ROWS * NW * n) >> 4 : rows >> 4) : (NW <= V_BLOCK ? NW * (n - MY_K) / V_BLOCK : g / V_BLOCK);
    const unsigned lo = x ? at_lo[1] : at_lo[0], hi = x ? at_hi[1] : at_hi[0];
    const int row = x ? at_row[1] : at_row[0];
    const auto block = __builtin_amdgcn_make_buffer_rsrc((void*)(((unsigned long)hi << 32) | lo), 0, 0x7fffffff, 0x00020000);
    if (keys)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(block, (__attribute__((address_space(3))) void*)(size_t)(lds_k + stage_off + g * 1024), 16,
                                               k_lane ^ (unsigned)((rows & (NP - 1)) << 4), (row + swap23(rows & 15)) * (HD * 2), 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(block, (__attribute__((address_space(3))) void*)(size_t)(lds_v + stage_off + g * 1024), 16,
                                               v_lane, v_from + row * 2 + (g % V_BLOCK) * 64 * P, 0, 0);
#endif
  };
  auto issue = [&](int i, unsigned stage_off) __attribute__((always_inline)) {
    find_turn(i);
#pragma unroll
    for (int n = 0; n < MY_LOADS; ++n) load_one(stage_off, n);
  };
  // this group's turns are turns grp, grp + NG, ...; i counts them, and turn i goes through stage i % ST
  const int n_turns = max(0, (n_blk + 1) / 2), n_iter = (n_turns + NG - 1) / NG;      // n_iter: the first group's, the most
  const int my_turns = max(0, (n_turns - grp + NG - 1) / NG);
  constexpr int AHEAD = ST - 1;
  // The queries of a workgroup of many groups, which all take the same rows, come through LDS as well: QL loads a wavefront of whole rows (piece c
  // of row r in place c ^ (r & (NP - 1))).  As operands from memory, a row in every lane, they were 64 loads a tile of 64 cycles each of the unit that
  // takes addresses, in front of a tile's first scores.  (us a launch at 16 heads, 8 for keys, before and now: 2,048 tokens 40.0 -> 38.3, 77 8.2
  // -> 7.5, 504 behind 500 20.6 -> 19.8; 2,048 at 32 heads 74.4 -> 72.2.)
  if constexpr (QL > 0) {
    const char* rows = reinterpret_cast<const char*>(q + (size_t)head * HD);
#pragma unroll
    for (int j = 0; j < QL; ++j) {
      const int g = wid + NG * NW * j, r = g * K_ROWS + lane / NP;
      const char* src = rows + (size_t)min(first + r, row_end - 1) * ((size_t)n_head * HD * 2) + (((lane % NP) ^ (r & (NP - 1))) << 4);
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(size_t)((unsigned)(size_t)smem + Lds::QUERIES + g * 1024), 16, 0, 0);
    }
  }
  // the first run's blocks and first turns are asked for before the queries are waited for: those arrive meanwhile
  // (a workgroup whose run of keys is empty walks nothing, and nothing may be on its way into LDS
  // when it goes on to the merge)
  const int under_way = min(AHEAD, my_turns);
  if (n_turns) {
    ask_run(0);
    place_run(0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i)
      if (i < my_turns) issue(i, i * NEXT);
    if (n_blk > 64) ask_run(1);
  }

  v4u qf[CB][KS];
  int my_pos[CB];
  bool col_ok[CB];
  if constexpr (QL > 0) {
    vm_wait_turns<MY_LOADS, ST + 1>(under_way);
    __builtin_amdgcn_s_barrier();
    static_assert(CB == 1, "a column block a wavefront");
    const int r = wave * 32 + r32;
    const unsigned at = (unsigned)(size_t)smem + Lds::QUERIES + r * (HD * 2);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      asm volatile("ds_read_b128 %0, %1" : "=v"(qf[0][ks]) : "v"(at + (((ks * 2 + h) ^ (r & (NP - 1))) << 4)));
    lgkm_wait(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[0][ks]));
  }
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int row = w_first + cb * 32 + r32;
    col_ok[cb] = row < row_end;
    my_pos[cb] = start + (row - row0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if constexpr (QL > 0) {
        if (!col_ok[cb]) qf[cb][ks] = v4u{0, 0, 0, 0};
        continue;
      }
      qf[cb][ks] = v4u{0, 0, 0, 0};
      if (col_ok[cb]) {
        const uint4 t = *reinterpret_cast<const uint4*>(q + ((size_t)row * n_head + head) * HD + ks * 16 + h * 8);
        qf[cb][ks] = v4u{t.x, t.y, t.z, t.w};
      }
    }
  }
  float mx[CB], l[CB];
  floatx16 o[CB][DB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    mx[cb] = -INFINITY;
    l[cb] = 0.f;
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[cb][d][i] = 0.f;
  }

  // One turn of 32 keys from a stage for this wavefront's columns, in two steps: the scores, then the
  // softmax and the second product.  plain (the same in every lane): every key of the turn is visible
  // to every column and written: no compare at all.
  auto turn_scores = [&](auto stage_tag, floatx16* sc, auto between) __attribute__((always_inline)) {
    constexpr unsigned SOFF = decltype(stage_tag)::value * NEXT;
    // ---- the fragments: keys now, values right behind them
    v4u kf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[ks]) : "v"(k_addr[ks]), "n"(SOFF));
    // ---- S^T = K . Q^T
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[cb][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (cb == 0) {
          lgkm_wait(KS - 1 - ks);        // the first ks + 1 of the KS reads have arrived
          asm volatile("" : "+v"(kf[ks]));
        }
        sc[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[ks]),
                                                         __builtin_bit_cast(bf16x8, qf[cb][ks]), sc[cb], 0, 0, 0);
        if (cb == 0) between(ks);
      }
    }
  };
  auto turn_rest = [&](auto stage_tag, int key0, bool plain, const floatx16* sc) __attribute__((always_inline)) {
    constexpr unsigned SOFF = decltype(stage_tag)::value * NEXT;
    // the value fragments are asked for now and waited for after the softmax
    v4u vf[DB][2];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(vf[d][tt]) : "v"(v_addr), "n"(SOFF + tt * (HD * 32) + d * 1024));

    // ---- masks, the online softmax and O^T += V^T . P^T, column block by column block: the matrix
    // core works on one block's second product while the next block's softmax runs.  The scores stay
    // as the first product left them: the maximum is taken over them and scaled once (the scale is
    // positive), and the scale goes into the multiply-add of the exponent.
    // element i of a lane: key key0 + 16 (i / 8) + 8 h + 4 ((i / 4) % 2) + i % 4
    // (the keys' numbers are worked out behind the branches that need them, not before the loop and kept
    // in registers: the compiler takes `hm` for something the branch has made)
    int hm = h;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      float sv[16], cv[16];
      // a soft cap (the same in every lane) before the masks: cap tanh(s scale / cap), left in the units of the bare product
#pragma unroll
      for (int i = 0; i < 16; ++i) cv[i] = sc[cb][i];
      if (softcap > 0.f) {
        const float r = scale / softcap, back = softcap / scale;
#pragma unroll
        for (int i = 0; i < 16; ++i) cv[i] = tanh_fast(cv[i] * r) * back;
      }
      if (plain) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sv[i] = cv[i];
      } else {
        asm volatile("" : "+v"(hm));
        const int hi = col_ok[cb] ? my_pos[cb] : -1;
        const int lo = (window > 0) ? my_pos[cb] - window + 1 : 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = key0 + 16 * (i >> 3) + 8 * hm + 4 * ((i >> 2) & 1) + (i & 3);
          const bool see = (key <= hi) & (key >= lo);      // bitwise on purpose: selects, no branches
          sv[i] = see ? cv[i] : -INFINITY;
        }
      }
      float bm = sv[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) bm = fmaxf(bm, sv[i]);
      {
        const LanePair p = lane_pair<32>(bm);
        bm = fmaxf(p.a, p.b);
      }
      const float m_new = fmaxf(mx[cb], bm * scale2);
      const float m_safe = (m_new == -INFINITY) ? 0.f : m_new;
      float ps = 0.f;
      float pv[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        pv[i] = __builtin_amdgcn_exp2f(fmaf(sv[i], scale2, -m_safe));
        ps += pv[i];
      }
      v4u pf[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        pf[tt] = v4u{pack_bf16x2(pv[8 * tt], pv[8 * tt + 1]), pack_bf16x2(pv[8 * tt + 2], pv[8 * tt + 3]),
                     pack_bf16x2(pv[8 * tt + 4], pv[8 * tt + 5]), pack_bf16x2(pv[8 * tt + 6], pv[8 * tt + 7])};
      // the running maximum settles after a few turns; then nothing needs rescaling
      if (__builtin_amdgcn_ballot_w64(m_new != mx[cb]) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(mx[cb] - m_safe);
        l[cb] *= alpha;
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[cb][d][i] *= alpha;
        mx[cb] = m_new;
      }
      l[cb] += ps;

      if (cb == 0) {
        // the value fragments have had the first block's softmax to arrive
        lgkm_wait(0);
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) asm volatile("" : "+v"(vf[d][tt]));
        if (!plain) {
          if (key0 + PF_KEYS - 1 > v_limit || key0 < g_lo) {
            // rows never written, and the stand-in page read for a block that was given back or
            // lies past the end, may hold anything, NaN included, and 0 * NaN is NaN
            asm volatile("" : "+v"(hm));
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
              for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                  const int key = key0 + 16 * tt + 8 * hm + e;
                  const bool drop = (key > v_limit) | (key < g_lo);
                  const unsigned keep = drop ? ((e & 1) ? 0x0000FFFFu : 0xFFFF0000u) : 0xFFFFFFFFu;
                  vf[d][tt][e >> 1] &= keep;
                }
          }
        }
      }
#pragma unroll
      for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          o[cb][d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[d][tt]),
                                                             __builtin_bit_cast(bf16x8, pf[tt]), o[cb][d], 0, 0, 0);
    }
  };

  // Run 1 has been asked for, with the first turns on their way; the others are asked for as the loads enter the run before, and placed a turn
  // later.
  int placed = 0, entered = 0;      // the last run placed, and the last that loads have been asked from
  for (int i0 = 0; i0 < n_iter; i0 += ST) {
    // ST turns, each with its stage as a constant
    unrolled_while<ST>([&](auto si_tag) __attribute__((always_inline)) {
      constexpr int si = decltype(si_tag)::value;
      const int i = i0 + si;
      if (i >= n_iter) return false;
      // this wavefront's part of the group's turn i has landed: only its turns issued after it (at
      // most AHEAD - 1) may be outstanding.  Then the group's wavefronts wait for each other: the
      // whole turn has landed, and everyone is done with the turn before, whose stage turn
      // i + AHEAD goes into.
      vm_wait_turns<MY_LOADS, ST>(max(0, min(AHEAD - 1, my_turns - 1 - i)));
      group_sync();
      const int key0 = (blk_lo + 2 * (i * NG + grp)) * 16;
      // nothing of this turn is visible to this wavefront: it only helps loading
      const bool idle = i >= my_turns || w_rows == 0 || key0 > w_pos_last || key0 + PF_KEYS - 1 < w_lo;
      const bool more = i + AHEAD < my_turns;
      if (more) {
        if (placed == entered && 64 * (entered + 1) < n_blk) place_run(++placed);
        const int r = ((i + AHEAD) * NG + grp) >> 5;
        find_turn(i + AHEAD);
        if (idle) {
#pragma unroll
          for (int n = 0; n < MY_LOADS; ++n) load_one(((si + AHEAD) % ST) * NEXT, n);
        }
        if (r != entered) {
          entered = r;
          if (64 * (r + 1) < n_blk) ask_run(r + 1);
        }
      }
      if (idle) return true;
      // Turn i + AHEAD goes into the stage that turn i - 1 has left, a load behind each of the first product's matrix instructions: asked for
      // at once the wavefronts' loads queue at the unit that takes addresses, and nothing is on the matrix cores meanwhile (2,048 tokens
      // 32.7 us, so 32.0; 6,000 228, 224).
      constexpr unsigned to = ((si + AHEAD) % ST) * NEXT;
      floatx16 sc[CB];
      if (more)
        turn_scores(si_tag, sc, [&](int ks) __attribute__((always_inline)) {
#pragma unroll
          for (int n = 0; n < MY_LOADS; ++n)
            if (n * KS / MY_LOADS == ks) load_one(to, n);
          __builtin_amdgcn_sched_barrier(0);
        });
      else
        turn_scores(si_tag, sc, [](int) {});
      const bool plain = (key0 + PF_KEYS - 1 <= w_pos_first) && (w_rows == WROWS) &&
                         (window <= 0 || key0 >= w_pos_last - window + 1);
      turn_rest(si_tag, key0, plain, sc);
      return true;
    });
  }
  // every wavefront of the group is done with the stages before the merge (or the next tile) writes into them
  group_sync();

  // ---- the result: o[cb][d][i] is dim 32 d + 8 (i / 4) + 4 h + i % 4 of token (column) r32 of block cb.
  // `first_val`, `count_tag`: which of a lane's DB * 16 values of a block (value v = 16 d + i) these are; a
  // lane's values come in fours of consecutive dims.
  auto write_out = [&](int cb, const float* val, int first_val, auto count_tag, float m_all, float lt) __attribute__((always_inline)) {
    constexpr int n_val = decltype(count_tag)::value;
    if (!col_ok[cb]) return;
    const int row = w_first + cb * 32 + r32;
    if (n_splits > 1) {
      const size_t at = ((size_t)row * n_head + head) * n_splits + split;
      float* po = part_o + at * HD;
#pragma unroll
      for (int j = 0; j < n_val; j += 4) {
        const int v = first_val + j;
        *reinterpret_cast<float4*>(po + 32 * (v >> 4) + 8 * ((v & 15) >> 2) + 4 * h) =
            make_float4(val[j], val[j + 1], val[j + 2], val[j + 3]);
      }
      if (h == 0 && first_val == 0) reinterpret_cast<float2*>(part_ml)[at] = make_float2(m_all, lt);
      return;
    }
    const float inv = sink_join(sink, head, m_all, lt) / lt;
    bf16_t* dst = out + ((size_t)row * n_head + head) * HD;
#pragma unroll
    for (int j = 0; j < n_val; j += 4) {
      const int v = first_val + j;
      *reinterpret_cast<uint2*>(dst + 32 * (v >> 4) + 8 * ((v & 15) >> 2) + 4 * h) =
          make_uint2(pack_bf16x2(val[j] * inv, val[j + 1] * inv), pack_bf16x2(val[j + 2] * inv, val[j + 3] * inv));
    }
  };
  if constexpr (NG == 1) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      float val[DB * 16];
#pragma unroll
      for (int v = 0; v < DB * 16; ++v) val[v] = o[cb][v >> 4][v & 15];
      write_out(cb, val, 0, std::integral_constant<int, DB * 16>{}, mx[cb], l[cb] + __shfl_xor(l[cb], 32, 64));
    }
  } else {
    // The groups merge their partial results through LDS (the stages are free now), each group the
    // values it owns: values VPG g .. VPG (g + 1) - 1 of every lane are group g's.  A group leaves the
    // values it does not own (in their order, four to a slot of 16 bytes a lane), its maximum and its sum in its part of LDS; after a
    // barrier it reads the others' contributions to its own values, adds them to its own (scaled first) in the order of the groups, each by
    // one multiply-add (written out: left to the compiler, which product of a sum is rounded first changes with the code around it), and
    // writes them out.  The code stands once for each group, so that which registers these are is known where it is compiled (as a
    // choice between registers by the group's number, value by value, a tile's end took 4,400 cycles; 2,048 tokens 38.0 us, now 36.4, 77 7.5,
    // now 7.05, 2,048 at 32 heads 73.2, now 70.0).
    constexpr int VALS = DB * 16, VPG = VALS / NG, FOURS = (VALS - VPG) / 4, PART = (FOURS * 16 + 8) * 64;
    static_assert(VALS % NG == 0 && VPG % 4 == 0, "a group owns whole fours of values");
    static_assert(NG * NW * PART <= Lds::QUERIES, "the partial results fit into the stages");
    typedef __attribute__((address_space(3))) floatx4 lds_four;
    typedef __attribute__((address_space(3))) ti_float2v lds_two;
    // slot i (values 4 i .. of those left) of group g's wavefront, and behind the slots its maximum and sum
    const unsigned part0 = (unsigned)(size_t)smem + wave * PART;
    auto four_of = [&](int g, int i) __attribute__((always_inline)) { return (lds_four*)(size_t)(part0 + g * (NW * PART) + i * 1024 + lane * 16); };
    auto ml_of = [&](int g) __attribute__((always_inline)) { return (lds_two*)(size_t)(part0 + g * (NW * PART) + FOURS * 1024 + lane * 8); };
    // only the workgroup's barrier tells that every group is done with its stages
    if constexpr (NW == 1) __syncthreads();
    auto merge = [&](auto tag, int cb) __attribute__((always_inline)) {
      constexpr int G = decltype(tag)::value, FIRST = G * VPG;      // this group, and its first value
#pragma unroll
      for (int i = 0; i < FOURS; ++i) {
        constexpr auto at = [](int sl) { return sl < FIRST ? sl : sl + VPG; };
        const int v = at(4 * i);
        *four_of(G, i) = floatx4{o[cb][v >> 4][v & 15], o[cb][v >> 4][(v & 15) + 1], o[cb][v >> 4][(v & 15) + 2], o[cb][v >> 4][(v & 15) + 3]};
      }
      *ml_of(G) = ti_float2v{mx[cb], l[cb]};
      __syncthreads();
      ti_float2v ml[NG];
#pragma unroll
      for (int g = 0; g < NG; ++g) ml[g] = *ml_of(g);
      floatx4 theirs[NG][VPG / 4];
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int j = 0; j < VPG / 4; ++j)
          if (g != G) theirs[g][j] = *four_of(g, (FIRST + (G > g ? -VPG : 0)) / 4 + j);
      float m_all = ml[0].x;
#pragma unroll
      for (int g = 1; g < NG; ++g) m_all = fmaxf(m_all, ml[g].x);
      const float m_safe = (m_all == -INFINITY) ? 0.f : m_all;
      float a_g[NG], l_all = 0.f;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        a_g[g] = __builtin_amdgcn_exp2f(ml[g].x - m_safe);
        l_all = fmaf(ml[g].y, a_g[g], l_all);
      }
      const float a_own = __builtin_amdgcn_exp2f(mx[cb] - m_safe);
      float val[VPG];
#pragma unroll
      for (int j = 0; j < VPG; ++j) val[j] = o[cb][(FIRST + j) >> 4][(FIRST + j) & 15] * a_own;
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int j = 0; j < VPG; ++j)
          if (g != G) val[j] = fmaf(theirs[g][j / 4][j % 4], a_g[g], val[j]);
      write_out(cb, val, FIRST, std::integral_constant<int, VPG>{}, m_all, l_all + __shfl_xor(l_all, 32, 64));
    };
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      if (cb > 0) __syncthreads();                   // the block before has been read
      unrolled_while<NG>([&](auto tag) __attribute__((always_inline)) {      // (the same in every lane)
        if (grp == decltype(tag)::value) merge(tag, cb);
        return true;
      });
    }
  }
  // the next tile's loads go into the LDS that the merge has just read
  if (PAIRED && NG > 1) __syncthreads();
  }   // slot
}

template <int HD, int NG, int NW = 4, int ST = PF_STAGES, bool PAIRED = false, int CB = 1, bool TOGETHER = false>
__global__ void __launch_bounds__(64 * NW * NG)
attn_prefill_lds_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ pool,
                        const int* __restrict__ table, int table_stride, const int* __restrict__ tiles,
                        int n_tiles, const int* __restrict__ entries, bf16_t* __restrict__ out, int n_head,
                        int n_kv, int P, float scale, int window, float* __restrict__ part_o = nullptr,
                        float* __restrict__ part_ml = nullptr, float softcap = 0.f, const float* __restrict__ sink = nullptr) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  prefill_tiles<HD, NG, NW, ST, PAIRED, CB, TOGETHER>(smem, blockIdx.x, blockIdx.y, gridDim.x, gridDim.z, blockIdx.z, q, pool, table,
                                            table_stride, tiles, n_tiles, entries, out, n_head, n_kv, P, scale, window, part_o,
                                            part_ml, softcap, sink);
}

// ============================================== portions and single tokens in one launch
// A step that holds portions beside decoded tokens: the first n_tiles * n_head workgroups take a tile of 64 rows
// each (the unpaired kernel above), the others a run of a single token's context (by records), walked by eight
// wavefronts.  The tiles are bound by their softmax and leave memory idle, the single tokens by what a compute unit
// reads: side by side they take about as long as the longer of the two.
template <int HD>
__global__ void __launch_bounds__(512)
attn_step_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ pool, const int* __restrict__ table, int table_stride,
                 const int* __restrict__ tiles, int n_tiles, const int* __restrict__ entries, const int* __restrict__ runs,
                 int run_stride, int group, bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml,
                 int n_head, int n_kv, int P, float scale, int window, float softcap, const float* __restrict__ sink) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int n_pre = n_tiles * n_head, id = blockIdx.x;
  if (id < n_pre) {
    prefill_tiles<HD, 4, 2, 2, false, 1, false>(smem, id % n_tiles, id / n_tiles, n_tiles, 1, 0, q, pool, table, table_stride, tiles,
                                         n_tiles, entries, out, n_head, n_kv, P, scale, window, nullptr, nullptr, softcap, sink);
  } else {
    const int at = id - n_pre, ways = n_kv * ((group + 15) / 16);
    decode_run<HD, false, 8, 1>(*reinterpret_cast<StagedMerge<HD, 8, 1>*>(smem), at / ways, at % ways, 0, q, pool, table,
                                          table_stride, nullptr, nullptr, nullptr, out, part_o, part_ml, n_head, n_kv, P, scale,
                                          window, 1, QKPrep{}, softcap, sink, DecodeRuns{runs, run_stride}, group);
  }
}

// ------------------------------------------------------------------ dispatch
static int check_common(const char* what, int n_head, int n_kv, int hd, int P, int table_stride) {
  if (!(hd == 32 || hd == 64 || hd == 128)) {
    ti_set_error("%s: head_dim %d is not served by the matrix-core kernels (32, 64, 128)", what, hd);
    return 3;
  }
  if (P % 16 != 0) {
    ti_set_error("%s: page size %d is not a multiple of 16", what, P);
    return 3;
  }
  if (n_head <= 0 || n_kv <= 0 || n_head % n_kv != 0 || table_stride <= 0) {
    ti_set_error("%s: heads %d / kv_heads %d / table_stride %d", what, n_head, n_kv, table_stride);
    return 1;
  }
  return 0;
}

// compute units of the current device (asked once)
static int compute_units() {
  static int n = 0;
  if (n == 0) {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      n = v;
    else
      n = 256;
  }
  return n;
}

// Decode rows.  rows: which rows of the step (nullptr: rows 0..n_rows-1).  n_splits > 1 needs
// part_o (float [n_rows, n_head, n_splits, hd]) and part_ml (float [n_rows, n_head, n_splits, 2]).
// Returns 3 for sizes these kernels do not serve.
// The soft cap of the call under way: the entry points whose names end in `_capped_bf16` set it around a call of
// the plain ones, which hand it to their kernels (0: none).
static thread_local float g_softcap = 0.f;
// The sinks of the call under way (float [n_head] in device memory, or null): `ti_attention_bf16_sink` sets them for the calling
// thread's next calls, which hand them to the kernels that finish a column.
static thread_local const float* g_sink = nullptr;
extern "C" void ti_attention_bf16_sink(const float* sink) { g_sink = sink; }

template <bool PREP>
static int launch_decode(const void* q, const void* pool, const int* table, int table_stride, const int* pos,
                         const int* slot, const int* rows, void* out, float* part_o, float* part_ml, int n_rows,
                         int n_head, int n_kv, int hd, int page_size, float scale, int window, int n_splits,
                         QKPrep prep, hipStream_t stream) {
  TI_REQUIRE(n_splits >= 1 && n_splits <= MERGE_MAX_SPLITS, "attention_decode: bad split count %d (1..%d)", n_splits, MERGE_MAX_SPLITS);
  TI_REQUIRE(n_splits == 1 || (part_o && part_ml), "attention_decode: splits need partial buffers");
  TI_REQUIRE(slot || table_stride <= DEC_TABLE_LDS, "attention_decode: without slots a table row has at most %d entries, not %d",
             DEC_TABLE_LDS, table_stride);
  if (n_rows == 0) return 0;
  const int parts = (n_head / n_kv + 15) / 16;
  TI_REQUIRE(n_kv * parts <= 65535, "attention_decode: too many heads");
  dim3 grid(n_rows, n_kv * parts, n_splits);
#define TI_DEC(H)                                                                                          \
  case H:                                                                                                  \
    attn_decode_kernel<H, PREP><<<grid, 256, 0, stream>>>((const bf16_t*)q, (const bf16_t*)pool, table,     \
                                                          table_stride, pos, slot, rows, (bf16_t*)out,      \
                                                          part_o, part_ml, n_head, n_kv, page_size,         \
                                                          scale, window, n_splits, prep, g_softcap, g_sink);  \
    if (n_splits > 1)                                                                                       \
      attn_merge_kernel<H><<<dim3(n_rows, n_head), (H < 64 ? 64 : H), 0, stream>>>(part_o, part_ml, rows,   \
                                                                                  (bf16_t*)out, n_head,    \
                                                                                  n_splits, g_sink);       \
    break;
  switch (hd) {
    TI_DEC(64) TI_DEC(128)
    case 32:
      if constexpr (!PREP) {
        attn_decode_kernel<32, false><<<grid, 256, 0, stream>>>((const bf16_t*)q, (const bf16_t*)pool, table,
                                                                table_stride, pos, slot, rows, (bf16_t*)out,
                                                                part_o, part_ml, n_head, n_kv, page_size, scale,
                                                                window, n_splits, prep, g_softcap, g_sink);
        if (n_splits > 1)
          attn_merge_kernel<32><<<dim3(n_rows, n_head), 64, 0, stream>>>(part_o, part_ml, rows, (bf16_t*)out,
                                                                         n_head, n_splits, g_sink);
      }
      break;
  }
#undef TI_DEC
  TI_LAUNCH_CHECK();
  return 0;
}

extern "C" int ti_attention_decode_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                        const int* pos, const int* slot, const int* rows, void* out,
                                        float* part_o, float* part_ml, int n_rows, int n_head, int n_kv, int hd,
                                        int page_size, float scale, int window, int n_splits,
                                        hipStream_t stream) {
  int rc = check_common("attention_decode", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  return launch_decode<false>(q, pool, table, table_stride, pos, slot, rows, out, part_o, part_ml, n_rows, n_head,
                              n_kv, hd, page_size, scale, window, n_splits, QKPrep{}, stream);
}

// The same for rows 0..n_rows-1 of a step, starting from the 32-bit projections: qkv is float
// [n_rows, row_width] with the q heads first and, if write_kv, the k heads and v heads after
// them.  Per-head norm (q_w, k_w: float [hd] or nullptr), rotation (inv_freq float [hd/2] or
// nullptr; rope_table float [table_len, hd/2, 2] or nullptr) and the write of each row's key
// and value at its own position happen inside the attention kernel.  Returns 3 for what it
// does not serve: head sizes other than 64 and 128, more than 16 q heads per kv head.
extern "C" int ti_attention_decode_prepared_bf16(const float* qkv, int row_width, const float* q_w,
                                                 const float* k_w, float eps, const float* inv_freq,
                                                 const float* rope_table, int table_len, void* pool, int write_kv,
                                                 const int* table, int table_stride, const int* pos,
                                                 const int* slot, void* out, float* part_o, float* part_ml,
                                                 int n_rows, int n_head, int n_kv, int hd, int page_size,
                                                 float scale, int window, int n_splits, hipStream_t stream) {
  int rc = check_common("attention_decode_prepared", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  if (hd == 32 || n_head / n_kv > 16 || ((uintptr_t)q_w & 15) || ((uintptr_t)rope_table & 15)) {
    ti_set_error("attention_decode_prepared: head_dim %d with %d q heads per kv head is not served (or a norm "
                 "weight or the sin/cos table is not 16-byte aligned)", hd, n_head / n_kv);
    return 3;
  }
  TI_REQUIRE(qkv && row_width >= (n_head + (write_kv ? 2 * n_kv : 0)) * hd && row_width % 4 == 0 &&
                 ((uintptr_t)qkv & 15) == 0,
             "attention_decode_prepared: the projections do not fit (row_width %d)", row_width);
  TI_REQUIRE(inv_freq || !rope_table, "attention_decode_prepared: a sin/cos table without inv_freq");
  QKPrep prep{qkv, row_width, q_w, k_w, eps, inv_freq, (const float2*)rope_table, table_len,
              write_kv ? (bf16_t*)pool : nullptr};
  return launch_decode<true>(nullptr, pool, table, table_stride, pos, slot, nullptr, out, part_o, part_ml, n_rows,
                             n_head, n_kv, hd, page_size, scale, window, n_splits, prep, stream);
}

// What the kernels through LDS reach behind a block's descriptor: a page of all heads' keys and values.
static bool prefill_page_fits(int n_kv, int hd, int P) { return 4L * n_kv * P * hd < 0x7fffffffL; }

static int g_prefill_groups = 0;   // for measurements: 1 or 2 wavefront groups per workgroup, 0 = by the launch
static int g_prefill_lds = 1;
static int g_decode_stages = 0;    // LDS stages a wavefront of the decode kernel by records at a head size of 128, 0 = by the launch
// 1: head sizes 64 and 128 take the kernel that shares keys and values through LDS
// (default); 0: every head size takes the kernel that reads them per wavefront

// Portions of prompts.  tiles: int [n_tiles, 2] = (entry, first row), each tile 128 rows, best from the one that sees the most keys on;
// entries: int [n_entries, 4] = (row0, n_tokens, start_pos, -); table row e belongs to entry e.
extern "C" int ti_attention_prefill_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                         const int* tiles, const int* entries, void* out, int n_tiles,
                                         int n_head, int n_kv, int hd, int page_size, float scale, int window,
                                         hipStream_t stream) {
  int rc = check_common("attention_prefill", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  TI_REQUIRE(n_head <= 65535, "attention_prefill: too many heads");
  if (n_tiles == 0) return 0;
  dim3 grid(n_tiles, n_head);
  if (g_prefill_lds && (hd == 64 || hd == 128) && prefill_page_fits(n_kv, hd, page_size)) {
    // two groups of wavefronts per workgroup when the launch would else leave a SIMD with one wavefront
    const int groups = g_prefill_groups ? g_prefill_groups : ((long)n_tiles * n_head < 512 ? 2 : 1);
    const int lds = groups * PF_STAGES * 2 * PF_KEYS * hd * 2;
    static bool ready = false;          // allow more than 64 KiB of dynamic LDS, once
    if (!ready) {
      const int most = 2 * PF_STAGES * 2 * PF_KEYS * 128 * 2;
      if (hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<128, 1>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, most / 2) != hipSuccess ||
          hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<128, 2>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, most) != hipSuccess ||
          hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<64, 1>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, most / 4) != hipSuccess ||
          hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<64, 2>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, most / 2) != hipSuccess) {
        ti_set_error("attention_prefill: cannot reserve %d bytes of LDS", most);
        return 2;
      }
      ready = true;
    }
#define TI_PLDS(H, G)                                                                                          \
  attn_prefill_lds_kernel<H, G><<<grid, 256 * G, lds, stream>>>((const bf16_t*)q, (const bf16_t*)pool, table,   \
                                                                table_stride, tiles, n_tiles, entries,          \
                                                                (bf16_t*)out, n_head, n_kv, page_size, scale,   \
                                                                window, nullptr, nullptr, g_softcap, g_sink)
    if (hd == 128 && groups == 2) TI_PLDS(128, 2);
    else if (hd == 128) TI_PLDS(128, 1);
    else if (groups == 2) TI_PLDS(64, 2);
    else TI_PLDS(64, 1);
#undef TI_PLDS
    TI_LAUNCH_CHECK();
    return 0;
  }
#define TI_PRE(H)                                                                                          \
  case H:                                                                                                  \
    attn_prefill_kernel<H><<<grid, 512, 0, stream>>>((const bf16_t*)q, (const bf16_t*)pool, table,          \
                                                     table_stride, tiles, entries, (bf16_t*)out, n_head,    \
                                                     n_kv, page_size, scale, window, g_softcap, g_sink);    \
    break;
  switch (hd) {
    TI_PRE(32) TI_PRE(64) TI_PRE(128)
  }
#undef TI_PRE
  TI_LAUNCH_CHECK();
  return 0;
}

// The same for launches of few tiles.  tiles: int [n_tiles, 2] = (entry, first row) of tiles of 64 rows, ordered from the
// tile that sees the most keys to the one that sees the fewest.  A workgroup takes a tile, the heaviest ones of all heads
// first, or where the caller asks for pairs (1) tile b and tile n_tiles - 1 - b, one after the other; 2: a tile, its heads together (see
// prefill_tiles); four groups of two wavefronts take the turns of keys in rotation.  Returns 3 for head sizes other than 64 and 128 and for pages of 2 GiB and more.
extern "C" int ti_attention_prefill_paired_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                                const int* tiles, const int* entries, void* out, int n_tiles,
                                                int n_head, int n_kv, int hd, int page_size, float scale,
                                                int window, int n_rows, float* part_o, float* part_ml,
                                                int n_splits, int paired, hipStream_t stream) {
  int rc = check_common("attention_prefill_paired", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  if (hd == 32) {
    ti_set_error("attention_prefill_paired: head_dim 32 is not served (64, 128)");
    return 3;
  }
  if (!prefill_page_fits(n_kv, hd, page_size)) {
    ti_set_error("attention_prefill_paired: pages of 2 GiB and more are not served");
    return 3;
  }
  TI_REQUIRE(n_head <= 65535, "attention_prefill_paired: too many heads");
  TI_REQUIRE(n_splits >= 1 && n_splits <= 8 && (n_splits == 1 || (part_o && part_ml && n_rows > 0)),
             "attention_prefill_paired: 1 to 8 runs of keys, more than one with buffers for their results");
  if (n_tiles == 0) return 0;
  constexpr int NG = 4, NW = 2, ST = 2, CB = 1;
  const int lds = hd == 128 ? PrefillLds<128, NG, NW, ST>::BYTES : PrefillLds<64, NG, NW, ST>::BYTES;
  static bool ready = false;          // allow more than 64 KiB of dynamic LDS, once
  if (!ready) {
    if (hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<128, NG, NW, ST, true, CB>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<128, NG, NW, ST>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<64, NG, NW, ST, true, CB>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<64, NG, NW, ST>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<128, NG, NW, ST, false, CB>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<128, NG, NW, ST>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<128, NG, NW, ST, false, CB, true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<128, NG, NW, ST>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<64, NG, NW, ST, false, CB, true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<64, NG, NW, ST>::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_prefill_lds_kernel<64, NG, NW, ST, false, CB>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, PrefillLds<64, NG, NW, ST>::BYTES) != hipSuccess) {
      ti_set_error("attention_prefill_paired: cannot reserve the LDS");
      return 2;
    }
    ready = true;
  }
  const bool pairs = paired == 1;
  dim3 grid(pairs ? (n_tiles + 1) / 2 : n_tiles, n_head, n_splits);
#define TI_GO(H, PAIRED, TOGETHER)                                                                                \
  attn_prefill_lds_kernel<H, NG, NW, ST, PAIRED, CB, TOGETHER><<<grid, 64 * NW * NG, lds, stream>>>(                            \
      (const bf16_t*)q, (const bf16_t*)pool, table, table_stride, tiles, n_tiles, entries, (bf16_t*)out, n_head, \
      n_kv, page_size, scale, window, part_o, part_ml, g_softcap, g_sink)
  const bool together = paired == 2 && n_kv % 8 != 0;
  if (hd == 128 && pairs) TI_GO(128, true, false);
  else if (hd == 128 && together) TI_GO(128, false, true);
  else if (hd == 128) TI_GO(128, false, false);
  else if (pairs) TI_GO(64, true, false);
  else if (together) TI_GO(64, false, true);
  else TI_GO(64, false, false);
#undef TI_GO
  if (n_splits > 1) {
    // every row of the step has its runs (rows of single tokens too: theirs are not read by anyone)
    if (hd == 128)
      attn_merge_kernel<128><<<dim3(n_rows, n_head), 128, 0, stream>>>(part_o, part_ml, nullptr, (bf16_t*)out, n_head,
                                                                     n_splits, g_sink);
    else
      attn_merge_kernel<64><<<dim3(n_rows, n_head), 64, 0, stream>>>(part_o, part_ml, nullptr, (bf16_t*)out, n_head,
                                                                   n_splits, g_sink);
  }
  TI_LAUNCH_CHECK();
  return 0;
}

// What a launch by records needs: n_runs records of run_stride ints, and where rows are cut (n_rows > 0) the rows' records
// int [n_rows][4] and buffers for the runs' results, [n_runs][n_head][hd] and [n_runs][n_head][2].
static int check_runs(const char* what, const int* runs, int n_runs, int run_stride, const int* rows, int n_rows, const float* part_o,
                      const float* part_ml) {
  TI_REQUIRE(runs && n_runs > 0 && n_runs <= 65535 && run_stride >= TI_RUN_HEAD, "%s: records (%d of %d ints)", what, n_runs, run_stride);
  TI_REQUIRE(n_rows == 0 || (n_rows > 0 && rows && part_o && part_ml), "%s: rows in several runs need records and buffers", what);
  return 0;
}

// ti_attention_decode_prepared_bf16 by records (see DecodeRuns).  Serves the same sizes.
extern "C" int ti_attention_decode_runs_bf16(const float* qkv, int row_width, const float* q_w, const float* k_w, float eps,
                                             const float* inv_freq, const float* rope_table, int table_len, void* pool, int write_kv,
                                             const int* table, int table_stride, const int* runs, int n_runs, int run_stride,
                                             const int* rows, int n_rows, void* out, float* part_o, float* part_ml, int n_head, int n_kv,
                                             int hd, int page_size, float scale, int window, hipStream_t stream) {
  int rc = check_common("attention_decode_runs", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  if (hd == 32 || n_head / n_kv > 16 || ((uintptr_t)q_w & 15) || ((uintptr_t)rope_table & 15)) {
    ti_set_error("attention_decode_runs: head_dim %d with %d q heads per kv head is not served (or a norm "
                 "weight or the sin/cos table is not 16-byte aligned)", hd, n_head / n_kv);
    return 3;
  }
  TI_REQUIRE(qkv && row_width >= (n_head + (write_kv ? 2 * n_kv : 0)) * hd && row_width % 4 == 0 && ((uintptr_t)qkv & 15) == 0,
             "attention_decode_runs: the projections do not fit (row_width %d)", row_width);
  TI_REQUIRE(inv_freq || !rope_table, "attention_decode_runs: a sin/cos table without inv_freq");
  rc = check_runs("attention_decode_runs", runs, n_runs, run_stride, rows, n_rows, part_o, part_ml);
  if (rc) return rc;
  static bool ready = false;          // allow more than 64 KiB of dynamic LDS, once
  if (!ready) {
    if (hipFuncSetAttribute((const void*)attn_decode_runs_kernel<128, 1>, hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(StagedMerge<128, 4, 1>)) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_decode_runs_kernel<128, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(StagedMerge<128, 4, 2>)) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_decode_runs_kernel<64, 2>, hipFuncAttributeMaxDynamicSharedMemorySize, sizeof(StagedMerge<64, 4, 2>)) != hipSuccess) {
      ti_set_error("attention_decode_runs: cannot reserve the LDS");
      return 2;
    }
    ready = true;
  }
#define TI_GO(H, S)                                                                                                          \
  attn_decode_runs_kernel<H, S><<<dim3(n_kv, n_runs), 256, sizeof(StagedMerge<H, 4, S>), stream>>>(                                                     \
      runs, run_stride, n_head / n_kv, qkv, row_width, n_kv, (const float2*)rope_table, (const bf16_t*)pool, page_size, table_len, \
      q_w, k_w, table, table_stride, window, inv_freq, write_kv ? (bf16_t*)pool : nullptr, eps, scale, (bf16_t*)out, part_o, part_ml)
  if (hd == 64) TI_GO(64, 2);
  // two stages (133 KiB) where a unit has one workgroup at most; one (69 KiB) where two share it, so that one walks while the other starts
  else if (g_decode_stages ? g_decode_stages == 2 : n_kv * n_runs <= compute_units()) TI_GO(128, 2);
  else TI_GO(128, 1);
#undef TI_GO
  if (n_rows) {
    if (hd == 128) attn_merge_kernel<128, true><<<dim3(n_rows, n_head), 128, 0, stream>>>(part_o, part_ml, rows, (bf16_t*)out, n_head, 0, nullptr);
    else attn_merge_kernel<64, true><<<dim3(n_rows, n_head), 64, 0, stream>>>(part_o, part_ml, rows, (bf16_t*)out, n_head, 0, nullptr);
  }
  TI_LAUNCH_CHECK();
  return 0;
}

// Portions (tiles of 64 rows as above, unpaired, whole) and the single-token rows of the same step (by records) in one
// launch; softcap as for the entry points below.  Returns 3 for head sizes other than 64 and 128.
extern "C" int ti_attention_step_bf16(const void* q, const void* pool, const int* table, int table_stride, const int* tiles,
                                      const int* entries, int n_tiles, const int* runs, int n_runs, int run_stride, const int* rows,
                                      int n_rows, void* out, float* part_o, float* part_ml, int n_head, int n_kv, int hd, int page_size,
                                      float scale, float softcap, int window, hipStream_t stream) {
  int rc = check_common("attention_step", n_head, n_kv, hd, page_size, table_stride);
  if (rc) return rc;
  if (hd == 32) {
    ti_set_error("attention_step: head_dim 32 is not served (64, 128)");
    return 3;
  }
  if (!prefill_page_fits(n_kv, hd, page_size)) {
    ti_set_error("attention_step: pages of 2 GiB and more are not served");
    return 3;
  }
  TI_REQUIRE(n_tiles > 0 && tiles && entries, "attention_step: no tiles");
  rc = check_runs("attention_step", runs, n_runs, run_stride, rows, n_rows, part_o, part_ml);
  if (rc) return rc;
  const int parts = (n_head / n_kv + 15) / 16;
  const long grid = (long)n_tiles * n_head + (long)n_runs * n_kv * parts;
  TI_REQUIRE(grid <= 0x7fffffL, "attention_step: too many workgroups");
  typedef PrefillLds<128, 4, 2, 2> Lds128;
  typedef PrefillLds<64, 4, 2, 2> Lds64;
  static_assert(sizeof(StagedMerge<128, 8, 1>) <= Lds128::BYTES && sizeof(StagedMerge<64, 8, 1>) <= Lds64::BYTES, "the runs' stages and merge fit");
  static bool ready = false;          // allow more than 64 KiB of dynamic LDS, once
  if (!ready) {
    if (hipFuncSetAttribute((const void*)attn_step_kernel<128>, hipFuncAttributeMaxDynamicSharedMemorySize, Lds128::BYTES) != hipSuccess ||
        hipFuncSetAttribute((const void*)attn_step_kernel<64>, hipFuncAttributeMaxDynamicSharedMemorySize, Lds64::BYTES) != hipSuccess) {
      ti_set_error("attention_step: cannot reserve the LDS");
      return 2;
    }
    ready = true;
  }
  const float cap = softcap > 0.f ? softcap : 0.f;
#define TI_GO(H)                                                                                                              \
  do {                                                                                                                        \
    attn_step_kernel<H><<<(unsigned)grid, 512, Lds##H::BYTES, stream>>>((const bf16_t*)q, (const bf16_t*)pool, table, table_stride, \
                                                                     tiles, n_tiles, entries, runs, run_stride, n_head / n_kv,  \
                                                                     (bf16_t*)out, part_o, part_ml,                              \
                                                                     n_head, n_kv, page_size, scale, window, cap, g_sink);       \
    if (n_rows)                                                                                                               \
      attn_merge_kernel<H, true><<<dim3(n_rows, n_head), H, 0, stream>>>(part_o, part_ml, rows, (bf16_t*)out, n_head, 0, g_sink); \
  } while (0)
  if (hd == 128) TI_GO(128);
  else TI_GO(64);
#undef TI_GO
  TI_LAUNCH_CHECK();
  return 0;
}

// The three entry points above with soft-capped scores: s <- softcap tanh(s / softcap) before the softmax.
struct CapScope {
  explicit CapScope(float cap) { g_softcap = cap > 0.f ? cap : 0.f; }
  ~CapScope() { g_softcap = 0.f; }
};
extern "C" int ti_attention_decode_capped_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                               const int* pos, const int* slot, const int* rows, void* out, float* part_o,
                                               float* part_ml, int n_rows, int n_head, int n_kv, int hd, int page_size,
                                               float scale, float softcap, int window, int n_splits, hipStream_t stream) {
  CapScope cap(softcap);
  return ti_attention_decode_bf16(q, pool, table, table_stride, pos, slot, rows, out, part_o, part_ml, n_rows, n_head, n_kv, hd,
                                  page_size, scale, window, n_splits, stream);
}
extern "C" int ti_attention_prefill_capped_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                                const int* tiles, const int* entries, void* out, int n_tiles, int n_head,
                                                int n_kv, int hd, int page_size, float scale, float softcap, int window,
                                                hipStream_t stream) {
  CapScope cap(softcap);
  return ti_attention_prefill_bf16(q, pool, table, table_stride, tiles, entries, out, n_tiles, n_head, n_kv, hd, page_size, scale,
                                   window, stream);
}
extern "C" int ti_attention_prefill_paired_capped_bf16(const void* q, const void* pool, const int* table, int table_stride,
                                                       const int* tiles, const int* entries, void* out, int n_tiles, int n_head,
                                                       int n_kv, int hd, int page_size, float scale, float softcap, int window,
                                                       int n_rows, float* part_o, float* part_ml, int n_splits, int paired,
                                                       hipStream_t stream) {
  CapScope cap(softcap);
  return ti_attention_prefill_paired_bf16(q, pool, table, table_stride, tiles, entries, out, n_tiles, n_head, n_kv, hd, page_size,
                                          scale, window, n_rows, part_o, part_ml, n_splits, paired, stream);
}

// ------------------------------------------------------------------- tests and measurements
// One entry for every choice above that a test or a measurement may want to force (names as in
// tinyinfer_kernels_tuning.h); process-wide in the library, applied and reset around its calls by the
// host library's Ops.  Returns 0, or 1 for an unknown name.
extern "C" void ti_tuning_reset() {
  g_prefill_groups = 0;
  g_prefill_lds = 1;
  g_decode_stages = 0;
}
extern "C" int ti_tuning_set(const char* name, long value) {
  const std::string n = name ? name : "";
  if (n == "prefill_groups") g_prefill_groups = (int)value;
  else if (n == "prefill_use_lds") g_prefill_lds = (int)value;
  else if (n == "decode_stages") g_decode_stages = (int)value;
  else return 1;
  return 0;
}
