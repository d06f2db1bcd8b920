// Sampling on the device: greedy argmax (of equal logits the lowest index wins,
// as src/cuda/sample.cu:5-11) and temperature sampling with
// optional top-k and top-p cuts (src/main.cpp:40-83 does these
// on the host with a sort).  Several workgroups read a long row, and one finishes it.
//
// Temperature sampling draws by inverse CDF over the index order from one
// uniform number per row, which the host derives from (seed, request, number of
// tokens generated), so a draw does not depend on what else is in the batch.
// The cuts are the k-th largest logit and the logit at which the descending
// cumulative mass reaches top_p, both found on the order-preserving integer
// image of the floats: by radix with many workgroups a row where there is a
// top-k cut, else by 32 steps of bisection each in one workgroup.  Every sum is
// reduced in a fixed order, so the result is reproducible.
#include <algorithm>
#include <mutex>

#include "common.h"
#include "tinyinfer_kernels.h"

TI_ERROR_API

#define SNT 1024

__device__ __forceinline__ uint32_t order_key(float f) {
  uint32_t u = __float_as_uint(f);
  if (u == 0x80000000u) u = 0u;                  // -0 and +0 are equal logits
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ int block_sum_int(int v, int* red) {
#pragma unroll
  for (int o = TI_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, TI_WAVE);
  __syncthreads();
  if ((threadIdx.x & (TI_WAVE - 1)) == 0) red[threadIdx.x / TI_WAVE] = v;
  __syncthreads();
  int t = 0;
#pragma unroll
  for (int i = 0; i < SNT / TI_WAVE; ++i) t += red[i];
  return t;
}

__device__ int row_argmax(const float* __restrict__ row, int V, float* s_val, int* s_idx) {
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = threadIdx.x; i < V; i += SNT) {
    const float v = row[i];
    if (v > bv || (bi == 0x7fffffff && v == v)) {   // first finite or -inf value, then strictly greater
      bv = v;
      bi = i;
    }
  }
#pragma unroll
  for (int o = TI_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, TI_WAVE);
    const int oi = __shfl_xor(bi, o, TI_WAVE);
    if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  }
  __syncthreads();
  if ((threadIdx.x & (TI_WAVE - 1)) == 0) {
    s_val[threadIdx.x / TI_WAVE] = bv;
    s_idx[threadIdx.x / TI_WAVE] = bi;
  }
  __syncthreads();
  float fv = s_val[0];
  int fi = s_idx[0];
  for (int i = 1; i < SNT / TI_WAVE; ++i) {
    const float ov = s_val[i];
    const int oi = s_idx[i];
    if (oi != 0x7fffffff && (fi == 0x7fffffff || ov > fv || (ov == fv && oi < fi))) {
      fv = ov;
      fi = oi;
    }
  }
  return fi == 0x7fffffff ? 0 : fi;
}

__global__ void __launch_bounds__(SNT)
argmax_kernel(const float* __restrict__ logits, int* __restrict__ out, int V) {
  __shared__ float s_val[SNT / TI_WAVE];
  __shared__ int s_idx[SNT / TI_WAVE];
  const int r = blockIdx.x;
  const int best = row_argmax(logits + (size_t)r * V, V, s_val, s_idx);
  if (threadIdx.x == 0) out[r] = best;
}

// Greedy choice of a long row in two steps, so that a row is read by many
// workgroups at once: grid (rows, ARG_PARTS) finds the best of each slice, then
// one wavefront per row picks among the ARG_PARTS winners (lowest index on ties).
#define ARG_PARTS 64
__global__ void __launch_bounds__(256)
argmax_part_kernel(const float* __restrict__ logits, float* __restrict__ part_val, int* __restrict__ part_idx,
                   int V) {
  __shared__ float s_val[4];
  __shared__ int s_idx[4];
  const int r = blockIdx.x, c = blockIdx.y;
  const int chunk = (V + ARG_PARTS - 1) / ARG_PARTS;
  const int b = c * chunk, e = min(V, b + chunk);
  const float* row = logits + (size_t)r * V;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  for (int i = b + threadIdx.x; i < e; i += 256) {
    const float v = row[i];
    if (v > bv || (bi == 0x7fffffff && v == v)) {
      bv = v;
      bi = i;
    }
  }
#pragma unroll
  for (int o = TI_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, TI_WAVE);
    const int oi = __shfl_xor(bi, o, TI_WAVE);
    if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  }
  if ((threadIdx.x & 63) == 0) {
    s_val[threadIdx.x >> 6] = bv;
    s_idx[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      const float ov = s_val[w];
      const int oi = s_idx[w];
      if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) {
        bv = ov;
        bi = oi;
      }
    }
    part_val[r * ARG_PARTS + c] = bv;
    part_idx[r * ARG_PARTS + c] = bi;
  }
}

__global__ void __launch_bounds__(64)
argmax_final_kernel(const float* __restrict__ part_val, const int* __restrict__ part_idx, int* __restrict__ out) {
  const int r = blockIdx.x;
  float bv = part_val[r * ARG_PARTS + threadIdx.x];
  int bi = part_idx[r * ARG_PARTS + threadIdx.x];
#pragma unroll
  for (int o = TI_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, TI_WAVE);
    const int oi = __shfl_xor(bi, o, TI_WAVE);
    if (oi != 0x7fffffff && (bi == 0x7fffffff || ov > bv || (ov == bv && oi < bi))) {
      bv = ov;
      bi = oi;
    }
  }
  if (threadIdx.x == 0) out[r] = bi == 0x7fffffff ? 0 : bi;
}

// What the rows of a call ask for: in memory of the device's, or up to S_VALUES rows of it in the launch's own arguments, which
// costs no copy (one of 1 KiB takes 3 us on the stream and as long on the host).
struct SampleRow {
  float temp;
  int top_k;
  float top_p, uni;
};
struct RowsInMemory {
  const float* temp;
  const int* top_k;
  const float *top_p, *uni;
  __device__ __forceinline__ SampleRow at(int r) const { return SampleRow{temp[r], top_k[r], top_p[r], uni[r]}; }
};
#define S_VALUES 64
struct RowsByValue {
  SampleRow row[S_VALUES];
  __device__ __forceinline__ SampleRow at(int r) const { return row[r]; }
};

// temp[r] <= 0: greedy.  top_k[r] <= 0 or >= V: no top-k cut.  top_p[r] >= 1: no top-p cut.
// One workgroup walks the whole row some seventy times: the way for the rows that the two short
// kernels below do not serve, and for a caller without their workspace.
__device__ void sample_row_by_bisection(const float* __restrict__ logits, SampleRow want, int* __restrict__ out, int V, int r) {
  __shared__ float s_val[SNT / TI_WAVE];
  __shared__ int s_idx[SNT / TI_WAVE];
  __shared__ float s_chunk[SNT];
  __shared__ int s_pick;
  const float* row = logits + (size_t)r * V;
  const float T = want.temp;
  const int best = row_argmax(row, V, s_val, s_idx);
  if (!(T > 0.f)) {
    if (threadIdx.x == 0) out[r] = best;
    return;
  }
  const float mx = row[best];
  const float inv_t = 1.0f / T;

  uint32_t cut = 0;   // keep keys >= cut
  const int k = want.top_k;
  if (k > 0 && k < V) {
    uint32_t prefix = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = prefix | (1u << bit);
      int c = 0;
      for (int i = threadIdx.x; i < V; i += SNT) c += (row[i] == row[i] && order_key(row[i]) >= cand) ? 1 : 0;
      c = block_sum_int(c, s_idx);
      if (c >= k) prefix = cand;
    }
    cut = prefix;
  }
  const float p_keep = want.top_p;
  if (p_keep < 1.0f) {
    float s = 0.f;
    for (int i = threadIdx.x; i < V; i += SNT) {
      const float v = row[i];
      if (v == v && order_key(v) >= cut) s += expf((v - mx) * inv_t);
    }
    const float total = block_sum<SNT>(s, s_val);
    const float need = p_keep * total;
    uint32_t prefix = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t cand = prefix | (1u << bit);
      float ms = 0.f;
      for (int i = threadIdx.x; i < V; i += SNT) {
        const float v = row[i];
        if (v == v && order_key(v) >= cand && order_key(v) >= cut) ms += expf((v - mx) * inv_t);
      }
      ms = block_sum<SNT>(ms, s_val);
      if (ms >= need) prefix = cand;
    }
    if (prefix > cut) cut = prefix;
  }

  // inverse CDF over the index order; thread t owns indices [t*C, (t+1)*C)
  const int C = (V + SNT - 1) / SNT;
  const int b = threadIdx.x * C, e = min(V, b + C);
  float cs = 0.f;
  for (int i = b; i < e; ++i) {
    const float v = row[i];
    if (v == v && order_key(v) >= cut) cs += expf((v - mx) * inv_t);
  }
  s_chunk[threadIdx.x] = cs;
  if (threadIdx.x == 0) s_pick = -1;
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0.f;
    for (int i = 0; i < SNT; ++i) total += s_chunk[i];
    const float target = want.uni * total;
    float acc = 0.f;
    int owner = -1, last_nonzero = 0;
    for (int i = 0; i < SNT; ++i) {
      if (s_chunk[i] > 0.f) last_nonzero = i;
      if (owner < 0 && s_chunk[i] > 0.f && target < acc + s_chunk[i]) {
        owner = i;
        break;
      }
      acc += s_chunk[i];
    }
    if (owner < 0) {   // rounding pushed the target past the end: the last kept entry
      owner = last_nonzero;
      acc = -1.f;      // marks "take the owner's last kept index"
    }
    // walk the owner's chunk
    const int ob = owner * C, oe = min(V, ob + C);
    int pick = -1, last = -1;
    float a = acc;
    for (int i = ob; i < oe; ++i) {
      const float v = row[i];
      if (!(v == v) || order_key(v) < cut) continue;
      last = i;
      if (acc < 0.f) continue;
      a += expf((v - mx) * inv_t);
      if (target < a) {
        pick = i;
        break;
      }
    }
    s_pick = pick >= 0 ? pick : (last >= 0 ? last : best);
  }
  __syncthreads();
  if (threadIdx.x == 0) out[r] = s_pick;
}

template <class Rows>
__global__ void __launch_bounds__(SNT)
sample_kernel(const float* __restrict__ logits, Rows rows, int* __restrict__ out, int V) {
  sample_row_by_bisection(logits, rows.at(blockIdx.x), out, V, blockIdx.x);
}

// ------------------------------------------------------------ the same draw in two short kernels
// A row of 151,936 logits cut to its 512 largest: the kernel above takes 0.9 ms (1.8 with a top-p
// cut), as long as a whole decode step, because one workgroup reads the row once per bit of the
// answer.  Here the k-th largest key is found by radix, and many workgroups share a row:
//   part    a workgroup holds S_SPAN keys of a row in registers, finds its own k-th largest (counts of the keys'
//           upper 12 bits in LDS, and of the next 10 and the last 10 where a bin holds too many) and leaves
//           what is at or above it, or in its bin, as (key, index) pairs: the row's k largest are among them.  It says as
//           well from where up its own share of the k, k / parts, lies;
//   finish  one workgroup per row: at least k keys lie at or above the least of the parts' shares, so it takes those pairs alone (some
//           700 of 10,000 for k = 512), finds the k-th key among them the same way, keeps it and those above,
//           sorts what is kept by logit where there is a top-p cut and sums the weights in that order, sorts
//           what is left by index and draws by inverse CDF.  Sums are scans of a fixed shape.
// It draws what the kernel above draws, up to the rounding of sums that are taken in another order.
// Rows that it does not serve (no top-k cut, a cut beyond S_MAX_K, more keys of a part that are equal
// at the row's cut than it has room for) are left to that kernel's walk, inside the last kernel.  A part may hold thousands of equal
// keys at its own k-th while the row's cut lies above them (a masked row: a few logits a part beside as many masked ones as there are):
// it leaves what is above them and says which they are, and the row is served if k pairs are above all of those.  (64 rows of
// 151,936 with 1,000 logits left at random, us: a cut of 50 61, of 500 with a top-p cut 81; when such parts sent their rows to the walk
// 1,016 and 3,872.)
//
// 64 rows of 151,936, greedy, top-k 50 and top-p, 512 and 20 in turn, us: three passes over the row's memory and a finish
// with two sorts by rank 9.9 + 12.9 + 14.3 + 23.0; this 13.4 + 16.8.  Of the first, 9.5 are the loads and the counts (39 MB, and a
// workgroup's counts wait for its loads); the second is a chain of some thirty short steps with a barrier each (a greedy row's 6.8).
// Parts of 8,192 keys 13.1 + 18.1; without the shares the finish's counts of 10,000 pairs a row took 3 us more.
#define S_BITS 12
#define S_BINS (1 << S_BITS)
#define S_BITS2 10                               // the next digits
#define S_BINS2 (1 << S_BITS2)
#define S_CAND 4096                              // pairs a workgroup may leave of its part, and the finish may keep
#define S_MAX_K 3584                             // the largest cut served: room for equals and for a bin's others
#define S_NT 512
#define S_LOADS 20                               // keys a thread holds
#define S_SPAN (S_NT * S_LOADS)
static_assert(S_BITS + 2 * S_BITS2 == 32, "a key is three digits");

__device__ __forceinline__ float key_value(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}
// the cut that the radix kernels find for a row: a greedy row is a cut to the largest key; 0: not served
__device__ __forceinline__ int served_cut(const SampleRow& want, int V) {
  const int k = want.temp > 0.f ? want.top_k : 1;
  return (k > 0 && k < V && k <= S_MAX_K) ? k : 0;
}

// The sum of v over this lane and those below it: shifts inside rows of 16 lanes and two broadcasts, no trip through LDS.
__device__ __forceinline__ int wave_prefix(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // row_shr:1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // lane 15 of a row to the next, 31 to the upper half
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// Which of BINS counts in LDS holds the k-th largest key, how many keys lie in the bins above it, and how many in it.  Every
// thread of the workgroup's NT calls it and gets all three; what it leaves in the counts is zero.
// k beyond the number of keys: the lowest bin that holds a key.  No keys: bin -1.  share_bin: the bin of the share-th largest, 0 where
// there are fewer.
template <int BINS, int NT>
__device__ void bin_of_kth(int* s_bins, int k, int* s_wave, int* s_res, int& bin, int& above, int& in, int share = 0, int* share_bin = nullptr) {
  constexpr int OWN = BINS / NT, WAVES = NT / TI_WAVE;
  const int t = threadIdx.x, lane = t & (TI_WAVE - 1), wave = t / TI_WAVE;
  int* own = s_bins + BINS - OWN * (t + 1);        // the first threads own the highest bins
  int c[OWN], mine = 0;
  if constexpr (OWN % 4 == 0) {
#pragma unroll
    for (int j = 0; j < OWN; j += 4) {
      int4* p = reinterpret_cast<int4*>(own + j);
      const int4 q = *p;
      *p = make_int4(0, 0, 0, 0);
      c[j] = q.x, c[j + 1] = q.y, c[j + 2] = q.z, c[j + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int j = 0; j < OWN; ++j) {
      c[j] = own[j];
      own[j] = 0;
    }
  }
#pragma unroll
  for (int j = 0; j < OWN; ++j) mine += c[j];
  int run = wave_prefix(mine), total = 0;
  if (lane == TI_WAVE - 1) s_wave[wave] = run;
  run -= mine;                                     // keys in the bins above this thread's
  if (t == 0) s_res[0] = -1, s_res[1] = 0, s_res[2] = 0, s_res[3] = 0;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    const int n = s_wave[w];
    if (w < wave) run += n;
    total += n;
  }
  const int kk = k < total ? k : total;
  if (kk >= 1) {
#pragma unroll
    for (int j = OWN - 1; j >= 0; --j) {
      if (run < kk && run + c[j] >= kk) s_res[0] = BINS - OWN * (t + 1) + j, s_res[1] = run, s_res[2] = c[j];
      if (run < share && run + c[j] >= share) s_res[3] = BINS - OWN * (t + 1) + j;
      run += c[j];
    }
  }
  __syncthreads();
  bin = s_res[0];
  above = s_res[1];
  in = s_res[2];
  if (share_bin) *share_bin = s_res[3];
  __syncthreads();
}

// Where this lane's `n` entries go behind *s_count: one counter's step a wavefront.  All lanes call it.
__device__ __forceinline__ int next_places(int* s_count, int n) {
  const int upto = wave_prefix(n), all = __builtin_amdgcn_readlane(upto, TI_WAVE - 1);
  if (all == 0) return 0;
  int at = 0;
  if ((threadIdx.x & (TI_WAVE - 1)) == 0) at = atomicAdd(s_count, all);
  return __builtin_amdgcn_readfirstlane(at) + upto - n;
}

// Counts the digits of the lanes that are `on`.  What shares the first such lane's digit is added at once: thousands of masked
// logits are one key, and a step each on one counter takes 30 us a digit (138 us for the latter rows above).  For the digits behind the
// first: there it took ordinary rows 3.7 us of 27.  All lanes call it.
__device__ __forceinline__ void count_digit(int* s_bins, bool on, int digit) {
  const unsigned long long lanes = __ballot(on);
  if (lanes == 0) return;
  const int first = __builtin_ctzll(lanes), shared = __builtin_amdgcn_readlane(digit, first);
  const int n = __popcll(__ballot(on && digit == shared));
  if ((int)(threadIdx.x & (TI_WAVE - 1)) == first) atomicAdd(&s_bins[shared], n);
  else if (on && digit != shared) atomicAdd(&s_bins[digit], 1);
}

// grid (parts of `span` keys, rows), span a multiple of 4, at most S_SPAN.  WIDE: rows of whole float4s on their boundaries, four
// neighbours a load.  left [row][parts], pairs [row][parts][S_CAND] (key << 32 | ~index).  (64 registers a thread: four workgroups to a unit, so that 64 rows of 15 parts are one round.)
struct PartLeft {
  int pairs;
  uint32_t share;      // the key from which the part's share lies
  uint32_t over;       // the k-th key, if it has more equals than there is room for: the part's pairs are those above it (0: no such key)
};
template <bool WIDE, class Rows>
__global__ void __launch_bounds__(S_NT)
sample_part_kernel(const float* __restrict__ logits, Rows rows, PartLeft* __restrict__ left, unsigned long long* __restrict__ pairs,
                   int V, int span) {
  __shared__ __attribute__((aligned(16))) int s_bins[S_BINS];
  __shared__ int s_wave[S_NT / TI_WAVE], s_res[4], s_count;
  const int r = blockIdx.y, t = threadIdx.x;
  const int k = served_cut(rows.at(r), V);
  if (k == 0) return;                              // the whole workgroup
  const float* row = logits + (size_t)r * V;
  const size_t part = (size_t)r * gridDim.x + blockIdx.x;
  const int base = blockIdx.x * span, end = min(V, base + span);
  const float none = __uint_as_float(0x7fc00000u);
  float v[S_LOADS];
  // key u of a thread is the row's base + place(u)
  const auto place = [&](int u) { return WIDE ? S_NT * (u & ~3) + 4 * t + (u & 3) : S_NT * u + t; };
#pragma unroll
  for (int u = 0; u < S_LOADS; u += WIDE ? 4 : 1) {
    const int i = base + place(u);
    if (WIDE) {
      const float4 q = i < end ? *reinterpret_cast<const float4*>(row + i) : make_float4(none, none, none, none);
      v[u] = q.x, v[u + 1] = q.y, v[u + 2] = q.z, v[u + 3] = q.w;
    } else {
      v[u] = i < end ? row[i] : none;
    }
  }
  for (int i = t; i < S_BINS / 4; i += S_NT) reinterpret_cast<int4*>(s_bins)[i] = make_int4(0, 0, 0, 0);
  if (t == 0) s_count = 0;
  __syncthreads();
  uint32_t key[S_LOADS];                           // 0, which is no number's: NaN is never drawn
#pragma unroll
  for (int u = 0; u < S_LOADS; ++u) {
    key[u] = v[u] == v[u] ? order_key(v[u]) : 0;
    if (key[u]) atomicAdd(&s_bins[key[u] >> (32 - S_BITS)], 1);
  }
  __syncthreads();
  int bin, above, in, share_bin, taken = 0, need = k, shift = 32 - S_BITS;      // taken: keys above the prefix
  bin_of_kth<S_BINS, S_NT>(s_bins, need, s_wave, s_res, bin, above, in, (k + gridDim.x - 1) / gridDim.x, &share_bin);
  if (bin < 0) {
    if (t == 0) left[part] = PartLeft{0, 0, 0};
    return;
  }
  uint32_t prefix = bin;
  // few more than k is good enough: the finish looks at 15 such parts of a row of 151,936
  const int enough = min(S_CAND, max(1024, k + 512));
  while (above + taken + in > enough && shift > 0) {
    taken += above;
    need -= above;
#pragma unroll
    for (int u = 0; u < S_LOADS; ++u)
      count_digit(s_bins, key[u] && (key[u] >> shift) == prefix, (int)((key[u] >> (shift - S_BITS2)) & (S_BINS2 - 1)));
    __syncthreads();
    bin_of_kth<S_BINS2, S_NT>(s_bins, need, s_wave, s_res, bin, above, in);
    prefix = (prefix << S_BITS2) | (uint32_t)bin;
    shift -= S_BITS2;
  }
  unsigned long long* mine = pairs + part * S_CAND;
  const uint32_t over = above + taken + in > S_CAND ? prefix : 0;         // (a whole key then: all its digits have been looked at)
  const uint32_t least = over ? over + 1 : max(prefix << shift, 1u);       // fewer than k keys are above the k-th
  int n = 0;
#pragma unroll
  for (int u = 0; u < S_LOADS; ++u) n += key[u] >= least ? 1 : 0;
  int at = next_places(&s_count, n);
#pragma unroll
  for (int u = 0; u < S_LOADS; ++u)
    if (key[u] >= least) mine[at++] = ((unsigned long long)key[u] << 32) | (uint32_t)~(base + place(u));
  __syncthreads();
  if (t == 0) left[part] = PartLeft{s_count, (uint32_t)share_bin << (32 - S_BITS), over};
}

// sorts a[0..n) of LDS downwards by the entries' upper words, n <= S_CAND; every thread of the workgroup
// calls it.  Up to S_BY_RANK entries each thread counts the entries above its own and puts it there (reads of four keys
// that the whole wavefront shares, no barrier between them); entries with equal
// upper words take neighbouring places in the order in which they come.  More entries are sorted by a
// bitonic network on the whole entries, a barrier a stage.  tmp: room for S_BY_RANK entries, as many counters and as many keys.
#define S_BY_RANK 1024
__device__ void sort_down(unsigned long long* a, int n, unsigned long long* tmp) {
  if (n <= S_BY_RANK) {
    int* taken = reinterpret_cast<int*>(tmp + S_BY_RANK);
    uint32_t* keys = reinterpret_cast<uint32_t*>(taken + S_BY_RANK);
    const int i = threadIdx.x;
    unsigned long long x = 0;
    if (i < n) {
      x = a[i];
      taken[i] = 0;
    }
    if (i < ((n + 3) & ~3)) keys[i] = (uint32_t)(x >> 32);         // beyond n: 0, above nothing
    __syncthreads();
    if (i < n) {
      const uint32_t mine = (uint32_t)(x >> 32);
      int above = 0;
      for (int j = 0; j < n; j += 4) {
        const uint4 q = *reinterpret_cast<const uint4*>(keys + j);
        above += (q.x > mine) + (q.y > mine) + (q.z > mine) + (q.w > mine);
      }
      a[above + atomicAdd(&taken[above], 1)] = x;
    }
    __syncthreads();
    return;
  }
  int p2 = 1;
  while (p2 < n) p2 <<= 1;
  for (int i = n + threadIdx.x; i < p2; i += SNT) a[i] = 0ull;     // below every pair
  __syncthreads();
  for (int size = 2; size <= p2; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = threadIdx.x; t < p2 / 2; t += SNT) {
        const int lo = ((t & ~(stride - 1)) << 1) | (t & (stride - 1)), hi = lo + stride;
        const bool down = (lo & size) == 0;
        const unsigned long long x = a[lo], y = a[hi];
        if ((x < y) == down) {
          a[lo] = y;
          a[hi] = x;
        }
      }
      __syncthreads();
    }
}

// running sums of w[0..n), n <= 4 SNT, in place (each entry's sum includes it); returns the sum of all.
// Thread t owns entries 4 t .. 4 t + 3; a wavefront scans its threads' sums with shuffles, the wavefronts'
// totals are added in order.
__device__ float scan_in_place(float* w, int n, float* s_wave) {
  const int t = threadIdx.x, lane = t & (TI_WAVE - 1), wave = t / TI_WAVE;
  float e[4], local = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    e[j] = 4 * t + j < n ? w[4 * t + j] : 0.f;
    local += e[j];
  }
  float run = local;
#pragma unroll
  for (int o = 1; o < TI_WAVE; o <<= 1) {
    const float v = __shfl_up(run, o, TI_WAVE);
    if (lane >= o) run += v;
  }
  const float upto = __shfl_up(run, 1, TI_WAVE);
  __syncthreads();
  if (lane == TI_WAVE - 1) s_wave[wave] = run;
  __syncthreads();
  float acc = 0.f, total = 0.f;
  for (int i = 0; i < SNT / TI_WAVE; ++i) {
    if (i == wave) acc = total;
    total += s_wave[i];
  }
  if (lane > 0) acc += upto;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    acc += e[j];
    if (4 * t + j < n) w[4 * t + j] = acc;
  }
  __syncthreads();
  return total;
}

// how many of the pairs a[0..n), sorted downwards by key, have a key of at least `key` (a[0] has)
__device__ int pairs_at_least(const unsigned long long* a, int n, uint32_t key, int* s_n) {
  for (int i = threadIdx.x; i < n; i += SNT)
    if ((uint32_t)(a[i] >> 32) >= key && (i + 1 == n || (uint32_t)(a[i + 1] >> 32) < key)) *s_n = i + 1;
  __syncthreads();
  const int m = *s_n;
  __syncthreads();
  return m;
}

// sorts the pairs a[0..n) of LDS, (key, ~index) with indices below V, by index; the result is in b as (~index, key).  A count by the
// indices' upper bits gives every pair its bucket's range, and within a bucket it counts the smaller ones.  n <= S_CAND; every thread
// calls it.  s_bins: 2 SNT counters.
__device__ void sort_by_index(const unsigned long long* a, unsigned long long* tmp, unsigned long long* b, int n, int V, int* s_bins, int* s_wave) {
  const int t = threadIdx.x, lane = t & (TI_WAVE - 1), wave = t / TI_WAVE;
  const int bits = max(0, 32 - __clz(V - 1) - 11);           // indices of a bucket: 2^bits, 2 SNT buckets
  static_assert(2 * SNT == 2048, "eleven bits of buckets");
  s_bins[2 * t] = s_bins[2 * t + 1] = 0;
  __syncthreads();
  for (int i = t; i < n; i += SNT) atomicAdd(&s_bins[~(uint32_t)a[i] >> bits], 1);
  __syncthreads();
  const int c0 = s_bins[2 * t], c1 = s_bins[2 * t + 1];
  int run = wave_prefix(c0 + c1);
  if (lane == TI_WAVE - 1) s_wave[wave] = run;
  __syncthreads();
  run -= c0 + c1;
#pragma unroll
  for (int w = 0; w < SNT / TI_WAVE; ++w)
    if (w < wave) run += s_wave[w];
  s_bins[2 * t] = run;                                       // where the bucket starts; after the next loop where it ends
  s_bins[2 * t + 1] = run + c0;
  __syncthreads();
  for (int i = t; i < n; i += SNT) tmp[atomicAdd(&s_bins[~(uint32_t)a[i] >> bits], 1)] = a[i];
  __syncthreads();
  for (int i = t; i < n; i += SNT) {
    const unsigned long long x = tmp[i];
    const uint32_t index = ~(uint32_t)x, bucket = index >> bits;
    const int lo = bucket ? s_bins[bucket - 1] : 0, hi = s_bins[bucket];
    int at = lo;
    for (int j = lo; j < hi; ++j) at += ~(uint32_t)tmp[j] < index ? 1 : 0;
    b[at] = (x << 32) | (x >> 32);
  }
  __syncthreads();
}

template <class Rows>
__global__ void __launch_bounds__(SNT)
sample_finish_kernel(const float* __restrict__ logits, Rows rows, int* __restrict__ out, const PartLeft* __restrict__ left,
                     const unsigned long long* __restrict__ pairs, int parts, int V) {
  __shared__ __attribute__((aligned(16))) unsigned long long s_pair[S_CAND], s_tmp[S_CAND];
  __shared__ float s_w[S_CAND];
  __shared__ __attribute__((aligned(16))) int s_bins[S_BINS];
  __shared__ float s_wave[SNT / TI_WAVE];
  __shared__ int s_iwave[SNT / TI_WAVE], s_res[4];
  __shared__ int s_n, s_at, s_m;
  __shared__ uint32_t s_max, s_from, s_over;
  const int r = blockIdx.x, t = threadIdx.x, lane = t & (TI_WAVE - 1), wave = t / TI_WAVE;
  const SampleRow want = rows.at(r);
  const int k = served_cut(want, V);
  if (k == 0) {
    sample_row_by_bisection(logits, want, out, V, r);
    return;
  }
  const float T = want.temp, p_keep = want.top_p, u = want.uni;
  // a wavefront takes parts wave, wave + 16, ...: f(eight pairs, or 0) by all lanes, eight loads under way at a time;
  // a part's first go out beside the load of its count (what lies beyond it is room of the part's, whatever it holds)
  const auto each = [&](auto f) {
    for (int b = wave; b < parts; b += SNT / TI_WAVE) {
      const unsigned long long* seg = pairs + ((size_t)r * parts + b) * S_CAND + lane;
      unsigned long long x[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = seg[TI_WAVE * j];
      const int n = left[(size_t)r * parts + b].pairs;
      for (int i0 = 0; i0 < n; i0 += 8 * TI_WAVE) {
        if (i0) {
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] = i0 + TI_WAVE * j + lane < n ? seg[i0 + TI_WAVE * j] : 0ull;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (i0 + TI_WAVE * j + lane >= n) x[j] = 0ull;
        f(x);
      }
    }
  };
  reinterpret_cast<int4*>(s_bins)[t] = make_int4(0, 0, 0, 0);
  static_assert(S_BINS == 4 * SNT, "four bins a thread");
  if (t == 0) s_at = 0x7fffffff, s_m = 0, s_max = 0, s_over = 0, s_from = 0xffffffffu;
  __syncthreads();
  for (int b = t; b < parts; b += SNT) {
    const PartLeft c = left[(size_t)r * parts + b];
    atomicMin(&s_from, c.share);
    if (c.over) atomicMax(&s_over, c.over);
  }
  __syncthreads();
  const uint32_t over = s_over;                    // keys up to here may be missing
  const uint32_t from = over ? max(s_from, over + 1) : s_from;
  // the pairs at or above `key`, in LDS as far as they fit
  const auto gather = [&](uint32_t key) {
    const uint32_t least = max(key, 1u);           // (0 is no pair)
    each([&](const unsigned long long* x) {
      int n = 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) n += (uint32_t)(x[j] >> 32) >= least ? 1 : 0;
      int at = next_places(&s_m, n);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if ((uint32_t)(x[j] >> 32) >= least) {
          if (at < S_CAND) s_tmp[at] = x[j];
          ++at;
        }
    });
    __syncthreads();
  };
  gather(from);
  int bin, above, in, taken = 0, need = k, shift = 32, got = s_m;      // taken: keys above the prefix
  uint32_t prefix = 0;
  const auto digit = [&](unsigned long long x) {
    const uint32_t key = (uint32_t)(x >> 32);
    if (x && (shift == 32 || (key >> shift) == prefix))
      atomicAdd(&s_bins[shift == 32 ? key >> (32 - S_BITS) : (key >> (shift - S_BITS2)) & (S_BINS2 - 1)], 1);
  };
  const auto next = [&]() {                        // the digit that `digit` has counted
    __syncthreads();
    if (shift == 32) {
      bin_of_kth<S_BINS, SNT>(s_bins, need, s_iwave, s_res, bin, above, in);
      prefix = bin;
      shift = 32 - S_BITS;
    } else {
      bin_of_kth<S_BINS2, SNT>(s_bins, need, s_iwave, s_res, bin, above, in);
      prefix = (prefix << S_BITS2) | (uint32_t)bin;
      shift -= S_BITS2;
    }
    taken += above;
    need -= above;
  };
  if (over && got < k) {                           // the row's cut is `over`, whose equals are too many
    sample_row_by_bisection(logits, want, out, V, r);
    return;
  }
  if (got == 0) {                                  // a row of NaN
    if (t == 0) out[r] = 0;
    return;
  }
  if (got > S_CAND) {                              // shares that are no guide: by digits over all pairs, until few enough are left
    do {
      each([&](const unsigned long long* x) {
        for (int j = 0; j < 8; ++j) digit(x[j]);
      });
      next();
    } while (taken + in > S_CAND && shift > 0);
    got = taken + in;
    if (got <= S_CAND) {
      if (t == 0) s_m = 0;
      __syncthreads();
      gather(prefix << shift);
    }
  }
  if (got > S_CAND) {
    sample_row_by_bisection(logits, want, out, V, r);
    return;
  }
  const int n = s_m;                               // the rest of the k-th key from these
  constexpr int PER = S_CAND / SNT;
  unsigned long long mine[PER];                    // pairs t, t + SNT, ...
#pragma unroll
  for (int j = 0; j < PER; ++j) mine[j] = t + SNT * j < n ? s_tmp[t + SNT * j] : 0ull;
  __syncthreads();
  if (t == 0) s_m = 0;
  __syncthreads();
  while (shift > 0) {
#pragma unroll
    for (int j = 0; j < PER; ++j)
      digit(mine[j]);
    next();
  }
  const uint32_t cut = prefix;
  if (!(T > 0.f)) {                                // of equal logits the lowest index
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (mine[j] && (uint32_t)(mine[j] >> 32) == cut) atomicMin(&s_at, (int)~(uint32_t)mine[j]);
    __syncthreads();
    if (t == 0) out[r] = s_at;
    return;
  }
  uint32_t largest = 0;
  int kept = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t key = (uint32_t)(mine[j] >> 32);
    kept += key >= cut ? 1 : 0;                    // (the cut is some number's key, not 0)
    largest = max(largest, key);
  }
  int place = next_places(&s_m, kept);
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if ((uint32_t)(mine[j] >> 32) >= cut) s_pair[place++] = mine[j];
  if (largest) atomicMax(&s_max, largest);
  __syncthreads();
  int m = s_m;
  const float mx = key_value(s_max);
  const float inv_t = 1.0f / T;
  if (p_keep < 1.0f) {
    sort_down(s_pair, m, s_tmp);
    for (int i = t; i < m; i += SNT) s_w[i] = expf((key_value((uint32_t)(s_pair[i] >> 32)) - mx) * inv_t);
    __syncthreads();
    const float need_mass = p_keep * scan_in_place(s_w, m, s_wave);
    for (int i = t; i < m; i += SNT)
      if (s_w[i] >= need_mass) atomicMin(&s_at, i);
    __syncthreads();
    const int j = s_at;                            // the first pair at which the mass from the top reaches it
    __syncthreads();
    if (t == 0) s_at = 0x7fffffff;
    if (j < m) m = pairs_at_least(s_pair, m, (uint32_t)(s_pair[j] >> 32), &s_n);   // its equals stay
    else __syncthreads();
  }
  // what is left, in the order of the indices
  sort_by_index(s_pair, s_tmp, s_pair, m, V, s_bins, s_iwave);
  for (int i = t; i < m; i += SNT) s_w[i] = expf((key_value((uint32_t)s_pair[i]) - mx) * inv_t);
  __syncthreads();
  const float target = u * scan_in_place(s_w, m, s_wave);
  for (int i = t; i < m; i += SNT)
    if (target < s_w[i]) atomicMin(&s_at, i);
  __syncthreads();
  if (t == 0) {
    const int at = s_at < m ? s_at : m - 1;        // rounding pushed the target past the end: the last one kept
    out[r] = (int)~(uint32_t)(s_pair[at] >> 32);
  }
}

// scratch: 2 * n_rows * 64 four-byte words, or nullptr (then one workgroup reads a whole row)
extern "C" int ti_argmax(const float* logits, int* out, void* scratch, int n_rows, int V, hipStream_t stream) {
  TI_REQUIRE(n_rows >= 0 && V > 0, "argmax: bad sizes rows=%d V=%d", n_rows, V);
  if (n_rows == 0) return 0;
  if (scratch && V >= 16384) {
    float* pv = (float*)scratch;
    int* pi = (int*)scratch + (size_t)n_rows * ARG_PARTS;
    argmax_part_kernel<<<dim3(n_rows, ARG_PARTS), 256, 0, stream>>>(logits, pv, pi, V);
    argmax_final_kernel<<<n_rows, 64, 0, stream>>>(pv, pi, out);
  } else {
    argmax_kernel<<<n_rows, SNT, 0, stream>>>(logits, out, V);
  }
  TI_LAUNCH_CHECK();
  return 0;
}

// The same greedy choice for callers that cannot allocate (code under HIP graph capture, tight
// serving loops, harnesses that forbid hipMalloc): the two-stage kernels above, with their partial
// results in a file-scope device array instead of a workspace argument.  Each GPU holds its own
// copy of the array (128 KiB) until the process ends; its address on a device is asked for once,
// with that device current, and kept.  Nothing in the array has to start at zero: the first stage
// writes every slot of the rows it is given before the second stage reads them.  Every call on a
// GPU shares that GPU's array, so calls that overlap on one GPU (two streams, two threads) race.
#define ARGMAX_STATIC_MAX_ROWS 256
static __device__ __align__(256) unsigned int scratch[2 * ARG_PARTS * ARGMAX_STATIC_MAX_ROWS];
#define ARGMAX_STATIC_MAX_DEVICES 64
static void* g_scratch_ptr[ARGMAX_STATIC_MAX_DEVICES];     // per device: where `scratch` lies there
static std::mutex g_scratch_mutex;

extern "C" int ti_argmax_static(const float* logits, int* out, int n_rows, int V, hipStream_t stream) {
  TI_REQUIRE(n_rows >= 0 && V > 0, "argmax_static: bad sizes rows=%d V=%d", n_rows, V);
  TI_REQUIRE(n_rows <= ARGMAX_STATIC_MAX_ROWS,
             "argmax_static: %d rows are more than the %d its fixed scratch array serves (use ti_argmax with a workspace)",
             n_rows, ARGMAX_STATIC_MAX_ROWS);
  if (n_rows == 0) return 0;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  TI_REQUIRE(e == hipSuccess && dev >= 0 && dev < ARGMAX_STATIC_MAX_DEVICES, "argmax_static: no current device (%s)",
             hipGetErrorString(e));
  void* ptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      TI_REQUIRE(e == hipSuccess && p, "argmax_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
      g_scratch_ptr[dev] = p;
    }
    ptr = g_scratch_ptr[dev];
  }
  float* pv = (float*)ptr;
  int* pi = (int*)ptr + (size_t)n_rows * ARG_PARTS;
  argmax_part_kernel<<<dim3(n_rows, ARG_PARTS), 256, 0, stream>>>(logits, pv, pi, V);
  argmax_final_kernel<<<n_rows, 64, 0, stream>>>(pv, pi, out);
  TI_LAUNCH_CHECK();
  return 0;
}

static int sample_parts(int V) { return std::max(1, (V + S_SPAN - 1) / S_SPAN); }
extern "C" long ti_sample_scratch_bytes(int n_rows, int V) { return (long)n_rows * sample_parts(V) * (S_CAND * 8 + (long)sizeof(PartLeft)); }

template <class Rows>
static void launch_sample(const float* logits, const Rows& rows, int* out, void* scratch, int n_rows, int V, hipStream_t stream) {
  if (!scratch) {
    sample_kernel<<<n_rows, SNT, 0, stream>>>(logits, rows, out, V);
    return;
  }
  const int parts = sample_parts(V), span = ((V + parts - 1) / parts + 3) & ~3;      // parts of a size: equal shares
  const dim3 grid(parts, n_rows);
  auto* pairs = (unsigned long long*)scratch;
  auto* left = (PartLeft*)(pairs + (size_t)n_rows * parts * S_CAND);
  if (V % 4 == 0 && ((uintptr_t)logits & 15) == 0)
    sample_part_kernel<true><<<grid, S_NT, 0, stream>>>(logits, rows, left, pairs, V, span);
  else
    sample_part_kernel<false><<<grid, S_NT, 0, stream>>>(logits, rows, left, pairs, V, span);
  sample_finish_kernel<<<n_rows, SNT, 0, stream>>>(logits, rows, out, left, pairs, parts, V);
}

// scratch: ti_sample_scratch_bytes(n_rows, V) bytes on a boundary of 8, or nullptr (then one workgroup walks a whole row)
extern "C" int ti_sample(const float* logits, const float* temp, const int* top_k, const float* top_p,
                         const float* uni, int* out, void* scratch, int n_rows, int V, hipStream_t stream) {
  TI_REQUIRE(n_rows >= 0 && V > 0, "sample: bad sizes rows=%d V=%d", n_rows, V);
  if (n_rows == 0) return 0;
  launch_sample(logits, RowsInMemory{temp, top_k, top_p, uni}, out, scratch, n_rows, V, stream);
  TI_LAUNCH_CHECK();
  return 0;
}

extern "C" int ti_sample_by_value(const float* logits, const float* temp, const int* top_k, const float* top_p,
                                  const float* uni, int* out, void* scratch, int n_rows, int V, hipStream_t stream) {
  TI_REQUIRE(n_rows >= 0 && V > 0, "sample: bad sizes rows=%d V=%d", n_rows, V);
  for (int r0 = 0; r0 < n_rows; r0 += S_VALUES) {
    const int n = std::min(S_VALUES, n_rows - r0);
    RowsByValue rows = {};
    for (int i = 0; i < n; ++i) rows.row[i] = SampleRow{temp[r0 + i], top_k[r0 + i], top_p[r0 + i], uni[r0 + i]};
    launch_sample(logits + (size_t)r0 * V, rows, out + r0, scratch, n, V, stream);
    TI_LAUNCH_CHECK();
  }
  return 0;
}
