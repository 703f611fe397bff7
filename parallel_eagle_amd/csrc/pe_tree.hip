// Tree masks, the greedy acceptance walk and in-place KV compaction.
//
// pe_tree_masks replaces tree_depths / tree_allow_mask / tree_position_ids
// (src/pe/masks.py:118-156) with one small kernel that turns `parents` into a
// per-node ancestor bitmask (bit u of bits[t] set iff u is t or an ancestor of t),
// the node depth and its RoPE position P + depth.
//
// pe_accept_tree is accept_tree_cached (src/pe/decode/verify.py:104-125): the
// argmax of the root logit and of every node row (first index among equal
// maxima, as torch.argmax), then the walk that descends into the first child (in
// node order) whose token equals the current argmax. It runs on the device so
// the host reads back one small result instead of syncing per depth.
//
// pe_kv_compact keeps rows [0, P) and the accepted path: row P + path[i] moves
// to P + i. path[i] >= i and path is increasing, so ascending i never
// overwrites a row still to be read; only |path| rows per layer/head move
// instead of index_select copying the whole cache (src/pe/target.py:194-201).

#include "pe_common.h"

#include <mutex>

namespace {

// Depth, position P + depth and ancestor bits of the T nodes of one tree
// (parents in the tree's own numbering), by the threads of one block.
__device__ void tree_masks_rows(const int32_t* __restrict__ parents, int T, int64_t P, uint64_t* __restrict__ bits,
                                int words, int64_t* __restrict__ positions, int32_t* __restrict__ depths,
                                int32_t* status) {
  for (int t = threadIdx.x; t < T; t += blockDim.x) {
    uint64_t b[PE_TREE_MAX_WORDS] = {0ull, 0ull, 0ull, 0ull};
    int depth = 0;
    bool bad = false;
    int a = t;
    // walk up: each step must go to a strictly smaller index
    for (int steps = 0; steps <= T; ++steps) {
      b[a >> 6] |= 1ull << (a & 63);
      const int p = parents[a];
      if (p == -1) break;
      if (p < -1 || p >= a) { bad = true; break; }
      a = p;
      ++depth;
    }
    if (bad && status) atomicOr(status, PE_ERR_TREE);
    for (int w = 0; w < words; ++w) bits[(int64_t)t * words + w] = bad ? 0ull : b[w];
    if (positions) positions[t] = P + depth;
    if (depths) depths[t] = depth;
  }
}

__global__ void tree_masks_kernel(const int32_t* __restrict__ parents, int T, int64_t P, uint64_t* __restrict__ bits,
                                  int words, int64_t* __restrict__ positions, int32_t* __restrict__ depths,
                                  int32_t* status) {
  tree_masks_rows(parents, T, P, bits, words, positions, depths, status);
}

// Batched trees: block b handles sequence b's rows [seq_row0[b], seq_row0[b+1]).
__global__ void tree_masks_batch_kernel(const int32_t* __restrict__ parents, const int32_t* __restrict__ seq_row0,
                                        const int64_t* __restrict__ seq_prefix, int max_rows,
                                        uint64_t* __restrict__ bits, int words, int64_t* __restrict__ positions,
                                        int32_t* __restrict__ depths, int32_t* status) {
  const int b = blockIdx.x;
  const int r0 = seq_row0[b], T = seq_row0[b + 1] - r0;
  if (T < 0 || T > max_rows || r0 < 0) {
    if (threadIdx.x == 0 && status) atomicOr(status, PE_ERR_TREE);
    return;
  }
  tree_masks_rows(parents + r0, T, seq_prefix[b], bits + (int64_t)r0 * words, words,
                  positions ? positions + r0 : nullptr, depths ? depths + r0 : nullptr, status);
}

__global__ void allow_dense_kernel(const uint64_t* __restrict__ bits, int T, int words, int64_t P,
                                   uint8_t* __restrict__ allow) {
  const int64_t n = P + T;
  const int64_t total = n * n;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
    const int64_t i = idx / n, j = idx % n;
    uint8_t v;
    if (i < P) {
      v = j <= i;
    } else if (j < P) {
      v = 1;
    } else {
      const int t = (int)(i - P), u = (int)(j - P);
      v = (bits[(int64_t)t * words + (u >> 6)] >> (u & 63)) & 1ull;
    }
    allow[idx] = v;
  }
}

template <int DT>
__global__ __launch_bounds__(256) void bias_to_bits_kernel(const typename Elem<DT>::T* __restrict__ bias, int64_t ld,
                                                           int T, int64_t P, float masked_below,
                                                           uint64_t* __restrict__ bits, int words, int32_t* status) {
  const int t = blockIdx.x;
  __shared__ unsigned long long w[PE_TREE_MAX_WORDS];
  if (threadIdx.x < PE_TREE_MAX_WORDS) w[threadIdx.x] = 0ull;
  __syncthreads();
  const int64_t S = P + T;
  int err = 0;
  for (int64_t j = threadIdx.x; j < S; j += blockDim.x) {
    const float v = Elem<DT>::load(bias, (int64_t)t * ld + j);
    const bool allowed = v == 0.f;
    const bool masked = v <= masked_below;
    if (!allowed && !masked) err = 1;
    if (j < P) {
      if (!allowed) err = 1;
    } else if (allowed) {
      const int u = (int)(j - P);
      atomicOr(&w[u >> 6], 1ull << (u & 63));
    }
  }
  if (err && status) atomicOr(status, PE_ERR_MASK);
  __syncthreads();
  if (threadIdx.x < words) bits[(int64_t)t * words + threadIdx.x] = w[threadIdx.x];
}

// Row argmax with torch.argmax's semantics: the largest value, a NaN beats
// every number, and among equal maxima (or NaNs) the lowest index wins.
constexpr int kArgThreads = 1024;

// The largest element of a thread's share of a row: 16-byte vectors t, t +
// kArgThreads, ... in increasing index order, then single elements past the
// last whole vector (all of them when the row is not 16-byte aligned). Returns
// the first element of the largest arg_key (bi < 0: none).
//
// 16-bit rows are compared two elements at a time: (magnitude ^ sign) - sign
// orders them as signed 16-bit integers with -0 equal to +0, so a vector costs
// 3 packed operations per element pair more than its load, instead of a
// conversion, a NaN test and a 32-bit key per element; the best vector is kept
// whole and searched once at the end. NaNs (a magnitude past infinity's) are
// only detected: `nan` then tells the caller that the result counts numbers
// only (fp32 keys hold them). kArgVec vectors (a 152064-element row's whole
// share) are in flight at a time; one workgroup reads a row, so its CU's load
// rate is the bound (26 rows of 152064 bf16 elements, replayed: 16.9 us with
// 32-bit keys and 8 vectors in flight, 9.9 us like this).
typedef short s16x2_t __attribute__((ext_vector_type(2)));
constexpr int kArgVec = 10;

template <int DT>
__device__ __forceinline__ void share_best(const typename Elem<DT>::T* __restrict__ x, int64_t V, int64_t nvec,
                                           uint32_t& bk, int& bi, bool& nan) {
  typedef typename Elem<DT>::T T;
  constexpr int kPer = 16 / sizeof(T);
  bk = 0;  // below every real key
  bi = -1;
  nan = false;
  if constexpr (DT == PE_DTYPE_F32) {
    for (int64_t v0 = 0; v0 < nvec; v0 += (int64_t)kArgVec * kArgThreads) {
      u32x4_t buf[kArgVec];
#pragma unroll
      for (int k = 0; k < kArgVec; ++k) {
        const int64_t vi = v0 + (int64_t)k * kArgThreads + threadIdx.x;
        if (vi < nvec) buf[k] = *(const u32x4_t*)(x + vi * kPer);
      }
#pragma unroll
      for (int k = 0; k < kArgVec; ++k) {
        const int64_t vi = v0 + (int64_t)k * kArgThreads + threadIdx.x;
        if (vi < nvec) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const uint32_t key = arg_key(__uint_as_float(buf[k][j]));
            if (key > bk) {
              bk = key;
              bi = (int)(vi * kPer + j);
            }
          }
        }
      }
    }
  } else {
    constexpr uint32_t kInf = DT == PE_DTYPE_BF16 ? 0x7f80u : 0x7c00u;
    int best = -32768, bv = -1;  // below every number's key
    u32x4_t bw = {0, 0, 0, 0};
    uint32_t mag = 0;  // packed maximum of the magnitudes
    typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
    auto key2 = [](uint32_t w) -> s16x2_t {
      const s16x2_t sg = __builtin_bit_cast(s16x2_t, w) >> 15;
      return (__builtin_bit_cast(s16x2_t, w & 0x7fff7fffu) ^ sg) - sg;
    };
    for (int64_t v0 = 0; v0 < nvec; v0 += (int64_t)kArgVec * kArgThreads) {
      u32x4_t buf[kArgVec];
#pragma unroll
      for (int k = 0; k < kArgVec; ++k) {
        const int64_t vi = v0 + (int64_t)k * kArgThreads + threadIdx.x;
        if (vi < nvec) buf[k] = *(const u32x4_t*)(x + vi * kPer);
      }
#pragma unroll
      for (int k = 0; k < kArgVec; ++k) {
        const int64_t vi = v0 + (int64_t)k * kArgThreads + threadIdx.x;
        if (vi < nvec) {
          s16x2_t m = key2(buf[k][0]);
#pragma unroll
          for (int j = 1; j < 4; ++j) m = __builtin_elementwise_max(m, key2(buf[k][j]));
#pragma unroll
          for (int j = 0; j < 4; ++j)
            mag = __builtin_bit_cast(
                uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, mag),
                                                    __builtin_bit_cast(u16x2_t, buf[k][j] & 0x7fff7fffu)));
          const int top = max((int)m[0], (int)m[1]);
          if (top > best) {
            best = top;
            bv = (int)vi;
            bw = buf[k];
          }
        }
      }
    }
    nan = (mag & 0xffffu) > kInf || (mag >> 16) > kInf;
    if (bv >= 0) {
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        const s16x2_t m = key2(bw[j]);
        if (m[1] == best) bi = bv * kPer + 2 * j + 1;
        if (m[0] == best) bi = bv * kPer + 2 * j;
      }
      // the winner's own 32-bit key
      uint32_t e = bw[0];
#pragma unroll
      for (int j = 1; j < 4; ++j) e = ((bi >> 1) & 3) == j ? bw[j] : e;
      const uint16_t bits = (uint16_t)((bi & 1) ? e >> 16 : e);
      bk = arg_key(Elem<DT>::load(&bits, 0));
    }
  }
  for (int64_t i = nvec * kPer + threadIdx.x; i < V; i += kArgThreads) {
    const float v = Elem<DT>::load(x, i);
    if constexpr (DT != PE_DTYPE_F32) nan |= v != v;
    const uint32_t key = arg_key(v);
    if (key > bk) {
      bk = key;
      bi = (int)i;
    }
  }
  if constexpr (DT == PE_DTYPE_F32) nan = bk == 0xFFFFFFFFu;  // a NaN's key, the largest
}

// Whole 16-byte vectors of a row (none when it is not 16-byte aligned).
template <int DT>
__device__ __forceinline__ int64_t row_vectors(const typename Elem<DT>::T* x, int64_t V) {
  return (((uintptr_t)x) & 15) == 0 ? V / (16 / (int64_t)sizeof(typename Elem<DT>::T)) : 0;
}

// One block of kArgThreads per row: every thread's best, then the block's with
// (key descending, index ascending). A thread whose 16-bit share holds a NaN
// goes through its vectors again for the first one (every NaN has the largest
// key); the fp32 search and the single elements have its key already.
template <int DT>
__device__ int row_argmax(const typename Elem<DT>::T* __restrict__ x, int64_t V, int32_t* out) {
  uint32_t bk;
  int bi;
  bool nan;
  const int64_t nvec = row_vectors<DT>(x, V);
  share_best<DT>(x, V, nvec, bk, bi, nan);
  if constexpr (DT != PE_DTYPE_F32) {
    if (nan) {
      constexpr int kPer = 8;
      bool found = false;
      for (int64_t vi = threadIdx.x; vi < nvec && !found; vi += kArgThreads)
        for (int j = 0; j < kPer && !found; ++j) {
          const float v = Elem<DT>::load(x, vi * kPer + j);
          if (v != v) {
            bk = arg_key(v);
            bi = (int)(vi * kPer + j);
            found = true;
          }
        }
    }
  }
  auto better = [](uint32_t k2, int i2, uint32_t k1, int i1) {  // (k2, i2) beats (k1, i1)
    if (i2 < 0) return false;
    if (i1 < 0) return true;
    return k2 > k1 || (k2 == k1 && i2 < i1);
  };
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t k2 = __shfl_xor(bk, o, 64);
    const int i2 = __shfl_xor(bi, o, 64);
    if (better(k2, i2, bk, bi)) {
      bk = k2;
      bi = i2;
    }
  }
  __shared__ uint32_t wk[kArgThreads / 64];
  __shared__ int wi[kArgThreads / 64];
  if ((threadIdx.x & 63) == 0) {
    wk[threadIdx.x >> 6] = bk;
    wi[threadIdx.x >> 6] = bi;
  }
  __syncthreads();
  int i1 = -1;
  if (threadIdx.x == 0) {
    uint32_t k1 = wk[0];
    i1 = wi[0];
    for (int w = 1; w < kArgThreads / 64; ++w)
      if (better(wk[w], wi[w], k1, i1)) {
        k1 = wk[w];
        i1 = wi[w];
      }
    if (out) *out = i1;
  }
  return i1;
}

// Row argmax from per-column-group keys (arg_key64, written by the lm_head
// GEMM's argmax epilogue): the largest key and its column; the result is
// valid in thread 0.
__device__ int row_argmax_keys(const uint64_t* __restrict__ keys, int groups) {
  uint64_t best = 0;  // below every real key
  for (int i = threadIdx.x; i < groups; i += kArgThreads) {
    const uint64_t k = keys[i];
    best = k > best ? k : best;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t k = shfl_xor_u64(best, o);
    best = k > best ? k : best;
  }
  __shared__ uint64_t wk[kArgThreads / 64];
  if ((threadIdx.x & 63) == 0) wk[threadIdx.x >> 6] = best;
  __syncthreads();
  int idx = -1;
  if (threadIdx.x == 0) {
    uint64_t b = wk[0];
    for (int w = 1; w < kArgThreads / 64; ++w) b = wk[w] > b ? wk[w] : b;
    idx = b ? (int)(0xFFFFFFFFu - (uint32_t)b) : -1;
  }
  return idx;
}

template <int DT>
__global__ __launch_bounds__(kArgThreads) void argmax_rows_kernel(const typename Elem<DT>::T* __restrict__ x,
                                                                  int64_t ld, int64_t V, int32_t* __restrict__ out) {
  row_argmax<DT>(x + (int64_t)blockIdx.x * ld, V, out + blockIdx.x);
}

// One launch does the whole acceptance. Block r finds the argmax of row r
// (row 0 = root logit, rows 1..T = node logits) and publishes it in
// work[1 + r]; the last block to count itself on work[0] (every row's argmax
// is then visible) resets that counter and walks the tree. The counter sits
// at index 0 whatever T is, so one scratch buffer serves calls of any size. The walk stages every
// node's argmax, parent and token in LDS; one wave then follows the greedy
// path, each step a ballot over the nodes for the first child of the current
// node whose token equals the current truth (at most kWalkMax nodes).
constexpr int kWalkMax = 64 * PE_TREE_MAX_WORDS;

// Batched trees (seq_row0 non-null): blockIdx.y = sequence b, whose root row
// is root + b * ld_root, node rows start at row seq_row0[b], scratch at
// work + b * (T + 2) and result at out + b * (T + 2), T being the largest
// tree; blocks past the sequence's own node count leave at once.
template <int DT>
__global__ __launch_bounds__(kArgThreads) void accept_kernel(const typename Elem<DT>::T* __restrict__ root,
                                                             int64_t ld_root,
                                                             const typename Elem<DT>::T* __restrict__ nodes,
                                                             int64_t ld, int64_t V, int32_t* __restrict__ work,
                                                             int T, const int32_t* __restrict__ seq_row0,
                                                             const int64_t* __restrict__ tokens,
                                                             const int32_t* __restrict__ parents,
                                                             int32_t* __restrict__ out,
                                                             const uint64_t* __restrict__ node_keys, int groups) {
  if (seq_row0) {
    const int b = blockIdx.y, r0 = seq_row0[b];
    root += b * ld_root;
    nodes += (int64_t)r0 * ld;
    work += (int64_t)b * (T + 2);
    out += (int64_t)b * (T + 2);
    tokens += r0;
    parents += r0;
    T = min(max(seq_row0[b + 1] - r0, 0), T);
    if ((int)blockIdx.x > T) return;
  }
  int32_t* const counter = work;
  int32_t* const amax = work + 1;
  const int r = blockIdx.x;
  const typename Elem<DT>::T* x = (r == 0) ? root : nodes + (int64_t)(r - 1) * ld;
  // node rows from the lm_head's argmax keys when the caller has them
  const int best = (node_keys && r > 0) ? row_argmax_keys(node_keys + (int64_t)(r - 1) * groups, groups)
                                        : row_argmax<DT>(x, V, nullptr);
  __shared__ int s_last;
  if (threadIdx.x == 0) {
    // The row's argmax is stored at agent scope (past this die's L2) and
    // acknowledged before the block counts itself, and the last block reads
    // every argmax at agent scope, so it sees all of them. (An acquire-release
    // count would write back and invalidate the whole L2 in every block.)
    __hip_atomic_store(amax + r, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = old == T;
    if (old == T) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  __shared__ int32_t s_amax[kWalkMax + 1], s_par[kWalkMax];
  __shared__ int64_t s_tok[kWalkMax];
  const int n = min(T, kWalkMax);
  for (int t = threadIdx.x; t <= n; t += kArgThreads)
    s_amax[t] = __hip_atomic_load(amax + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int t = threadIdx.x; t < n; t += kArgThreads) {
    s_par[t] = parents[t];
    s_tok[t] = tokens[t];
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x;
  int cur = -1, len = 0;
  int truth = s_amax[0];
  for (;;) {
    int nxt = -1;
    for (int base = 0; base < n; base += 64) {
      const int t = base + lane;
      const bool hit = t < n && s_par[t] == cur && s_tok[t] == (int64_t)truth;
      const uint64_t b = __ballot(hit);
      if (b) {
        nxt = base + (int)__builtin_ctzll(b);
        break;
      }
    }
    if (nxt < 0 || len >= n) break;
    if (lane == 0) out[2 + len] = nxt;
    ++len;
    cur = nxt;
    truth = s_amax[1 + nxt];
  }
  if (lane == 0) {
    out[0] = len;
    out[1] = truth;
  }
}

// grid: (L * nkv, 2 for K/V, batch); threads over 16-byte chunks of a row.
// Batched (seq_prefix non-null): sequence b = blockIdx.z has its cache at
// seq_bytes * b, its prefix seq_prefix[b] and its result at res + b * res_stride.
__global__ void kv_compact_kernel(uint8_t* __restrict__ kc, uint8_t* __restrict__ vc, int64_t cap, int64_t row_bytes,
                                  int64_t P, const int32_t* __restrict__ res, const int64_t* __restrict__ seq_prefix,
                                  int64_t seq_bytes, int res_stride) {
  if (seq_prefix) {
    const int b = blockIdx.z;
    P = seq_prefix[b];
    res += (int64_t)b * res_stride;
    kc += b * seq_bytes;
    vc += b * seq_bytes;
  }
  const int len = res[0];
  uint8_t* base = (blockIdx.y == 0 ? kc : vc) + (int64_t)blockIdx.x * cap * row_bytes;
  const int64_t nchunk = row_bytes / 16;
  for (int i = 0; i < len; ++i) {
    const int src = res[2 + i];
    if (src == i || src < 0 || P + src >= cap || P + i >= cap) continue;
    const uint4* s = (const uint4*)(base + (P + src) * row_bytes);
    uint4* d = (uint4*)(base + (P + i) * row_bytes);
    for (int64_t c = threadIdx.x; c < nchunk; c += blockDim.x) d[c] = s[c];
    __syncthreads();
  }
}

// validate keep (strictly increasing, < cap) and find the first i with keep[i] != i
__global__ void kv_keep_check_kernel(const int64_t* __restrict__ keep, int64_t n, int64_t cap,
                                     int64_t* __restrict__ first, int32_t* status) {
  __shared__ unsigned long long fmin;
  if (threadIdx.x == 0) fmin = (unsigned long long)n;
  __syncthreads();
  int err = 0;
  for (int64_t i = threadIdx.x; i < n; i += blockDim.x) {
    const int64_t k = keep[i];
    if (k < 0 || k >= cap || (i > 0 && keep[i - 1] >= k)) err = 1;
    if (k != i) atomicMin(&fmin, (unsigned long long)i);
  }
  if (err && status) atomicOr(status, PE_ERR_INDEX);
  __syncthreads();
  if (threadIdx.x == 0) *first = err ? n : (int64_t)fmin;
}

__global__ void kv_gather_kernel(uint8_t* __restrict__ kc, uint8_t* __restrict__ vc, int64_t cap, int64_t row_bytes,
                                 const int64_t* __restrict__ keep, int64_t n, const int64_t* __restrict__ first) {
  const int64_t f = *first;
  uint8_t* base = (blockIdx.y == 0 ? kc : vc) + (int64_t)blockIdx.x * cap * row_bytes;
  const int64_t nchunk = row_bytes / 16;
  for (int64_t i = f; i < n; ++i) {
    const int64_t src = keep[i];
    if (src == i) continue;
    const uint4* s = (const uint4*)(base + src * row_bytes);
    uint4* d = (uint4*)(base + i * row_bytes);
    for (int64_t c = threadIdx.x; c < nchunk; c += blockDim.x) d[c] = s[c];
    __syncthreads();
  }
}

// Beam tree proposal (propose_tree, src/pe/decode/tree.py:34-55) in three
// launches (two for short rows, see kShortRow).
//   * draft_topk_kernel: one block per depth row. Every thread finds the best
//     element of its share of the row; one wave then takes the row's top c_d
//     tokens in (value descending, index ascending) order: the best of the
//     1024 shares, whose owner's share (about V / 1024 elements, read across
//     the wave) is searched for its next best. Streaming the row again for
//     every token took 199 us for five rows of 152064 at five tokens each;
//     this takes 20 us (a row is one CU's 304 KB), the sums below 8.
//   * draft_expsum_kernel: the row's sum of exp(x - max) in fp32. The sum keeps
//     the order of 1024 strided partial sums (element i in partial i % 1024,
//     increasing i), the partials of 64 neighbours added by a butterfly: block
//     s owns the 64 partials of slice s and computes their exponentials in
//     parallel, one wave adds them up in order. (Sums of equal logits over
//     different rows tie up to these roundings, so the order decides trees.)
//   * beam_kernel: logarithms of the rows' sums (slices in order), the
//     candidates' log-probabilities (x - max) - log(sum), then one block walks
//     the depths; candidate (parent p, rank j in the row) scores cum[p] +
//     lp[j] in float64, and its position in the stable descending order of the
//     candidate list (parent-major, as the reference builds it) is counted
//     directly: j for its own parent, plus, for every other parent, the
//     candidates that score higher (or equal, for parents before it), found by
//     binary search since each parent's scores do not increase with j.
constexpr int kBeamThreads = 256;
constexpr int kSlices = kArgThreads / 64;  // slices of 64 partial sums
constexpr int kExpTile = 128;              // elements of a partial sum staged at a time
constexpr int kExpThreads = 512;
// Up to this row length draft_topk_kernel takes the sums itself, one thread per
// partial sum, and the second launch is left out: five rows at two tokens each
// take 15.5 us of 2048 elements with one launch less and 17.0 with it, 17.9 and
// 18.0 of 16384, 20.8 and 19.0 of 32000.
constexpr int64_t kShortRow = 16384;
static_assert(kSlices <= PE_PROPOSE_MAX_WIDTH, "a row's slice sums are staged in its log-probability scratch");

struct BeamShape {
  int k;
  int width[PE_PROPOSE_MAX_DEPTH];  // nodes kept at depth d
  int cand[PE_PROPOSE_MAX_DEPTH];   // candidates per parent: min(top_k, width[d])
};

// (k2, i2) before (k1, i1) in the order key descending, index ascending; i < 0 is "none"
__device__ __forceinline__ bool key_before(uint32_t k2, int i2, uint32_t k1, int i1) {
  if (i2 < 0) return false;
  if (i1 < 0) return true;
  return k2 > k1 || (k2 == k1 && i2 < i1);
}

// wave-wide (key, index) reduction; every lane gets the result
__device__ __forceinline__ void wave_best(uint32_t& bk, int& bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t k2 = __shfl_xor(bk, o, 64);
    const int i2 = __shfl_xor(bi, o, 64);
    if (key_before(k2, i2, bk, bi)) {
      bk = k2;
      bi = i2;
    }
  }
}

// A row with a NaN, without a finite value or with +inf flags PE_ERR_VALUE and
// leaves token -1 in its first place.
template <int DT>
__global__ __launch_bounds__(kArgThreads) void draft_topk_kernel(const typename Elem<DT>::T* __restrict__ logits,
                                                                 int64_t ld, int64_t V, BeamShape bs,
                                                                 int32_t* __restrict__ tok_out,
                                                                 float* __restrict__ sums, int32_t* status) {
  const int d = blockIdx.x;
  const typename Elem<DT>::T* x = logits + (int64_t)d * ld;
  constexpr int kPer = 16 / sizeof(typename Elem<DT>::T);
  const int64_t nvec = row_vectors<DT>(x, V);
  __shared__ uint32_t s_key[kArgThreads];
  __shared__ int s_idx[kArgThreads];
  uint32_t bk;
  int bi;
  bool nan;
  share_best<DT>(x, V, nvec, bk, bi, nan);
  s_key[threadIdx.x] = bk;
  s_idx[threadIdx.x] = bi;
  nan = __syncthreads_or(nan);
  const int lane = threadIdx.x & 63;
  int32_t* out = tok_out + d * PE_PROPOSE_MAX_WIDTH;
  // the best of this lane's 16 shares (lane, lane + 64, ...)
  uint32_t lk = 0;
  int li = -1;
  auto scan = [&]() {
    lk = 0;
    li = -1;
#pragma unroll
    for (int q = 0; q < kArgThreads / 64; ++q) {
      const uint32_t k2 = s_key[lane + 64 * q];
      const int i2 = s_idx[lane + 64 * q];
      if (key_before(k2, i2, lk, li)) {
        lk = k2;
        li = i2;
      }
    }
  };
  uint32_t pk = 0;
  int pi = -1;
  if (threadIdx.x < 64) {
    scan();
    pk = lk;
    pi = li;
    wave_best(pk, pi);
  }
  if (sums) {
    // a short row: partial sum t by thread t, slice w by wave w
    __shared__ int s_first;
    if (threadIdx.x == 0) s_first = pi;
    __syncthreads();
    const float mx = Elem<DT>::load(x, s_first);
    float s = 0.f;
    for (int64_t i = threadIdx.x; i < V; i += kArgThreads) s += expf(Elem<DT>::load(x, i) - mx);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) sums[d * PE_PROPOSE_MAX_WIDTH + (threadIdx.x >> 6)] = s;
  }
  if (threadIdx.x >= 64) return;
  const int c = bs.cand[d];
  for (int j = 0; j < c; ++j) {
    if (j > 0) {
      pk = lk;
      pi = li;
      wave_best(pk, pi);
    } else {
      const float mx = Elem<DT>::load(x, pi);
      if (nan || !(mx > -INFINITY) || mx == INFINITY) {
        if (lane == 0) {
          out[0] = -1;
          if (status) atomicOr(status, PE_ERR_VALUE);
        }
        return;
      }
    }
    if (lane == 0) out[j] = pi;
    if (j + 1 == c) break;
    // the owner's next best after (pk, pi)
    const bool in_vec = pi < nvec * kPer;
    const int owner = (int)((in_vec ? pi / kPer : pi - nvec * kPer) % kArgThreads);
    const int64_t nv = nvec > owner ? (nvec - owner + kArgThreads - 1) / kArgThreads : 0;
    uint32_t k1 = 0;
    int i1 = -1;
    auto offer = [&](int64_t i) {
      const uint32_t key = arg_key(Elem<DT>::load(x, i));
      if (key_before(pk, pi, key, (int)i) && key_before(key, (int)i, k1, i1)) {
        k1 = key;
        i1 = (int)i;
      }
    };
#pragma unroll 4
    for (int64_t q = lane; q < nv * kPer; q += 64) offer((owner + (q / kPer) * kArgThreads) * kPer + q % kPer);
    for (int64_t i = nvec * kPer + owner + (int64_t)lane * kArgThreads; i < V; i += 64 * kArgThreads) offer(i);
    wave_best(k1, i1);
    if (lane == (owner & 63)) {
      s_key[owner] = k1;
      s_idx[owner] = i1;
      scan();
    }
  }
}

// grid (kSlices, depth rows)
template <int DT>
__global__ __launch_bounds__(kExpThreads) void draft_expsum_kernel(const typename Elem<DT>::T* __restrict__ logits,
                                                                   int64_t ld, int64_t V,
                                                                   const int32_t* __restrict__ tok,
                                                                   float* __restrict__ sums) {
  const int slice = blockIdx.x, d = blockIdx.y;
  const typename Elem<DT>::T* x = logits + (int64_t)d * ld;
  const int first = tok[d * PE_PROPOSE_MAX_WIDTH];
  if (first < 0) return;  // an invalid row (the whole block leaves)
  const float mx = Elem<DT>::load(x, first);
  __shared__ float e[kExpTile][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t part = slice * 64 + lane;
  const int64_t n = part < V ? (V - part + kArgThreads - 1) / kArgThreads : 0;  // this lane's elements
  const int64_t most = slice * 64 < V ? (V - slice * 64 + kArgThreads - 1) / kArgThreads : 0;
  float s = 0.f;
  for (int64_t j0 = 0; j0 < most; j0 += kExpTile) {
    const int64_t j1 = min(most, j0 + kExpTile);
#pragma unroll 4
    for (int64_t j = j0 + wave; j < j1; j += kExpThreads / 64)
      if (j < n) e[j - j0][lane] = expf(Elem<DT>::load(x, part + j * kArgThreads) - mx);
    __syncthreads();
    if (wave == 0) {
      const int64_t m = min(n, j1) - j0;
#pragma unroll 8
      for (int64_t j = 0; j < m; ++j) s += e[j][lane];
    }
    __syncthreads();
  }
  if (wave != 0) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) sums[d * PE_PROPOSE_MAX_WIDTH + slice] = s;
}

// lp: the rows' slice sums on entry, their candidates' log-probabilities on return.
template <int DT>
__global__ __launch_bounds__(kBeamThreads) void beam_kernel(const typename Elem<DT>::T* __restrict__ logits,
                                                            int64_t ld, BeamShape bs, float* __restrict__ lp,
                                                            const int32_t* __restrict__ tok,
                                                            int64_t* __restrict__ node_tokens,
                                                            int32_t* __restrict__ parents, const int32_t* status) {
  __shared__ float s_sum[PE_PROPOSE_MAX_DEPTH][kSlices];
  __shared__ float s_lp[PE_PROPOSE_MAX_DEPTH][PE_PROPOSE_MAX_WIDTH];
  __shared__ int s_tok[PE_PROPOSE_MAX_DEPTH][PE_PROPOSE_MAX_WIDTH];
  __shared__ double cum[PE_PROPOSE_MAX_WIDTH], ncum[PE_PROPOSE_MAX_WIDTH], row[PE_PROPOSE_MAX_WIDTH];
  __shared__ int node[PE_PROPOSE_MAX_WIDTH];
  int bad = status && (*status & PE_ERR_VALUE);
  for (int i = threadIdx.x; i < bs.k * PE_PROPOSE_MAX_WIDTH; i += kBeamThreads) {
    const int d = i / PE_PROPOSE_MAX_WIDTH, j = i % PE_PROPOSE_MAX_WIDTH;
    if (j < kSlices) s_sum[d][j] = lp[i];
    if (j < bs.cand[d]) s_tok[d][j] = tok[i];
    if (j == 0) bad |= tok[i] < 0;
  }
  if (__syncthreads_or(bad)) return;
  for (int i = threadIdx.x; i < bs.k * PE_PROPOSE_MAX_WIDTH; i += kBeamThreads) {
    const int d = i / PE_PROPOSE_MAX_WIDTH, j = i % PE_PROPOSE_MAX_WIDTH;
    if (j >= bs.cand[d]) continue;
    const typename Elem<DT>::T* x = logits + (int64_t)d * ld;
    const float mx = Elem<DT>::load(x, s_tok[d][0]);
    float s = 0.f;
    for (int w = 0; w < kSlices; ++w) s += s_sum[d][w];
    const float v = (Elem<DT>::load(x, s_tok[d][j]) - mx) - logf(s);
    s_lp[d][j] = v;
    lp[i] = v;
  }
  int nb = 1, base = 0;
  if (threadIdx.x == 0) {
    cum[0] = 0.0;
    node[0] = -1;
  }
  __syncthreads();
  for (int d = 0; d < bs.k; ++d) {
    const int c = bs.cand[d];
    const int n = nb * c;
    const int kept = min(bs.width[d], n);
    if (threadIdx.x < c) row[threadIdx.x] = (double)s_lp[d][threadIdx.x];
    __syncthreads();
    for (int q = threadIdx.x; q < n; q += kBeamThreads) {
      const int p = q / c, j = q - p * c;
      const double sc = cum[p] + row[j];
      int r = j;
      for (int p2 = 0; p2 < nb && r < kept; ++p2) {
        if (p2 == p) continue;
        // count j2 with cum[p2] + row[j2] > sc (>= sc for parents listed before p)
        int lo = 0, hi = c;
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          const double s2 = cum[p2] + row[mid];
          if (p2 < p ? s2 >= sc : s2 > sc)
            lo = mid + 1;
          else
            hi = mid;
        }
        r += lo;
      }
      if (r < kept) {
        ncum[r] = sc;
        node_tokens[base + r] = s_tok[d][j];
        parents[base + r] = node[p];
      }
    }
    __syncthreads();
    if (threadIdx.x < kept) {
      cum[threadIdx.x] = ncum[threadIdx.x];
      node[threadIdx.x] = base + threadIdx.x;
    }
    __syncthreads();
    base += kept;
    nb = kept;
  }
}

int esize(int dtype) { return dtype == PE_DTYPE_F32 ? 4 : 2; }

}  // namespace

extern "C" int pe_tree_masks(const int32_t* parents, int T, int64_t P, uint64_t* bits, int words, int64_t* positions,
                             int32_t* depths, int32_t* status, void* stream) {
  if (!parents || !bits || T <= 0 || P < 0 || words <= 0 || words > PE_TREE_MAX_WORDS) return PE_ERR_ARG;
  if (T > 64 * words) return PE_ERR_TREE;
  tree_masks_kernel<<<1, 256, 0, (hipStream_t)stream>>>(parents, T, P, bits, words, positions, depths, status);
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_tree_masks_batch(const int32_t* parents, const int32_t* seq_row0, const int64_t* seq_prefix, int batch,
                                   int max_seq_rows, uint64_t* bits, int words, int64_t* positions, int32_t* depths,
                                   int32_t* status, void* stream) {
  if (!parents || !seq_row0 || !seq_prefix || !bits || batch <= 0 || max_seq_rows <= 0 || words <= 0 ||
      words > PE_TREE_MAX_WORDS)
    return PE_ERR_ARG;
  if (max_seq_rows > 64 * words) return PE_ERR_TREE;
  tree_masks_batch_kernel<<<batch, 256, 0, (hipStream_t)stream>>>(parents, seq_row0, seq_prefix, max_seq_rows, bits,
                                                                   words, positions, depths, status);
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_tree_allow_dense(const uint64_t* bits, int T, int words, int64_t P, uint8_t* allow, void* stream) {
  if (!bits || !allow || T <= 0 || P < 0 || words <= 0 || words > PE_TREE_MAX_WORDS || T > 64 * words)
    return PE_ERR_ARG;
  const int64_t n = P + T;
  int64_t g = (n * n + 255) / 256;
  if (g > 65536) g = 65536;
  allow_dense_kernel<<<(int)g, 256, 0, (hipStream_t)stream>>>(bits, T, words, P, allow);
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_bias_to_bits(const void* bias, int64_t ld_bias, int dtype, int T, int64_t P, uint64_t* bits,
                               int words, int32_t* status, void* stream) {
  if (!bias || !bits || T <= 0 || P < 0 || words <= 0 || words > PE_TREE_MAX_WORDS) return PE_ERR_ARG;
  if (T > 64 * words) return PE_ERR_TREE;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case PE_DTYPE_F32:
      bias_to_bits_kernel<PE_DTYPE_F32><<<T, 256, 0, st>>>((const float*)bias, ld_bias, T, P, -1.7014117e38f, bits,
                                                           words, status);
      break;
    case PE_DTYPE_BF16:
      bias_to_bits_kernel<PE_DTYPE_BF16><<<T, 256, 0, st>>>((const uint16_t*)bias, ld_bias, T, P, -1.69e38f, bits,
                                                            words, status);
      break;
    case PE_DTYPE_F16:
      bias_to_bits_kernel<PE_DTYPE_F16><<<T, 256, 0, st>>>((const uint16_t*)bias, ld_bias, T, P, -32752.f, bits,
                                                           words, status);
      break;
    default:
      return PE_ERR_ARG;
  }
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_argmax_rows(const void* x, int64_t ld, int rows, int64_t V, int dtype, int32_t* out_idx,
                              void* stream) {
  if (!x || !out_idx || rows <= 0 || V <= 0) return PE_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  switch (dtype) {
    case PE_DTYPE_F32: argmax_rows_kernel<PE_DTYPE_F32><<<rows, kArgThreads, 0, st>>>((const float*)x, ld, V, out_idx); break;
    case PE_DTYPE_BF16: argmax_rows_kernel<PE_DTYPE_BF16><<<rows, kArgThreads, 0, st>>>((const uint16_t*)x, ld, V, out_idx); break;
    case PE_DTYPE_F16: argmax_rows_kernel<PE_DTYPE_F16><<<rows, kArgThreads, 0, st>>>((const uint16_t*)x, ld, V, out_idx); break;
    default: return PE_ERR_ARG;
  }
  PE_CHECK_LAUNCH();
  return PE_OK;
}

namespace {

// batch == 0: one tree of T nodes; batch >= 1: seq_row0 [batch + 1] splits the
// node rows into trees of at most T nodes each.
int launch_accept(const void* root_logit, int64_t ld_root, const void* node_logits, int64_t ld, int T, int64_t V,
                  int dtype, const int32_t* seq_row0, int batch, const int64_t* node_tokens, const int32_t* parents,
                  int32_t* out, int32_t* work, hipStream_t st, const uint64_t* node_keys = nullptr,
                  int groups = 0) {
  const dim3 grid(T + 1, batch > 0 ? batch : 1);
  switch (dtype) {
    case PE_DTYPE_F32:
      accept_kernel<PE_DTYPE_F32><<<grid, kArgThreads, 0, st>>>((const float*)root_logit, ld_root,
                                                                (const float*)node_logits, ld, V, work, T, seq_row0,
                                                                node_tokens, parents, out, node_keys, groups);
      break;
    case PE_DTYPE_BF16:
      accept_kernel<PE_DTYPE_BF16><<<grid, kArgThreads, 0, st>>>((const uint16_t*)root_logit, ld_root,
                                                                 (const uint16_t*)node_logits, ld, V, work, T,
                                                                 seq_row0, node_tokens, parents, out, node_keys,
                                                                 groups);
      break;
    case PE_DTYPE_F16:
      accept_kernel<PE_DTYPE_F16><<<grid, kArgThreads, 0, st>>>((const uint16_t*)root_logit, ld_root,
                                                                (const uint16_t*)node_logits, ld, V, work, T,
                                                                seq_row0, node_tokens, parents, out, node_keys,
                                                                groups);
      break;
    default:
      return PE_ERR_ARG;
  }
  PE_CHECK_LAUNCH();
  return PE_OK;
}

int check_accept_args(const void* root_logit, const void* node_logits, int T, int64_t V, int dtype,
                      const int64_t* node_tokens, const int32_t* parents, const int32_t* out) {
  if (!root_logit || !out || T < 0 || V <= 0) return PE_ERR_ARG;
  if (dtype != PE_DTYPE_F32 && dtype != PE_DTYPE_BF16 && dtype != PE_DTYPE_F16) return PE_ERR_ARG;
  if (T > 0 && (!node_logits || !node_tokens || !parents)) return PE_ERR_ARG;
  if (T > kWalkMax) return PE_ERR_TREE;
  return PE_OK;
}

// The acceptance scratch of pe_accept_tree_noalloc: an arrival counter and
// the row argmaxes of a tree of up to kWalkMax nodes. One copy per GPU, kept
// for the life of the process; calls on one GPU share it.
static __device__ __align__(256) int32_t scratch[kWalkMax + 2];

// Device address of `scratch` per device (the array's name is a host-side
// stand-in in host code), looked up once per device with that device current.
int32_t* scratch_ptr() {
  static std::mutex mu;
  static int32_t* ptrs[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    ptrs[dev] = (int32_t*)p;
  }
  return ptrs[dev];
}

__global__ void zero_counter_kernel(int32_t* counter) { *counter = 0; }

}  // namespace

extern "C" int pe_accept_tree(const void* root_logit, const void* node_logits, int64_t ld, int T, int64_t V, int dtype,
                              const int64_t* node_tokens, const int32_t* parents, int32_t* out, int32_t* work,
                              void* stream) {
  int rc = check_accept_args(root_logit, node_logits, T, V, dtype, node_tokens, parents, out);
  if (rc != PE_OK) return rc;
  if (!work) return PE_ERR_ARG;
  return launch_accept(root_logit, 0, node_logits, ld, T, V, dtype, nullptr, 0, node_tokens, parents, out, work,
                       (hipStream_t)stream);
}

extern "C" int pe_accept_tree_keys(const void* root_logit, int64_t V, int dtype, const uint64_t* node_keys,
                                   int groups, int T, const int64_t* node_tokens, const int32_t* parents, int32_t* out,
                                   int32_t* scratch, void* stream) {
  if (!root_logit || !out || !scratch || T < 0 || V <= 0) return PE_ERR_ARG;
  if (dtype != PE_DTYPE_F32 && dtype != PE_DTYPE_BF16 && dtype != PE_DTYPE_F16) return PE_ERR_ARG;
  if (T > 0 && (!node_keys || groups <= 0 || !node_tokens || !parents)) return PE_ERR_ARG;
  if (T > kWalkMax) return PE_ERR_TREE;
  return launch_accept(root_logit, 0, nullptr, 0, T, V, dtype, nullptr, 0, node_tokens, parents, out, scratch,
                       (hipStream_t)stream, node_keys, groups);
}

extern "C" int pe_accept_tree_batch(const void* root_logits, int64_t ld_root, const void* node_logits, int64_t ld,
                                    int64_t V, int dtype, const int32_t* seq_row0, int batch, int max_seq_rows,
                                    const int64_t* node_tokens, const int32_t* parents, int32_t* out, int32_t* scratch,
                                    void* stream) {
  if (!root_logits || !node_logits || !seq_row0 || !node_tokens || !parents || !out || !scratch || batch <= 0 ||
      max_seq_rows <= 0 || V <= 0 || ld_root < V || ld < V)
    return PE_ERR_ARG;
  if (dtype != PE_DTYPE_F32 && dtype != PE_DTYPE_BF16 && dtype != PE_DTYPE_F16) return PE_ERR_ARG;
  if (max_seq_rows > kWalkMax) return PE_ERR_TREE;
  return launch_accept(root_logits, ld_root, node_logits, ld, max_seq_rows, V, dtype, seq_row0, batch, node_tokens,
                       parents, out, scratch, (hipStream_t)stream);
}

extern "C" int pe_accept_tree_noalloc(const void* root_logit, const void* node_logits, int64_t ld, int T, int64_t V,
                                      int dtype, const int64_t* node_tokens, const int32_t* parents, int32_t* out,
                                      void* stream) {
  int rc = check_accept_args(root_logit, node_logits, T, V, dtype, node_tokens, parents, out);
  if (rc != PE_OK) return rc;  // T > PE_ACCEPT_NOALLOC_MAX_NODES: PE_ERR_TREE
  int32_t* work = scratch_ptr();
  if (!work) return PE_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  // the counter starts at zero: cleared by a kernel (no memset node if the
  // caller captures this call in a graph)
  zero_counter_kernel<<<1, 1, 0, st>>>(work);
  PE_CHECK_LAUNCH();
  return launch_accept(root_logit, 0, node_logits, ld, T, V, dtype, nullptr, 0, node_tokens, parents, out, work, st);
}

extern "C" int pe_propose_tree(const void* logits, int64_t ld, int k, int64_t V, int dtype, const int32_t* widths,
                               int top_k, int64_t* node_tokens, int32_t* parents, int32_t* n_nodes, void* scratch,
                               int32_t* status, void* stream) {
  if (!logits || !widths || !node_tokens || !parents || !n_nodes || !scratch || k < 1 || k > PE_PROPOSE_MAX_DEPTH ||
      V < 1 || V > INT32_MAX || ld < V || top_k < 1)
    return PE_ERR_ARG;
  BeamShape bs{};
  bs.k = k;
  int nb = 1, total = 0;
  for (int d = 0; d < k; ++d) {
    const int w = widths[d];
    if (w < 1 || w > PE_PROPOSE_MAX_WIDTH) return PE_ERR_ARG;
    bs.width[d] = w;
    bs.cand[d] = min(top_k, w);
    if (bs.cand[d] > V) return PE_ERR_ARG;
    nb = min(w, nb * bs.cand[d]);
    total += nb;
  }
  *n_nodes = total;
  float* lp = (float*)scratch;
  int32_t* tok = (int32_t*)((char*)scratch + (size_t)k * PE_PROPOSE_MAX_WIDTH * sizeof(float));
  hipStream_t st = (hipStream_t)stream;
#define PE_PROPOSE(D)                                                                                            \
  do {                                                                                                          \
    const Elem<D>::T* x = (const Elem<D>::T*)logits;                                                            \
    const bool short_row = V <= kShortRow;                                                                      \
    draft_topk_kernel<D><<<k, kArgThreads, 0, st>>>(x, ld, V, bs, tok, short_row ? lp : nullptr, status);        \
    PE_CHECK_LAUNCH();                                                                                          \
    if (!short_row) {                                                                                           \
      draft_expsum_kernel<D><<<dim3(kSlices, k), kExpThreads, 0, st>>>(x, ld, V, tok, lp);                       \
      PE_CHECK_LAUNCH();                                                                                        \
    }                                                                                                           \
    beam_kernel<D><<<1, kBeamThreads, 0, st>>>(x, ld, bs, lp, tok, node_tokens, parents, status);                \
    PE_CHECK_LAUNCH();                                                                                          \
  } while (0)
  switch (dtype) {
    case PE_DTYPE_F32: PE_PROPOSE(PE_DTYPE_F32); break;
    case PE_DTYPE_BF16: PE_PROPOSE(PE_DTYPE_BF16); break;
    case PE_DTYPE_F16: PE_PROPOSE(PE_DTYPE_F16); break;
    default: return PE_ERR_ARG;
  }
#undef PE_PROPOSE
  return PE_OK;
}

extern "C" int pe_kv_compact(void* k_cache, void* v_cache, int L, int nkv, int64_t cap, int hd, int dtype, int64_t P,
                             const int32_t* accept_out, void* stream) {
  if (!k_cache || !v_cache || !accept_out || L <= 0 || nkv <= 0 || hd <= 0 || P < 0) return PE_ERR_ARG;
  const int64_t row_bytes = (int64_t)hd * esize(dtype);
  if (row_bytes % 16) return PE_ERR_ARG;
  dim3 grid(L * nkv, 2);
  kv_compact_kernel<<<grid, 64, 0, (hipStream_t)stream>>>((uint8_t*)k_cache, (uint8_t*)v_cache, cap, row_bytes, P,
                                                         accept_out, nullptr, 0, 0);
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_kv_compact_batch(void* k_cache, void* v_cache, int batch, int64_t cache_seq_stride, int L, int nkv,
                                   int64_t cap, int hd, int dtype, const int64_t* seq_prefix, const int32_t* accept_out,
                                   int max_seq_rows, void* stream) {
  if (!k_cache || !v_cache || !accept_out || !seq_prefix || batch <= 0 || L <= 0 || nkv <= 0 || hd <= 0 ||
      max_seq_rows <= 0)
    return PE_ERR_ARG;
  const int64_t row_bytes = (int64_t)hd * esize(dtype);
  if (row_bytes % 16 || cache_seq_stride < (int64_t)L * nkv * cap * hd) return PE_ERR_ARG;
  dim3 grid(L * nkv, 2, batch);
  kv_compact_kernel<<<grid, 64, 0, (hipStream_t)stream>>>((uint8_t*)k_cache, (uint8_t*)v_cache, cap, row_bytes, 0,
                                                         accept_out, seq_prefix, cache_seq_stride * esize(dtype),
                                                         2 + max_seq_rows);
  PE_CHECK_LAUNCH();
  return PE_OK;
}

extern "C" int pe_kv_gather(void* k_cache, void* v_cache, int L, int nkv, int64_t cap, int hd, int dtype,
                            const int64_t* keep, int64_t n_keep, int32_t* status, void* stream) {
  if (!k_cache || !v_cache || !keep || !status || L <= 0 || nkv <= 0 || hd <= 0 || n_keep < 0 || n_keep > cap)
    return PE_ERR_ARG;
  if (n_keep == 0) return PE_OK;
  const int64_t row_bytes = (int64_t)hd * esize(dtype);
  if (row_bytes % 16) return PE_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  // `first` lives in the status word's neighbour: callers pass status as int32[4] (8-byte aligned at +8)
  int64_t* first = (int64_t*)(status + 2);
  kv_keep_check_kernel<<<1, 256, 0, st>>>(keep, n_keep, cap, first, status);
  PE_CHECK_LAUNCH();
  dim3 grid(L * nkv, 2);
  kv_gather_kernel<<<grid, 64, 0, st>>>((uint8_t*)k_cache, (uint8_t*)v_cache, cap, row_bytes, keep, n_keep, first);
  PE_CHECK_LAUNCH();
  return PE_OK;
}
