// Fused beam-search step over trie-constrained candidates: mask -> top-K ->
// expand token rows -> advance trie nodes.
//
// Reference: python/flashrec/kernel/beam_trie.py:536-633
// (genrec_mask_topk_expand, whose PyTorch branch defines the result) and its
// CUDA kernel python/flashrec/kernel/csrc/beam_trie.cuh:548-757, whose
// choices for what the PyTorch branch leaves open are kept: candidates are
// ranked by score descending, then flat index (b * C + c) ascending; with
// masking on, masked candidates (and -inf scores) are never picked, and when
// fewer than K remain the missing picks are (-inf, index 0, parent 0,
// token top_tokens[n][0][0]); rows b >= K of the token / node planes are
// copied unchanged; with expansion off nothing is advanced either.
// Candidate rule (beam_trie.cuh:37-49): node < 0 accepts every token,
// otherwise allow[node][tok - token_base] with tok outside the table refused;
// transition (:51-64): node < 0 stays, tok outside the table -> invalid_node,
// else next_node[node][tok - token_base].  NaN scores are treated as masked.
//
// Layout for MI355X.  Per request the candidates are BW beams x C columns,
// each beam's C sorted descending (they come from a per-row sorted top-k).  A
// candidate is one 64-bit key: the orderable bits of its score in the high
// word, the complement of its flat index in the low word, so keys are distinct
// and "larger key" is exactly the ranking above.  Both kernels are a chain of
// latencies (one request's beam step takes as long as eight requests'), so
// they select instead of merging: a 2048-bin LDS histogram of the key range,
// narrowed to the bin that holds the K-th key until few enough keys are left
// (select_top), is a handful of barriers where a tree of pairwise merges was
// a binary search and a walk of dependent LDS reads per level.
//   kernel 1, one workgroup per (request, slice of BS beams): each wave
//     compacts its beams' valid candidates into per-beam lists of at most K
//     keys (ballot prefix sums; stops at K); the slice's best K of them, in
//     no particular order, go to the caller's scratch;
//   kernel 2, one workgroup per request: selects at most 1024 keys that hold
//     the top K from the slices' lists, sorts them (one key per thread),
//     writes vals / parents / tokens / indices, then the expanded token rows
//     and the advanced trie nodes.
// 8 x 512 beams x 1024 candidates -> top 512: 34.0 + 33.6 us with merge trees,
// 18.2 + 18.3 so; 1 x 512 33.6 + 33.7 -> 15.4 + 17.8; 8 x 35 21.4 + 10.6 -> 10.1
// + 8.4, both together 5.6 less with narrow beams and few lists told apart (below).
// What is left is latency: kernel 2 is one CU per request.
#include <mutex>
#include <type_traits>

#include "fr_common.h"

namespace fr {

struct GenrecArgs {
  float* out_vals;        // [N, K]
  int64_t* out_parents;   // [N, K]
  int64_t* out_tokens;    // [N, K]
  int64_t* out_indices;   // [N, K]
  uint64_t* scratch;      // [N, S, 1 + K]
  const float* cum;       // [N, BW]
  const float* lp;        // [N, BW, C]
  const int64_t* tok;     // [N, BW, C]
  const int64_t* nodes;   // [N, BW] or null
  const uint8_t* allow;   // [n_nodes, vsz] or null
  const int64_t* tin;     // [N, BW, L] or null
  int64_t* tout;          // [N, BW, L] or null
  const void* next;       // [n_nodes, vsz] int64 or int32 (next_i32), or null
  int next_i32;
  int64_t* nout;          // [N, BW] or null
  const uint8_t* do_exp;  // [N] or null (all)
  const int32_t* col;     // [N]
  int64_t token_base, n_nodes, vsz, invalid_node;
  float neg_inf;
  int N, BW, C, K, L, S, BS;
  int apply_mask, apply_expand, apply_advance;
};

constexpr int kListKeys = 8192;  // keys per LDS list buffer (64 KB)

__device__ __forceinline__ uint32_t order_bits(float v) {
  const uint32_t u = __float_as_uint(v);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float from_order_bits(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o);
}
__device__ __forceinline__ uint64_t make_key(float v, uint32_t idx) {
  return (static_cast<uint64_t>(order_bits(v)) << 32) | static_cast<uint64_t>(~idx);
}
__device__ __forceinline__ float key_val(uint64_t k) { return from_order_bits(static_cast<uint32_t>(k >> 32)); }
__device__ __forceinline__ uint32_t key_idx(uint64_t k) { return ~static_cast<uint32_t>(k); }

constexpr int kBins = 2048;  // select_top's histogram

// LDS of select_top.
struct SelectLds {
  uint32_t hist[kBins];
  uint32_t wsum[16];
  uint64_t hi[16], lo[16];
  uint64_t edge[2];  // bin of the K-th key, keys before it
  uint32_t at;       // keys in it
};

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
  const uint32_t lo = __shfl_xor(static_cast<uint32_t>(v), m, 64);
  const uint32_t hi = __shfl_xor(static_cast<uint32_t>(v >> 32), m, 64);
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Largest and smallest nonzero of the block's keys (PER per thread).
template <int PER>
__device__ __forceinline__ void key_range(const uint64_t (&key)[PER], uint64_t& hi, uint64_t& lo, SelectLds& L) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  hi = 0;
  lo = ~0ull;
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    hi = key[r] > hi ? key[r] : hi;
    lo = key[r] != 0 && key[r] < lo ? key[r] : lo;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint64_t h = shfl_xor_u64(hi, o), l = shfl_xor_u64(lo, o);
    hi = h > hi ? h : hi;
    lo = l < lo ? l : lo;
  }
  if (lane == 0) {
    L.hi[wave] = hi;
    L.lo[wave] = lo;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    hi = L.hi[w] > hi ? L.hi[w] : hi;
    lo = L.lo[w] < lo ? L.lo[w] : lo;
  }
}

// Inclusive sum over the block's threads in order (one barrier).
__device__ __forceinline__ uint32_t block_scan(uint32_t v, SelectLds& L) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  if (lane == 63) L.wsum[wave] = v;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 16; ++w) v += w < wave ? L.wsum[w] : 0u;
  return v;
}

// A threshold that at least K and at most `cap` >= K of the block's `n` keys
// (PER per thread, 0: none; all distinct) reach; 1 when n <= cap.  1024
// threads, all of which call this with the same n, K, cap.
template <int PER>
__device__ __forceinline__ uint64_t select_top(const uint64_t (&key)[PER], int n, int K, int cap, SelectLds& L) {
  if (n <= cap) return 1;
  uint64_t hi, lo;
  key_range<PER>(key, hi, lo, L);
  uint32_t sure = 0;  // keys above hi
  for (;;) {
    const uint64_t range = hi - lo;
    const int bits = range == 0 ? 0 : 64 - __builtin_clzll(range);
    const int shift = bits > 11 ? bits - 11 : 0;  // 2048 bins
    L.hist[threadIdx.x] = L.hist[threadIdx.x + 1024] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < PER; ++r)
      if (key[r] >= lo && key[r] <= hi) atomicAdd(&L.hist[(hi - key[r]) >> shift], 1u);
    __syncthreads();
    // bins 2 t and 2 t + 1 of thread t, scanned over the block
    const uint32_t c0 = L.hist[2 * threadIdx.x], c1 = L.hist[2 * threadIdx.x + 1];
    const uint32_t run = block_scan(c0 + c1, L);
    const uint32_t need = static_cast<uint32_t>(K) - sure;
    const uint32_t b0 = run - c0 - c1, b1 = run - c1;  // keys before each bin
    if (b0 < need && need <= b1) {
      L.edge[0] = 2 * threadIdx.x;
      L.edge[1] = b0;
      L.at = c0;
    } else if (b1 < need && need <= run) {
      L.edge[0] = 2 * threadIdx.x + 1;
      L.edge[1] = b1;
      L.at = c1;
    }
    __syncthreads();
    const uint64_t bin = L.edge[0];
    const uint32_t before = static_cast<uint32_t>(L.edge[1]), in = L.at;
    const uint64_t top = hi - (bin << shift);  // the bin holds keys top - width + 1 .. top
    const uint64_t width = 1ull << shift;
    const uint64_t low = top - lo < width ? lo : top - width + 1;
    if (sure + before + in <= static_cast<uint32_t>(cap) || shift == 0) return low;
    sure += before;
    hi = top;
    lo = low;
  }
}

// Position threadIdx.x + 1024 r of lists of K entries as (list, entry).
struct ListAt {
  int l, i, dl, di;
  __device__ __forceinline__ explicit ListAt(int K)
      : l(static_cast<int>(threadIdx.x) / K), i(static_cast<int>(threadIdx.x) % K), dl(1024 / K), di(1024 % K) {}
  __device__ __forceinline__ void next(int K) {
    l += dl;
    i += di;
    if (i >= K) {
      i -= K;
      ++l;
    }
  }
};

// Sorts the first `n` <= 1024 keys of `keys` descending in place: each key's
// place is its bin's start (2048 bins over the keys' range) plus its rank
// among the few keys of its bin.  Keys that crowd a bin (more than 32) are
// sorted by a bitonic network instead.  `buf` holds 1024 keys; 1024 threads.
__device__ __forceinline__ void sort_desc(uint64_t* keys, int n, uint64_t* buf, SelectLds& L) {
  const int t = threadIdx.x;
  const uint64_t key[1] = {t < n ? keys[t] : 0};
  if (n <= 64) {  // one wave, in registers; a network as wide as the keys
    if (t < 64) {
      uint64_t v = key[0];
      for (int k = 2; k < 2 * n; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
          const uint64_t o = shfl_xor_u64(v, j);
          const bool want_max = ((t & j) == 0) == ((t & k) == 0);
          v = want_max == (v < o) ? o : v;
        }
      keys[t] = v;
    }
    __syncthreads();
    return;
  }
  uint64_t hi, lo;
  key_range<1>(key, hi, lo, L);
  const uint64_t range = n > 0 ? hi - lo : 0;
  const int bits = range == 0 ? 0 : 64 - __builtin_clzll(range);
  const int shift = bits > 11 ? bits - 11 : 0;
  L.hist[t] = L.hist[t + 1024] = 0;
  if (t == 0) L.at = 0;
  __syncthreads();
  const uint32_t bin = t < n ? static_cast<uint32_t>((hi - key[0]) >> shift) : 0u;
  const uint32_t r = t < n ? atomicAdd(&L.hist[bin], 1u) : 0u;
  __syncthreads();
  const uint32_t c0 = L.hist[2 * t], c1 = L.hist[2 * t + 1];
  if (c0 > 32 || c1 > 32) L.at = 1;
  const uint32_t run = block_scan(c0 + c1, L);
  L.hist[2 * t] = run - c0 - c1;
  L.hist[2 * t + 1] = run - c1;
  __syncthreads();
  if (L.at == 0) {
    uint32_t s = 0, e = 0;
    if (t < n) {
      s = L.hist[bin];
      e = bin + 1 < kBins ? L.hist[bin + 1] : static_cast<uint32_t>(n);
      buf[s + r] = key[0];
    }
    __syncthreads();
    uint32_t place = s;
    for (uint32_t m = s; m < e; ++m) place += buf[m] > key[0] ? 1u : 0u;
    if (t < n) keys[place] = key[0];
    __syncthreads();
    return;
  }
  uint64_t v = key[0];
  int width = 2;
  while (width < n) width <<= 1;
  for (int k = 2; k <= width; k <<= 1) {
    for (int j = k >> 1; j > 0; j >>= 1) {
      uint64_t o;
      if (j < 64) {
        o = shfl_xor_u64(v, j);
      } else {
        __syncthreads();
        buf[t] = v;
        __syncthreads();
        o = buf[t ^ j];
      }
      const bool want_max = ((t & j) == 0) == ((t & k) == 0);
      v = want_max == (v < o) ? o : v;
    }
  }
  __syncthreads();
  keys[t] = v;
  __syncthreads();
}

constexpr int kRowBytes = 1024;   // widest allow row looked up through LDS
constexpr int kSliceWaves = 16;  // one wave per beam of a slice (BS <= 16)

__global__ __launch_bounds__(64 * kSliceWaves) void genrec_slice_topk(GenrecArgs a) {
  static_assert(kSliceWaves == 16, "select_top's 1024 threads");
  __shared__ uint64_t buf[kListKeys];
  __shared__ SelectLds sel;
  __shared__ __attribute__((aligned(16))) uint8_t rows[kSliceWaves][kRowBytes];  // the beams' rows of the allow table
  __shared__ int len[kSliceWaves];
  __shared__ uint32_t cursor;
  const int n = blockIdx.x / a.S, s = blockIdx.x - (blockIdx.x / a.S) * a.S;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b0 = s * a.BS;
  const int nb = a.BW - b0 < a.BS ? a.BW - b0 : a.BS;
  const bool mask = a.apply_mask && a.allow != nullptr && a.nodes != nullptr;
  // wave j compacts beam j of the slice (BS <= kSliceWaves): its list at
  // buf + j * K.  The beam's candidates go in groups of kPre chunks of 64: the
  // scores and tokens of the whole group are loaded, then all of its trie
  // lookups are issued, then the chunks are compacted in order (ballot prefix
  // sums, stopping at K): two memory round trips per group.  Loads are
  // unconditional on clamped indices: under a lane's condition each would
  // wait for the one before it.  Narrow beams take groups of one or four chunks:
  // the instructions of sixteen, and of sixteen keys a thread in kernel 2, were
  // most of a small step (both kernels: 1 beam of 16 candidates 13.8 -> 8.1 us, 20
  // beams of 40 21.6 -> 15.3).
  if (wave < nb) {
    const int b = b0 + wave;
    const float cb = a.cum[static_cast<int64_t>(n) * a.BW + b];
    const int64_t node = mask ? a.nodes[static_cast<int64_t>(n) * a.BW + b] : -1;
    const float* lpb = a.lp + (static_cast<int64_t>(n) * a.BW + b) * a.C;
    const int64_t* tkb = a.tok + (static_cast<int64_t>(n) * a.BW + b) * a.C;
    const bool lookup = node >= 0 && a.n_nodes > 0 && a.vsz > 0;  // (node < 0 accepts every token)
    const uint8_t* allow = nullptr;
    if (lookup) allow = a.allow + (node > a.n_nodes - 1 ? a.n_nodes - 1 : node) * a.vsz;
    // A row of up to 1 KB is read once, 16 bytes a lane, and looked up in LDS:
    // 1024 candidates are 16 gathers of 64 single bytes, and a gather takes
    // the address path a cycle a lane (8 us of a 512-beam step).
    const bool staged = lookup && a.vsz <= kRowBytes && a.vsz % 16 == 0 && (reinterpret_cast<uintptr_t>(allow) & 15) == 0;
    if (staged && 16 * lane < a.vsz)
      *reinterpret_cast<u32x4*>(rows[wave] + 16 * lane) = *reinterpret_cast<const u32x4*>(allow + 16 * lane);
    int count = 0;
    auto group = [&](int g0, auto pre_c) __attribute__((always_inline)) {
      constexpr int kPre = decltype(pre_c)::value;
      float v[kPre];
      int64_t rel[kPre];
#pragma unroll
      for (int u = 0; u < kPre; ++u) {
        const int c = g0 + 64 * u + lane, cc = c < a.C ? c : a.C - 1;
        v[u] = cb + lpb[cc];
        rel[u] = lookup ? tkb[cc] - a.token_base : 0;
      }
      uint32_t in[kPre] = {};
      if (staged) {
#pragma unroll
        for (int u = 0; u < kPre; ++u) in[u] = rows[wave][rel[u] >= 0 && rel[u] < a.vsz ? rel[u] : 0];
      } else if (lookup) {
#pragma unroll
        for (int u = 0; u < kPre; ++u) in[u] = allow[rel[u] >= 0 && rel[u] < a.vsz ? rel[u] : 0];
      }
#pragma unroll
      for (int u = 0; u < kPre; ++u) {
        const int c = g0 + 64 * u + lane;
        bool ok = c < a.C && count < a.K && v[u] == v[u];  // NaN: never picked
        if (mask) ok = ok && v[u] != a.neg_inf && (node < 0 || lookup);
        if (lookup) ok = ok && rel[u] >= 0 && rel[u] < a.vsz && in[u] != 0;
        const uint64_t bal = __ballot(ok);
        const int pos = count + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                                    static_cast<uint32_t>(bal >> 32),
                                    __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(bal), 0u)));
        if (ok && pos < a.K) buf[wave * a.K + pos] = make_key(v[u], static_cast<uint32_t>(b * a.C + c));
        count += __builtin_popcountll(bal);
      }
    };
    if (a.C <= 64) group(0, std::integral_constant<int, 1>{});
    else if (a.C <= 256) group(0, std::integral_constant<int, 4>{});
    else
      for (int g0 = 0; g0 < a.C && count < a.K; g0 += 1024) group(g0, std::integral_constant<int, 16>{});
    if (lane == 0) len[wave] = count < a.K ? count : a.K;
  } else if (lane == 0) {
    len[wave] = 0;
  }
  if (threadIdx.x == 0) cursor = 0;
  __syncthreads();
  int total = 0;
#pragma unroll
  for (int j = 0; j < kSliceWaves; ++j) total += len[j];
  uint64_t* const out = a.scratch + (static_cast<int64_t>(n) * a.S + s) * (1 + a.K);
  if (threadIdx.x == 0) out[0] = static_cast<uint64_t>(total < a.K ? total : a.K);
  constexpr int kPer = kListKeys / 1024;
  uint64_t key[kPer];
  ListAt at(a.K);
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const bool ok = at.l < nb && at.i < len[at.l < nb ? at.l : 0];
    key[r] = ok ? buf[threadIdx.x + r * 1024] : 0;
    at.next(a.K);
  }
  // the rest of the list: 0, no key (kernel 2 then reads whole lists without
  // waiting for their lengths)
  for (int i = total + static_cast<int>(threadIdx.x); i < a.K; i += 1024) out[1 + i] = 0;
  const uint64_t least = select_top<kPer>(key, total, a.K, a.K, sel);
#pragma unroll
  for (int r = 0; r < kPer; ++r)
    if (key[r] >= least) out[1 + atomicAdd(&cursor, 1u)] = key[r];
}

__global__ __launch_bounds__(1024) void genrec_request_topk_expand(GenrecArgs a) {
  __shared__ uint64_t acc[1024];  // keys that hold the top K of the lists read so far
  __shared__ SelectLds sel;
  __shared__ int len[64];
  __shared__ uint32_t cursor;
  __shared__ int64_t sel_parent[1024];
  __shared__ int64_t sel_token[1024];
  const int n = blockIdx.x;
  const int K = a.K;
  const uint64_t* lists = a.scratch + static_cast<int64_t>(n) * a.S * (1 + K);
  // The slices' lists go in groups of G that fill the threads' registers (one
  // key a thread where that holds all of them); the keys kept from the groups
  // before ride along.
  // keys kept: up to twice K's power of two, so that one histogram pass mostly
  // does and the sort below stays short
  int cap = 2;
  while (cap < K) cap <<= 1;
  cap = cap < 512 ? 2 * cap : 1024;
  int held = 0;
  auto select = [&](auto per_c) __attribute__((always_inline)) {
    constexpr int kPer = decltype(per_c)::value;
    const int G = kPer * 1024 / K < 64 ? kPer * 1024 / K : 64;  // (len[] holds 64)
    for (int g0 = 0; g0 < a.S; g0 += G) {
      const int gs = a.S - g0 < G ? a.S - g0 : G;
      const uint64_t* gl = lists + static_cast<int64_t>(g0) * (1 + K);
      if (threadIdx.x == 0) cursor = 0;
      uint64_t key[kPer + 1];
      ListAt at(K);
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const uint64_t x = gl[at.l < gs ? static_cast<uint32_t>(at.l * (1 + K) + 1 + at.i) : 0u];
        key[r] = at.l < gs ? x : 0;
        at.next(K);
      }
      if (threadIdx.x < 64)
        len[threadIdx.x] = static_cast<int>(threadIdx.x) < gs ? static_cast<int>(gl[threadIdx.x * (1 + K)]) : 0;
      __syncthreads();
      key[kPer] = static_cast<int>(threadIdx.x) < held ? acc[threadIdx.x] : 0;
      int total = len[threadIdx.x & 63];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o, 64);
      total += held;
      __syncthreads();  // acc, len and the cursor are read
      const uint64_t least = select_top<kPer + 1>(key, total, K, cap, sel);
#pragma unroll
      for (int r = 0; r <= kPer; ++r)
        if (key[r] != 0 && key[r] >= least) acc[atomicAdd(&cursor, 1u)] = key[r];
      __syncthreads();
      held = static_cast<int>(cursor);
      __syncthreads();
    }
  };
  if (a.S * K <= 1024) select(std::integral_constant<int, 1>{});
  else select(std::integral_constant<int, 16>{});
  sort_desc(acc, held, reinterpret_cast<uint64_t*>(sel_parent), sel);
  const uint64_t* res = acc;
  const int got = held < K ? held : K;
  const int64_t* tkn = a.tok + static_cast<int64_t>(n) * a.BW * a.C;
  for (int k = threadIdx.x; k < K; k += blockDim.x) {
    float v = a.neg_inf;
    uint32_t idx = 0;
    if (k < got) {
      v = key_val(res[k]);
      idx = key_idx(res[k]);
    }
    const int64_t parent = k < got ? static_cast<int64_t>(idx / static_cast<uint32_t>(a.C)) : 0;
    const int64_t token = tkn[idx];
    const int64_t o = static_cast<int64_t>(n) * K + k;
    a.out_vals[o] = v;
    a.out_parents[o] = parent;
    a.out_tokens[o] = token;
    a.out_indices[o] = static_cast<int64_t>(idx);
    sel_parent[k] = parent;
    sel_token[k] = token;
  }
  const bool expand = a.apply_expand && a.tin != nullptr && a.tout != nullptr &&
                      (a.do_exp == nullptr || a.do_exp[n] != 0);
  if (!expand) return;
  __syncthreads();
  const int col = a.col[n] < 0 ? 0 : a.col[n];
  const int64_t* tin = a.tin + static_cast<int64_t>(n) * a.BW * a.L;
  int64_t* tout = a.tout + static_cast<int64_t>(n) * a.BW * a.L;
  for (int64_t e = threadIdx.x; e < static_cast<int64_t>(a.BW) * a.L; e += blockDim.x) {
    const int b = static_cast<int>(e / a.L), c = static_cast<int>(e - static_cast<int64_t>(b) * a.L);
    if (b >= K) {
      tout[e] = tin[e];
    } else if (c == col) {
      tout[e] = sel_token[b];
    } else {
      int64_t p = sel_parent[b];
      p = p < 0 ? 0 : (p > a.BW - 1 ? a.BW - 1 : p);
      tout[e] = tin[p * a.L + c];
    }
  }
  if (a.apply_advance && a.next != nullptr && a.nodes != nullptr && a.nout != nullptr) {
    const int64_t* nin = a.nodes + static_cast<int64_t>(n) * a.BW;
    int64_t* nout = a.nout + static_cast<int64_t>(n) * a.BW;
    for (int b = threadIdx.x; b < a.BW; b += blockDim.x) {
      if (b >= K) {
        nout[b] = nin[b];
        continue;
      }
      int64_t p = sel_parent[b];
      p = p < 0 ? 0 : (p > a.BW - 1 ? a.BW - 1 : p);
      const int64_t old = nin[p];
      int64_t nx;
      if (old < 0) {
        nx = old;
      } else {
        const int64_t rel = sel_token[b] - a.token_base;
        if (rel < 0 || rel >= a.vsz || a.n_nodes <= 0) {
          nx = a.invalid_node;
        } else {
          const int64_t safe = old > a.n_nodes - 1 ? a.n_nodes - 1 : old;
          const int64_t cell = safe * a.vsz + rel;
          nx = a.next_i32 ? static_cast<int64_t>(static_cast<const int32_t*>(a.next)[cell])
                          : static_cast<const int64_t*>(a.next)[cell];
        }
      }
      nout[b] = nx;
    }
  }
}

}  // namespace fr

using namespace fr;

extern "C" int fr_genrec_scratch_bytes(int64_t N, int64_t BW, int64_t K) {
  if (N <= 0 || BW <= 0 || K <= 0 || K > 1024) return -1;
  const int64_t BS = kListKeys / K < 16 ? kListKeys / K : 16;
  const int64_t S = (BW + BS - 1) / BS;
  const int64_t bytes = N * S * (1 + K) * 8;
  return bytes > 0x7FFFFFFF ? -1 : static_cast<int>(bytes);
}

// Argument checks shared by both entry points; the scratch is checked by
// each (caller's buffer, or the library's static one).
static int genrec_check(float* out_vals, int64_t* out_parents, int64_t* out_tokens, int64_t* out_indices,
                        const float* cum, const float* top_logprobs, const int64_t* top_tokens,
                        const int32_t* col, int64_t N, int64_t BW, int64_t C, int64_t K, int64_t L) {
  if (N < 0 || BW <= 0 || C <= 0 || K <= 0 || L < 0) return FR_EINVAL;
  if (N == 0) return FR_OK;
  if (!out_vals || !out_parents || !out_tokens || !out_indices || !cum || !top_logprobs || !top_tokens ||
      !col)
    return FR_EINVAL;
  if (K > 1024 || K > BW * C || BW * C > 0x7FFFFFFF) return FR_EUNSUPPORTED;
  return FR_OK;
}

static int genrec_launch(
    float* out_vals, int64_t* out_parents, int64_t* out_tokens, int64_t* out_indices, void* scratch,
    const float* cum, const float* top_logprobs, const int64_t* top_tokens,
    const int64_t* node_ids, const uint8_t* allow_table, const int64_t* token_ids_in,
    int64_t* token_ids_out, const void* next_node, int64_t* node_ids_out, const uint8_t* do_expand,
    const int32_t* col, int64_t token_base, int64_t n_nodes, int64_t vsz, int64_t invalid_node,
    int64_t N, int64_t BW, int64_t C, int64_t K, int64_t L, int apply_mask, int apply_expand,
    int apply_advance, int next_i32, void* stream) {
  if (apply_mask && node_ids && allow_table && n_nodes > 0 && vsz <= 0) return FR_EINVAL;
  if (apply_expand && (!token_ids_in || !token_ids_out || L <= 0)) return FR_EINVAL;
  if (apply_expand && token_ids_in == token_ids_out) return FR_EINVAL;  // rows gather from other rows
  GenrecArgs a{};
  a.out_vals = out_vals;
  a.out_parents = out_parents;
  a.out_tokens = out_tokens;
  a.out_indices = out_indices;
  a.scratch = static_cast<uint64_t*>(scratch);
  a.cum = cum;
  a.lp = top_logprobs;
  a.tok = top_tokens;
  a.nodes = node_ids;
  a.allow = allow_table;
  a.tin = token_ids_in;
  a.tout = token_ids_out;
  a.next = next_node;
  a.next_i32 = next_i32 ? 1 : 0;
  a.nout = node_ids_out;
  a.do_exp = do_expand;
  a.col = col;
  a.token_base = token_base;
  a.n_nodes = n_nodes;
  a.vsz = vsz;
  a.invalid_node = invalid_node;
  a.neg_inf = -__builtin_inff();
  a.N = static_cast<int>(N);
  a.BW = static_cast<int>(BW);
  a.C = static_cast<int>(C);
  a.K = static_cast<int>(K);
  a.L = static_cast<int>(L);
  a.BS = kListKeys / a.K < 16 ? kListKeys / a.K : 16;
  a.S = (a.BW + a.BS - 1) / a.BS;
  a.apply_mask = apply_mask;
  a.apply_expand = apply_expand;
  a.apply_advance = apply_advance;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(genrec_slice_topk, dim3(static_cast<unsigned>(N * a.S)), dim3(64 * kSliceWaves), 0, st, a);
  hipLaunchKernelGGL(genrec_request_topk_expand, dim3(static_cast<unsigned>(N)), dim3(1024), 0, st, a);
  return hipGetLastError() == hipSuccess ? FR_OK : FR_ELAUNCH;
}

extern "C" int fr_genrec_mask_topk_expand(
    float* out_vals, int64_t* out_parents, int64_t* out_tokens, int64_t* out_indices, void* scratch,
    int64_t scratch_bytes, const float* cum, const float* top_logprobs, const int64_t* top_tokens,
    const int64_t* node_ids, const uint8_t* allow_table, const int64_t* token_ids_in,
    int64_t* token_ids_out, const void* next_node, int64_t* node_ids_out, const uint8_t* do_expand,
    const int32_t* col, int64_t token_base, int64_t n_nodes, int64_t vsz, int64_t invalid_node,
    int64_t N, int64_t BW, int64_t C, int64_t K, int64_t L, int apply_mask, int apply_expand,
    int apply_advance, int next_i32, void* stream) {
  const int rc = genrec_check(out_vals, out_parents, out_tokens, out_indices, cum, top_logprobs, top_tokens,
                              col, N, BW, C, K, L);
  if (rc != FR_OK || N == 0) return rc;
  if (!scratch) return FR_EINVAL;
  const int need = fr_genrec_scratch_bytes(N, BW, K);
  if (need < 0 || scratch_bytes < need) return FR_EINVAL;
  return genrec_launch(out_vals, out_parents, out_tokens, out_indices, scratch, cum, top_logprobs,
                       top_tokens, node_ids, allow_table, token_ids_in, token_ids_out, next_node,
                       node_ids_out, do_expand, col, token_base, n_nodes, vsz, invalid_node, N, BW, C, K, L,
                       apply_mask, apply_expand, apply_advance, next_i32, stream);
}

// ---- The same step with no allocation anywhere: the slice lists live in a
// static device array of FR_GENREC_NOALLOC_SCRATCH_BYTES (every GPU the
// library runs on holds its own copy until the process ends).  Its device
// address is looked up once per device, with that device current; host code
// never passes the array's name to a kernel (on the host that name is a
// stand-in, not a device address).  The slice kernel writes every list entry
// the request kernel reads, so nothing needs clearing between calls.  All
// calls on one GPU share the array: calls that overlap on one GPU (other
// streams, other threads) race.
static __device__ __align__(256) uint64_t genrec_static_scratch[FR_GENREC_NOALLOC_SCRATCH_BYTES / 8];

static void* genrec_static_scratch_ptr() {
  static std::mutex mu;
  static void* ptrs[kMaxDevices] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(mu);
  if (ptrs[dev] == nullptr) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(genrec_static_scratch)) != hipSuccess) return nullptr;
    ptrs[dev] = p;
  }
  return ptrs[dev];
}

extern "C" int fr_genrec_mask_topk_expand_noalloc(
    float* out_vals, int64_t* out_parents, int64_t* out_tokens, int64_t* out_indices, const float* cum,
    const float* top_logprobs, const int64_t* top_tokens, const int64_t* node_ids,
    const uint8_t* allow_table, const int64_t* token_ids_in, int64_t* token_ids_out,
    const void* next_node, int64_t* node_ids_out, const uint8_t* do_expand, const int32_t* col,
    int64_t token_base, int64_t n_nodes, int64_t vsz, int64_t invalid_node, int64_t N, int64_t BW,
    int64_t C, int64_t K, int64_t L, int apply_mask, int apply_expand, int apply_advance, int next_i32,
    void* stream) {
  const int rc = genrec_check(out_vals, out_parents, out_tokens, out_indices, cum, top_logprobs, top_tokens,
                              col, N, BW, C, K, L);
  if (rc != FR_OK || N == 0) return rc;
  const int need = fr_genrec_scratch_bytes(N, BW, K);
  if (need < 0 || need > FR_GENREC_NOALLOC_SCRATCH_BYTES) return FR_ETOOLARGE;
  void* scratch = genrec_static_scratch_ptr();
  if (scratch == nullptr) return FR_ELAUNCH;
  return genrec_launch(out_vals, out_parents, out_tokens, out_indices, scratch, cum, top_logprobs,
                       top_tokens, node_ids, allow_table, token_ids_in, token_ids_out, next_node,
                       node_ids_out, do_expand, col, token_base, n_nodes, vsz, invalid_node, N, BW, C, K, L,
                       apply_mask, apply_expand, apply_advance, next_i32, stream);
}
