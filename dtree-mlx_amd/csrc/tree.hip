// Draft-tree construction on the GPU (build_dtree_tree, dtree_runtime.py:82-163):
// per-depth top-k of the draft logits with log-probs = logit - logsumexp(row),
// then the best-first heap over cumulative log-probs, written straight into the
// verify step's descriptor (tokens, positions = P + depth, parents, ancestor
// bitsets; compile_dtree_tree, dtree_runtime.py:166-192).
//
// Three launches, all graph-capturable:
//   1. topk_chunk_kernel  (row, 8192-logit chunk): chunk max and sum of
//      exp(x - max), and the chunk's top-k by a bound (bounded_topk) or, where
//      that does not thin the chunk out, a four-digit radix select;
//   2. topk_merge_kernel  (row): the union of the chunk candidates (which
//      holds the row's top-k) selected the same way and sorted; log-probs
//      from the merged logsumexp;
//   3. heap_kernel        (one wavefront): the reference's heap order.
//
// Order rules that make the tree identical to the reference's given the same
// top-k lists and log-probs:
//   * a row's top-k is sorted by (logit desc, token id asc);
//   * heap entries compare as the Python tuples (-logw, ranks, ...): larger
//     logw first, then the lexicographically smaller rank tuple (a prefix
//     before its extensions). logw is a double built with the reference's
//     operation order (sibling: (logw - lp[d][r]) + lp[d][r + 1]; child:
//     logw + lp[d + 1][0]); rank tuples are packed 7 bits per level (value
//     rank + 1, zero past the end) into a 128-bit big-endian key, so they
//     compare as integers.
#include "common.h"

namespace dtree {
namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 8192;                // logits per workgroup in pass 1
constexpr int kE1 = kChunk / kThreads;      // contiguous logits per thread
constexpr int kCand = 4096;                 // candidates per row in pass 2
constexpr int kE2 = kCand / kThreads;
constexpr int kMaxK = 127;                  // rank + 1 fits the 7-bit level field
constexpr int kMaxDepth = 18;               // 18 levels x 7 bits in 128 bits
constexpr int kMaxEntries = 256;            // heap entries: 1 + 2 * budget

__device__ __forceinline__ uint32_t ordered_bits(float x) {
  const uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}

// Wave-wide unsigned maximum (in every lane) by the cross-lane adders of the
// vector unit: six dependent operations, where shuffles go through LDS.
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
  auto step = [&](uint32_t o) { v = max(v, o); };
  step(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // row_shr:1
  step(__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  step(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1, 3
  step(__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2, 3
  return __builtin_amdgcn_readlane(v, 63);
}

struct SelectLds {
  uint32_t hist[256];
  uint32_t wave_sum[kThreads / 64];
  uint32_t prefix, need, take_all, n_out;
  unsigned long long list[128];
};

// Block-wide exclusive prefix sum over threads in thread order.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, SelectLds& s) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  uint32_t inc = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t u = __shfl_up(inc, o);
    if (lane >= o) inc += u;
  }
  if (lane == 63) s.wave_sum[w] = inc;
  __syncthreads();
  uint32_t before = 0;
  for (int i = 0; i < w; ++i) before += s.wave_sum[i];
  __syncthreads();
  return before + inc - v;
}

// The workgroup's top K (K <= 128) elements, sorted descending by the 64-bit
// key (hi << 32 | lo), into s.list[0 .. K). Thread t holds positions
// E*t .. E*t + E - 1; among elements with equal hi the selection keeps the
// smallest positions (the callers make position order agree with lo order).
// Fewer than K valid elements: all of them, the rest of the list is zero.
template <int E>
__device__ void select_topk(const uint32_t (&hi)[E], const uint32_t (&lo)[E], const bool (&valid)[E], int K,
                            SelectLds& s) {
  const int t = threadIdx.x;
  uint32_t prefix = 0, need = (uint32_t)K;
  bool take_all = false;
  for (int shift = 24; shift >= 0; shift -= 8) {
    s.hist[t] = 0;  // kThreads == 256 bins
    __syncthreads();
    const uint32_t hmask = shift == 24 ? 0u : (0xFFFFFFFFu << (shift + 8));
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (valid[e] && (hi[e] & hmask) == (prefix & hmask)) atomicAdd(&s.hist[(hi[e] >> shift) & 255u], 1u);
    __syncthreads();
    if (t < 64) {
      // lane l owns bins 255 - 4l .. 252 - 4l (descending digit order)
      uint32_t c[4], sum = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        c[j] = s.hist[255 - 4 * t - j];
        sum += c[j];
      }
      uint32_t inc = sum;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(inc, o);
        if (t >= o) inc += u;
      }
      const uint32_t total = __shfl(inc, 63);
      if (shift == 24 && total <= need) {
        if (t == 0) {
          s.take_all = 1u;
          s.prefix = 0u;
          s.need = 0u;
        }
      } else {
        uint32_t before = inc - sum;
        // the digit where the running count first reaches `need`
        for (int j = 0; j < 4; ++j) {
          if (before < need && before + c[j] >= need) {
            s.take_all = 0u;
            s.prefix = prefix | ((uint32_t)(255 - 4 * t - j) << shift);
            s.need = need - before;
          }
          before += c[j];
        }
      }
    }
    __syncthreads();
    take_all = s.take_all != 0u;
    prefix = s.prefix;
    need = s.need;
    if (take_all) break;
  }
  // T = prefix is the K-th largest hi; keep every hi > T and the first `need`
  // elements (position order) with hi == T.
  uint32_t eq = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) eq += (!take_all && valid[e] && hi[e] == prefix) ? 1u : 0u;
  if (t == 0) s.n_out = 0;
  uint32_t rank = block_exclusive_scan(eq, s);  // also orders n_out's reset before the appends
  for (int e = 0; e < E; ++e) {
    if (!valid[e]) continue;
    bool keep = take_all || hi[e] > prefix;
    if (!keep && hi[e] == prefix) {
      keep = rank < need;
      ++rank;
    }
    if (keep) {
      const uint32_t slot = atomicAdd(&s.n_out, 1u);
      s.list[slot] = ((unsigned long long)hi[e] << 32) | lo[e];
    }
  }
  __syncthreads();
  const uint32_t n = s.n_out;
  int kp = 1;
  while (kp < K) kp <<= 1;
  for (int i = t; i < kp; i += kThreads)
    if ((uint32_t)i >= n) s.list[i] = 0ull;
  __syncthreads();
  // bitonic sort of kp entries, descending
  for (int size = 2; size <= kp; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (t < kp / 2) {
        const int i = 2 * t - (t & (stride - 1));
        const int j = i + stride;
        const bool desc = (i & size) == 0;
        const unsigned long long a = s.list[i], b = s.list[j];
        if ((a < b) == desc) {
          s.list[i] = b;
          s.list[j] = a;
        }
      }
      __syncthreads();
    }
  }
}

constexpr int kShort = 256;  // candidates that bounded_topk ranks
struct ShortLds {
  __attribute__((aligned(16))) uint32_t tmax[kThreads];
  unsigned long long cand[kShort];
  uint32_t bound, n;
};

// The same list by a bound: the K-th largest of the threads' own maxima is at
// most the K-th largest element, so the elements from it on (about K of them
// when the values are spread over the threads) hold the top K; they are
// compacted, and each is placed by counting the larger ones. hi[e] of an
// invalid element is 0. The maxima are compared by their upper 24 bits, then
// by thread. False (same in every thread) if more than kShort elements reach the bound - many
// equal values, or the largest ones in few threads - or if fewer than K threads
// hold any: the radix select has to take over.
template <int E>
__device__ bool bounded_topk(const uint32_t (&hi)[E], const uint32_t (&lo)[E], int K, ShortLds& b,
                             unsigned long long* list) {
  const int t = threadIdx.x;
  uint32_t m = 0;
#pragma unroll
  for (int e = 0; e < E; ++e) m = max(m, hi[e]);
  m = (m & ~255u) | (uint32_t)(255 - t);
  b.tmax[t] = m;
  if (t == 0) {
    b.bound = 0;
    b.n = 0;
  }
  __syncthreads();
  int above = 0;
#pragma unroll 8
  for (int i = 0; i < kThreads; i += 4) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(&b.tmax[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) above += v[j] > m ? 1 : 0;
  }
  if (above == K - 1) b.bound = m & ~255u;
  __syncthreads();
  const uint32_t bound = b.bound;
  if (bound == 0) return false;
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (hi[e] >= bound) {
      const uint32_t slot = atomicAdd(&b.n, 1u);
      if (slot < (uint32_t)kShort) b.cand[slot] = ((unsigned long long)hi[e] << 32) | lo[e];
    }
  __syncthreads();
  const int n = (int)b.n;
  if (n > kShort) return false;
  if (t < n) {
    const unsigned long long key = b.cand[t];
    int rank = 0;
    for (int i = 0; i < n; ++i) rank += b.cand[i] > key ? 1 : 0;
    if (rank < K) list[rank] = key;
  }
  __syncthreads();
  return true;
}

__device__ __forceinline__ float block_max(float v, float* red) {
  const int t = threadIdx.x;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  float r = red[0];
  for (int i = 1; i < kThreads / 64; ++i) r = fmaxf(r, red[i]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int t = threadIdx.x;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  if ((t & 63) == 0) red[t >> 6] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < kThreads / 64; ++i) r += red[i];
  __syncthreads();
  return r;
}

struct TreeParams {
  const float* logits;
  int ld, depth, vocab, k, budget, chunks, root, past;
  unsigned long long* part_keys;  // [depth][chunks][k]
  float2* part_ms;                // [depth][chunks] (max, sum exp(x - max))
  int* top_tok;                   // [depth][k]
  float* top_lp;                  // [depth][k]
  DtreeStepDesc* desc;
  int* tree_out;                  // optional [1 + 3 * DTREE_MAX_NODES]
  int* topk_ids;                  // optional [depth][k] copies of top_tok / top_lp
  float* topk_lp;
};

// Latency-bound. Measured, 15 rows of 151936 logits, top 24: 13.5 us by the
// bound, 22.6 by the radix select alone (its first digit, sign and exponent,
// puts most of 8192 histogram increments on a few LDS words).
__global__ __launch_bounds__(kThreads) void topk_chunk_kernel(TreeParams p) {
  __shared__ SelectLds s;
  __shared__ ShortLds b;
  __shared__ float red[kThreads / 64];
  const int row = blockIdx.y, chunk = blockIdx.x, t = threadIdx.x;
  const int base = chunk * kChunk + kE1 * t;
  const float* src = p.logits + (size_t)row * p.ld;
  float x[kE1];
  bool valid[kE1];
#pragma unroll
  for (int q = 0; q < kE1 / 4; ++q) {
    const int i = base + 4 * q;
    const bool in = i < p.vocab;  // vocab % 4 == 0: whole float4 groups
    const f32x4_t v = in ? *reinterpret_cast<const f32x4_t*>(src + i) : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x[4 * q + j] = v[j];
      valid[4 * q + j] = in;
    }
  }
  float m = -__builtin_inff();
#pragma unroll
  for (int e = 0; e < kE1; ++e)
    if (valid[e]) m = fmaxf(m, x[e]);
  m = block_max(m, red);
  float se = 0.f;
#pragma unroll
  for (int e = 0; e < kE1; ++e)
    if (valid[e] && m > -__builtin_inff()) se += expf(x[e] - m);
  se = block_sum(se, red);
  if (t == 0) p.part_ms[row * p.chunks + chunk] = make_float2(m, se);
  uint32_t hi[kE1], lo[kE1];
#pragma unroll
  for (int e = 0; e < kE1; ++e) {
    hi[e] = valid[e] ? ordered_bits(x[e]) : 0u;
    lo[e] = ~(uint32_t)(base + e);  // smaller token id sorts first among equal logits
  }
  if (!bounded_topk<kE1>(hi, lo, p.k, b, s.list)) select_topk<kE1>(hi, lo, valid, p.k, s);
  unsigned long long* dst = p.part_keys + ((size_t)row * p.chunks + chunk) * p.k;
  for (int i = t; i < p.k; i += kThreads) dst[i] = s.list[i];
}

// As above: 7.1 us for 15 rows of 19 x 24 candidates, 10.4 by the radix
// select alone.
__global__ __launch_bounds__(kThreads) void topk_merge_kernel(TreeParams p) {
  __shared__ SelectLds s;
  __shared__ ShortLds b;
  __shared__ float red[kThreads / 64];
  const int row = blockIdx.x, t = threadIdx.x;
  const int n = p.chunks * p.k;
  const unsigned long long* src = p.part_keys + (size_t)row * n;
  uint32_t hi[kE2], lo[kE2];
  // a chunk's candidates are sorted: neighbours go to different threads
#pragma unroll
  for (int e = 0; e < kE2; ++e) {
    const int i = kThreads * e + t;
    const unsigned long long key = i < n ? src[i] : 0ull;
    hi[e] = (uint32_t)(key >> 32);
    lo[e] = (uint32_t)key;
  }
  // logsumexp of the row from the chunk partials
  float mm = -__builtin_inff();
  for (int c = t; c < p.chunks; c += kThreads) mm = fmaxf(mm, p.part_ms[row * p.chunks + c].x);
  mm = block_max(mm, red);
  float ss = 0.f;
  for (int c = t; c < p.chunks; c += kThreads) {
    const float2 ms = p.part_ms[row * p.chunks + c];
    if (ms.x > -__builtin_inff()) ss += ms.y * expf(ms.x - mm);
  }
  ss = block_sum(ss, red);
  const float lse = mm + logf(ss);
  if (!bounded_topk<kE2>(hi, lo, p.k, b, s.list)) {
    bool valid[kE2];
#pragma unroll
    for (int e = 0; e < kE2; ++e) {
      const int i = kE2 * t + e;  // candidates of chunk c precede chunk c + 1's: position order = token id order
      const unsigned long long key = i < n ? src[i] : 0ull;
      hi[e] = (uint32_t)(key >> 32);
      lo[e] = (uint32_t)key;
      valid[e] = key != 0ull;
    }
    select_topk<kE2>(hi, lo, valid, p.k, s);
  }
  for (int i = t; i < p.k; i += kThreads) {
    const unsigned long long key = s.list[i];
    const int tok = (int)~(uint32_t)key;
    const float lp = from_ordered((uint32_t)(key >> 32)) - lse;
    p.top_tok[row * p.k + i] = tok;
    p.top_lp[row * p.k + i] = lp;
    if (p.topk_ids) p.topk_ids[row * p.k + i] = tok;
    if (p.topk_lp) p.topk_lp[row * p.k + i] = lp;
  }
}

// Rank tuple field of level j (1-based): r0 holds levels 1..9, r1 levels 10..18.
__device__ __forceinline__ void add_level(unsigned long long& r0, unsigned long long& r1, int level,
                                          unsigned long long v) {
  if (level <= 9)
    r0 += v << (64 - 7 * level);
  else
    r1 += v << (64 - 7 * (level - 9));
}

// A heap entry's logw as an unsigned integer of the same order (NaN: the
// smallest) and back.
__device__ __forceinline__ unsigned long long ordered_key(double x) {
  if (x != x) return 0ull;
  const unsigned long long b = (unsigned long long)__double_as_longlong(x + 0.0);  // -0 compares as +0
  return (b >> 63) ? ~b : (b | 1ull << 63);
}
__device__ __forceinline__ double key_logw(unsigned long long k) {
  return __longlong_as_double((long long)((k >> 63) ? k & ~(1ull << 63) : ~k));
}

__device__ __forceinline__ unsigned long long readlane64(unsigned long long v, int lane) {
  return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), lane) << 32) |
         (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}

// One wavefront; a serial chain of `budget` pops. Everything a pop needs is in
// registers (entry i of the heap in lane i % 64, slot i / 64 of ES; node i alike
// in NS slots) or in LDS (the top-k lists); its winner is found by DPP maxima
// over the keys' halves, and only equal keys go on to the ranks. Bound by the
// instructions of a pop, hence the slot counts as template arguments. Measured,
// 24 pops over 15 rows: 15 us with one slot, 24.4 with four; with the
// entries in LDS, shuffles of (logw, ranks, index) and the lists read from
// memory at every pop, 40 us.
template <int ES, int NS>
__global__ __launch_bounds__(64) void heap_kernel(TreeParams p) {
  constexpr int NW = 2 * NS;  // bitset words that NS slots of nodes use
  static_assert(NW <= DTREE_MASK_WORDS && 64 * NS <= DTREE_MAX_NODES, "nodes of the descriptor");
  __shared__ float s_lp[kMaxDepth * kMaxK];
  __shared__ int s_tok[kMaxDepth * kMaxK];
  const int lane = threadIdx.x;
  unsigned long long key[ES], r0[ES], r1[ES];
  int meta[ES];  // parent | depth << 8 | rank << 16; -1 = no entry
  int tok[NS], par[NS], dep[NS];
  uint32_t anc[NS][NW];
#pragma unroll
  for (int s = 0; s < ES; ++s) {
    key[s] = r0[s] = r1[s] = 0ull;
    meta[s] = -1;
  }
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    tok[s] = dep[s] = 0;
    par[s] = -1;
#pragma unroll
    for (int w = 0; w < NW; ++w) anc[s][w] = 0u;
  }
  if (lane == 0) {  // node 0, the root
    tok[0] = p.root;
    anc[0][0] = 1u;
  }
  int n_ent = 0, nodes = 0;
  if (p.budget > 0 && p.depth > 0) {
    const int n = p.depth * p.k;
#pragma unroll 8
    for (int i = lane; i < n; i += 64) {
      s_lp[i] = p.top_lp[i];
      s_tok[i] = p.top_tok[i];
    }
    __syncthreads();
    if (lane == 0) {
      key[0] = ordered_key((double)s_lp[0]);
      r0[0] = 1ull << 57;  // ranks (0,)
      meta[0] = 0 | (1 << 8) | (0 << 16);
    }
    n_ent = 1;
  }
  while (nodes < p.budget && n_ent > 0) {
    unsigned long long bk = key[0], b0 = r0[0], b1 = r1[0];
    int bm = meta[0], bs = 0;
#pragma unroll
    for (int s = 1; s < ES; ++s)
      if (n_ent > 64 * s && meta[s] >= 0 &&
          (bm < 0 || key[s] > bk || (key[s] == bk && (r0[s] < b0 || (r0[s] == b0 && r1[s] < b1))))) {
        bk = key[s];
        b0 = r0[s];
        b1 = r1[s];
        bm = meta[s];
        bs = s;
      }
    bool in = bm >= 0;
    unsigned long long win = __ballot(in);
    if (win == 0ull) break;  // heap empty
    auto narrow = [&](uint32_t v) {
      const uint32_t m = wave_umax(in ? v : 0u);
      in = in && v == m;
      win = __ballot(in);
    };
    narrow((uint32_t)(bk >> 32));
    if (win & (win - 1ull)) narrow((uint32_t)bk);
    if (win & (win - 1ull)) {  // equal logw: the smaller rank tuple
      narrow(~(uint32_t)(b0 >> 32));
      narrow(~(uint32_t)b0);
      narrow(~(uint32_t)(b1 >> 32));
      narrow(~(uint32_t)b1);
    }
    const int src = __builtin_ctzll(win);
    const double bl = key_logw(readlane64(bk, src));
    const unsigned long long w0 = readlane64(b0, src), w1 = readlane64(b1, src);
    const int m = __builtin_amdgcn_readlane(bm, src), slot = ES > 1 ? __builtin_amdgcn_readlane(bs, src) : 0;
    const int parent = m & 255, d = (m >> 8) & 255, r = m >> 16, at = (d - 1) * p.k + r;
    const int idx = ++nodes;
    const int token = s_tok[at];
    // Two new entries in two lanes' slots: the sibling with ranks[:-1] +
    // (rank + 1,) and the first child with ranks + (0,).
    const bool sib = r + 1 < p.k, child = d < p.depth;
    const int es = n_ent, ec = n_ent + (sib ? 1 : 0);
    n_ent = ec + (child ? 1 : 0);
    const bool is_c = child && lane == (ec & 63);
    const double lp_add = (double)s_lp[is_c ? d * p.k : at + (sib ? 1 : 0)];
    const double base = is_c ? bl : bl - (double)s_lp[at];
    const unsigned long long nk = ordered_key(base + lp_add);
    unsigned long long q0 = w0, q1 = w1;
    add_level(q0, q1, d + (is_c ? 1 : 0), 1ull);
    const int nm = is_c ? idx | ((d + 1) << 8) : parent | (d << 8) | ((r + 1) << 16);
    const int e = is_c ? ec : sib && lane == (es & 63) ? es : -1;
#pragma unroll
    for (int s = 0; s < ES; ++s) {
      if (slot == s && lane == src) meta[s] = -1;
      if (e >= 0 && (e >> 6) == s) {
        key[s] = nk;
        r0[s] = q0;
        r1[s] = q1;
        meta[s] = nm;
      }
    }
    uint32_t a[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      a[w] = (uint32_t)__builtin_amdgcn_readlane((int)anc[0][w], parent & 63);
#pragma unroll
      for (int s = 1; s < NS; ++s)
        if ((parent >> 6) == s) a[w] = (uint32_t)__builtin_amdgcn_readlane((int)anc[s][w], parent & 63);
      if (w == idx / 32) a[w] |= 1u << (idx % 32);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (lane + 64 * s == idx) {
        tok[s] = token;
        par[s] = parent;
        dep[s] = d;
#pragma unroll
        for (int w = 0; w < NW; ++w) anc[s][w] = a[w];
      }
  }
  // descriptor: root + nodes in pop order, rows past L cleared
  const int L = nodes + 1;
  DtreeStepDesc* dd = p.desc;
#pragma unroll
  for (int s = 0; s < DTREE_MAX_NODES / 64; ++s) {
    const int i = lane + 64 * s, sn = s < NS ? s : 0;
    const bool has = s < NS;
    dd->tokens[i] = has ? tok[sn] : 0;
    dd->positions[i] = i < L ? p.past + dep[sn] : 0;
    dd->parents[i] = has ? par[sn] : -1;
#pragma unroll
    for (int w = 0; w < DTREE_MASK_WORDS; ++w) dd->ancestors[i][w] = has && w < NW ? anc[sn][w < NW ? w : 0] : 0u;
    dd->accepted[i] = 0;
    dd->posterior[i] = 0;
    if (p.tree_out && i > 0) {
      p.tree_out[i] = has ? tok[sn] : 0;
      p.tree_out[DTREE_MAX_NODES + i] = has ? dep[sn] : 0;
      p.tree_out[2 * DTREE_MAX_NODES + i] = has ? par[sn] : -1;
    }
  }
  if (lane == 0) {
    dd->past_length = p.past;
    dd->num_nodes = L;
    dd->n_accepted = 0;
    dd->bonus_token = -1;
    if (p.tree_out) p.tree_out[0] = nodes;
  }
}

size_t tree_ws_layout(int depth, int vocab, int k, size_t* off_ms, size_t* off_tok, size_t* off_lp) {
  const int chunks = (vocab + kChunk - 1) / kChunk;
  size_t o = (size_t)depth * chunks * k * sizeof(unsigned long long);
  *off_ms = o;
  o += (size_t)depth * chunks * sizeof(float2);
  o = (o + 255) / 256 * 256;
  *off_tok = o;
  o += (size_t)depth * k * sizeof(int);
  o = (o + 255) / 256 * 256;
  *off_lp = o;
  o += (size_t)depth * k * sizeof(float);
  return (o + 255) / 256 * 256;
}

}  // namespace
}  // namespace dtree

using namespace dtree;

extern "C" size_t dtree_tree_build_workspace_bytes(int32_t depth, int32_t vocab, int32_t topk) {
  if (depth <= 0 || vocab <= 0 || topk <= 0) return 0;
  size_t a, b, c;
  return tree_ws_layout(depth, vocab, topk, &a, &b, &c);
}

extern "C" int dtree_tree_build(const float* logits, int32_t ld, int32_t depth, int32_t vocab, int32_t topk,
                                int32_t budget, int32_t root_token, int32_t past_length, void* workspace,
                                size_t workspace_bytes, DtreeStepDesc* desc, int32_t* tree_out, int32_t* topk_ids,
                                float* topk_logprobs, hipStream_t stream) {
  DTREE_REQUIRE(desc, "tree_build: null desc");
  DTREE_REQUIRE(budget >= 0 && budget <= DTREE_MAX_NODES - 1, "tree_build: budget must be in [0, 127]");
  DTREE_REQUIRE(depth >= 0 && depth <= kMaxDepth, "tree_build: depth (draft rows) must be in [0, 18]");
  DTREE_REQUIRE(past_length >= 0 && past_length <= (1 << 30) - kMaxDepth, "tree_build: past_length");
  DTREE_REQUIRE(root_token >= 0, "tree_build: root_token");
  TreeParams p{};
  p.depth = depth;
  p.budget = budget;
  p.root = root_token;
  p.past = past_length;
  p.desc = desc;
  p.tree_out = tree_out;
  p.topk_ids = topk_ids;
  p.topk_lp = topk_logprobs;
  if (budget > 0 && depth > 0) {
    DTREE_REQUIRE(logits && workspace, "tree_build: null logits / workspace");
    DTREE_REQUIRE(vocab > 0 && vocab % 4 == 0 && ld >= vocab && ld % 4 == 0 && ((uintptr_t)logits & 15) == 0,
                  "tree_build: vocab and ld multiples of 4, ld >= vocab, 16-byte aligned logits");
    DTREE_REQUIRE(topk >= 1 && topk <= kMaxK && topk <= vocab, "tree_build: topk must be in [1, min(127, vocab)]");
    const int chunks = (vocab + kChunk - 1) / kChunk;
    DTREE_REQUIRE((size_t)chunks * topk <= (size_t)kCand, "tree_build: vocab / 8192 * topk must be <= 4096");
    size_t off_ms, off_tok, off_lp;
    const size_t need = tree_ws_layout(depth, vocab, topk, &off_ms, &off_tok, &off_lp);
    DTREE_REQUIRE(workspace_bytes >= need, "tree_build: workspace too small");
    char* ws = static_cast<char*>(workspace);
    p.logits = logits;
    p.ld = ld;
    p.vocab = vocab;
    p.k = topk;
    p.chunks = chunks;
    p.part_keys = reinterpret_cast<unsigned long long*>(ws);
    p.part_ms = reinterpret_cast<float2*>(ws + off_ms);
    p.top_tok = reinterpret_cast<int*>(ws + off_tok);
    p.top_lp = reinterpret_cast<float*>(ws + off_lp);
    topk_chunk_kernel<<<dim3(chunks, depth), kThreads, 0, stream>>>(p);
    DTREE_LAUNCH_CHECK("tree_build: top-k pass");
    topk_merge_kernel<<<depth, kThreads, 0, stream>>>(p);
    DTREE_LAUNCH_CHECK("tree_build: merge pass");
  }
  // 1 + 2 budget heap entries and 1 + budget nodes, 64 to a slot
  if (budget <= 31) heap_kernel<1, 1><<<1, 64, 0, stream>>>(p);
  else if (budget <= 63) heap_kernel<2, 1><<<1, 64, 0, stream>>>(p);
  else heap_kernel<4, 2><<<1, 64, 0, stream>>>(p);
  DTREE_LAUNCH_CHECK("tree_build: heap");
  return DTREE_OK;
}
