// Causal attention of a prompt segment over the paged KV cache (the prefill's
// forward_with_hidden_states, adapters.py:494-533; custom_qwen35_model.py:
// 961-1097): one launch appends the segment's K / V rows to the cache, one
// scores every row of the segment against the prefix and the rows before it.
//
// * A workgroup is four waves of one KV group; a wave owns 32 rows of one query
//   head. The waves' (row block, head) pairs are consecutive with the head
//   fastest, so with four heads per group they share one causal range, and
//   every K / V page (64 keys) is loaded once per workgroup, straight to LDS,
//   where its MFMA fragments are contiguous kilobytes (the cache's layout).
//   The next page is in flight during the current one.
// * S^T = K Q^T and O^T = V^T P^T, as in the tree kernels: a lane owns one query
//   row, the softmax statistics are lane-local (one exchange with lane ^ 32),
//   and P goes to the second product straight from the registers of the first.
//   q and P are split pairs of bf16 (16 significant bits); K and V are the
//   cache's bf16 values.
// * Few rows over a long prefix are split over key ranges (causal_parts): a
//   workgroup walks one range of its rows' pages and leaves O, m and l in fp32
//   in the caller's workspace, and causal_combine_kernel adds the ranges.
// * Row blocks with the longest ranges start first; the groups alternate, so a
//   group's workgroups share an XCD's L2 when the groups divide the eight.
//
// Bound by the matrix cores (both products twice, for the split pairs) in the
// workgroups with the longest range: a page costs a wave 64 (D 128) or 128 MFMAs
// of 32 clocks. Measured, 32 heads of 128, 8 groups, 1000 rows, no prefix: 48 us
// + 6 us append, where a tree-attention launch per 128 rows took 194 us in eight
// launches; 16 gated heads of 256, 4 groups, 4096 rows: 369 us in one segment,
// 0.96 ms in four of 1024, where the launches per 128 rows took 1.95 ms. Key
// ranges, 8192-key prefix, without / with them: 32 heads of 128, 128 rows 281 /
// 64 us, 512 rows 293 / 170; 16 gated heads of 256, 128 rows 591 / 78 us, 512
// rows 610 / 186, 1000 rows 659 / 350 (a tree-attention launch per 128 rows: 70,
// 272; 83, 325, 673).
#include <algorithm>

#include "lds_load.h"

namespace dtree {
namespace {

constexpr float kNegInf = -1e30f;

struct CausalParams {
  const float* qkv; int ld_qkv, q_stride, k_off, v_off;
  const uint16_t* q_norm; const uint16_t* k_norm; float eps;
  const float* cos; const float* sin;  // [rows][R / 2]
  uint16_t* kp; uint16_t* vp; const int* page_table;
  uint16_t* out; uint16_t* out_lo; int ld_out, out_tiled, out_h16;
  int Hq, Hkv, past, n, rows;  // rows: n padded to whole 32-row blocks
  float scale_log2;
  int parts;  // key ranges per workgroup of rows (1: the kernel writes `out` itself)
  float* part; float* part_ml;  // of every (range, workgroup, wave): O^T fragments [32 D], m and l [2][32]
};

// Workgroup w of a group takes (row block, head) pairs 4 w .. 4 w + 3, a wave
// each; `items` pairs per group.
__host__ __device__ __forceinline__ int causal_groups(int items) { return (items + 3) / 4; }

// Pages that workgroup w's rows need (none: it has padding rows alone).
__device__ __forceinline__ int causal_tiles(const CausalParams& p, int w, int G, int items) {
  if (32 * (4 * w / G) >= p.n) return 0;
  const int rbl = min(4 * w + 3, items - 1) / G;  // the workgroup's last row block
  return (min(p.past + 32 * (rbl + 1), p.past + p.n) + DTREE_PAGE - 1) / DTREE_PAGE;
}

// Pages of one of its key ranges (the last may be shorter, ranges past it empty).
constexpr int kMinRange = 2;
__host__ __device__ __forceinline__ int causal_range(int tiles, int parts) {
  const int per = (tiles + parts - 1) / parts;
  return per > kMinRange ? per : kMinRange;
}

// A lane's values of dims 32 db .. of its row: scaled, gated, stored.
template <int D, bool GATED>
__device__ __forceinline__ void causal_store(const CausalParams& p, const f32x16_t& o, float inv, int row, int hq, int db,
                                             int h) {
  const bool valid = row < p.n;
  const float* gate = p.qkv + (size_t)row * p.ld_qkv + hq * p.q_stride + D;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int d = 32 * db + 8 * q + 4 * h;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = valid ? o[4 * q + e] * inv : 0.f;
    if constexpr (GATED) {
      const f32x4_t gt = *reinterpret_cast<const f32x4_t*>(gate + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = valid ? y[e] / (1.0f + __expf(-gt[e])) : 0.f;
    }
    const int col = hq * D + d;
    const size_t oi = p.out_tiled ? tiled_index(row, col, p.ld_out) : (size_t)row * p.ld_out + col;
    store_act4(p.out, p.out_lo, oi, y, p.out_h16);
  }
}

// K / V rows of the segment into the cache. A workgroup owns one page of one KV
// head: four threads per K row (RMSNorm, RoPE pairs inside a thread, 16-byte
// runs of 8 dims), then 8-position runs of one V dim per thread.
template <int D, int R>
__global__ __launch_bounds__(256) void causal_append_kernel(CausalParams p) {
  const int pg = p.past / DTREE_PAGE + blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  const size_t blk = ((size_t)p.page_table[pg] * p.Hkv + g) * (DTREE_PAGE * D);
  const int first = pg * DTREE_PAGE - p.past;  // segment row of slot 0
  {
    const int slot = tid >> 2, j = tid & 3, row = first + slot;
    const bool in = row >= 0 && row < p.n;
    const int rr = in ? row : 0;
    constexpr int RP = R / 8;          // rotated pairs per thread: dims RP j .. and R / 2 + RP j ..
    constexpr int NP = (D - R) / 4;    // unrotated dims per thread
    constexpr int NV = 2 * RP + NP;
    auto dim = [&](int i) { return i < RP ? RP * j + i : i < 2 * RP ? R / 2 + RP * j + i - RP : R + NP * j + i - 2 * RP; };
    const float* src = p.qkv + (size_t)rr * p.ld_qkv + p.k_off + g * D;
    float v[NV], ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i += 4) {
      const f32x4_t x = *reinterpret_cast<const f32x4_t*>(src + dim(i));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[i + e] = x[e];
    }
    if (p.k_norm) {
#pragma unroll
      for (int i = 0; i < NV; ++i) ss += v[i] * v[i];
      ss += dpp<0xB1>(ss);
      ss += dpp<0x4E>(ss);
      const float rs = rsqrtf(ss * (1.0f / D) + p.eps);
#pragma unroll
      for (int i = 0; i < NV; ++i) v[i] *= rs * bf2f(p.k_norm[dim(i)]);
    }
#pragma unroll
    for (int i = 0; i < RP; ++i) {
      const float cs = p.cos[(size_t)rr * (R / 2) + RP * j + i], sn = p.sin[(size_t)rr * (R / 2) + RP * j + i];
      const float a = v[i], b = v[RP + i];
      v[i] = a * cs - b * sn;
      v[RP + i] = a * sn + b * cs;
    }
    if (in) {
#pragma unroll
      for (int i = 0; i < NV; i += 8)
        *reinterpret_cast<u32x4_t*>(p.kp + blk + kv_k_off(slot, dim(i), D)) =
            u32x4_t{pack_bf2(v[i], v[i + 1]), pack_bf2(v[i + 2], v[i + 3]), pack_bf2(v[i + 4], v[i + 5]),
                    pack_bf2(v[i + 6], v[i + 7])};
    }
  }
#pragma unroll
  for (int u = tid; u < 8 * D; u += 256) {
    const int s0 = 8 * (u / D), d = u % D, r0 = first + s0;
    if (r0 + 7 < 0 || r0 >= p.n) continue;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int row = min(max(r0 + e, 0), p.n - 1);
      v[e] = p.qkv[(size_t)row * p.ld_qkv + p.v_off + g * D + d];
    }
    uint16_t* o = p.vp + blk + kv_v_off(s0, d, D);
    if (r0 >= 0 && r0 + 7 < p.n) {
      *reinterpret_cast<u32x4_t*>(o) =
          u32x4_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (r0 + e >= 0 && r0 + e < p.n) o[e] = f2bf(v[e]);
    }
  }
}

// v = hi + lo, eight bf16 pairs.
__device__ __forceinline__ void split_pair8(const float (&v)[8], u32x4_t& hi, u32x4_t& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = v[2 * i], b = v[2 * i + 1];
    hi[i] = pack_bf2(a, b);
    lo[i] = pack_bf2(a - __uint_as_float(hi[i] << 16), b - __uint_as_float(hi[i] & 0xffff0000u));
  }
}

// Zeroes the keys of a V^T fragment from `end` on (first: the fragment's first
// key): cache slots past the segment may hold anything, and 0 * NaN is NaN.
__device__ __forceinline__ u32x4_t clip_keys(u32x4_t v, int first, int end) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v[i] &= (first + 2 * i < end ? 0xffffu : 0u) | (first + 2 * i + 1 < end ? 0xffff0000u : 0u);
  return v;
}

// SPLIT: one of p.parts key ranges of the rows, to the workspace.
template <int D, int R, bool GATED, bool SPLIT>
__global__ __launch_bounds__(256, D == 128 ? 2 : 1) void causal_attn_kernel(CausalParams p) {
  constexpr int NJ = D / 16, ND = D / 32, PB = DTREE_PAGE * D * 2;  // bytes of a page's K (or V)
  constexpr int PW = 2 * PB / 1024 / 4;                             // 1 KB pieces per wave and page
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2][2 * PB];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // key ranges cover the live rows alone (causal_combine_kernel writes all rows)
  const int G = p.Hq / p.Hkv, items = G * ((SPLIT ? p.n + 31 : p.rows) / 32), nw = causal_groups(items);
  const int g = blockIdx.x % p.Hkv, b = blockIdx.x / p.Hkv, part = SPLIT ? b % p.parts : 0;
  const int w = nw - 1 - (SPLIT ? b / p.parts : b);
  const int item = 4 * w + wave, rb = item / G, hq = g * G + item % G;
  const int row0 = 32 * rb, row = row0 + c;
  const bool live = item < items && row0 < p.n;
  const int end = p.past + p.n;                                         // keys in the cache
  const int kend = live ? min(p.past + row0 + 32, end) : 0;             // keys this wave needs
  int first = 0, tiles = causal_tiles(p, w, G, items);
  if constexpr (SPLIT) {
    const int per = causal_range(tiles, p.parts);
    first = part * per;
    tiles = min(tiles, first + per);
    if (first >= tiles) return;  // (uniform; the ranges are counted alike in the combine)
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&smem[0][0];
  auto issue = [&](int t) {
    const size_t blk = ((size_t)p.page_table[t] * p.Hkv + g) * (DTREE_PAGE * D);
    const u32x4_t kr = strip_rsrc(p.kp + blk, PB), vr = strip_rsrc(p.vp + blk, PB);
    const unsigned lds = lds0 + (t & 1) * (2 * PB) + wave * (PW * 512);
#pragma unroll
    for (int i = 0; i < PW / 2; ++i) lds_load16(kr, wave * (PW * 512) + 1024 * i + 16 * lane, lds + 1024 * i);
#pragma unroll
    for (int i = 0; i < PW / 2; ++i) lds_load16(vr, wave * (PW * 512) + 1024 * i + 16 * lane, lds + PB + 1024 * i);
  };
  if (first < tiles) issue(first);
  // This lane's dims 16 j + 8 h .. + 7 of its query row: q_norm, RoPE (pairs j,
  // j + R / 32 in one lane), softmax scale in log2 units, split.
  u32x4_t qh[NJ], ql[NJ];
  if (live) {
    const float* src = p.qkv + (size_t)row * p.ld_qkv + hq * p.q_stride + 8 * h;
    float q[NJ][8];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4_t a = *reinterpret_cast<const f32x4_t*>(src + 16 * j);
      const f32x4_t b = *reinterpret_cast<const f32x4_t*>(src + 16 * j + 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[j][i] = a[i];
        q[j][4 + i] = b[i];
      }
    }
    if (p.q_norm) {
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += q[j][i] * q[j][i];
      ss += __shfl_xor(ss, 32);
      const float rs = rsqrtf(ss * (1.0f / D) + p.eps);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        u32x4_t nwv;  // (a weight at any 2-byte address, as the tree kernels take it)
        __builtin_memcpy(&nwv, p.q_norm + 16 * j + 8 * h, sizeof(nwv));
#pragma unroll
        for (int i = 0; i < 8; ++i)
          q[j][i] *= rs * __uint_as_float((i & 1) ? (nwv[i >> 1] & 0xffff0000u) : (nwv[i >> 1] << 16));
      }
    }
#pragma unroll
    for (int j = 0; j < R / 32; ++j) {
      const float* cp = p.cos + (size_t)row * (R / 2) + 16 * j + 8 * h;
      const float* sp = p.sin + (size_t)row * (R / 2) + 16 * j + 8 * h;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float a = q[j][i], b = q[j + R / 32][i], cs = cp[i], sn = sp[i];
        q[j][i] = a * cs - b * sn;
        q[j + R / 32][i] = a * sn + b * cs;
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
#pragma unroll
      for (int i = 0; i < 8; ++i) q[j][i] *= p.scale_log2;
      split_pair8(q[j], qh[j], ql[j]);
    }
  }
  f32x16_t o[ND];
#pragma unroll
  for (int db = 0; db < ND; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  float m_run = kNegInf, l_run = 0.f;
  for (int t = first; t < tiles; ++t) {
    stage_wait<0>();  // page t has landed for every wave, and every wave has read page t - 1
    if (t + 1 < tiles) issue(t + 1);
    const int k0 = DTREE_PAGE * t;
    if (k0 >= kend) continue;
    const unsigned char* kb = smem[t & 1] + 16 * lane;
    const unsigned char* vb = kb + PB;
    f32x16_t s[2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[b][r] = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const u32x4_t kf = *reinterpret_cast<const u32x4_t*>(kb + (b * NJ + j) * 1024);
        s[b] = mfma32(kf, qh[j], s[b]);
        s[b] = mfma32(kf, ql[j], s[b]);
      }
    // register r of block b: key k0 + 32 b + 16 (r / 8) + 8 h + r % 8
    if (k0 + DTREE_PAGE > p.past + row0) {
      const int lim = p.past + row - k0 - 8 * h;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * b + 16 * (r >> 3) + (r & 7) > lim) s[b][r] = kNegInf;
    }
    float mx = kNegInf;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[b][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (__any(mx > m_run)) {  // some row's maximum grew: rescale
      const float m_new = fmaxf(m_run, mx), alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < ND; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    }
    const bool clip = k0 + DTREE_PAGE > end;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pv[e] = fast_exp2(s[st >> 1][8 * (st & 1) + e] - m_run);
        l_run += pv[e];
      }
      u32x4_t ph, pl;
      split_pair8(pv, ph, pl);
#pragma unroll
      for (int db = 0; db < ND; ++db) {
        u32x4_t vf = *reinterpret_cast<const u32x4_t*>(vb + (st * ND + db) * 1024);
        if (clip) vf = clip_keys(vf, k0 + 16 * st + 8 * h, end);
        o[db] = mfma32(vf, ph, o[db]);
        o[db] = mfma32(vf, pl, o[db]);
      }
    }
  }
  if (item >= items) return;
  const float l = l_run + __shfl_xor(l_run, 32);
  if constexpr (SPLIT) {
    const size_t u = ((size_t)(part * nw + w) * p.Hkv + g) * 4 + wave;
    f32x4_t* po = reinterpret_cast<f32x4_t*>(p.part + u * (32 * D)) + lane;
#pragma unroll
    for (int db = 0; db < ND; ++db)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        po[(4 * db + q) * 64] = f32x4_t{o[db][4 * q], o[db][4 * q + 1], o[db][4 * q + 2], o[db][4 * q + 3]};
    p.part_ml[u * 64 + lane] = h ? l : m_run;
    return;
  }
  const float inv = row < p.n ? 1.f / l : 0.f;
#pragma unroll
  for (int db = 0; db < ND; ++db) causal_store<D, GATED>(p, o[db], inv, row, hq, db, h);
}

// The key ranges' partial results into `out`: a wave per 32 dims of a (row
// block, head) pair, the lanes as in the kernel above, so every partial is read
// as whole kilobytes. A range whose keys lie past a row contributes nothing to
// it (its weight is 0 next to the first range's, which holds key 0).
template <int D, bool GATED>
__global__ __launch_bounds__(256) void causal_combine_kernel(CausalParams p) {
  constexpr int ND = D / 32;
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);  // (row block, head, dims), dims fastest
  const int db = unit % ND, hq = unit / ND % p.Hq, rb = unit / ND / p.Hq;
  if (32 * rb >= p.rows) return;
  const int G = p.Hq / p.Hkv, g = hq / G, item = rb * G + hq % G, items = G * ((p.n + 31) / 32);
  const int nw = causal_groups(items), w = item / 4, row = 32 * rb + c;
  f32x16_t o;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[r] = 0.f;
  float inv = 0.f;
  if (32 * rb < p.n) {
    const int all = causal_tiles(p, w, G, items), per = causal_range(all, p.parts), used = (all + per - 1) / per;
    const size_t u0 = ((size_t)w * p.Hkv + g) * 4 + item % 4, du = (size_t)nw * p.Hkv * 4;
    const float* ml = p.part_ml + u0 * 64 + c;
    float m = kNegInf, l = 0.f;
#pragma unroll 4
    for (int s = 0; s < used; ++s) m = fmaxf(m, ml[s * du * 64]);
    const f32x4_t* po = reinterpret_cast<const f32x4_t*>(p.part + u0 * (32 * D)) + 256 * db + lane;
#pragma unroll 4
    for (int s = 0; s < used; ++s) {
      const float k = fast_exp2(ml[s * du * 64] - m);
      l += k * ml[s * du * 64 + 32];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4_t v = po[s * du * (8 * D) + 64 * q];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[4 * q + e] = fmaf(k, v[e], o[4 * q + e]);
      }
    }
    inv = row < p.n ? 1.f / l : 0.f;
  }
  causal_store<D, GATED>(p, o, inv, row, hq, db, h);
}

__global__ __launch_bounds__(256) void rope_positions_kernel(int first, int rows, int half, float base, float* cos_out,
                                                             float* sin_out) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= rows * half) return;
  const int m = e / half, i = e % half;
  const double inv = exp(-log((double)base) * (2.0 * i) / (2.0 * half));
  const double ang = (double)(first + m) * inv;
  cos_out[e] = (float)cos(ang);
  sin_out[e] = (float)sin(ang);
}

// Workgroups that fill an MI355X's 256 CUs once. A workgroup walks its pages one
// after another and uses its CU's matrix cores by itself (head_dim 128, 2048 rows
// over 8192 keys: two on every CU, 4.2 us a page; 300 rows, one on a third of
// them: 2.1), so rows that leave CUs idle are split over key ranges up to this
// many workgroups.
constexpr int kFill = 256;

// Workspace of one key range of every workgroup.
size_t causal_part_bytes(int D, int groups) { return (size_t)groups * 4 * (32 * D + 64) * sizeof(float); }

// Ranges pay once they save more than the second kernel costs, about 5 us: two
// pages' walk at head_dim 256 (4.5 us a page; 5 pages, 300 rows: 52 -> 40 us),
// four at 128 (2.1 us; 13 pages, 300 rows: 40 -> 35, but 5 pages 24.5 -> 27.8).
int causal_parts(int D, int groups, int past, int n) {
  const int pages = (past + n + DTREE_PAGE - 1) / DTREE_PAGE;
  if (pages < (D == 128 ? 8 : 4)) return 1;
  return std::max(1, std::min(kFill / groups, pages / kMinRange));
}

}  // namespace
}  // namespace dtree

using namespace dtree;

extern "C" int dtree_rope_positions(int32_t first_position, int32_t rows, int32_t rope_dims, float rope_base,
                                    float* rope_cos, float* rope_sin, hipStream_t stream) {
  DTREE_REQUIRE(rope_cos && rope_sin, "rope_positions: null pointer");
  DTREE_REQUIRE(first_position >= 0 && rows > 0 && rows <= (1 << 20), "rope_positions: first_position >= 0, rows");
  DTREE_REQUIRE(rope_dims > 0 && rope_dims % 2 == 0 && rope_dims <= 1024, "rope_positions: rope_dims");
  const int n = rows * (rope_dims / 2);
  rope_positions_kernel<<<(n + 255) / 256, 256, 0, stream>>>(first_position, rows, rope_dims / 2, rope_base, rope_cos,
                                                              rope_sin);
  DTREE_LAUNCH_CHECK("rope_positions launch");
  return DTREE_OK;
}

extern "C" size_t dtree_causal_attention_workspace_bytes(int32_t head_dim) {
  return head_dim > 0 ? causal_part_bytes(head_dim, kFill) : 0;
}

extern "C" int dtree_causal_attention_split(const DtreeAttnArgs* a, int32_t past_length, int32_t num_rows,
                                            void* workspace, size_t workspace_bytes, hipStream_t stream) {
  DTREE_REQUIRE(a, "causal_attention: null args");
  DTREE_REQUIRE(a->qkv && a->rope_cos && a->rope_sin && a->k_pages && a->v_pages && a->page_table && a->out,
                "causal_attention: null pointer");
  const int D = a->head_dim, R = a->rope_dims ? a->rope_dims : D;
  DTREE_REQUIRE((D == 128 && R == 128 && !a->gated) || (D == 256 && R == 64 && a->gated),
                "causal_attention: head_dim 128 with 128 rotary dims, or gated head_dim 256 with 64, are compiled");
  DTREE_REQUIRE(a->num_kv_heads > 0 && a->num_heads > 0 && a->num_heads % a->num_kv_heads == 0,
                "causal_attention: num_heads % num_kv_heads");
  const int G = a->num_heads / a->num_kv_heads;  // the groups the tree steps take
  DTREE_REQUIRE(G == 2 || G == 4 || (G == 8 && D == 128), "causal_attention: GQA group of 2, 4 or 8 (8: head_dim 128)");
  DTREE_REQUIRE(past_length >= 0 && num_rows >= 1 && a->rows_padded >= num_rows && a->rows_padded % 32 == 0 &&
                    a->rows_padded <= (1 << 20) && past_length <= (1 << 28),
                "causal_attention: num_rows in [1, rows_padded], rows_padded a multiple of 32");
  const int qs = a->gated ? 2 * D : D;
  const int width = a->num_heads * qs + 2 * a->num_kv_heads * D;
  DTREE_REQUIRE(a->ld_qkv >= width && a->ld_qkv % 4 == 0 && ((uintptr_t)a->qkv & 15) == 0,
                "causal_attention: qkv rows of [q | k | v] heads, 16-byte aligned");
  DTREE_REQUIRE(((uintptr_t)a->k_pages & 15) == 0 && ((uintptr_t)a->v_pages & 15) == 0,
                "causal_attention: the pages must be 16-byte aligned");
  const int od = a->num_heads * D;
  DTREE_REQUIRE(((uintptr_t)a->out & 7) == 0 && ((uintptr_t)a->out_lo & 7) == 0 &&
                    (a->out_layout == DTREE_W_ROWMAJOR ? a->ld_out >= od && a->ld_out % 4 == 0
                                                       : (a->out_layout == DTREE_W_TILED ||
                                                          a->out_layout == DTREE_W_TILED_F16) &&
                                                             a->ld_out == od),
                "causal_attention: out layout (8-byte aligned; tiled needs ld_out == num_heads * head_dim)");
  CausalParams p{};
  p.qkv = a->qkv; p.ld_qkv = a->ld_qkv; p.q_stride = qs;
  p.k_off = a->num_heads * qs; p.v_off = p.k_off + a->num_kv_heads * D;
  p.q_norm = a->q_norm; p.k_norm = a->k_norm; p.eps = a->eps; p.cos = a->rope_cos; p.sin = a->rope_sin;
  p.kp = a->k_pages; p.vp = a->v_pages; p.page_table = a->page_table;
  p.out_h16 = a->out_layout == DTREE_W_TILED_F16;
  p.out = a->out; p.out_lo = p.out_h16 ? nullptr : a->out_lo; p.ld_out = a->ld_out;
  p.out_tiled = a->out_layout != DTREE_W_ROWMAJOR;
  p.Hq = a->num_heads; p.Hkv = a->num_kv_heads; p.past = past_length; p.n = num_rows; p.rows = a->rows_padded;
  p.scale_log2 = a->scale * 1.4426950408889634f;
  const int live = causal_groups(G * ((num_rows + 31) / 32)) * p.Hkv;
  p.parts = causal_parts(D, live, past_length, num_rows);
  // without room for two ranges, one: the kernel then needs no workspace
  const size_t fit = workspace && ((uintptr_t)workspace & 15) == 0 ? workspace_bytes / causal_part_bytes(D, live) : 0;
  if ((size_t)p.parts > fit) p.parts = std::max(1, (int)fit);
  p.part = static_cast<float*>(workspace);
  if (p.part) p.part_ml = p.part + (size_t)p.parts * live * 4 * (32 * D);
  const int pages = (past_length + num_rows - 1) / DTREE_PAGE - past_length / DTREE_PAGE + 1;
  const dim3 agrid(pages, p.Hkv);
  const int grid = p.parts > 1 ? live * p.parts : causal_groups(G * (p.rows / 32)) * p.Hkv;
  const int cgrid = (p.rows / 32 * p.Hq * (D / 32) + 3) / 4;
  if (D == 128) {
    causal_append_kernel<128, 128><<<agrid, 256, 0, stream>>>(p);
    DTREE_LAUNCH_CHECK("causal_attention append launch");
    if (p.parts == 1) causal_attn_kernel<128, 128, false, false><<<grid, 256, 0, stream>>>(p);
    else causal_attn_kernel<128, 128, false, true><<<grid, 256, 0, stream>>>(p);
    if (p.parts > 1) causal_combine_kernel<128, false><<<cgrid, 256, 0, stream>>>(p);
  } else {
    causal_append_kernel<256, 64><<<agrid, 256, 0, stream>>>(p);
    DTREE_LAUNCH_CHECK("causal_attention append launch");
    if (p.parts == 1) causal_attn_kernel<256, 64, true, false><<<grid, 256, 0, stream>>>(p);
    else causal_attn_kernel<256, 64, true, true><<<grid, 256, 0, stream>>>(p);
    if (p.parts > 1) causal_combine_kernel<256, true><<<cgrid, 256, 0, stream>>>(p);
  }
  DTREE_LAUNCH_CHECK("causal_attention launch");
  return DTREE_OK;
}

extern "C" int dtree_causal_attention(const DtreeAttnArgs* a, int32_t past_length, int32_t num_rows,
                                      hipStream_t stream) {
  return dtree_causal_attention_split(a, past_length, num_rows, nullptr, 0, stream);
}
