// Long-M GEMM Y[M, N] = X[M, K] * W[N, K]^T for the prompt prefill (rows a
// multiple of 128), dense weights. Compute-bound: the design goal is MFMA
// issue, so the tile, not the weight stream, is what each workgroup shares.
//
// * Both operands are in the tiled layout (32-row x 64-column blocks, four
//   1 KB MFMA fragments in lane order), so a fragment goes from memory to LDS
//   by one direct 16-byte-per-lane load of one wave and from LDS to registers
//   by one contiguous 16-byte read: no staging registers, no bank conflicts.
// * A stage is half a K block (32 K: two fragments of every row and column
//   block). NST stages are in LDS; the loads of stage s + NST - 1 are issued
//   when stage s starts, and the only waits are for the stage two fragments
//   ahead, with the younger stages' loads left in flight.
// * Fragments are read from LDS one step (one fragment index) ahead of their
//   MFMAs into a second register set, so a wave's LDS reads, its barrier and
//   its stage wait lie under the previous step's MFMAs.
// * The MFMA is issued as W * X^T: a lane then holds four consecutive output
//   columns of one row per accumulator quad, so the epilogues run from the
//   registers: 16-byte fp32 rows, 8-byte activation pieces that are
//   contiguous across lanes in the tiled layout, the SwiGLU partner in the
//   same lane and the row's sum of squares one lane exchange away.
// * Narrow outputs (fewer tiles than CUs) run eight waves on a 128 x 128 tile,
//   two groups of four on the two halves of every K block: two waves per SIMD
//   cover each other's waits (N 2560, K 9728, 1024 rows: 79 us with four
//   waves, 65 with eight).
//
// Bound by MFMA issue on the wide tiles (a 256 x 256 tile with no loads at all
// takes 85 % of its time; the card's clock falls to about 2 GHz under it) and by
// the ~100 GB/s a CU loads on the narrow ones. Measured against the kernel
// this one replaced (128 x 128 tiles staged through registers, one barrier per
// 64 K): Qwen3-4B's gate/up and down over 1024 rows 368 -> 197 us (0.42 ->
// 0.79 PFLOP/s); N 24576, K 4096, 4096 rows 1403 -> 699 us (1.18 PFLOP/s).
#include "gemm_long.h"

namespace dtree {
namespace {

// Tile of a workgroup: GM x GN waves, each MB x NB 32 x 32 blocks, KS times:
// with KS = 2 a second group of waves takes the other half of every K block.
template <int MB_, int NB_, int GM_, int GN_, int NST_, int KS_ = 1>
struct Tile {
  static constexpr int MB = MB_, NB = NB_, GM = GM_, GN = GN_, NST = NST_, KS = KS_;
  static constexpr int WAVES = GM * GN * KS, THREADS = 64 * WAVES;
  static constexpr int TM = 32 * MB * GM, TN = 32 * NB * GN;
};

constexpr int kSub = 2;  // fragments per row / column block that a wave reads of a stage

// Direct load of 16 bytes per lane into LDS (lane l's land at lds + 16 l).
// Offsets past the resource's size read zero without a memory access. Not the
// builtin: the compiler would order every later LDS read behind all such
// loads; the stage waits below do it by count. The load has no register
// result, and the callers wait for it before its LDS is read or released.
// s_nop 4 covers m0 and a resource word that a VALU lane read has just written.
__device__ __forceinline__ int uni(uint32_t v) { return __builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ void lds_load16(u32x4_t r, unsigned off, unsigned lds_addr) {
  typedef int s32x4_t __attribute__((ext_vector_type(4)));
  const s32x4_t rsrc = s32x4_t{uni(r[0]), uni(r[1]), uni(r[2]), uni(r[3])};
  const int lds = uni(lds_addr);
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds), "v"(off), "s"(rsrc) : "memory");
}

// This wave's loads but the N youngest have landed and its LDS reads are done;
// then the workgroup barrier.
template <int N>
__device__ __forceinline__ void stage_wait() {
  static_assert(N <= 63, "vmcnt is 6 bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

__device__ __forceinline__ u32x4_t strip_rsrc(const void* p, unsigned bytes) {
  const uint64_t a = (uint64_t)p;
  return u32x4_t{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32) & 0xffff),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

template <bool VEC>
__device__ __forceinline__ void st4f(float* p, const float (&v)[4]) {
  if constexpr (VEC) {
    *reinterpret_cast<f32x4_t*>(p) = f32x4_t{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = v[i];
  }
}

// Four consecutive activations of row m from column col (col % 4 == 0; they
// lie in one 8-element run of the tiled layout).
template <bool VEC>
__device__ __forceinline__ void st4_act(const LongParams& p, int m, int col, const float (&v)[4]) {
  const size_t oi = p.out_tiled ? tiled_index(m, col, p.ld_out_bf16) : (size_t)m * p.ld_out_bf16 + col;
  if constexpr (VEC) {
    store_act4(p.out_bf16, p.out_lo, oi, v, p.out_h16);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (p.out_h16) {
      p.out_bf16[oi + i] = f2h(v[i]);
    } else {
      const uint16_t hi = f2bf(v[i]);
      p.out_bf16[oi + i] = hi;
      if (p.out_lo) p.out_lo[oi + i] = f2bf(v[i] - bf2f(hi));
    }
  }
}

// Epilogue of one wave's MB x NB accumulator blocks: block (j, i) holds
// columns n0 + 32 j + 8 q + 4 h + e (register 4 q + e) of row m0 + 32 i + c.
template <int NB, int MB, int EPI, bool VEC>
__device__ __forceinline__ void long_epilogue(const LongParams& p, f32x16_t (&acc)[NB][MB], const float* rs,
                                              int R, int mw, int n0) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int rb = R + mw + 32 * i;  // rows of this block
    if (rb >= p.rows) break;
    const int m = rb + c;
    if constexpr (EPI == DTREE_EPI_RESIDUAL) {
      // the block row's residuals in flight together
      f32x4_t xo[NB][4];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        if (n0 + 32 * j >= p.n) break;
        const float* xp = p.out_f32 + (size_t)m * p.ld_out_f32 + n0 + 32 * j + 4 * h;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (VEC) xo[j][q] = *reinterpret_cast<const f32x4_t*>(xp + 8 * q);
          else xo[j][q] = f32x4_t{xp[8 * q], xp[8 * q + 1], xp[8 * q + 2], xp[8 * q + 3]};
        }
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int cb = n0 + 32 * j;
        if (cb >= p.n) break;
        float sq = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int col = cb + 8 * q + 4 * h;
          float g[4], xv[4], xg[4];
          if constexpr (VEC) {
            const u32x2_t gw = *reinterpret_cast<const u32x2_t*>(p.next_norm + col);
#pragma unroll
            for (int e = 0; e < 4; ++e) g[e] = bf2f((uint16_t)(gw[e >> 1] >> (16 * (e & 1))));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) g[e] = bf2f(p.next_norm[col + e]);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            xv[e] = xo[j][q][e] + acc[j][i][4 * q + e];
            xg[e] = xv[e] * g[e];
            sq += xv[e] * xv[e];
          }
          st4f<VEC>(p.out_f32 + (size_t)m * p.ld_out_f32 + col, xv);
          st4_act<VEC>(p, m, col, xg);
          if (p.hidden_out) {
            uint16_t* hp = p.hidden_out + (size_t)m * p.ld_hidden + col;
            if constexpr (VEC) {
              *reinterpret_cast<u32x2_t*>(hp) = u32x2_t{pack_bf2(xv[0], xv[1]), pack_bf2(xv[2], xv[3])};
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e) hp[e] = f2bf(xv[e]);
            }
          }
        }
        sq += __shfl_xor(sq, 32);
        if (h == 0) p.ss_out[ss_index(cb >> 5, m, p.n >> 5)] = sq;
      }
    } else {
      const float r = rs[mw + 32 * i + c];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int cb = n0 + 32 * j;
        if (cb >= p.n) break;
        if constexpr (EPI == DTREE_EPI_SWIGLU) {
          // 16 gate rows then 16 up rows of the weight per 32 columns
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[e] = silu_f(acc[j][i][4 * q + e] * r) * (acc[j][i][8 + 4 * q + e] * r);
            st4_act<VEC>(p, m, (cb >> 1) + 8 * q + 4 * h, v);
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int col = cb + 8 * q + 4 * h;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = acc[j][i][4 * q + e] * r;
            if constexpr (EPI == DTREE_EPI_STORE_F32) st4f<VEC>(p.out_f32 + (size_t)m * p.ld_out_f32 + col, v);
            else st4_act<VEC>(p, m, col, v);
          }
        }
      }
    }
  }
}

// RMSNorm row scales of the tile's rows into rs: wave w takes row blocks w,
// w + WAVES, ..; the two half-waves take alternate statistics tiles.
template <class T>
__device__ __forceinline__ void long_row_scale(const LongParams& p, int R, int wave, float* rs) {
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  for (int b = wave; b < T::TM / 32; b += T::WAVES) {
    float r = 1.f;
    if (p.ss_in && R + 32 * b < p.rows) {
      const float* s = p.ss_in + ss_index(0, R + 32 * b, p.ss_tiles) + c;
      float a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = 0.f;
      int t = h;
      for (; t + 14 < p.ss_tiles; t += 16)
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] += s[(size_t)(t + 2 * u) * 32];
      for (; t < p.ss_tiles; t += 2) a[0] += s[(size_t)t * 32];
      float tot = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
      tot += __shfl_xor(tot, 32);
      r = rsqrtf(tot * p.inv_norm_dim + p.eps);
    }
    if (h == 0) rs[32 * b + c] = r;
  }
}

// Tile of workgroup b, as (row tile, column tile). The tiles are cut into one
// contiguous run per XCD (workgroups go round-robin over the eight) of an
// order that walks bands of kBand rows: column tile by column tile, rows
// fastest. The 32 tiles an XCD runs at a time then share their row and column
// strips about evenly through its L2.
constexpr int kBand = 1024;
__device__ __forceinline__ int2 xcd_tile(int b, int tiles, int ntn, int tm) {
  const int x = b & 7, i = b >> 3, q = tiles >> 3, r = tiles & 7;
  const int id = x * q + min(x, r) + i;
  const int ntm = tiles / ntn, bm = kBand / tm;  // row tiles, and per band
  const int band = id / (bm * ntn), in = id - band * bm * ntn;
  const int rows = min(bm, ntm - band * bm);     // row tiles of this band
  const int nt = in / rows;
  return int2{band * bm + in - nt * rows, nt};
}

template <class T, int EPI, bool H, int NPL>
__global__ __launch_bounds__(T::THREADS) void long_kernel(LongParams p) {
  constexpr int MB = T::MB, NB = T::NB, NST = T::NST;
  constexpr int KS = T::KS, SUB = kSub * KS;                           // fragments per block and stage
  constexpr int ACH = T::TM / 32 * NPL * SUB, BCH = T::TN / 32 * SUB;  // 1 KB pieces per stage
  constexpr int CH = ACH + BCH, STAGE = CH * 1024;
  constexpr int PW = (CH + T::WAVES - 1) / T::WAVES;  // pieces per wave (the last may be padding)
  constexpr bool PAD = CH % T::WAVES != 0;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NST * STAGE + (PAD ? 1024 : 0)];
  __shared__ float rs[T::TM];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kg = KS > 1 ? wave / (T::GM * T::GN) : 0, wt = wave - kg * (T::GM * T::GN);
  const int wm = wt / T::GN, wn = wt % T::GN;
  const int2 mn = xcd_tile(blockIdx.x, p.tiles, p.ntn, T::TM);
  const int R = mn.x * T::TM, N0 = mn.y * T::TN;
  const int nkb = p.k >> 6, S = p.k / (16 * SUB);
  const unsigned strip = (unsigned)nkb * 4096u;  // bytes of one 32-row strip
  const size_t xo = (size_t)R * p.k, wo = (size_t)N0 * p.k;
  const unsigned xbytes = (unsigned)min(T::TM, p.rows - R) / 32u * strip;
  const u32x4_t xr = strip_rsrc(p.x + xo, xbytes);
  const u32x4_t xlr = strip_rsrc((NPL > 1 ? p.x_lo : p.x) + xo, xbytes);
  const u32x4_t wr = strip_rsrc(p.w + wo, (unsigned)min(T::TN, p.n - N0) / 32u * strip);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  // Piece wave + WAVES j of stage s: activation pieces (plane, row block,
  // fragment), then weight pieces (column block, fragment). Past the last
  // stage or piece the load reads nothing, so every wave always has the same
  // number in flight.
  auto issue = [&](int s, int j) {
    const int ch = wave + T::WAVES * j;
    const bool isa = ch < ACH, pad = PAD && ch >= CH;
    const int a = isa ? ch : ch - ACH;
    const int plane = NPL > 1 && isa && a >= ACH / NPL;
    const int ap = plane ? a - ACH / NPL : a;
    const unsigned off = (unsigned)(ap / SUB) * strip + (unsigned)(ap % SUB + SUB * s) * 1024u;
    const unsigned lds = lds0 + (pad ? (unsigned)(NST * STAGE) : (unsigned)((s % NST) * STAGE + 1024 * ch));
    lds_load16(isa ? (plane ? xlr : xr) : wr, (s < S && !pad ? off : kOob) + 16u * lane, lds);
  };
  f32x16_t acc[NB][MB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;
  u32x4_t fa[2][MB * NPL], fb[2][NB];
  // fragment r of step (s, f) into register set `set`: the weight blocks, then
  // the activation blocks in the order of the MFMAs
  auto frag = [&](int s, int f, int set, int r) {
    const unsigned char* st = smem + (s % NST) * STAGE + 16 * lane;
    if (r < NB) {
      fb[set][r] = *reinterpret_cast<const u32x4_t*>(st + (ACH + (wn * NB + r) * SUB + kSub * kg + f) * 1024);
    } else {
      const int i = (r - NB) / NPL, pl = (r - NB) % NPL;
      fa[set][r - NB] = *reinterpret_cast<const u32x4_t*>(st + (pl * (ACH / NPL) + (wm * MB + i) * SUB + kSub * kg + f) * 1024);
    }
  };
  // One step: the MFMAs of fragment set f with the next step's fragment reads
  // and this step's share of the stage loads spread between them.
  constexpr int NM = MB * NB * NPL, NF = NB + MB * NPL;
  auto step = [&](int s, int f) {
    const bool last = f + 1 == kSub;
    const int j0 = PW * f / kSub, j1 = PW * (f + 1) / kSub, items = NF + j1 - j0;
    int done = 0;
#pragma unroll
    for (int k = 0; k < NM; ++k) {
      const int i = k / (NB * NPL), pl = (k / NB) % NPL, j = k % NB;
      if constexpr (H) acc[j][i] = mfma32_f16(fb[f & 1][j], fa[f & 1][i * NPL + pl], acc[j][i]);
      else acc[j][i] = mfma32(fb[f & 1][j], fa[f & 1][i * NPL + pl], acc[j][i]);
#pragma unroll
      for (; done * NM < (k + 1) * items && done < items; ++done) {
        if (done < NF) frag(last ? s + 1 : s, last ? 0 : f + 1, (f + 1) & 1, done);
        else issue(s + NST - 1, j0 + done - NF);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
#pragma unroll
    for (int j = 0; j < PW; ++j) issue(s, j);
  if constexpr (EPI != DTREE_EPI_RESIDUAL) long_row_scale<T>(p, R, wave, rs);
  stage_wait<(NST - 2) * PW>();
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): from here the compiler counts LDS reads alone
#pragma unroll
  for (int r = 0; r < NF; ++r) frag(0, 0, 0, r);
  for (int s = 0; s < S; ++s) {
#pragma unroll
    for (int f = 0; f < kSub; ++f) {
      // Before the last step: stage s + 1 has landed for every wave, and every
      // wave has read all of stage s, so the next iteration may overwrite it.
      // This iteration's loads overwrite stage s - 1.
      if (f + 1 == kSub) stage_wait<(NST - 3) * PW + PW * (kSub - 1) / kSub>();
      __builtin_amdgcn_sched_barrier(0);
      step(s, f);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into this LDS outlives the workgroup
  const int mw = 32 * MB * wm, n0 = N0 + 32 * NB * wn;
  if constexpr (KS > 1) {
    // The two K halves: the waves of a pair swap half of their row blocks
    // through LDS, each adds and finishes the half it keeps.
    static_assert(MB % 2 == 0 && T::GM * T::GN * NB * MB * 4096 <= NST * STAGE, "the exchange fits the stages");
    constexpr int HB = MB / 2;
    stage_wait<0>();  // every wave's loads and reads of the stages are done
    f32x4_t* ex = reinterpret_cast<f32x4_t*>(smem) + (size_t)wt * (2 * NB * HB * 256) + lane;
    auto slot = [&](int g, int j, int i, int q) { return ex + (((g * NB + j) * HB + i) * 4 + q) * 64; };
    f32x16_t half[NB][HB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < HB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = kg ? acc[j][i][4 * q + e] : acc[j][HB + i][4 * q + e];
          *slot(kg, j, i, q) = v;
#pragma unroll
          for (int e = 0; e < 4; ++e) half[j][i][4 * q + e] = kg ? acc[j][HB + i][4 * q + e] : acc[j][i][4 * q + e];
        }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < HB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4_t v = *slot(1 - kg, j, i, q);
#pragma unroll
          for (int e = 0; e < 4; ++e) half[j][i][4 * q + e] += v[e];
        }
    if (p.vec) long_epilogue<NB, HB, EPI, true>(p, half, rs, R, mw + 32 * HB * kg, n0);
    else long_epilogue<NB, HB, EPI, false>(p, half, rs, R, mw + 32 * HB * kg, n0);
  } else {
    if (p.vec) long_epilogue<NB, MB, EPI, true>(p, acc, rs, R, mw, n0);
    else long_epilogue<NB, MB, EPI, false>(p, acc, rs, R, mw, n0);
  }
}

template <class T, bool H, int NPL>
int launch_tile(LongParams p, int epi, hipStream_t st) {
  p.ntn = (p.n + T::TN - 1) / T::TN;
  const long long tiles = (long long)((p.rows + T::TM - 1) / T::TM) * p.ntn;
  DTREE_REQUIRE(tiles < (1LL << 31), "gemm_long: grid too large");
  p.tiles = (int)tiles;
  switch (epi) {
    case DTREE_EPI_STORE_F32: long_kernel<T, DTREE_EPI_STORE_F32, H, NPL><<<p.tiles, T::THREADS, 0, st>>>(p); break;
    case DTREE_EPI_RESIDUAL:
      if constexpr (T::TN <= 256) long_kernel<T, DTREE_EPI_RESIDUAL, H, NPL><<<p.tiles, T::THREADS, 0, st>>>(p);
      break;
    case DTREE_EPI_SWIGLU: long_kernel<T, DTREE_EPI_SWIGLU, H, NPL><<<p.tiles, T::THREADS, 0, st>>>(p); break;
    default: long_kernel<T, DTREE_EPI_STORE_BF16, H, NPL><<<p.tiles, T::THREADS, 0, st>>>(p); break;
  }
  DTREE_LAUNCH_CHECK("gemm_long launch");
  return DTREE_OK;
}

using T128x128 = Tile<2, 2, 2, 2, 4>;      // bf16 weights
using T128x128k = Tile<2, 2, 2, 2, 4, 2>;
using T256x128 = Tile<2, 2, 4, 2, 6>;
using T256x192 = Tile<2, 3, 4, 2, 5>;
using T256x256 = Tile<4, 2, 2, 4, 4>;
using T256x320 = Tile<2, 5, 4, 2, 4>;
using T256x384 = Tile<4, 3, 2, 4, 3>;

// Tile shape for fp16 operands. One workgroup runs per CU, so a launch takes
// ceil(tiles / CUs) rounds of one tile time each; the shape with the least
// rounds x tile time wins. `cost` is the tile time in us per 64 K with every
// CU busy (a CU's share of the load bandwidth bounds the narrow tiles, MFMA
// issue the wide ones; per output element 256 x 256 is the cheapest). Measured
// for 1024 rows, us (128x128 / 256x128 / 256x192 / 256x256 / 256x320 /
// 256x384): N 2560 K 9728 65 / 110 / 160 / 179 / 238 / 306; N 6144 K 2560
// 48 / 42 / 53 / 61 / 70 / 85; N 12352 K 2560 102 / 89 / 112 / 77 / 81 / 103;
// N 19456 K 2560 136 / 129 / 120 / 133 / 98 / 108; N 24576 K 4096 244 / 212 /
// 201 / 209 / 243 / 186; 4096 rows, N 24576 K 4096: 950 / 827 / 775 / 699 /
// 697 / 728. The two widest do not take the residual epilogue (its preloaded
// rows would not fit their registers).
enum { kT128x128, kT256x128, kT256x192, kT256x256, kT256x320, kT256x384, kTiles };
struct TileCost { int tm, tn; float cost; };
constexpr TileCost kTileCost[kTiles] = {{128, 128, 0.55f}, {256, 128, 0.75f}, {256, 192, 1.08f},
                                        {256, 256, 1.30f}, {256, 320, 1.62f}, {256, 384, 2.05f}};

int pick_tile(int rows, int n, int epi, int cus) {
  int best = 0;
  float bt = 0.f;
  for (int i = 0; i < kTiles; ++i) {
    if (i >= kT256x320 && epi == DTREE_EPI_RESIDUAL) break;
    const TileCost& c = kTileCost[i];
    const long long tiles = (long long)((rows + c.tm - 1) / c.tm) * ((n + c.tn - 1) / c.tn);
    const float t = (float)((tiles + cus - 1) / cus) * c.cost;
    if (i == 0 || t < bt) {
      best = i;
      bt = t;
    }
  }
  return best;
}

}  // namespace

int launch_long_dense(LongParams p, int epi, bool h16, int cus, hipStream_t st) {
  if (!h16)
    return p.x_lo ? launch_tile<T128x128, false, 2>(p, epi, st) : launch_tile<T128x128, false, 1>(p, epi, st);
  switch (pick_tile(p.rows, p.n, epi, cus)) {
    case kT256x128: return launch_tile<T256x128, true, 1>(p, epi, st);
    case kT256x192: return launch_tile<T256x192, true, 1>(p, epi, st);
    case kT256x256: return launch_tile<T256x256, true, 1>(p, epi, st);
    case kT256x320: return launch_tile<T256x320, true, 1>(p, epi, st);
    case kT256x384: return launch_tile<T256x384, true, 1>(p, epi, st);
    default: return launch_tile<T128x128k, true, 1>(p, epi, st);
  }
}

}  // namespace dtree
