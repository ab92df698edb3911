// Long-M GEMM Y[M, N] = X[M, K] * W[N, K]^T for the prompt prefill (rows a
// multiple of 128). Compute-bound: the design goal is MFMA
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
//   cover each other's waits (N 2560, K 9728, 1024 rows, repeated by itself: 79
//   us with four waves, 65 with eight; as the down projection of a prompt, behind
//   gate/up, 89).
//
// Bound by MFMA issue on the wide tiles (a 256 x 256 tile with no loads at all
// takes 85 % of its time; the card's clock falls to about 2 GHz under it) and by
// the ~100 GB/s a CU loads on the narrow ones. Measured against the kernel
// this one replaced (128 x 128 tiles staged through registers, one barrier per
// 64 K): Qwen3-4B's gate/up and down over 1024 rows 368 -> 197 us (0.42 ->
// 0.79 PFLOP/s); N 24576, K 4096, 4096 rows 1403 -> 699 us (1.18 PFLOP/s).
#include "gemm_long.h"
#include "lds_load.h"

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

// Epilogues of the workgroup's finished accumulators (the stages' LDS is free
// again after the first barrier in here). With KS = 2 the waves of a pair swap
// half of their row blocks through LDS, and each adds and finishes the half it
// keeps. `turn` brings acc[j][i] into the epilogue's layout in place if the
// kernel accumulates another one; its scratch is 32 x 36 floats per wave.
template <class T, int EPI, class Turn>
__device__ __forceinline__ void long_finish(const LongParams& p, f32x16_t (&acc)[T::NB][T::MB], unsigned char* smem,
                                            const float* rs, int wave, int R, int N0, Turn turn) {
  constexpr int MB = T::MB, NB = T::NB;
  const int lane = threadIdx.x & 63;
  const int kg = T::KS > 1 ? wave / (T::GM * T::GN) : 0, wt = wave - kg * (T::GM * T::GN);
  const int wm = wt / T::GN, wn = wt % T::GN;
  const int mw = 32 * MB * wm, n0 = N0 + 32 * NB * wn;
  float* scratch = reinterpret_cast<float*>(smem) + wave * (32 * 36);
  stage_wait<0>();  // every wave's loads and reads of the stages are done
  if constexpr (T::KS > 1) {
    static_assert(MB % 2 == 0, "a pair of waves swaps half of its row blocks");
    constexpr int HB = MB / 2;
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
    __syncthreads();
    turn(half, scratch);
    if (p.vec) long_epilogue<NB, HB, EPI, true>(p, half, rs, R, mw + 32 * HB * kg, n0);
    else long_epilogue<NB, HB, EPI, false>(p, half, rs, R, mw + 32 * HB * kg, n0);
  } else {
    turn(acc, scratch);
    if (p.vec) long_epilogue<NB, MB, EPI, true>(p, acc, rs, R, mw, n0);
    else long_epilogue<NB, MB, EPI, false>(p, acc, rs, R, mw, n0);
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
  const unsigned wbytes = (unsigned)min(T::TN, p.n - N0) / 32u * strip;
  const u32x4_t xr = strip_rsrc(p.x + xo, xbytes);
  const u32x4_t wr = strip_rsrc(p.w + wo, wbytes);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  // Piece wave + WAVES j of stage s: activation pieces (plane, row block,
  // fragment), then weight pieces (column block, fragment). Past the last
  // stage or piece the load reads nothing, so every wave always has the same
  // number in flight.
  // Two planes: the piece's base, size, offset and place are kept in scalar
  // registers. Chosen among three resources at every load they went through
  // scratch, whose waits also wait for the stage loads just issued (N 19456,
  // K 2560, 1024 rows: 1229 us, so 219). For one plane the choice between two
  // is the faster form (N 2560, K 9728, 1024 rows, bf16: 79 us, in registers 82).
  constexpr bool WORDS = NPL > 1;
  uint32_t plo[PW], phi[PW], psize[PW], poff[PW];
  if constexpr (WORDS) {
    static_assert(!PAD, "two planes deal their pieces out evenly");
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int ch = wave + T::WAVES * j;
      const bool isa = ch < ACH, low = isa && ch >= ACH / NPL;
      const int ap = !isa ? ch - ACH : low ? ch - ACH / NPL : ch;
      const uint64_t base = isa ? (uint64_t)((low ? p.x_lo : p.x) + xo) : (uint64_t)(p.w + wo);
      plo[j] = uni((uint32_t)base);
      phi[j] = uni((uint32_t)(base >> 32) & 0xffffu);
      psize[j] = uni(isa ? xbytes : wbytes);
      poff[j] = uni((unsigned)(ap / SUB) * strip + (unsigned)(ap % SUB) * 1024u);
      // opaque from here on: kept instead of being made again per stage
      asm volatile("" : "+s"(plo[j]), "+s"(phi[j]), "+s"(psize[j]), "+s"(poff[j]));
    }
  }
  auto issue = [&](int s, int j) {
    const int ch = wave + T::WAVES * j;
    if constexpr (WORDS) {
      lds_load16_s(plo[j], phi[j], psize[j] & (uint32_t)((s - S) >> 31),
                   poff[j] + (unsigned)s * (SUB * 1024u) + 16u * lane, lds0 + (s % NST) * STAGE + 1024 * ch);
    } else {
      const bool isa = ch < ACH, pad = PAD && ch >= CH;
      const int ap = isa ? ch : ch - ACH;
      const unsigned off = (unsigned)(ap / SUB) * strip + (unsigned)(ap % SUB + SUB * s) * 1024u;
      const unsigned lds = lds0 + (pad ? (unsigned)(NST * STAGE) : (unsigned)((s % NST) * STAGE + 1024 * ch));
      lds_load16(isa ? xr : wr, (s < S && !pad ? off : kOob) + 16u * lane, lds);
    }
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
  long_finish<T, EPI>(p, acc, smem, rs, wave, R, N0, [](auto&, float*) {});
}

// ---- q4 group-64 weights ---------------------------------------------------------
// The same tiles and pipeline over 4-bit weights with bf16 activations. A K
// block is one quantisation group and one stage (per K group of the tile): the
// activation fragments, 1 KB of nibbles and 32 (scale, bias) words per column
// block, all by direct loads.
//
// y = sum_g s_g sum_k x_k q_k + b_g sum_k x_k. The nibbles enter the MFMA as
// bf16 16 + q (exact), so per group
//   acc += s * (x . (16 + q)),  and  acc += (b - 16 s) * sum(x).
// (128 + q would save a shift in seven unpacking operations, but up to eight
// groups' 128 s sum(x) stand in the accumulators until the second term takes
// them out, and their rounding stays: against 64 bits, K 4096, relative error
// 9.3e-7 with 128 and 2.0e-7 with 16, 6.0e-7 with 128 and the second term added
// group by group; with activations of mean 4, 3.3e-7, 1.0e-7 and 2.1e-7. The
// shift costs 1 to 2 % of the time.)
// The first is a fresh four-MFMA sum per 32 x 32 block folded in by one FMA per
// element, under the next block's MFMAs. The second is a product over the
// groups, [rows x groups] x [groups x columns], so it runs on MFMA as well, once
// per eight groups: each group's sum(x) (dot products with ones, one wave per
// row block) and b - 16 s (one wave per column block) go to an LDS ring as
// fp32; both are split into three bf16 parts (24 significant bits), and three
// MFMAs cover the six products down to 2^-16, two of them side by side in the
// 16 K slots (the lane halves). As FMAs it would cost as many again as the
// first fold, which with the nibble unpacking is what bounds the kernel.
//
// The accumulators are X W^T here (a scale is then one value per lane) and are
// turned into the epilogues' layout through LDS once per tile.
//
// Measured against the kernel this one replaced (128 x 128 tiles through
// registers, both folds as FMAs, sum(x) by MFMA in every wave): the 9B-shaped
// MLP (gate/up and down) over 300 tokens 477 -> 240 us; N 24576, K 4096, 4096
// rows 847 us (0.97 PFLOP/s; the fp16 tiles reach 1.18). Bound by a wave's own
// instruction chain (folds, unpacking, load issue, waits): a lone wave per SIMD
// takes as long per stage as two, and deeper pipelines change nothing. With the
// folds beginning under their block's last MFMA and the load resources remade
// from vector registers at every load it was 248 us and 913 us (with 128 + q,
// then 236 and 827).
constexpr int kRing = 8;        // groups per correction step
constexpr int kRingStride = 12; // floats per ring row (16-byte reads, spread over the banks)

// Nibbles as bf16 16 + q: the nibble in mantissa bits 3 to 6.
__device__ __forceinline__ u32x4_t q4_pairs16(uint32_t w, uint32_t m, uint32_t e) {
  return u32x4_t{((w << 3) & m) | e, ((w >> 1) & m) | e, ((w >> 5) & m) | e, ((w >> 9) & m) | e};
}

// Sum of the eight bf16 of w, added to s.
__device__ __forceinline__ float bf8_sum(u32x4_t w, float s) {
  const bf16x2_t one = __builtin_bit_cast(bf16x2_t, 0x3f803f80u);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, (uint32_t)w[i]), one, s, false);
  return s;
}

// a + the other half-wave's a. As row_pair_sum (common.h): one asm sequence,
// since the compiler folds the two results of the swap of equal registers.
__device__ __forceinline__ float half_pair_sum(float a) {
  float b;
  asm volatile("v_mov_b32 %1, %0\n\ts_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_add_f32 %0, %0, %1"
               : "+v"(a), "=&v"(b));
  return a;
}

// v = hi + mid + lo, each bf16, to about 24 significant bits.
__device__ __forceinline__ void split3(const float (&v)[8], u32x4_t& hi, u32x4_t& mid, u32x4_t& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = v[2 * i], b = v[2 * i + 1];
    hi[i] = pack_bf2(a, b);
    const float a1 = a - __uint_as_float(hi[i] << 16), b1 = b - __uint_as_float(hi[i] & 0xffff0000u);
    mid[i] = pack_bf2(a1, b1);
    lo[i] = pack_bf2(a1 - __uint_as_float(mid[i] << 16), b1 - __uint_as_float(mid[i] & 0xffff0000u));
  }
}

template <class T, int EPI, int NPL>
__global__ __launch_bounds__(T::THREADS) void longq_kernel(LongParams p) {
  constexpr int MB = T::MB, NB = T::NB, NST = T::NST, KS = T::KS, WT = T::GM * T::GN;
  constexpr int RB = T::TM / 32, CB = T::TN / 32;
  constexpr int PA = RB * NPL * 4, CHK = PA + CB + 1;  // 1 KB pieces per K block: x, nibbles, scale words
  constexpr int CH = KS * CHK, STAGE = CH * 1024;
  constexpr int PW = (CH + T::WAVES - 1) / T::WAVES;
  constexpr bool PAD = CH % T::WAVES != 0;
  static_assert(CB <= 8, "one piece holds the tile's scale words");
  static_assert(NST * STAGE >= T::WAVES * 32 * 36 * 4 && (KS == 1 || NST * STAGE >= WT * NB * MB * 4096),
                "long_finish's scratch");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[NST * STAGE + (PAD ? 1024 : 0)];
  __shared__ __attribute__((aligned(16))) float xring[KS][T::TM][kRingStride], cring[KS][T::TN][kRingStride];
  __shared__ float rs[T::TM];
  const int t = threadIdx.x, lane = t & 63, c = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int kg = KS > 1 ? wave / WT : 0, wt = wave - kg * WT;
  const int wm = wt / T::GN, wn = wt % T::GN;
  const int2 mn = xcd_tile(blockIdx.x, p.tiles, p.ntn, T::TM);
  const int R = mn.x * T::TM, N0 = mn.y * T::TN;
  const unsigned nkb = (unsigned)p.k >> 6;
  const int S = (int)nkb / KS;  // KS = 2 takes an even number of K blocks
  const unsigned mrb = (unsigned)min(T::TM, p.rows - R) / 32u, ncb = (unsigned)min(T::TN, p.n - N0) / 32u;
  const size_t xo = (size_t)R * p.k, cb0 = (size_t)(N0 >> 5) * nkb;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  // Piece wave + WAVES j of every stage: its strips' base and size, its offset
  // in stage 0, the offset's step per stage and its place in a stage.
  // (A piece past the last has size 0, reads nothing and keeps the counts equal.)
  uint32_t plo[PW], phi[PW], psize[PW], poff[PW], pstep[PW], plds[PW], pstage[PW];
  uint32_t pmask[PW];
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const int ch = wave + T::WAVES * j;
    const int g = KS > 1 ? ch / CHK : 0, q = ch - g * CHK;
    const bool pad = PAD && ch >= CH;
    const bool isx = q < PA, isw = !isx && q < PA + CB, low = NPL > 1 && isx && q >= PA / NPL;
    const int a = isx ? (low ? q - PA / NPL : q) : q - PA;
    const unsigned kstep = isx ? 4096u : isw ? 1024u : 128u;  // bytes of one K block of a strip
    const uint64_t base = isx ? (uint64_t)((low ? p.x_lo : p.x) + xo)
                              : isw ? (uint64_t)(p.w + cb0 * 512) : (uint64_t)(p.w_sb + cb0 * 64);
    plo[j] = uni((uint32_t)base);
    phi[j] = uni((uint32_t)(base >> 32) & 0xffffu);
    psize[j] = uni(pad ? 0u : (isx ? mrb : ncb) * nkb * kstep);
    poff[j] = uni((isx ? (unsigned)(a >> 2) : isw ? (unsigned)a : 0u) * nkb * kstep + g * kstep +
                  (isx ? (a & 3) * 1024u : 0u));
    pstep[j] = uni(KS * kstep);
    plds[j] = uni(lds0 + (pad ? NST * STAGE : 1024 * ch));
    pstage[j] = uni(pad ? 0u : ~0u);  // padding has one place for all stages
    pmask[j] = uni(isx || isw ? 0u : ~0u);  // scale words: eight lanes per column block
    // opaque from here on: kept in scalar registers instead of being made again per stage
    asm volatile("" : "+s"(plo[j]), "+s"(phi[j]), "+s"(psize[j]), "+s"(poff[j]), "+s"(pstep[j]), "+s"(plds[j]),
                 "+s"(pstage[j]));
  }
  const unsigned lane16 = 16u * lane, lane_s = (unsigned)(lane >> 3) * nkb * 128u + 16u * (lane & 7) - lane16;
  // `at`: the stage's LDS offset. Past the last stage the size is 0 (no branch
  // and no select: the stage loop stays one block, as its order is written).
  auto issue = [&](int s, unsigned at, int j) {
    const uint32_t live = (uint32_t)((s - S) >> 31);
    lds_load16_s(plo[j], phi[j], psize[j] & live, poff[j] + (unsigned)s * pstep[j] + lane16 + (lane_s & pmask[j]),
                 plds[j] + (at & pstage[j]));
  };
  f32x16_t acc[NB][MB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.f;
  uint32_t nib_m, nib_e;  // in registers: the three-operand form takes no literal
  asm("s_mov_b32 %0, 0x00780078" : "=s"(nib_m));
  asm("v_mov_b32 %0, 0x41804180" : "=v"(nib_e));
  constexpr int NT = MB * NB;
  // row blocks whose sums, and column blocks whose ring entries, a wave makes
  constexpr int NSUM = MB > T::GN ? MB / T::GN : 1, NCR = (CB + WT - 1) / WT;
  static_assert((MB % T::GN == 0 || T::GN % MB == 0) && NT % 2 == 0 && 2 * NSUM <= NT - NB && CB % (NCR * 2) == 0,
                "sums shared out evenly and done before the last row block; running sums alternate");
  u32x4_t fa[4 * NPL], wq[NB], bq[NB][4];
  uint32_t sbw[NB], cw[NCR];
  float sc[NB];
  f32x16_t au[2];
  const unsigned char* kbase = smem + kg * (CHK * 1024);
  auto read_a = [&](unsigned at, int i, int f, int pl) {
    fa[f * NPL + pl] = *reinterpret_cast<const u32x4_t*>(
        kbase + at + ((pl * RB + wm * MB + i) * 4 + f) * 1024 + 16 * lane);
  };
  auto read_w = [&](unsigned at, int j) {
    const unsigned char* st = kbase + at + PA * 1024;
    wq[j] = *reinterpret_cast<const u32x4_t*>(st + (wn * NB + j) * 1024 + 16 * lane);
    sbw[j] = *reinterpret_cast<const uint32_t*>(st + CB * 1024 + (wn * NB + j) * 128 + 4 * c);
    if (j < NCR) cw[j] = *reinterpret_cast<const uint32_t*>(st + CB * 1024 + min(wt * NCR + j, CB - 1) * 128 + 4 * c);
  };
  auto unpack = [&](int j, int f) {
    bq[j][f] = q4_pairs16(wq[j][f], nib_m, nib_e);
  };
  // sum(x) of the group for this wave's row blocks (both lane halves hold and
  // write the same value, as do waves that share a row block)
  const int srow = wm * MB + (MB > T::GN ? wn * NSUM : wn % MB);
  u32x4_t sx[4 * NPL];
  float ssum[2];
  auto sum_read = [&](unsigned at, int e, int f) {
#pragma unroll
    for (int pl = 0; pl < NPL; ++pl)
      sx[f * NPL + pl] = *reinterpret_cast<const u32x4_t*>(kbase + at + ((pl * RB + srow + e) * 4 + f) * 1024 + 16 * lane);
  };
  auto sum_add = [&](int f) {
#pragma unroll
    for (int pl = 0; pl < NPL; ++pl) ssum[f & 1] = bf8_sum(sx[f * NPL + pl], f < 2 && pl == 0 ? 0.f : ssum[f & 1]);
  };
  // A third of block v's sum, under the next block's MFMAs 1 .. 3 (its own last
  // one is still running under MFMA 0).
  auto fold = [&](int v, int f, float scale) {
#pragma unroll
    for (int r = 16 * (f - 1) / 3; r < 16 * f / 3; ++r)
      acc[v % NB][v / NB][r] = fmaf(scale, au[v & 1][r], acc[v % NB][v / NB][r]);
  };
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
#pragma unroll
    for (int j = 0; j < PW; ++j) issue(s, s * STAGE, j);
  if constexpr (EPI != DTREE_EPI_RESIDUAL) long_row_scale<T>(p, R, wave, rs);
  stage_wait<(NST - 2) * PW>();
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): from here the compiler counts LDS operations alone
#pragma unroll
  for (int j = 0; j < NB; ++j) read_w(0, j);
#pragma unroll
  for (int f = 0; f < 4; ++f)
#pragma unroll
    for (int pl = 0; pl < NPL; ++pl) read_a(0, 0, f, pl);
#pragma unroll
  for (int f = 0; f < 4; ++f) unpack(0, f);
#pragma unroll
  for (int j = 0; j < NB; ++j) sc[j] = 0.f;
  float sc0 = __uint_as_float(sbw[0] << 16);  // column block 0's scale of the stage to come
#pragma unroll
  for (int r = 0; r < 16; ++r) au[(NT - 1) & 1][r] = 0.f;
  // LDS offsets of stages s, s + 1 and s + NST - 1
  unsigned cur = 0, nxt = STAGE, fut = (NST - 1) * STAGE;
  auto advance = [](unsigned& o) { o = o + STAGE == NST * STAGE ? 0u : o + STAGE; };
  for (int s = 0; s < S; ++s) {
    const int slot = s & (kRing - 1);
    const float last = sc[NB - 1];
    sc[0] = sc0;
#pragma unroll
    for (int j = 1; j < NB; ++j) sc[j] = __uint_as_float(sbw[j] << 16);
#pragma unroll
    for (int e = 0; e < NCR; ++e)
      cring[kg][min(wt * NCR + e, CB - 1) * 32 + c][slot] =
          fmaf(-16.f, __uint_as_float(cw[e] << 16), __uint_as_float(cw[e] & 0xffff0000u));
    // Block u = (row block i, column block j): its four MFMAs, with the previous
    // block's fold, the unpacking of the column block needed next, the next
    // row block's fragments, the ring's row sums and this stage's share of the
    // loads between them.
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int i = u / NB, j = u % NB;
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        __builtin_amdgcn_sched_barrier(0);
        // Inside the last row block: stage s + 1 has landed for every wave, every
        // wave has read all of stage s, and the ring holds this group.
        if (j == 0 && i + 1 == MB && f == 2) stage_wait<(NST - 3) * PW + PW * (NT - NB) / NT>();
#pragma unroll
        for (int pl = 0; pl < NPL; ++pl) {
          if (f == 0 && pl == 0) {
            f32x16_t z;
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r] = 0.f;
            au[u & 1] = mfma32(fa[0], bq[j][0], z);
          } else {
            au[u & 1] = mfma32(fa[f * NPL + pl], bq[j][f], au[u & 1]);
          }
          if (j + 1 == NB) {  // the next row block's fragments take this one's registers
            if (i + 1 < MB) read_a(cur, i + 1, f, pl);
            else read_a(nxt, 0, f, pl);
          }
        }
        if (f > 0) {
          if (u > 0) fold(u - 1, f, sc[(u - 1) % NB]);
          else fold(NT - 1, f, last);  // the previous stage's last block
        }
        if (u + 1 < NB) unpack(u + 1, f);
        if (u + 1 == NT) unpack(0, f);
        if (u < 2 * NSUM) {
          if (u % 2 == 0) sum_read(cur, u / 2, f);
          else sum_add(f);
          if (u % 2 == 1 && f == 3) xring[kg][(srow + u / 2) * 32 + c][slot] = half_pair_sum(ssum[0] + ssum[1]);
        }
        if (i + 1 == MB && j == 0 && f == 2) {
#pragma unroll
          for (int jj = 0; jj < NB; ++jj) read_w(nxt, jj);
        }
        if (f == 3) {
#pragma unroll
          for (int d = PW * u / NT; d < PW * (u + 1) / NT; ++d) issue(s + NST - 1, fut, d);
        }
      }
    }
    sc0 = __uint_as_float(sbw[0] << 16);
    advance(cur);
    advance(nxt);
    advance(fut);
    if (slot == kRing - 1 || s + 1 == S) {
      // the ring's groups: acc += sum(x) (b - 16 s), three bf16 parts each
      const int valid = slot + 1;
      auto parts = [&](const float* row, u32x4_t (&o)[3]) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(row), b = *reinterpret_cast<const f32x4_t*>(row + 4);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = e < valid ? (e < 4 ? a[e & 3] : b[e & 3]) : 0.f;
        split3(v, o[0], o[1], o[2]);
      };
      u32x4_t cp[NB][2];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        u32x4_t o[3];
        parts(cring[kg][(wn * NB + j) * 32 + c], o);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          cp[j][0][e] = h ? o[1][e] : o[0][e];
          cp[j][1][e] = h ? o[0][e] : o[2][e];
        }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        u32x4_t o[3], x3;
        parts(xring[kg][(wm * MB + i) * 32 + c], o);
#pragma unroll
        for (int e = 0; e < 4; ++e) x3[e] = h ? o[2][e] : o[0][e];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          acc[j][i] = mfma32(o[0], cp[j][0], acc[j][i]);  // hi hi + hi mid
          acc[j][i] = mfma32(o[1], cp[j][0], acc[j][i]);  // mid hi + mid mid
          acc[j][i] = mfma32(x3, cp[j][1], acc[j][i]);    // hi lo + lo hi
        }
      }
      lds_barrier();  // the next group's entries overwrite the ring
    }
  }
#pragma unroll
  for (int f = 1; f < 4; ++f) fold(NT - 1, f, sc[NB - 1]);
  long_finish<T, EPI>(p, acc, smem, rs, wave, R, N0, [&](auto& a, float* buf) {
#pragma unroll
    for (auto& aj : a)
#pragma unroll
      for (auto& blk : aj) {
#pragma unroll
        for (int r = 0; r < 16; ++r) buf[acc_row(r, h) * 36 + c] = blk[r];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(buf + c * 36 + 8 * q + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) blk[4 * q + e] = v[e];
        }
      }
  });
}

enum Mode { kBf16, kBf16Lo, kF16, kQ4, kQ4Lo };

template <class T, int EPI, Mode M>
void launch_kernel(const LongParams& p, hipStream_t st) {
  if constexpr (M == kQ4) longq_kernel<T, EPI, 1><<<p.tiles, T::THREADS, 0, st>>>(p);
  else if constexpr (M == kQ4Lo) longq_kernel<T, EPI, 2><<<p.tiles, T::THREADS, 0, st>>>(p);
  else long_kernel<T, EPI, M == kF16, M == kBf16Lo ? 2 : 1><<<p.tiles, T::THREADS, 0, st>>>(p);
}

template <class T, Mode M>
int launch_tile(LongParams p, int epi, hipStream_t st) {
  p.ntn = (p.n + T::TN - 1) / T::TN;
  const long long tiles = (long long)((p.rows + T::TM - 1) / T::TM) * p.ntn;
  DTREE_REQUIRE(tiles < (1LL << 31), "gemm_long: grid too large");
  p.tiles = (int)tiles;
  switch (epi) {
    case DTREE_EPI_STORE_F32: launch_kernel<T, DTREE_EPI_STORE_F32, M>(p, st); break;
    case DTREE_EPI_RESIDUAL:
      if constexpr (T::TN <= 256) launch_kernel<T, DTREE_EPI_RESIDUAL, M>(p, st);
      break;
    case DTREE_EPI_SWIGLU: launch_kernel<T, DTREE_EPI_SWIGLU, M>(p, st); break;
    default: launch_kernel<T, DTREE_EPI_STORE_BF16, M>(p, st); break;
  }
  DTREE_LAUNCH_CHECK("gemm_long launch");
  return DTREE_OK;
}

using Q128x128lo = Tile<2, 2, 2, 2, 3>;      // with the low activation plane
using Q128x128k = Tile<2, 2, 2, 2, 3, 2>;
using Q128x256 = Tile<2, 2, 2, 4, 3>;
using Q256x192 = Tile<2, 3, 4, 2, 3>;
using Q256x256 = Tile<4, 2, 2, 4, 3>;
using T128x128 = Tile<2, 2, 2, 2, 4>;      // bf16 weights
using T64x64k = Tile<2, 1, 1, 2, 4, 2>;
using T64x128k = Tile<2, 2, 1, 2, 4, 2>;
using T128x128k = Tile<2, 2, 2, 2, 4, 2>;
using T256x128 = Tile<2, 2, 4, 2, 6>;
using T256x192 = Tile<2, 3, 4, 2, 5>;
using T256x256 = Tile<4, 2, 2, 4, 4>;
using T256x320 = Tile<2, 5, 4, 2, 4>;
using T256x384 = Tile<4, 3, 2, 4, 3>;

// Tile shape for fp16 operands. A launch is taken as ceil(tiles / CUs) rounds of
// one tile time each (a CU's LDS holds one workgroup, but two of the 64 x 64
// tiles, which is in their cost); the shape with the least rounds x tile time
// wins. `cost` is the tile time in us per 64 K with every CU busy (a CU's share of the load bandwidth bounds the narrow tiles, MFMA
// issue the wide ones; per output element 256 x 256 is the cheapest). Measured
// for 1024 rows, us, each product repeated by itself (128x128 / 256x128 / 256x192 / 256x256 / 256x320 /
// 256x384): N 2560 K 9728 65 / 110 / 160 / 179 / 238 / 306; N 6144 K 2560
// 48 / 42 / 53 / 61 / 70 / 85; N 12352 K 2560 102 / 89 / 112 / 77 / 81 / 103;
// N 19456 K 2560 136 / 129 / 120 / 133 / 98 / 108; N 24576 K 4096 244 / 212 /
// 201 / 209 / 243 / 186; 4096 rows, N 24576 K 4096: 950 / 827 / 775 / 699 /
// 697 / 728. The two smallest are for short prompts (64x64 / 64x128 / 128x128):
// 128 rows, N 6144 K 2560 14 / 17 / 21; 384 rows, N 2560 K 9728 38 / 48 / 56;
// 768 rows, the same 65 / 54 / 60. The two widest do not take the residual epilogue (its preloaded
// rows would not fit their registers).
struct TileCost { int tm, tn; float cost; };
enum { kT64x64, kT64x128, kT128x128, kT256x128, kT256x192, kT256x256, kT256x320, kT256x384, kTiles };
constexpr TileCost kTileCost[kTiles] = {{64, 64, 0.25f}, {64, 128, 0.35f}, {128, 128, 0.55f}, {256, 128, 0.75f},
                                        {256, 192, 1.08f}, {256, 256, 1.30f}, {256, 320, 1.62f}, {256, 384, 2.05f}};
// The same for q4 weights (one or two K blocks per stage; 128 x 128 tiles need
// an even number of them). Measured with nibbles as 128 + q, 1 to 2 % below the
// present times, us at 1024 rows (128x128 / 128x256 / 256x192 /
// 256x256): N 2560 K 9728 106 / 179 / 237 / 286; N 12352 K 2560 136 / 111 / 143
// / 88; N 24576 K 4096 290 / 256 / 231 / 261; 4096 rows, N 24576 K 4096: 1141
// / 1021 / 920 / 846; N 2560 K 9728: 316 / 369 / 259 / 289.
enum { kQ128x128, kQ128x256, kQ256x192, kQ256x256, kQTiles };
constexpr TileCost kQTileCost[kQTiles] = {{128, 128, 0.75f}, {128, 256, 1.33f}, {256, 192, 1.80f}, {256, 256, 2.20f}};

// The first of `count` shapes from `from` on with the least rounds x cost.
int pick_tile(const TileCost* cost, int from, int count, int rows, int n, int cus) {
  int best = from;
  float bt = 0.f;
  for (int i = from; i < count; ++i) {
    const TileCost& c = cost[i];
    const long long tiles = (long long)((rows + c.tm - 1) / c.tm) * ((n + c.tn - 1) / c.tn);
    const float t = (float)((tiles + cus - 1) / cus) * c.cost;
    if (i == from || t < bt) {
      best = i;
      bt = t;
    }
  }
  return best;
}

}  // namespace

namespace {
int dense_tile(int epi, int rows, int n, int cus) {
  return pick_tile(kTileCost, 0, epi == DTREE_EPI_RESIDUAL ? kT256x320 : kTiles, rows, n, cus);
}
int q4_tile(int rows, int n, int k, int cus) {
  return pick_tile(kQTileCost, k % 128 ? kQ128x256 : kQ128x128, kQTiles, rows, n, cus);
}
}  // namespace

int long_tile(bool q4, bool h16, bool lo, int epi, int rows, int n, int k, int cus) {
  if (q4 ? lo : !h16) return 1000 * 128 + 128;
  const TileCost& c = q4 ? kQTileCost[q4_tile(rows, n, k, cus)] : kTileCost[dense_tile(epi, rows, n, cus)];
  return 1000 * c.tm + c.tn;
}

int launch_long_dense(LongParams p, int epi, bool h16, int cus, hipStream_t st) {
  if (!h16)
    return p.x_lo ? launch_tile<T128x128, kBf16Lo>(p, epi, st) : launch_tile<T128x128, kBf16>(p, epi, st);
  switch (dense_tile(epi, p.rows, p.n, cus)) {
    case kT64x64: return launch_tile<T64x64k, kF16>(p, epi, st);
    case kT64x128: return launch_tile<T64x128k, kF16>(p, epi, st);
    case kT256x128: return launch_tile<T256x128, kF16>(p, epi, st);
    case kT256x192: return launch_tile<T256x192, kF16>(p, epi, st);
    case kT256x256: return launch_tile<T256x256, kF16>(p, epi, st);
    case kT256x320: return launch_tile<T256x320, kF16>(p, epi, st);
    case kT256x384: return launch_tile<T256x384, kF16>(p, epi, st);
    default: return launch_tile<T128x128k, kF16>(p, epi, st);
  }
}

int launch_long_q4(LongParams p, int epi, int cus, hipStream_t st) {
  if (p.x_lo) return launch_tile<Q128x128lo, kQ4Lo>(p, epi, st);
  switch (q4_tile(p.rows, p.n, p.k, cus)) {
    case kQ128x256: return launch_tile<Q128x256, kQ4>(p, epi, st);
    case kQ256x192: return launch_tile<Q256x192, kQ4>(p, epi, st);
    case kQ256x256: return launch_tile<Q256x256, kQ4>(p, epi, st);
    default: return launch_tile<Q128x128k, kQ4>(p, epi, st);
  }
}

}  // namespace dtree
