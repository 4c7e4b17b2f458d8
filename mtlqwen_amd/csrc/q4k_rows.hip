// GEMMs of 9 to 64 rows with hi/lo activations for gfx950: decode batches,
// short prompts and the LM head's rows, for every weight type.  The weights
// enter the MFMAs as the decode GEMVs' exact quant x scale products and the
// activations as two fp16 parts (about 22 significant bits), so the results
// keep the GEMVs' precision while the weights are read once for all rows.
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include "q4k_mid.h"

namespace q4k {
namespace {

// ---- B operands ---------------------------------------------------------------
// Per weight type: the loads of a tile-block into LDS and its raw words there
// (the Tg* policies), the block constants, and the B fragments of MFMAs u and
// 4 + u as fp16 products whose block factor d (kFold) is applied to the fp32
// sums of the block; kMin: the min term, dmin times the 16x16x16 MFMA of the
// sub-block sums with bmin (32 m_j; k = 0..7 the hi parts, 8..15 the lo ones).
struct RxQ4K : TgQ4K {
  static constexpr bool kFold = true, kMin = true, kShortSums = true;
  struct K {
    float d, dmin;
    h2_t mul_lo, add_lo, mul_hi, add_hi;
    h4_t bmin;
  };
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    // bmin of lane group g: sub-blocks 4 (g & 1) .. + 3 for the hi and the lo
    // sums; block_consts gives those of g < 2 and zero for the others.
    const BlockConsts a = block_consts(r.hd, lane >> 4);
    k.d = a.d;
    k.dmin = a.dmin;
    k.mul_lo = a.mul_lo;
    k.add_lo = a.add_lo;
    k.mul_hi = a.mul_hi;
    k.add_hi = a.add_hi;
    const uint32_t m03 = r.hd.z & 0x3F3F3F3Fu, m47 = ((r.hd.w >> 4) & 0x0F0F0F0Fu) | ((r.hd.z >> 2) & 0x30303030u);
    const uint32_t mb = (lane & 16) ? m47 : m03;
    const h2_t k32 = {(_Float16)32.0f, (_Float16)32.0f}, kneg32768 = {(_Float16)-32768.0f, (_Float16)-32768.0f};
    const h2_t m01 = __builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(0x64646464u, mb, 0x04010400u)), k32, kneg32768);
    const h2_t m23 = __builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(0x64646464u, mb, 0x04030402u)), k32, kneg32768);
    k.bmin = h4_t{m01[0], m01[1], m23[0], m23[1]};
  }
  static __device__ __forceinline__ void frags(const K& k, const W& w, int, h8_t& blo, h8_t& bhi) {
    blo = quant_times_scale(w.q.x, w.q.y, 0x000F000Fu, 0x64006400u, k.mul_lo, k.add_lo);
    bhi = quant_times_scale(w.q.x, w.q.y, 0x00F000F0u, 0x64006400u, k.mul_hi, k.add_hi);
  }
};

struct RxQ5K : TgQ5K {
  static constexpr bool kFold = true, kMin = true, kShortSums = false;
  struct K : RxQ4K::K {
    uint32_t h0, h1;
  };
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    RxQ4K::R q;
    q.hd = r.hd;
    RxQ4K::consts(k, q, lane);
    k.h0 = r.h.x;
    k.h1 = r.h.y;
  }
  static __device__ __forceinline__ void frags(const K& k, const W& w, int u, h8_t& blo, h8_t& bhi) {
    const uint32_t src[4] = {w.q.x, w.q.x >> 8, w.q.y, w.q.y >> 8};
    u4_t lo, hi;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t b0 = and_or(move_bits(k.h0, 4 * u + t, 4), 0x00100010u, 0x64006400u);
      const uint32_t b1 = and_or(move_bits(k.h1, 4 * u + t, 8), 0x01000100u, 0x64006400u);
      lo[t] = as_u32(__builtin_elementwise_fma(as_h2(and_or(src[t], 0x000F000Fu, b0)), k.mul_lo, k.add_lo));
      hi[t] = as_u32(__builtin_elementwise_fma(as_h2(and_or(src[t], 0x00F000F0u, b1)), k.mul_hi, k.add_hi));
    }
    blo = __builtin_bit_cast(h8_t, lo);
    bhi = __builtin_bit_cast(h8_t, hi);
  }
};

struct RxQ6K : TgQ6K {
  static constexpr bool kFold = true, kMin = false, kShortSums = false;
  struct K {
    float d, dmin;
    h2_t mul[4], add[4];  // of scale byte i: sc / 16 and -96 sc
  };
  static __device__ __forceinline__ void consts(K& k, const R& r, int) {
    k.d = half_bits_to_float(r.d & 0xffffu);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2_t p = as_h2(__builtin_amdgcn_perm(0x64646464u, r.sc, 0x04000400u | (uint32_t)i | ((uint32_t)i << 16)));
      k.mul[i] = __builtin_elementwise_fma(p, h2_splat(0.0625f), h2_splat(-72.0f));
      k.add[i] = k.mul[i] * h2_splat(-1536.0f);
    }
  }
  static __device__ __forceinline__ h8_t half_triple(uint32_t A, uint32_t B, uint32_t C, int p, h2_t mul, h2_t add) {
    const uint32_t m6 = 0x03F003F0u, m4 = 0x00F000F0u, m2 = 0x03000300u, magic = 0x64006400u;
    u4_t o;
    if (p == 0) {
      o[0] = and_or(A, m6, magic);
      o[1] = and_or(A >> 6, m6, magic);
      o[2] = and_or(B, m6, magic);
      o[3] = and_or(B >> 6, m6, magic);
    } else {
      o[0] = and_or(C, m6, magic);
      o[1] = and_or(C >> 6, m6, magic);
      o[2] = and_or(A << 4, m4, and_or(B << 8, m2, magic));
      o[3] = and_or(C << 4, m4, and_or(B << 6, m2, magic));
    }
    u4_t f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const uint32_t v = o[t];
      f[t] = as_u32(__builtin_elementwise_fma(as_h2(v), mul, add));
    }
    return __builtin_bit_cast(h8_t, f);
  }
  static __device__ __forceinline__ void frags(const K& k, const W& w, int u, h8_t& blo, h8_t& bhi) {
    blo = half_triple(w.a0, w.b0, w.c0, u & 1, k.mul[u >> 1], k.add[u >> 1]);
    bhi = half_triple(w.a1, w.b1, w.c1, u & 1, k.mul[2 + (u >> 1)], k.add[2 + (u >> 1)]);
  }
};

struct RxQ8_0 : TgQ8_0 {
  static constexpr bool kFold = false, kMin = false, kShortSums = false;  // q * d, rounded once to fp16
  struct K : TgQ8_0::K {
    float d, dmin;
  };
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    TgQ8_0::consts(k, r, lane);
  }
  static __device__ __forceinline__ void frags(const K& k, const W& w, int u, h8_t& blo, h8_t& bhi) {
    TgQ8_0::dequant(k, w, u, blo, bhi);
  }
};

struct RxIQ4XS : TgIQ4XS {
  static constexpr bool kFold = true, kMin = false, kShortSums = false;
  struct K {
    float d, dmin;
    h2_t mul0, add0, mul1, add1;  // ls - 32 and -1152 (ls - 32) of sub-blocks 2g, 2g + 1
  };
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    const int j = 2 * (lane >> 4);
    const uint32_t sh = r.hd.x >> 16, sl = r.hd.y;
    k.d = half_bits_to_float(r.hd.x & 0xffffu);
    k.mul0 = h2_splat((float)((int)(((sl >> (4 * j)) & 15u) | (((sh >> (2 * j)) & 3u) << 4)) - 32));
    k.mul1 = h2_splat((float)((int)(((sl >> (4 * j + 4)) & 15u) | (((sh >> (2 * j + 2)) & 3u) << 4)) - 32));
    k.add0 = k.mul0 * h2_splat(-1152.0f);
    k.add1 = k.mul1 * h2_splat(-1152.0f);
  }
  static __device__ __forceinline__ h8_t frag(uint32_t w, h2_t mul, h2_t add) {
    const uint32_t vlo = FmtIQ4XS::lookup(w), vhi = FmtIQ4XS::lookup_hi(w);
    auto f = [&](uint32_t v, uint32_t sel) { return as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(0x64646464u, v, sel)), mul, add)); };
    return __builtin_bit_cast(h8_t, u4_t{f(vlo, 0x04010400u), f(vlo, 0x04030402u), f(vhi, 0x04010400u), f(vhi, 0x04030402u)});
  }
  static __device__ __forceinline__ void frags(const K& k, const W& w, int, h8_t& blo, h8_t& bhi) {
    blo = frag(w.lo, k.mul0, k.add0);
    bhi = frag(w.hi, k.mul1, k.add1);
  }
};

// ---- the kernel --------------------------------------------------------------
// Workgroup = 8 waves: two K-groups (u-steps 2h and 2h + 1 of each half block)
// of four column groups of two column tiles; all rows (RT row tiles, staged
// as 2 RT: hi and lo) in every workgroup.  Items are (column block, K-slice);
// a workgroup takes items blockIdx, blockIdx + grid, ... and its LDS rings
// (activations NS - 1 half blocks ahead, weights NB blocks) run on across
// them: after the last block of an item the first of the next is already
// under way.  GATED: the wave's two column tiles are one of the gate and the
// same one of the up matrix.
template <class P, int RT>
struct RowsShape {
  static constexpr int kASlot = RT * 8192, kBSlot = 8 * P::kTB, kXch = 2 * 4 * 2 * 1024;
  static constexpr int kXs = P::kMin ? RT * 512 : 0, kXsSlots = P::kMin ? 4 : 0;
  static constexpr int kNS = RT >= 3 ? 2 : RT == 2 ? 3 : 4;
  static constexpr int kLeft = 160 * 1024 - kNS * kASlot - kXch - kXs * kXsSlots - 256;
  static constexpr int kNB = kLeft / kBSlot < 4 ? kLeft / kBSlot : 4;
  static_assert(kNB >= 2, "two blocks of weights");
  static constexpr int kB0 = kNS * kASlot, kX0 = kB0 + kNB * kBSlot, kXs0 = kX0 + kXch, kRs0 = kXs0 + kXs * kXsSlots;
  static constexpr int kLds = kRs0 + 256;  // the rows' unscale factors last
};

template <class P, int RT, bool GATED, int KGI>
__device__ __forceinline__ void rows_run(const MidArgs& a, uint8_t* lds, int wave, int lane) {
  using M = RowsShape<P, RT>;
  constexpr int CT = 2, OT = GATED ? 1 : 2, NS = M::kNS, NB = M::kNB, AD = NS - 1, VT = 2 * RT;
  constexpr int LA = RT, LB = P::kNL;  // one tile-block per wave and block
  constexpr int W0 = mid_wait_count(0, 0, AD, NB, LA, LB), W1 = mid_wait_count(1, 0, AD, NB, LA, LB);
  const int cg = wave & 3, ntiles = a.n >> 4, items = a.cblocks * a.slices;
  const int mine = (items - 1 - (int)blockIdx.x) / (int)gridDim.x + 1;  // items of this workgroup
  // Items of one workgroup are of one slice (slices > 1: one item each).
  const int slice = (int)blockIdx.x % a.slices;
  const int kb0 = slice * a.nb / a.slices, nbr = (slice + 1) * a.nb / a.slices - kb0, steps = 2 * nbr;
  const int total = mine * steps, btotal = mine * nbr;
  auto item_tile = [&](int i) { return (((int)blockIdx.x + i * (int)gridDim.x) / a.slices * 4 + cg) * OT; };
  // This wave loads column KGI of its column group.
  auto weights = [&](int i) {
    const int oc = item_tile(i) + (GATED ? 0 : KGI);
    return uniform_ptr((GATED && KGI == 1 ? a.wu : a.w) + ((size_t)(oc < ntiles ? oc : ntiles - 1) * a.nb + kb0) * P::kTB);
  };
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds)), voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;
  const uint8_t* const xa =
      uniform_ptr(reinterpret_cast<const uint8_t*>(a.xh) + (size_t)kb0 * 65536 + (size_t)((wave >> 2) * 16 + (wave & 3) * RT) * 1024);
  const uint8_t* const xsb =
      uniform_ptr(reinterpret_cast<const uint8_t*>(a.xs) + (P::kMin ? ((size_t)kb0 * RT + (wave < RT ? wave : 0)) * 512 : 0));
  // Cursors of the next activations (step of the item) and weights (block of
  // the item, item) to load, and how many have been.
  int at = 0, ab = 0, an = 0, bb = 0, bi = 0, bn = 0;
  uint32_t aslot = 0, bslot = 0;
  const uint8_t* wp = weights(0);
  auto issue_a = [&] {
    if constexpr (P::kMin) {
      // The block's sub-block sums with its first half (wave w: row tile w).
      if ((at & 1) == 0 && wave < RT) {
        const uint32_t l = lds0 + M::kXs0 + (uint32_t)((an >> 1) & 3) * M::kXs + (uint32_t)wave * 512;
        lds_dma4<0>(xsb + (size_t)ab * (RT * 512), voff4, l);
        lds_dma4<256>(xsb + (size_t)ab * (RT * 512), voff4, l);
      }
    }
    const uint8_t* src = xa + (size_t)at * 32768;
    const uint32_t l = lds0 + aslot * M::kASlot + (uint32_t)wave * (RT * 1024);
    lds_dma16<0>(src, voff16, l);
    if constexpr (RT > 1)
      lds_dma16<1024>(src, voff16, l);
    if constexpr (RT > 2)
      lds_dma16<2048>(src, voff16, l);
    if constexpr (RT > 3)
      lds_dma16<3072>(src, voff16, l);
    aslot = aslot + 1 == NS ? 0 : aslot + 1;
    ++an;
    ++at;
    ab = at >> 1;
    if (at == steps)
      at = ab = 0;
  };
  auto issue_b = [&] {
    P::issue(wp + (size_t)bb * P::kTB, voff16, voff4,
             __builtin_amdgcn_readfirstlane(lds0 + M::kB0 + bslot * M::kBSlot + (uint32_t)(cg * CT + KGI) * P::kTB), lane);
    bslot = bslot + 1 == NB ? 0 : bslot + 1;
    ++bn;
    if (++bb == nbr) {
      bb = 0;
      ++bi;
      wp = weights(bi < mine ? bi : mine - 1);
    }
  };
  const uint8_t* const bl = lds + M::kB0 + cg * CT * P::kTB;

  // Prologue; short items (fewer than AD steps or NB blocks in all) load
  // some of them again so that the loads always number the same.
  if (wave == 0)
    lds_dma4<0>(uniform_ptr(reinterpret_cast<const uint8_t*>(a.rowscale)), voff4, lds0 + M::kRs0);
  issue_b();
#pragma unroll
  for (int t = 0; t < AD; ++t)
    issue_a();
#pragma unroll
  for (int b = 1; b < NB; ++b)
    issue_b();
  mid_wait<AD * LA + (NB - 1) * LB>();
  __syncthreads();
  typename P::K kk[CT];
  h8_t blo[CT], bhi[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    typename P::R r;
    typename P::W w;
    P::raw(r, bl + c * P::kTB, lane);
    P::consts(kk[c], r, lane);
    P::words(w, bl + c * P::kTB, KGI, lane);
    P::frags(kk[c], w, KGI, blo[c], bhi[c]);
  }
  // Up to 32 rows of Q4_K (kShortSums): fp32 sums of four blocks at a time, and a
  // step's low parts before its high ones, so that no sum runs over all of K in
  // full size: N = 66048, K = 4096 against 64 bits 1.80e-7, in one run 2.15e-7;
  // the staged GEMV, whose waves sum one or two blocks, 1.82e-7 (times even:
  // N = 248320, 9 rows 166 against 162 us, 24 rows 207 against 208).  The other
  // types' sums are already closer than the GEMV groups' that they replace
  // (Q5_K 1.94e-7 against 2.05e-7).
  constexpr bool SHORT = P::kShortSums && RT <= 2;
  f4_t acc[RT][CT], blk[RT][CT], far[SHORT ? RT : 1][CT];
  uint32_t as = 0, bs = 0;
  int t = 0, xslot = 0;
  for (int it = 0; it < mine; ++it) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        acc[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (SHORT) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          far[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int b = 0; b < nbr; ++b) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh, ++t) {
        if (total - t > (AD > 2 * NB - 2 ? AD : 2 * NB - 2)) {
          if (hh == 0)
            mid_wait<W0>();
          else
            mid_wait<W1>();
        } else {
          mid_wait<0>();
        }
        __syncthreads();  // step t's operands of every wave landed; step t - 1 fully read
        __builtin_amdgcn_sched_barrier(0);
        if (an < total)
          issue_a();
        if (hh == 1 && bn < btotal)
          issue_b();
        const uint32_t bsn = hh == 0 ? bs : bs + 1 == NB ? 0 : bs + 1;
        const uint8_t* const al = lds + as * M::kASlot + KGI * 2 * VT * 1024 + 16 * lane;
        const uint8_t* const bnx = bl + bsn * M::kBSlot;
        __builtin_amdgcn_sched_barrier(0);
        h8_t af[2][VT];
#pragma unroll
        for (int v = 0; v < VT; ++v)
          af[0][v] = *reinterpret_cast<const h8_t*>(al + (2 * v) * 1024);
        typename P::R r[CT];
        typename P::W wv[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          if (hh == 1)
            P::raw(r[c], bnx + c * P::kTB, lane);
          P::words(wv[c], bnx + c * P::kTB, 2 * (1 - hh) + KGI, lane);
        }
#pragma unroll
        for (int v = 0; v < VT; ++v)
          af[1][v] = *reinterpret_cast<const h8_t*>(al + (2 * v + 1) * 1024);
        // hi then lo parts of every row tile, low- then high-nibble fragments
        // (SHORT: lo parts first, then hi).
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int h = SHORT ? i & 1 : i >> 1, p = SHORT ? 1 - (i >> 1) : i & 1;
#pragma unroll
          for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
              if constexpr (P::kFold)
                blk[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[h][2 * rt + p], h ? bhi[c] : blo[c],
                                                                    hh == 0 && i == 0 ? f4_t{0.0f, 0.0f, 0.0f, 0.0f} : blk[rt][c], 0, 0, 0);
              else
                acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[h][2 * rt + p], h ? bhi[c] : blo[c], acc[rt][c], 0, 0, 0);
            }
        }
        float d[CT], dmin[CT];
        h4_t bmin[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          d[c] = kk[c].d;
          dmin[c] = kk[c].dmin;
          if constexpr (P::kMin)
            bmin[c] = kk[c].bmin;
          if (hh == 1)
            P::consts(kk[c], r[c], lane);
          P::frags(kk[c], wv[c], 2 * (1 - hh) + KGI, blo[c], bhi[c]);
        }
        if constexpr (P::kFold) {
          if (hh == 1) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
              for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  acc[rt][c][v] = fmaf(d[c], blk[rt][c][v], acc[rt][c][v]);
          }
        }
        if constexpr (P::kMin && KGI == 0) {
          if (hh == 0) {
            const uint8_t* const xl = lds + M::kXs0 + (xslot & 3) * M::kXs + 8 * lane;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
              const h4_t xv = *reinterpret_cast<const h4_t*>(xl + rt * 512);
#pragma unroll
              for (int c = 0; c < CT; ++c) {
                const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(xv, bmin[c], f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  acc[rt][c][v] = fmaf(-dmin[c], cm[v], acc[rt][c][v]);
              }
            }
          }
        }
        as = as + 1 == NS ? 0 : as + 1;
        bs = bsn;
        __builtin_amdgcn_sched_barrier(0);
      }
      ++xslot;
      if constexpr (SHORT) {
        if ((b & 3) == 3 || b + 1 == nbr) {
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int c = 0; c < CT; ++c) {
              far[rt][c] += acc[rt][c];
              acc[rt][c] = b + 1 == nbr ? far[rt][c] : f4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
      }
    }
    // The two K-groups' sums, two row tiles at a time: of the pair the wave of
    // K-group 0 finishes the even row tile, that of K-group 1 the odd one.
    const int tile0 = item_tile(it);
    f4_t* const give = reinterpret_cast<f4_t*>(lds + M::kX0) + wave * (CT * 64) + lane;
    const f4_t* const take = reinterpret_cast<const f4_t*>(lds + M::kX0) + (wave ^ 4) * (CT * 64) + lane;
#pragma unroll
    for (int i = 0; i < (RT + 1) / 2; ++i) {
      const int other = 2 * i + 1 - KGI, own = 2 * i + KGI;
      if (i > 0)
        __syncthreads();
      if (other < RT) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          give[c * 64] = acc[other][c];
      }
      __syncthreads();
      if (own < RT && 16 * own < a.m) {
        f4_t s[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c)
          s[c] = acc[own][c] + take[c * 64];
        if (a.slices > 1) {
          const int wide = GATED ? 2 * ntiles : ntiles, live = (a.m + 15) >> 4;
          f4_t* part = reinterpret_cast<f4_t*>(a.part) + ((size_t)slice * live + own) * wide * 64 + lane;
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            const int oc = tile0 + (GATED ? 0 : c);
            if (oc < ntiles)
              part[(size_t)(oc + (GATED && c == 1 ? ntiles : 0)) * 64] = s[c];
          }
        } else {
#pragma unroll
          for (int c = 0; c < OT; ++c)
            if (tile0 + c < ntiles)
              mid_epilogue_tile<GATED>(a, own, tile0 + c, lane, s[c], s[GATED ? 1 : c],
                                       *reinterpret_cast<const f4_t*>(lds + M::kRs0 + 64 * own + 16 * (lane >> 4)));
        }
      }
    }
  }
  mid_wait<0>();
}

template <class P, int RT, bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void rows_gemm_kernel(MidArgs a) {
  using M = RowsShape<P, RT>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[M::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wave < 4)
    rows_run<P, RT, GATED, 0>(a, lds, wave, lane);
  else
    rows_run<P, RT, GATED, 1>(a, lds, wave, lane);
}

template <class P, int RT, bool GATED>
hipError_t rows_launch(hipStream_t s, MidArgs a, int cus) {
  const int ntiles = a.n / 16;
  a.cblocks = GATED ? (ntiles + 3) / 4 : (ntiles + 7) / 8;
  const int items = a.cblocks * a.slices;
  const int grid = a.slices > 1 || items < cus ? items : cus;
  const DispatchEvents ev = dispatch_events();
  if (a.slices > 1)
    dispatch_events() = DispatchEvents{ev.start, nullptr};
  (void)dispatch(rows_gemm_kernel<P, RT, GATED>, dim3((unsigned)grid), dim3(512), s, a);
  if (a.slices > 1) {
    dispatch_events() = DispatchEvents{nullptr, ev.stop};
    (void)launch_mid_reduce(s, a, GATED);
    dispatch_events() = ev;
  }
  return hipGetLastError();
}

template <class P, bool GATED>
hipError_t rows_launch_rt(hipStream_t s, const MidArgs& a, int cus) {
  switch ((a.m + 15) / 16) {
    case 1:
      return rows_launch<P, 1, GATED>(s, a, cus);
    case 2:
      return rows_launch<P, 2, GATED>(s, a, cus);
    case 3:
      return rows_launch<P, 3, GATED>(s, a, cus);
    case 4:
      if constexpr (!P::kShortSums)  // Q4_K comes with at most 48 rows
        return rows_launch<P, 4, GATED>(s, a, cus);
      [[fallthrough]];
    default:
      return hipErrorInvalidValue;
  }
}

template <class P>
hipError_t rows_launch_any(hipStream_t s, const MidArgs& a, bool gated, int cus) {
  return gated ? rows_launch_rt<P, true>(s, a, cus) : rows_launch_rt<P, false>(s, a, cus);
}

}  // namespace

hipError_t launch_rows_gemm(hipStream_t s, const MidArgs& a, uint32_t type, bool gated, int cus) {
  if (a.m < 1 || a.m > 64 || a.n % 16 != 0 || a.n < 16 || a.slices < 1 || a.slices > a.nb || (a.slices > 1 && !a.part) || (gated && !a.wu) || !a.xs)
    return hipErrorInvalidValue;
  switch (type) {
    case kTypeQ4_K:
      // Q4_K pairs take the decode and rows GEMVs.
      return gated ? hipErrorInvalidValue : rows_launch_rt<RxQ4K, false>(s, a, cus);
    case kTypeQ5_K:
      return rows_launch_any<RxQ5K>(s, a, gated, cus);
    case kTypeQ6_K:
      return rows_launch_any<RxQ6K>(s, a, gated, cus);
    case kTypeQ8_0:
      return rows_launch_any<RxQ8_0>(s, a, gated, cus);
    case kTypeIQ4_XS:
      return rows_launch_any<RxIQ4XS>(s, a, gated, cus);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace q4k
