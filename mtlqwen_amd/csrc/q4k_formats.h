// Format policies of the weight types, shared by the kernel sources: the
// decode GEMVs' (Fmt*: the registers of one tile-block per lane, their loads
// and the MFMA operands as exact quant x scale products) and the prefill
// GEMMs' (Tg*: a tile-block in LDS, dequantised to the reference's prefill
// tile value).
#pragma once
#include "q4k_device.h"

namespace q4k {
namespace {

struct XF {
  h8_t f[8];
  float dv[4];
  h4_t xs;
};

template <bool MIN>
__device__ __forceinline__ void load_xf(XF& xf, const DecodePack& pk, size_t b, int lane) {
  const u4_t* fr = pk.frag + b * 8 * 64 + lane;
#pragma unroll
  for (int fs = 0; fs < 8; ++fs)
    xf.f[fs] = __builtin_bit_cast(h8_t, fr[fs * 64]);
  const float* ds = pk.dsc + b * 8 + 4 * ((lane >> 4) & 1);
#pragma unroll
  for (int v = 0; v < 4; ++v)
    xf.dv[v] = ds[v];
  if constexpr (MIN)
    xf.xs = pk.xs[b * 64 + lane];
}

__device__ __forceinline__ h2_t h2_splat(float v) {
  return h2_t{(_Float16)v, (_Float16)v};
}

// Outputs o = 8a .. 8a+7 of Q6_K triple (A, B, C) times their scale: b0 = MFMA
// 2a's four B dwords, b1 = MFMA 2a + 1's (layout in q4k_internal.h).
__device__ __forceinline__ void q6_triple(uint32_t A, uint32_t B, uint32_t C, h2_t mul, h2_t add, h8_t& b0, h8_t& b1) {
  const uint32_t m6 = 0x03F003F0u, m4 = 0x00F000F0u, m2 = 0x03000300u, magic = 0x64006400u;
  const uint32_t o0 = and_or(A, m6, magic), o1 = and_or(A >> 6, m6, magic);
  const uint32_t o2 = and_or(B, m6, magic), o3 = and_or(B >> 6, m6, magic);
  const uint32_t o4 = and_or(C, m6, magic), o5 = and_or(C >> 6, m6, magic);
  const uint32_t o6 = and_or(A << 4, m4, and_or(B << 8, m2, magic));
  const uint32_t o7 = and_or(C << 4, m4, and_or(B << 6, m2, magic));
  auto f = [&](uint32_t o) { return as_u32(__builtin_elementwise_fma(as_h2(o), mul, add)); };
  b0 = __builtin_bit_cast(h8_t, u4_t{f(o0), f(o1), f(o2), f(o3)});
  b1 = __builtin_bit_cast(h8_t, u4_t{f(o4), f(o5), f(o6), f(o7)});
}

// Each policy also names the shape of its persistent form: kPW waves (16:
// one block of x each, within 128 VGPRs, four waves per SIMD; 8: two blocks
// each, two waves per SIMD) and kPT column tiles per item, the measured best
// that does not spill.
struct FmtQ6K {
  static constexpr int kTB = kQ6TileBlockBytes;
  static constexpr bool kMin = false;
  static constexpr int kPW = 16, kPT = 2;
  struct U {
    u4_t s0, s1, s2;
    uint32_t sc, d;
  };
  static __device__ __forceinline__ void load(U& u, const uint8_t* src, int lane) {
    u.s0 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src) + lane);
    u.s1 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + 1024) + lane);
    u.s2 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + 2048) + lane);
    u.sc = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(src + kQ6ScaleOffset) + lane);
    u.d = *(reinterpret_cast<const uint16_t*>(src + kQ6DOffset) + (lane & 15));
  }
  static __device__ __forceinline__ void mac(const U& u, const XF& x, int, f4_t& acc) {
    const float d = half_bits_to_float(u.d & 0xffffu);
    f4_t c0 = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, c1 = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    // Triple tr = dwords 3tr..3tr+2 of the lane's twelve (named directly: a
    // local array of them is not always kept in registers).
    auto triple = [&](int tr, uint32_t A, uint32_t B, uint32_t C) {
      // fp16 1152 + sc -> sc / 16 (exact), and -96 sc.
      const uint32_t sel = 0x04000400u | (uint32_t)tr | ((uint32_t)tr << 16);
      const h2_t p = as_h2(__builtin_amdgcn_perm(0x64646464u, u.sc, sel));
      const h2_t mul = __builtin_elementwise_fma(p, h2_splat(0.0625f), h2_splat(-72.0f));
      const h2_t add = mul * h2_splat(-1536.0f);
      h8_t b0, b1;
      q6_triple(A, B, C, mul, add, b0, b1);
      c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[2 * tr], b0, c0, 0, 0, 0);
      c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[2 * tr + 1], b1, c1, 0, 0, 0);
    };
    triple(0, u.s0[0], u.s0[1], u.s0[2]);
    triple(1, u.s0[3], u.s1[0], u.s1[1]);
    triple(2, u.s1[2], u.s1[3], u.s2[0]);
    triple(3, u.s2[1], u.s2[2], u.s2[3]);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[v] = fmaf(c0[v] + c1[v], d * x.dv[v], acc[v]);
  }
};

struct FmtQ8_0 {
  static constexpr int kTB = kTileN * kQ8BlockBytes;
  static constexpr bool kMin = false;
  static constexpr int kPW = 16, kPT = 2;
  struct U {
    u4_t s[4];
    uint32_t d;
  };
  static __device__ __forceinline__ void load(U& u, const uint8_t* src, int lane) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      u.s[j] = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + 1024 * j) + lane);
    u.d = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(src + 4096) + lane);
  }
  static __device__ __forceinline__ void mac(const U& u, const XF& x, int, f4_t& acc) {
    // d of the lane's two records, each in both halves.
    const h2_t d0 = as_h2(__builtin_amdgcn_perm(u.d, u.d, 0x01000100u)), d1 = as_h2(__builtin_amdgcn_perm(u.d, u.d, 0x03020302u));
    const h2_t k1152 = h2_splat(-1152.0f);
    f4_t c0 = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, c1 = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int fs = 0; fs < 8; ++fs) {
      const u4_t sl = u.s[fs >> 1];
      const uint32_t w0 = sl[2 * (fs & 1)], w1 = sl[2 * (fs & 1) + 1];
      const h2_t d = fs < 4 ? d0 : d1;
      auto q = [&](uint32_t w, uint32_t sel) { return as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) + k1152) * d); };
      const h8_t b = __builtin_bit_cast(h8_t, u4_t{q(w0, 0x04010400u), q(w0, 0x04030402u), q(w1, 0x04010400u), q(w1, 0x04030402u)});
      if (fs & 1)
        c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[fs], b, c1, 0, 0, 0);
      else
        c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[fs], b, c0, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[v] = fmaf(c0[v] + c1[v], x.dv[v], acc[v]);
  }
};

struct FmtQ5K {
  static constexpr int kTB = kTileN * kQ5BlockBytes;
  static constexpr bool kMin = true;
  static constexpr int kPW = 8, kPT = 2;
  struct U {
    u4_t q0, q1, hd;
    uint32_t h0, h1;
  };
  static __device__ __forceinline__ void load(U& u, const uint8_t* src, int lane) {
    u.q0 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src) + lane);
    u.q1 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + kSlabBytes) + lane);
    u.hd = *(reinterpret_cast<const u4_t*>(src + kHeaderOffset) + (lane & 15));
    typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
    const u2_t h = __builtin_nontemporal_load(reinterpret_cast<const u2_t*>(src + 2304) + lane);
    u.h0 = h[0];
    u.h1 = h[1];
  }
  // Fifth bits of B dword k (= 4 (fs % 4) + t) moved to bit P of each half,
  // or'ed with the fp16 bias 0x6400.
  template <int P>
  static __device__ __forceinline__ uint32_t bias(uint32_t h, int k) {
    const uint32_t moved = k < P ? h << (P - k) : h >> (k - P);
    return and_or(moved, (1u << P) | (1u << (16 + P)), 0x64006400u);
  }
  static __device__ __forceinline__ void mac(const U& u, const XF& x, int lane, f4_t& acc) {
    const BlockConsts kc = block_consts(u.hd, lane >> 4);
    f4_t cl = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, ch = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u4_t qq = s < 2 ? u.q0 : u.q1;
      const uint32_t wa = qq[2 * (s & 1)], wb = qq[2 * (s & 1) + 1];
      const uint32_t src[4] = {wa, wa >> 8, wb, wb >> 8};
      u4_t lo, hi;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        lo[t] = as_u32(__builtin_elementwise_fma(as_h2(and_or(src[t], 0x000F000Fu, bias<4>(u.h0, 4 * s + t))), kc.mul_lo, kc.add_lo));
        hi[t] = as_u32(__builtin_elementwise_fma(as_h2(and_or(src[t], 0x00F000F0u, bias<8>(u.h1, 4 * s + t))), kc.mul_hi, kc.add_hi));
      }
      cl = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[s], __builtin_bit_cast(h8_t, lo), cl, 0, 0, 0);
      ch = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[4 + s], __builtin_bit_cast(h8_t, hi), ch, 0, 0, 0);
    }
    const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(x.xs, kc.bmin, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[v] += fmaf(kc.d, cl[v] + ch[v], -kc.dmin * cm[v]) * x.dv[v];
  }
};

// Q4_K itself in the same form (the tiled layout of q4k_internal.h), for the
// wide decode projections (the LM head) the persistent form serves best.
struct FmtQ4K {
  static constexpr int kTB = kTileBlockBytes;
  static constexpr bool kMin = true;
  static constexpr int kPW = 16, kPT = 2;
  struct U {
    u4_t q0, q1, hd;
  };
  static __device__ __forceinline__ void load(U& u, const uint8_t* src, int lane) {
    u.q0 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src) + lane);
    u.q1 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + kSlabBytes) + lane);
    u.hd = *(reinterpret_cast<const u4_t*>(src + kHeaderOffset) + (lane & 15));
  }
  static __device__ __forceinline__ void mac(const U& u, const XF& x, int lane, f4_t& acc) {
    const BlockConsts kc = block_consts(u.hd, lane >> 4);
    f4_t cl = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, ch = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u4_t qq = s < 2 ? u.q0 : u.q1;
      const uint32_t wa = qq[2 * (s & 1)], wb = qq[2 * (s & 1) + 1];
      const h8_t blo = quant_times_scale(wa, wb, 0x000F000Fu, 0x64006400u, kc.mul_lo, kc.add_lo);
      const h8_t bhi = quant_times_scale(wa, wb, 0x00F000F0u, 0x64006400u, kc.mul_hi, kc.add_hi);
      cl = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[s], blo, cl, 0, 0, 0);
      ch = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[4 + s], bhi, ch, 0, 0, 0);
    }
    const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(x.xs, kc.bmin, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[v] += fmaf(kc.d, cl[v] + ch[v], -kc.dmin * cm[v]) * x.dv[v];
  }
};

struct FmtIQ4XS {
  static constexpr int kTB = kTileN * kIQ4BlockBytes;
  static constexpr bool kMin = false;
  static constexpr int kPW = 16, kPT = 2;
  struct U {
    u4_t q0, q1;
    uint2 hd;
  };
  static __device__ __forceinline__ void load(U& u, const uint8_t* src, int lane) {
    u.q0 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src) + lane);
    u.q1 = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + 1024) + lane);
    u.hd = *(reinterpret_cast<const uint2*>(src + 2048) + (lane & 15));
  }
  // Codebook entries (iq4nl, quant_linear.metal:5) + 128 as bytes, four per word.
  static constexpr uint32_t kT0 = 0x3F2D1801u, kT1 = 0x766A5D4Fu, kT2 = 0xA6998D81u, kT3 = 0xF1D9C5B5u;
  // Four codebook bytes for the four 4-bit indices at bits 0..3 of each byte of w.
  static __device__ __forceinline__ uint32_t lookup(uint32_t w) {
    const uint32_t t = w & 0x07070707u;
    const uint32_t a = __builtin_amdgcn_perm(kT1, kT0, t), b = __builtin_amdgcn_perm(kT3, kT2, t);
    // Selector byte 0x0C gives 0x00, 0x0D gives 0xFF: a byte mask of bit 3.
    const uint32_t m = __builtin_amdgcn_perm(0u, 0u, and_or(w >> 3, 0x01010101u, 0x0C0C0C0Cu));
    return (m & b) | (~m & a);
  }
  // The same for the indices at bits 4..7 of each byte.  Bit 3 of index b is
  // bit 7 of byte b, which selectors 8..11 turn into a byte mask directly
  // (0x00 or 0xFF from bit 15 / 31 of the second source, bit 15 / 31 of the
  // first): bytes 1, 3 from w, bytes 0, 2 from w << 8.
  static __device__ __forceinline__ uint32_t lookup_hi(uint32_t w) {
    const uint32_t t = (w >> 4) & 0x07070707u;
    const uint32_t a = __builtin_amdgcn_perm(kT1, kT0, t), b = __builtin_amdgcn_perm(kT3, kT2, t);
    const uint32_t m = __builtin_amdgcn_perm(w << 8, w, 0x090B080Au);
    return (m & b) | (~m & a);
  }
  static __device__ __forceinline__ void mac(const U& u, const XF& x, int lane, f4_t& acc) {
    const int g = lane >> 4;
    const uint32_t sh = u.hd.x >> 16, sl = u.hd.y;
    const float d = half_bits_to_float(u.hd.x & 0xffffu);
    // ls - 32 of sub-blocks 2g (MFMAs 0..3) and 2g + 1 (MFMAs 4..7).
    const int j0 = 2 * g;
    const int ls0 = (int)(((sl >> (4 * j0)) & 15u) | (((sh >> (2 * j0)) & 3u) << 4)) - 32;
    const int ls1 = (int)(((sl >> (4 * j0 + 4)) & 15u) | (((sh >> (2 * j0 + 2)) & 3u) << 4)) - 32;
    const h2_t mul0 = h2_splat((float)ls0), mul1 = h2_splat((float)ls1);
    const h2_t add0 = mul0 * h2_splat(-1152.0f), add1 = mul1 * h2_splat(-1152.0f);
    f4_t c0 = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, c1 = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int fs = 0; fs < 8; ++fs) {
      const uint32_t w = (fs < 4 ? u.q0 : u.q1)[fs & 3];
      const uint32_t vlo = lookup(w), vhi = lookup_hi(w);
      const h2_t mul = fs < 4 ? mul0 : mul1, add = fs < 4 ? add0 : add1;
      auto f = [&](uint32_t v, uint32_t sel) {
        return as_u32(__builtin_elementwise_fma(as_h2(__builtin_amdgcn_perm(0x64646464u, v, sel)), mul, add));
      };
      const h8_t b = __builtin_bit_cast(h8_t, u4_t{f(vlo, 0x04010400u), f(vlo, 0x04030402u), f(vhi, 0x04010400u), f(vhi, 0x04030402u)});
      if (fs & 1)
        c1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[fs], b, c1, 0, 0, 0);
      else
        c0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.f[fs], b, c0, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
      acc[v] = fmaf(c0[v] + c1[v], d * x.dv[v], acc[v]);
  }
};

// Bit `from` (and from + 16) of h moved to bit `to` (and to + 16).
__device__ __forceinline__ uint32_t move_bits(uint32_t h, int from, int to) {
  return from >= to ? h >> (from - to) : h << (to - from);
}

// Two fp16 pairs from four fp32 values, each rounded once: the four values
// are formed before either conversion (the empty asm keeps them apart from
// it), so that no conversion directly follows the v_fma_mix that wrote its
// source (that adjacency costs two wait states).
__device__ __forceinline__ void pack_h2x2(float a0, float a1, float b0, float b1, uint32_t& lo, uint32_t& hi) {
  asm("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
  lo = as_u32(h2_t{(_Float16)a0, (_Float16)a1});
  hi = as_u32(h2_t{(_Float16)b0, (_Float16)b1});
}

__device__ __forceinline__ uint32_t lds_u32(const uint8_t* p) {
  return *reinterpret_cast<const uint32_t*>(p);
}

struct TgQ5K {
  static constexpr int kTB = kTileN * kQ5BlockBytes, kCT = 4, kAS = 4, kNL = 5, kVPM = 2;
  struct R {
    u4_t hd;
    uint2 h;
  };
  struct K {
    float dl, cl, dh, ch;
    uint32_t h0, h1;
  };
  struct W {
    uint2 q;
  };
  static __device__ __forceinline__ void issue(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l, int) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<kSlabBytes>(src, v16, l);
    lds_dma4<kHeaderOffset>(src, v4, l);
    lds_dma4<2304>(src, v4, l);
    lds_dma4<2560>(src, v4, l);
  }
  static __device__ __forceinline__ void raw(R& r, const uint8_t* tb, int lane) {
    r.hd = *reinterpret_cast<const u4_t*>(tb + kHeaderOffset + 16 * (lane & 15));
    r.h = *reinterpret_cast<const uint2*>(tb + 2304 + 8 * lane);
  }
  // Sub-blocks 2g (low nibbles) and 2g + 1 (high nibbles): d * sc times
  // 2^24 (2^20), and -dmin * m.
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    uint32_t p0, p1;
    scale_min_packed(r.hd, lane >> 4, p0, p1);
    const float d = half_bits_to_float(r.hd.x & 0xffffu), dm = half_bits_to_float(r.hd.x >> 16);
    k.dl = d * (float)(p0 & 0xffu) * 0x1p24f;
    k.cl = -dm * (float)((p0 >> 16) & 0xffu);
    k.dh = d * (float)(p1 & 0xffu) * 0x1p20f;
    k.ch = -dm * (float)((p1 >> 16) & 0xffu);
    k.h0 = r.h.x;
    k.h1 = r.h.y;
  }
  static __device__ __forceinline__ void words(W& w, const uint8_t* tb, int u, int lane) {
    w.q = *reinterpret_cast<const uint2*>(tb + (u >> 1) * kSlabBytes + 16 * lane + 8 * (u & 1));
  }
  // B dword t of MFMA u (low nibbles): fifth bits at bit 4u + t (+16) of h0;
  // of MFMA 4 + u (high nibbles): the same bits of h1.  The value is the fp16
  // denormal (q + 16h) * 2^-24 (low nibble at bit 0, fifth bit at bit 4) or
  // (q + 16h) * 2^-20 (nibble at bits 4..7, fifth bit at bit 8).
  static __device__ __forceinline__ void dequant(const K& k, const W& w, int u, h8_t& blo, h8_t& bhi) {
    const uint32_t lw[4] = {w.q.x, w.q.x >> 8, w.q.y, w.q.y >> 8};
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const h2_t ql = as_h2(and_or(lw[t], 0x000F000Fu, move_bits(k.h0, 4 * u + t, 4) & 0x00100010u));
      const h2_t qh = as_h2(and_or(lw[t], 0x00F000F0u, move_bits(k.h1, 4 * u + t, 8) & 0x01000100u));
      pack_h2x2(__builtin_fmaf((float)ql[0], k.dl, k.cl), __builtin_fmaf((float)ql[1], k.dl, k.cl), __builtin_fmaf((float)qh[0], k.dh, k.ch),
                __builtin_fmaf((float)qh[1], k.dh, k.ch), lo[t], hi[t]);
    }
    blo = __builtin_bit_cast(h8_t, u4_t{lo[0], lo[1], lo[2], lo[3]});
    bhi = __builtin_bit_cast(h8_t, u4_t{hi[0], hi[1], hi[2], hi[3]});
  }
};

struct TgQ6K {
  static constexpr int kTB = kQ6TileBlockBytes, kCT = 4, kAS = 3, kNL = 5, kVPM = 2;
  struct R {
    uint32_t sc, d;
  };
  // d * sc of the lane's four scale bytes (MFMAs u and 4 + u take bytes u / 2
  // and 2 + u / 2), formed once per block.
  struct K {
    float ds[4];
  };
  // Triples u / 2 (MFMA u) and 2 + u / 2 (MFMA 4 + u); C only for odd u.
  struct W {
    uint32_t a0, b0, c0, a1, b1, c1;
  };
  static __device__ __forceinline__ void issue(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l, int lane) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<1024>(src, v16, l);
    lds_dma16<2048>(src, v16, l);
    lds_dma4<kQ6ScaleOffset>(src, v4, l);
    if (lane < 8)  // the 16 rows' d: 32 bytes
      lds_dma4<kQ6DOffset>(src, v4, l);
  }
  static __device__ __forceinline__ void raw(R& r, const uint8_t* tb, int lane) {
    r.sc = lds_u32(tb + kQ6ScaleOffset + 4 * lane);
    r.d = *reinterpret_cast<const uint16_t*>(tb + kQ6DOffset + 2 * (lane & 15));
  }
  // Scale byte i is stored sc + 128: d * sc = fma(sc + 128, d, -128 d), exact.
  static __device__ __forceinline__ void consts(K& k, const R& r, int) {
    const float d = half_bits_to_float(r.d), m128 = -128.0f * d;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      k.ds[i] = __builtin_fmaf((float)((r.sc >> (8 * i)) & 0xffu), d, m128);
  }
  static __device__ __forceinline__ uint32_t dword(const uint8_t* tb, int j, int lane) {
    return lds_u32(tb + (j >> 2) * 1024 + 16 * lane + 4 * (j & 3));
  }
  static __device__ __forceinline__ void words(W& w, const uint8_t* tb, int u, int lane) {
    const int a = 3 * (u >> 1);
    w.a0 = dword(tb, a, lane);
    w.b0 = dword(tb, a + 1, lane);
    w.a1 = dword(tb, a + 6, lane);
    w.b1 = dword(tb, a + 7, lane);
    w.c0 = (u & 1) ? dword(tb, a + 2, lane) : 0u;
    w.c1 = (u & 1) ? dword(tb, a + 8, lane) : 0u;
  }
  // Outputs 8a + 4p .. 8a + 4p + 3 of triple (A, B, C) (p = u & 1) as fp16
  // 64 + q (bias 0x5400: bit 4 of a half is 1), then d*sc*(q - 32) exactly.
  static __device__ __forceinline__ h8_t triple(uint32_t A, uint32_t B, uint32_t C, int p, float ds) {
    const uint32_t m6 = 0x03F003F0u, m4 = 0x00F000F0u, m2 = 0x03000300u, bias = 0x54005400u;
    uint32_t o[4];
    if (p == 0) {
      o[0] = and_or(A, m6, bias);
      o[1] = and_or(A >> 6, m6, bias);
      o[2] = and_or(B, m6, bias);
      o[3] = and_or(B >> 6, m6, bias);
    } else {
      o[0] = and_or(C, m6, bias);
      o[1] = and_or(C >> 6, m6, bias);
      o[2] = and_or(A << 4, m4, and_or(B << 8, m2, bias));
      o[3] = and_or(C << 4, m4, and_or(B << 6, m2, bias));
    }
    const float c = -96.0f * ds;
    uint32_t r[4];
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
      const h2_t q = as_h2(o[t]), p = as_h2(o[t + 1]);
      pack_h2x2(__builtin_fmaf((float)q[0], ds, c), __builtin_fmaf((float)q[1], ds, c), __builtin_fmaf((float)p[0], ds, c),
                __builtin_fmaf((float)p[1], ds, c), r[t], r[t + 1]);
    }
    return __builtin_bit_cast(h8_t, u4_t{r[0], r[1], r[2], r[3]});
  }
  // Scale of MFMA u: byte u / 2 of the lane's scale dword; of MFMA 4 + u:
  // byte 2 + u / 2.
  static __device__ __forceinline__ void dequant(const K& k, const W& w, int u, h8_t& blo, h8_t& bhi) {
    blo = triple(w.a0, w.b0, w.c0, u & 1, k.ds[u >> 1]);
    bhi = triple(w.a1, w.b1, w.c1, u & 1, k.ds[2 + (u >> 1)]);
  }
};

struct TgQ8_0 {
  static constexpr int kTB = kTileN * kQ8BlockBytes, kCT = 2, kAS = 5, kNL = 5, kVPM = 2;
  struct R {
    uint32_t dd;
  };
  struct K {
    h2_t dl, dh;
  };
  struct W {
    uint2 lo, hi;
  };
  static __device__ __forceinline__ void issue(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l, int) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<1024>(src, v16, l);
    lds_dma16<2048>(src, v16, l);
    lds_dma16<3072>(src, v16, l);
    lds_dma4<0>(src + 4096, v4, l + 4096);  // past the instruction offset's range
  }
  static __device__ __forceinline__ void raw(R& r, const uint8_t* tb, int lane) {
    r.dd = lds_u32(tb + 4096 + 4 * lane);
  }
  // d of records 2g (MFMAs 0..3) and 2g + 1 (MFMAs 4..7), in both halves.
  static __device__ __forceinline__ void consts(K& k, const R& r, int) {
    k.dl = as_h2(__builtin_amdgcn_perm(r.dd, r.dd, 0x01000100u));
    k.dh = as_h2(__builtin_amdgcn_perm(r.dd, r.dd, 0x03020302u));
  }
  static __device__ __forceinline__ void words(W& w, const uint8_t* tb, int u, int lane) {
    w.lo = *reinterpret_cast<const uint2*>(tb + (u >> 1) * 1024 + 16 * lane + 8 * (u & 1));
    w.hi = *reinterpret_cast<const uint2*>(tb + (2 + (u >> 1)) * 1024 + 16 * lane + 8 * (u & 1));
  }
  // Byte q ^ 0x80 as fp16 1024 + (q + 128), minus 1152 (exact), times d.
  static __device__ __forceinline__ h8_t frag(uint2 v, h2_t d) {
    auto q = [&](uint32_t x, uint32_t sel) { return as_u32((as_h2(__builtin_amdgcn_perm(0x64646464u, x, sel)) + h2_splat(-1152.0f)) * d); };
    return __builtin_bit_cast(h8_t, u4_t{q(v.x, 0x04010400u), q(v.x, 0x04030402u), q(v.y, 0x04010400u), q(v.y, 0x04030402u)});
  }
  static __device__ __forceinline__ void dequant(const K& k, const W& w, int, h8_t& blo, h8_t& bhi) {
    blo = frag(w.lo, k.dl);
    bhi = frag(w.hi, k.dh);
  }
};

// Q8_0 with four column tiles per wave: two blocks of its 4352-byte
// tile-blocks per column do not fit beside an A ring, so B streams in half
// tile-blocks through three half-slots per column (typed_gemm_tile_half).
// Half 0 of a tile-block holds the quant slabs of u-steps 0, 1 (slabs 0 and
// 2: the low and high MFMA fragments) and the d row, half 1 the slabs of
// u-steps 2, 3 (slabs 1 and 3).  A half-slot: [low slab 1 KB][high slab
// 1 KB][d row 256 B].
struct TgQ8_0W : TgQ8_0 {
  static constexpr int kCT = 4, kAS = 3, kHS = 2304, kL0 = 3, kL1 = 2;
  static constexpr bool kHalf = true;
  static __device__ __forceinline__ void issue_half0(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<1024>(src + 1024, v16, l);  // slab 2 into [1 KB, 2 KB)
    lds_dma4<0>(src + 4096, v4, l + 2048);
  }
  static __device__ __forceinline__ void issue_half1(const uint8_t* src, uint32_t v16, uint32_t l) {
    lds_dma16<0>(src + 1024, v16, l);     // slab 1
    lds_dma16<1024>(src + 2048, v16, l);  // slab 3 into [1 KB, 2 KB)
  }
  static __device__ __forceinline__ void raw_half(R& r, const uint8_t* hs, int lane) {
    r.dd = lds_u32(hs + 2048 + 4 * lane);
  }
  static __device__ __forceinline__ void words_half(W& w, const uint8_t* hs, int u, int lane) {
    w.lo = *reinterpret_cast<const uint2*>(hs + 16 * lane + 8 * (u & 1));
    w.hi = *reinterpret_cast<const uint2*>(hs + 1024 + 16 * lane + 8 * (u & 1));
  }
};

template <class P, class = void>
struct TgIsHalf {
  static constexpr bool value = false;
};
template <class P>
struct TgIsHalf<P, decltype((void)P::kHalf)> {
  static constexpr bool value = P::kHalf;
};

struct TgIQ4XS {
  static constexpr int kTB = kTileN * kIQ4BlockBytes, kCT = 4, kAS = 5, kNL = 3, kVPM = 4;
  struct R {
    uint2 hd;
  };
  struct K {
    float dl, cl, dh, ch;
  };
  struct W {
    uint32_t lo, hi;
  };
  static __device__ __forceinline__ void issue(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l, int lane) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<1024>(src, v16, l);
    if (lane < 32)  // the 16 rows' 8-byte headers: 128 bytes
      lds_dma4<2048>(src, v4, l);
  }
  static __device__ __forceinline__ void raw(R& r, const uint8_t* tb, int lane) {
    r.hd = *reinterpret_cast<const uint2*>(tb + 2048 + 8 * (lane & 15));
  }
  // Sub-blocks 2g (MFMAs 0..3) and 2g + 1 (4..7): dl = d * (ls - 32) and
  // -1152 dl, both exact.
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    const int j = 2 * (lane >> 4);
    const uint32_t sh = r.hd.x >> 16, sl = r.hd.y;
    const float d = half_bits_to_float(r.hd.x & 0xffffu);
    const int ls0 = (int)(((sl >> (4 * j)) & 15u) | (((sh >> (2 * j)) & 3u) << 4));
    const int ls1 = (int)(((sl >> (4 * j + 4)) & 15u) | (((sh >> (2 * j + 2)) & 3u) << 4));
    k.dl = d * (float)(ls0 - 32);
    k.cl = -1152.0f * k.dl;
    k.dh = d * (float)(ls1 - 32);
    k.ch = -1152.0f * k.dh;
  }
  static __device__ __forceinline__ void words(W& w, const uint8_t* tb, int u, int lane) {
    w.lo = lds_u32(tb + 16 * lane + 4 * u);
    w.hi = lds_u32(tb + 1024 + 16 * lane + 4 * u);
  }
  // Codebook value + 128 per byte (FmtIQ4XS::lookup) as fp16 1152 + v, then
  // dl * v exactly.
  static __device__ __forceinline__ h8_t frag(uint32_t wq, float dl, float cl) {
    const uint32_t vlo = FmtIQ4XS::lookup(wq), vhi = FmtIQ4XS::lookup_hi(wq);
    const uint32_t p[4] = {__builtin_amdgcn_perm(0x64646464u, vlo, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, vlo, 0x04030402u),
                           __builtin_amdgcn_perm(0x64646464u, vhi, 0x04010400u), __builtin_amdgcn_perm(0x64646464u, vhi, 0x04030402u)};
    uint32_t r[4];
#pragma unroll
    for (int t = 0; t < 4; t += 2) {
      const h2_t v = as_h2(p[t]), w = as_h2(p[t + 1]);
      pack_h2x2(__builtin_fmaf((float)v[0], dl, cl), __builtin_fmaf((float)v[1], dl, cl), __builtin_fmaf((float)w[0], dl, cl),
                __builtin_fmaf((float)w[1], dl, cl), r[t], r[t + 1]);
    }
    return __builtin_bit_cast(h8_t, u4_t{r[0], r[1], r[2], r[3]});
  }
  static __device__ __forceinline__ void dequant(const K& k, const W& w, int, h8_t& blo, h8_t& bhi) {
    blo = frag(w.lo, k.dl, k.cl);
    bhi = frag(w.hi, k.dh, k.ch);
  }
};

// Q4_K on the same template, two column tiles per wave (128 columns per
// workgroup): for prefill grids that the 256-column Q4_K GEMM leaves short of
// the CUs.  The dequantisation is that GEMM's (fp16 denormal nibbles, one
// fp32 fma with d*sc*2^24 or d*sc*2^20 and -dmin*m): the reference's value
// exactly.
struct TgQ4K {
  static constexpr int kTB = kTileBlockBytes, kCT = 2, kAS = 5, kNL = 3, kVPM = 2;
  struct R {
    u4_t hd;
  };
  struct K {
    float dl, cl, dh, ch;
  };
  struct W {
    uint2 q;
  };
  static __device__ __forceinline__ void issue(const uint8_t* src, uint32_t v16, uint32_t v4, uint32_t l, int) {
    lds_dma16<0>(src, v16, l);
    lds_dma16<kSlabBytes>(src, v16, l);
    lds_dma4<kHeaderOffset>(src, v4, l);
  }
  static __device__ __forceinline__ void raw(R& r, const uint8_t* tb, int lane) {
    r.hd = *reinterpret_cast<const u4_t*>(tb + kHeaderOffset + 16 * (lane & 15));
  }
  static __device__ __forceinline__ void consts(K& k, const R& r, int lane) {
    uint32_t p0, p1;
    scale_min_packed(r.hd, lane >> 4, p0, p1);
    const float d = half_bits_to_float(r.hd.x & 0xffffu), dm = half_bits_to_float(r.hd.x >> 16);
    k.dl = d * (float)(p0 & 0xffu) * 0x1p24f;
    k.cl = -dm * (float)((p0 >> 16) & 0xffu);
    k.dh = d * (float)(p1 & 0xffu) * 0x1p20f;
    k.ch = -dm * (float)((p1 >> 16) & 0xffu);
  }
  static __device__ __forceinline__ void words(W& w, const uint8_t* tb, int u, int lane) {
    w.q = *reinterpret_cast<const uint2*>(tb + (u >> 1) * kSlabBytes + 16 * lane + 8 * (u & 1));
  }
  static __device__ __forceinline__ void dequant(const K& k, const W& w, int, h8_t& blo, h8_t& bhi) {
    const uint32_t lw[4] = {w.q.x, w.q.x >> 8, w.q.y, w.q.y >> 8};
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const h2_t ql = as_h2(lw[t] & 0x000F000Fu), qh = as_h2(lw[t] & 0x00F000F0u);
      pack_h2x2(__builtin_fmaf((float)ql[0], k.dl, k.cl), __builtin_fmaf((float)ql[1], k.dl, k.cl), __builtin_fmaf((float)qh[0], k.dh, k.ch),
                __builtin_fmaf((float)qh[1], k.dh, k.ch), lo[t], hi[t]);
    }
    blo = __builtin_bit_cast(h8_t, u4_t{lo[0], lo[1], lo[2], lo[3]});
    bhi = __builtin_bit_cast(h8_t, u4_t{hi[0], hi[1], hi[2], hi[3]});
  }
};

// A policy with two column tiles per wave (128 columns per workgroup) and a
// 5-slot A ring, for grids the 4-tile form leaves short of the CUs.
template <class P>
struct Narrow : P {
  static constexpr int kCT = 2, kAS = 5;
};

// Three column tiles per wave (192 columns per workgroup): the B ring is
// three quarters of the 4-tile form's, which leaves LDS for a deeper A ring
// (Q6_K: 5 slots instead of 3) or more MFMAs per A fragment read (Q8_0).
template <class P, int AS>
struct Mid : P {
  static constexpr int kCT = 3, kAS = AS;
};

// Six column tiles per wave (384 columns per workgroup, or 192 output
// columns of the gated GEMM: three gate and three up tiles) with a 3-slot A
// ring (156 KB of LDS with Q4_K, 150 KB with IQ4_XS): each A fragment read
// from LDS feeds six column tiles.
template <class P>
struct Six : P {
  static constexpr int kCT = 6, kAS = 3;
};
// IQ4_XS: six vector instructions per MFMA in the schedule (with 2 to 5 the
// plain GEMM's epilogue spills two VGPRs around the loop).
template <>
struct Six<TgIQ4XS> : TgIQ4XS {
  static constexpr int kCT = 6, kAS = 3, kVPM = 6;
};

}  // namespace
}  // namespace q4k
