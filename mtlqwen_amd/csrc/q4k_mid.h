// Device code shared by the GEMMs of the middle row counts (q4k_mid.hip,
// q4k_rows.hip): the accounting of their LDS-DMA loads and their epilogue.
#pragma once
#include "q4k_formats.h"

namespace q4k {
namespace {

// Load accounting.  A wave issues A(t + AD) (LA loads) at step t, then, at
// odd steps t = 2 b + 1, its share of B(b + NB) (LB loads); the prologue
// issues B(0), A(0 .. AD - 1), B(1 .. NB - 1).  At the top of step t A(t + lead)
// must have landed and, at odd steps, B((t + 1) / 2) (read from there on).  vmcnt
// counts in issue order, so the wait is the number of loads issued after the
// later of the two: the smallest over the steps of one parity, the first ones
// (whose loads come from the prologue) included.
constexpr int mid_loads_after(int t, int lead, int ad, int nb, int la, int lb) {
  // Position of the last required load, and of the end, counted in loads.
  int pos = lb, need = 0;  // after B(0)
  for (int i = 0; i < ad; ++i) {
    pos += la;
    if (i == t + lead)
      need = pos;
  }
  for (int b = 1; b < nb; ++b) {
    pos += lb;
    if ((t & 1) && b == (t + 1) / 2)
      need = pos > need ? pos : need;
  }
  for (int s = 0; s < t; ++s) {
    pos += la;
    if (s + ad == t + lead)
      need = pos > need ? pos : need;
    if (s & 1) {
      pos += lb;
      if ((t & 1) && (s - 1) / 2 + nb == (t + 1) / 2)
        need = pos > need ? pos : need;
    }
  }
  return pos - need;
}
constexpr int mid_wait_count(int parity, int lead, int ad, int nb, int la, int lb) {
  int n = 63;
  for (int t = parity; t < 32; t += 2) {
    const int v = mid_loads_after(t, lead, ad, nb, la, lb);
    n = v < n ? v : n;
  }
  return n;
}

template <int N>
__device__ __forceinline__ void mid_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ f4_t mid_rowscale(const MidArgs& a, int rt0, int lane) {
  return *reinterpret_cast<const f4_t*>(a.rowscale + 16 * rt0 + 4 * (lane >> 4));
}

template <typename OutT>
__device__ __forceinline__ void mid_store(const MidArgs& a, int row, size_t col, float v, float rs) {
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const size_t off = (size_t)row * a.n + col;
  float acc_v = v * rs;
  if (sizeof(OutT) == 2)
    acc_v = round_half(acc_v);
  float out = acc_v;
  if (a.post == 1)
    out = acc_v + load_elem(reinterpret_cast<const OutT*>(a.aux), off);
  else if (a.post == 2)
    out = silu(load_elem(reinterpret_cast<const OutT*>(a.aux), off)) * acc_v;
  asm("" : "+v"(out));  // the fp32 value first: fused into the conversion the product would round once instead of twice
  store_elem(y, off, out);
}

template <typename OutT>
__device__ __forceinline__ void mid_store_gated(const MidArgs& a, int row, size_t col, float gv, float uv, float rs) {
  OutT* y = reinterpret_cast<OutT*>(a.y);
  gv *= rs;
  uv *= rs;
  if (sizeof(OutT) == 2) {
    gv = round_half(gv);
    uv = round_half(uv);
  }
  float out = silu(gv) * uv;
  asm("" : "+v"(out));
  store_elem(y, (size_t)row * a.n + col, out);
}

// Epilogue of the rows of one 16 x 16 accumulator tile (row tile rt0, output
// column tile ct): lane 16g + i holds rows 4g .. 4g + 3 of column i, whose
// unscale factors are rs.
template <bool GATED>
__device__ __forceinline__ void mid_epilogue_tile(const MidArgs& a, int rt0, int ct, int lane, const f4_t& v, const f4_t& up, const f4_t& rs) {
  const int row0 = 16 * rt0 + 4 * (lane >> 4);
  const size_t col = (size_t)ct * 16 + (lane & 15);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = row0 + e;
    if (row >= a.m)
      continue;
    if constexpr (GATED) {
      if (a.dtype == kF32)
        mid_store_gated<float>(a, row, col, v[e], up[e], rs[e]);
      else
        mid_store_gated<_Float16>(a, row, col, v[e], up[e], rs[e]);
    } else {
      if (a.dtype == kF32)
        mid_store<float>(a, row, col, v[e], rs[e]);
      else
        mid_store<_Float16>(a, row, col, v[e], rs[e]);
    }
  }
}

}  // namespace
}  // namespace q4k
