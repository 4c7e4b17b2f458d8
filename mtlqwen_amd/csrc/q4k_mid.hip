// GEMMs of the middle row counts for gfx950: prefill passes too small to fill
// the chip with 128 x 256 tiles.
//
//  mid_gemm_kernel    column tiles x K-slices over all CUs, weights from
//                     global memory straight into registers
//  mid_reduce_kernel  sums the K-slices and applies the epilogue
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include <type_traits>

#include "q4k_formats.h"

namespace q4k {
namespace {


// ---- the kernel --------------------------------------------------------------
// y = post(x W^T) for row blocks of 16 RT rows.  Workgroup = 8 waves = KG
// K-groups x 8 / KG column groups of CT column tiles; it takes one row block,
// one column block and one K-slice (blocks [kb0, kb0 + nbr)).  A step is half
// a block, u-steps 2h and 2h + 1: with KG = 2 the waves of K-group kg take
// u-step 2h + kg, with KG = 1 every wave takes both.  The activations of a
// step (RT x 4 KB) arrive by LDS-DMA in a ring of NS slots, NS - 1 steps
// ahead, the tile-blocks of a block in a ring of NB slots; each tile-block is
// dequantised once per K-group, into registers, and multiplied into all RT
// row tiles.
template <class P, int RT, int CT, int KG, int NS, int NB>
struct MidShape {
  static constexpr int kCG = 8 / KG, kTiles = kCG * CT, kASlot = RT * 4096, kBSlot = kTiles * P::kTB;
  static constexpr int kLds = NS * kASlot + NB * kBSlot, kHR = KG == 2 ? RT / 2 : RT;
  static_assert(kLds <= 160 * 1024, "LDS of one workgroup");
  static_assert(KG == 1 || 8 * (RT / 2) * CT * 1024 <= kLds, "K-group exchange");
};

// Load accounting.  A wave issues A(t + AD) (LA loads) at step t, then, at
// odd steps t = 2 b + 1, its share of B(b + NB) (LB loads); the prologue
// issues B(0), A(0 .. AD - 1), B(1 .. NB - 1).  At the top of step t A(t) must
// have landed and, at odd steps, B((t + 1) / 2) (read from there on).  vmcnt
// counts in issue order, so the wait is the number of loads issued after the
// later of the two: the smallest over the steps of one parity, the first ones
// (whose loads come from the prologue) included.
constexpr int mid_loads_after(int t, int ad, int nb, int la, int lb) {
  // Position of the last required load, and of the end, counted in loads.
  int pos = lb, need = 0;  // after B(0)
  for (int i = 0; i < ad; ++i) {
    pos += la;
    if (i == t + 1)
      need = pos;
  }
  for (int b = 1; b < nb; ++b) {
    pos += lb;
    if ((t & 1) && b == (t + 1) / 2)
      need = pos > need ? pos : need;
  }
  for (int s = 0; s < t; ++s) {
    pos += la;
    if (s + ad == t + 1)
      need = pos > need ? pos : need;
    if (s & 1) {
      pos += lb;
      if ((t & 1) && (s - 1) / 2 + nb == (t + 1) / 2)
        need = pos > need ? pos : need;
    }
  }
  return pos - need;
}
constexpr int mid_wait_count(int parity, int ad, int nb, int la, int lb) {
  int n = 63;
  for (int t = parity; t < 32; t += 2) {
    const int v = mid_loads_after(t, ad, nb, la, lb);
    n = v < n ? v : n;
  }
  return n;
}

template <int N>
__device__ __forceinline__ void mid_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
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
// column tile ct): lane 16g + i holds rows 4g .. 4g + 3 of column i.
template <bool GATED>
__device__ __forceinline__ void mid_epilogue_tile(const MidArgs& a, int rt0, int ct, int lane, const f4_t& v, const f4_t& up) {
  const int row0 = 16 * rt0 + 4 * (lane >> 4);
  const size_t col = (size_t)ct * 16 + (lane & 15);
  const f4_t rs = *reinterpret_cast<const f4_t*>(a.rowscale + row0);
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

// The steps of one wave of K-group KGI (compile-time, so that the u-steps and
// with them the dequantisation's shifts are).
template <class P, int RT, int CT, int KG, int NS, int NB, bool GATED, int KGI>
__device__ __forceinline__ void mid_steps(const MidArgs& a, uint8_t* lds, int by, int cb, int kb0, int nbr, int wave, int lane, f4_t (&acc)[RT][CT]) {
  using M = MidShape<P, RT, CT, KG, NS, NB>;
  constexpr int OT = GATED ? CT / 2 : CT, AD = NS - 1, NU = 2 / KG;
  // Tile-blocks this wave loads per block: its columns', shared out between
  // the two waves that use them (KG = 2; one column: by the first).
  constexpr int MB = KG == 1 ? CT : CT % 2 == 0 ? CT / 2 : KGI == 0 ? CT : 0;
  constexpr int MB0 = KG == 2 && CT % 2 == 0 ? KGI * (CT / 2) : 0;
  constexpr int LA = RT / 2, LB = MB * P::kNL;
  constexpr int W0 = mid_wait_count(0, AD, NB, LA, LB), W1 = mid_wait_count(1, AD, NB, LA, LB);
  const int cg = KG == 1 ? wave : wave & 3, ntiles = a.n >> 4, steps = 2 * nbr;
  const int ct0 = (cb * M::kCG + cg) * OT;
  const uint8_t* wcol[MB > 0 ? MB : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int c = MB0 + i, oc = ct0 + (GATED ? c % OT : c);
    wcol[i] = uniform_ptr((GATED && c >= OT ? a.wu : a.w) + ((size_t)(oc < ntiles ? oc : ntiles - 1) * a.nb + kb0) * P::kTB);
  }
  constexpr int RB8 = 8 / RT;  // row blocks per 128 staged rows
  // This wave's RT / 2 fragments of a step: u-step wave / 4 of the two, of
  // whose 2 RT fragments (of this row block) the wave % 4-th quarter.
  const uint8_t* const xa = uniform_ptr(reinterpret_cast<const uint8_t*>(a.xh) + ((size_t)(by / RB8) * a.nb + kb0) * 65536 +
                                        (size_t)((wave >> 2) * 16 + (by % RB8) * 2 * RT + (wave & 3) * (RT / 2)) * 1024);
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds)), voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;
  const uint32_t a0w = lds0 + (uint32_t)wave * (RT / 2 * 1024), b0 = lds0 + NS * M::kASlot;
  auto issue_a = [&](int t, uint32_t slot) {
    const uint8_t* src = xa + (size_t)t * 32768;
    const uint32_t l = a0w + slot * M::kASlot;
    lds_dma16<0>(src, voff16, l);
    lds_dma16<1024>(src, voff16, l);
    if constexpr (RT == 8) {
      lds_dma16<2048>(src, voff16, l);
      lds_dma16<3072>(src, voff16, l);
    }
  };
  auto issue_b = [&](int b, uint32_t slot) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
      P::issue(wcol[i] + (size_t)b * P::kTB, voff16, voff4, __builtin_amdgcn_readfirstlane(b0 + slot * M::kBSlot + (uint32_t)(cg * CT + MB0 + i) * P::kTB),
               lane);
  };
  const uint8_t* const bl = lds + NS * M::kASlot + cg * CT * P::kTB;  // this column group's tile-blocks in a B slot

  issue_b(0, 0);
#pragma unroll
  for (int t = 0; t < AD; ++t)
    issue_a(t < steps ? t : steps - 1, t);
#pragma unroll
  for (int b = 1; b < NB; ++b)
    issue_b(b < nbr ? b : nbr - 1, b);
  mid_wait<AD * LA + (NB - 1) * LB>();
  __syncthreads();
  typename P::K kk[CT];
  h8_t blo[NU][CT], bhi[NU][CT];
  {
    typename P::R r[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::raw(r[c], bl + c * P::kTB, lane);
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::consts(kk[c], r[c], lane);
#pragma unroll
    for (int ui = 0; ui < NU; ++ui)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        typename P::W w;
        P::words(w, bl + c * P::kTB, ui + KGI, lane);
        P::dequant(kk[c], w, ui + KGI, blo[ui][c], bhi[ui][c]);
      }
  }
  uint32_t as = 0, bs = 0;  // ring slots of step t and of its block
  h8_t af[2][RT];
  mid_wait<(AD - 1) * LA + (NB - 1) * LB>();  // A(0) of this wave
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
    af[0][rt] = *reinterpret_cast<const h8_t*>(lds + KGI * 2 * RT * 1024 + 16 * lane + 2 * rt * 1024);
  for (int b = 0; b < nbr; ++b) {
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      const int t = 2 * b + hh;
      // Near the end fewer loads follow the ones waited for.
      const int rest = steps - t;  // steps from t on
      if (rest > (AD > 2 * NB - 2 ? AD : 2 * NB - 2)) {
        if (hh == 0)
          mid_wait<W0>();
        else
          mid_wait<W1>();
      } else {
        mid_wait<0>();
      }
      __syncthreads();  // step t's operands of every wave landed; step t - 1 fully read
      __builtin_amdgcn_sched_barrier(0);
      const uint32_t an = as == 0 ? NS - 1 : as - 1;  // slot of step t - 1
      if (t + AD < steps)
        issue_a(t + AD, an);
      if (hh == 1 && b + NB < nbr)
        issue_b(b + NB, bs);
      const uint32_t bsn = hh == 0 ? bs : bs + 1 == NB ? 0 : bs + 1;  // B slot of step t + 1
      const uint8_t* const al = lds + as * M::kASlot + KGI * 2 * RT * 1024 + 16 * lane;
      const uint32_t asn = as + 1 == NS ? 0 : as + 1;
      const uint8_t* const aln = lds + asn * M::kASlot + KGI * 2 * RT * 1024 + 16 * lane;
      const uint8_t* const bn = bl + bsn * M::kBSlot;
      __builtin_amdgcn_sched_barrier(0);
      typename P::R r[CT];
      if (hh == 1) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          P::raw(r[c], bn + c * P::kTB, lane);
      }
      typename P::W wv[NU][CT];
#pragma unroll
      for (int ui = 0; ui < NU; ++ui)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          P::words(wv[ui][c], bn + c * P::kTB, 2 * (1 - hh) + ui + KGI, lane);
      h8_t nlo[NU][CT], nhi[NU][CT];
#pragma unroll
      for (int ui = 0; ui < NU; ++ui) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          // The A fragments of the next group of MFMAs, the next step's
          // first at the end.
          const int i = 2 * ui + h, j = i + 1;
          const uint8_t* const src = j < 2 * NU ? al + (j / 2 * 2 * RT + (j & 1)) * 1024 : aln;
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            af[j & 1][rt] = *reinterpret_cast<const h8_t*>(src + 2 * rt * 1024);
#pragma unroll
          for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
              acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i & 1][rt], h ? bhi[ui][c] : blo[ui][c], acc[rt][c], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          if (hh == 1 && ui == 0)
            P::consts(kk[c], r[c], lane);
          P::dequant(kk[c], wv[ui][c], 2 * (1 - hh) + ui + KGI, nlo[ui][c], nhi[ui][c]);
        }
      }
#pragma unroll
      for (int ui = 0; ui < NU; ++ui)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          blo[ui][c] = nlo[ui][c];
          bhi[ui][c] = nhi[ui][c];
          asm volatile("" : "+v"(blo[ui][c]), "+v"(bhi[ui][c]));  // formed in this step, under its MFMAs
        }
      as = asn;
      bs = bsn;
      // The raw words first, then each MFMA followed by an LDS read (the
      // next group's fragments) and vector work.
      if (hh == 1)
        __builtin_amdgcn_sched_group_barrier(0x100, CT + CT * NU, 0);
      else
        __builtin_amdgcn_sched_group_barrier(0x100, CT * NU, 0);
#pragma unroll
      for (int i = 0; i < 2 * NU * RT * CT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i % (RT * CT) < RT)
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (hh == 1)
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        else
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  mid_wait<0>();
}

template <class P, int RT, int CT, int KG, int NS, int NB, bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mid_gemm_kernel(MidArgs a) {
  using M = MidShape<P, RT, CT, KG, NS, NB>;
  constexpr int OT = GATED ? CT / 2 : CT;
  __shared__ __attribute__((aligned(16))) uint8_t lds[M::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = KG == 1 ? wave : wave & 3, kg = KG == 1 ? 0 : wave >> 2;
  // Workgroup -> (row block, column block, K-slice).  Workgroup L runs on XCD
  // L % 8: the row blocks of one (column block, slice) share an XCD (its
  // weights), and slices are dealt so that an XCD reads few slices of x.
  const int xcd = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
  const int by = j % a.rblocks, p = (j / a.rblocks) * 8 + xcd;
  if (p >= a.cblocks * a.slices)
    return;
  const int slice = p % a.slices, cb = p / a.slices;
  const int kb0 = slice * a.nb / a.slices, nbr = (slice + 1) * a.nb / a.slices - kb0;
  const int ntiles = a.n >> 4;
  const int ct0 = (cb * M::kCG + cg) * OT;
  f4_t acc[RT][CT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int c = 0; c < CT; ++c)
      acc[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  if (KG == 1 || kg == 0)
    mid_steps<P, RT, CT, KG, NS, NB, GATED, 0>(a, lds, by, cb, kb0, nbr, wave, lane, acc);
  else
    mid_steps<P, RT, CT, KG, NS, NB, GATED, KG - 1>(a, lds, by, cb, kb0, nbr, wave, lane, acc);

  // K-groups: each wave of a pair keeps half of the row tiles and takes the
  // other wave's sums of them (in either order the same two terms).
  f4_t sum[M::kHR][CT];
  int rt_first = 0;
  if constexpr (KG == 2) {
    constexpr int H = RT / 2;
    __syncthreads();  // every wave has read its last operands, and no load is in flight
    f4_t* mine = reinterpret_cast<f4_t*>(lds) + wave * (H * CT * 64) + lane;
    const f4_t* other = reinterpret_cast<const f4_t*>(lds) + (wave ^ 4) * (H * CT * 64) + lane;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        mine[(h * CT + c) * 64] = kg ? acc[h][c] : acc[H + h][c];
        sum[h][c] = kg ? acc[H + h][c] : acc[h][c];
      }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        sum[h][c] += other[(h * CT + c) * 64];
    rt_first = kg * H;
  } else {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int c = 0; c < CT; ++c)
        sum[rt][c] = acc[rt][c];
  }
  const int row_tile = by * RT + rt_first, live = (a.m + 15) >> 4;
  if (a.slices > 1) {
    // Slice sums in accumulator order: [slice][row tile][column tile][lane].
    const int wide = GATED ? 2 * ntiles : ntiles;
    f4_t* part = reinterpret_cast<f4_t*>(a.part) + (size_t)slice * live * wide * 64 + lane;
#pragma unroll
    for (int h = 0; h < M::kHR; ++h)
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int oc = ct0 + (GATED ? c % OT : c);
        if (row_tile + h < live && oc < ntiles)
          part[((size_t)(row_tile + h) * wide + oc + (GATED && c >= OT ? ntiles : 0)) * 64] = sum[h][c];
      }
    return;
  }
#pragma unroll
  for (int h = 0; h < M::kHR; ++h)
#pragma unroll
    for (int c = 0; c < OT; ++c)
      if (row_tile + h < live && ct0 + c < ntiles)
        mid_epilogue_tile<GATED>(a, row_tile + h, ct0 + c, lane, sum[h][c], sum[h][GATED ? OT + c : c]);
}

// One wave per 16 x 16 output tile: the slices' sums in slice order, then the
// epilogue.
template <bool GATED>
__global__ __launch_bounds__(256) void mid_reduce_kernel(MidArgs a) {
  const int lane = threadIdx.x & 63, ntiles = a.n >> 4, live = (a.m + 15) >> 4;
  const int item = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (item >= live * ntiles)
    return;
  const int rt = item / ntiles, ct = item % ntiles, wide = GATED ? 2 * ntiles : ntiles;
  const f4_t* part = reinterpret_cast<const f4_t*>(a.part) + ((size_t)rt * wide + ct) * 64 + lane;
  const size_t stride = (size_t)live * wide * 64;
  f4_t s = part[0], u = GATED ? part[(size_t)ntiles * 64] : f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
  for (int i = 1; i < a.slices; ++i) {
    s += part[i * stride];
    if (GATED)
      u += part[i * stride + (size_t)ntiles * 64];
  }
  mid_epilogue_tile<GATED>(a, rt, ct, lane, s, u);
}

template <class P, int RT, int CT, bool GATED>
hipError_t mid_launch(hipStream_t s, MidArgs a) {
  constexpr int KG = 2, kTiles = 4 * CT * P::kTB;
  // Ring depths that fit 160 KB: activations first (three slots of 32 KB, or
  // four of 16), then up to four blocks of weights.
  constexpr int NS = RT == 8 ? 3 : 4, kLeft = 160 * 1024 - NS * RT * 4096, NB = kLeft / kTiles < 4 ? kLeft / kTiles : 4;
  static_assert(NB >= 2, "two blocks of weights");
  constexpr int OT = GATED ? CT / 2 : CT;
  const int ntiles = a.n / 16;
  a.cblocks = (ntiles + 4 * OT - 1) / (4 * OT);
  a.rblocks = (a.m + 16 * RT - 1) / (16 * RT);
  const int grid = (a.cblocks * a.slices + 7) / 8 * 8 * a.rblocks;
  // Two launches when K is sliced: the dispatch events (launch timing) span both.
  const DispatchEvents ev = dispatch_events();
  if (a.slices > 1)
    dispatch_events() = DispatchEvents{ev.start, nullptr};
  (void)dispatch(mid_gemm_kernel<P, RT, CT, KG, NS, NB, GATED>, dim3((unsigned)grid), dim3(512), s, a);
  if (a.slices > 1) {
    dispatch_events() = DispatchEvents{nullptr, ev.stop};
    const int items = (a.m + 15) / 16 * ntiles;
    (void)dispatch(mid_reduce_kernel<GATED>, dim3((unsigned)((items + 3) / 4)), dim3(256), s, a);
    dispatch_events() = ev;
  }
  return hipGetLastError();
}

template <class P, int CT, bool GATED>
hipError_t mid_launch_rt(hipStream_t s, const MidArgs& a, int rt) {
  return rt == 4 ? mid_launch<P, 4, CT, GATED>(s, a) : mid_launch<P, 8, CT, GATED>(s, a);
}

}  // namespace

// Row counts whose 128 x 64 tiles fit the CUs in one round.  There the
// 128 x 256 and 128 x 128 tilings of the pipelined GEMMs leave most CUs idle
// (32 of 256 at N = 4096, M <= 128) and K is walked by one workgroup alone:
// measured with the staging, fp16, this form against those,
//   N = 4096, K = 4096:   M = 64 20.3 / 46.5 us, 128 24.3 / 48.4, 512 40.0 / 52.3
//   N = 4096, K = 12288:  M = 64 38.4 / 107.8, 128 45.1 / 111.8, 512 94.0 / 113.9
//   gate/up N = 12288:    M = 64 40.7 / 70.5, 128 48.2 / 73.3
//   N = 8192, K = 4096:   M = 128 31.6 / 49.9, 256 39.4 / 52.2
//   N = 1024, K = 4096:   M = 64 16.3 / 46.4, 1024 33.2 / 54.6
// and past the round: N = 4096, M = 640 65.0 / 54.0, gate/up M = 160
// 85.9 / 74.0, N = 8192 M = 320 63.5 / 53.0.  The rule depends on the shape
// of one projection only, so a gate/up pair takes the same form, the same
// K-slices and the same order of sums in one launch as in two.
// The K-slices fill the CUs that the tiles leave idle, each at least two
// blocks long.  The row tiles per workgroup (64 or 128 rows) are those whose
// rounds take less time; a block of a workgroup took 0.85 us plus 0.155 us
// per row tile.
MidPlan mid_plan(int m, int n, int nb, int cus) {
  MidPlan p;
  // The tiling switches of the pipelined GEMMs name forms of theirs.
  static const bool forced = [] {
    for (const char* name : {"Q4K_GEMM_NARROW", "Q4K_GEMM2_SPLIT", "Q4K_GEMM2_SPLIT_B", "Q4K_GEMM2_PERSIST", "Q4K_GEMM_XCD_ROWS", "Q4K_GEMM_MID",
                             "Q4K_TYPED_MID", "Q4K_TYPED_Q8W", "Q4K_GEMM_GATED_SIX", "Q4K_GEMM_SIX"})
      if (const char* v = getenv(name))
        if (*v)
          return true;
    return false;
  }();
  const int cb = (n / 16 + 3) / 4;  // 64-column blocks
  if (forced || m < 1 || n < 64 || (long long)cb * ((m + 127) / 128) > cus)
    return p;
  const size_t row_floats = (size_t)((m + 15) / 16 * 16) * n * 2;  // one slice's sums of a gate/up pair
  int best = 0;
  for (int rt : {8, 4}) {
    const int tiles = cb * ((m + 16 * rt - 1) / (16 * rt));
    int s = cus / tiles < nb / 2 ? cus / tiles : nb / 2;
    if (s > kMidMaxSlices)
      s = kMidMaxSlices;
    while (s > 1 && s * row_floats > kMidPartFloats)
      --s;
    if (s < 1)
      s = 1;
    const int time = (tiles * s + cus - 1) / cus * ((nb + s - 1) / s) * (85 * 2 + 31 * rt);
    if (!p.rt || time < best) {
      best = time;
      p.rt = rt;
      p.slices = s;
    }
  }
  p.part_floats = p.slices > 1 ? p.slices * row_floats : 0;
  return p;
}

hipError_t launch_mid(hipStream_t s, MidArgs a, uint32_t type, const MidPlan& plan, bool gated) {
  if ((plan.rt != 4 && plan.rt != 8) || a.m < 1 || a.n % 16 != 0 || plan.slices < 1 || plan.slices > a.nb || (plan.slices > 1 && !a.part) || (gated && !a.wu))
    return hipErrorInvalidValue;
  a.slices = plan.slices;
  switch (type) {
    case kTypeQ4_K:
      return gated ? mid_launch_rt<TgQ4K, 2, true>(s, a, plan.rt) : mid_launch_rt<TgQ4K, 1, false>(s, a, plan.rt);
    case kTypeQ5_K:
      return mid_launch_rt<TgQ5K, 1, false>(s, a, plan.rt);
    case kTypeQ6_K:
      return mid_launch_rt<TgQ6K, 1, false>(s, a, plan.rt);
    case kTypeQ8_0:
      return mid_launch_rt<TgQ8_0, 1, false>(s, a, plan.rt);
    case kTypeIQ4_XS:
      return mid_launch_rt<TgIQ4XS, 1, false>(s, a, plan.rt);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace q4k
