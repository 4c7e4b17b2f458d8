// GEMMs of the middle row counts for gfx950: prefill passes too small to fill
// the chip with 128 x 256 tiles.
//
//  mid_gemm_kernel    column tiles x K-slices over all CUs, activations and
//                     weights through LDS-DMA rings
//  mid_reduce_kernel  sums the K-slices and applies the epilogue
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include "q4k_mid.h"

namespace q4k {
namespace {

// ---- the kernel --------------------------------------------------------------
// y = post(x W^T) for row blocks of 16 RT rows.  Workgroup = 8 waves = 2
// K-groups x 4 column groups of CT column tiles; it takes one row block, one
// column block and one K-slice (blocks [kb0, kb0 + nbr)).  A step is half a
// block, u-steps 2h and 2h + 1, of which the waves of K-group kg take 2h + kg.  The activations of a
// step (RT x 4 KB) arrive by LDS-DMA in a ring of NS slots, NS - 1 steps
// ahead, the tile-blocks of a block in a ring of NB slots; each tile-block is
// dequantised once per K-group, into registers, and multiplied into all RT
// row tiles.
template <class P, int RT, int CT, int NS, int NB>
struct MidShape {
  static constexpr int kCG = 4, kTiles = kCG * CT, kASlot = RT * 4096, kBSlot = kTiles * P::kTB;
  static constexpr int kLds = NS * kASlot + NB * kBSlot, kHR = RT / 2;
  static_assert(kLds <= 160 * 1024, "LDS of one workgroup");
  static_assert(8 * (RT / 2) * CT * 1024 <= kLds, "K-group exchange");
};

// The steps of one wave of K-group KGI (compile-time, so that the u-steps and
// with them the dequantisation's shifts are).
template <class P, int RT, int CT, int NS, int NB, bool GATED, int KGI>
__device__ __forceinline__ void mid_steps(const MidArgs& a, uint8_t* lds, int by, int cb, int kb0, int nbr, int wave, int lane, f4_t (&acc)[RT][CT]) {
  using M = MidShape<P, RT, CT, NS, NB>;
  // With four row tiles a step's loads are issued after its first MFMAs, which
  // need nothing but what the previous step read (gate/up 4096 -> 12288 at 64
  // rows 34.6 -> 30.7 us, down 26.3 -> 24.6); with eight, where the MFMAs of a
  // step cover them, before (the late issue took 1 to 3 % more).
  constexpr bool kLate = RT == 4;
  constexpr int OT = GATED ? CT / 2 : CT, AD = NS - 1;
  // Tile-blocks this wave loads per block: its columns', shared out between
  // the two waves that use them (one column: by the first).
  constexpr int MB = CT % 2 == 0 ? CT / 2 : KGI == 0 ? CT : 0;
  constexpr int MB0 = CT % 2 == 0 ? KGI * (CT / 2) : 0;
  constexpr int LA = RT / 2, LB = MB * P::kNL;
  constexpr int W0 = mid_wait_count(0, 1, AD, NB, LA, LB), W1 = mid_wait_count(1, 1, AD, NB, LA, LB);
  const int cg = wave & 3, ntiles = a.n >> 4, steps = 2 * nbr;
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
  h8_t blo[CT], bhi[CT];
  {
    typename P::R r[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::raw(r[c], bl + c * P::kTB, lane);
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::consts(kk[c], r[c], lane);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      typename P::W w;
      P::words(w, bl + c * P::kTB, KGI, lane);
      P::dequant(kk[c], w, KGI, blo[c], bhi[c]);
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
      const uint32_t bsn = hh == 0 ? bs : bs + 1 == NB ? 0 : bs + 1;  // B slot of step t + 1
      const uint8_t* const al = lds + as * M::kASlot + KGI * 2 * RT * 1024 + 16 * lane;
      const uint32_t asn = as + 1 == NS ? 0 : as + 1;
      const uint8_t* const aln = lds + asn * M::kASlot + KGI * 2 * RT * 1024 + 16 * lane;
      const uint8_t* const bn = bl + bsn * M::kBSlot;
      typename P::R r[CT];
      typename P::W wv[CT];
      h8_t nlo[CT], nhi[CT];
      auto issue = [&] {
        if (t + AD < steps)
          issue_a(t + AD, an);
        if (hh == 1 && b + NB < nbr)
          issue_b(b + NB, bs);
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // The MFMAs on the low- or high-nibble fragments, under them the reads
        // of the next A fragments (the next step's first ones at the end) and
        // half of the next step's dequantisation.
        if (h == 0) {
          if (!kLate)
            issue();
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            if (hh == 1)
              P::raw(r[c], bn + c * P::kTB, lane);
            P::words(wv[c], bn + c * P::kTB, 2 * (1 - hh) + KGI, lane);
          }
        }
        const uint8_t* const src = h == 0 ? al + 1024 : aln;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          af[1 - h][rt] = *reinterpret_cast<const h8_t*>(src + 2 * rt * 1024);
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[h][rt], h ? bhi[c] : blo[c], acc[rt][c], 0, 0, 0);
#pragma unroll
        for (int c = h * CT / 2; c < (h + 1) * CT / 2; ++c) {
          if (hh == 1)
            P::consts(kk[c], r[c], lane);
          P::dequant(kk[c], wv[c], 2 * (1 - hh) + KGI, nlo[c], nhi[c]);
          asm volatile("" : "+v"(nlo[c]), "+v"(nhi[c]));  // formed in this step, under its MFMAs
        }
        if (h == 0) {
          if (hh == 1)
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * CT, 0);
          else
            __builtin_amdgcn_sched_group_barrier(0x100, CT, 0);
        }
#pragma unroll
        for (int k = 0; k < RT * CT; ++k) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (k < RT)
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          if (hh == 1)
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          else
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
        if (kLate)
          __builtin_amdgcn_sched_barrier(0);
        if (kLate && h == 0)
          issue();
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        blo[c] = nlo[c];
        bhi[c] = nhi[c];
      }
      as = asn;
      bs = bsn;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  mid_wait<0>();
}

template <class P, int RT, int CT, int NS, int NB, bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void mid_gemm_kernel(MidArgs a) {
  using M = MidShape<P, RT, CT, NS, NB>;
  constexpr int OT = GATED ? CT / 2 : CT;
  __shared__ __attribute__((aligned(16))) uint8_t lds[M::kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = wave & 3, kg = wave >> 2;
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
  if (kg == 0)
    mid_steps<P, RT, CT, NS, NB, GATED, 0>(a, lds, by, cb, kb0, nbr, wave, lane, acc);
  else
    mid_steps<P, RT, CT, NS, NB, GATED, 1>(a, lds, by, cb, kb0, nbr, wave, lane, acc);

  // K-groups: each wave of a pair keeps half of the row tiles and takes the
  // other wave's sums of them (in either order the same two terms).
  f4_t sum[M::kHR][CT];
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
  const int row_tile = by * RT + kg * H, live = (a.m + 15) >> 4;
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
        mid_epilogue_tile<GATED>(a, row_tile + h, ct0 + c, lane, sum[h][c], sum[h][GATED ? OT + c : c], mid_rowscale(a, row_tile + h, lane));
}

// Activations of few rows in the GEMM order: one row per workgroup of 512
// threads, so that a pass of 128 rows uses 128 CUs (8 rows per workgroup use
// 16).  Workgroup L runs on XCD L % 8: the 8 rows that share each 128-byte
// line of the staged operand go to one XCD, whose L2 puts the line together.
// CPT chunks of 8 elements per thread stay in registers between the row
// maximum (and, with NORM, the sum of squares) and the conversion; CPT == 0:
// x is read twice.
// SPLIT: a row is staged as two, hi = fp16(v) as staged row 32 (r / 16) +
// r % 16 and lo = fp16(v - hi) 16 rows on (about 22 significant bits), and xs
// receives each 32-element sub-block's sum / 32, hi/lo too, as the A operand
// of v_mfma_f32_16x16x16_f16 per (block, row tile): lane 16 G + r % 16 holds
// sub-blocks 4 (G & 1) .. + 3, the low parts for G >= 2.
template <typename InT, int CPT, bool NORM, bool SPLIT>
__global__ __launch_bounds__(512) void stage_row_kernel(const InT* __restrict__ x, _Float16* __restrict__ xo, float* __restrict__ rowscale, int m,
                                                        int k, const float* __restrict__ nw, float eps, _Float16* __restrict__ xs) {
  constexpr int T = 512, N = CPT > 0 ? CPT : 1;
  const int j8 = (int)blockIdx.x >> 3, row = ((j8 >> 3) * 8 + ((int)blockIdx.x & 7)) * 8 + (j8 & 7);
  if (row >= m)
    return;
  const int tid = threadIdx.x, chunks = k >> 3, nb = k >> 8;
  const InT* xr = x + (size_t)row * k;
  float v[N][8];
  float mx = 0.0f, ss = 0.0f;
  auto read = [&](int c, float (&o)[8]) {
    load8(xr + (size_t)c * 8, o);
    if (NORM) {
      float w8[8];
      load8(nw + (size_t)c * 8, w8);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        ss = fmaf(o[i], o[i], ss);
        o[i] *= w8[i];
      }
    }
  };
  if constexpr (CPT > 0) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = tid + T * j;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[j][i] = 0.0f;
      if (c < chunks)
        read(c, v[j]);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mx = fmaxf(mx, fabsf(v[j][i]));
    }
  } else {
    for (int c = tid; c < chunks; c += T) {
      read(c, v[0]);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mx = fmaxf(mx, fabsf(v[0][i]));
    }
  }
  __shared__ float red[2][8];
  mx = max64_lanes(mx);
  if (NORM) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      ss += __shfl_xor(ss, off);
  }
  if ((tid & 63) == 0) {
    red[0][tid >> 6] = mx;
    red[1][tid >> 6] = ss;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 8; ++w)
    mx = fmaxf(mx, red[0][w]);
  float r = 1.0f;
  if (NORM) {
    r = 1.0f / sqrtf(sum8_pairs(red[1]) / (float)k + eps);
    mx *= r;
  }
  float up, down;
  pow2_scale(mx, up, down);
  if (tid == 0)
    rowscale[row] = down;
  const float cs = NORM ? up * r : up;
  // Whole groups of 4 lanes (one sub-block) call it together.
  auto put = [&](int c, const float (&o)[8]) {
    h8_t h;
    if constexpr (SPLIT) {
      h8_t lo;
      float sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // One fp32 value for both parts: fused into the conversions, hi would
        // be rounded once where it is stored and its residual taken from
        // another rounding of the product (cs is no power of two with NORM).
        float t = o[i] * cs;
        asm("" : "+v"(t));
        h[i] = (_Float16)t;
        lo[i] = (_Float16)(t - (float)h[i]);
        sum += t;
      }
      const int vrow = 32 * (row >> 4) + (row & 15);
      *reinterpret_cast<h8_t*>(xo + gemm_frag_offset(vrow, c, nb)) = h;
      *reinterpret_cast<h8_t*>(xo + gemm_frag_offset(vrow + 16, c, nb)) = lo;
      sum += dpp_f<kDppQuadSwap1>(sum);
      sum += dpp_f<kDppQuadSwap2>(sum);
      if ((c & 3) == 0) {
        const float s32 = sum * 0.03125f;
        const _Float16 sh = (_Float16)s32;
        const int jb = (c >> 2) & 7;
        _Float16* p = xs + (((size_t)(c >> 5) * ((m + 15) >> 4) + (row >> 4)) * 64 + 16 * (jb >> 2) + (row & 15)) * 4 + (jb & 3);
        p[0] = sh;
        p[128] = (_Float16)(s32 - (float)sh);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        h[i] = (_Float16)(o[i] * cs);
      *reinterpret_cast<h8_t*>(xo + gemm_frag_offset(row, c, nb)) = h;
    }
  };
  if constexpr (CPT > 0) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = tid + T * j;
      if (c < chunks)
        put(c, v[j]);
    }
  } else {
    for (int c = tid; c < chunks; c += T) {
      read(c, v[0]);
      put(c, v[0]);
    }
  }
}

template <typename InT, bool NORM, bool SPLIT>
void stage_rows(hipStream_t s, const InT* x, _Float16* xo, float* rowscale, int m, int k, const float* nw, float eps, _Float16* xs) {
  const dim3 grid((unsigned)((m + 63) / 64 * 64)), block(512);
  if (k <= 4096)
    (void)dispatch(stage_row_kernel<InT, 1, NORM, SPLIT>, grid, block, s, x, xo, rowscale, m, k, nw, eps, xs);
  else if (k <= 12288)
    (void)dispatch(stage_row_kernel<InT, 3, NORM, SPLIT>, grid, block, s, x, xo, rowscale, m, k, nw, eps, xs);
  else
    (void)dispatch(stage_row_kernel<InT, 0, NORM, SPLIT>, grid, block, s, x, xo, rowscale, m, k, nw, eps, xs);
}

template <typename InT>
void stage_rows_any(hipStream_t s, const InT* x, _Float16* xo, float* rowscale, int m, int k, const float* nw, float eps, _Float16* xs) {
  if (xs)
    nw ? stage_rows<InT, true, true>(s, x, xo, rowscale, m, k, nw, eps, xs) : stage_rows<InT, false, true>(s, x, xo, rowscale, m, k, nw, eps, xs);
  else
    nw ? stage_rows<InT, true, false>(s, x, xo, rowscale, m, k, nw, eps, xs) : stage_rows<InT, false, false>(s, x, xo, rowscale, m, k, nw, eps, xs);
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
  mid_epilogue_tile<GATED>(a, rt, ct, lane, s, u, mid_rowscale(a, rt, lane));
}

template <class P, int RT, int CT, bool GATED>
hipError_t mid_launch(hipStream_t s, MidArgs a) {
  constexpr int kTiles = 4 * CT * P::kTB;
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
  (void)dispatch(mid_gemm_kernel<P, RT, CT, NS, NB, GATED>, dim3((unsigned)grid), dim3(512), s, a);
  if (a.slices > 1) {
    dispatch_events() = DispatchEvents{nullptr, ev.stop};
    (void)launch_mid_reduce(s, a, GATED);
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

hipError_t launch_stage_rows(hipStream_t s, const void* x, int dtype, _Float16* xo, float* rowscale, int m, int k, const float* norm_w, float eps,
                             _Float16* xs) {
  if (dtype == kF32)
    stage_rows_any(s, static_cast<const float*>(x), xo, rowscale, m, k, norm_w, eps, xs);
  else
    stage_rows_any(s, static_cast<const _Float16*>(x), xo, rowscale, m, k, norm_w, eps, xs);
  return hipGetLastError();
}

hipError_t launch_mid_reduce(hipStream_t s, const MidArgs& a, bool gated) {
  const int items = (a.m + 15) / 16 * (a.n / 16);
  if (gated)
    (void)dispatch(mid_reduce_kernel<true>, dim3((unsigned)((items + 3) / 4)), dim3(256), s, a);
  else
    (void)dispatch(mid_reduce_kernel<false>, dim3((unsigned)((items + 3) / 4)), dim3(256), s, a);
  return hipGetLastError();
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
