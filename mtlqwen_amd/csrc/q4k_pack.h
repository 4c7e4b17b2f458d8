// The in-register pack of up to 8 rows of x into MFMA operands, shared by the
// decode GEMVs that take x as the caller stores it (no staging launch).
#pragma once
#include "q4k_formats.h"

namespace q4k {
namespace {

// ----------------------------------------------------------------------------
// In-register activation packing (m <= 8 rows, K = 4096).  A wave owns BPW
// consecutive K-blocks (rotated by workgroup, so that the workgroups of one L2
// read different parts of x first), loads them from x (one coalesced 1 KB load
// per (block, row)) and, under its first weight loads, turns them into the MFMA
// operands in the layout of the decode pack (pack_block_row):
//  - x passes through LDS so that lane 16g + i holds elements
//    64g + 32 (i / 8) + [0, 32) of row i % 8 (rows >= m read as zero);
//  - each (row, block) is scaled by a power of two that puts its largest
//    magnitude in [2^14, 2^15) and split into hi = h(t), lo = h(t - hi);
//  - lanes i and i ^ 8 (one DPP row rotation) trade halves so that lanes
//    i < 8 hold the high parts of elements 64g + [0, 64) of row i and lanes
//    i >= 8 the low parts: the A fragments of v_mfma_f32_16x16x32_f16, rows
//    8..15 carrying the low parts;
//  - each lane's 32 elements are one sub-block; their sums / 32 (hi / lo)
//    are gathered into the min-term operand of v_mfma_f32_16x16x16_f16.
// About 500 vector instructions per block, 2 us in all.
// ----------------------------------------------------------------------------
constexpr int kDppRowRor8 = 0x128;  // lane i <- lane (i + 8) % 16 within 16 lanes

template <int BANKS>
__device__ __forceinline__ uint32_t ror8_into(uint32_t old, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, kDppRowRor8, 0xF, BANKS, false);
}

// Registers of one packed x block: A fragments, min-term operand and the
// unscale factors of this lane's C rows (4g + v) & 7.
struct XBlock {
  h8_t frag[8];
  h4_t xs;
  float dv[4];
};

// Converts the 32 values t0 (elements 64g + 32 (i / 8) + [0, 32) of row i % 8,
// lane 16g + i) of one block into the block's operands.
__device__ __forceinline__ void pack_x_regs(const float (&xv)[32], int lane, XBlock& xb) {
  const int g = lane >> 4, i = lane & 15, half = i >> 3;
  // Largest magnitude of the (row, block): own 32, the partner half, the four
  // lane groups.
  float mx = 0.0f;
#pragma unroll
  for (int e = 0; e < 32; ++e)
    mx = fmaxf(mx, fabsf(xv[e]));
  mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, mx), kDppRowRor8, 0xF, 0xF, false)));
  mx = fmaxf(mx, __shfl_xor(mx, 16));
  mx = fmaxf(mx, __shfl_xor(mx, 32));
  float up = 1.0f, down = 1.0f;
  if (mx > 0.0f && mx <= FLT_MAX) {
    int ex;
    frexpf(mx, &ex);
    ex = ex < -80 ? -80 : ex;
    up = ldexpf(1.0f, 15 - ex);
    down = ldexpf(1.0f, ex - 15);
  }
  uint32_t hw[16], lw[16];
  float sum = 0.0f;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const float t0 = xv[2 * v] * up, t1 = xv[2 * v + 1] * up;
    sum += t0 + t1;
    // Both parts rounded to nearest, as the staging kernels round them: hi + lo
    // then holds 23 significant bits of the larger elements, where a truncated
    // hi leaves a residual of up to a whole ulp and lo drops one bit more (rows
    // 4096 -> 1024, m = 8, against 64 bits: 1.69e-7, truncated 1.91e-7).  The
    // opaque values keep hi at one v_cvt_pk_f16_f32, not converted again element
    // by element for its residual, and the residuals in fp32 until theirs
    // (4096 -> 1024, m = 8, Q6_K 5.97 us; truncated 6.13).
    uint32_t hp = __builtin_bit_cast(uint32_t, h2_t{(_Float16)t0, (_Float16)t1});
    asm("" : "+v"(hp));
    const h2_t h = __builtin_bit_cast(h2_t, hp);
    float l0 = t0 - (float)h[0], l1 = t1 - (float)h[1];
    asm("" : "+v"(l0), "+v"(l1));
    const h2_t l = h2_t{(_Float16)l0, (_Float16)l1};
    hw[v] = __builtin_bit_cast(uint32_t, h);
    lw[v] = __builtin_bit_cast(uint32_t, l);
  }
  // Fragments 0..3 (elements 64g + [0, 32)): own high parts in lanes i < 8,
  // the partner's low parts in lanes i >= 8 (banks 2, 3 take the rotation).
  // Fragments 4..7 (64g + [32, 64)): the partner's high parts in lanes i < 8,
  // own low parts in lanes i >= 8.
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    u4_t f0, f1;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      f0[v] = ror8_into<0xC>(hw[4 * s + v], lw[4 * s + v]);
      f1[v] = ror8_into<0x3>(lw[4 * s + v], hw[4 * s + v]);
    }
    xb.frag[s] = __builtin_bit_cast(h8_t, f0);
    xb.frag[4 + s] = __builtin_bit_cast(h8_t, f1);
  }
  // Sub-block sums / 32 as (hi, lo) halves; lane 16G + r (G < 2) gathers
  // sub-blocks 4G + c (c = 0..3) of row r % 8 from lanes 16 (2G + c / 2) +
  // r % 8 + 8 (c % 2), taking the high halves for r < 8 and the low for r >= 8.
  const float s32 = sum * 0.03125f;
  const _Float16 sh = (_Float16)s32;
  const _Float16 sl = (_Float16)(s32 - (float)sh);
  const uint32_t shl = (uint32_t)__builtin_bit_cast(uint16_t, sh) | ((uint32_t)__builtin_bit_cast(uint16_t, sl) << 16);
  const int G = g & 1, r8 = i & 7;
  uint32_t got[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    got[c] = (uint32_t)__shfl((int)shl, 16 * (2 * G + (c >> 1)) + r8 + 8 * (c & 1));
  const uint32_t sel = half ? 0x07060302u : 0x05040100u;  // low or high halves of a pair of dwords
  const uint32_t x01 = __builtin_amdgcn_perm(got[1], got[0], sel), x23 = __builtin_amdgcn_perm(got[3], got[2], sel);
  xb.xs = g < 2 ? __builtin_bit_cast(h4_t, uint2{x01, x23}) : h4_t{(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
  // Unscale factors of C rows 4 (g & 1) + v (the same in every lane of a row).
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float d0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, down), v));
    const float d1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, down), 4 + v));
    xb.dv[v] = (g & 1) ? d1 : d0;
  }
}

// x of wave w, re-ordered for the register pack: [block][lane][32 + 4]
// floats (the 4-float pad makes the 16-byte reads of 16 lanes hit 64
// distinct banks), BPW blocks per wave.  The partial sums reuse the wave's
// own region at the end.
constexpr int kGuXRow = 36;
template <int BPW>
constexpr int gu_wave_floats() {
  return BPW * 64 * kGuXRow;
}

// The x of one workgroup, packed: its wave loads K-blocks bw .. bw + BPW - 1
// of all 8 rows (one coalesced load per (block, row), lane l
// holding elements 4l..4l+3; rows >= m read row 0 and are zeroed), calls
// issue_first() once its x has landed, and turns its blocks into MFMA
// operands in registers (through its LDS region; W = 8 or 16).  NORM: x
// is RMS-normalised on the way in (native_ops.metal:6-40, the norm
// forward.cpp:114 applies before the MLP): the W waves hold all of x between
// them, so each row's sum of squares is their partial sums (ssq [wave][row])
// added after one barrier, and every element becomes
// (x * rsqrt(sum / k + eps)) * w before the pack.
template <typename OutT, bool NORM, int W, int BPW, typename Issue>
__device__ __forceinline__ void gate_up_pack_x(const GemvArgs& a, float* xl, float (*ssq)[8], int bw, XBlock (&xb)[BPW],
                                               Issue&& issue_first) {
  constexpr int kXRow = kGuXRow;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float xv[BPW][8][4];
#pragma unroll
  for (int j = 0; j < BPW; ++j)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const OutT* p = reinterpret_cast<const OutT*>(a.x) + (size_t)(r < a.m ? r : 0) * a.k + (size_t)(bw + j) * 256 + 4 * lane;
      if (sizeof(OutT) == 4) {
        const f4_t v4 = *reinterpret_cast<const f4_any_t*>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          xv[j][r][e] = v4[e];
      } else {
        const h4_t v4 = *reinterpret_cast<const h4_any_t*>(p);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          xv[j][r][e] = (float)v4[e];
      }
    }
  f4_t nw[BPW];
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < BPW; ++j)
      nw[j] = *reinterpret_cast<const f4_any_t*>(a.norm_w + (size_t)(bw + j) * 256 + 4 * lane);
  }
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (NORM) {
    float ss[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      ss[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < BPW; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          ss[r] = fmaf(xv[j][r][e], xv[j][r][e], ss[r]);
    }
    // The eight sums over the lanes by halving: a lane gives the other half of
    // the rows it holds for its own, until lanes 8r .. 8r + 7 hold row r's (10
    // shuffles; 48 with every lane summing every row).
#pragma unroll
    for (int n = 4; n > 0; n >>= 1) {
      const bool up = lane & (8 * n);
#pragma unroll
      for (int r = 0; r < n; ++r) {
        const float give = up ? ss[r] : ss[r + n];
        ss[r] = (up ? ss[r + n] : ss[r]) + __shfl_xor(give, 8 * n);
      }
    }
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
      ss[0] += __shfl_xor(ss[0], off);
    if ((lane & 7) == 0)
      ssq[wave][lane >> 3] = ss[0];
    __syncthreads();
    // Row r's scale in lanes 8r .. 8r + 7, one square root and division for all.
    // (With every sum and scale formed in every lane the norm took 5 us of a
    // call; so 1.2: 8 rows of 4096 -> 1024 Q4_K 11.2 -> 7.5 us, Q6_K 11.5 -> 7.4.)
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w += 8)
      tot += ssq[w + (lane & 7)][lane >> 3];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1)
      tot += __shfl_xor(tot, off);
    const int scales = __builtin_bit_cast(int, 1.0f / sqrtf(tot / (float)a.k + a.eps));
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const float scale = __builtin_bit_cast(float, __builtin_amdgcn_readlane(scales, 8 * r));
#pragma unroll
      for (int j = 0; j < BPW; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          xv[j][r][e] = (xv[j][r][e] * scale) * nw[j][e];
    }
  }
  // Element e = 4 lane of row r goes to pack lane 16 (e / 64) + r + 8 ((e / 32) & 1),
  // float (e & 31) of its 32.
  float* const xw = xl + (size_t)wave * gu_wave_floats<BPW>();
  const int dl = 16 * (lane >> 4) + 8 * ((lane >> 3) & 1), doff = 4 * (lane & 7);
#pragma unroll
  for (int j = 0; j < BPW; ++j)
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      f4_t v4;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v4[e] = r < a.m ? xv[j][r][e] : 0.0f;
      *reinterpret_cast<f4_t*>(xw + (j * 64 + dl + r) * kXRow + doff) = v4;
    }
  // The first weight loads go out once x has landed, not with it: issued
  // together, every wave's first units queue ahead of the x of later
  // workgroups (measured: kernel 15.0 against 15.6 us at config 1).  The
  // LDS transposition and the register pack below run under them.
  __builtin_amdgcn_sched_barrier(0);
  issue_first();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < BPW; ++j) {
    float t32[32];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const f4_t v4 = *reinterpret_cast<const f4_t*>(xw + (j * 64 + lane) * kXRow + 4 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        t32[4 * c + e] = v4[e];
    }
    pack_x_regs(t32, lane, xb[j]);
  }
}

}  // namespace
}  // namespace q4k
