// Q4_K linear() kernels for gfx950 (MI355X / CDNA4), and the other GGUF
// weight types on the same surface.
//
// Beside this file: q4k_decode.hip (decode_gemv_kernel: up to 8 rows, K = 4096),
// q4k_rows.hip (rows_gemm_kernel: 9 to 63 rows) and q4k_mid.hip (mid_gemm_kernel
// and stage_row_kernel: prefills too small to fill the CUs here).
//
//  stage_x_kernel, stage_gemm_kernel, stage_pack_kernel
//                   activations -> fp16 operands with power-of-two scales
//  q4k_gemv_kernel  staged decode GEMV (up to 48 rows), optionally gated
//  q4k_gemv_splitk_kernel    split-K decode GEMV (K = 12288)
//  typed_gemv_kernel, typed_gemv_persistent_kernel
//                   decode GEMVs over a format policy (Q6_K, Q8_0, Q5_K,
//                   IQ4_XS; Q4_K for the wide LM head)
//  q4k_gemm2_kernel, typed_gemm_kernel
//                   pipelined prefill GEMMs on v_mfma_f32_16x16x32_f16
//  gather_rows_kernel, relayout_kernel, typed_relayout_kernel
//  embedding_kernel, embedding_batch_kernel, rms_norm_kernel, rms_norm8_kernel
//                   the path's neighbours in a pass (token embedding
//                   gather-dequant, RMS norm / LM-head rms_norm_gather)
//
// Reference semantics: backend/metal/kernel/quant_linear.metal and
// backend/metal/kernel/fused_kernels.metal.
#include <float.h>
#include <hip/hip_runtime.h>
#include <stdlib.h>

#include "q4k_pack.h"

namespace q4k {
namespace {

// ----------------------------------------------------------------------------
// Activation staging.  One workgroup of 512 threads per row (K = 4096, 40
// rows: 3.4 us against 5.3 with 256).  Rows of up to 512 * 8 * kStageRegChunks
// elements are held in registers between the max reduction and the
// conversion (one read of x); longer rows are read twice.
// ----------------------------------------------------------------------------
constexpr int kStageThreads = 512, kStageRegChunks = 3;

// Maximum of mx and sum of ss over the workgroup's threads (one barrier).
__device__ __forceinline__ void block_max_sum(float& mx, float& ss) {
  __shared__ float red[2][kStageThreads / 64];
  mx = max64_lanes(mx);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    ss += __shfl_xor(ss, off);
  if ((threadIdx.x & 63) == 0) {
    red[0][threadIdx.x >> 6] = mx;
    red[1][threadIdx.x >> 6] = ss;
  }
  __syncthreads();
  static_assert(kStageThreads == 8 * 64, "sum8_pairs");
#pragma unroll
  for (int w = 0; w < 8; ++w)
    mx = fmaxf(mx, red[0][w]);
  ss = sum8_pairs(red[1]);
}

// Fused RMS norm of a staged row (native_ops.metal:6-40): the staging
// kernels multiply each element by its weight w[k] as it is read, sum the
// squares of the unweighted elements, and fold rsqrt(sum / k + eps) into the
// power-of-two conversion scale.
struct RowNorm {
  const float* w = nullptr;
  float eps = 0.0f;
};

// Converts and stores one 8-element chunk; all threads of the workgroup
// must call it together (the sub-block sum is reduced over 4 lanes).
template <int MODE>
__device__ __forceinline__ void stage_store(_Float16* xo, _Float16* xs, _Float16* xe, int row, int c, bool live, int m, int k, int nb,
                                            const float* v, float up) {
  h8_t hi, lo;
  float sum = 0.0f, res = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    // One fp32 value for both parts (with a norm `up` is no power of two, and
    // a product fused into the conversions would be rounded differently in
    // the stored part and in its residual).
    float t = v[i] * up;
    asm("" : "+v"(t));
    hi[i] = (_Float16)t;
    const float r = t - (float)hi[i];
    lo[i] = (_Float16)r;
    sum += t;
    res += r;
  }
  if (live) {
    *reinterpret_cast<h8_t*>(xo + frag_offset(row, c, nb)) = hi;
    if (MODE == kStageFragSplit)
      *reinterpret_cast<h8_t*>(xo + frag_offset(m + row, c, nb)) = lo;
  }
  // Chunks 4q..4q+3 (lanes 4q..4q+3) form one sub-block.
  sum += __shfl_xor(sum, 1);
  sum += __shfl_xor(sum, 2);
  res += __shfl_xor(res, 1);
  res += __shfl_xor(res, 2);
  if (live && (c & 3) == 0) {
    const float s32 = sum * 0.03125f;
    const _Float16 sh = (_Float16)s32;
    const int b = c >> 5, j = (c >> 2) & 7;
    xs[xs_offset(row, b, j, nb)] = sh;
    if (MODE == kStageFragSplit)
      xs[xs_offset(m + row, b, j, nb)] = (_Float16)(s32 - (float)sh);
    // The sub-block's sum of fp16 rounding residuals (the mean-quant
    // correction's A operand; |.| <= 32 half-ulps of 2^15), zero for hi/lo
    // fragments, whose low parts carry the residuals.
    if (MODE == kStageFrag) {
      xe[xs_offset(row, b, j, nb)] = (_Float16)res;
    } else {
      xe[xs_offset(row, b, j, nb)] = (_Float16)0.0f;
      xe[xs_offset(m + row, b, j, nb)] = (_Float16)0.0f;
    }
  }
}

// Loads chunk c (8 elements) of row xr; with NORM, multiplies each element by
// its norm weight and adds the squares of the unweighted elements to ss.
template <bool NORM, typename InT>
__device__ __forceinline__ void load8_norm(const InT* xr, const float* nw, int c, float* v, float& ss) {
  load8(xr + (size_t)c * 8, v);
  if (NORM) {
    float w8[8];
    load8(nw + (size_t)c * 8, w8);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ss = fmaf(v[i], v[i], ss);
      v[i] *= w8[i];
    }
  }
}

template <typename InT, int MODE, bool NORM>
__global__ __launch_bounds__(kStageThreads) void stage_x_kernel(const InT* __restrict__ x, _Float16* __restrict__ xo, _Float16* __restrict__ xs,
                                                      float* __restrict__ rowscale, int m, int k, RowNorm nrm) {
  const int row = blockIdx.x;
  const InT* xr = x + (size_t)row * k;
  const int chunks = k >> 3, nb = k >> 8;
  const bool in_regs = chunks <= kStageThreads * kStageRegChunks;
  // The residual sums' plane follows the sub-block sums (of m rows, or 2m
  // for hi/lo fragments, whose residual sums are written as zeros).
  _Float16* const xe = xs + xs_plane_halves(MODE == kStageFragSplit ? 2 * m : m, nb);
  float v[kStageRegChunks][8] = {};
  float mx = 0.0f, ss = 0.0f;
  if (in_regs) {
#pragma unroll
    for (int j = 0; j < kStageRegChunks; ++j) {
      const int c = threadIdx.x + kStageThreads * j;
      if (c < chunks) {
        load8_norm<NORM>(xr, nrm.w, c, v[j], ss);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          mx = fmaxf(mx, fabsf(v[j][i]));
      }
    }
  } else {
    for (int c = threadIdx.x; c < chunks; c += kStageThreads) {
      float t[8];
      load8_norm<NORM>(xr, nrm.w, c, t, ss);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mx = fmaxf(mx, fabsf(t[i]));
    }
  }
  float r = 1.0f;
  block_max_sum(mx, ss);
  if (NORM) {
    r = 1.0f / sqrtf(ss / (float)k + nrm.eps);
    mx *= r;
  }
  float up, down;
  pow2_scale(mx, up, down);
  if (threadIdx.x == 0)
    rowscale[row] = down;
  const float cs = NORM ? up * r : up;
  if (in_regs) {
#pragma unroll
    for (int j = 0; j < kStageRegChunks; ++j) {
      const int c = threadIdx.x + kStageThreads * j;
      if (kStageThreads * j < chunks)  // uniform: whole groups of 4 lanes take part
        stage_store<MODE>(xo, xs, xe, row, c, c < chunks, m, k, nb, v[j], cs);
    }
  } else {
    for (int c0 = 0; c0 < chunks; c0 += kStageThreads) {
      const int c = c0 + threadIdx.x;
      float t[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      float unused = 0.0f;
      if (c < chunks)
        load8_norm<NORM>(xr, nrm.w, c, t, unused);
      stage_store<MODE>(xo, xs, xe, row, c, c < chunks, m, k, nb, t, cs);
    }
  }
}

// ----------------------------------------------------------------------------
// Decode pack (m <= 8): x converted once into the MFMA operands of the
// persistent and per-item GEMVs, per 256-element block b:
//   frag[b][s][l]  16 B: A fragment s (v_mfma_f32_16x16x32_f16) of lane l =
//                  16g + i: elements 64g + 32 (s / 4) + 8 (s % 4) + [0, 8)
//                  of row i (i < 8: high fp16 parts, i >= 8: low parts of
//                  row i - 8; zero for rows >= m);
//   xs[b][l]       8 B: min-term A operand (v_mfma_f32_16x16x16_f16) of lane
//                  l = 16G + i: sub-block sums / 32 of sub-blocks 4G..4G+3
//                  (high / low parts as above; zero for G >= 2);
//   dsc[b][r]      float: unscale factor of row r in block b.
// Each (row, block) is scaled by a power of two that puts its largest
// magnitude in [2^14, 2^15); hi + lo carries about 22 significant bits.
// One 64-thread workgroup per (block, row); lane l holds elements 4l..4l+3.
// ----------------------------------------------------------------------------
// Packs the four elements v of lane l (elements 4l..4l+3 of row r of one
// block) into the block's fragments frag_b [8][64], min-term operands xs_b
// [64] and unscale factors dsc_b [8]; the 64 lanes of one wave call it
// together.  The pointers may be global or LDS.
__device__ __forceinline__ void pack_block_row(const float (&v)[4], int r, int l, u4_t* frag_b, h4_t* xs_b, float* dsc_b) {
  const float amax = max64_lanes(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
  float up = 1.0f, down = 1.0f;
  if (amax > 0.0f && amax <= FLT_MAX) {
    int ex;
    frexpf(amax, &ex);
    ex = ex < -80 ? -80 : ex;
    up = ldexpf(1.0f, 15 - ex);
    down = ldexpf(1.0f, ex - 15);
  }
  const float t0 = v[0] * up, t1 = v[1] * up, t2 = v[2] * up, t3 = v[3] * up;
  const h2_t h01 = __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(t0, t1));
  const h2_t h23 = __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(t2, t3));
  const h2_t l01 = __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(t0 - (float)h01[0], t1 - (float)h01[1]));
  const h2_t l23 = __builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_pkrtz(t2 - (float)h23[0], t3 - (float)h23[1]));
  // Element e = 4l: lane group g = e / 64, fragment s = 4 ((e / 32) & 1) +
  // (e / 8) & 3, half offset e & 7 (0 or 4).
  const int e = 4 * l, g = e >> 6, fs = 4 * ((e >> 5) & 1) + ((e >> 3) & 3), h0 = e & 7;
  uint2* fh = reinterpret_cast<uint2*>(reinterpret_cast<_Float16*>(frag_b + fs * 64 + 16 * g + r) + h0);
  uint2* fl = reinterpret_cast<uint2*>(reinterpret_cast<_Float16*>(frag_b + fs * 64 + 16 * g + r + 8) + h0);
  *fh = uint2{__builtin_bit_cast(uint32_t, h01), __builtin_bit_cast(uint32_t, h23)};
  *fl = uint2{__builtin_bit_cast(uint32_t, l01), __builtin_bit_cast(uint32_t, l23)};
  // Sub-block j = l / 8: eight lanes.
  const float sum = sum8_lanes((t0 + t1) + (t2 + t3));
  _Float16* xsh = reinterpret_cast<_Float16*>(xs_b);
  if ((l & 7) == 0) {
    const int j = l >> 3;
    const float s32 = sum * 0.03125f;
    const _Float16 sh = (_Float16)s32;
    xsh[(16 * (j >> 2) + r) * 4 + (j & 3)] = sh;
    xsh[(16 * (j >> 2) + r + 8) * 4 + (j & 3)] = (_Float16)(s32 - (float)sh);
  }
  if (r == 0 && l < 32)  // lanes 32..63 of the min-term operand
    xs_b[32 + l] = h4_t{(_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f, (_Float16)0.0f};
  if (l == 0)
    dsc_b[r] = down;
}

// GEMM staging (kStageGemm) with 8 rows per workgroup: thread t converts row
// t / 32 of the workgroup's 8, chunks (8 elements) t % 32 + 32 j.  The 8
// rows' 16-byte pieces of one fragment lane group are one 128-byte line, so
// every line is written whole by one workgroup (row-per-workgroup staging
// leaves 8 workgroups, on different XCDs, writing 16 bytes of each line).
// TPR threads per row (32, or 64 for long rows: 512 threads per workgroup).
// CPT > 0: the row's K / (8 TPR) <= CPT chunks per thread stay in registers
// between the maximum and the conversion; CPT == 0: x is read twice.  With
// 64 threads per row the 8 pieces of a line come from 8 waves at different
// times, and lines left the L2 partly written (1.38 x the output bytes
// written at K = 12288): those rows pass their pieces through LDS, half of
// the chunks at a time, and 8 consecutive lanes then store each line whole.
// Reduction over the lanes of one staged row: lanes 0..31 and 32..63 of a
// wave are two rows (TPR = 32), or the whole wave is one (TPR = 64).
template <int TPR, bool MAX>
__device__ __forceinline__ float row_reduce(float v) {
  auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
  v = op(v, dpp_f<kDppQuadSwap1>(v));
  v = op(v, dpp_f<kDppQuadSwap2>(v));
  v = op(v, dpp_f<kDppHalfMirror>(v));
  v = op(v, dpp_f<kDppRowMirror>(v));
  const int b = __builtin_bit_cast(int, v);
  const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 0)), r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 16));
  const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 32)), r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, 48));
  return TPR == 64 ? op(op(r0, r1), op(r2, r3)) : (threadIdx.x & 63) < 32 ? op(r0, r1) : op(r2, r3);
}

template <typename InT, int CPT, int TPR, bool NORM>
__global__ __launch_bounds__(8 * TPR) void stage_gemm_kernel(const InT* __restrict__ x, _Float16* __restrict__ xo, float* __restrict__ rowscale,
                                                             int m, int k, RowNorm nrm) {
  static_assert(TPR == 32 || TPR == 64, "one row per half wave or per wave");
  const int t = threadIdx.x, q = t & (TPR - 1);
  const int row = blockIdx.x * 8 + t / TPR;
  const bool live = row < m;
  const int nb = k >> 8, cpt = (k >> 3) / TPR;
  const InT* xr = x + (size_t)(live ? row : 0) * k;
  float v[CPT > 0 ? CPT : 1][8];
  float mx = 0.0f, ss = 0.0f;
#pragma unroll
  for (int j = 0; j < (CPT > 0 ? CPT : 1); ++j)
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[j][i] = 0.0f;
  if (CPT > 0) {
#pragma unroll
    for (int j = 0; j < CPT; ++j)
      if (live && j < cpt)
        load8_norm<NORM>(xr, nrm.w, q + TPR * j, v[j], ss);
#pragma unroll
    for (int j = 0; j < CPT; ++j)
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mx = fmaxf(mx, fabsf(v[j][i]));
  } else if (live) {
    for (int j = 0; j < cpt; ++j) {
      float w[8];
      load8_norm<NORM>(xr, nrm.w, q + TPR * j, w, ss);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        mx = fmaxf(mx, fabsf(w[i]));
    }
  }
  mx = row_reduce<TPR, true>(mx);
  float r = 1.0f;
  if (NORM) {
    r = 1.0f / sqrtf(row_reduce<TPR, false>(ss) / (float)k + nrm.eps);
    mx *= r;
  }
  float up, down;
  pow2_scale(mx, up, down);
  // Rows past m write nothing; with the LDS path their waves stay for its
  // barriers.
  if (!live && !(CPT > 0 && TPR == 64))
    return;
  if (q == 0 && live)
    rowscale[row] = down;
  const float cs = NORM ? up * r : up;
  auto put = [&](int j, const float* w) {
    h8_t h;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      h[i] = (_Float16)(w[i] * cs);
    *reinterpret_cast<h8_t*>(xo + gemm_frag_offset(row, q + TPR * j, nb)) = h;
  };
  if constexpr (CPT > 0 && TPR == 64) {
    // LDS piece (chunk, row of the 8) at 16 (8 chunk + row); CPT / 2 chunks
    // of every thread per half.
    constexpr int HALF = (CPT + 1) / 2;
    __shared__ __attribute__((aligned(16))) h8_t piece[HALF * TPR * 8];
    const int r8 = t / TPR;
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      if (hf)
        __syncthreads();  // the first half's stores have read their pieces
#pragma unroll
      for (int jj = 0; jj < HALF; ++jj) {
        const int j = hf * HALF + jj;
        if (j < CPT && j < cpt) {
          h8_t h;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            h[i] = (_Float16)(v[j][i] * cs);
          piece[(jj * TPR + q) * 8 + r8] = h;
        }
      }
      __syncthreads();
      // Thread t stores piece (chunk (t / 8) + 64 i of the half, row t % 8):
      // lanes 8c .. 8c + 7 write one whole line.
      const int pr = t & 7, pc = t >> 3;
      const int prow = blockIdx.x * 8 + pr;
#pragma unroll
      for (int i = 0; i < HALF; ++i) {
        const int jj = i, j = hf * HALF + jj, c = pc + TPR * j;
        if (j < CPT && j < cpt && prow < m)
          *reinterpret_cast<h8_t*>(xo + gemm_frag_offset(prow, c, nb)) = piece[(jj * TPR + pc) * 8 + pr];
      }
    }
  } else if (CPT > 0) {
#pragma unroll
    for (int j = 0; j < (CPT > 0 ? CPT : 1); ++j)
      if (j < cpt)
        put(j, v[j]);
  } else {
    for (int j = 0; j < cpt; ++j) {
      float w[8];
      float unused = 0.0f;
      load8_norm<NORM>(xr, nrm.w, q + TPR * j, w, unused);
      put(j, w);
    }
  }
}

template <typename InT>
__global__ __launch_bounds__(64) void stage_pack_kernel(const InT* __restrict__ x, u4_t* __restrict__ frag, h4_t* __restrict__ xs,
                                                        float* __restrict__ dsc, int m, int k) {
  const int b = blockIdx.x >> 3, r = blockIdx.x & 7, l = threadIdx.x;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (r < m) {
    const InT* p = x + (size_t)r * k + (size_t)b * 256 + 4 * l;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = (float)p[e];
  }
  pack_block_row(v, r, l, frag + (size_t)b * 8 * 64, xs + (size_t)b * 64, dsc + (size_t)b * 8);
}

// ----------------------------------------------------------------------------
// GEMV (decode / small prefill / gated decode).
//
// Workgroup = W waves over T column tiles (16T output columns); the K blocks
// are split into W contiguous ranges, one per wave, and the partial sums are
// reduced through LDS.  Per tile-block a wave issues three fully contiguous
// 16-byte loads per lane (two quant slabs + header) and, per 16-row tile of
// activations, 8 MFMAs with B = q*sc (exact fp16) plus one 16x16x16 MFMA of
// the sub-block sums against 32*m_j, then acc += d * C_q - dmin * C_m in fp32
// -- the decode form of quant_linear.metal:288-302 with the integer parts on
// the matrix core.
// ----------------------------------------------------------------------------
template <int T, int NM>
struct TileWords {
  u4_t q0[NM][T], q1[NM][T], hd[NM][T];
};

template <int T, int NM>
__device__ __forceinline__ void load_tile_words(TileWords<T, NM>& tw, const GemvArgs& a, int ct0, int b, int nb, int lane, int col) {
#pragma unroll
  for (int mi = 0; mi < NM; ++mi)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint8_t* p = (mi ? a.wu : a.w) + ((size_t)(ct0 + t) * nb + b) * kTileBlockBytes;
      tw.q0[mi][t] = *reinterpret_cast<const u4_t*>(p + 16 * lane);
      tw.q1[mi][t] = *reinterpret_cast<const u4_t*>(p + kSlabBytes + 16 * lane);
      tw.hd[mi][t] = *reinterpret_cast<const u4_t*>(p + kHeaderOffset + 16 * col);
    }
}

// BPW > 0: every wave owns exactly BPW blocks (nb == W * BPW) and issues all of
// their weight loads at once; BPW == 0: any split, with a one-block prefetch.
template <int RT, int T, int W, int BPW, bool GATED, typename OutT>
__global__ __launch_bounds__(64 * W) void q4k_gemv_kernel(GemvArgs a) {
  constexpr int NM = GATED ? 2 : 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g = lane >> 4, col = lane & 15;
  const int nb = a.nb;
  const int ct0 = blockIdx.x * T;
  const int b0 = nb * wave / W, b1 = nb * (wave + 1) / W;

  f4_t acc[NM][T][RT];
#pragma unroll
  for (int mi = 0; mi < NM; ++mi)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
        acc[mi][t][rt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // Dead activation rows (>= a.rows, inside the padded 16-row tiles) are
  // loaded unmasked: in a matrix product a garbage A row only reaches its own
  // C row, which the epilogue never reads.  Branch-free loads keep the vmcnt
  // waits exact.
  // The min-term operand: lanes 0..31 the sub-block sums / 32, lanes 32..63
  // (k = 8..15) the sub-blocks' sums of fp16 rounding residuals from the
  // plane after them (zeros for hi/lo rows), as in the rows GEMV.
  const h4_t* const xsrc = reinterpret_cast<const h4_t*>(a.xs + (lane >= 32 ? xs_plane_halves(a.rows, nb) : 0));
  auto load_x = [&](h8_t (&xa)[RT][8], h4_t (&xsa)[RT], int b) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const h8_t* xp = reinterpret_cast<const h8_t*>(a.xf) + (size_t)(rt * nb + b) * 8 * 64 + lane;
#pragma unroll
      for (int s = 0; s < 8; ++s)
        xa[rt][s] = xp[s * 64];
      xsa[rt] = xsrc[(size_t)(rt * nb + b) * 32 + (lane & 31)];
    }
  };
  auto compute = [&](const TileWords<T, NM>& cur, const h8_t (&xa)[RT][8], const h4_t (&xsa)[RT]) {
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const BlockConsts kc = block_consts(cur.hd[mi][t], g);
        f4_t cq[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
          cq[rt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const u4_t q = u < 2 ? cur.q0[mi][t] : cur.q1[mi][t];
          const uint32_t wa = q[2 * (u & 1)], wb = q[2 * (u & 1) + 1];
          const h8_t blo = quant_times_scale(wa, wb, 0x000F000Fu, 0x64006400u, kc.mul_lo, kc.add_lo);
          const h8_t bhi = quant_times_scale(wa, wb, 0x00F000F0u, 0x64006400u, kc.mul_hi, kc.add_hi);
#pragma unroll
          for (int rt = 0; rt < RT; ++rt) {
            cq[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[rt][u], blo, cq[rt], 0, 0, 0);
            cq[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[rt][4 + u], bhi, cq[rt], 0, 0, 0);
          }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          // mean-quant correction of the fp16 rounding (k = 8 + j; single
          // fp16 rows, m >= 25, need at least two row tiles: one holds only
          // hi/lo rows), then the min term: sum_j (xs_j / 32) * (32 m_j)
          if constexpr (RT >= 2)
            cq[rt] = __builtin_amdgcn_mfma_f32_16x16x16f16(xsa[rt], kc.bsc, cq[rt], 0, 0, 0);
          const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(xsa[rt], kc.bmin, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; ++v)
            acc[mi][t][rt][v] = fmaf(kc.d, cq[rt][v], fmaf(-kc.dmin, cm[v], acc[mi][t][rt][v]));
        }
      }
  };

  if constexpr (BPW > 0) {
    // Issue order for the in-order vmcnt counter: block 0's activations, all
    // BPW blocks' weights, then each later block's activations just in time.
    TileWords<T, NM> tw[BPW];
    h8_t xa[RT][8];
    h4_t xsa[RT];
    load_x(xa, xsa, b0);
#pragma unroll
    for (int j = 0; j < BPW; ++j)
      load_tile_words(tw[j], a, ct0, b0 + j, nb, lane, col);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      if (j > 0)
        load_x(xa, xsa, b0 + j);
      compute(tw[j], xa, xsa);
    }
  } else {
    TileWords<T, NM> cur, next;
    if (b0 < b1)
      load_tile_words(cur, a, ct0, b0, nb, lane, col);
    for (int b = b0; b < b1; ++b) {
      h8_t xa[RT][8];
      h4_t xsa[RT];
      load_x(xa, xsa, b);
      __builtin_amdgcn_sched_barrier(0);
      if (b + 1 < b1)
        load_tile_words(next, a, ct0, b + 1, nb, lane, col);
      __builtin_amdgcn_sched_barrier(0);
      compute(cur, xa, xsa);
      cur = next;
    }
  }

  // Cross-wave reduction through LDS in [wave][matrix][tile][row][column]
  // order (the C fragment of lane l is rows 4*(l/16)+v, column l%16).
  constexpr int ROWS = RT * 16;
  __shared__ float red[W][NM][T][ROWS][16];
#pragma unroll
  for (int mi = 0; mi < NM; ++mi)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          red[wave][mi][t][rt * 16 + 4 * g + v][col] = acc[mi][t][rt][v];
  __syncthreads();

  // Epilogue: one thread per output (row, column); split rows add their low half.
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  for (int item = tid; item < a.m * 16 * T; item += 64 * W) {
    const int row = item / (16 * T), c = item % (16 * T), t = c >> 4, cc = c & 15;
    float s[NM];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi) {
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w)
        v += red[w][mi][t][row][cc];
      if (a.split) {
#pragma unroll
        for (int w = 0; w < W; ++w)
          v += red[w][mi][t][a.m + row][cc];
      }
      s[mi] = v;
    }
    const float scale = a.rowscale[row];
    const size_t o = (size_t)row * a.n + (size_t)(ct0 + t) * 16 + cc;
    float out;
    if (GATED) {
      float gv = s[0] * scale, uv = s[NM - 1] * scale;
      if (sizeof(OutT) == 2) {
        gv = round_half(gv);
        uv = round_half(uv);
      }
      out = silu(gv) * uv;
    } else {
      float acc_v = s[0] * scale;
      if (sizeof(OutT) == 2)
        acc_v = round_half(acc_v);
      out = a.post == 1 ? acc_v + load_elem(aux, o) : a.post == 2 ? silu(load_elem(aux, o)) * acc_v : acc_v;
    }
    store_elem(y, o, out);
  }
}

// ----------------------------------------------------------------------------
// Load helpers of the GEMVs that stream weights through LDS.
// ----------------------------------------------------------------------------

// ----------------------------------------------------------------------------
// GEMV for staged activations of 17..48 fragment rows (the decode pass of a
// speculative batch, up to 8 queries x 5 rows), K = 2048 .. 12288.
//
// The work split of the fused gate/up GEMV over the staged fp16 fragments
// (stage_x_kernel, one power-of-two scale per row; split rows carry the low
// parts) of the RT row tiles: workgroup = one item of T column tiles of NM
// matrices (NM = 2: gate and up), 8 waves; wave w owns K-blocks bw ..
// bw + BPW - 1 (bw = BPW ((w + item) % 8)) of the item's NM T (matrix, tile)
// pairs, U = BPW NM T units.  The wave loads a block's fragments for all RT
// row tiles once (RT x 8 KB from the staging) and every unit of that block
// multiplies them: RT x 8 v_mfma_f32_16x16x32_f16 and RT min-term MFMAs per
// tile-block dequantised once.  A CU thus reads the staged x once per T
// column tiles of NM matrices; the one-tile GEMV reads it once per column
// tile, and at M = 40 its gated launch was bound by those reads (768
// workgroups x 384 KB).  Units stream two ahead as in the fused gate/up
// GEMV; a block's fragments replace the previous block's after its units
// (one L2 round trip per block and wave, which the SIMD's other wave
// covers).  The 8 waves' partial sums meet in LDS in wave order.
// KS > 1 K-slices: workgroup b takes slice b % KS (blocks 8 BPW of them) of
// column group b / KS, so that KS times fewer column groups, each of KS
// times more column tiles, read all of x; each slice's workgroup writes its
// sums (written through to memory) and the last of the KS to arrive (a
// per-group counter, reset by it) adds them in slice order and runs the
// epilogue.  No workgroup waits for another.
// ----------------------------------------------------------------------------
template <int NM, int T, int RT, int BPW, typename OutT, int KS = 1>
__global__ __launch_bounds__(512) void q4k_gemv_rows_kernel(GemvArgs a) {
  constexpr int W = 8, MT = NM * T, U = BPW * MT, ROWS = 16 * RT, DQ = 2;
  __shared__ float red[W][MT][ROWS][16];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int item = blockIdx.x / KS, ks = blockIdx.x % KS, nb = a.nb;
  const int bw = ks * (W * BPW) + BPW * ((wave + item) % W);
  const size_t tile_bytes = (size_t)nb * kTileBlockBytes;

  u4_t hdr[U], q0[U], q1[U];
  auto issue_unit = [&](int u) {
    const int j = u / MT, mt = u - j * MT, mi = mt / T, t = mt - mi * T;
    const uint8_t* src = (mi ? a.wu : a.w) + ((size_t)item * T + t) * tile_bytes + (size_t)(bw + j) * kTileBlockBytes;
    hdr[u] = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + kHeaderOffset) + col);
    q0[u] = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src) + lane);
    q1[u] = __builtin_nontemporal_load(reinterpret_cast<const u4_t*>(src + kSlabBytes) + lane);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Dead fragment rows (>= a.rows inside the last row tile) are loaded as
  // they are: a garbage A row reaches only its own C row, never stored.
  h8_t xa[RT][8];
  // The min-term MFMA's A operand: lanes 0..31 (k = 0..7) the sub-block sums
  // / 32; lanes 32..63 (k = 8..15) the sub-blocks' sums of fp16 rounding
  // residuals, from the plane after the sums that stage_x_kernel writes
  // (zeros for hi/lo fragments).  Each of the two MFMAs that read it has a
  // zero B operand for the other half's k.
  h4_t xsa[RT];
  const h4_t* const xsrc = reinterpret_cast<const h4_t*>(a.xs + (lane >= 32 ? xs_plane_halves(a.rows, nb) : 0));
  auto load_x = [&](int b) {
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const h8_t* xp = reinterpret_cast<const h8_t*>(a.xf) + (size_t)(rt * nb + b) * 8 * 64 + lane;
#pragma unroll
      for (int s = 0; s < 8; ++s)
        xa[rt][s] = xp[s * 64];
      xsa[rt] = xsrc[(size_t)(rt * nb + b) * 32 + (lane & 31)];
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  load_x(bw);
#pragma unroll
  for (int u = 0; u < (DQ < U ? DQ : U); ++u)
    issue_unit(u);

  f4_t acc[MT][RT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      acc[mt][rt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = u / MT, mt = u - j * MT;
    __builtin_amdgcn_sched_barrier(0);
    if (u > 0 && mt == 0)
      load_x(bw + j);
    if (u + DQ < U)
      issue_unit(u + DQ);
    const BlockConsts kc = block_consts(hdr[u], g);
    f4_t cq[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
      cq[rt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const u4_t qq = s < 2 ? q0[u] : q1[u];
      const uint32_t wa = qq[2 * (s & 1)], wb = qq[2 * (s & 1) + 1];
      const h8_t blo = quant_times_scale(wa, wb, 0x000F000Fu, 0x64006400u, kc.mul_lo, kc.add_lo);
      const h8_t bhi = quant_times_scale(wa, wb, 0x00F000F0u, 0x64006400u, kc.mul_hi, kc.add_hi);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        cq[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[rt][s], blo, cq[rt], 0, 0, 0);
        cq[rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[rt][4 + s], bhi, cq[rt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      // Mean-quant correction of the fp16 rounding: sum_j E_j * 7.5 sc_j
      // (k = 8 + j), E_j = the sub-block's sum of rounding residuals: the
      // part of the q-term's error common to every column.
      if constexpr (RT >= 2)
        cq[rt] = __builtin_amdgcn_mfma_f32_16x16x16f16(xsa[rt], kc.bsc, cq[rt], 0, 0, 0);
      // min term: sum_j (xs_j / 32) * (32 m_j), k = sub-block
      const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(xsa[rt], kc.bmin, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[mt][rt][v] = fmaf(kc.d, cq[rt][v], fmaf(-kc.dmin, cm[v], acc[mt][rt][v]));
      // Each unit's sums are folded here: otherwise the compiler defers the
      // folds and keeps every unit's MFMA results live.
      asm volatile("" : "+v"(acc[mt][rt]));
    }
  }

  // C fragment of lane l: rows 4 (l / 16) + v of each row tile, column l % 16.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[wave][mt][rt * 16 + 4 * g + v][col] = acc[mt][rt][v];
  __syncthreads();
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  constexpr int EPI = 16 * T;
  // This workgroup's sum of output o (row o / EPI, column o % EPI) of
  // matrix mi: the waves in order, then (split rows) the low parts.
  auto wave_sum = [&](int o, int mi) {
    const int row = o / EPI, c = o % EPI, t = c >> 4, cc = c & 15;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w)
      v += red[w][mi * T + t][row][cc];
    if (a.split) {
#pragma unroll
      for (int w = 0; w < W; ++w)
        v += red[w][mi * T + t][a.m + row][cc];
    }
    return v;
  };
  // K-slices: outputs of slice k2 of matrix mi at part + ((item KS + k2) NM
  // + mi) ROWS EPI + o.  Per thread at most PER outputs (o = tid + 512 r).
  constexpr int PER = (ROWS * EPI + 64 * W - 1) / (64 * W);
  float sl[PER][NM];
  if constexpr (KS > 1) {
    float* const mine = a.part + ((size_t)item * KS + ks) * NM * ROWS * EPI;
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int o = tid + r * 64 * W;
      if (o < a.m * EPI) {
#pragma unroll
        for (int mi = 0; mi < NM; ++mi)
          store_coherent(mine + mi * ROWS * EPI + o, wave_sum(o, mi));
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0)
      s_last = count_arrival(&a.counters[item]) == KS - 1;
    __syncthreads();
    if (!s_last)
      return;
    // Every slice's sums, loaded together, then added in slice order.
    float pv[PER][NM][KS];
    const float* const grp = a.part + (size_t)item * KS * NM * ROWS * EPI;
#pragma unroll
    for (int r = 0; r < PER; ++r) {
      const int o0 = tid + r * 64 * W, o = o0 < a.m * EPI ? o0 : 0;
#pragma unroll
      for (int mi = 0; mi < NM; ++mi)
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2)
          pv[r][mi][k2] = load_coherent(grp + (k2 * NM + mi) * ROWS * EPI + o);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int r = 0; r < PER; ++r)
#pragma unroll
      for (int mi = 0; mi < NM; ++mi) {
        float v = 0.0f;
#pragma unroll
        for (int k2 = 0; k2 < KS; ++k2) {
          hold(pv[r][mi][k2]);
          v += pv[r][mi][k2];
        }
        sl[r][mi] = v;
      }
    if (tid == 0)
      reset_counter(&a.counters[item]);  // ready for the next launch
  }
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int o = tid + r * 64 * W;
    if (o >= a.m * EPI)
      break;
    const int row = o / EPI, c = o % EPI, t = c >> 4, cc = c & 15;
    float s[NM];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
      s[mi] = (KS > 1 ? sl[r][mi] : wave_sum(o, mi)) * a.rowscale[row];
    const size_t off = (size_t)row * a.n + ((size_t)item * T + t) * 16 + cc;
    float out;
    if (NM == 2) {
      float gv = s[0], uv = s[NM - 1];
      if (sizeof(OutT) == 2) {
        gv = round_half(gv);
        uv = round_half(uv);
      }
      out = silu(gv) * uv;
    } else {
      float acc_v = s[0];
      if (sizeof(OutT) == 2)
        acc_v = round_half(acc_v);
      out = a.post == 1 ? acc_v + load_elem(aux, off) : a.post == 2 ? silu(load_elem(aux, off)) * acc_v : acc_v;
    }
    store_elem(y, off, out);
  }
}

// ----------------------------------------------------------------------------
// Split-K GEMV (m <= 8 rows, split hi/lo into one 16-row activation tile).
//
// Each CU of a persistent launch would otherwise pull all of x from L2 (32 MB
// across the chip for m = 8, K = 4096, fp32) before its first MFMA.  Here
// workgroup b covers column group `grp` (T tiles of NM matrices) over one
// K-slice `ks` of BPS blocks, so it reads only its slice of x:
//  1. the workgroup converts its slice of x once into LDS: A fragments
//     (fp16 high parts in rows 0..7, low parts in rows 8..15, per-(row, slice)
//     power-of-two scale) and the min-term fragments (sub-block sums / 32);
//  2. wave w owns (matrix, tile) pairs w, w + 8, ... (PW of them) and streams
//     their tile-blocks of the slice through a private LDS ring with DP
//     block-steps in flight; a block-step is PW independent MFMA chains
//     over one set of A fragments;
//  3. each wave writes its slice partials (hi + lo rows combined, unscaled)
//     to the workspace; the last workgroup of the group to arrive (a device-
//     scope counter, reset by that workgroup) sums the KS slices in slice
//     order and runs the epilogue.  No workgroup ever waits for another.
// Workgroups of one group are placed on one XCD (workgroup b runs on XCD
// b % 8), so their partials meet in one L2.
// ----------------------------------------------------------------------------
// Bytes of LDS one split-K slice uses.
// The slice of x as read: one row of one block per (block, row) pair, 1 KB
// of fp32 (512 B of fp16) at a stride of 1040 B, so that the 8 rows' 128-byte
// reads of the pack fall in different banks.
constexpr int kSplitkStageStride = 1040;
template <int NM, int T, int BPS, int DP>
constexpr int splitk_lds_bytes() {
  return 8 * DP * (NM * T / 8) * kTileBlockBytes + BPS * 8 * 64 * 16 + BPS * 64 * 8 + BPS * 8 * 4 + BPS * 8 * kSplitkStageStride;
}

// One workgroup's K-slice ks of column group grp (see above), over LDS of
// splitk_lds_bytes().
template <int NM, int T, int KS, int BPS, int DP, typename OutT>
__device__ __forceinline__ void splitk_slice(const GemvArgs& a, uint8_t* lds, int* s_last, float* __restrict__ part, int* __restrict__ counters,
                                             int grp, int ks) {
  constexpr int W = 8, MT = NM * T, PW = MT / W;
  static_assert(MT % W == 0, "whole (matrix, tile) pairs per wave");
  // LDS: the rings, then the slice's decode pack (fragments, min-term
  // operands, unscale factors: the same layout as in global memory).
  constexpr int kFragBytes = BPS * 8 * 64 * 16;  // [BPS][8 fragments][64 lanes] x 16 B
  constexpr int kXsBytes = BPS * 64 * 8;         // [BPS][64 lanes] x 4 halves
  constexpr int kDscBytes = BPS * 8 * 4;         // [BPS][8 rows]
  constexpr int kStageBytes = BPS * 8 * kSplitkStageStride;  // the slice of x as read, per (block, row) pair
  constexpr int kSlots = DP * PW;                // ring slots per wave
  constexpr int kRingBytes = W * kSlots * kTileBlockBytes;
  static_assert(kRingBytes + kFragBytes + kXsBytes + kDscBytes + kStageBytes == splitk_lds_bytes<NM, T, BPS, DP>(), "LDS layout");
  uint8_t* const stage = lds + kRingBytes + kFragBytes + kXsBytes + kDscBytes;
  u4_t* const xf = reinterpret_cast<u4_t*>(lds + kRingBytes);
  _Float16* const xs = reinterpret_cast<_Float16*>(lds + kRingBytes + kFragBytes);
  const float* const dscl = reinterpret_cast<const float*>(lds + kRingBytes + kFragBytes + kXsBytes);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int nb = a.nb, kb0 = ks * BPS;
  uint8_t* const ring = lds + (size_t)wave * kSlots * kTileBlockBytes;
  const uint32_t ring0 = lds_addr(ring);
  const uint32_t voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;

  // Block-step i of this wave: block kb0 + i of each of its PW pairs, into
  // slot group i % DP.  Steps past the end re-load the last one (L2 hits),
  // so every step issues exactly 3 * PW loads.
  auto issue = [&](int i) {
    __builtin_amdgcn_sched_barrier(0);
    const int bb = i < BPS ? i : BPS - 1;
    const int sg = i % DP;
#pragma unroll
    for (int pw = 0; pw < PW; ++pw) {
      const int mt = wave + W * pw, mi = mt / T, t = mt - mi * T;
      const size_t ct = (size_t)grp * T + t;
      const uint8_t* src = uniform_ptr((mi ? a.wu : a.w) + (ct * nb + kb0 + bb) * kTileBlockBytes);
      const uint32_t l = __builtin_amdgcn_readfirstlane(ring0 + (uint32_t)(sg * PW + pw) * kTileBlockBytes);
      lds_dma16<0>(src, voff16, l);
      lds_dma16<kSlabBytes>(src, voff16, l);
      lds_dma4<kHeaderOffset>(src, voff4, l);
    }
  };

  // 1. The workgroup packs its slice of x into LDS (the decode pack layout,
  // see stage_pack_kernel): wave w converts (block, row) pairs w, w + 8, ...
  // of the slice.  The slice arrives by LDS DMA like the weights, issued
  // before them; a wait that leaves the weight loads in flight
  // (vmcnt(3 * PW * DP)) then covers x alone.  (Compiler-visible loads of x
  // would be waited for with vmcnt(0): the compiler does not count the
  // weight DMAs, so that wait would also cover the first weight steps.)
  constexpr int PPW = BPS * 8 / W;  // (block, row) pairs per wave
  static_assert(BPS * 8 % W == 0, "whole pairs per wave");
  static_assert(3 * PW * DP <= 63, "vmcnt range");
  const OutT* const xin = reinterpret_cast<const OutT*>(a.x);
  const bool live = (wave & 7) < a.m;  // row (wave + 8j) & 7 of every pair of this wave
  if (live) {
#pragma unroll
    for (int j = 0; j < PPW; ++j) {
      const int pr = wave + W * j, r = pr & 7;
      const OutT* src = xin + (size_t)r * a.k + (size_t)(kb0 + (pr >> 3)) * 256;
      const uint32_t l = __builtin_amdgcn_readfirstlane(lds_addr(stage + (size_t)pr * kSplitkStageStride));
      if (sizeof(OutT) == 4) {
        lds_dma16<0>(uniform_ptr(reinterpret_cast<const uint8_t*>(src)), voff16, l);
      } else {
        lds_dma4<0>(uniform_ptr(reinterpret_cast<const uint8_t*>(src)), voff4, l);
        lds_dma4<256>(uniform_ptr(reinterpret_cast<const uint8_t*>(src)), voff4, l);
      }
    }
  }
  __builtin_amdgcn_s_barrier();  // the workgroup's x requests ahead of its weight requests
#pragma unroll
  for (int i = 0; i < DP; ++i)
    issue(i);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PW * DP) : "memory");
  __syncthreads();
  // Wave w < BPS packs block w of the slice, all 8 rows, as the fused gate/up
  // GEMV packs its blocks: lane 16 g + 8 h + r takes elements 64 g + 32 h +
  // [0, 32) of row r (128 contiguous bytes of the stage), so that the row
  // maximum and the sub-block sums are mostly in-lane, and writes the block's
  // fragments, min-term operands and unscale factors to LDS.  Rows >= m are
  // zero.
  static_assert(BPS <= W, "one block per packing wave");
  if (wave < BPS) {
    const int r = lane & 7, e0 = 64 * (lane >> 4) + 32 * ((lane >> 3) & 1);
    const uint8_t* src = stage + (size_t)(8 * wave + r) * kSplitkStageStride;
    float t32[32];
    if (sizeof(OutT) == 4) {
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const f4_t v4 = *reinterpret_cast<const f4_t*>(src + 4 * e0 + 16 * c);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          t32[4 * c + e] = v4[e];
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const h8_t v8 = *reinterpret_cast<const h8_t*>(src + 2 * e0 + 16 * c);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          t32[8 * c + e] = (float)v8[e];
      }
    }
    if (r >= a.m) {
#pragma unroll
      for (int e = 0; e < 32; ++e)
        t32[e] = 0.0f;
    }
    XBlock xb;
    pack_x_regs(t32, lane, xb);
#pragma unroll
    for (int f = 0; f < 8; ++f)
      xf[((size_t)wave * 8 + f) * 64 + lane] = __builtin_bit_cast(u4_t, xb.frag[f]);
    reinterpret_cast<h4_t*>(xs)[(size_t)wave * 64 + lane] = xb.xs;
    if (lane == 0 || lane == 16) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        const_cast<float*>(dscl)[wave * 8 + (lane >> 2) + v] = xb.dv[v];
    }
  }
  __syncthreads();

  // 2. Stream the slice's tile-blocks of this wave's pairs.
  f4_t acc[PW];
#pragma unroll
  for (int pw = 0; pw < PW; ++pw)
    acc[pw] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < BPS; ++i) {
    // 3 * PW loads per step: with DP steps outstanding, this marks step i.
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PW * (DP - 1)) : "memory");
    const u4_t* sl = reinterpret_cast<const u4_t*>(ring + (size_t)(i % DP) * PW * kTileBlockBytes);
    u4_t q0[PW], q1[PW], hd[PW];
#pragma unroll
    for (int pw = 0; pw < PW; ++pw) {
      const u4_t* su = sl + pw * (kTileBlockBytes / 16);
      q0[pw] = su[lane];
      q1[pw] = su[kSlabBytes / 16 + lane];
      hd[pw] = su[kHeaderOffset / 16 + col];
    }
    h8_t xa[8];
#pragma unroll
    for (int f = 0; f < 8; ++f)
      xa[f] = __builtin_bit_cast(h8_t, xf[(i * 8 + f) * 64 + lane]);
    const h4_t xsa = *reinterpret_cast<const h4_t*>(xs + (i * 64 + lane) * 4);
    // Unscale factors of this lane's C rows (4g + v) & 7 in block i.
    const f4_t dv = *reinterpret_cast<const f4_t*>(dscl + i * 8 + 4 * (g & 1));
    // The step is in registers: its slots take the step DP ahead.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(i + DP);
#pragma unroll
    for (int pw = 0; pw < PW; ++pw) {
      const BlockConsts kc = block_consts(hd[pw], g);
      f4_t cl = f4_t{0.0f, 0.0f, 0.0f, 0.0f}, ch = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const u4_t qq = u < 2 ? q0[pw] : q1[pw];
        const uint32_t wa = qq[2 * (u & 1)], wb = qq[2 * (u & 1) + 1];
        const h8_t blo = quant_times_scale(wa, wb, 0x000F000Fu, 0x64006400u, kc.mul_lo, kc.add_lo);
        const h8_t bhi = quant_times_scale(wa, wb, 0x00F000F0u, 0x64006400u, kc.mul_hi, kc.add_hi);
        cl = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[u], blo, cl, 0, 0, 0);
        ch = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[4 + u], bhi, ch, 0, 0, 0);
      }
      const f4_t cm = __builtin_amdgcn_mfma_f32_16x16x16f16(xsa, kc.bmin, f4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[pw][v] += fmaf(kc.d, cl[v] + ch[v], -kc.dmin * cm[v]) * dv[v];
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // 3. Slice partials: C row r (lanes g < 2) plus its low part r + 8 (lanes
  // g + 2), unscaled; layout [grp][ks][mt][8 rows][16 columns].  They are
  // written through to memory (system-coherent stores) and read back the
  // same way, so no cache of any XCD needs flushing; the counter is a
  // device-scope atomic.
#pragma unroll
  for (int pw = 0; pw < PW; ++pw) {
    const int mt = wave + W * pw;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float tot = acc[pw][v] + __shfl_xor(acc[pw][v], 32);
      const int row = 4 * g + v;
      if (g < 2 && row < a.m)
        store_coherent(part + ((((size_t)grp * KS + ks) * MT + mt) * 8 + row) * 16 + col, tot);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0)
    *s_last = count_arrival(&counters[grp]) == KS - 1;
  __syncthreads();
  if (!*s_last)
    return;
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  constexpr int EPI = 16 * T;  // outputs per row of a group
  // The outputs of the group this thread finishes (at most PER of them), with
  // all their loads (the KS slice partials, and aux) issued before a single
  // wait: the reduction costs one memory round trip, not two per output.
  constexpr int PER = (8 * EPI + 64 * W - 1) / (64 * W);
  float pv[PER][NM][KS], av[PER];
  size_t offs[PER];
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    const int o0 = tid + r * 64 * W, o = o0 < a.m * EPI ? o0 : 0;
    const int row = o / EPI, c = o % EPI, t = c >> 4, cc = c & 15;
#pragma unroll
    for (int mi = 0; mi < NM; ++mi)
#pragma unroll
      for (int k2 = 0; k2 < KS; ++k2)
        pv[r][mi][k2] = load_coherent(part + ((((size_t)grp * KS + k2) * MT + mi * T + t) * 8 + row) * 16 + cc);
    offs[r] = (size_t)row * a.n + ((size_t)grp * T + t) * 16 + cc;
    av[r] = NM == 1 && a.post != 0 ? load_elem(aux, offs[r]) : 0.0f;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int r = 0; r < PER; ++r) {
    if (tid + r * 64 * W >= a.m * EPI)
      break;
    float sm[NM];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi) {
      float v = 0.0f;
#pragma unroll
      for (int k2 = 0; k2 < KS; ++k2) {
        hold(pv[r][mi][k2]);
        v += pv[r][mi][k2];
      }
      sm[mi] = v;
    }
    float out;
    if (NM == 2) {
      float gv = sm[0], uv = sm[NM - 1];
      if (sizeof(OutT) == 2) {
        gv = round_half(gv);
        uv = round_half(uv);
      }
      out = silu(gv) * uv;
    } else {
      float acc_v = sm[0];
      if (sizeof(OutT) == 2)
        acc_v = round_half(acc_v);
      out = a.post == 1 ? acc_v + av[r] : a.post == 2 ? silu(av[r]) * acc_v : acc_v;
    }
    store_elem(y, offs[r], out);
  }
  if (tid == 0)
    reset_counter(&counters[grp]);  // ready for the next launch
}

// Workgroup b: slice (b / 8) % KS of group (b % 8) + 8 ((b / 8) / KS), so the
// KS slices of a group run on one XCD (b % 8).
template <int NM, int T, int KS, int BPS, int DP, typename OutT>
__global__ __launch_bounds__(512) void q4k_gemv_splitk_kernel(GemvArgs a, float* __restrict__ part, int* __restrict__ counters) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[splitk_lds_bytes<NM, T, BPS, DP>()];
  __shared__ int s_last;
  const int sidx = (int)blockIdx.x >> 3;
  splitk_slice<NM, T, KS, BPS, DP, OutT>(a, lds, &s_last, part, counters, ((int)blockIdx.x & 7) + 8 * (sidx / KS), sidx % KS);
}


// ----------------------------------------------------------------------------
// Pipelined GEMM (prefill, N a multiple of 256).
//
// Workgroup tile 128 rows x 256 columns, 4 waves; wave w owns columns
// [64w, 64w + 64) (4 column tiles) of all 128 rows (8 row tiles), so every
// weight element is dequantised once per workgroup and each A fragment read
// from LDS feeds 4 column tiles.  K runs in u-steps of v_mfma_f32_16x16x32_f16
// pairs: u-step t = 4 * block + u covers, in every row, elements
// 64g + 8u + [0, 8) (low nibbles, fragment u) and 64g + 32 + 8u + [0, 8)
// (high nibbles, fragment 4 + u) of the block, for lane groups g.
//  - A: the activations, staged in the GEMM order (gemm_frag_offset: one
//    contiguous 16 KB run per (row block, u-step)), stream through a
//    5-slot LDS ring shared by the 4 waves (16 KB per u-step: 8 row tiles
//    x 2 fragments), loaded with global_load_lds_dwordx4 four u-steps ahead;
//    one barrier per u-step.
//  - B: each wave streams the tile-blocks of its 4 column tiles through a
//    private 2-block LDS ring (one block ahead) and dequantises in
//    registers to h(d*sc*q - dmin*m), the fp32 expression rounded to fp16
//    once (the reference's prefill tile value, quant_linear.metal:43,45).
// Loads: per u-step a wave issues its 4 fragments of A(t + 4) and, at the
// first u-step of a block, the 4 tile-blocks (12 loads) of the next block,
// one fragment (and one tile-block) per column group so that the load
// issue is spread over the step.
// ----------------------------------------------------------------------------
constexpr int kG2M = 128, kG2N = 256, kG2AS = 5, kG2AD = 4;  // A ring slots, A distance
// Time of one 128-column tile (two column tiles per wave) in tenths of a
// 256-column tile's, for the choice between the two tilings.
constexpr int kGemmNarrowTileTime = 6;
constexpr int kG2ASlot = 16 * 1024;                    // 8 row tiles x 2 fragments x 1 KB
constexpr int kG2BWave = 2 * 4 * kTileBlockBytes;      // per wave: 2 blocks x 4 tile-blocks

// Epilogues of a wave's 128-row tile.  The accumulators hold one column per
// lane (4-byte pieces of 16 columns): stored as they are, the residual or gate
// (aux) came in pieces of 32 or 64 bytes whose latency showed once per row
// tile.  Each row tile therefore passes through the wave's own LDS (its B ring,
// idle once its loads have landed: no barrier) and leaves as 4 consecutive
// columns per lane, and the aux of a whole batch of row tiles is loaded, 4
// columns per lane, before the first of them is stored.  N = 12288, K = 4096,
// post 1, before and after: fp16 Q8_0 M = 1531 215 -> 184 us, M = 2048 270 ->
// 231, Q6_K M = 2048 291 -> 249, Q4_K 256 -> 215, IQ4_XS 287 -> 247; fp32 Q8_0
// 245 -> 233, Q6_K 263 -> 249 and, with six column tiles, Q4_K at M = 1531 223
// -> 200, at M = 2048 242 -> 225.
constexpr int kEpiLd(int cols) {
  return cols + 4;  // floats per LDS row: the two row halves of a write fall in different banks
}

template <typename OutT>
struct Quad;
template <>
struct Quad<float> {
  typedef f4_t type;
};
template <>
struct Quad<_Float16> {
  typedef h4_t type;
};

// Four consecutive outputs (or aux values); vec: the pointer is aligned to them.
template <typename OutT>
__device__ __forceinline__ typename Quad<OutT>::type load_quad(const OutT* p, bool vec) {
  typedef typename Quad<OutT>::type Q;
  if (vec)
    return *reinterpret_cast<const Q*>(p);
  return Q{p[0], p[1], p[2], p[3]};
}

template <typename OutT>
__device__ __forceinline__ void store_quad(OutT* p, typename Quad<OutT>::type v, bool vec) {
  if (vec) {
    *reinterpret_cast<typename Quad<OutT>::type*>(p) = v;
  } else {
    p[0] = v[0];
    p[1] = v[1];
    p[2] = v[2];
    p[3] = v[3];
  }
}

// LDS written by some lanes of a wave and read by others: the wave's LDS
// accesses execute in order, and the fences keep the compiler from moving them
// across this point (they emit no instruction at wavefront scope).
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// `value(rt, c, v)` forms the output (before aux) of accumulator element v of
// row tile rt and output column tile c (of NC, nct of them inside n); wl is
// wave-private LDS of at least 16 kEpiLd(16 NC) floats.
template <typename OutT, int POST, int NC, int BR, typename F>
__device__ __forceinline__ void gemm2_flush(const GemmArgs& a, float* wl, int mt0, int ct0, int lane, int nct, F value) {
  typedef typename Quad<OutT>::type Q;
  constexpr int LD = kEpiLd(16 * NC), LPR = 4 * NC, RPP = 64 / LPR, NP = (16 + RPP - 1) / RPP;  // lanes per row, rows per pass, passes
  static_assert(8 % BR == 0, "batches of row tiles");
  asm volatile("" : "+v"(lane));  // nothing of the epilogue is formed ahead of the K loop, beside its registers
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  const int g = lane >> 4, col = lane & 15;
  const int lr = lane / LPR, lc = lane % LPR;
  const bool live = lr < RPP && (lc >> 2) < nct;
  const size_t col0 = (size_t)ct0 * 16 + 4 * lc;
  const bool vec = ((reinterpret_cast<uintptr_t>(y) | (POST ? reinterpret_cast<uintptr_t>(aux) : 0)) & (4 * sizeof(OutT) - 1)) == 0;
#pragma unroll
  for (int b = 0; b < 8; b += BR) {
    Q av[POST ? BR : 1][NP];
    if constexpr (POST != 0) {
#pragma unroll
      for (int r = 0; r < BR; ++r)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          const int lrow = p * RPP + lr, row = (mt0 + b + r) * 16 + lrow;
          av[r][p] = Q{};
          if (live && lrow < 16 && row < a.m)
            av[r][p] = load_quad(aux + (size_t)row * a.n + col0, vec);
        }
    }
#pragma unroll
    for (int r = 0; r < BR; ++r) {
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int c = 0; c < NC; ++c)
          wl[(4 * g + v) * LD + 16 * c + col] = value(b + r, c, v);
      wave_order();
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int lrow = p * RPP + lr, row = (mt0 + b + r) * 16 + lrow;
        if (live && lrow < 16 && row < a.m) {
          const f4_t t = *reinterpret_cast<const f4_t*>(wl + lrow * LD + 4 * lc);
          Q o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float out = t[e];
            if constexpr (POST == 1)
              out += (float)av[r][p][e];
            if constexpr (POST == 2)
              out *= silu((float)av[r][p][e]);
            // The fp32 value is formed before any conversion to fp16: fused
            // into the conversion (v_fma_mix) the product would round once
            // instead of twice, as the reference's half(silu(g) * u) does.
            asm("" : "+v"(out));
            o[e] = (OutT)out;
          }
          store_quad(y + (size_t)row * a.n + col0, o, vec);
        }
      }
      wave_order();
    }
  }
}

// Row tiles whose aux is loaded together: as many as the registers hold.  Beside
// six column tiles' accumulators that is 16 registers, two column tiles of two
// (fp32) or four row tiles (N = 12288, K = 4096, M = 2048, post 1: Q4_K fp32 224
// us, fp16 215, against 241 and 231 for one row tile of three columns).
template <typename OutT, int CT>
constexpr int epi_batch() {
  return CT > 4 ? 8 / (int)sizeof(OutT) : CT * sizeof(OutT) <= 16 ? 8 : 4;
}

template <typename OutT, int POST, int CT>
__device__ __forceinline__ void gemm2_epilogue(const GemmArgs& a, const f4_t (&acc)[8][CT], int mt0, int ct0, int lane, int nct, float* wl) {
  // The tile's 128 row scales behind the transposing buffer (the staging
  // buffers cover whole 128-row tiles, so the loads stay in bounds).
  float* const lrs = wl + 16 * kEpiLd(16 * CT);
  *reinterpret_cast<float2*>(lrs + 2 * lane) = *reinterpret_cast<const float2*>(a.rowscale + mt0 * 16 + 2 * lane);
  wave_order();
  const int g = lane >> 4;
  if constexpr (POST == 0) {
    // Nothing to wait for: the pieces of 16 columns leave as they are (through
    // LDS N = 12288, M = 2048 took 2 to 12 us more).
    OutT* y = reinterpret_cast<OutT*>(a.y);
    const size_t col0 = (size_t)ct0 * 16 + (lane & 15);
#pragma unroll
    for (int rt = 0; rt < 8; ++rt) {
      const f4_t rs = *reinterpret_cast<const f4_t*>(lrs + 16 * rt + 4 * g);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = (mt0 + rt) * 16 + 4 * g + v;
        if (row >= a.m)
          continue;
#pragma unroll
        for (int c = 0; c < CT; ++c)
          if (c < nct)
            store_elem(y, (size_t)row * a.n + col0 + 16 * c, acc[rt][c][v] * rs[v]);
      }
    }
  } else {
    constexpr int NC = CT > 4 ? 2 : CT;
#pragma unroll
    for (int c0 = 0; c0 < CT; c0 += NC)
      gemm2_flush<OutT, POST, NC, epi_batch<OutT, CT>()>(a, wl, mt0, ct0 + c0, lane, nct - c0, [&](int rt, int c, int v) {
        const float t = acc[rt][c0 + c][v] * lrs[16 * rt + 4 * g + v];
        return sizeof(OutT) == 2 ? round_half(t) : t;
      });
  }
}

// The gated GEMM's wave tile of 128 rows and CT / 2 output column tiles: the
// gate tiles (columns 0 .. CT / 2 - 1 of acc) and the up tiles (the rest) of
// the same output column tiles combine as in the two-call form: SiLU(gate) *
// up, each of gate and up first unscaled and, for fp16 outputs, rounded to
// fp16 (the gate value the first call stores, the up value the second call's
// epilogue forms).  nct of the output tiles lie inside n.
template <typename OutT, int CT>
__device__ __forceinline__ void gemm2_epilogue_gated(const GemmArgs& a, const f4_t (&acc)[8][CT], int mt0, int ct0, int lane, int nct, float* wl) {
  constexpr int H = CT / 2;  // output tiles: gate columns 0 .. H - 1, up columns H .. CT - 1
  float* const lrs = wl + 16 * kEpiLd(16 * H);
  *reinterpret_cast<float2*>(lrs + 2 * lane) = *reinterpret_cast<const float2*>(a.rowscale + mt0 * 16 + 2 * lane);
  wave_order();
  const int g = lane >> 4;
  gemm2_flush<OutT, 0, H, 8>(a, wl, mt0, ct0, lane, nct, [&](int rt, int c, int v) {
    const float rs = lrs[16 * rt + 4 * g + v];
    float gv = acc[rt][c][v] * rs, uv = acc[rt][H + c][v] * rs;
    if (sizeof(OutT) == 2) {
      gv = round_half(gv);
      uv = round_half(uv);
    }
    return silu(gv) * uv;
  });
}

// Tile order of the persistent GEMMs.  Workgroup b runs on XCD b % 8 (the
// dispatcher deals workgroups to the eight XCDs in turn).  In the plain order
// tile t = b + i * grid has column block t % tiles_x, so an XCD owns whole
// column blocks and streams the A operand of every row block.  With rg > 0
// the tile grid is cut into 8 rectangles of tiles_y / rg row blocks by
// tiles_x / (8 / rg) column blocks, one per XCD, and the XCD's workgroups
// take its tiles column by column, so that the tiles running together on one
// XCD share the A of a few row blocks and the B of a few column blocks in
// that XCD's L2.
struct TileMap {
  int tiles_x, tiles;  // column blocks, all tiles
  int rg;              // 0: plain order; else row groups (8 / rg column groups)
  int rows, cols;      // rectangle of one XCD (rg > 0)
};

__device__ __forceinline__ int tile_count(const TileMap& m) {
  if (m.rg == 0)
    return ((int)blockIdx.x < m.tiles) ? (m.tiles - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
  const int per = (int)gridDim.x >> 3, j = (int)blockIdx.x >> 3;
  const int rect = m.rows * m.cols;
  return j < rect ? (rect - 1 - j) / per + 1 : 0;
}

// The i-th tile of this workgroup as (column block, row block).
__device__ __forceinline__ void tile_at(const TileMap& m, int i, int& bx, int& by) {
  if (m.rg == 0) {
    const int t = (int)blockIdx.x + i * (int)gridDim.x;
    bx = t % m.tiles_x;
    by = t / m.tiles_x;
    return;
  }
  const int x = (int)blockIdx.x & 7, per = (int)gridDim.x >> 3;
  const int l = ((int)blockIdx.x >> 3) + i * per;
  const int cg = 8 / m.rg;
  by = (x / cg) * m.rows + l % m.rows;
  bx = (x % cg) * m.cols + l / m.rows;
}

// One 128 x 256 output tile (column block bx, row block by).  Column tiles
// at or past ntiles = n / 16 (a last, partial column block) load the last
// column tile (in bounds) and store nothing.  GATED: the workgroup's 128
// output columns of the gated GEMM; wave w takes output column tiles
// ct0 = 8 bx + 2 w and ct0 + 1, whose gate tiles are its B columns 0, 1 and
// whose up tiles (a.wu) are its columns 2, 3.
template <typename OutT, bool GATED, bool SPLIT>
__device__ __forceinline__ void gemm2_tile(const GemmArgs& a, uint8_t* lds, int bx, int by, int ntiles, int kb0, int nbr, int item,
                                           int* s_last) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  // Blocks [kb0, kb0 + nbr) of K (all of them unless SPLIT); u-steps and
  // ring positions count from kb0.
  const int nb = a.nb, steps = 4 * nbr;
  const int mt0 = by * (kG2M / 16);                         // first row tile
  const int ct0 = GATED ? bx * 8 + 2 * wave : bx * (kG2N / 16) + 4 * wave;  // this wave's first column tile
  const uint32_t aring = lds_addr(lds);
  uint8_t* const bring = lds + kG2AS * kG2ASlot + wave * kG2BWave;
  const uint32_t bring0 = lds_addr(bring);
  const uint32_t voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;
  const _Float16* const xh = a.xh;

  // A(t, i): fragment i of this wave's 4 (of the 16) fragments of u-step t
  // (clamped to the last u-step past the end).
  auto issue_a = [&](int t, int i) {
    const int tc = t < steps ? t : steps - 1;
    const int b = kb0 + (tc >> 2), u = tc & 3;
    const int f = 4 * wave + i;
    const _Float16* src = xh + ((((size_t)by * nb + b) * 4 + u) * 16 + f) * 512;
    const uint32_t l = __builtin_amdgcn_readfirstlane(aring + (uint32_t)(t % kG2AS) * kG2ASlot + (uint32_t)f * 1024);
    lds_dma16<0>(uniform_ptr(reinterpret_cast<const uint8_t*>(src)), voff16, l);
  };
  // B(blk, c): tile-block c of block blk (clamped) into ring half blk & 1.
  auto issue_b = [&](int blk, int c) {
    const int bc = kb0 + (blk < nbr ? blk : nbr - 1);
    const int cc = GATED ? ct0 + (c & 1) : ct0 + c;
    const int ct = cc < ntiles ? cc : ntiles - 1;
    const uint8_t* const wm = GATED && c >= 2 ? a.wu : a.w;
    const uint8_t* src = uniform_ptr(wm + ((size_t)ct * nb + bc) * kTileBlockBytes);
    const uint32_t l = __builtin_amdgcn_readfirstlane(bring0 + (uint32_t)((blk & 1) * 4 + c) * kTileBlockBytes);
    lds_dma16<0>(src, voff16, l);
    lds_dma16<kSlabBytes>(src, voff16, l);
    lds_dma4<kHeaderOffset>(src, voff4, l);
  };

  // Block constants of the 4 column tiles, in fp32, from the 4 headers (this
  // lane's column) of one block: for sub-block 2g (low nibbles) d * sc * 2^24
  // and -dmin * m, for sub-block 2g + 1 (high nibbles) d * sc * 2^20 and
  // -dmin * m.  All are exact in fp32 (11-bit d times a 6-bit field, times a
  // power of two).
  float dsl[4], csl[4], dsh[4], csh[4];
  auto block_const = [&](int c, const u4_t& hd) {
    uint32_t p0, p1;
    scale_min_packed(hd, g, p0, p1);
    const float d = half_bits_to_float(hd.x & 0xffffu), dmin = half_bits_to_float(hd.x >> 16);
    dsl[c] = d * (float)(p0 & 0xffu) * 0x1p24f;
    csl[c] = -dmin * (float)((p0 >> 16) & 0xffu);
    dsh[c] = d * (float)(p1 & 0xffu) * 0x1p20f;
    csh[c] = -dmin * (float)((p1 >> 16) & 0xffu);
  };
  // B fragments of column tile c from its two raw words (words 2(u & 1),
  // 2(u & 1) + 1 of slab u / 2 for u-step u), with the block constants: the
  // reference's prefill tile value h(d * sc * q - dmin * m), formed in fp32
  // and rounded to fp16 once (quant_linear.metal:43,45), bit for bit.
  // w & 0x000F000F puts two low nibbles into the low bits of two fp16
  // halves: the denormals q * 2^-24 (w & 0x00F000F0: 16 q * 2^-24 for two
  // high nibbles).  One v_fma_mix_f32 per weight, which takes fp16 denormal
  // sources at their exact value, forms q * (d * sc * 2^24) - dmin * m (2^20
  // for the high nibbles) with the product exact and one rounding to fp32,
  // and one v_cvt_pk_f16_f32 per pair rounds to fp16.  The empty asm keeps
  // the fp32 results apart from the conversion: fused, they become
  // v_fma_mixlo/mixhi_f16 pairs writing the two halves of one register, a
  // dependent chain that measured 6 % slower.  The nibble masks live in
  // registers, as plain values that the scheduler sees as vector ALU work.
  uint32_t m_lo = 0x000F000Fu, m_hi = 0x00F000F0u;
  asm volatile("" : "+v"(m_lo), "+v"(m_hi));
  auto dequant_words = [&](int c, uint2 wv, h8_t& blo, h8_t& bhi) {
    const uint32_t lw[4] = {wv.x, wv.x >> 8, wv.y, wv.y >> 8};
    u4_t lo, hi;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const h2_t ql = as_h2(lw[e] & m_lo);
      const h2_t qh = as_h2(lw[e] & m_hi);
      float a0 = __builtin_fmaf((float)ql[0], dsl[c], csl[c]), a1 = __builtin_fmaf((float)ql[1], dsl[c], csl[c]);
      float b0 = __builtin_fmaf((float)qh[0], dsh[c], csh[c]), b1 = __builtin_fmaf((float)qh[1], dsh[c], csh[c]);
      asm("" : "+v"(a0), "+v"(a1), "+v"(b0), "+v"(b1));
      lo[e] = as_u32(h2_t{(_Float16)a0, (_Float16)a1});
      hi[e] = as_u32(h2_t{(_Float16)b0, (_Float16)b1});
    }
    blo = __builtin_bit_cast(h8_t, lo);
    bhi = __builtin_bit_cast(h8_t, hi);
  };

  // Accumulators: 32 MFMA tiles, zeroed and pinned to AGPRs (the loop-carried
  // values then stay in AGPRs instead of being copied through VGPRs).
  f4_t acc[8][4];
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      acc[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[rt][c]));
    }

#pragma unroll
  for (int c = 0; c < 4; ++c)
    issue_b(0, c);
#pragma unroll
  for (int t = 0; t < kG2AD; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      issue_a(t, i);
  // B(0) and A(0) landed: A(1..3) (12 loads) were issued after them.
  asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  // Dequantisation runs one column behind the MFMAs: column c of u-step
  // t + 1 is dequantised under the MFMAs of column c + 1 of u-step t, and
  // column 3 under those of column 0 of u-step t + 1 (from words kept in
  // wv3), so that every column's MFMAs have vector work to cover.  At the
  // last u-step of a block the next block's constants of column c are
  // computed under column c's MFMAs, after column 3 of the current u-step
  // (old constants) was dequantised and before column c's first use.
  h8_t bclo[4], bchi[4];  // dequantised B fragments of the current u-step
  uint2 wv3;              // raw words of column 3 for the current u-step
  {
    u4_t hd[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      hd[c] = *reinterpret_cast<const u4_t*>(bring + c * kTileBlockBytes + kHeaderOffset + 16 * col);
      block_const(c, hd[c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
      dequant_words(c, *reinterpret_cast<const uint2*>(bring + c * kTileBlockBytes + 16 * lane), bclo[c], bchi[c]);
    wv3 = *reinterpret_cast<const uint2*>(bring + 3 * kTileBlockBytes + 16 * lane);
  }
  // A in the loop: this wave's 4 fragments of u-step t are 4 consecutive KB
  // at xa + 16 KB * t of the staging and at 4 KB * wave of ring slot t % 5;
  // fragment i is the instruction offset 1 KB * i.  The ring addresses of
  // the slot read (ar) and written (aw) roll instead of being recomputed.
  const uint8_t* const xa = reinterpret_cast<const uint8_t*>(xh) + ((size_t)by * nb * 64 + (size_t)kb0 * 64 + 4 * wave) * 1024;
  const uint32_t aend = aring + kG2AS * kG2ASlot;
  uint32_t ar = aring, aw = aring + kG2AD * kG2ASlot + 4096u * (uint32_t)wave;
  for (int blk = 0; blk < nbr; ++blk) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * blk + u;
      const int ta = t + kG2AD < steps ? t + kG2AD : steps - 1;
      const uint8_t* const asrc = uniform_ptr(xa + (size_t)ta * 16384);
      // Own loads issued after A(t) (during u-steps t - 4 .. t - 1, in the
      // order of the column groups below): 15 at u = 0 (the 3 of B tile 3
      // that follow A(t) at u-step t - 4, then 3 x 4), 24 at u = 1, 2, 3.
      // At u = 3 B(blk + 1), issued at u-step t - 3 after A(t), must have
      // landed too: 8 loads follow it.  (A(0) is waited for in the prologue.)
      if (u == 0)
        asm volatile("s_waitcnt vmcnt(15)" ::: "memory");
      else if (u == 3)
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else
        asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
      __syncthreads();  // A(t) of every wave landed; u-step t - 1 fully read
      __builtin_amdgcn_sched_barrier(0);
      // LDS reads of the step: the 16 A fragments of u-step t ([row tile][low,
      // high]), then (u = 3) the headers of the next block, then the raw B
      // words of u-step t + 1.  At u = 3 that is the next block, whose B
      // landed before A(t) (issued at u = 0).
      const int bn = u == 3 ? blk + 1 : blk, un = (u + 1) & 3;
      const uint8_t* aslot = lds + (ar - aring);
      h8_t af[16];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        af[i] = *reinterpret_cast<const h8_t*>(aslot + i * 1024 + 16 * lane);
      const uint8_t* bslot = bring + (size_t)((bn & 1) * 4) * kTileBlockBytes;
      u4_t hd[4];
      if (u == 3) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          hd[c] = *reinterpret_cast<const u4_t*>(bslot + c * kTileBlockBytes + kHeaderOffset + 16 * col);
      }
      uint2 wv[4];
#pragma unroll
      for (int c = 0; c < 4; ++c)
        wv[c] = *reinterpret_cast<const uint2*>(bslot + c * kTileBlockBytes + (un >> 1) * kSlabBytes + 16 * lane + 8 * (un & 1));
      __builtin_amdgcn_sched_barrier(0);
      // Column tile c: its 16 MFMAs of u-step t, then its B fragments of
      // u-step t + 1 replace the ones just consumed.  The dequantisation of
      // column c runs under the MFMAs of column c + 1.
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c == 0)
          dequant_words(3, wv3, bclo[3], bchi[3]);  // column 3 of this u-step
        // Low-nibble fragments over the 8 row tiles, then the high ones:
        // neighbouring MFMAs are independent.
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt], bclo[c], acc[rt][c], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt + 1], bchi[c], acc[rt][c], 0, 0, 0);
        if (u == 3)
          block_const(c, hd[c]);
        if (c > 0)
          dequant_words(c - 1, wv[c - 1], bclo[c - 1], bchi[c - 1]);
        // The loads of the column group, spread over the step: fragment c
        // of A(t + 4) and, at u = 0, tile-block c of B(blk + 1).
        if (c == 0)
          lds_dma16<0>(asrc, voff16, aw);
        else if (c == 1)
          lds_dma16<1024>(asrc, voff16, aw);
        else if (c == 2)
          lds_dma16<2048>(asrc, voff16, aw);
        else
          lds_dma16<3072>(asrc, voff16, aw);
        if (u == 0)
          issue_b(blk + 1, c);
      }
      wv3 = wv[3];
      ar = ar + kG2ASlot == aend ? aring : ar + kG2ASlot;
      aw = aw + kG2ASlot >= aend ? aw + kG2ASlot - kG2AS * kG2ASlot : aw + kG2ASlot;
      // Schedule of the step: the LDS reads first, then each MFMA followed
      // by a share of the vector work (the next step's dequantisation, and
      // at u = 3 the next block's constants), so that no vector work is
      // left after the last MFMA.
      if (u == 3) {
        __builtin_amdgcn_sched_group_barrier(0x100, 24, 0);
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
        }
      } else {
        __builtin_amdgcn_sched_group_barrier(0x100, 20, 0);
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // Pin the accumulators to AGPRs at the loop exit, so that the epilogue's
  // element reads do not pull copies of them into the loop.
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      asm volatile("" : "+a"(acc[rt][c]));

  if constexpr (SPLIT) {
    // Two K-segments per tile (items 2 tile, 2 tile + 1).  A segment that
    // finds the other already arrived (its accumulators in memory and the
    // counter at 1) stores nothing; otherwise it stores its accumulators
    // (written through to memory), counts its arrival, and the second to
    // arrive adds the other's and runs the epilogue.  fp32 addition
    // commutes, so the result does not depend on which segment is last.
    constexpr size_t kWaveFloats = 32 * 64 * 4;
    int* const ctr = &a.counters[item >> 1];
    if (tid == 0)
      *s_last = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 0;
    __syncthreads();
    if (!*s_last) {
      float* const mine = a.part + ((size_t)item * 4 + wave) * kWaveFloats + 4 * lane;
#pragma unroll
      for (int rt = 0; rt < 8; ++rt)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          store_coherent4(mine + (rt * 4 + c) * 256, acc[rt][c]);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0)
        *s_last = count_arrival(ctr) == 1;
      __syncthreads();
      if (!*s_last)
        return;
    }
    const float* const other = a.part + ((size_t)(item ^ 1) * 4 + wave) * kWaveFloats + 4 * lane;
    f4_t pv[8][4];
#pragma unroll
    for (int rt = 0; rt < 8; ++rt)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        pv[rt][c] = load_coherent4(other + (rt * 4 + c) * 256);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
    for (int rt = 0; rt < 8; ++rt)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        hold(pv[rt][c]);
        acc[rt][c] += pv[rt][c];
      }
    if (tid == 0)
      reset_counter(ctr);  // ready for the next launch
  }

  // One straight-line epilogue per post code.
  float* const elds = reinterpret_cast<float*>(bring);  // this wave's B ring: its loads have landed
  if constexpr (GATED) {
    const int nct2 = ntiles - ct0 >= 2 ? 2 : ntiles - ct0 > 0 ? ntiles - ct0 : 0;
    gemm2_epilogue_gated<OutT>(a, acc, mt0, ct0, lane, nct2, elds);
    return;
  }
  const int nct = ntiles - ct0 >= 4 ? 4 : ntiles - ct0 > 0 ? ntiles - ct0 : 0;
  if (a.post == 0)
    gemm2_epilogue<OutT, 0>(a, acc, mt0, ct0, lane, nct, elds);
  else if (a.post == 1)
    gemm2_epilogue<OutT, 1>(a, acc, mt0, ct0, lane, nct, elds);
  else
    gemm2_epilogue<OutT, 2>(a, acc, mt0, ct0, lane, nct, elds);
}

// Persistent launch: workgroup b takes its tiles in the order of the tile
// map.  Consecutive tiles of a workgroup reuse its LDS rings; a barrier
// separates the last reads of one tile from the first loads of the next.
// SPLIT: items 2 t and 2 t + 1 are the two K-segments of tile t (plain tile
// order): with a.split_q > 0 workgroup t < tiles takes segment 0 of tile t
// and workgroup tiles + r segments 1 of tiles r, r + R, ... (R workgroups
// past the tiles), else the workgroups take the items in turn.
template <typename OutT, bool GATED, bool SPLIT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void q4k_gemm2_kernel(GemmArgs a, TileMap map) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[kG2AS * kG2ASlot + 4 * kG2BWave];
  __shared__ int s_last;
  if constexpr (SPLIT) {
    // This workgroup's items: first, first + step, ... below 2 x tiles (one
    // call site of the tile body, which is inlined).
    const int b = a.split_b, tiles = map.tiles, g = (int)blockIdx.x;
    int first = g, step = (int)gridDim.x;
    if (a.split_q > 0) {
      first = g < tiles ? 2 * g : 2 * (g - tiles) + 1;
      step = g < tiles ? 2 * tiles : 2 * ((int)gridDim.x - tiles);
    }
    for (int it = first; it < 2 * tiles; it += step) {
      if (it != first)
        __syncthreads();
      const int tile = it >> 1, ks = it & 1;
      gemm2_tile<OutT, GATED, true>(a, lds, tile % map.tiles_x, tile / map.tiles_x, a.n / 16, ks ? b : 0, ks ? a.nb - b : b, it, &s_last);
    }
  } else {
    const int count = tile_count(map);
    for (int i = 0; i < count; ++i) {
      if (i > 0)
        __syncthreads();
      int bx, by;
      tile_at(map, i, bx, by);
      gemm2_tile<OutT, GATED, false>(a, lds, bx, by, a.n / 16, 0, a.nb, 0, &s_last);
    }
  }
}

// ----------------------------------------------------------------------------
// Measured MFMA ceiling: the GEMM's instruction (v_mfma_f32_16x16x32_f16) back
// to back, 32 independent accumulators per wave, one wave per SIMD, operands
// in registers -- the rate a kernel of this instruction can reach on the box
// (clock under a dense MFMA load included).  The result is stored so that
// nothing is dead; its value is meaningless.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mfma_ceiling_kernel(float* out, int iters) {
  const int lane = threadIdx.x & 63;
  f4_t acc[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    acc[i] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
    asm volatile("" : "+a"(acc[i]));
  }
  h8_t a0, a1, b0, b1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    a0[i] = (_Float16)(0.001f * (float)(lane + i));
    a1[i] = (_Float16)(0.002f * (float)(lane - i));
    b0[i] = (_Float16)(0.003f * (float)(i - lane));
    b1[i] = (_Float16)(0.004f * (float)(i + 1));
  }
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 32; ++i)
      acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(i & 1 ? a1 : a0, i & 2 ? b1 : b0, acc[i], 0, 0, 0);
  }
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    asm volatile("" : "+a"(acc[i]));
    sum += acc[i][0] + acc[i][3];
  }
  out[(size_t)blockIdx.x * 256 + threadIdx.x] = sum;
}

// ----------------------------------------------------------------------------
// Measured streaming-read ceiling: a plain read of n16 16-byte words with
// non-temporal loads (as the GEMVs stream their weights), up to four in
// flight per lane, over the grid the caller gives.  The xor of each lane's words is stored only
// if it hits a fixed value, which keeps the loads alive without a store
// stream of its own.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void stream_read_kernel(const u4_t* __restrict__ p, size_t n16, uint32_t* out) {
  const size_t stride = (size_t)gridDim.x * 256;
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  uint32_t acc = 0;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const u4_t a = __builtin_nontemporal_load(p + i), b = __builtin_nontemporal_load(p + i + stride);
    const u4_t c = __builtin_nontemporal_load(p + i + 2 * stride), d = __builtin_nontemporal_load(p + i + 3 * stride);
    acc ^= (a.x ^ a.y ^ a.z ^ a.w) ^ (b.x ^ b.y ^ b.z ^ b.w) ^ (c.x ^ c.y ^ c.z ^ c.w) ^ (d.x ^ d.y ^ d.z ^ d.w);
  }
  for (; i < n16; i += stride) {
    const u4_t a = __builtin_nontemporal_load(p + i);
    acc ^= a.x ^ a.y ^ a.z ^ a.w;
  }
  if (acc == 0x9E3779B9u)
    out[blockIdx.x] = acc;
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, uint32_t v, uint32_t n) {
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    p[i] = v;
}

// ----------------------------------------------------------------------------
// Row gather and device re-layout.
// ----------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void gather_rows_kernel(const T* __restrict__ x, T* __restrict__ out, int k, GatherIndex idx) {
  const int r = blockIdx.x;
  const T* src = x + (size_t)idx.src[r] * k;
  T* dst = out + (size_t)r * k;
  for (int i = threadIdx.x; i < k; i += 256)
    dst[i] = src[i];
}


// ----------------------------------------------------------------------------
// Token embedding (quant_linear.metal:572-591, embedding_q4_k): output row t
// is row ids[t] of a Q4_K table kept in the tiled device layout, dequantised.
// One 256-thread workgroup per (block, row); thread e forms element e of the
// block from its byte (e / 64) * 32 + e % 32 (high nibble when e & 32) and
// sub-block e / 32, as (d * sc) * q - dmin * m with each product and the
// difference rounded once (no contraction; the CPU oracle's order).  Ids
// outside [0, n) give a zero row.
// ----------------------------------------------------------------------------
template <typename OutT>
__device__ __forceinline__ void embedding_elem(const uint8_t* __restrict__ w, int id, OutT* __restrict__ y, int n, int nb, int t, int b, int e) {
#pragma clang fp contract(off)
  float v = 0.0f;
  if (id >= 0 && id < n) {
    const int i = id & 15;
    const uint8_t* tb = w + ((size_t)(id >> 4) * nb + b) * kTileBlockBytes;
    const uint8_t* hd = tb + kHeaderOffset + 16 * i;
    const uint8_t* q12 = hd + 4;
    // 6-bit scale and min of sub-block j (quant_linear.metal:12-20).
    const int j = e >> 5;
    uint32_t sc, mn;
    if (j < 4) {
      sc = q12[j] & 63u;
      mn = q12[j + 4] & 63u;
    } else {
      sc = (q12[j + 4] & 15u) | ((uint32_t)(q12[j - 4] >> 6) << 4);
      mn = (uint32_t)(q12[j + 4] >> 4) | ((uint32_t)(q12[j] >> 6) << 4);
    }
    // Quant byte p of the GGUF record: lane 16 (p / 32) + i of slab (p / 16) & 1,
    // word (p / 4) & 3, with the word's two middle bytes swapped.
    const int p = (e >> 6) * 32 + (e & 31), o = p & 31, bw = o & 3;
    const int sbw = bw == 1 ? 2 : bw == 2 ? 1 : bw;
    const uint8_t qb = tb[(o >> 4) * kSlabBytes + 16 * (16 * (p >> 5) + i) + (o & 12) + sbw];
    const uint32_t q = (e & 32) ? (uint32_t)(qb >> 4) : (uint32_t)(qb & 15);
    const float d = half_bits_to_float((uint32_t)hd[0] | ((uint32_t)hd[1] << 8));
    const float dmin = half_bits_to_float((uint32_t)hd[2] | ((uint32_t)hd[3] << 8));
    const float dsc = d * (float)sc;
    const float val = dsc * (float)q;
    const float mterm = dmin * (float)mn;
    v = val - mterm;
  }
  store_elem(y, (size_t)t * nb * 256 + (size_t)b * 256 + e, v);
}

template <typename OutT>
__global__ __launch_bounds__(256) void embedding_kernel(const uint8_t* __restrict__ w, const int32_t* __restrict__ ids, OutT* __restrict__ y, int n,
                                                        int nb) {
  embedding_elem(w, ids[blockIdx.y], y, n, nb, (int)blockIdx.y, (int)blockIdx.x, (int)threadIdx.x);
}

// The same over a packed batch, each row's token resolved in the kernel
// (quant_linear.metal:577-584 mode 0 with queryRow, batch.hpp:19-23): row t
// belongs to the first query q with t < start[q] + count[q] and takes the
// request buffer's token tokens[slot[q] * capacity + position[q] + t -
// start[q]].
template <typename OutT>
__global__ __launch_bounds__(256) void embedding_batch_kernel(const uint8_t* __restrict__ w, const int32_t* __restrict__ tokens, OutT* __restrict__ y,
                                                              int n, int nb, EmbedQueries qs) {
  const uint32_t t = blockIdx.y;
  uint32_t q = 0;
  while (q + 1 < qs.n && t >= qs.start[q] + qs.count[q])
    ++q;
  const int id = tokens[(size_t)qs.slot[q] * qs.capacity + qs.position[q] + (t - qs.start[q])];
  embedding_elem(w, id, y, n, nb, (int)t, (int)blockIdx.x, (int)threadIdx.x);
}

// ----------------------------------------------------------------------------
// RMS norm (native_ops.metal:6-40): y[r] = x[s] * rsqrt(sum(x[s]^2) / k + eps)
// * w, s = idx.src[r] for rms_norm_gather (the LM-head rows, batch.hpp:25-29)
// or s = r.  One 256-thread workgroup per output row; fp32 sum of squares
// (wave shuffle reduction, then across the 4 waves).  Rows of up to
// 256 * kNormRegs elements stay in registers between the two passes (one
// read of x); longer rows are read again.
// ----------------------------------------------------------------------------
constexpr int kNormRegs = 16;

// RMS norm of one row per workgroup of 512 threads, 8 elements (one 16- or
// two 16-byte loads) per thread and chunk, the row in registers between the
// sum of squares and the scaling, against the general form's 16 single-element
// loads per thread (rows of 4096, replayed back to back): 40 fp16 rows 6.1 ->
// 3.3 us, 5 6.0 -> 3.2, 2048 10.2 -> 7.8; fp32 40 rows 5.0 -> 3.4, 2048 13.3 -> 13.5
// (bandwidth either way).
constexpr int kNormChunks = 3;
template <typename T>
__global__ __launch_bounds__(512) void rms_norm8_kernel(const T* __restrict__ x, const float* __restrict__ w, T* y, int k, float eps, GatherIndex idx,
                                                        int gather) {
  const int r = blockIdx.x, tid = threadIdx.x, chunks = k >> 3;
  const T* xr = x + (size_t)(gather ? idx.src[r] : (uint32_t)r) * k;
  float v[kNormChunks][8];
  float ss = 0.0f;
#pragma unroll
  for (int j = 0; j < kNormChunks; ++j) {
    const int c = tid + 512 * j;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[j][i] = 0.0f;
    if (c < chunks)
      load8(xr + (size_t)c * 8, v[j]);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      ss = fmaf(v[j][i], v[j][i], ss);
  }
  float nw[kNormChunks][8];
#pragma unroll
  for (int j = 0; j < kNormChunks; ++j)
    if (tid + 512 * j < chunks)
      load8(w + (size_t)(tid + 512 * j) * 8, nw[j]);
  __shared__ float part[8];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    ss += __shfl_xor(ss, off);
  if ((tid & 63) == 0)
    part[tid >> 6] = ss;
  __syncthreads();
  const float scale = 1.0f / sqrtf(sum8_pairs(part) / (float)k + eps);
  T* yr = y + (size_t)r * k;
#pragma unroll
  for (int j = 0; j < kNormChunks; ++j) {
    const int c = tid + 512 * j;
    if (c < chunks) {
      typedef T t8 __attribute__((ext_vector_type(8)));
      t8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        o[i] = (T)((v[j][i] * scale) * nw[j][i]);
      *reinterpret_cast<t8*>(yr + (size_t)c * 8) = o;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void rms_norm_kernel(const T* __restrict__ x, const float* __restrict__ w, T* y, int k, float eps, GatherIndex idx,
                                                       int gather) {
  __shared__ float part[4];
  const int r = blockIdx.x, tid = threadIdx.x;
  const T* xr = x + (size_t)(gather ? idx.src[r] : (uint32_t)r) * k;
  float v[kNormRegs];
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < kNormRegs; ++i) {
    const int d = tid + 256 * i;
    v[i] = d < k ? (float)xr[d] : 0.0f;
    ss = fmaf(v[i], v[i], ss);
  }
  for (int d = tid + 256 * kNormRegs; d < k; d += 256) {
    const float t = (float)xr[d];
    ss = fmaf(t, t, ss);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    ss += __shfl_xor(ss, off);
  if ((tid & 63) == 0)
    part[tid >> 6] = ss;
  __syncthreads();
  const float total = (part[0] + part[1]) + (part[2] + part[3]);
  const float scale = 1.0f / sqrtf(total / (float)k + eps);
  T* yr = y + (size_t)r * k;
#pragma unroll
  for (int i = 0; i < kNormRegs; ++i) {
    const int d = tid + 256 * i;
    if (d < k)
      yr[d] = (T)((v[i] * scale) * w[d]);
  }
  for (int d = tid + 256 * kNormRegs; d < k; d += 256)
    yr[d] = (T)(((float)xr[d] * scale) * w[d]);
}

__device__ __forceinline__ uint32_t swap_middle_bytes(uint32_t v) {
  return (v & 0xff0000ffu) | ((v & 0x0000ff00u) << 8) | ((v & 0x00ff0000u) >> 8);
}

// One workgroup of 64 lanes per tile-block.
__global__ __launch_bounds__(64) void relayout_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t n, uint32_t nb) {
  const size_t tb = blockIdx.x;
  const uint32_t c = (uint32_t)(tb / nb), b = (uint32_t)(tb % nb);
  const int lane = threadIdx.x, i = lane & 15, g = lane >> 4;
  const uint8_t* blk = src + ((size_t)(16 * c + i) * nb + b) * kBlockBytes;
  uint8_t* out = dst + tb * kTileBlockBytes;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint8_t* q = blk + 16 + 32 * g + 16 * h;
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = swap_middle_bytes((uint32_t)q[4 * j] | ((uint32_t)q[4 * j + 1] << 8) | ((uint32_t)q[4 * j + 2] << 16) | ((uint32_t)q[4 * j + 3] << 24));
    *reinterpret_cast<u4_t*>(out + h * kSlabBytes + 16 * lane) = u4_t{w[0], w[1], w[2], w[3]};
  }
  if (g == 0) {
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (uint32_t)blk[4 * j] | ((uint32_t)blk[4 * j + 1] << 8) | ((uint32_t)blk[4 * j + 2] << 16) | ((uint32_t)blk[4 * j + 3] << 24);
    *reinterpret_cast<u4_t*>(out + kHeaderOffset + 16 * i) = u4_t{w[0], w[1], w[2], w[3]};
  }
}

// ----------------------------------------------------------------------------
// The other GGUF types on the same linear() surface: Q6_K (the LM head of real
// files, mixed-type down projections), Q8_0, Q5_K and IQ4_XS
// (quant_linear.metal:50-115 dequant, :329-570 decode GEMVs, :620-662 shapes;
// fused_kernels.metal:80-200).
//
// GEMV for m <= 8 rows (decode, small prefill, LM head) over the decode pack
// of x (hi / lo fp16 rows 0..7 / 8..15, per-(row, block) power-of-two scale;
// the sub-block sums for the Q5_K min term).  A format policy F supplies the
// per-lane registers of one tile-block (U), their loads, and `mac`: the eight
// B operands of v_mfma_f32_16x16x32_f16 in fp16, the MFMAs, and the tile-
// block's contribution scaled into the lane's four accumulator rows:
//   Q6_K   (q - 32) * sc per dword: (w & 0x03F003F0) | 0x6400 = 1024 + 16q for
//          two quants stored at bits 4..9 of each half, one v_pk_fma_f16 with
//          (sc / 16, -96 sc); d * row unscale after the MFMAs.
//   Q8_0   q * d per dword: v_perm_b32 of two biased bytes with 0x64 bytes is
//          1024 + 128 + q; v_pk_add_f16 -1152 leaves q, v_pk_mul_f16 by the
//          record's d (one rounding); row unscale after the MFMAs.
//   Q5_K   the Q4_K nibble decode with the fifth bit or'ed into the fp16 bias
//          (16 for low nibbles, 256 for high ones), q * sc exact (<= 1953), the
//          min term on a 16x16x16 MFMA of the sub-block sums.
//   IQ4_XS codebook lookup of four indices per v_perm_b32 pair (entries 0..7,
//          8..15, selected by bit 3 with v_bfi_b32), biased bytes to fp16 as for
//          Q8_0, one v_pk_fma_f16 with (ls - 32, -1152 (ls - 32)).
// Products above 2048 in magnitude (Q6_K, IQ4_XS) and q * d (Q8_0) are
// rounded once to fp16; the reference's prefill tiles round every dequantised
// weight to fp16 (quant_linear.metal:65,83,98,112).
//
// Workgroup = 8 waves; wave w takes blocks w, w + 8, ...  The persistent form
// (K = 4096, 16 blocks: two per wave) keeps each wave's x fragments in
// registers and streams every item (T column tiles) it owns through one
// register window that runs across item boundaries; partial sums alternate
// between two LDS buffers, one barrier per item.  The other form (any K)
// takes one item per workgroup, double-buffers the next block's x fragments
// and streams its T tile-blocks per block through a window DQ deep.
// ----------------------------------------------------------------------------

template <typename OutT, int W = 8>
__device__ __forceinline__ void typed_epilogue(const GemvArgs& a, const float* part, int t_count, int tile0, int ntiles) {
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  const int tid = threadIdx.x;
  for (int o = tid; o < a.m * 16 * t_count; o += 64 * W) {
    const int row = o / (16 * t_count), c = o % (16 * t_count), t = c >> 4, cc = c & 15;
    if (tile0 + t >= ntiles)
      continue;
    float acc_v = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w)
      acc_v += part[((w * t_count + t) * 8 + row) * 16 + cc];
    if (sizeof(OutT) == 2)
      acc_v = round_half(acc_v);
    const size_t off = (size_t)row * a.n + (size_t)(tile0 + t) * 16 + cc;
    const float out = a.post == 1 ? acc_v + load_elem(aux, off) : a.post == 2 ? silu(load_elem(aux, off)) * acc_v : acc_v;
    store_elem(y, off, out);
  }
}

template <class F, int T, int DQ, typename OutT>
__global__ __launch_bounds__(512) void typed_gemv_kernel(GemvArgs a) {
  constexpr int W = 8;
  static_assert(DQ <= T || T == 1, "window");
  constexpr int D = DQ < T ? DQ : T;
  __shared__ float part[W][T][8][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int nb = a.nb, ntiles = a.n >> 4, tile0 = blockIdx.x * T;
  const size_t tile_bytes = (size_t)nb * F::kTB;
  const int nbw = wave < nb ? (nb - 1 - wave) / W + 1 : 0;

  typename F::U ring[T];
  auto issue = [&](int t, int bi) {
    const int tile = tile0 + t < ntiles ? tile0 + t : ntiles - 1;
    F::load(ring[t], a.w + (size_t)tile * tile_bytes + (size_t)(wave + W * bi) * F::kTB, lane);
  };
  f4_t acc[T];
#pragma unroll
  for (int t = 0; t < T; ++t)
    acc[t] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
  if (nbw > 0) {
    XF xc, xn;
    load_xf<F::kMin>(xc, a.pack, (size_t)wave, lane);
#pragma unroll
    for (int t = 0; t < D; ++t)
      issue(t, 0);
    for (int bi = 0; bi < nbw; ++bi) {
      const bool more = bi + 1 < nbw;
      if (more)
        load_xf<F::kMin>(xn, a.pack, (size_t)(wave + W * (bi + 1)), lane);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        // Take slot t before the window's next issue, which may reuse it.
        const typename F::U cur = ring[t];
        const int tn = t + D;
        if (tn < T)
          issue(tn, bi);
        else if (more)
          issue(tn - T, bi + 1);
        F::mac(cur, xc, lane, acc[t]);
      }
      if (more)
        xc = xn;
    }
  }
  // C row 4g + v: lanes g < 2 add the low parts held 32 lanes up.
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float tot = acc[t][v] + __shfl_xor(acc[t][v], 32);
      if (g < 2)
        part[wave][t][4 * g + v][col] = tot;
    }
  __syncthreads();
  typed_epilogue<OutT>(a, &part[0][0][0][0], T, tile0, ntiles);
}

template <class F, int T, int DQ, int W, typename OutT>
__global__ __launch_bounds__(64 * W) void typed_gemv_persistent_kernel(GemvArgs a, int items) {
  constexpr int BPW = 16 / W, U = BPW * T;
  static_assert(W * BPW == 16 && DQ <= U, "16 blocks; window");
  __shared__ float part[2][W][T][8][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int ntiles = a.n >> 4;
  const size_t tile_bytes = (size_t)(W * BPW) * F::kTB;
  int item = blockIdx.x;
  if (item >= items)
    return;

  XF xf[BPW];
#pragma unroll
  for (int j = 0; j < BPW; ++j)
    load_xf<F::kMin>(xf[j], a.pack, (size_t)(wave + W * j), lane);
  typename F::U ring[U];
  auto issue = [&](int u, int it) {
    const int j = u / T, t = u - j * T;
    const int tile = it * T + t < ntiles ? it * T + t : ntiles - 1;
    F::load(ring[u], a.w + (size_t)tile * tile_bytes + (size_t)(wave + W * j) * F::kTB, lane);
  };
#pragma unroll
  for (int u = 0; u < DQ; ++u)
    issue(u, item);
  for (int it = 0; item < items; ++it, item += gridDim.x) {
    const int next = item + (int)gridDim.x;
    f4_t acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
      acc[t] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = u / T, t = u - j * T;
      const typename F::U cur = ring[u];
      if (u + DQ < U)
        issue(u + DQ, item);
      else if (next < items)
        issue(u + DQ - U, next);
      F::mac(cur, xf[j], lane, acc[t]);
    }
    float(*pb)[T][8][16] = part[it & 1];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float tot = acc[t][v] + __shfl_xor(acc[t][v], 32);
        if (g < 2)
          pb[wave][t][4 * g + v][col] = tot;
      }
    __syncthreads();
    typed_epilogue<OutT, W>(a, &pb[0][0][0][0], T, item * T, ntiles);
  }
}

// ----------------------------------------------------------------------------
// Prefill GEMM for the other weight types (Q5_K, Q6_K, Q8_0, IQ4_XS).
//
// The pipelined GEMM of the Q4_K path with its B operand taken from a policy
// of the type's tile-block (layouts in q4k_internal.h): the same A ring over
// the activations in the GEMM staging order, a private 2-block B ring per
// wave filled by LDS-DMA, and per u-step u the B fragments of MFMA fs = u
// (low) and fs = 4 + u (high) of each column tile dequantised in registers to
// the reference's prefill tile value (quant_linear.metal:49-115): its fp32
// expression rounded once to fp16, bit for bit.
//   Q5_K   h(d*sc*(q + 16h) - dmin*m): q + 16h as an fp16 denormal (as the
//          Q4_K nibbles), then one fp32 fma with d*sc*2^24 and -dmin*m (both
//          exact), the single fp32 rounding of the reference's expression.
//   Q6_K   h(d*sc*(q - 32)): the product has at most 23 significant bits, so
//          fma(64 + q, d*sc, -96 d*sc) is exact.
//   Q8_0   h(d*q): 19 bits; one fp16 multiply rounds the exact product once.
//   IQ4_XS h(d*(ls - 32)*v): 23 bits; fma(1152 + v, dl, -1152 dl) is exact.
// Per type: kCT column tiles per wave and kAS A ring slots (A loaded kAS - 1
// u-steps ahead), so that both rings fit the 160 KB of LDS; kNL DMA loads per
// tile-block; kVPM vector instructions scheduled after each MFMA (measured:
// 2 for Q5_K, Q6_K and Q8_0, 3-5 percent faster than 3 or 4 at M = 2048; 4
// for IQ4_XS).  Column tiles past n (a multiple of 16, not of the
// workgroup's width) load the last tile and store nothing.  Wrappers set
// other widths: Narrow (2 tiles), Mid (3), Six (6, with a 3-slot A ring;
// also the gated Q4_K GEMM, GATED), and TgQ8_0W streams Q8_0's B in half
// tile-blocks so that four tiles fit.
// ----------------------------------------------------------------------------

// Load accounting of the typed GEMM.  A wave issues per u-step its 4 A
// fragments of A(t + kAS - 1) spread over its kCT column groups, each group's
// share followed, at u = 0, by the kNL loads of that column's tile-block of
// the next block.  vmcnt is in order, so A(t) has landed once no more than
// the loads issued after its last fragment are outstanding.
constexpr int tg_mod4(int v) {
  return ((v % 4) + 4) % 4;
}
constexpr int tg_step_loads(int u, int ct, int nl) {
  return 4 + (u == 0 ? ct * nl : 0);
}
// Loads issued after A(t)'s last fragment (issued at u-step t - ad) up to the
// top of u-step t, u = t % 4; at u = 3 also no more than the 8 loads of
// u-steps 1 and 2, which follow the next block's B (issued at u = 0).
constexpr int tg_wait(int u, int ad, int ct, int nl) {
  int n = tg_mod4(u - ad) == 0 ? nl : 0;
  for (int j = 1; j < ad; ++j)
    n += tg_step_loads(tg_mod4(u - j), ct, nl);
  return u == 3 && n > 8 ? 8 : n;
}
// In the first block A(1 .. ad - 1) come from the prologue (after B(0), before
// any u-step): the steady-state wait must not exceed the loads that really
// follow them there.  (A(0) is waited for by the prologue itself.)
constexpr bool tg_first_block_ok(int ad, int ct, int nl) {
  for (int t = 1; t < ad && t < 4; ++t) {
    int after = 4 * (ad - 1 - t);
    for (int s = 0; s < t; ++s)
      after += tg_step_loads(s % 4, ct, nl);
    if (after < tg_wait(t, ad, ct, nl))
      return false;
  }
  return true;
}

template <int N>
__device__ __forceinline__ void vm_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt field");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One 128 x (64 kCT) output tile (column block bx, row block by); ntiles =
// n / 16.  The step structure is the Q4_K GEMM's: the LDS reads of a u-step
// first (the 16 A fragments, at u = 3 the next block's per-column data, the
// raw B words of u-step t + 1), then per column tile its 16 MFMAs with the
// dequantisation of the previous column for u-step t + 1 under them (the
// last column's under the first column of the next u-step).
// GATED: the gated GEMM (SiLU(gate) * up of a.w and a.wu): the wave's
// columns 0 .. CT / 2 - 1 are output column tiles ct0 .. of the gate matrix,
// the others the same tiles of the up matrix; ct0 counts output tiles.
template <class P, typename OutT, bool GATED = false>
__device__ __forceinline__ void typed_gemm_tile(const GemmArgs& a, uint8_t* lds, int bx, int by, int ntiles) {
  constexpr int CT = P::kCT, AS = P::kAS, AD = AS - 1, NL = P::kNL, TB = P::kTB;
  constexpr int OT = GATED ? CT / 2 : CT;  // output column tiles per wave
  static_assert(tg_first_block_ok(AD, CT, NL), "first-block load accounting");
  static_assert(!GATED || CT % 2 == 0, "gate and up tiles in pairs");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = a.nb, steps = 4 * nb;
  const int mt0 = by * (kG2M / 16);
  const int ct0 = bx * (4 * OT) + OT * wave;
  const uint32_t aring = lds_addr(lds);
  uint8_t* const bring = lds + AS * kG2ASlot + wave * (2 * CT * TB);
  const uint32_t bring0 = lds_addr(bring);
  const uint32_t voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;
  // A: this wave's 4 fragments of u-step t are 4 consecutive KB at
  // xa + 16 KB * t of the staging and at 4 KB * wave of ring slot t % AS;
  // fragment i is the instruction offset 1 KB * i.  The ring addresses of
  // the slot read (ar) and written (aw) roll from step to step.
  const uint8_t* const xa = uniform_ptr(reinterpret_cast<const uint8_t*>(a.xh) + ((size_t)by * nb * 64 + 4 * (size_t)wave) * 1024);
  const uint32_t aend = aring + AS * kG2ASlot;
  auto frag_a = [&](const uint8_t* src, uint32_t l, int i) {
    if (i == 0)
      lds_dma16<0>(src, voff16, l);
    else if (i == 1)
      lds_dma16<1024>(src, voff16, l);
    else if (i == 2)
      lds_dma16<2048>(src, voff16, l);
    else
      lds_dma16<3072>(src, voff16, l);
  };
  // B: column c's tile-blocks start at wcol[c] (column tiles past n read the
  // last one); block blk goes to ring half blk & 1.
  const uint8_t* wcol[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) {
    const int oc = ct0 + (GATED ? c % OT : c);
    wcol[c] = uniform_ptr((GATED && c >= OT ? a.wu : a.w) + (size_t)(oc < ntiles ? oc : ntiles - 1) * nb * TB);
  }
  auto issue_b = [&](int blk, int c) {
    const int bc = blk < nb ? blk : nb - 1;
    const uint32_t l = __builtin_amdgcn_readfirstlane(bring0 + (uint32_t)((blk & 1) * CT + c) * TB);
    P::issue(wcol[c] + (size_t)bc * TB, voff16, voff4, l, lane);
  };

  f4_t acc[8][CT];
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[rt][c]));
    }

#pragma unroll
  for (int c = 0; c < CT; ++c)
    issue_b(0, c);
#pragma unroll
  for (int t = 0; t < AD; ++t) {
    const uint8_t* src = xa + (size_t)(t < steps ? t : steps - 1) * 16384;
    const uint32_t l = aring + (uint32_t)t * kG2ASlot + 4096u * (uint32_t)wave;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      frag_a(src, l, i);
  }
  vm_wait<4 * (AD - 1)>();  // B(0) and A(0)
  typename P::K kk[CT];
  h8_t bclo[CT], bchi[CT];
  typename P::W wl;  // raw words of the last column for the current u-step
  {
    typename P::R r[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::raw(r[c], bring + c * TB, lane);
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::consts(kk[c], r[c], lane);
#pragma unroll
    for (int c = 0; c < CT - 1; ++c) {
      typename P::W w;
      P::words(w, bring + c * TB, 0, lane);
      P::dequant(kk[c], w, 0, bclo[c], bchi[c]);
    }
    P::words(wl, bring + (CT - 1) * TB, 0, lane);
  }
  uint32_t ar = aring, aw = aring + AD * kG2ASlot + 4096u * (uint32_t)wave;
  for (int blk = 0; blk < nb; ++blk) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * blk + u;
      const int ta = t + AD < steps ? t + AD : steps - 1;
      const uint8_t* const asrc = xa + (size_t)ta * 16384;
      if (u == 0)
        vm_wait<tg_wait(0, AD, CT, NL)>();
      else if (u == 1)
        vm_wait<tg_wait(1, AD, CT, NL)>();
      else if (u == 2)
        vm_wait<tg_wait(2, AD, CT, NL)>();
      else
        vm_wait<tg_wait(3, AD, CT, NL)>();
      __syncthreads();  // A(t) of every wave landed; u-step t - 1 fully read
      __builtin_amdgcn_sched_barrier(0);
      const int bn = u == 3 ? blk + 1 : blk, un = (u + 1) & 3;
      const uint8_t* aslot = lds + (ar - aring);
      h8_t af[16];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        af[i] = *reinterpret_cast<const h8_t*>(aslot + i * 1024 + 16 * lane);
      const uint8_t* bslot = bring + (size_t)((bn & 1) * CT) * TB;
      typename P::R r[CT];
      if (u == 3) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          P::raw(r[c], bslot + c * TB, lane);
      }
      typename P::W wv[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c)
        P::words(wv[c], bslot + c * TB, un, lane);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (c == 0)
          P::dequant(kk[CT - 1], wl, u, bclo[CT - 1], bchi[CT - 1]);
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt], bclo[c], acc[rt][c], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt + 1], bchi[c], acc[rt][c], 0, 0, 0);
        if (u == 3)
          P::consts(kk[c], r[c], lane);
        if (c > 0)
          P::dequant(kk[c - 1], wv[c - 1], un, bclo[c - 1], bchi[c - 1]);
#pragma unroll
        for (int i = 4 * c / CT; i < 4 * (c + 1) / CT; ++i)
          frag_a(asrc, aw, i);
        if (u == 0)
          issue_b(blk + 1, c);
      }
      wl = wv[CT - 1];
      ar = ar + kG2ASlot == aend ? aring : ar + kG2ASlot;
      aw = aw + kG2ASlot >= aend ? aw + kG2ASlot - AS * kG2ASlot : aw + kG2ASlot;
      __builtin_amdgcn_sched_group_barrier(0x100, 64, 0);
#pragma unroll
      for (int i = 0; i < 16 * CT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, P::kVPM, 0);
      }
    }
  }
  vm_wait<0>();
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < CT; ++c)
      asm volatile("" : "+a"(acc[rt][c]));

  float* const elds = reinterpret_cast<float*>(bring);  // this wave's B ring: its loads have landed
  if constexpr (GATED) {
    const int nct2 = ntiles - ct0 >= OT ? OT : ntiles - ct0 > 0 ? ntiles - ct0 : 0;
    gemm2_epilogue_gated<OutT>(a, acc, mt0, ct0, lane, nct2, elds);
    return;
  }
  const int nct = ntiles - ct0 >= CT ? CT : ntiles - ct0 > 0 ? ntiles - ct0 : 0;
  if (a.post == 0)
    gemm2_epilogue<OutT, 0>(a, acc, mt0, ct0, lane, nct, elds);
  else if (a.post == 1)
    gemm2_epilogue<OutT, 1>(a, acc, mt0, ct0, lane, nct, elds);
  else
    gemm2_epilogue<OutT, 2>(a, acc, mt0, ct0, lane, nct, elds);
}

// typed_gemm_tile with B in half tile-blocks (policies with kHalf): per
// column three half-slots, half h (half h % 2 of block h / 2) in slot h % 3.
// Half 1 of block blk + 1 is issued at u-step 1 of block blk into the slot of
// half 0 of blk (last read at u-step 0), half 0 of block blk + 2 at u-step 3
// into the slot of half 1 of blk (last read at u-step 2); each is read three
// or four u-steps after its issue.  The A ring has kAS = 3 slots (A two
// u-steps ahead).  Loads in issue order per u-step and column group c: A
// fragment c of A(t + 2), then at u = 1 column c's half 1 (kL1 loads), at
// u = 3 its half 0 (kL0 loads).  Every half read at u-step t was issued
// before A(t), so the wait for A(t) covers it: the loads after A(t)'s last
// fragment are column 3's half of u-step t - 2 and all of u-step t - 1, that
// is 4 + CT kL0 (u = 0), kL0 + 4 (u = 1), 4 + CT kL1 (u = 2), kL1 + 4
// (u = 3); at u-step 1 of the first block only A(2) follows A(1) (the
// prologue issues no B after it), so the wait there is 4.
template <class P, typename OutT>
__device__ __forceinline__ void typed_gemm_tile_half(const GemmArgs& a, uint8_t* lds, int bx, int by, int ntiles) {
  constexpr int CT = P::kCT, AS = P::kAS, AD = AS - 1, TB = P::kTB, HS = P::kHS, L0 = P::kL0, L1 = P::kL1;
  static_assert(AD == 2 && CT == 4, "the wait counts below assume A two u-steps ahead and four column groups");
  constexpr int W0 = 4 + CT * L0, W1 = L0 + 4, W2 = 4 + CT * L1, W3 = L1 + 4;
  static_assert(W0 < 64 && W2 < 64, "vmcnt field");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = a.nb, steps = 4 * nb;
  const int mt0 = by * (kG2M / 16);
  const int ct0 = bx * (4 * CT) + CT * wave;
  const uint32_t aring = lds_addr(lds);
  uint8_t* const bring = lds + AS * kG2ASlot + wave * (3 * CT * HS);
  const uint32_t bring0 = lds_addr(bring);
  const uint32_t voff16 = 16u * (uint32_t)lane, voff4 = 4u * (uint32_t)lane;
  const uint8_t* const xa = uniform_ptr(reinterpret_cast<const uint8_t*>(a.xh) + ((size_t)by * nb * 64 + 4 * (size_t)wave) * 1024);
  const uint32_t aend = aring + AS * kG2ASlot;
  auto frag_a = [&](const uint8_t* src, uint32_t l, int i) {
    if (i == 0)
      lds_dma16<0>(src, voff16, l);
    else if (i == 1)
      lds_dma16<1024>(src, voff16, l);
    else if (i == 2)
      lds_dma16<2048>(src, voff16, l);
    else
      lds_dma16<3072>(src, voff16, l);
  };
  const uint8_t* wcol[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c)
    wcol[c] = uniform_ptr(a.w + (size_t)(ct0 + c < ntiles ? ct0 + c : ntiles - 1) * nb * TB);
  // Half s of block blk (clamped to the last block) of column c into slot sl.
  auto issue_half = [&](int blk, int s, int c, int sl) {
    const int bc = blk < nb ? blk : nb - 1;
    const uint32_t l = __builtin_amdgcn_readfirstlane(bring0 + (uint32_t)((sl * CT + c) * HS));
    if (s == 0)
      P::issue_half0(wcol[c] + (size_t)bc * TB, voff16, voff4, l);
    else
      P::issue_half1(wcol[c] + (size_t)bc * TB, voff16, l);
  };
  auto hslot = [&](int sl, int c) { return bring + (size_t)(sl * CT + c) * HS; };

  f4_t acc[8][CT];
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      acc[rt][c] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
      asm volatile("" : "+a"(acc[rt][c]));
    }

  // Prologue: half 0 and 1 of block 0 and half 0 of block 1 into slots 0, 1,
  // 2, then A(0), A(1); everything but A(1) waited for.
#pragma unroll
  for (int c = 0; c < CT; ++c)
    issue_half(0, 0, c, 0);
#pragma unroll
  for (int c = 0; c < CT; ++c)
    issue_half(0, 1, c, 1);
#pragma unroll
  for (int c = 0; c < CT; ++c)
    issue_half(1, 0, c, 2);
#pragma unroll
  for (int t = 0; t < AD; ++t) {
    const uint8_t* src = xa + (size_t)(t < steps ? t : steps - 1) * 16384;
    const uint32_t l = aring + (uint32_t)t * kG2ASlot + 4096u * (uint32_t)wave;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      frag_a(src, l, i);
  }
  vm_wait<4>();
  typename P::K kk[CT];
  h8_t bclo[CT], bchi[CT];
  typename P::W wl;
  {
    typename P::R r[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::raw_half(r[c], hslot(0, c), lane);
#pragma unroll
    for (int c = 0; c < CT; ++c)
      P::consts(kk[c], r[c], lane);
#pragma unroll
    for (int c = 0; c < CT - 1; ++c) {
      typename P::W w;
      P::words_half(w, hslot(0, c), 0, lane);
      P::dequant(kk[c], w, 0, bclo[c], bchi[c]);
    }
    P::words_half(wl, hslot(0, CT - 1), 0, lane);
  }
  uint32_t ar = aring, aw = aring + AD * kG2ASlot + 4096u * (uint32_t)wave;
  // Slots of half 0 and half 1 of block blk and of half 0 of block blk + 1.
  int s0 = 0, s1 = 1, s2 = 2;
  for (int blk = 0; blk < nb; ++blk) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * blk + u;
      const int ta = t + AD < steps ? t + AD : steps - 1;
      const uint8_t* const asrc = xa + (size_t)ta * 16384;
      if (u == 0)
        vm_wait<W0>();
      else if (u == 1) {
        if (blk == 0)
          vm_wait<4>();
        else
          vm_wait<W1>();
      } else if (u == 2)
        vm_wait<W2>();
      else
        vm_wait<W3>();
      __syncthreads();  // A(t) of every wave landed; u-step t - 1 fully read
      __builtin_amdgcn_sched_barrier(0);
      const int un = (u + 1) & 3;
      const int ws = u == 0 ? s0 : u == 3 ? s2 : s1;  // slot of the words of u-step t + 1
      const uint8_t* aslot = lds + (ar - aring);
      h8_t af[16];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        af[i] = *reinterpret_cast<const h8_t*>(aslot + i * 1024 + 16 * lane);
      typename P::R r[CT];
      if (u == 3) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          P::raw_half(r[c], hslot(s2, c), lane);
      }
      typename P::W wv[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c)
        P::words_half(wv[c], hslot(ws, c), un, lane);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        if (c == 0)
          P::dequant(kk[CT - 1], wl, u, bclo[CT - 1], bchi[CT - 1]);
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt], bclo[c], acc[rt][c], 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 8; ++rt)
          acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[2 * rt + 1], bchi[c], acc[rt][c], 0, 0, 0);
        if (u == 3)
          P::consts(kk[c], r[c], lane);
        if (c > 0)
          P::dequant(kk[c - 1], wv[c - 1], un, bclo[c - 1], bchi[c - 1]);
        frag_a(asrc, aw, c);
        if (u == 1)
          issue_half(blk + 1, 1, c, s0);
        else if (u == 3)
          issue_half(blk + 2, 0, c, s1);
      }
      wl = wv[CT - 1];
      ar = ar + kG2ASlot == aend ? aring : ar + kG2ASlot;
      aw = aw + kG2ASlot >= aend ? aw + kG2ASlot - AS * kG2ASlot : aw + kG2ASlot;
      __builtin_amdgcn_sched_group_barrier(0x100, 64, 0);
#pragma unroll
      for (int i = 0; i < 16 * CT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, P::kVPM, 0);
      }
    }
    const int sn = s2;
    s2 = s1;
    s1 = s0;
    s0 = sn;
  }
  vm_wait<0>();
#pragma unroll
  for (int rt = 0; rt < 8; ++rt)
#pragma unroll
    for (int c = 0; c < CT; ++c)
      asm volatile("" : "+a"(acc[rt][c]));

  float* const elds = reinterpret_cast<float*>(bring);  // this wave's half-slots: their loads have landed
  const int nct = ntiles - ct0 >= CT ? CT : ntiles - ct0 > 0 ? ntiles - ct0 : 0;
  if (a.post == 0)
    gemm2_epilogue<OutT, 0>(a, acc, mt0, ct0, lane, nct, elds);
  else if (a.post == 1)
    gemm2_epilogue<OutT, 1>(a, acc, mt0, ct0, lane, nct, elds);
  else
    gemm2_epilogue<OutT, 2>(a, acc, mt0, ct0, lane, nct, elds);
}

template <class P>
constexpr int tg_lds_bytes() {
  if constexpr (TgIsHalf<P>::value)
    return P::kAS * kG2ASlot + 4 * 3 * P::kCT * P::kHS;
  else
    return P::kAS * kG2ASlot + 4 * 2 * P::kCT * P::kTB;
}

// Persistent over the (column block, row block) tiles, as the Q4_K GEMM.
template <class P, typename OutT, bool GATED = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void typed_gemm_kernel(GemmArgs a, TileMap map, int ntiles) {
  __shared__ __attribute__((aligned(16))) uint8_t lds[tg_lds_bytes<P>()];
  static_assert(tg_lds_bytes<P>() <= 160 * 1024, "LDS of one workgroup");
  const int count = tile_count(map);
  for (int i = 0; i < count; ++i) {
    if (i > 0)
      __syncthreads();
    int bx, by;
    tile_at(map, i, bx, by);
    if constexpr (TgIsHalf<P>::value)
      typed_gemm_tile_half<P, OutT>(a, lds, bx, by, ntiles);
    else
      typed_gemm_tile<P, OutT, GATED>(a, lds, bx, by, ntiles);
  }
}

// One workgroup of 64 lanes per tile-block (encode_lane, q4k_internal.h).
__global__ __launch_bounds__(64) void typed_relayout_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, uint32_t nb, uint32_t type) {
  const size_t tb = blockIdx.x;
  const uint32_t c = (uint32_t)(tb / nb), b = (uint32_t)(tb % nb);
  const int lane = threadIdx.x;
  const size_t bb = (size_t)type_block_bytes(type);
  encode_lane(type, src + ((size_t)(16 * c + (lane & 15)) * nb + b) * bb, dst + tb * 16 * bb, lane);
}

int env_int(const char* name, int fallback) {
  const char* v = getenv(name);
  return v && *v ? atoi(v) : fallback;
}

template <int RT, int T, int W, int BPW, bool GATED>
hipError_t gemv_launch(hipStream_t s, const GemvArgs& a, int dtype) {
  const dim3 grid((unsigned)(a.n / (16 * T))), block(64 * W);
  if (dtype == kF32)
    (void)dispatch(q4k_gemv_kernel<RT, T, W, BPW, GATED, float>, grid, block, s, a);
  else
    (void)dispatch(q4k_gemv_kernel<RT, T, W, BPW, GATED, _Float16>, grid, block, s, a);
  return hipGetLastError();
}

// One row tile: the block count per wave is fixed at compile time when the
// waves split nb evenly into at most 4 blocks each.
template <int T, bool GATED>
hipError_t gemv_one_row_tile(hipStream_t s, const GemvArgs& a, int dtype, int waves) {
  static const bool generic = env_int("Q4K_GEMV_GENERIC", 0) != 0;
  const int bpw = !generic && a.nb % waves == 0 ? a.nb / waves : 0;
  if (waves == 16) {
    if (bpw == 1)
      return gemv_launch<1, T, 16, 1, GATED>(s, a, dtype);
    if constexpr (T == 1 && !GATED) {  // the other BPW=3 instances spill
      if (bpw == 3)
        return gemv_launch<1, T, 16, 3, GATED>(s, a, dtype);
    }
    return gemv_launch<1, T, 16, 0, GATED>(s, a, dtype);
  }
  if (waves == 8) {
    if (bpw == 2)
      return gemv_launch<1, T, 8, 2, GATED>(s, a, dtype);
    return gemv_launch<1, T, 8, 0, GATED>(s, a, dtype);
  }
  if (bpw == 4)
    return gemv_launch<1, T, 4, 4, GATED>(s, a, dtype);
  return gemv_launch<1, T, 4, 0, GATED>(s, a, dtype);
}

template <int RT, bool GATED>
hipError_t gemv_multi_row_tile(hipStream_t s, const GemvArgs& a, int dtype, int waves, int tiles) {
  if constexpr (!GATED) {
    if (tiles == 2)
      return gemv_launch<RT, 2, 4, 0, false>(s, a, dtype);
  }
  if (waves >= 8)
    return gemv_launch<RT, 1, 8, 0, GATED>(s, a, dtype);
  return gemv_launch<RT, 1, 4, 0, GATED>(s, a, dtype);
}

// Instances kept within the register file (no spills): 16 waves only with
// one row tile; two column tiles only with one row tile and no gate/up pair.
template <bool GATED>
hipError_t gemv_dispatch(hipStream_t s, const GemvArgs& a, int dtype, const GemvShape& shape) {
  if (shape.row_tiles == 1) {
    if constexpr (!GATED) {
      if (shape.tiles == 2)
        return gemv_one_row_tile<2, false>(s, a, dtype, shape.waves);
    }
    return gemv_one_row_tile<1, GATED>(s, a, dtype, shape.waves);
  }
  if (shape.row_tiles == 2)
    return gemv_multi_row_tile<2, GATED>(s, a, dtype, shape.waves, shape.tiles);
  return gemv_multi_row_tile<3, GATED>(s, a, dtype, shape.waves, shape.tiles);
}

}  // namespace

namespace {

// Split-K instances: (NM, T, KS, BPS, DP).  A group is T column tiles of NM
// matrices; KS slices of BPS blocks each.
struct SplitkInst {
  int nm, t, ks, bps;
};
constexpr SplitkInst kSplitk[] = {
    {1, 8, 8, 6},  // K = 12288 (nb = 48), N a multiple of 1024: 8 tiles x 8 slices of 6 blocks
};

template <int NM, int T, int KS, int BPS, int DP>
hipError_t splitk_launch(hipStream_t s, const GemvArgs& a, int dtype, int grid, float* part, int* counters) {
  if (dtype == kF32)
    (void)dispatch(q4k_gemv_splitk_kernel<NM, T, KS, BPS, DP, float>, dim3((unsigned)grid), dim3(512), s, a, part, counters);
  else
    (void)dispatch(q4k_gemv_splitk_kernel<NM, T, KS, BPS, DP, _Float16>, dim3((unsigned)grid), dim3(512), s, a, part, counters);
  return hipGetLastError();
}

}  // namespace

bool gemv_splitk_plan(int m, int n, int nb, bool gated, int cus, SplitkPlan* plan) {
  static const int forced = env_int("Q4K_GEMV_SPLITK", -1);  // -1 auto, -2 off, else instance
  if (forced == -2 || m < 1 || m > 8 || n % 16 != 0)
    return false;
  const int tiles = n / 16, nm = gated ? 2 : 1;
  int best = -1, best_grid = 0;
  for (int i = 0; i < (int)(sizeof(kSplitk) / sizeof(kSplitk[0])); ++i) {
    const SplitkInst& c = kSplitk[i];
    if (forced >= 0 && i != forced)
      continue;
    if (c.nm != nm || c.ks * c.bps != nb || tiles % c.t != 0 || (tiles / c.t) % 8 != 0)
      continue;
    const int grid = tiles / c.t * c.ks;
    // Prefer the largest grid that fills at most one workgroup per CU, then
    // the smallest grid above that.
    const bool fits = grid <= cus, best_fits = best_grid <= cus;
    if (best < 0 || (fits && (!best_fits || grid > best_grid)) || (!fits && !best_fits && grid < best_grid)) {
      best = i;
      best_grid = grid;
    }
  }
  if (best < 0)
    return false;
  const SplitkInst& c = kSplitk[best];
  plan->inst = best;
  plan->groups = tiles / c.t;
  plan->ks = c.ks;
  plan->mt = c.nm * c.t;
  plan->grid = best_grid;
  return true;
}

size_t gemv_splitk_part_floats(const SplitkPlan& plan) {
  return (size_t)plan.groups * plan.ks * plan.mt * 8 * 16;
}

hipError_t launch_gemv_splitk(hipStream_t s, const GemvArgs& a, int dtype, const SplitkPlan& plan, float* part, int* counters) {
  (void)plan.inst;  // one instance
  // Two block-steps in flight per wave: measured faster than four (shorter
  // memory queues, as for the fused gate/up GEMV).
  return splitk_launch<1, 8, 8, 6, 2>(s, a, dtype, plan.grid, part, counters);
}

// Column tiles per workgroup of the rows GEMV (0: not this kernel).  Gated
// pairs at K = 4096 take 3 (one workgroup per CU at N = 12288): at M = 40
// 19.4 us against 26.7 on the one-tile GEMV.  Plain projections with K =
// 12288 take the most of 3, 2, 1 that still gives every CU a workgroup, or
// 1 (M = 40, N = 4096: 19.1 against 20.5 us).  Plain projections at K = 4096
// stay on the staged GEMV, which already splits K over 8 waves with two
// column tiles where that fills the CUs (measured as fast or faster).
RowsPlan gemv_rows_plan(int rows, int nb, int n, bool gated, int cus) {
  static const int forced = env_int("Q4K_GEMV_ROWS", -1);  // -1 auto, 0 off, 1..3 column tiles
  static const int slices_env = env_int("Q4K_GEMV_ROWS_SLICES", -1);  // -1 auto, 1 one slice, 3 three
  RowsPlan p;
  if (forced == 0 || rows <= 16 || rows > 16 * kGemvMaxRowTiles || n % 16 != 0)
    return p;
  const int ctiles = n / 16;
  if (gated) {
    if (nb != 16)
      return p;
    const int t = forced > 0 ? forced : 3;
    if (ctiles % t == 0 && (forced > 0 || ctiles / t >= cus))
      p.tiles = t;
    return p;
  }
  if (nb != 48 && !(forced > 0 && nb == 16))
    return p;
  // K = 12288: three K-slices of 4 column tiles when the column groups fill
  // the CUs in one round -- each CU then reads a third of x for 4 column
  // tiles instead of all of it for one (M = 40, N = 4096: 64 groups x 3).
  const bool slices_ok = nb == 48 && forced <= 0 && ctiles % 4 == 0 && (ctiles / 4) * 3 <= cus;
  if (slices_env == 3 ? nb == 48 && ctiles % 4 == 0 : slices_env != 1 && slices_ok) {
    p.tiles = 4;
    p.slices = 3;
    return p;
  }
  if (forced > 0) {
    if (ctiles % forced == 0)
      p.tiles = forced;
    return p;
  }
  p.tiles = 1;
  for (int t = 3; t >= 1; --t)
    if (ctiles % t == 0 && ctiles / t >= cus) {
      p.tiles = t;
      break;
    }
  return p;
}

size_t gemv_rows_part_floats(const RowsPlan& p, int n) {
  return p.slices > 1 ? (size_t)(n / (16 * p.tiles)) * p.slices * (16 * kGemvMaxRowTiles) * (16 * p.tiles) : 0;
}

template <int NM, int T, int RT, int BPW, int KS = 1>
hipError_t gemv_rows_launch(hipStream_t s, const GemvArgs& a, int dtype) {
  const dim3 grid((unsigned)(a.n / (16 * T) * KS)), block(512);
  if (dtype == kF32)
    (void)dispatch(q4k_gemv_rows_kernel<NM, T, RT, BPW, float, KS>, grid, block, s, a);
  else
    (void)dispatch(q4k_gemv_rows_kernel<NM, T, RT, BPW, _Float16, KS>, grid, block, s, a);
  return hipGetLastError();
}

// K = 4096 (2 blocks per wave) and, for plain projections, K = 12288 (6).
template <int NM, int T, int RT>
hipError_t gemv_rows_bpw(hipStream_t s, const GemvArgs& a, int dtype) {
  if (a.nb == 16)
    return gemv_rows_launch<NM, T, RT, 2>(s, a, dtype);
  if constexpr (NM == 1) {
    if (a.nb == 48)
      return gemv_rows_launch<NM, T, RT, 6>(s, a, dtype);
  }
  return hipErrorInvalidValue;
}

template <int NM, int T>
hipError_t gemv_rows_rt(hipStream_t s, const GemvArgs& a, int dtype) {
  return a.rows <= 32 ? gemv_rows_bpw<NM, T, 2>(s, a, dtype) : gemv_rows_bpw<NM, T, 3>(s, a, dtype);
}

hipError_t launch_gemv_rows(hipStream_t s, const GemvArgs& a, int dtype, const RowsPlan& p, bool gated) {
  const int tiles = p.tiles;
  if (a.rows <= 16 || a.rows > 16 * kGemvMaxRowTiles || (a.nb != 16 && a.nb != 48) || tiles < 1 || a.n % (16 * tiles) != 0 ||
      a.rows != (a.split ? 2 * a.m : a.m))
    return hipErrorInvalidValue;
  if (p.slices != 1) {
    // K = 12288: three K-slices of four column tiles (2 blocks per wave).
    // (Two slices of two column tiles, 3 blocks per wave and all 256 CUs,
    // measured the same config-2 pass: 78.9-81.3 against 79.4-79.7 us.)
    if (gated || p.slices != 3 || tiles != 4 || a.nb != 48 || !a.part || !a.counters)
      return hipErrorInvalidValue;
    return a.rows <= 32 ? gemv_rows_launch<1, 4, 2, 2, 3>(s, a, dtype) : gemv_rows_launch<1, 4, 3, 2, 3>(s, a, dtype);
  }
  if (gated) {
    if (a.nb != 16)
      return hipErrorInvalidValue;
    switch (tiles) {
      case 3: return gemv_rows_rt<2, 3>(s, a, dtype);
      case 2: return gemv_rows_rt<2, 2>(s, a, dtype);
      case 1: return gemv_rows_rt<2, 1>(s, a, dtype);
      default: return hipErrorInvalidValue;
    }
  }
  switch (tiles) {
    case 3: return gemv_rows_rt<1, 3>(s, a, dtype);
    case 2: return gemv_rows_rt<1, 2>(s, a, dtype);
    case 1: return gemv_rows_rt<1, 1>(s, a, dtype);
    default: return hipErrorInvalidValue;
  }
}

template <typename InT, bool NORM>
hipError_t stage_launch(hipStream_t s, const InT* x, _Float16* xo, _Float16* xs, float* rowscale, int m, int k, int mode, RowNorm nrm) {
  const dim3 grid((unsigned)m), block(kStageThreads);
  if (mode == kStageFrag)
    (void)dispatch(stage_x_kernel<InT, kStageFrag, NORM>, grid, block, s, x, xo, xs, rowscale, m, k, nrm);
  else if (mode == kStageGemm && k / 256 <= 16)
    (void)dispatch(stage_gemm_kernel<InT, 16, 32, NORM>, dim3((unsigned)((m + 7) / 8)), dim3(256), s, x, xo, rowscale, m, k, nrm);
  else if (mode == kStageGemm && k % 512 == 0 && k / 512 <= 24)  // K <= 12288: one read of x, 64 threads per row
    (void)dispatch(stage_gemm_kernel<InT, 24, 64, NORM>, dim3((unsigned)((m + 7) / 8)), dim3(512), s, x, xo, rowscale, m, k, nrm);
  else if (mode == kStageGemm)
    (void)dispatch(stage_gemm_kernel<InT, 0, 32, NORM>, dim3((unsigned)((m + 7) / 8)), dim3(256), s, x, xo, rowscale, m, k, nrm);
  else
    (void)dispatch(stage_x_kernel<InT, kStageFragSplit, NORM>, grid, block, s, x, xo, xs, rowscale, m, k, nrm);
  return hipGetLastError();
}

hipError_t launch_stage_pack(hipStream_t s, const void* x, int dtype, const DecodePack& pk, int m, int k) {
  const dim3 grid((unsigned)(k / 256 * 8)), block(64);
  if (dtype == kF32)
    (void)dispatch(stage_pack_kernel<float>, grid, block, s, static_cast<const float*>(x), pk.frag, pk.xs, pk.dsc, m, k);
  else
    (void)dispatch(stage_pack_kernel<_Float16>, grid, block, s, static_cast<const _Float16*>(x), pk.frag, pk.xs, pk.dsc, m, k);
  return hipGetLastError();
}

hipError_t launch_stage_x(hipStream_t s, const void* x, int dtype, _Float16* xo, _Float16* xs, float* rowscale, int m, int k, int mode,
                          const float* norm_w, float eps) {
  if (m <= 0)
    return hipSuccess;
  // One row per workgroup while 8 rows per workgroup leave CUs idle (fp32 /
  // fp16, one row against eight: K = 4096, M = 128 3.2 / 3.3 against 5.4 /
  // 7.2 us, M = 1024 7.5 / 7.8 against 7.6 / 12.4; K = 12288, M = 128 4.8 /
  // 4.9 against 12.8 / 14.3, M = 1024 15.8 / 14.4 against 17.1 / 20.7; past
  // that M = 2048 28.6 / 23.5 against 24.1 / 21.0).
  if (mode == kStageGemm && m <= 1024)
    return launch_stage_rows(s, x, dtype, xo, rowscale, m, k, norm_w, eps);
  RowNorm nrm;
  nrm.w = norm_w;
  nrm.eps = eps;
  if (dtype == kF32)
    return norm_w ? stage_launch<float, true>(s, static_cast<const float*>(x), xo, xs, rowscale, m, k, mode, nrm)
                  : stage_launch<float, false>(s, static_cast<const float*>(x), xo, xs, rowscale, m, k, mode, nrm);
  return norm_w ? stage_launch<_Float16, true>(s, static_cast<const _Float16*>(x), xo, xs, rowscale, m, k, mode, nrm)
                : stage_launch<_Float16, false>(s, static_cast<const _Float16*>(x), xo, xs, rowscale, m, k, mode, nrm);
}

GemvShape gemv_shape(int rows, int n, int nb, bool gated, int cus) {
  GemvShape sh;
  sh.row_tiles = rows <= 16 ? 1 : rows <= 32 ? 2 : 3;
  // One 16-column tile per workgroup (two for very wide outputs, one row tile,
  // no gate/up pair), and enough waves per workgroup -- each taking 1/waves
  // of K -- for about 12-16 resident waves per CU across the grid.
  const int ctiles = n / 16;
  static const int env_tiles = env_int("Q4K_GEMV_TILES", 0), env_waves = env_int("Q4K_GEMV_WAVES", 0);
  sh.tiles = (sh.row_tiles == 1 && !gated && n % 32 == 0 && ctiles >= 4096) ? 2 : 1;
  // More than one row tile: each workgroup reads all of the staged x (its
  // launches fit about 4 us + 14 us per MB of x a CU reads).  Between one
  // and two workgroups per CU, two column tiles per workgroup (4 waves) take
  // one round with half the x reads per tile: at M = 40, N = 6144 (the QKV
  // projection, 384 tiles) 11.7 us against 14.6.  Narrower outputs lose CUs
  // that way (N = 4096: 12.5 against 9.4 us), and gate/up pairs, three
  // workgroups per CU, measured 34.3 against 26.7 us (three tiles: 27.9).
  if (sh.row_tiles > 1 && !gated && ctiles % 2 == 0 && ctiles > cus && ctiles <= 2 * cus)
    sh.tiles = 2;
  if (env_tiles == 1 || (env_tiles == 2 && sh.row_tiles == 1 && !gated && n % 32 == 0))
    sh.tiles = env_tiles;
  const int groups = ctiles / sh.tiles;
  int waves = groups >= 1024 ? 4 : groups >= 512 ? 4 : groups >= 320 ? 8 : 16;
  if (env_waves == 4 || env_waves == 8 || env_waves == 16)
    waves = env_waves;
  while (waves > 4 && waves > nb)
    waves >>= 1;
  if (sh.row_tiles > 1 && waves > 8)
    waves = 8;
  sh.waves = waves;
  return sh;
}

hipError_t launch_gemv(hipStream_t s, const GemvArgs& a, int dtype, const GemvShape& shape, bool gated) {
  if (shape.row_tiles < 1 || shape.row_tiles > kGemvMaxRowTiles || a.n % (16 * shape.tiles) != 0 || a.rows > 16 * shape.row_tiles ||
      a.rows != (a.split ? 2 * a.m : a.m))
    return hipErrorInvalidValue;
  return gated ? gemv_dispatch<true>(s, a, dtype, shape) : gemv_dispatch<false>(s, a, dtype, shape);
}

bool gemm2_supported(int m, int n) {
  return n > 0 && n % 16 == 0 && m > 0;
}

int gemm2_rows(int m) {
  return (m + kG2M - 1) / kG2M * kG2M;
}

hipError_t launch_stream_read(hipStream_t s, const void* p, size_t bytes, uint32_t* out, int blocks) {
  (void)dispatch(stream_read_kernel, dim3((unsigned)blocks), dim3(256), s, static_cast<const u4_t*>(p), bytes / 16, out);
  return hipGetLastError();
}

hipError_t launch_mfma_ceiling(hipStream_t s, float* out, int blocks, int iters) {
  hipLaunchKernelGGL(mfma_ceiling_kernel, dim3((unsigned)blocks), dim3(256), 0, s, out, iters);
  return hipGetLastError();
}

// The tile map of a persistent GEMM launch of `grid` workgroups over a
// tiles_y x tiles_x tile grid: the XCD rectangles when the grid deals the
// same number of workgroups to each XCD and the rectangles divide the grid
// (Q4K_GEMM_XCD_ROWS: row groups, default 4; 0 keeps the plain order).
TileMap make_tile_map(int tiles_x, int tiles_y, int grid) {
  static const int rg_env = env_int("Q4K_GEMM_XCD_ROWS", 4);
  TileMap m{tiles_x, tiles_x * tiles_y, 0, 0, 0};
  const int rg = rg_env == 1 || rg_env == 2 || rg_env == 4 || rg_env == 8 ? rg_env : 0;
  if (rg && grid % 8 == 0 && tiles_y % rg == 0 && tiles_x % (8 / rg) == 0) {
    m.rg = rg;
    m.rows = tiles_y / rg;
    m.cols = tiles_x / (8 / rg);
  }
  return m;
}

template <class P, bool GATED = false>
hipError_t typed_gemm_launch(hipStream_t s, const GemmArgs& a, int dtype, int cus);

// Rounds of workgroups (tiles / CUs, rounded up) of the 256-column and
// 128-column tilings, weighted by the time of one tile of each.
bool gemm2_narrow(int tiles256, int tiles128, int cus) {
  static const int forced = env_int("Q4K_GEMM_NARROW", -1);  // -1 auto, 0 off, 1 always
  if (forced >= 0)
    return forced == 1;
  const int r4 = (tiles256 + cus - 1) / cus, r2 = (tiles128 + cus - 1) / cus;
  return r2 * kGemmNarrowTileTime < r4 * 10;
}

// 192 columns per workgroup (the typed template's Q4_K policy with three
// column tiles per wave) when the 256-column tiles leave CUs idle and the
// 192-column ones fill between three quarters of the CUs and all of them in
// one round.  At M = 821 the N = 6144 projection (168 256-column tiles, 224
// of 192) measured 55.0 us against 59.6 in K-segments and 64.3 unsplit; the
// N = 4096 one (154 tiles) 59.4 against 51.5 on 128 columns, which it keeps.
// The accumulation order and the dequantised values are those of the
// 256-column GEMM, and the K-split defers to this rule, so the gated GEMM
// stays bit-identical to the two-call form.  Q4K_GEMM_MID: -1 auto, 0
// never, 1 always (for the plain Q4_K GEMM).
static bool gemm2_mid(int m, int n, int cus) {
  static const int forced = env_int("Q4K_GEMM_MID", -1);
  if (forced >= 0)
    return forced == 1;
  const int tiles_y = (m + kG2M - 1) / kG2M;
  const int t4 = (n + kG2N - 1) / kG2N * tiles_y, t3 = (n / 16 + 11) / 12 * tiles_y;
  return t4 < cus && t3 <= cus && 4 * t3 >= 3 * cus;
}

// Segments 1 per workgroup on the CUs that `tiles` workgroups leave free.
static int split_segments_per_wg(int tiles, int cus) {
  const int free = cus - tiles;
  return (tiles + free - 1) / free;
}

// K-split of the pipelined GEMM when its 256-column tiles leave CUs idle:
// segment 0 of each tile (blocks [0, b)) on a workgroup of its own, segments
// 1 (the other nb - b blocks) q to a workgroup on the CUs the tiles leave
// free, q = tiles / free CUs rounded up.
//  - q = 1 (the tiles fill at most half the CUs) and K >= 8192: two halves
//    (b = nb / 2).  At M = 821 the K = 12288 down projection (112 tiles)
//    measured 113.6 us against 123.9 on the 128-column template; longer
//    segments 0 (b = 27, 30: 119.0, 128.0 us) do not pay for the exchange
//    they hide.  At K = 4096 the 112-tile O projection measured 56.0 us split
//    against 50.4 on the template, which it keeps.
//  - q = 2 and K >= 4096: b = q nb / (q + 1) rounded up, so that the q
//    segments 1 of a workgroup take no longer than one segment 0.  The
//    N = 6144 projection's 168 tiles at M = 821 (b = 11) measured 58.9-60.9
//    us for b = 10..13 against 64.3 unsplit: the segments 0 run at 5.4 us
//    per block against 4.0 unsplit, so that 252 workgroups gain only 8 %
//    over 168.
//  - q = 3, K >= 8192, N < K and the free CUs at least 7/8 filled (192 tiles on
//    256 CUs): b as for q = 2.  K = 12288 -> N = 4096 at M = 1536 170.1-172.0
//    us against 177.2-178.0 unsplit, K = 12288 -> 8192 at M = 768 163.9
//    against 176.4, K = 8192 -> 4096 at M = 1536 119.8 against 123.6.  Less
//    filled it gains nothing (176 tiles, M = 1408: 168.2-172.7 against
//    159.9-173.4), and neither does K = 4096 (-> 4096, M = 1536: 71.4
//    against 68.5).  A gate/up pair takes the same b (its bits are the two
//    calls') and loses by it (8192 -> 8192 at M = 768 276 us against 232):
//    pairs widen, so the rule keeps to projections that narrow.
//  - Otherwise no split.  The few free CUs then hold q short segments each, whose
//    exchanges follow one another: N = 12288 at M = 640 (q = 15) measured 182
//    us against 77.7 unsplit, its gate/up pair 251 against 139; N = 8192 at
//    M = 821 (q = 7) 102 against 73.2; K = 12288 -> 4096 at M = 1700 (q = 7)
//    215 against 197, at M = 1920 (q = 15) 273 against 206.
// Returns b, or 0 for no split.  Q4K_GEMM2_SPLIT=0 turns the split off;
// Q4K_GEMM2_SPLIT_B forces b (for every shape with tiles < CUs and b < nb).
int gemm2_split_b(int m, int n, int nb, int cus) {
  static const int on = env_int("Q4K_GEMM2_SPLIT", 1);
  static const int b_env = env_int("Q4K_GEMM2_SPLIT_B", 0);
  const int tiles = ((n + kG2N - 1) / kG2N) * ((m + kG2M - 1) / kG2M);
  if (!on || tiles >= cus || gemm2_mid(m, n, cus))
    return 0;
  if (b_env > 0)
    return b_env < nb ? b_env : 0;
  const int q = split_segments_per_wg(tiles, cus);
  if (q == 1)
    return nb >= 32 ? nb / 2 : 0;
  const bool three = q == 3 && nb >= 32 && n < 256 * nb && 8 * tiles >= 21 * (cus - tiles);
  return (q == 2 && nb >= 16) || three ? (q * nb + q) / (q + 1) : 0;
}

void gemm2_split_workspace(int m, int n, bool gated, size_t* part_floats, size_t* counters) {
  const int tiles_x = gated ? (n / 16 + 7) / 8 : (n + kG2N - 1) / kG2N, tiles = tiles_x * ((m + kG2M - 1) / kG2M);
  *part_floats = (size_t)2 * tiles * 4 * 32 * 64 * 4;
  *counters = (size_t)tiles;
}

namespace {
// Segments 0 one per workgroup and segments 1 q per workgroup past them
// when the launch's own tiles leave CUs free, else both dealt round robin
// (the gated GEMM, twice the plain GEMM's tiles, takes the plain GEMM's b).
template <bool GATED>
hipError_t gemm2_split_launch(hipStream_t s, GemmArgs a, int dtype, int tiles_x, int tiles_y, int cus, int b) {
  const int tiles = tiles_x * tiles_y;
  a.split_b = b;
  a.split_q = tiles < cus ? split_segments_per_wg(tiles, cus) : 0;
  const int grid = a.split_q > 0 ? tiles + (tiles + a.split_q - 1) / a.split_q : (2 * tiles < cus ? 2 * tiles : cus);
  const TileMap map{tiles_x, tiles, 0, 0, 0};
  if (dtype == kF32)
    (void)dispatch(q4k_gemm2_kernel<float, GATED, true>, dim3((unsigned)grid), dim3(256), s, a, map);
  else
    (void)dispatch(q4k_gemm2_kernel<_Float16, GATED, true>, dim3((unsigned)grid), dim3(256), s, a, map);
  return hipGetLastError();
}
}  // namespace

// Six column tiles per wave (384 columns per workgroup) for a plain GEMM
// when its rounds of workgroups over the CUs take no longer than those of
// the 256-column tiling, a 384-column tile counted as 1.375 of a 256-column
// one (at M = 2048, N = 12288, K = 4096: Q4_K 182.6 us against 199-202 with
// four tiles per wave, IQ4_XS 208-210 against 224-225).  Q4K_GEMM_SIX: -1
// auto, 0 never, 1 always (the Q4_K and IQ4_XS GEMMs).
static bool gemm_six(int tiles256, int tiles384, int cus) {
  static const int forced = env_int("Q4K_GEMM_SIX", -1);
  if (forced >= 0)
    return forced == 1;
  const int r4 = (tiles256 + cus - 1) / cus, r6 = (tiles384 + cus - 1) / cus;
  return 11 * r6 <= 8 * r4;
}

hipError_t launch_gemm2(hipStream_t s, const GemmArgs& a, int dtype, int cus) {
  if (!gemm2_supported(a.m, a.n) || a.nb < 1)
    return hipErrorInvalidValue;
  const int tiles_x = (a.n + kG2N - 1) / kG2N, tiles_y = (a.m + kG2M - 1) / kG2M, tiles = tiles_x * tiles_y;
  if (const int b = gemm2_split_b(a.m, a.n, a.nb, cus)) {
    if (!a.part || !a.counters)
      return hipErrorInvalidValue;
    return gemm2_split_launch<false>(s, a, dtype, tiles_x, tiles_y, cus, b);
  }
  if (gemm2_mid(a.m, a.n, cus))
    return typed_gemm_launch<Mid<TgQ4K, 5>>(s, a, dtype, cus);
  if (gemm_six(tiles, ((a.n / 16 + 23) / 24) * tiles_y, cus))
    return typed_gemm_launch<Six<TgQ4K>>(s, a, dtype, cus);
  if (gemm2_narrow(tiles, ((a.n / 16 + 7) / 8) * tiles_y, cus))
    return typed_gemm_launch<TgQ4K>(s, a, dtype, cus);
  static const int persist = env_int("Q4K_GEMM2_PERSIST", 1);
  const int grid = persist && tiles > cus ? cus : tiles;
  const TileMap map = make_tile_map(tiles_x, tiles_y, grid);
  const dim3 block(256);
  if (dtype == kF32)
    (void)dispatch(q4k_gemm2_kernel<float, false>, dim3((unsigned)grid), block, s, a, map);
  else
    (void)dispatch(q4k_gemm2_kernel<_Float16, false>, dim3((unsigned)grid), block, s, a, map);
  return hipGetLastError();
}

// The gated GEMM on the typed template with six B column tiles per wave
// (three gate and three up tiles: 192 output columns per workgroup, against
// 128 for q4k_gemm2_kernel) when its rounds of workgroups over the CUs take
// no longer, a 192-column tile counted as 1.375 of a 128-column one (at
// M = 2048, N = 12288, K = 4096 the plain GEMM measured 182.6 us with six
// column tiles per wave against 199-202 us with four).  Its accumulation
// order and dequantised values are those of q4k_gemm2_kernel, so it stays
// bit-identical to the gate-then-up calls.  Q4K_GEMM_GATED_SIX: -1 auto, 0
// never, 1 always.
static bool gemm2_gated_six(int tiles128, int tiles192, int cus) {
  static const int forced = env_int("Q4K_GEMM_GATED_SIX", -1);
  if (forced >= 0)
    return forced == 1;
  const int r4 = (tiles128 + cus - 1) / cus, r6 = (tiles192 + cus - 1) / cus;
  return 11 * r6 <= 8 * r4;
}

hipError_t launch_gemm2_gated(hipStream_t s, const GemmArgs& a, int dtype, int cus) {
  if (!gemm2_supported(a.m, a.n) || a.nb < 1 || !a.wu)
    return hipErrorInvalidValue;
  // 128 output columns (256 B columns: gate and up) per tile.
  const int tiles_x = (a.n / 16 + 7) / 8, tiles_y = (a.m + kG2M - 1) / kG2M, tiles = tiles_x * tiles_y;
  // K-segments exactly when, and where, the plain GEMM of this shape splits,
  // so that the gated launch stays bit-identical to the gate-then-up calls.
  if (const int b = gemm2_split_b(a.m, a.n, a.nb, cus)) {
    if (!a.part || !a.counters)
      return hipErrorInvalidValue;
    return gemm2_split_launch<true>(s, a, dtype, tiles_x, tiles_y, cus, b);
  }
  if (gemm2_gated_six(tiles, ((a.n / 16 + 11) / 12) * tiles_y, cus))
    return typed_gemm_launch<Six<TgQ4K>, true>(s, a, dtype, cus);
  const int grid = tiles > cus ? cus : tiles;
  const TileMap map = make_tile_map(tiles_x, tiles_y, grid);
  const dim3 block(256);
  if (dtype == kF32)
    (void)dispatch(q4k_gemm2_kernel<float, true>, dim3((unsigned)grid), block, s, a, map);
  else
    (void)dispatch(q4k_gemm2_kernel<_Float16, true>, dim3((unsigned)grid), block, s, a, map);
  return hipGetLastError();
}

hipError_t launch_fill_u32(hipStream_t s, uint32_t* p, uint32_t v, uint32_t n) {
  if (n == 0)
    return hipSuccess;
  const unsigned grid = (n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024;
  (void)dispatch(fill_u32_kernel, dim3(grid), dim3(256), s, p, v, n);
  return hipGetLastError();
}

hipError_t launch_gather(hipStream_t s, const void* x, void* out, int k, int dtype, const GatherIndex& idx) {
  if (idx.rows == 0)
    return hipSuccess;
  const dim3 grid(idx.rows), block(256);
  if (dtype == kF32)
    (void)dispatch(gather_rows_kernel<float>, grid, block, s, static_cast<const float*>(x), static_cast<float*>(out), k, idx);
  else
    (void)dispatch(gather_rows_kernel<_Float16>, grid, block, s, static_cast<const _Float16*>(x), static_cast<_Float16*>(out), k, idx);
  return hipGetLastError();
}

hipError_t launch_embedding_batch(hipStream_t s, const uint8_t* w, const int32_t* tokens, const EmbedQueries& qs, void* y, int rows, int n, int k,
                                  int dtype) {
  if (rows == 0)
    return hipSuccess;
  const dim3 grid((unsigned)(k / 256), (unsigned)rows), block(256);
  if (dtype == kF32)
    (void)dispatch(embedding_batch_kernel<float>, grid, block, s, w, tokens, static_cast<float*>(y), n, k / 256, qs);
  else
    (void)dispatch(embedding_batch_kernel<_Float16>, grid, block, s, w, tokens, static_cast<_Float16*>(y), n, k / 256, qs);
  return hipGetLastError();
}

hipError_t launch_embedding(hipStream_t s, const uint8_t* w, const int32_t* ids, void* y, int rows, int n, int k, int dtype) {
  if (rows == 0)
    return hipSuccess;
  const dim3 grid((unsigned)(k / 256), (unsigned)rows), block(256);
  if (dtype == kF32)
    (void)dispatch(embedding_kernel<float>, grid, block, s, w, ids, static_cast<float*>(y), n, k / 256);
  else
    (void)dispatch(embedding_kernel<_Float16>, grid, block, s, w, ids, static_cast<_Float16*>(y), n, k / 256);
  return hipGetLastError();
}

template <typename T>
static void rms_norm_rows(hipStream_t s, const void* x, const float* w, void* y, int rows, int k, float eps, const GatherIndex& gi, int gather) {
  const dim3 grid((unsigned)rows);
  const T* xt = static_cast<const T*>(x);
  T* yt = static_cast<T*>(y);
  // Eight elements at a time where rows and addresses allow it.
  const uintptr_t at = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(w);
  if (k % 8 == 0 && k <= 8 * 512 * kNormChunks && at % 16 == 0)
    (void)dispatch(rms_norm8_kernel<T>, grid, dim3(512), s, xt, w, yt, k, eps, gi, gather);
  else
    (void)dispatch(rms_norm_kernel<T>, grid, dim3(256), s, xt, w, yt, k, eps, gi, gather);
}

hipError_t launch_rms_norm(hipStream_t s, const void* x, const float* w, void* y, int rows, int k, float eps, int dtype, const GatherIndex* idx) {
  if (rows == 0)
    return hipSuccess;
  GatherIndex gi{};
  if (idx)
    gi = *idx;
  if (dtype == kF32)
    rms_norm_rows<float>(s, x, w, y, rows, k, eps, gi, idx ? 1 : 0);
  else
    rms_norm_rows<_Float16>(s, x, w, y, rows, k, eps, gi, idx ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_relayout(hipStream_t s, const uint8_t* src, uint8_t* dst, uint32_t n, uint32_t k) {
  const uint32_t nb = k / 256;
  const size_t tiles = (size_t)(n / 16) * nb;
  if (tiles == 0)
    return hipSuccess;
  (void)dispatch(relayout_kernel, dim3((unsigned)tiles), dim3(64), s, src, dst, n, nb);
  return hipGetLastError();
}

template <class F, int T, int DQ>
hipError_t typed_gemv_launch(hipStream_t s, const GemvArgs& a, int dtype) {
  const int ntiles = a.n / 16;
  const dim3 grid((unsigned)((ntiles + T - 1) / T)), block(512);
  if (dtype == kF32)
    (void)dispatch(typed_gemv_kernel<F, T, DQ, float>, grid, block, s, a);
  else
    (void)dispatch(typed_gemv_kernel<F, T, DQ, _Float16>, grid, block, s, a);
  return hipGetLastError();
}

template <class F, int T, int DQ, int W = 8>
hipError_t typed_persistent_launch(hipStream_t s, const GemvArgs& a, int dtype, int cus) {
  const int items = (a.n / 16 + T - 1) / T;
  const dim3 grid((unsigned)(items < cus ? items : cus)), block(64 * W);
  if (dtype == kF32)
    (void)dispatch(typed_gemv_persistent_kernel<F, T, DQ, W, float>, grid, block, s, a, items);
  else
    (void)dispatch(typed_gemv_persistent_kernel<F, T, DQ, W, _Float16>, grid, block, s, a, items);
  return hipGetLastError();
}

// K = 4096 with at least 16 column tiles per CU: the persistent form
// (F::kPW waves, F::kPT tiles per item).  Otherwise column tiles per
// workgroup: the most (of 4, 2, 1) that still gives every CU at least two
// workgroups.
template <class F>
hipError_t typed_gemv_dispatch(hipStream_t s, const GemvArgs& a, int dtype, int cus) {
  const int ntiles = a.n / 16;
  static const int persistent = env_int("Q6K_GEMV_PERSISTENT", -1);  // -1 auto, 0 off, 1 on
  if (a.nb == 16 && persistent != 0 && (persistent > 0 || ntiles >= 16 * cus))
    return typed_persistent_launch<F, F::kPT, 2, F::kPW>(s, a, dtype, cus);
  static const int forced = env_int("Q6K_GEMV_TILES", 0);
  const int t = forced == 1 || forced == 2 || forced == 4 ? forced : ntiles >= 8 * cus ? 4 : ntiles >= 4 * cus ? 2 : 1;
  if (t == 4)
    return typed_gemv_launch<F, 4, 2>(s, a, dtype);
  if (t == 2)
    return typed_gemv_launch<F, 2, 2>(s, a, dtype);
  return typed_gemv_launch<F, 1, 2>(s, a, dtype);
}

// The Q4_K LM-head shape (K = 4096, at least 16 column tiles per CU, m <= 8)
// on the persistent form.
bool q4k_persistent_supported(int m, int nb, int n, int cus) {
  static const int on = env_int("Q4K_GEMV_PERSISTENT", 1);
  return on && m >= 1 && m <= 8 && nb == 16 && n % 16 == 0 && n / 16 >= 16 * cus;
}

hipError_t launch_q4k_persistent(hipStream_t s, const GemvArgs& a, int dtype, int cus) {
  return typed_persistent_launch<FmtQ4K, FmtQ4K::kPT, 2, FmtQ4K::kPW>(s, a, dtype, cus);
}

hipError_t launch_typed_gemv(hipStream_t s, const GemvArgs& a, uint32_t type, int dtype, int cus) {
  switch (type) {
    case kTypeQ4_K:
      return typed_gemv_dispatch<FmtQ4K>(s, a, dtype, cus);
    case kTypeQ6_K:
      return typed_gemv_dispatch<FmtQ6K>(s, a, dtype, cus);
    case kTypeQ8_0:
      return typed_gemv_dispatch<FmtQ8_0>(s, a, dtype, cus);
    case kTypeQ5_K:
      return typed_gemv_dispatch<FmtQ5K>(s, a, dtype, cus);
    case kTypeIQ4_XS:
      return typed_gemv_dispatch<FmtIQ4XS>(s, a, dtype, cus);
    default:
      return hipErrorInvalidValue;
  }
}

template <class P, bool GATED>
hipError_t typed_gemm_launch(hipStream_t s, const GemmArgs& a, int dtype, int cus) {
  constexpr int OT = GATED ? P::kCT / 2 : P::kCT;  // output column tiles per wave
  const int ntiles = a.n / 16, tiles_x = (ntiles + 4 * OT - 1) / (4 * OT);
  const int tiles_y = (a.m + kG2M - 1) / kG2M, tiles = tiles_x * tiles_y;
  const int g = tiles > cus ? cus : tiles;
  const TileMap map = make_tile_map(tiles_x, tiles_y, g);
  const dim3 grid((unsigned)g), block(256);
  if (dtype == kF32)
    (void)dispatch(typed_gemm_kernel<P, float, GATED>, grid, block, s, a, map, ntiles);
  else
    (void)dispatch(typed_gemm_kernel<P, _Float16, GATED>, grid, block, s, a, map, ntiles);
  return hipGetLastError();
}

bool typed_gemm_supported(uint32_t type, int m, int n) {
  const bool served = type == kTypeQ5_K || type == kTypeQ6_K || type == kTypeQ8_0 || type == kTypeIQ4_XS;
  return served && m > 0 && n > 0 && n % 16 == 0;
}

// Rounds of workgroups of the 192-column Q8_0 tiling against the 128-column
// one, each weighted by its columns per tile.
static bool q8_mid(int ntiles, int tiles_y, int cus) {
  static const int forced = env_int("Q4K_TYPED_MID", -1);
  if (forced >= 0)
    return forced == 1;
  const int r3 = ((ntiles + 11) / 12 * tiles_y + cus - 1) / cus, r2 = ((ntiles + 7) / 8 * tiles_y + cus - 1) / cus;
  return 3 * r3 <= 2 * r2;
}

// Four column tiles per wave with B in half tile-blocks (TgQ8_0W) where its
// rounds of workgroups over the CUs take no longer than those of the three-
// and two-tile forms, each round weighted by the time of one tile of that
// form: at M = 2048 a 192-column tile took 0.80 and a 128-column tile 0.61 of
// a 256-column tile's time (N = 12288, K = 4096: 190.6 us against 202.1 with
// three tiles per wave; N = 4096, K = 12288: 178.6 against 219.0 with two).
// Q4K_TYPED_Q8W: -1 auto, 0 never, 1 always; Q4K_TYPED_MID set (0 or 1)
// turns the auto choice of this form off as well.
static bool q8_wide(int ntiles, int tiles_y, int cus) {
  static const int forced = env_int("Q4K_TYPED_Q8W", -1);
  static const int mid = env_int("Q4K_TYPED_MID", -1);
  if (forced >= 0)
    return forced == 1;
  if (mid >= 0)
    return false;
  auto rounds = [&](int cols) { return ((ntiles * 16 + cols - 1) / cols * tiles_y + cus - 1) / cus; };
  const int r4 = rounds(256), r3 = rounds(192), r2 = rounds(128);
  return 100 * r4 <= 80 * r3 && 100 * r4 <= 61 * r2;
}

hipError_t launch_typed_gemm(hipStream_t s, const GemmArgs& a, uint32_t type, int dtype, int cus) {
  if (!typed_gemm_supported(type, a.m, a.n) || a.nb < 1)
    return hipErrorInvalidValue;
  const int ntiles = a.n / 16, tiles_y = (a.m + kG2M - 1) / kG2M;
  const bool narrow = gemm2_narrow(((ntiles + 15) / 16) * tiles_y, ((ntiles + 7) / 8) * tiles_y, cus);
  switch (type) {
    case kTypeQ5_K:
      return narrow ? typed_gemm_launch<Narrow<TgQ5K>>(s, a, dtype, cus) : typed_gemm_launch<TgQ5K>(s, a, dtype, cus);
    case kTypeQ6_K:
      return narrow ? typed_gemm_launch<Narrow<TgQ6K>>(s, a, dtype, cus) : typed_gemm_launch<TgQ6K>(s, a, dtype, cus);
    case kTypeQ8_0:
      // Four column tiles per wave on the half tile-block ring (q8_wide), or
      // two (two blocks of its tile-blocks per column fit beside an A ring),
      // or three where the 192-column grid takes no more time in rounds:
      // three tiles read each A fragment for half as many MFMAs again (at
      // M = 2048 the N = 12288 GEMM measured 211 instead of 243 us; Q6_K and
      // Q5_K measured slower with three, also with a 5-slot A ring).
      // Q4K_TYPED_MID: -1 auto, 0 never, 1 always.
      if (q8_wide(ntiles, tiles_y, cus))
        return typed_gemm_launch<TgQ8_0W>(s, a, dtype, cus);
      if (q8_mid(ntiles, tiles_y, cus))
        return typed_gemm_launch<Mid<TgQ8_0, 3>>(s, a, dtype, cus);
      return typed_gemm_launch<TgQ8_0>(s, a, dtype, cus);
    default:
      if (gemm_six(((ntiles + 15) / 16) * tiles_y, ((ntiles + 23) / 24) * tiles_y, cus))
        return typed_gemm_launch<Six<TgIQ4XS>>(s, a, dtype, cus);
      return narrow ? typed_gemm_launch<Narrow<TgIQ4XS>>(s, a, dtype, cus) : typed_gemm_launch<TgIQ4XS>(s, a, dtype, cus);
  }
}

hipError_t launch_typed_relayout(hipStream_t s, const uint8_t* src, uint8_t* dst, uint32_t n, uint32_t k, uint32_t type) {
  const uint32_t nb = k / 256;
  const size_t tiles = (size_t)(n / 16) * nb;
  if (tiles == 0)
    return hipSuccess;
  if (type_block_bytes(type) == 0 || type == kTypeQ4_K)
    return hipErrorInvalidValue;
  (void)dispatch(typed_relayout_kernel, dim3((unsigned)tiles), dim3(64), s, src, dst, nb, type);
  return hipGetLastError();
}

}  // namespace q4k
