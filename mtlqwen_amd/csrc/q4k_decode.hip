// Decode GEMV of up to 8 rows with K = 4096, every weight type, a plain
// projection or a gate/up pair, in one launch: x (RMS-normalised on the way in,
// if asked) is packed in registers by the workgroups that multiply it.
//
// Bound by memory and by the latency before the weights stream: a call's time is
// about 5.2 us plus 1.3 us (Q4_K; 7 TB/s) per column tile that a CU takes.  With
// separate staging (or norm and pack) launches in front, 8 rows took, before
// and after: Q4_K N = 1024 8.0 -> 5.9 us, 4096 8.7 -> 6.4, 12288 14.1 -> 9.4,
// 24576 23.1 -> 15.2, 49152 38.3 -> 29.3; Q6_K 4096 8.9 -> 7.1, 12288 18.1 ->
// 11.0; Q8_0 4096 9.1 -> 6.7, 12288 18.2 -> 12.1; a Q4_K pair of N = 8192 14.7
// -> 11.1 (of 12288 14.7, bandwidth either way).
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include "q4k_pack.h"

namespace q4k {
namespace {

// Workgroup = W waves over the 16 blocks of K (BPW = 16 / W each) and T column
// tiles of NM matrices.  A wave's tile-blocks ("units") are requested once its
// x has landed, two in flight.
template <class F, int NM, int T, int W, typename OutT, bool NORM>
__global__ __launch_bounds__(64 * W) void decode_gemv_kernel(GemvArgs a) {
  constexpr int BPW = 16 / W, MT = NM * T, U = BPW * MT, DQ = U < 2 ? U : 2, WF = gu_wave_floats<BPW>();
  static_assert(MT * 8 * 16 <= WF, "partials fit the x region");
  __shared__ __attribute__((aligned(16))) float xl[W * WF];
  __shared__ float ssq[W][8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, col = lane & 15;
  const int ntiles = a.n >> 4, tile0 = blockIdx.x * T;
  const int bw = ((wave + (int)blockIdx.x) % W) * BPW;
  const size_t tile_bytes = (size_t)16 * F::kTB;
  typename F::U un[U];
  auto issue_unit = [&](int u) {
    const int j = u / MT, mt = u - j * MT, t = mt % T;
    const int tile = tile0 + t < ntiles ? tile0 + t : ntiles - 1;
    F::load(un[u], (mt < T ? a.w : a.wu) + (size_t)tile * tile_bytes + (size_t)(bw + j) * F::kTB, lane);
    __builtin_amdgcn_sched_barrier(0);
  };
  XBlock xb[BPW];
  gate_up_pack_x<OutT, NORM, W, BPW>(a, xl, ssq, bw, xb, [&] {
#pragma unroll
    for (int u = 0; u < DQ; ++u)
      issue_unit(u);
  });
  f4_t acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    acc[mt] = f4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = u / MT;
    __builtin_amdgcn_sched_barrier(0);
    if (u + DQ < U)
      issue_unit(u + DQ);
    XF xf;
#pragma unroll
    for (int s = 0; s < 8; ++s)
      xf.f[s] = xb[j].frag[s];
    xf.xs = xb[j].xs;
#pragma unroll
    for (int v = 0; v < 4; ++v)
      xf.dv[v] = xb[j].dv[v];
    F::mac(un[u], xf, lane, acc[u - j * MT]);
  }
  // C row 4g + v, lanes g < 2 adding the low parts held 32 lanes up; the
  // waves' sums meet in LDS in the order of their blocks' waves.
  float* const xw = xl + (size_t)wave * WF;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float tot = acc[mt][v] + __shfl_xor(acc[mt][v], 32);
      if (g < 2)
        xw[(mt * 8 + 4 * g + v) * 16 + col] = tot;
    }
  __syncthreads();
  OutT* y = reinterpret_cast<OutT*>(a.y);
  const OutT* aux = reinterpret_cast<const OutT*>(a.aux);
  for (int o = tid; o < a.m * 16 * T; o += 64 * W) {
    const int row = o / (16 * T), c = o % (16 * T), t = c >> 4, cc = c & 15;
    if (tile0 + t >= ntiles)
      continue;
    const size_t off = (size_t)row * a.n + (size_t)(tile0 + t) * 16 + cc;
    float acc_v[NM];
#pragma unroll
    for (int mi = 0; mi < NM; ++mi) {
      acc_v[mi] = 0.0f;
#pragma unroll
      for (int w = 0; w < W; ++w)
        acc_v[mi] += xl[w * WF + ((mi * T + t) * 8 + row) * 16 + cc];
      if (sizeof(OutT) == 2)
        acc_v[mi] = round_half(acc_v[mi]);
    }
    float out;
    if constexpr (NM == 2)
      out = silu(acc_v[0]) * acc_v[1];
    else
      out = a.post == 1 ? acc_v[0] + load_elem(aux, off) : a.post == 2 ? silu(load_elem(aux, off)) * acc_v[0] : acc_v[0];
    store_elem(y, off, out);
  }
}

template <class F, int NM, int T, int W>
hipError_t decode_launch(hipStream_t s, const GemvArgs& a, int dtype) {
  const dim3 grid((unsigned)((a.n / 16 + T - 1) / T)), block(64 * W);
  if (dtype == kF32)
    a.norm_w ? (void)dispatch(decode_gemv_kernel<F, NM, T, W, float, true>, grid, block, s, a)
             : (void)dispatch(decode_gemv_kernel<F, NM, T, W, float, false>, grid, block, s, a);
  else
    a.norm_w ? (void)dispatch(decode_gemv_kernel<F, NM, T, W, _Float16, true>, grid, block, s, a)
             : (void)dispatch(decode_gemv_kernel<F, NM, T, W, _Float16, false>, grid, block, s, a);
  return hipGetLastError();
}

// Sixteen waves (128 registers) hold up to four tiles, eight the larger ones
// (N = 8192, two tiles: 7.8 us against 8.1 with eight).
template <class F, int NM, int T>
hipError_t decode_tiles_launch(hipStream_t s, const GemvArgs& a, int dtype) {
  return decode_launch<F, NM, T, NM * T <= 4 ? 16 : 8>(s, a, dtype);
}

// Column tiles per workgroup: of those built, the fewest whose workgroups take
// the fewest rounds over the CUs.  A workgroup's x costs every round about 5 us
// and a tile 1.3, and an idle tile costs too: N = 12288 took 9.4 us with three
// tiles (one round), 10.3 with four, 13.4 with two; N = 16384 11.6 with four,
// 14.2 with two, 14.3 with six; N = 24576 15.2 with six, 17.8 with three.
int decode_tiles(int ntiles, int cus, bool gated) {
  const int most = gated ? 3 : 6;
  int best = 1, rounds = (ntiles + cus - 1) / cus;
  for (int t = 2; t <= most; t += t == 4 ? 2 : 1) {
    const int r = (ntiles + t * cus - 1) / (t * cus);
    if (r < rounds) {
      best = t;
      rounds = r;
    }
  }
  return best;
}

template <class F>
hipError_t decode_dispatch(hipStream_t s, const GemvArgs& a, int dtype, int cus) {
  const int t = decode_tiles(a.n / 16, cus, a.wu != nullptr);
  if (a.wu)
    return t == 1 ? decode_tiles_launch<F, 2, 1>(s, a, dtype) : t == 2 ? decode_tiles_launch<F, 2, 2>(s, a, dtype) : decode_tiles_launch<F, 2, 3>(s, a, dtype);
  switch (t) {
    case 1: return decode_tiles_launch<F, 1, 1>(s, a, dtype);
    case 2: return decode_tiles_launch<F, 1, 2>(s, a, dtype);
    case 3: return decode_tiles_launch<F, 1, 3>(s, a, dtype);
    case 4: return decode_tiles_launch<F, 1, 4>(s, a, dtype);
    default: return decode_tiles_launch<F, 1, 6>(s, a, dtype);
  }
}

}  // namespace

// Plain outputs stay narrower than the persistent GEMV's (16 column tiles per
// CU), which packs x once per CU.
bool decode_gemv_supported(int m, int nb, int n, bool gated, int cus) {
  if (m < 1 || m > 8 || nb != 16 || n % 16 != 0)
    return false;
  if (gated) {
    static const bool on = [] {
      const char* v = getenv("Q4K_GEMV_GATE_UP");
      return !v || !*v || atoi(v) != 0;
    }();
    return on;
  }
  // The plain GEMVs' own switches name forms of theirs.
  static const bool off = [] {
    for (const char* name : {"Q4K_GEMV_GENERIC", "Q4K_GEMV_WAVES", "Q4K_GEMV_TILES", "Q6K_GEMV_PERSISTENT", "Q6K_GEMV_TILES"})
      if (const char* v = getenv(name))
        if (*v)
          return true;
    return false;
  }();
  return !off && n / 16 < 16 * cus;
}

hipError_t launch_decode_gemv(hipStream_t s, const GemvArgs& a, uint32_t type, int dtype, int cus) {
  if (a.m < 1 || a.m > 8 || a.nb != 16 || a.n % 16 != 0)
    return hipErrorInvalidValue;
  switch (type) {
    case kTypeQ4_K:
      return decode_dispatch<FmtQ4K>(s, a, dtype, cus);
    case kTypeQ6_K:
      return decode_dispatch<FmtQ6K>(s, a, dtype, cus);
    case kTypeQ8_0:
      return decode_dispatch<FmtQ8_0>(s, a, dtype, cus);
    case kTypeQ5_K:
      return decode_dispatch<FmtQ5K>(s, a, dtype, cus);
    case kTypeIQ4_XS:
      return decode_dispatch<FmtIQ4XS>(s, a, dtype, cus);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace q4k
