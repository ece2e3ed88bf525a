// moe_expert.hip - grouped INT4 expert kernels for small token tiles (decode).
//
// Arithmetic (the reference's INT4 GEMV, tools/cmdlist/kernels.cpp:148-201,
// restated for bf16 activations): y[m][n] = sum_g s[n][g] * sum_{k in g}
// q[n][k] * x[m][k].  The inner sum runs on bf16 MFMA
// (v_mfma_f32_4x4x4bf16_1k): each packed nibble becomes the bf16 value
// 136 + q (bit pattern 0x4300 | (q + 8), two nibbles per AND-OR), the
// accumulator of every group starts at -136 * sum_{k in g} x[m][k] (that sum
// comes from the same MFMA against a ones operand), so after the group's
// MFMAs it holds sum q*x, and the group scale is applied once per
// accumulator in fp32.
//
// One block = one work item: a tile of at most DEC_MT tokens routed to one
// expert x 16 * RG * WR weight rows (moe_expert_item.h).  Decode is bound by
// weight bytes in flight, so every wave issues all its weight loads at once.
//
// MODE 0: gate and up together, epilogue silu(g)*u -> act (bf16, MFMA
//         order).
// MODE 1: down, epilogue o (bf16) per dispatch position; the combine kernel
//         sums a token's k + 1 rows in slot order.
#include <hip/hip_ext.h>

#include "moe_common.h"
#include "moe_internal.h"
#include "moe_expert_item.h"

namespace {

constexpr int MAX_WAVES = 16;  // 1024 threads

template <int SD, int KBW, int RG, int MODE>
__global__ __launch_bounds__(1024) void k_expert_lds(ExpertArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tile_id = blockIdx.x / a.n_slabs, slab = blockIdx.x % a.n_slabs;
  int n_tiles;
  const int4 t = sload_tile(a.tiles, a.n_tiles, tile_id, n_tiles);
  if (tile_id >= n_tiles) return;
  expert_lds_item<SD, KBW, RG, DEC_MT, MODE, false, false, true>(a, t, slab, lds);
}

}  // namespace

#ifdef AINFER_DECODE_TRACE
extern "C" int ainfer_debug_land_expert(void *host) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_dland), sizeof(g_dland)) == hipSuccess ? 0 : -1;
}
#endif

// KBW k-groups per wave (the preferred count, raised until one row group
// fits in 16 waves, lowered until it divides both K group counts), WK =
// waves along K, WR = row groups per block.
#ifndef EXPERT_WAVES
#define EXPERT_WAVES 4  // waves per expert item (K-split x row groups)
#endif
bool expert_geometry(int mode, int H, int I, int Is, int pref_kbw, int *KBW, int *WK,
                     int *WR) {
  const int KBr = (mode == 0 ? H : I) / 128;
  const int KBs = (mode == 0 ? H : (Is > 0 ? Is : I)) / 128;
  const int KBmax = KBr > KBs ? KBr : KBs;
  int kbw = pref_kbw < 1 ? 1 : (pref_kbw > 4 ? 4 : pref_kbw);
  while ((KBmax + kbw - 1) / kbw > MAX_WAVES && kbw < 4) kbw *= 2;
  while (kbw > 1 && (KBr % kbw || KBs % kbw)) kbw /= 2;
  if ((KBmax + kbw - 1) / kbw > MAX_WAVES || KBr % kbw || KBs % kbw) return false;
  const int wk = KBmax / kbw;
  int wr = EXPERT_WAVES / wk;
  if (wr < 1) wr = 1;
  *KBW = kbw;
  *WK = wk;
  *WR = wr;
  return true;
}


hipEvent_t g_kev_start = nullptr, g_kev_stop = nullptr;

template <int SD, int MODE>
void launch_kbw(int kbw, unsigned grid, int threads, size_t lds, const ExpertArgs &a,
                hipStream_t s) {
  auto go = [&](auto kern) {
    if (g_kev_start) {  // profiling: the kernel's own start and end
      hipExtLaunchKernelGGL(kern, dim3(grid), dim3(threads), (uint32_t)lds, s, g_kev_start,
                            g_kev_stop, 0u, a);
      g_kev_start = g_kev_stop = nullptr;
    } else {
      kern<<<grid, threads, lds, s>>>(a);
    }
  };
  constexpr int RG = stream_rg(MODE);
  if (kbw == 1)
    go(k_expert_lds<SD, 1, RG, MODE>);
  else if (kbw == 2)
    go(k_expert_lds<SD, 2, RG, MODE>);
  else
    go(k_expert_lds<SD, 4, RG, MODE>);
}

void set_expert_launch_events(hipEvent_t start, hipEvent_t stop) {
  g_kev_start = start;
  g_kev_stop = stop;
}

hipError_t launch_expert_stream(int mode, int scale_dtype, ExpertArgs a, int max_tiles,
                                int pref_kbw, hipStream_t s) {
  if (max_tiles <= 0) return hipSuccess;
  const int rg = stream_rg(mode);
  int kbw;
  if (!expert_geometry(mode, a.H, a.I, a.Is, pref_kbw, &kbw, &a.WK, &a.WR))
    return hipErrorInvalidValue;
  const int Nmax = mode == 0 ? (a.I > a.Is ? a.I : a.Is) : a.H;
  a.n_slabs = (Nmax + 16 * rg * a.WR - 1) / (16 * rg * a.WR);
  const int threads = a.WK * a.WR * 64;
  // A staging; the K-split partials reuse it when they fit (expert_lds_item, ALIAS)
  const size_t lds = (size_t)a.WK * a.WR * item_lds_per_wave(DEC_MT, kbw, rg, mode);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  const long grid = (long)max_tiles * a.n_slabs;
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  if (mode == 0) {
    if (scale_dtype == AINFER_SCALE_FP16)
      launch_kbw<AINFER_SCALE_FP16, 0>(kbw, (unsigned)grid, threads, lds, a, s);
    else
      launch_kbw<AINFER_SCALE_BF16, 0>(kbw, (unsigned)grid, threads, lds, a, s);
  } else {
    if (scale_dtype == AINFER_SCALE_FP16)
      launch_kbw<AINFER_SCALE_FP16, 1>(kbw, (unsigned)grid, threads, lds, a, s);
    else
      launch_kbw<AINFER_SCALE_BF16, 1>(kbw, (unsigned)grid, threads, lds, a, s);
  }
  return hipGetLastError();
}
