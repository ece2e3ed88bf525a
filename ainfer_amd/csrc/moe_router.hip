// moe_router.hip - router for gfx950: MFMA logits, exact candidate refine,
// top-k, renormalised weights, sigmoid shared gate.
//
// The top-k must equal, bit for bit, the top-k of the fp32 logits computed in
// the lane-strided chunk order (include/ainfer_moe.h).  Computing that order
// for all E experts is a latency-bound VALU job, so the router runs in two
// kernels:
//
//  k_router_mfma: approximate logits on bf16 MFMA (products exact, fp32
//    accumulation in the hardware's order) plus the 2-norm of every router
//    weight row.
//  k_select: one wave or one workgroup per token.  With L_k the k-th largest approximate
//    logit and d >= |approx - exact| + |canonical - exact| for every expert,
//    any expert whose canonical logit can reach the canonical top-k has
//    approx >= L_k - 2d (the top-k experts by approx all have canonical >=
//    L_k - d).  Those candidates are recomputed in the canonical order and
//    the top-k is taken among them: the result equals the top-k over all E
//    canonical logits.  d is a rigorous fp32 summation bound: for n products
//    accumulated with one rounding each (to nearest or toward zero),
//    |error| <= n * 2^-23 * sum|x_i w_i| <= n * 2^-23 * ||x|| * ||w_e||
//    (Cauchy-Schwarz), taken for both paths, plus margins for the bias
//    addition and for denormal flushing.  When many logits tie, every expert
//    becomes a candidate and the same code recomputes all of them.
//
// The dispatch for T <= 64 runs in k_select's last block (dispatch_small_block,
// moe_dispatch.h).
#include <string.h>

#include "moe_common.h"
#include "moe_dispatch.h"
#include "moe_gemm_parts.h"
#include "moe_topk.h"
#include "moe_internal.h"

#ifdef AINFER_DECODE_TRACE
__device__ unsigned long long g_strace[4096][8];
#define STRACE(I) \
  if ((threadIdx.x & 63) == 0 && (!COOP || threadIdx.x == 0) && t < 4096) \
  g_strace[t][I] = __builtin_amdgcn_s_memrealtime()
extern "C" int ainfer_debug_strace(void *host) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_strace), sizeof(g_strace)) == hipSuccess ? 0 : -1;
}
#else
#define STRACE(I)
#endif

namespace {

// ---------------------------------------------------------------------------
// Approximate logits.  Block = NW waves over one (16-expert, 16*MS-token)
// tile; wave w takes k-slice [w*H/NW, (w+1)*H/NW) in 32-wide MFMA steps.
// Lane l: expert row l%16, k offset 8*(l/16) inside each step (A and B use
// the same k mapping, so both operands load 16 contiguous bytes).
// ---------------------------------------------------------------------------
template <int MS>
__global__ __launch_bounds__(1024) void k_router_mfma(const uint16_t *__restrict__ x,
                                                      const uint16_t *__restrict__ rw,
                                                      const float *__restrict__ bias,
                                                      float *__restrict__ approx,
                                                      float *__restrict__ wnorm,
                                                      int32_t *__restrict__ ticket, int T, int H,
                                                      int E, int NW) {
  extern __shared__ float red[];  // [NW][MS*256] partial logits, then [NW][16] norms
  // the last-block counter of the following k_select launch starts at 0
  if (ticket && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *ticket = 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int n = lane & 15, q = lane >> 4;
  const int e0 = blockIdx.x * 16, t0 = blockIdx.y * 16 * MS;
  const int e = min(e0 + n, E - 1);
  const int steps = H / (32 * NW);  // 32-wide k-steps of this wave
  const int kbase = wave * steps * 32;
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(x, (uint32_t)T * (uint32_t)H * 2u);
  f32x4 acc[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) acc[ms] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss = 0.0f;
  const uint16_t *wrow = rw + (size_t)e * H + kbase + 8 * q;
  uint32_t xoff[MS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms) {
    const int t = t0 + 16 * ms + n;
    xoff[ms] = t < T ? ((uint32_t)t * (uint32_t)H + (uint32_t)(kbase + 8 * q)) * 2u : BUF_OOB;
  }
  for (int s0 = 0; s0 < steps; s0 += 4) {
    u32x4 wv[4], xv[MS][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int ss_ = min(s0 + s, steps - 1);
      wv[s] = *(const u32x4 *)(wrow + 32 * ss_);
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
        xv[ms][s] = buf_load16(xr, xoff[ms] == BUF_OOB ? BUF_OOB : xoff[ms] + 64u * ss_);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if (s0 + s < steps) {
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) acc[ms] = mfma_bf16_16x16x32(xv[ms][s], wv[s], acc[ms]);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const float lo = __uint_as_float(wv[s][d] << 16), hi = __uint_as_float(wv[s][d] & 0xFFFF0000u);
          ss = __builtin_fmaf(lo, lo, ss);
          ss = __builtin_fmaf(hi, hi, ss);
        }
      }
    }
  }
  // partial logits: lane (q, n) holds tokens 4q+r of each m-subtile, expert n
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave * (MS * 256) + ms * 256 + (4 * q + r) * 16 + n] = acc[ms][r];
  ss += __shfl_xor(ss, 16, 64);
  ss += __shfl_xor(ss, 32, 64);
  float *nred = red + NW * MS * 256;
  if (q == 0) nred[wave * 16 + n] = ss;
  __syncthreads();
  for (int idx = threadIdx.x; idx < MS * 256; idx += blockDim.x) {
    const int ms = idx >> 8, cell = idx & 255;
    const int t = t0 + 16 * ms + (cell >> 4), ee = e0 + (cell & 15);
    if (t >= T || ee >= E) continue;
    float v = 0.0f;
    for (int w = 0; w < NW; ++w) v += red[w * (MS * 256) + idx];
    approx[(size_t)t * E + ee] = bias ? v + bias[ee] : v;
  }
  if (blockIdx.y == 0 && threadIdx.x < 16 && e0 + (int)threadIdx.x < E) {
    float v = 0.0f;
    for (int w = 0; w < NW; ++w) v += nred[w * 16 + threadIdx.x];
    wnorm[e0 + threadIdx.x] = sqrtf(v);
  }
}

// ---------------------------------------------------------------------------
// Canonical dots of 4 router rows with x in registers (lane l holds chunks l,
// l + 64, ...): per lane sequential fma in chunk order, then the xor butterfly
// 32, 16, ..., 1 of every row.  All rows' loads are issued before any math.  The
// butterfly halves the values at 32 and 16 (permlane swaps: lanes 16 b .. 16 b +
// 15 end with row b) and goes on inside the 16 lanes on the DPP path, 7 steps for
// the 4 rows where 24 ds_bpermutes did the same additions.  Returns row lane / 16.
// ---------------------------------------------------------------------------
constexpr int SEL_NB = 4;
template <int CH>
__device__ __forceinline__ float canon_dot4(const u32x4 (&xc)[CH], const uint16_t *const (&w)[SEL_NB],
                                            int lane, int nch) {
  u32x4 wv[SEL_NB][CH];
#pragma unroll
  for (int b = 0; b < SEL_NB; ++b)
#pragma unroll
    for (int j = 0; j < CH; ++j)
      wv[b][j] = *(const u32x4 *)(w[b] + (size_t)min(lane + 64 * j, nch - 1) * 8);
  float v[SEL_NB];
#pragma unroll
  for (int b = 0; b < SEL_NB; ++b) v[b] = 0.0f;
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    if (lane + 64 * j < nch) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float lo = __uint_as_float(xc[j][d] << 16), hi = __uint_as_float(xc[j][d] & 0xFFFF0000u);
#pragma unroll
        for (int b = 0; b < SEL_NB; ++b) {
          v[b] = __builtin_fmaf(lo, __uint_as_float(wv[b][j][d] << 16), v[b]);
          v[b] = __builtin_fmaf(hi, __uint_as_float(wv[b][j][d] & 0xFFFF0000u), v[b]);
        }
      }
    }
  }
  HalveSum<4, 32>::step(v, lane);
  HalveSum<2, 16>::step(v, lane);
  float r = v[0];
  auto mov = [](float f, auto ctrl, auto bank) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(f), __float_as_int(f),
                                                      decltype(ctrl)::value, 0xF,
                                                      decltype(bank)::value, false));
  };
  using std::integral_constant;
  r = r + mov(r, integral_constant<int, 0x128>(), integral_constant<int, 0xF>());  // row_ror 8: xor 8
  // xor 4: row_shl 4 (lane l takes l + 4) into the even quads, row_shr 4 into the odd ones
  const float up = mov(r, integral_constant<int, 0x104>(), integral_constant<int, 0x5>());
  const float dn = mov(r, integral_constant<int, 0x114>(), integral_constant<int, 0xA>());
  r = r + ((lane & 4) ? dn : up);
  r = r + mov(r, integral_constant<int, 0x4E>(), integral_constant<int, 0xF>());  // xor 2
  r = r + mov(r, integral_constant<int, 0xB1>(), integral_constant<int, 0xF>());  // xor 1
  return r;
}

constexpr int SEL_WAVES = 4;
constexpr int SEL_COOP_MAX_T = 1024;

// One wave per token, SEL_WAVES tokens per workgroup; or COOP (up to
// SEL_COOP_MAX_T, where one wave per token leaves most of the chip idle and a
// token's latency is the kernel's): one token per workgroup.  Wave 0 takes the
// approximate top-k and the candidate list, wave 1 writes the MFMA-order copy of
// x, and the candidates' canonical dots and the shared gate's are shared by all
// waves (E512 H2048 k10: T512 16.5 us by one wave per token, 9.5 COOP; T1500 17.1
// and 18.8).
// Bound by the latency of its serial parts at few tokens, by the reads of (k + 1)
// router rows per token through the L2s at many.  With one shuffle chain per row,
// the gate's dot on its own, x re-read after the top-k and lists of 1024 entries
// (3 workgroups per CU): T64 17.3 us, T512 16.5, T1500 19.9, T4096 39; H4096 T4096
// 105.  Now 14.4, 9.4, 17.0, 25.8 and 57.6.
//
// LATE_X (more than 512 experts, 1024 < H <= 2048, one wave per token): the row
// and the norms are loaded after the approximate top-k.  Held through it they take
// 13 VGPRs more than the 128 of 4 waves per SIMD; whole route, E1024 H2048 k8,
// spilled / with 3 waves / so: T2048 36.6, 34.1, 33.6 us, T4096 52.6, 54.3, 48.7
// (E700 H1536: T4096 38.9, 40.6, 35.1).
template <int NV, int CH, bool COOP>
__global__ __launch_bounds__(256, CH <= 4 ? 4 : 2) void k_select(const float *__restrict__ approx,
                                                const float *__restrict__ wnorm,
                                                const uint16_t *__restrict__ x,
                                                const uint16_t *__restrict__ rw,
                                                const float *__restrict__ bias,
                                                const uint16_t *__restrict__ gw,
                                                int32_t *__restrict__ topk_idx,
                                                float *__restrict__ topk_w,
                                                float *__restrict__ sgate,
                                                uint16_t *__restrict__ xperm,
                                                float *__restrict__ xsum, W8Rows w8, int T, int E,
                                                int k, int H, int has_shared, DispatchOut ds,
                                                int fused, unsigned long long *cmask,
                                                int32_t *ccount) {
  // candidate lists (E <= 64 NV)
  constexpr int LISTS = COOP ? 1 : SEL_WAVES;
  constexpr bool LATE_X = NV > 8 && CH == 4 && !COOP;
  __shared__ int cl[LISTS][64 * NV];
  __shared__ float cv[LISTS][64 * NV + 1];  // and the shared gate's dot
  __shared__ uint64_t s_cand[LISTS][64];
  __shared__ uint64_t s_sel[LISTS][16];
  __shared__ int s_nc;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t = COOP ? (int)blockIdx.x : (int)blockIdx.x * SEL_WAVES + wave;
  const int sw = COOP ? 0 : wave;  // this wave's LDS lists
  const bool lead = !COOP || wave == 0;
  if (t < T) {
    // the routing's loads first, then the MFMA-order copy of x (and its group
    // sums), which does not depend on it: its latency hides under the selection
    STRACE(0);
    const float *ar = approx + (size_t)t * E;
    const uint16_t *xrow = x + (size_t)t * H;
    const int nch = H >> 3;
    uint32_t key[NV];
    float av[NV], wn = 0.0f;
    u32x4 xc[CH];  // the x row in registers (canonical chunk layout)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = min(lane + 64 * i, E - 1);  // unconditional: loads issue together
      av[i] = lead ? ar[e] : 0.0f;
      if (!LATE_X) wn = fmaxf(wn, lead ? wnorm[e] : 0.0f);
    }
    auto load_x = [&]() {
#pragma unroll
      for (int j = 0; j < CH; ++j)
        xc[j] = *(const u32x4 *)(xrow + (size_t)min(lane + 64 * j, nch - 1) * 8);
    };
    if (!LATE_X) load_x();
    if ((xperm || w8.q) && (!COOP || wave == 1))
      write_xperm(xrow, xperm, xsum, t, H, lane, nullptr, 1.0f, w8.q, w8.s, w8.sum);
    STRACE(1);
    // ---- k-th largest approximate logit -------------------------------
#pragma unroll
    for (int i = 0; i < NV; ++i) key[i] = lane + 64 * i < E ? ordered_key(av[i]) : 0u;
    int seli = 0;
    uint32_t selk = 0u;
    if (lead) wave_topk_fast<NV>(key, E, k, lane, seli, selk, s_cand[sw], s_sel[sw]);
    STRACE(2);
    if (LATE_X) {
      load_x();
#pragma unroll
      for (int i = 0; i < NV; ++i) wn = fmaxf(wn, wnorm[min(lane + 64 * i, E - 1)]);
    }
    const uint32_t kth = (uint32_t)__builtin_amdgcn_readlane((int)selk, k - 1);
    float selv = 0.0f, sgv = 0.0f;
    {
      // ---- the row's norm (a bound: any order of the additions) -----------
      float xs = 0.0f;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        if (lane + 64 * j < nch) {
#pragma unroll
          for (int d = 0; d < 4; ++d) {
            const float lo = __uint_as_float(xc[j][d] << 16), hi = __uint_as_float(xc[j][d] & 0xFFFF0000u);
            xs = __builtin_fmaf(lo, lo, xs);
            xs = __builtin_fmaf(hi, hi, xs);
          }
        }
      }
      xs = row16_sum(xs);
      xs += __shfl_xor(xs, 16, 64);
      xs += __shfl_xor(xs, 32, 64);
      wn = __uint_as_float(wave_max_u32(__float_as_uint(wn)));  // norms: not negative
      // ---- candidate threshold --------------------------------------------
      const float lk = key_to_float(kth);
      const float nrm = sqrtf(xs) * wn * 1.0625f;
      const float d = 2.0f * (float)(H + 64) * 0x1p-23f * nrm;  // |approx - canonical|
      const float thr = lk - 2.0f * d - 0x1p-21f * (fabsf(lk) + 2.0f * d) - 1e-30f * (float)H;
      // ---- candidate list, expert-ascending -------------------------------
      int nc = 0;
      if (lead) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int e = lane + 64 * i;
          const bool c = e < E && key_to_float(key[i]) >= thr;
          const uint64_t b = __ballot(c);
          if (c) cl[sw][nc + __popcll(b & ((1ull << lane) - 1ull))] = e;
          nc += __popcll(b);
        }
        if (COOP && lane == 0) s_nc = nc;
      }
      __builtin_amdgcn_wave_barrier();
      if (COOP) {
        __syncthreads();
        nc = s_nc;
      }
      STRACE(3);
      // ---- canonical logits of the candidates, and the shared gate's -------
      {
        const int nr = nc + (gw ? 1 : 0), cstep = COOP ? SEL_WAVES * SEL_NB : SEL_NB;
        for (int c0 = COOP ? wave * SEL_NB : 0; c0 < nr; c0 += cstep) {
          const uint16_t *rows[SEL_NB];
#pragma unroll
          for (int b = 0; b < SEL_NB; ++b) {
            const int c = min(c0 + b, nr - 1);
            const int e = __builtin_amdgcn_readfirstlane(cl[sw][max(min(c, nc - 1), 0)]);
            rows[b] = c < nc ? rw + (size_t)e * H : gw;
          }
          const float v = canon_dot4<CH>(xc, rows, lane, nch);
          const int c = c0 + (lane >> 4);
          if ((lane & 15) == 0 && c < nr) cv[sw][c] = bias && c < nc ? v + bias[cl[sw][c]] : v;
        }
      }
      __builtin_amdgcn_wave_barrier();
      if (COOP) __syncthreads();
      STRACE(4);
      // ---- top-k among candidates (value desc, expert asc) ----------------
      if (!lead) {
        // helper waves are done
      } else if (nc < k) {
        // NaN in the row, the router or its norms: no threshold.  The
        // approximate selection stands (valid experts).
        selv = key_to_float(selk);
      } else if (nc <= 64 && k <= 16) {
        // rank of each candidate = candidates above it (unique composite keys)
        auto comp = [&](int i) {
          return ((uint64_t)ordered_key(cv[sw][i]) << 32) | (uint32_t)~(uint32_t)cl[sw][i];
        };
        const uint64_t mine = lane < nc ? comp(lane) : 0ull;
        int rk = 0;
        for (int j = 0; j < nc; ++j) rk += readlane_u64(mine, j) > mine ? 1 : 0;
        if (lane < nc && rk < k) s_sel[sw][rk] = ((uint64_t)(uint32_t)lane << 32) | (uint32_t)cl[sw][lane];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < k) {
          const uint64_t pk = s_sel[sw][lane];
          seli = (int)(uint32_t)pk;
          selv = cv[sw][(int)(pk >> 32)];
        }
      } else {
      uint32_t tmask = 0;  // taken bits per lane slot (nc <= 1024: 16 slots)
      for (int j = 0; j < k; ++j) {
        uint32_t bk = 0;
        int bs = 0x7FFFFFFF;
        for (int i = 0; i < 16 && lane + 64 * i < nc; ++i) {
          const uint32_t kk = ordered_key(cv[sw][lane + 64 * i]);
          if (!(tmask & (1u << i)) && (bs == 0x7FFFFFFF || kk > bk)) {
            bk = kk;
            bs = lane + 64 * i;
          }
        }
        const uint32_t wk = wave_max_u32(bk);
        const int ws = (int)wave_min_u32(bk == wk && bs != 0x7FFFFFFF ? (uint32_t)bs : 0xFFFFFFFFu);
        if ((ws & 63) == lane) tmask |= 1u << (ws >> 6);
        if (lane == j) {
          seli = cl[sw][ws];
          selv = cv[sw][ws];
        }
      }
      }
      STRACE(5);
      if (gw) sgv = cv[sw][nc];
      STRACE(6);
    }
    if (lead) {
      const float vmax = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(selv), 0));
      const float p = lane < k ? expf(selv - vmax) : 0.0f;
      float sum = 0.0f;
      for (int j = 0; j < k; ++j)
        sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), j));
      if (lane < k) {
        topk_idx[(size_t)t * k + lane] = seli;
        topk_w[(size_t)t * k + lane] = p / sum;
        // the dispatch's count and token mask of (64-token chunk, expert):
        // a sum and an OR over the chunk's picks, so the order of the
        // atomics does not matter (the counts sit just before the masks)
        if (cmask) {
          const size_t ce = (size_t)(t >> 6) * E + seli;
          atomicOr(cmask + ce, 1ull << (t & 63));
          atomicAdd(ccount + ce, 1);
        }
      }
      // ---- shared gate --------------------------------------------------
      float g = 1.0f;
      if (gw) g = 1.0f / (1.0f + expf(-sgv));
      if (lane == 0) sgate[t] = g;
    }
    STRACE(7);
  }
  if constexpr (!COOP) return;
  if (!fused) return;
  // ---- the last block runs the dispatch ---------------------------------
  __shared__ int is_last;
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    is_last = atomicAdd(ds.ticket, 1) == (int)gridDim.x - 1;
  }
  __syncthreads();
  if (!is_last) return;
  __threadfence();
  if (threadIdx.x == 0) atomicExch(ds.ticket, 0);
  dispatch_small_block(topk_idx, T, k, E, has_shared, ds);
}

template <int NV, bool COOP>
hipError_t launch_select_nv(int ch, unsigned grid, const float *approx, const float *wnorm,
                            const void *x, const void *rw, const float *bias, const void *gw,
                            int32_t *idx, float *w, float *sg, void *xperm, float *xsum, W8Rows w8, int T,
                            int E, int k, int H, int has_shared, const DispatchOut &ds, int fused,
                            unsigned long long *cmask, int32_t *ccount, hipStream_t s) {
#define SEL_ARGS                                                                            \
  approx, wnorm, (const uint16_t *)x, (const uint16_t *)rw, bias, (const uint16_t *)gw, idx, \
      w, sg, (uint16_t *)xperm, xsum, w8, T, E, k, H, has_shared, ds, fused, cmask, ccount
  switch (ch) {
  case 1: k_select<NV, 1, COOP><<<grid, 256, 0, s>>>(SEL_ARGS); break;
  case 2: k_select<NV, 2, COOP><<<grid, 256, 0, s>>>(SEL_ARGS); break;
  case 4: k_select<NV, 4, COOP><<<grid, 256, 0, s>>>(SEL_ARGS); break;
  default: k_select<NV, 8, COOP><<<grid, 256, 0, s>>>(SEL_ARGS); break;
  }
#undef SEL_ARGS
  return hipGetLastError();
}

}  // namespace

bool router_supported(int H, int E) { return H % 128 == 0 && H <= 4096 && E <= 1024; }

hipError_t launch_select(const float *approx, const float *wnorm,
                         const void *x, const void *rw, const float *bias, const void *gw,
                         int32_t *idx, float *w, float *sg, void *xperm, float *xsum, W8Rows w8, int T,
                         int H, int E, int k, int has_shared, const DispatchOut *fused,
                         hipStream_t s, unsigned long long *cmask = nullptr,
                         int32_t *ccount = nullptr) {
  const int ch = (H / 8 + 63) / 64;  // chunks per lane
  const int chp = ch <= 1 ? 1 : (ch <= 2 ? 2 : (ch <= 4 ? 4 : 8));
  const int nv = (E + 63) / 64;
  DispatchOut ds;
  memset(&ds, 0, sizeof ds);
  if (fused) ds = *fused;
  // one token per workgroup (k_select, COOP; it alone runs the fused dispatch)
  if (fused && T > SEL_COOP_MAX_T) return hipErrorInvalidValue;
  const bool coop = T <= SEL_COOP_MAX_T;
  const unsigned g = coop ? (unsigned)T : (T + SEL_WAVES - 1) / SEL_WAVES;
  const int fz = fused ? 1 : 0;
#define SEL_CALL(NVV)                                                                          \
  (coop ? launch_select_nv<NVV, true>(chp, g, approx, wnorm, x, rw, bias, gw, idx, \
                                              w, sg, xperm, xsum, w8, T, E, k, H, has_shared, ds, \
                                              fz, cmask, ccount, s)                           \
        : launch_select_nv<NVV, false>(chp, g, approx, wnorm, x, rw, bias, gw, idx, \
                                              w, sg, xperm, xsum, w8, T, E, k, H, has_shared, ds, \
                                              fz, cmask, ccount, s))
  if (nv <= 1) return SEL_CALL(1);
  if (nv <= 2) return SEL_CALL(2);
  if (nv <= 4) return SEL_CALL(4);
  if (nv <= 8) return SEL_CALL(8);
  return SEL_CALL(16);
#undef SEL_CALL
}

hipError_t launch_router_fast(const void *x, const void *rw, const float *bias, const void *gw,
                              float *approx, float *wnorm, int32_t *idx, float *w, float *sg,
                              void *xperm, float *xsum, int T, int H, int E, int k,
                              int has_shared, const DispatchOut *fused, hipStream_t s,
                              int32_t *ccount, unsigned long long *cmask, W8Rows w8) {
  if (T == 0) return hipSuccess;
  // ---- approximate logits + row norms ------------------------------------
  if (T >= GEMM_MIN_T) {
    // (and the chunk counts and masks zeroed: [ccount, cmask end), which
    // k_select fills for the dispatch)
    const size_t zb = cmask ? (size_t)((char *)(cmask + (size_t)((T + 63) / 64) * E) - (char *)ccount) : 0;
    hipError_t err = launch_router_gemm(x, rw, bias, approx, wnorm, T, H, E, (uint32_t *)ccount,
                                        (int)(zb / 4), s);
    if (err != hipSuccess) return err;
    return launch_select(approx, wnorm, x, rw, bias, gw, idx, w, sg, xperm,
                                xsum, w8, T, H, E, k, has_shared, fused, s, cmask, ccount);
  }
  // one 16-token tile per workgroup: more workgroups share the token reads
  // (c3 T=64: 55 -> 44 us against 64-token tiles; the router rows are
  // re-read from L2)
  constexpr int MS = 1;
  const int mt = 16 * MS;
  // decode: one token tile, K split over up to 16 waves; prefill: 4 waves
  int NW = T <= 64 ? H / 128 : 4;
  if (NW > 16) NW = 16;
  while (NW > 1 && (H % (32 * NW))) --NW;
  const dim3 grid((E + 15) / 16, (T + mt - 1) / mt);
  const size_t lds = sizeof(float) * ((size_t)NW * MS * 256 + NW * 16);
  k_router_mfma<MS><<<grid, NW * 64, lds, s>>>((const uint16_t *)x, (const uint16_t *)rw, bias,
                                               approx, wnorm, fused ? fused->ticket : nullptr, T,
                                               H, E, NW);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  // ---- refine + select ------------------------------------------------------
  return launch_select(approx, wnorm, x, rw, bias, gw, idx, w, sg, xperm, xsum,
                              w8, T, H, E, k, has_shared, fused, s);
}
