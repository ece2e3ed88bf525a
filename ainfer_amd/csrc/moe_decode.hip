// moe_decode.hip - the decode routing kernel (T <= 16 tokens), the down + combine
// kernel (down_combine_at: T = 1, and up to 4 tokens with at most 1024
// intermediate columns) and the fused expert kernel (T = 2 beyond that, where
// decode_geometry allows it).
//
// Measured on MI355X: a dependent kernel launch costs about 2.5 us, a flag
// handed from one workgroup to another through device memory about 0.8 us,
// same-address device atomics serialise at about 11 ns each, and an
// agent-scope release or acquire fence (a whole-L2 write-back or
// invalidate) about 20 ns, serialised.  So what meets inside a kernel meets
// through slots and counters that few workgroups touch, with data handed over by
// sc1 stores and loads instead of fences (moe_common.h):
//
//  k_route_decode   workgroups [0, NR): canonical router logits, one
//                   (one row x 1 or 2 tokens) unit per wave, each stored
//                   with an sc1 store as ~bits into a key slot of the sync
//                   region (never 0: the NaN 0xFFFFFFFF, which no bf16
//                   product or sum yields but a router bias may hold, is
//                   stored as 0xFFFFFFFE); workgroup NR (one wave per token)
//                   polls its token's slots
//                   until none is 0, clears them, takes the exact top-k, the
//                   weights and the shared gate, and builds the dispatch
//                   (tiles of at most DEC_MT tokens) from LDS.  A slot that is
//                   its own ready flag saves the store wait, barrier and
//                   counter round trip of an arrival.  Workgroup NR + 1
//                   writes x in MFMA order meanwhile.
//  k_experts_decode one workgroup per item: first every gate/up + SiLU item
//                   (tile-major, slab-minor), one arrival each on
//                   gu_done[tile]; then every down item, which requests its
//                   weights, waits for gu_done[tile] == gate/up slabs, reads
//                   the tile's act rows, writes its o rows, and counts one
//                   arrival per (token, row slab).  The (k+1)-th arrival of a
//                   (token, slab) sums the token's k + 1 rows of that slab in
//                   slot order (the combine).
//
//  k_down_combine   after the gate/up items (k_expert_lds, a launch of their
//                   own): each workgroup owns 8 or 16 output rows of every
//                   selected expert, so the combine is an LDS exchange and no
//                   counter is needed.
// Every other call runs k_expert_lds twice and k_combine.
//
// A wait only ever names work of lower workgroup index, and workgroups are
// dispatched in index order, so every awaited workgroup is already running.
// Waits are bounded (SPIN_MAX polls); one that runs out sets the error word
// of the sync region and carries on.  The error word is sticky: while it is
// set, every combine (this kernel's and k_combine) writes NaN outputs, so a
// call whose handoff failed, and every later call on that workspace until
// ainfer_moe_workspace_init clears it, returns visibly bad rows rather than
// silently wrong ones (a late arrival can leave a counter non-zero, which
// would let a later call's waits pass early).
//
// Every counter is reset by its last user (the logit slots by the selection
// workgroup, gu_done/dn_done by a tile's last down item, a (token, slab)
// counter by its last arrival), so the sync region is zero again when a call
// ends.  It must be zero before the first call (ainfer_moe_workspace_init).
//
// Debug builds with -DAINFER_DECODE_TRACE record per-workgroup timestamps.
#include <string.h>

#include <type_traits>

#include "moe_common.h"
#include "moe_expert_item.h"
#include "moe_internal.h"
#include "moe_topk.h"
#include "moe_decode_parts.h"

#ifdef AINFER_DECODE_TRACE
// debug builds only: per-workgroup timestamps (s_memrealtime, 100 MHz)
__device__ unsigned long long g_dtrace[2][1 << 15][5];
#define DTRACE_AT(K, X, I) \
  if (threadIdx.x == 0 && (X) < (1 << 15)) g_dtrace[K][X][I] = __builtin_amdgcn_s_memrealtime()
#define DTRACE(K, I) DTRACE_AT(K, blockIdx.x, I)
extern "C" int ainfer_debug_trace(void *host) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_dtrace), sizeof(g_dtrace)) == hipSuccess ? 0 : -1;
}
extern "C" int ainfer_debug_land(void *host) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_dland), sizeof(g_dland)) == hipSuccess ? 0 : -1;
}
#else
#define DTRACE(K, I)
#define DTRACE_AT(K, X, I)
#endif

namespace {

constexpr int RD_WAVES = 16;  // waves per k_route_decode workgroup
// Router units: one router row x TT tokens per wave (TT = 1 up to
// RD_TT1_MAX tokens, else 2: more, shorter units shorten the routing at few
// tokens; measured at T = 1, 4, 16 against 2 rows x 4 tokens: -2.9, -3.4,
// -0.5 us per layer).  At TT = 1 the workgroups have RD_W1 waves and a lane
// issues the loads of its whole row at once (c3 T=1: -1 us).
constexpr int RD_R = 1;       // router rows per wave
constexpr int RD_TT1_MAX = 4;
constexpr int RD_NB = 2;      // 8-element chunks per lane whose loads are issued together
#ifndef RD_W1
#define RD_W1 4    // waves per workgroup at T <= RD_TT1_MAX (the rows spread over more CUs)
#endif
#ifndef RD_NB1
#define RD_NB1 8   // chunks in flight at T <= RD_TT1_MAX: a whole row up to H = 4096
#endif
// RD_TT1_MAX < T <= RD_W2: two tokens per wave in workgroups of RD_W2 waves
// with RD_NB2 chunks in flight, so the 2048 units of c4 T=8 spread over all
// CUs instead of half of them (16-wave workgroups, which T > RD_W2 needs for
// its one selection wave per token).  c4 T=8 routing stage 13.8 -> 12.2 us
// per block; one token per wave in 8-wave workgroups: 12.4 us.
#ifndef RD_W2
#define RD_W2 8
#endif
#ifndef RD_NB2
#define RD_NB2 4
#endif
#ifndef RD_MID_TT
#define RD_MID_TT 2
#endif
static_assert(RD_W1 >= RD_TT1_MAX, "the selection runs one wave per token");
static_assert(DECODE_NORM_MAX_T <= RD_TT1_MAX, "the folded RMSNorm exists in the TT = 1 form only");
constexpr int SPIN_MAX = 1 << 20;
#ifndef DEC_WAVES_PER_SIMD
#define DEC_WAVES_PER_SIMD 6  // register budget of the expert kernel (<= 80 VGPRs)
#endif
#ifndef DEC_NW_MIN
#define DEC_NW_MIN 4  // waves per expert workgroup (at least)
#endif
#ifndef DEC_RG_GU
#define DEC_RG_GU 1  // 16-row groups per wave, gate/up items (16 x 2 rows x H)
#endif
#ifndef DEC_RG_DN
#define DEC_RG_DN 2  // 16-row groups per wave, down items
#endif

struct RouteDecodeArgs {
  const uint16_t *x, *rw, *gw;
  const float *bias;
  float *logits, *sgl;  // [T][E], [T]
  int32_t *idx;
  float *w, *sg;
  uint16_t *xperm;
  W8Rows w8;        // optional: W4A8 rows of the (normalized) x (sum null: natural order)
  DispatchOut ds;
  int32_t *sync;
  uint32_t *slots;  // [DECODE_MAX_T][E + 1] ~bits of the logits (sync region)
  NormIn norm;      // on: x is the residual stream, normalized here (RMSNorm)
  int T, H, E, k, has_shared, NR;
  int spin;         // polls before a wait gives up (0: at once)
};

// W waves per workgroup (T <= W: the selection runs one wave per token), NB
// chunks of 8 per lane whose loads are issued together
// NORM: x is the residual stream and the block's RMSNorm is applied here
// (T <= RD_TT1_MAX only: at two tokens per wave the extra registers cost
// more than the saved launch)
template <int NV, int RD_TT, int W, int NB, bool NORM>
__global__ __launch_bounds__(W * 64) void k_route_decode(RouteDecodeArgs a) {
  __shared__ uint64_t s_cand[W][68];
  __shared__ uint64_t s_sel[W][16];
  __shared__ int s_idx[W * 32];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int T = a.T, H = a.H, E = a.E, k = a.k;
  DTRACE(0, 0);
  if ((int)blockIdx.x < a.NR) {
    // ---- canonical logits of RD_R rows x RD_TT tokens per wave: lane l
    // sums 8-element chunks l, l+64, ... with fma in order, then the xor
    // butterfly (the oracle's mo_router_dot) ---------------------------------
    const int nrows = E + (a.gw ? 1 : 0);
    const int ngroups = (nrows + RD_R - 1) / RD_R;
    const int u = blockIdx.x * W + wave;
    const int rbase = (u % ngroups) * RD_R, t0 = (u / ngroups) * RD_TT;
    if (t0 < T) {
      const uint16_t *wr[RD_R];
#pragma unroll
      for (int i = 0; i < RD_R; ++i) {
        const int r = min(rbase + i, nrows - 1);
        wr[i] = r < E ? a.rw + (size_t)r * H : a.gw;
      }
      const int nch = H >> 3;
      // RMSNorm folded in: each token's scale from the x chunks the loop
      // below loads (the whole row: one pass, H <= 64 * NB * 8), then x
      // normalized per chunk
      static_assert(!NORM || 64 * NB * 8 >= 4096, "the folded RMSNorm needs the whole row");
      float inv[RD_TT];
#pragma unroll
      for (int j = 0; j < RD_TT; ++j) inv[j] = 1.0f;
      float acc[RD_R][RD_TT];
#pragma unroll
      for (int i = 0; i < RD_R; ++i)
#pragma unroll
        for (int j = 0; j < RD_TT; ++j) acc[i][j] = 0.0f;
      // NB chunks' loads in flight at once; the sums still run over
      // chunks l, l + 64, ... in order
      // (every lane takes part, H < 512 included: the RMSNorm's wave reductions
      // read all 64)
      for (int cb = lane; cb - lane < nch; cb += 64 * NB) {
        u32x4 wv[NB][RD_R], xv[NB][RD_TT], nv[NB];
        // x and the norm weight first: loads complete in issue order, so the
        // RMSNorm (which needs only them) runs while the router row, a cold
        // read from HBM, is still in flight
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int c = min(cb + 64 * b, nch - 1);
#pragma unroll
          for (int j = 0; j < RD_TT; ++j)
            xv[b][j] = *(const u32x4 *)(a.x + (size_t)min(t0 + j, T - 1) * H + (size_t)c * 8);
          nv[b] = NORM && a.norm.w ? *(const u32x4 *)(a.norm.w + (size_t)c * 8)
                                   : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int c = min(cb + 64 * b, nch - 1);
#pragma unroll
          for (int i = 0; i < RD_R; ++i) wv[b][i] = *(const u32x4 *)(wr[i] + (size_t)c * 8);
        }
        if constexpr (NORM) {
          // sum of squares in any order (rms_mean_f's tests hold for every
          // order), four independent fp64 chains per lane
#pragma unroll
          for (int j = 0; j < RD_TT; ++j) {
            double p4[4] = {0.0, 0.0, 0.0, 0.0};
            u16x2_t ek = {0x7F80, 0x7F80};
#pragma unroll
            for (int b = 0; b < NB; ++b)
              if (cb + 64 * b < nch) sumsq_chunk(xv[b][j], p4, ek);
            int emin = ek_emin(ek);
            // wave reductions on the DPP path (no LDS round trips on this
            // critical path); one value in every lane
            const double tot = wave_sum_f64((p4[0] + p4[1]) + (p4[2] + p4[3]));
            emin = (int)wave_min_u32((uint32_t)emin);
            inv[j] = rms_inv_finish(tot, emin, a.x + (size_t)min(t0 + j, T - 1) * H, H,
                                    a.norm.eps, lane);
          }
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int j = 0; j < RD_TT; ++j)
#pragma unroll
              for (int q = 0; q < 4; ++q) xv[b][j][q] = norm_pair(xv[b][j][q], nv[b][q], inv[j], a.norm);
          DTRACE(0, 2);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          // past the row end: computed on a clamped chunk and discarded, so
          // no load depends on a branch
          const bool in = cb + 64 * b < nch;
#pragma unroll
          for (int i = 0; i < RD_R; ++i)
#pragma unroll
            for (int j = 0; j < RD_TT; ++j) {
              float s = acc[i][j];
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                s = __builtin_fmaf(__uint_as_float(xv[b][j][q] << 16), __uint_as_float(wv[b][i][q] << 16), s);
                s = __builtin_fmaf(__uint_as_float(xv[b][j][q] & 0xFFFF0000u),
                                   __uint_as_float(wv[b][i][q] & 0xFFFF0000u), s);
              }
              acc[i][j] = in ? s : acc[i][j];
            }
        }
      }
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1)
#pragma unroll
        for (int i = 0; i < RD_R; ++i)
#pragma unroll
          for (int j = 0; j < RD_TT; ++j) acc[i][j] = acc[i][j] + __shfl_xor(acc[i][j], m, 64);
      DTRACE(0, 3);
      if (lane == 0) {
#pragma unroll
        for (int i = 0; i < RD_R; ++i)
#pragma unroll
          for (int j = 0; j < RD_TT; ++j) {
            const int r = rbase + i, t = t0 + j;
            if (r >= nrows || t >= T) continue;
            const float v = r < E && a.bias ? acc[i][j] + a.bias[r] : acc[i][j];
            // never 0, which the selection polls away: the one NaN whose ~bits
            // are 0 is stored as its neighbour
            st_dev(a.slots + (size_t)t * (E + 1) + r, max(~__float_as_uint(v), 1u));
          }
      }
    }
    DTRACE(0, 1);
    return;
  }
  const int t = wave;
  if ((int)blockIdx.x > a.NR) {
    // ---- workgroup NR + 1: the MFMA-order copy of x, one wave per token.
    // It does not depend on the routing; a workgroup of its own keeps it off
    // the selection's path (the selection polls as soon as it starts).
    if (t < T && (a.xperm || a.w8.q)) {
      const float inv = NORM ? row_rms_inv(a.x + (size_t)t * H, H, a.norm.eps, lane) : 1.0f;
      write_xperm(a.x + (size_t)t * H, a.xperm, nullptr, t, H, lane, NORM ? &a.norm : nullptr, inv,
                  a.w8.q, a.w8.s, a.w8.sum);
    }
    return;
  }
  // ---- the selection workgroup (NR): one wave per token (T <= W) ----------
  uint32_t raw[NV], graw = 0u;
  if (t < T) {
    uint32_t *sl = a.slots + (size_t)t * (E + 1);
    // poll the token's slots until every one is written (bounded)
    for (int it = 0;; ++it) {
#pragma unroll
      for (int i = 0; i < NV; ++i) raw[i] = ld_dev(sl + min(lane + 64 * i, E - 1));
      graw = ld_dev(sl + E);  // the shared gate's slot (stays 0 without one)
      uint32_t nz = graw | (a.gw ? 0u : 1u);
#pragma unroll
      for (int i = 0; i < NV; ++i) nz = min(nz, raw[i]);
      if (a.spin > 0 && __all(nz != 0u)) break;
      if (it >= a.spin) {
        if (lane == 0) atomicOr(a.sync + SY_ERR, 1);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    DTRACE(0, 4);
    uint32_t key[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) key[i] = lane + 64 * i < E ? ordered_key(__uint_as_float(~raw[i])) : 0u;
    const float sgl = __uint_as_float(~graw);
    int seli;
    uint32_t selk;
    wave_topk_fast<NV>(key, E, k, lane, seli, selk, s_cand[wave], s_sel[wave]);
    DTRACE(0, 1);
    const float selv = lane < k ? key_to_float(selk) : 0.0f;
    const float vmax = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(selv)));
    const float p = lane < k ? expf(selv - vmax) : 0.0f;
    float sum = 0.0f;  // in pick order, as the oracle
    for (int j = 0; j < k; ++j) sum += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), j));
    if (lane < k) {
      a.idx[(size_t)t * k + lane] = seli;
      a.w[(size_t)t * k + lane] = p / sum;
      s_idx[t * k + lane] = seli;
    }
    if (lane == 0) a.sg[t] = a.gw ? 1.0f / (1.0f + expf(-sgl)) : 1.0f;
  }
  DTRACE(0, 2);
  __syncthreads();
  if (a.ds.tiles) dispatch_decode<W>(s_idx, T, k, E, a.has_shared, a.ds);
  DTRACE(0, 3);
  // off the critical path: the logits output, and the slots cleared for
  // the next call
  if (t < T) {
    uint32_t *sl = a.slots + (size_t)t * (E + 1);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int e = lane + 64 * i;
      if (e < E) {
        st_dev(sl + e, 0u);
        a.logits[(size_t)t * E + e] = __uint_as_float(~raw[i]);
      }
    }
    if (a.gw && lane == 0) {
      st_dev(sl + E, 0u);
      a.sgl[t] = __uint_as_float(~graw);
    }
  }
}

struct ExpertsDecodeArgs {
  ExpertArgs gu, dn;  // WK, WR, n_slabs set (WK * WR waves in both)
  const float *w, *sg;
  const int32_t *inv;
  const uint16_t *resid;
  uint16_t *y;
  int32_t *sync;
  int max_tiles, cap;  // grid tiles; capacity of the per-tile counter arrays
  int spin;            // polls before a wait gives up (0: at once)
};

// One item per workgroup.  A down item only ever waits for gate/up items of
// lower index, which the dispatcher has started, so the waits end.
template <int SD, int KBW_GU, int RG_GU, int KBW_DN, int RG_DN>
__global__ __launch_bounds__(1024, DEC_WAVES_PER_SIMD) void k_experts_decode(ExpertsDecodeArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  // one counter per 256-byte line: same-line atomics and polls serialise
  int32_t *gu_done = a.sync + SY_TILES, *dn_done = gu_done + a.cap * SY_STRIDE,
          *cnt = dn_done + a.cap * SY_STRIDE;
  const int lane = threadIdx.x & 63;
  const int sg = a.gu.n_slabs, sd = a.dn.n_slabs;
  const int n_gu = a.max_tiles * sg;
  {
    const int item = blockIdx.x;
    // ---- item -> (kind, tile, slab): all gate/up items (tile-major,
    // slab-minor), then all down items ---------------------------------------
    const int is_gu = item < n_gu;
    const int r = is_gu ? item : item - n_gu, ns = is_gu ? sg : sd;
    const int tile = r / ns, slab = r % ns;
    int n_tiles;
    const int4 tt = sload_tile(is_gu ? a.gu.tiles : a.dn.tiles, a.gu.n_tiles, tile, n_tiles);
    if (tile >= n_tiles) return;
    DTRACE_AT(1, item, 0);
#ifdef AINFER_DECODE_TRACE
    if (threadIdx.x == 0) g_dtrace[1][item][4] = is_gu;
#endif
    // one item per workgroup, and no barrier before its loads: each wave
    // issues its weight loads as soon as it is launched (the waves of a
    // workgroup start up to about 1.5 us apart at the launch's start)
    if (is_gu) {
      // x (MFMA order) comes from the routing kernel: plain, cacheable loads
      expert_lds_item<SD, KBW_GU, RG_GU, DEC_MT, 0, true, false>(a.gu, tt, slab, lds);
      if (threadIdx.x >= 64) return;
      // wave 0: its act stores, then the arrival
      DTRACE_AT(1, item, 2);
      wait_stores();
      if (lane == 0) atomicAdd(&gu_done[tile * SY_STRIDE], 1);
      DTRACE_AT(1, item, 3);
      return;
    }
    const int4 td = tt;
    // the down weights are requested before the wait for the tile's act rows
    const int32_t *gdone = &gu_done[tile * SY_STRIDE];
    int32_t *err = a.sync + SY_ERR;
    expert_lds_item<SD, KBW_DN, RG_DN, DEC_MT, 1, true, true>(a.dn, td, slab, lds, [=]() {
      block_wait_geq(gdone, sg, err, a.spin);
      DTRACE_AT(1, item, 1);
    });
    if (threadIdx.x >= 64) return;
    DTRACE_AT(1, item, 2);
    // ---- wave 0: publish o; count this tile's down items and each token's
    // arrivals on this row slab --------------------------------------------
    wait_stores();
    if (lane == 0 && atomicAdd(&dn_done[tile * SY_STRIDE], 1) == sd - 1) {
      gu_done[tile * SY_STRIDE] = 0;  // all of the tile's down items have passed their wait
      dn_done[tile * SY_STRIDE] = 0;
    }
    const bool shared = td.x == a.dn.E;
    const int mcnt = td.z;
    const int has_shared = a.dn.Is > 0;
    const int k = a.dn.k, H = a.dn.H;
    int tok = -1;
    if (lane < mcnt) {
      const int pos = td.y + lane;
      const int tt = shared ? pos : a.dn.ptok[pos];
      int32_t *c = &cnt[(tt * sd + slab) * SY_STRIDE];
      if (atomicAdd(c, 1) == k + has_shared - 1) {
        *c = 0;
        tok = tt;
      }
    }
    DTRACE_AT(1, item, 3);
    if (__ballot(tok >= 0) == 0ull) return;
    // ---- combine of the completed (token, slab) pairs: slot order, as
    // k_combine -------------------------------------------------------------
    const __amdgpu_buffer_rsrc_t orr = make_rsrc(a.dn.o, 0x7FFFFFFFu);
    const int rows = 16 * RG_DN * a.dn.WR, r0 = slab * rows;
    const size_t Tk = (size_t)a.dn.T * k;
    // a wait of this or an earlier call on the workspace ran out (this
    // workgroup's own timeout is already visible here): NaN outputs
    const bool bad = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    constexpr int CB = 4;  // slots whose loads are issued together
    for (int i = 0; i < mcnt; ++i) {
      const int t = __builtin_amdgcn_readfirstlane(__shfl(tok, i, 64));
      if (t < 0) continue;
      for (int hr = lane; hr < rows; hr += 64) {
        const int h = min(r0 + hr, H - 1);
        float acc = 0.0f;
        for (int j0 = 0; j0 < k; j0 += CB) {
          uint16_t ov[CB];
          float wj[CB];
#pragma unroll
          for (int j = 0; j < CB; ++j) {
            const int jj = min(j0 + j, k - 1);
            const int pos = a.inv[(size_t)t * k + jj];
            wj[j] = a.w[(size_t)t * k + jj];
            ov[j] = ld_dev_u16(orr, (uint32_t)(((size_t)pos * H + h) * 2));
          }
#pragma unroll
          for (int j = 0; j < CB; ++j)
            if (j0 + j < k) acc = __builtin_fmaf(wj[j], bf16_to_f32(ov[j]), acc);
        }
        if (has_shared)
          acc = __builtin_fmaf(a.sg[t],
                               bf16_to_f32(ld_dev_u16(orr, (uint32_t)(((Tk + t) * H + h) * 2))), acc);
        if (a.resid) acc += bf16_to_f32(a.resid[(size_t)t * H + h]);
        if (r0 + hr < H) a.y[(size_t)t * H + h] = bad ? (uint16_t)0x7FC0u : f32_to_bf16(acc);
      }
    }
  }
}

// ---- T <= DC_MAX_T: down and combine in one launch -------------------------
// A workgroup owns ROWS = 4 Q output rows of every selected expert: its waves
// take the dispatch tiles in turn (a tile: one expert, all its tokens; the
// shared one last), each with all its weight loads in flight, the tiles' rows
// meet in LDS and one lane per (token, row) sums them in slot order.  Items of
// 32 rows of one expert that counted arrivals per row slab and combined on the
// last took 11.8 us at T = 1, H4096 I1024 k10 + shared (each waits for its sc1
// stores, an atomic, and the last for a read of the others' rows); this form
// 8.5 us.
// With few tiles and a long K (KS > 1, T = 1) KS waves share a tile's K.
// The arithmetic is the decode item's (moe_expert_item.h), bit for bit: per
// 32-wide chunk 8 MFMAs from -136 sum x and the group scale; then at KBW = 2
// (T <= 2) the 8 chunks of two groups added as ((c, c+4), (c, c+2), (c, c+1)),
// at KBW = 4 the 16 chunks of four groups with (c, c+8) first, at KBW = 1 (an odd
// number of groups) the 4 of one; then those sums in k order.
struct DownArgs {
  ExpertArgs dn;
  const float *w, *sg;
  const int32_t *inv;
  const uint16_t *resid;
  uint16_t *y;
  const int32_t *err;
  int has_shared, ks, max_tiles;
};
constexpr int DC_WMAX = 8;  // tiles at KS > 1

// scale dwords of a run's row: one per pair of groups, or (KBW = 1, where a
// row's pairs may straddle dwords) the dword holding each group's scale
constexpr int dc_scale_dma(int rpu, int rows, int kbw) { return (rpu * rows * (kbw == 1 ? 4 : 2) + 63) / 64; }
// LDS bytes per wave: the tile's token rows of the wave's K, then its scales
constexpr int dc_wave_lds(int rpu, int rows, int mt, int kbw) {
  return mt * rpu * 1024 + dc_scale_dma(rpu, rows, kbw) * 256;
}

// RPU: runs of 4 k-groups per wave (of the longer product, over KS); MT: most
// tokens of a tile
template <int SD, int RPU, int Q, int KBW, int MT>
__global__ __launch_bounds__(1024) void k_down_combine(DownArgs a) {
  constexpr int ROWS = 4 * Q;
  __shared__ float s_o[33 * MT][ROWS];
  __shared__ float s_wt[32 * MT];
  __shared__ int s_inv[32 * MT];
  __shared__ float s_part[MT == 1 && KBW == 2 ? DC_WMAX : 1][16][ROWS];  // KS > 1
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int DPR = KBW == 1 ? 4 : 2;  // scale dwords per run and row
  constexpr int SCD = RPU * ROWS * DPR, SCI = dc_scale_dma(RPU, ROWS, KBW);
  constexpr int SCO = MT * RPU * 1024;  // the scales' offset in the wave's LDS
  static_assert(MT == 1 || ROWS * MT <= 64, "wave 0 combines");
  const int tx = tid_opaque();
  const int wave = __builtin_amdgcn_readfirstlane(tx >> 6), lane = tx & 63;
  const int nw = blockDim.x >> 6, k = a.dn.k, H = a.dn.H, T = a.dn.T, KS = MT == 1 && KBW == 2 ? a.ks : 1;
  const int row0 = blockIdx.x * ROWS;
  // what the combine needs, requested before the weights
  const int ct = lane / ROWS, cr = lane % ROWS;  // wave 0: token and row of this lane
  float rv = 0.f, sgv = 0.f, wj = 0.f;
  int pj = 0;
  bool bad = false;
  if (tx < T * k) {
    wj = a.w[tx];
    pj = a.inv[tx];
  }
  if (wave == 0) {
    const int t = min(ct, T - 1);
    sgv = a.sg[t];
    if (a.resid) rv = bf16_to_f32(a.resid[(size_t)t * H + row0 + cr]);
    bad = *a.err != 0;
  }
  const int r4 = lane & 3, c = lane >> 2;
  uint8_t *wl = lds + wave * dc_wave_lds(RPU, ROWS, MT, KBW);
  const uint32_t wl32 = (uint32_t)(uintptr_t)wl;
  int n_tiles = a.max_tiles;
  for (int u = wave; u < n_tiles * KS; u += nw) {
    const int tile = u / KS, part = u % KS;
    const int4 t4 = sload_tile(a.dn.tiles, a.dn.n_tiles, tile, n_tiles);
    if (tile >= n_tiles) break;
    const int pos0 = t4.y, mcnt = t4.z;
    const bool shared = t4.x == a.dn.E;
    const int K = shared ? a.dn.Is : a.dn.I, KB = K >> 7;
    const size_t e = shared ? 0 : (size_t)t4.x;
    const uint8_t *w0 = shared ? a.dn.ws0 : a.dn.w0 + e * H * (K / 2);
    const uint16_t *s0 = shared ? a.dn.ss0 : a.dn.s0 + e * H * KB;
    const int h0 = part * RPU;  // first run of 4 groups
    // lane (r4, c): 32 nibbles of row r4 of a row quad at chunk 16 h + c
    u32x4 B[RPU][Q];
#pragma unroll
    for (int h = 0; h < RPU; ++h) {
      const int ch = min(16 * (h0 + h) + c, 4 * KB - 1);
#pragma unroll
      for (int q = 0; q < Q; ++q)
        B[h][q] = ldg_stream(w0 + (size_t)(row0 + 4 * q + r4) * (K / 2) + ch * 16);
    }
    // scales: dword (h, row, i) of DPR per row (KBW = 1: the aligned dword of
    // group 4 h + i; H rows are an even number, so it never ends past them)
#pragma unroll
    for (int i = 0; i < SCI; ++i) {
      const int d = min(64 * i + lane, SCD - 1);
      const int gi = DPR * (h0 + d / (DPR * ROWS)) + d % DPR, row = row0 + (d / DPR) % ROWS;
      const size_t at = (size_t)row * KB + (KBW == 1 ? min(gi, KB - 1) : 2 * min(gi, KB / 2 - 1));
      dma4(s0 + (at & ~(size_t)1), wl32 + SCO + i * 256);
    }
    // token rows in MFMA order: run h of row t at (t RPU + h) KB
    const uint8_t *act = (const uint8_t *)((shared ? a.dn.a_shared : a.dn.a_routed) + (size_t)pos0 * K);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      if (t >= mcnt) break;
#pragma unroll
      for (int h = 0; h < RPU; ++h)
        dma16(act + (size_t)t * K * 2 + min((h0 + h) * 1024 + lane * 16, K * 2 - 16),
              wl32 + (t * RPU + h) * 1024);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t magic;
    asm volatile("v_mov_b32 %0, 0x43084308" : "=v"(magic));
    const s16x4 ones = {0x3F80, 0x3F80, 0x3F80, 0x3F80};
    const uint32_t mask = 0x000F000Fu;
    const uint16_t *sl = (const uint16_t *)(wl + SCO);
    float gs[Q][MT];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t) gs[q][t] = 0.f;
#pragma unroll
    for (int h = 0; h < RPU; ++h) {
      if (4 * (h0 + h) >= KB) break;
      const uint8_t *xa = wl + ((MT == 1 ? 0 : min(r4, mcnt - 1)) * RPU + h) * 1024 + c * 64;
      s16x4 av[8];
#pragma unroll
      for (int jh = 0; jh < 8; ++jh) av[jh] = *(const s16x4 *)(xa + jh * 8);
      f32x4 xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int jh = 0; jh < 8; ++jh) xs = mfma_bf16_4x4x4(av[jh], ones, xs);
      const f32x4 c0 = xs * -136.0f;
      const bool in = 16 * (h0 + h) + c < 4 * KB;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        f32x4 acc = c0;
#pragma unroll
        for (int jh = 0; jh < 8; ++jh) {
          const int j = jh >> 1, hf = jh & 1;
          const uint32_t d0 = ((B[h][q][2 * hf] >> (4 * j)) & mask) ^ magic;
          const uint32_t d1 = ((B[h][q][2 * hf + 1] >> (4 * j)) & mask) ^ magic;
          acc = mfma_bf16_4x4x4(av[jh], __builtin_bit_cast(s16x4, u32x2{d0, d1}), acc);
        }
        const int sr = ROWS * h + 4 * q + r4, gr = c >> 2;
        const float sc = scale_to_f32<SD>(
            KBW == 1 ? sl[2 * (4 * sr + gr) + (((row0 + 4 * q + r4) * KB + 4 * (h0 + h) + gr) & 1)]
                     : sl[2 * (2 * sr + (gr >> 1)) + (gr & 1)]);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          if (t >= mcnt) break;
          float v = in ? acc[t] * sc : 0.f;
          if (KBW == 4) v += __shfl_xor(v, 32, 64);
          if (KBW > 1) v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (16 << 10) | 0x1F));
          v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (8 << 10) | 0x1F));
          v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), (4 << 10) | 0x1F));
          if (KBW == 4) {
            gs[q][t] += v;
          } else if (KBW == 1) {
            // group 4 h + i's sum in the lanes of chunk 4 i
#pragma unroll
            for (int i = 0; i < 4; ++i) gs[q][t] += __shfl(v, 16 * i + r4, 64);
          } else if (MT == 1 && KBW == 2 && KS > 1) {
            // lanes 0-31 hold groups 4 h, 4 h + 1; lanes 32-63 the next two
            if ((c & 7) == 0) s_part[tile][2 * (h0 + h) + (c >> 3)][4 * q + r4] = v;
          } else {
            gs[q][t] += v;
            gs[q][t] += __shfl_xor(v, 32, 64);
          }
        }
      }
    }
    if (lane < 4 && KS == 1) {
      const int o0 = (shared ? T * k : 0) + pos0;
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          if (t < mcnt) s_o[o0 + t][4 * q + r4] = bf16_to_f32(f32_to_bf16(gs[q][t]));
    }
    // this tile's LDS reads are done before the next tile's copies land there
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  if (tx < T * k) {
    s_wt[tx] = wj;
    s_inv[tx] = pj;
  }
  __syncthreads();
  if (MT == 1 && KBW == 2 && KS > 1) {  // T = 1: tile j's row is o row j (k: the shared one)
    const int nt = k + a.has_shared;
    for (int i = tx; i < nt * ROWS; i += blockDim.x) {
      const int tile = i / ROWS, r = i % ROWS, n = (tile == k ? a.dn.Is : a.dn.I) >> 8;
      float g = 0.f;
      for (int j = 0; j < n; ++j) g += s_part[tile][j][r];
      s_o[tile][r] = bf16_to_f32(f32_to_bf16(g));
    }
    __syncthreads();
  }
  if (wave != 0 || ct >= T) return;
  // ---- the combine, slot order (k_combine's arithmetic) ----------------------
  float acc = 0.f;
  for (int j = 0; j < k; ++j) acc = __builtin_fmaf(s_wt[ct * k + j], s_o[s_inv[ct * k + j]][cr], acc);
  if (a.has_shared) acc = __builtin_fmaf(sgv, s_o[T * k + ct][cr], acc);
  if (a.resid) acc += rv;
  a.y[(size_t)ct * H + row0 + cr] = bad ? (uint16_t)0x7FC0u : f32_to_bf16(acc);
}

}  // namespace

int g_spin_max = SPIN_MAX;

int decode_geometry(const ainfer_moe_shape &s, DecodeGeom *g) {
  int kbw, wk, wr;
  if (!expert_geometry(0, s.hidden, s.inter, s.shared_inter, 4, &kbw, &wk, &wr) || kbw != 4)
    return 0;
  g->wk_gu = wk;
  if (!expert_geometry(1, s.hidden, s.inter, s.shared_inter, 2, &kbw, &wk, &wr) || kbw != 2)
    return 0;
  g->wk_dn = wk;
  g->nw = g->wk_gu > g->wk_dn ? g->wk_gu : g->wk_dn;
  if (g->nw < DEC_NW_MIN) g->nw = DEC_NW_MIN;
  if (g->nw % g->wk_gu || g->nw % g->wk_dn || g->nw > 16) return 0;
  g->wr_gu = g->nw / g->wk_gu;
  g->wr_dn = g->nw / g->wk_dn;
  const int Ngu = s.inter > s.shared_inter ? s.inter : s.shared_inter;
  g->slabs_gu = (Ngu + 16 * DEC_RG_GU * g->wr_gu - 1) / (16 * DEC_RG_GU * g->wr_gu);
  g->slabs_dn = (s.hidden + 16 * DEC_RG_DN * g->wr_dn - 1) / (16 * DEC_RG_DN * g->wr_dn);
  // A staging only: the K-split partials reuse it (expert_lds_item, COH)
  const size_t lds_gu = (size_t)g->nw * item_lds_per_wave(DEC_MT, 4, DEC_RG_GU, 0);
  const size_t lds_dn = (size_t)g->nw * item_lds_per_wave(DEC_MT, 2, DEC_RG_DN, 1);
  g->lds = lds_gu > lds_dn ? lds_gu : lds_dn;
  if (g->lds > 64 * 1024) return 0;
  return 1;
}

hipError_t launch_route_decode(const void *x, const void *rw, const float *bias, const void *gw,
                               float *logits, float *sgl, int32_t *idx, float *w, float *sg,
                               void *xperm, int T, int H, int E, int k, int has_shared,
                               const DispatchOut *ds, int32_t *sync, uint32_t *slots,
                               const NormIn *norm, hipStream_t s, W8Rows w8) {
  if (T <= 0) return hipSuccess;
  if (T > DECODE_MAX_T || T > RD_WAVES || E > 1024) return hipErrorInvalidValue;
  RouteDecodeArgs a;
  memset(&a, 0, sizeof a);
  a.x = (const uint16_t *)x;
  a.rw = (const uint16_t *)rw;
  a.gw = (const uint16_t *)gw;
  a.bias = bias;
  a.logits = logits;
  a.sgl = sgl;
  a.idx = idx;
  a.w = w;
  a.sg = sg;
  a.xperm = (uint16_t *)xperm;
  a.w8 = w8;
  if (ds) a.ds = *ds;
  a.sync = sync;
  a.slots = slots;
  if (norm) a.norm = *norm;
  if (a.norm.on && T > RD_TT1_MAX) return hipErrorInvalidValue;  // see k_route_decode
  a.T = T;
  a.H = H;
  a.E = E;
  a.k = k;
  a.has_shared = has_shared;
  a.spin = g_spin_max;
  const int nrows = E + (gw ? 1 : 0);
  const bool mid = T > RD_TT1_MAX && T <= RD_W2;
  const int tt = T <= RD_TT1_MAX ? 1 : mid ? RD_MID_TT : 2;
  const int units = (nrows + RD_R - 1) / RD_R * ((T + tt - 1) / tt);
  const int wg = T <= RD_TT1_MAX ? RD_W1 : mid ? RD_W2 : RD_WAVES;
  a.NR = (units + wg - 1) / wg;
  const unsigned grid = a.NR + 2;  // router units, the selection, the x copy
  const int nv = (E + 63) / 64;
  auto go = [&](auto nv_c) {
    constexpr int NVc = decltype(nv_c)::value;
    if (T <= RD_TT1_MAX && a.norm.on)
      k_route_decode<NVc, 1, RD_W1, RD_NB1, true><<<grid, RD_W1 * 64, 0, s>>>(a);
    else if (T <= RD_TT1_MAX)
      k_route_decode<NVc, 1, RD_W1, RD_NB1, false><<<grid, RD_W1 * 64, 0, s>>>(a);
    else if (mid)
      k_route_decode<NVc, RD_MID_TT, RD_W2, RD_MID_TT == 1 ? RD_NB1 : RD_NB2, false>
          <<<grid, RD_W2 * 64, 0, s>>>(a);
    else
      k_route_decode<NVc, 2, RD_WAVES, RD_NB, false><<<grid, RD_WAVES * 64, 0, s>>>(a);
  };
  if (nv <= 1) go(std::integral_constant<int, 1>());
  else if (nv <= 2) go(std::integral_constant<int, 2>());
  else if (nv <= 4) go(std::integral_constant<int, 4>());
  else if (nv <= 8) go(std::integral_constant<int, 8>());
  else go(std::integral_constant<int, 16>());
  return hipGetLastError();
}

hipError_t launch_experts_decode(int scale_dtype, const DecodeGeom &g, ExpertArgs gu,
                                 ExpertArgs dn, const float *w, const float *sg,
                                 const int32_t *inv, const void *resid, void *y,
                                 int32_t *sync, int max_tiles, int cap, hipStream_t s) {
  if (max_tiles <= 0) return hipSuccess;
  if (max_tiles > cap) return hipErrorInvalidValue;
  ExpertsDecodeArgs a;
  memset(&a, 0, sizeof a);
  gu.WK = g.wk_gu;
  gu.WR = g.wr_gu;
  gu.n_slabs = g.slabs_gu;
  dn.WK = g.wk_dn;
  dn.WR = g.wr_dn;
  dn.n_slabs = g.slabs_dn;
  a.gu = gu;
  a.dn = dn;
  a.w = w;
  a.sg = sg;
  a.inv = inv;
  a.resid = (const uint16_t *)resid;
  a.y = (uint16_t *)y;
  a.sync = sync;
  a.max_tiles = max_tiles;
  a.cap = cap;
  a.spin = g_spin_max;
  const long grid = (long)max_tiles * (g.slabs_gu + g.slabs_dn);
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  const int threads = g.nw * 64;
  if (scale_dtype == AINFER_SCALE_FP16)
    k_experts_decode<AINFER_SCALE_FP16, 4, DEC_RG_GU, 2, DEC_RG_DN><<<(unsigned)grid, threads, g.lds, s>>>(a);
  else
    k_experts_decode<AINFER_SCALE_BF16, 4, DEC_RG_GU, 2, DEC_RG_DN><<<(unsigned)grid, threads, g.lds, s>>>(a);
  return hipGetLastError();
}

hipError_t launch_down_combine(int scale_dtype, const ExpertArgs &dn, int kbw, const float *w,
                               const float *sg, const int32_t *inv, const void *resid, void *y,
                               const int32_t *err, hipStream_t s) {
  const int Kmax = dn.I > dn.Is ? dn.I : dn.Is, has_shared = dn.Is > 0 ? 1 : 0;
  // (k-groups in whole waves of the item's split)
  if (dn.T < 1 || dn.T > DC_MAX_T || dn.k > 32 || dn.H % 128 ||
      (kbw != 1 && kbw != 2 && (kbw != 4 || dn.T == 1)) ||
      dn.I % (128 * kbw) || dn.Is % (128 * kbw) || Kmax > 4096)
    return hipErrorInvalidValue;
  DownArgs a;
  memset(&a, 0, sizeof a);
  a.dn = dn;
  a.w = w;
  a.sg = sg;
  a.inv = inv;
  a.resid = (const uint16_t *)resid;
  a.y = (uint16_t *)y;
  a.err = err;
  a.has_shared = has_shared;
  const int tiles = a.max_tiles = dn.T * dn.k + has_shared;  // at most
  int rpu = 1;
  while (512 * rpu < Kmax) rpu *= 2;
  // few tiles: KS waves share a tile's K
  a.ks = 1;
  while (dn.T == 1 && kbw == 2 && rpu > 1 && tiles <= DC_WMAX && tiles * a.ks * 2 <= 16) {
    a.ks *= 2;
    rpu /= 2;
  }
  if (dn.T > 1 && rpu > 2) return hipErrorInvalidValue;  // down_combine_at
  const int nw = tiles * a.ks < 16 ? tiles * a.ks : 16;
  using std::integral_constant;
  auto go = [&](auto sd_c, auto rpu_c, auto q_c, auto kbw_c, auto mt_c) {
    constexpr int SDc = decltype(sd_c)::value, R = decltype(rpu_c)::value,
                  Qc = decltype(q_c)::value, KW = decltype(kbw_c)::value,
                  M = decltype(mt_c)::value;
    k_down_combine<SDc, R, Qc, KW, M>
        <<<dn.H / (4 * Qc), nw * 64, (size_t)nw * dc_wave_lds(R, 4 * Qc, M, KW), s>>>(a);
  };
  // T > 1: 16 rows per workgroup where that still gives every CU one
  const bool wide = dn.H >= 16 * 256;
  auto go_t = [&](auto sd_c, auto rpu_c, auto kbw_c) {
    if (wide)
      go(sd_c, rpu_c, integral_constant<int, 4>(), kbw_c, integral_constant<int, 4>());
    else
      go(sd_c, rpu_c, integral_constant<int, 2>(), kbw_c, integral_constant<int, 4>());
  };
  auto go_r = [&](auto sd_c, auto kbw_c) {
    if (rpu == 1) go_t(sd_c, integral_constant<int, 1>(), kbw_c);
    else go_t(sd_c, integral_constant<int, 2>(), kbw_c);
  };
  auto go_1 = [&](auto sd_c, auto kbw_c) {
    using two = integral_constant<int, 2>;
    using one = integral_constant<int, 1>;
    if (rpu == 1) go(sd_c, one(), two(), kbw_c, one());
    else if (rpu == 2) go(sd_c, two(), two(), kbw_c, one());
    else if (rpu == 4) go(sd_c, integral_constant<int, 4>(), two(), kbw_c, one());
    else go(sd_c, integral_constant<int, 8>(), two(), kbw_c, one());
  };
  auto go_k = [&](auto sd_c) {
    using two = integral_constant<int, 2>;
    using one = integral_constant<int, 1>;
    if (dn.T > 1) {
      if (kbw == 1) go_r(sd_c, one());
      else if (kbw == 2) go_r(sd_c, two());
      else go_r(sd_c, integral_constant<int, 4>());
    } else if (kbw == 1) go_1(sd_c, one());
    else go_1(sd_c, two());
  };
  if (scale_dtype == AINFER_SCALE_FP16)
    go_k(integral_constant<int, AINFER_SCALE_FP16>());
  else
    go_k(integral_constant<int, AINFER_SCALE_BF16>());
  return hipGetLastError();
}

__global__ void k_zero_i32(int32_t *p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}


hipError_t launch_zero_i32(int32_t *p, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  k_zero_i32<<<(n + 255) / 256 < 1024 ? (n + 255) / 256 : 1024, 256, 0, s>>>(p, n);
  return hipGetLastError();
}
