// moe_internal.h - host-side launchers shared between the kernel files and
// the C-ABI implementation (moe_api.hip).  Not part of the public ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <cmath>

#include "../../include/ainfer_moe.h"

// Arguments of the grouped expert kernels (one launch covers the routed
// experts and the shared expert, whose tiles carry expert id E).
struct ExpertArgs {
  const uint8_t *w0, *w1;     // routed: gate, up (MODE 0) or down (MODE 1)
  const uint16_t *s0, *s1;    // their scales
  const uint8_t *ws0, *ws1;   // shared expert tensors
  const uint16_t *ss0, *ss1;
  const uint16_t *a_routed;   // MODE 0: x in MFMA order [T][H]; MODE 1: act [Tk][I]
  const uint16_t *a_shared;   // MODE 0: same x; MODE 1: act_s [T][Is]
  uint16_t *act;              // MODE 0 out: [Tk][I] bf16, MFMA order
  uint16_t *act_s;            // MODE 0 out: [T][Is]
  uint16_t *o;                // MODE 1 out: [Tk + T][H] bf16
  const int32_t *ptok;        // token of each dispatch position
  const int4 *tiles;          // (expert, first position, rows, 0)
  const int32_t *n_tiles;
  int T, k, E, H, I, Is;
  int WK, WR, n_slabs;        // set by the launcher
};

// Arguments of the prefill GEMM (moe_gemm.hip).
struct GemmArgs {
  const uint8_t *w0, *w1;
  const uint16_t *s0, *s1;
  const uint8_t *ws0, *ws1;
  const uint16_t *ss0, *ss1;
  const uint16_t *a_routed;   // MODE 0: x in MFMA order [T][H]; MODE 1: act [Tk][I]
  const uint16_t *a_shared;   // MODE 1: act_s [T][Is]
  uint16_t *act, *act_s;      // MODE 0 out
  uint16_t *o;                // MODE 1 out: [Tk + T][H] bf16
  const float *xsum;          // [T][H/128] -GEMM_NIB_OFFSET x the group sums of x
  float *asum, *asum_s;       // [Tk][I/128], [T][Is/128] the same of act (MODE 0 out)
  const int32_t *ptok;
  const int4 *tiles;
  const int32_t *n_tiles;
  int T, k, E, H, I, Is;
  int n_nblk;                 // set by the launcher
};
// Prefill router: approximate logits (+ bias) and router row norms, tiled bf16 MFMA GEMM.
// zbuf: zwords 32-bit words zeroed by the kernel (the dispatch counts and
// masks the following k_select fills), or null
hipError_t launch_router_gemm(const void *x, const void *rw, const float *bias, float *approx,
                              float *wnorm, int T, int H, int E, uint32_t *zbuf, int zwords,
                              hipStream_t s);
hipError_t launch_expert_gemm(int mode, int scale_dtype, GemmArgs a, int max_tiles,
                              hipStream_t s);
// token-tile height of the expert GEMMs (at most)
constexpr int GEMM_MT = 64;
// The height a call uses: the largest of 64, 32 and 16 that gives the gate/up
// stage an item for every CU, and 16 only up to 64 tokens per expert.  A lower
// tile re-reads weights through L2, but below one item per CU its shorter
// items run side by side (E8 k2 I1024, T = 128: 58 -> 48 us, in W4A8 66 -> 48;
// E66 k5 I128 T = 512: 109 -> 99 us, but 16 at T = 1024: 121 -> 128).
inline int gemm_mt(const ainfer_moe_shape &s, int T) {
  const long slots = (long)T * s.top_k, hit = slots < s.n_experts ? slots : s.n_experts;
  int mt = GEMM_MT;
  // tiles: the full ones and, on average, half a tile more per expert
  while (mt > 16 && (slots / mt + hit / 2) * (s.inter / 128) < 256 &&
         (mt > 32 || slots <= 64 * hit))
    mt /= 2;
  return mt;
}
#ifndef GEMM_WN
#define GEMM_WN 4       // waves per GEMM block, 64 weight rows each
#endif
// from this many tokens on the router's approximate logits come from the
// tiled GEMM (k_router_gemm), k_select runs one wave per token, and the
// experts always run as the grouped GEMM
constexpr int GEMM_MIN_T = 256;
// Experts as the grouped GEMM or as streaming items of at most DEC_MT tokens,
// for 16 < T.  The items re-read an expert's weights for every 4 of its
// tokens; the GEMM reads them once but needs enough items to fill the chip.
// Two lines, in tokens per expert (T k / E), and the GEMM is past both:
//  - 3.25.  Where both stages have items for every CU the two cross at 2.0
//    (H4096 E512 k10 I1024; T = 97: 584 us items, 591 GEMM; T = 133: 673, 630), 2.8
//    (H2048 E512 k10 I512; T = 133: 203, 208; T = 154: 222, 211; and E128 k8 I768),
//    3.0 (E256 k8 I256) and 3.25 (H3072 E324 k5 I256; T = 194: 143, 147; T = 233:
//    156, 152).  The line is the largest, so that none of these is slower by the
//    GEMM; below it the first ones' items are the slower ones, by up to 15%.
//  - C (1 / gate-up items + 1 / (2 x down items)).  With few items the GEMM waits
//    for one block's chain of groups per stage, whatever T is (down's weights are
//    half of gate/up's), while the items only grow with T.  C = the crossover over
//    that sum: 390 to 500 at H 2048 to 4096 (H3584 E20 k4 I128 crosses at 23: T = 80
//    51 us items, 56 GEMM; H3584 E66 k5 I128 at 6.4: T = 66 57, 62; H2048 E8 k2 I512
//    at 17, I4096 at 5.6; H2048 E4 k1 I1024 at 21), 300 to 450 at H 1280 and 1536,
//    220 to 260 at H1024 (E8 k2 I1024 at 7, E16 k4 I256 at 10), whose chains are
//    short, 60 to 140 at H512 (E8 k2 I256 at 13, E20 k4 I128 below 4); less where a
//    shared expert adds items (350 to 410 from H 2048 on).
inline bool expert_gemm_at(const ainfer_moe_shape &s, int T) {
  if (T >= GEMM_MIN_T) return true;
  if (T <= 16) return false;
  const long E = s.n_experts, slots = (long)T * s.top_k;
  const long gu = E * (s.inter / 128), dn = E * ((s.hidden + 255) / 256);
  const long C = s.hidden <= 512 ? 128 : s.hidden <= 1024 ? 256 : 432;
  return 4 * slots >= 13 * E && slots * 2 * gu * dn >= C * E * (gu + 2 * dn);
}

// Rows quantized for the W4A8 GEMM: codes in W8 order (write_xperm,
// moe_common.h), their scales per 128-wide group, -8 x each group's code sum.
struct W8Rows {
  int8_t *q = nullptr;
  float *s = nullptr;
  int32_t *sum = nullptr;
};
// Arguments of the W4A8 GEMM (moe_gemm_w4a8.hip).
struct W8GemmArgs {
  const uint8_t *w0, *w1, *ws0, *ws1;  // MODE 0: gate, up; MODE 1: down (w0 / ws0)
  const uint16_t *s0, *s1, *ss0, *ss1;
  W8Rows x, act, act_s;  // [T][H]; [T k][I], [T][Is] (MODE 0 out, MODE 1 in)
  float *o;              // MODE 1 out: [T k + T][H]
  const int32_t *ptok;
  const int4 *tiles;     // of at most GEMM_MT tokens
  const int32_t *n_tiles;
  int T, k, E, H, I, Is;
  int n_nblk;            // set by the launcher
};
// The W4A8 GEMM or 16-row GEMV blocks, from 2 tokens on.  The GEMM reads a weight
// once per tile, but where its items are few it waits for one item's chain of
// groups per stage; the blocks cut rows by 16 (us, blocks then GEMM).
//  Above 16 tokens the GEMM.  At 2 to 4 (down with the combine in it, intermediate
//  sizes to W8DC_MAX_K: I4096 H2048 E8 k2 T2 35, 45) from 24 gate/up items on
//  (H3584 E20 k4 I128 T4 30, 33; H2048 E512 k10 I512 T4 42, 32), and above I256
//  where gate/up's groups are no more than 0.9 of its items, of the experts that T
//  tokens hit on average (H4096 E32 k2 I512, 1.4 at T3: 29, 34; H4096 E64 k4 I512,
//  1.0 at T2: 33, 35, 0.7 at T3: 38, 36).
//  At 5 to 16 by groups over items, gate/up's + 10 times down's: up to 0.8, or 1.6
//  at I to 256.  At H2048
//  E32 k2 I1408 it is 1.2 at T8 (33, 33) and 0.7 at T16 (42, 36); H2048 E64 k2
//  I1024 0.8 at T8 (30, 32), 0.7 at T10 (34, 33); H4096 E32 k2 I512 1.2 at T5 (33,
//  38), 0.6 at T12 (43, 42); H4096 E6 k2 I1024 1.8 at T6 (35, 41); H2048 E4 k1
//  I1024 3.0 (T8 26, 30); H3584 E20 k4 I128 1.9 at T6 (31, 35), 1.5 at T12 (39,
//  38); H3584 E66 k5 I128 1.3 at T5 (40, 36).
inline bool w4a8_gemm_at(const ainfer_moe_shape &s, int T) {
  if (T > 16 || T < 2) return T > 1;
  if (s.inter > 2048 || s.shared_inter > 2048) return false;
  const int gi = s.inter / 128;
  const double E = s.n_experts, hit = E * (1.0 - std::pow(1.0 - s.top_k / E, T));
  const double gu = hit * gi, dn = hit * ((s.hidden + 255) / 256);
  const double chain = (s.hidden / 128) / gu;
  if (T <= 4) return (long)T * s.top_k * gi >= 24 && (gi <= 2 || chain <= 0.9);
  return chain + 10 * gi / dn <= (gi <= 2 ? 1.6 : 0.8);
}
hipError_t launch_w4a8_gemm(int mode, int scale_dtype, W8GemmArgs a, int max_tiles,
                            hipStream_t s);

// Outputs of the dispatch stage.  tiles: (expert, first position, rows,
// first row within the expert); shared-expert tiles carry expert id E and a
// token base.  ptok[pos] = token of dispatch position pos.
// the combine arrival counters, zeroed by the dispatch.  ticket is the
// last-block counter of the fused top-k + dispatch launch.
struct DispatchOut {
  int32_t *counts, *offsets, *perm, *inv, *ptok;
  int4 *tiles;
  int32_t *n_tiles;
  int32_t *ticket;
  int mt;  // tokens per tile of dispatch_small_block
};

hipError_t launch_fill(int kind, uint64_t seed, float std_, size_t n, void *out,
                       hipStream_t s);
hipError_t launch_rmsnorm(const void *x, const void *w, int mode, float eps, void *y,
                          int T, int H, hipStream_t s);
// ticket (may be NULL) is zeroed for the fused top-k + dispatch launch
hipError_t launch_router(const void *x, const void *rw, const float *bias, const void *gw,
                         float *logits, float *sg_logit, int32_t *ticket, int T, int H, int E,
                         hipStream_t s);
// Router: approximate MFMA logits -> exact candidate refine -> top-k,
// weights, shared gate, MFMA-order copy of x.  fused != NULL (T <= 64 only):
// the last block also runs the dispatch.  approx [T][E] and wnorm [E] are
// scratch.
bool router_supported(int H, int E);
// xsum (may be NULL): [T][H/128] -GEMM_NIB_OFFSET x the group sums of x for the prefill GEMM.
hipError_t launch_router_fast(const void *x, const void *rw, const float *bias, const void *gw,
                              float *approx, float *wnorm, int32_t *idx, float *w, float *sg,
                              void *xperm, float *xsum, int T, int H, int E, int k,
                              int has_shared, const DispatchOut *fused, hipStream_t s,
                              int32_t *ccount = nullptr, unsigned long long *cmask = nullptr,
                              W8Rows w8 = W8Rows());
// cmask non-null: the per-(64-token chunk, expert) token masks (and, in
// chunk_counts, the counts) the router's k_select already built
// (T >= GEMM_MIN_T), so no counting launch
hipError_t launch_dispatch(const int32_t *idx, int T, int k, int E, int mt, int has_shared,
                           int32_t *chunk_counts, int32_t *rank, const DispatchOut &ds,
                           hipStream_t s, const unsigned long long *cmask = nullptr);
// x in MFMA order (+ its per-128 group sums when xsum is non-null)
hipError_t launch_xperm(const void *x, void *xperm, float *xsum, int T, int H, hipStream_t s);
// expert output rows from dispatch-position order to slot order (H % 8 == 0)
hipError_t launch_gather_rows(const void *src, const int32_t *inv, void *dst, int T, int k,
                              int H, int has_shared, hipStream_t s);
// inv null: o's routed rows are in slot order (row t * k + j)
hipError_t launch_combine(const uint16_t *o, const int32_t *inv, const float *w, const float *sg,
                          int has_shared, const void *resid, void *y, int T, int k, int H,
                          const int32_t *err, hipStream_t s);
// The same combine (resid non-null, H % 8 == 0, H <= 4096, 16-byte aligned
// rows) followed by the next block's RMSNorm of each written row:
// h[t] = RMSNorm(y[t]) with `next` (weight, mode, eps), bit-identical to
// launch_rmsnorm on y.  One 256-thread block per token.
hipError_t launch_combine_norm(const uint16_t *o, const int32_t *inv, const float *w,
                               const float *sg, int has_shared, const void *resid, void *y,
                               int T, int k, int H, const int32_t *err, const NormIn &next,
                               void *h, hipStream_t s);
// polls a bounded device wait makes before it gives up (sets the workspace's
// error word); ainfer_moe_debug_spin_limit changes it for tests
extern int g_spin_max;
// false when the shape has no wave geometry (more than 16 waves along K)
bool expert_geometry(int mode, int H, int I, int Is, int pref_kbw, int *KBW, int *WK,
                     int *WR);
// the streaming items: 16-row groups per wave that share one load of the token
// rows (gate/up, down), and down's preferred k-groups per wave
#ifndef DEC_RG_GATE_UP
#define DEC_RG_GATE_UP 1
#endif
#ifndef DEC_RG_DOWN
#define DEC_RG_DOWN 2
#endif
#ifndef DEC_KBW_DOWN
#define DEC_KBW_DOWN 2
#endif
constexpr int stream_rg(int mode) { return mode == 0 ? DEC_RG_GATE_UP : DEC_RG_DOWN; }
// The next gate/up launch of launch_expert_stream goes through hipExtLaunchKernel
// with these start/stop events (one shot).
void set_expert_launch_events(hipEvent_t start, hipEvent_t stop);
// mode 0: gate/up + SiLU-mul; mode 1: down.  max_tiles bounds the tile list.
// pref_kbw: preferred 128-wide k-groups per wave (1, 2 or 4).
hipError_t launch_expert_stream(int mode, int scale_dtype, ExpertArgs a, int max_tiles,
                                int pref_kbw, hipStream_t s);

// LDS bytes per wave of a decode expert item (moe_expert_item.h): its A
// rows (MT x KBW * 256 B), its scales (KBW >= 2: one dword DMA per 256 B),
// and its K-split partials where they do not fit the A rows.
__host__ __device__ constexpr int item_scale_lds(int kbw, int rg, int mode) {
  return kbw >= 2 ? ((mode == 0 ? 2 : 1) * rg * 16 * kbw * 2 + 255) / 256 * 256 : 0;
}
__host__ __device__ constexpr int item_lds_per_wave(int mt, int kbw, int rg, int mode) {
  return mt * kbw * 256 + item_scale_lds(kbw, rg, mode) +
         (mt * kbw * 256 >= (mode == 0 ? 2 : 1) * rg * 1024 ? 0 : (mode == 0 ? 2 : 1) * rg * 1024);
}
constexpr int DEC_MT = 4;  // token rows of the streaming items' tiles
// largest T routed by the fused top-k + dispatch launch
constexpr int FUSED_DISPATCH_MAX_T = 64;


// ---- decode layer (moe_decode.hip), T <= DECODE_MAX_T ----
// (routed by k_route_decode: every logit in the canonical order; above, approximate logits and the
// canonical ones of the candidates)
constexpr int DECODE_MAX_T = 16;
// ainfer_moe_block_forward folds the RMSNorm into the decode routing kernel
// up to this many tokens (its one-token-per-wave form)
constexpr int DECODE_NORM_MAX_T = 4;
// up to this many tokens the expert stages run fused in one launch
// (k_experts_decode); above it as gate/up, down and combine launches (the
// fused items' handoffs cost more than the two launches they save)
#ifndef FUSED_EXPERTS_MAX_T
#define FUSED_EXPERTS_MAX_T 2
#endif
// sync region (int32 words at the start of the workspace, zero between calls):
// the error word, the per-tile and per-(token, slab) counters of the fused
// expert kernel, then the routing kernel's logit slots.  Counters sit
// SY_STRIDE words (256 bytes) apart.
enum { SY_STRIDE = 64, SY_ERR = 0, SY_TILES = SY_STRIDE };
struct DecodeGeom {
  int nw;                  // waves per expert workgroup
  int wk_gu, wr_gu, wk_dn, wr_dn;
  int slabs_gu, slabs_dn;  // row slabs per tile
  size_t lds;              // dynamic LDS bytes
};
// W4A8 GEMV numerics (moe_w4a8.hip)
// The MoE layer in W4A8 at decode sizes: the expert GEMVs and the fp32 combine.
struct W4A8Args {
  const uint8_t *w0, *w1, *ws0, *ws1;     // MODE 0: gate, up; MODE 1: down (w0/ws0)
  const uint16_t *s0, *s1, *ss0, *ss1;
  const int8_t *xq;                      // [T][H] x quantized
  const float *xs;                       // [T][H/128]
  float *act, *act_s;                    // MODE 0 out: [T*k][I], [T][Is]
  int8_t *aq, *aq_s;                     // MODE 1: act quantized (T > 1; written by the launch)
  float *as, *as_s;                      // their group scales
  float *o;                              // MODE 1 out: [T*k + T][H]
  const int32_t *ptok;
  const int4 *tiles;
  const int32_t *n_tiles;
  int T, k, E, H, I, Is;
};
// T > 1, tiles of at most 16 tokens: mode 0 gate/up + SiLU (act in fp32), mode 1
// act's quantization, then down
hipError_t launch_w4a8_expert(int mode, int scale_dtype, const W4A8Args &a, int max_tiles,
                              hipStream_t s);
hipError_t launch_act_quant_f32_pair(const float *x, int T, int K, int8_t *q, float *sq,
                                     const float *x2, int T2, int K2, int8_t *q2, float *sq2,
                                     hipStream_t s);
// T = 1: mode 0 gate/up + SiLU (act in fp32), mode 1 down (quantizes act in its
// blocks)
hipError_t launch_w4a8_expert_t1(int mode, int scale_dtype, const W4A8Args &a, int max_tiles,
                                 hipStream_t s);
// T <= DC_MAX_T, intermediate sizes up to W8DC_MAX_K: down (a's MODE 1 pointers)
// and the combine.  T = 1: act in a in fp32; else quantized in q, q_s.
constexpr int W8DC_MAX_K = 2048;
hipError_t launch_w4a8_down_combine(int scale_dtype, const W4A8Args &a, const W8Rows &q,
                                    const W8Rows &q_s, const float *w, const float *sg,
                                    const int32_t *inv, const void *resid, void *y,
                                    const int32_t *err, hipStream_t s);
hipError_t launch_combine_f32(const float *o, const int32_t *inv, const float *w,
                              const float *sg, int has_shared, const void *resid, void *y, int T,
                              int k, int H, const int32_t *err, hipStream_t s);
hipError_t launch_act_quant_i8(const void *x, int x_dtype, int T, int K, int8_t *q, float *sq,
                               hipStream_t s);
hipError_t launch_int4_gemv_i8(const uint8_t *P, const void *S, int scale_dtype, const int8_t *xq,
                               const float *sq, int M, int K, int T, float *y, hipStream_t s);
// 0 when the shape has no geometry for k_experts_decode (T = 2 then takes three launches)
int decode_geometry(const ainfer_moe_shape &s, DecodeGeom *g);
// router logits + top-k + weights + shared gate + x in MFMA order, and the
// dispatch (tiles of DEC_MT tokens) when ds != NULL
hipError_t launch_route_decode(const void *x, const void *rw, const float *bias, const void *gw,
                               float *logits, float *sgl, int32_t *idx, float *w, float *sg,
                               void *xperm, int T, int H, int E, int k, int has_shared,
                               const DispatchOut *ds, int32_t *sync, uint32_t *slots,
                               const NormIn *norm, hipStream_t s, W8Rows w8 = W8Rows());
// gate/up + SiLU, down and the combine (y = sum_j w_j o_j + g_s o_s (+ resid))
// in one launch
hipError_t launch_experts_decode(int scale_dtype, const DecodeGeom &g, ExpertArgs gu,
                                 ExpertArgs dn, const float *w, const float *sg,
                                 const int32_t *inv, const void *resid, void *y,
                                 int32_t *sync, int max_tiles, int cap, hipStream_t s);
// T <= DC_MAX_T: down and the combine; the gate/up items (launch_expert_stream)
// ran before.  kbw: the k-groups whose sums a wave of the down items adds (the
// order of the additions, as launch_expert_stream's at the same T).
constexpr int DC_MAX_T = 4;
// beyond one token a wave's LDS holds the token rows of up to 1024 columns
inline bool down_combine_at(const ainfer_moe_shape &s, int T) {
  return T == 1 || (T <= DC_MAX_T && s.inter <= 1024 && s.shared_inter <= 1024);
}
hipError_t launch_down_combine(int scale_dtype, const ExpertArgs &dn, int kbw, const float *w,
                               const float *sg, const int32_t *inv, const void *resid, void *y,
                               const int32_t *err, hipStream_t s);
hipError_t launch_zero_i32(int32_t *p, int n, hipStream_t s);

// k-groups per wave of the 4-token down items: whole 256-byte row segments
// once the down K (the intermediate size) has 8 groups or more
#ifndef DOWN_KBW4_MIN_I
#define DOWN_KBW4_MIN_I 1024  // c3 T=64: down 149.5 -> 139.5 us; c1 (I = 512) keeps 2
#endif
inline int down_kbw_of(const ainfer_moe_shape &s) {
  const int I = s.inter > s.shared_inter ? s.inter : s.shared_inter;
  return I >= DOWN_KBW4_MIN_I ? 4 : DEC_KBW_DOWN;
}

// ---- persistent decode stack (moe_stack.hip) ------------------------------
// One entry of the device layer table (ainfer_moe_stack_prepare).
struct StackLayer {
  ainfer_moe_weights w;
  const void *norm_w;  // RMSNorm weight [H] bf16, or null (unit)
  const void *pad;
};
struct StackGeom {
  int nw, wk_gu, wr_gu, wk_dn, wr_dn, kbw_dn, slabs_gu, slabs_dn;
  size_t lds;
};
// The stack kernel's workspace pieces: its counters and item flags (in the
// zeroed head of the workspace) and the per-layer regions.
struct StackWs {
  int32_t *flags;    // stack_flag_words
  int cap;           // tile capacity of the item flag arrays
  uint8_t *layers;   // n_layers regions of stack_layer_bytes(T)
  int32_t *err;
};
// bytes of one layer's region at T tokens (offs: the 6 piece offsets)
size_t stack_layer_bytes(const ainfer_moe_shape &s, int T, size_t *offs);
// false when the shape has no stack geometry at T tokens (use block_forward)
bool stack_geometry(const ainfer_moe_shape &s, int T, StackGeom *g);
int stack_flag_words(const ainfer_moe_shape &s, int cap);
hipError_t launch_decode_stack(int scale_dtype, const ainfer_moe_shape &s, const StackGeom &g,
                               const StackLayer *layers, int L, const void *x0, void *r, int T,
                               int norm_mode, float eps, const StackWs &w, hipStream_t st);
