// moe_gemm.hip - grouped INT4 expert GEMM for prefill (bf16 MFMA).
//
// As in the decode kernel (moe_expert.hip), weights become bf16 values a constant
// above q (here 24, nib_slice3), every 128-wide group accumulates from -24 *
// sum_{k in g} a[m][k] and the group's scale is applied with one fp32 fma per
// output, so the result is sum_g s_g * sum_{k in g} q * a.
// Restates the reference's INT4 GEMM (ChunkGemm, tools/cmdlist/kernels.cpp:
// 691-785; gemmMT4, tools/prefill/prefill.cpp:46-129) for bf16 MFMA.
//
// Block tile: at most 64 tokens (one expert tile of the dispatch) x 256
// weight rows (MODE 0 takes 128 gate rows and the matching 128 up rows, MODE
// 1 256 down rows), K in 128-wide groups.  4 waves along the rows, each all the
// tile's tokens x 64 rows: 2 x 2 tiles of v_mfma_f32_32x32x16_bf16 at 33 to 64
// tokens, 1 x 2 at 17 to 32, 1 x 4 of 16x16x32 up to 16.  16-token subtiles past
// the tile's count are not copied, and cost MFMAs only as the missing partner of
// a third one, so one kernel serves experts of one token (bound by streaming
// their weights) and of thousands (bound by the loop's issue).
//
// Why 64 tokens and 4 waves: two such blocks fit a CU (80 KB of LDS each, 2
// waves per SIMD together), so one block's prologue, barriers and epilogue
// run under the other's main loop, and a tile holds little padding.  Against
// one block of 8 waves on 128-token tiles with the experts of at most 32
// tokens in a 16-token streaming kernel (whole layer, H2048 E512 k10 I512):
// T = 1500 576 -> 319 us, T = 4096 Zipf 578 -> 477, 4 x 4096 2822 -> 2209;
// H2560 E96 k6 I896 T = 301 381 -> 191 us.  With the steps since then (32-wide
// MFMAs, a third stage, scales on the ring) 297, 435, 2065 and 167.
//
// Data movement: an LDS ring of 2 stages, 3 up to 32 tokens, one barrier per
// group.  Each stage holds one group of the token rows (256 B each, already in
// MFMA order), of the raw INT4 weight rows (64 B each), the dword of each weight
// row that holds its scale, and the token rows' group sums (for x from k_select,
// for act from this kernel's MODE 0 epilogue).  All of it arrives by global->LDS
// DMA (global_load_lds_dwordx4 and _dword: lane i of a wave lands at M0 + 16 i or
// 4 i), one or two groups ahead of the math, with no staging registers.  The
// DMA is issued from inline asm and its completion tracked with explicit
// vmcnt waits, so the compiler's conservative waits do not serialise the
// ring.  Rows are swizzled in 16-byte chunks (A: chunk c of row r at
// c ^ aswz(r); B: chunk q at q ^ bswz(r)) so that the lanes reading 16 rows
// at one column hit distinct bank groups.
#include <type_traits>

#include "moe_common.h"
#include "moe_internal.h"
#include "moe_gemm_parts.h"

#ifdef AINFER_GEMM_TRACE
// diagnostic builds only: per item (MODE * 16384 + item), the shader clock
// (s_memtime) at the item's start, before its main loop, after the loop's
// last barrier, and after its epilogue
__device__ unsigned long long g_gtrace[2 * 16384 * 4];
#define GTRACE(V) V
extern "C" int ainfer_debug_gemm_trace(void *host) {
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(g_gtrace), sizeof(g_gtrace)) == hipSuccess ? 0 : -1;
}
#else
#define GTRACE(V)
#endif

namespace {

constexpr int BM = GEMM_MT;  // tokens per tile: one token wave of 64

// Block geometry: WN waves along the weight rows; BN = 64 * WN rows per block.
template <int WN>
struct Geo {
  static constexpr int NW = WN;                      // waves
  static constexpr int THREADS = 64 * NW;
  static constexpr int BN = 64 * WN;                 // weight rows
  static constexpr int A_SUB = 16 * 256;             // bytes of a 16-token subtile per group
  static constexpr int B_STAGE = BN * 64;            // bytes per group
  // one ring stage at NMS token subtiles: A rows, B rows, a dword per B row
  // holding its scale, the group sums of 64 token rows
  static constexpr int stage(int nms) { return nms * A_SUB + B_STAGE + BN * 4 + BM * 4; }
  // two groups in flight where three stages fit (two blocks per CU, 80 KB each)
  static constexpr int stages(int nms) { return nms <= 2 ? 3 : 2; }
  static constexpr int RING = 3 * stage(2) > 2 * stage(4) ? 3 * stage(2) : 2 * stage(4);
  static constexpr int A_DMA = BM * 256 / (THREADS * 16);  // DMA per thread per group
  static constexpr int B_DMA = B_STAGE / (THREADS * 16);
  static constexpr int COLS = 32 * WN;               // MODE 0: act columns per block
  static_assert(BN == THREADS, "one lane per weight row copies its scales");
};

// A chunk swizzle: logical 16-byte chunk c of token row r sits at
// c ^ aswz(r), the 2-bit halves of r & 15 swapped.  The 16 rows that one
// fragment read touches at one logical chunk then spread over all 8
// 16-byte bank groups in each pair of k-quarter lanes (measured: 77% fewer
// LDS bank-conflict cycles than c ^ r).
__device__ __forceinline__ int aswz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

// Four bf16 pairs 24 + q of k-slice j of a packed 16-byte chunk
// (GEMM_NIB_OFFSET).  A nibble's two's complement value q is (nibble ^ 8) - 8,
// and a bf16 between 16 and 32 holds 16 + NN for the four upper bits NN of its
// mantissa, so the nibble pair shifted there, masked and xor'ed with `magic` =
// 0x41C041C0 (held in a register) is the pair 24 + q: a shift and one
// v_bitop3_b32.
//
// Why 24: the fp32 sums pass through the offset times sum a, whose rounding is
// what a dot is off by.  With the nibble in the mantissa's lower four bits
// (136 + q, one shift in four saved) a gate dot over 2048 columns of variance 1
// with |q| <= 7 was off by 1.7e-4 to 2.3e-4 (root mean square over dots that are
// 0 in 64 bits), where the 4-token items, which start anew every 32 columns, are
// off by 4e-5 to 7e-5; now 1.2e-5 to 1.9e-5.  The shift costs 1 to 2% (us, H2048
// E512 k10 I512: T192 216 -> 218, T1500 293 -> 296, T4096 516 -> 526; H2560 E96
// k6 I896 T301 168 -> 169, T2048 461 -> 469; H4096 I1024 T4096 1796 -> 1819).
__device__ __forceinline__ u32x4 nib_slice3(u32x4 b, int j, uint32_t magic) {
  u32x4 r;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    r[d] = ((j == 0 ? b[d] << 3 : b[d] >> (4 * j - 3)) & 0x00780078u) ^ magic;
  return r;
}

// D (TM x TM) += A B: 16 x 16 over 32 k, or 32 x 32 over 16 k
template <int TM, typename V>
__device__ __forceinline__ V mfma_bf16(u32x4 a, u32x4 b, V c) {
  if constexpr (TM == 16)
    return mfma_bf16_16x16x32(a, b, c);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// silu(g) * u by the hardware exp2 and reciprocal (about 1 ulp each, and the
// rounding of g log2 e under exp2) instead of silu_mul's expf and division, for
// tiles of more than 32 tokens in calls of GEMM_MIN_T or more, whose epilogue is
// VALU-bound: silu_mul there too takes 3% of such layers (us, H2048 E512 k10
// I512 T4096: 519 -> 535; H2560 E96 k6 I896 T2048: 459 -> 468; H4096 I1024
// T4096: 1820 -> 1841).  The other tiles wait for their weights, and silu_mul
// costs them at most 1% (T192 214 -> 215, T1500 286 -> 289, H2560 E96 T301 166.5
// either way).  An act differs by a few units of its last fp32 place, which its
// rounding to bf16 hides but for about one value in 65000.
// Large |g| behaves: exp2 -> inf gives rcp 0 and g * 0; exp2 -> 0 gives g.
__device__ __forceinline__ float silu_mul_fast(float g, float u) {
  const float e = __builtin_amdgcn_exp2f(g * -1.44269504088896341f);
  return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
}

// Byte selectors for v_perm_b32(recv, own, sel) in the epilogues' pair
// exchange: a lane holds rows (0, 1) of its column as own = r0 | r1 << 16
// (lower lane of the pair) or rows (2, 3) (upper lane), sends the other two
// rows to its partner and builds two dwords, each one row of the column
// pair (lower column in the low half).  Selector bytes 0-3 take own, 4-7
// recv.
__device__ __forceinline__ uint32_t pair_sel(bool upper, int d) {
  return upper ? (d == 0 ? 0x01000504u : 0x03020706u) : (d == 0 ? 0x05040100u : 0x07060302u);
}

// One item: expert tile lb / n_nblk (its entry t), column block lb % n_nblk.
template <int SD, int MODE, int WN>
__device__ __forceinline__ void gemm_item(const GemmArgs &a, const int lb, const int4 t) {
  using Gm = Geo<WN>;
  constexpr int BN = Gm::BN, NW = Gm::NW, THREADS = Gm::THREADS, COLS = Gm::COLS;
  // dynamic LDS: the ring; the epilogue's staging and row sums reuse it
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int n_nb = a.n_nblk;
  const int nb = lb % n_nb;
  const int e = t.x, pos0 = t.y, mcnt = t.z;
  const bool shared = e == a.E;
  // MODE 0: N = act columns (I or Is), block covers COLS of them; MODE 1: N = H, BN rows
  const int N = MODE == 0 ? (shared ? a.Is : a.I) : a.H;
  const int K = MODE == 0 ? a.H : (shared ? a.Is : a.I);
  const int G = K >> 7;
  if (nb * (MODE == 0 ? COLS : BN) >= N) return;

  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  GTRACE(const unsigned long long t0 = __builtin_amdgcn_s_memtime());
  const int tid = tid_opaque();  // per item: nothing lane-dependent is hoisted across items
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int wn = wave;

  // ---- per-thread DMA sources: A_DMA A slots and B_DMA B slots per stage ---
  // slot s = (i*NW + wave)*64 + lane, 16 bytes each.  The block-uniform part
  // of each address is a scalar base (advanced per group); a lane keeps one
  // 32-bit offset per slot.
  const uint8_t *abase;
  uint32_t aoff[Gm::A_DMA];
  if (MODE == 0)
    abase = (const uint8_t *)(a.a_routed + (shared ? (size_t)pos0 * a.H : 0));
  else
    abase = (const uint8_t *)((shared ? a.a_shared : a.a_routed) + (size_t)pos0 * K);
#pragma unroll
  for (int i = 0; i < Gm::A_DMA; ++i) {
    const int s = (i * NW + wave) * 64 + lane;
    const int r = s >> 4, c = (s & 15) ^ aswz(r);
    const int rr = min(r, mcnt - 1);
    // MODE 0 routed: a gathered token row, tok < T <= 4096 and H <= 4096
    const uint32_t row = MODE == 0 && !shared ? (uint32_t)a.ptok[pos0 + rr] : (uint32_t)rr;
    aoff[i] = row * (uint32_t)(MODE == 0 ? a.H : K) * 2u + (uint32_t)c * 16u;
  }
  const size_t rowb = (size_t)K / 2;
  const uint8_t *bbase[Gm::B_DMA];
  uint32_t boff[Gm::B_DMA];
#pragma unroll
  for (int i = 0; i < Gm::B_DMA; ++i) {
    const int s = (i * NW + wave) * 64 + lane;
    const int r = s >> 2, qq = (s & 3) ^ bswz(r);
    // the 16 B-rows of one (i, wave) lie on one side of COLS (16 | COLS)
    const int r0 = (i * NW + wave) * 16;
    int row;
    if (MODE == 0) {  // B-rows [0, COLS) gate, [COLS, 2 COLS) up
      bbase[i] = r0 < COLS ? (shared ? a.ws0 : a.w0 + (size_t)e * N * rowb)
                           : (shared ? a.ws1 : a.w1 + (size_t)e * N * rowb);
      row = nb * COLS + (r % COLS);
    } else {
      bbase[i] = shared ? a.ws0 : a.w0 + (size_t)e * N * rowb;
      row = nb * BN + r;
    }
    row = min(row, N - 1);
    boff[i] = (uint32_t)row * (uint32_t)rowb + (uint32_t)qq * 16u;
  }
  // 16-token subtiles that hold tokens (block-uniform): A slot i of a stage is
  // subtile i's rows, so the subtiles past the count are not copied
  const int nms = __builtin_amdgcn_readfirstlane(min(4, (mcnt + 15) >> 4));
  static_assert(Gm::A_DMA == 4 && NW == 4, "A slot i holds the rows of token subtile i");
  // scales: wave w copies B rows [64 w, +64), lane l the aligned dword that
  // holds row 64 w + l's scale of the group (the tensor's rows are a multiple
  // of 128, so the dword never ends past it); group sums: lane l token row l
  const uint16_t *sbase;
  uint32_t soff, xoff;
  const float *xbase;
  {
    const int r = wave * 64 + lane;
    int row;
    if (MODE == 0) {
      sbase = wave * 64 < COLS ? (shared ? a.ss0 : a.s0 + (size_t)e * N * G)
                               : (shared ? a.ss1 : a.s1 + (size_t)e * N * G);
      row = nb * COLS + (r % COLS);
    } else {
      sbase = shared ? a.ss0 : a.s0 + (size_t)e * N * G;
      row = nb * BN + r;
    }
    soff = (uint32_t)(min(row, N - 1) * G) * 2u;
    const int rr = min(lane, mcnt - 1);
    if (MODE == 0) {
      xbase = a.xsum + (shared ? (size_t)pos0 * G : 0);
      xoff = (uint32_t)((shared ? rr : a.ptok[pos0 + rr]) * G) * 4u;
    } else {
      xbase = (shared ? a.asum_s : a.asum) + (size_t)pos0 * G;
      xoff = (uint32_t)(rr * G) * 4u;
    }
  }
  const uint64_t abase_s = sbase64(abase), sbase_s = sbase64(sbase), xbase_s = sbase64(xbase);
  uint64_t bbase_s[Gm::B_DMA];
#pragma unroll
  for (int i = 0; i < Gm::B_DMA; ++i) bbase_s[i] = sbase64(bbase[i]);
  // DMA of group g into the ring stage at `base`, NMS token subtiles
  // (NMS + B_DMA + 2 instructions per wave; at NMS = 4 one fewer for a tile
  // of three subtiles)
  auto issue = [&](auto nms_c, int g, uint32_t base) {
    constexpr int NMS = decltype(nms_c)::value;
    constexpr uint32_t BO = NMS * Gm::A_SUB, SO = BO + Gm::B_STAGE, XO = SO + BN * 4;
#pragma unroll
    for (int i = 0; i < Gm::B_DMA; ++i)
      dma16s(boff[i], bbase_s[i] + (uint32_t)g * 64u, base + BO + (uint32_t)((i * NW + wave) * 1024));
    dma4s((soff + 2u * (uint32_t)g) & ~3u, sbase_s, base + SO + (uint32_t)(wave * 256));
#pragma unroll
    for (int i = 0; i < NMS; ++i)
      if (NMS < 4 || i < nms) dma16s(aoff[i], abase_s + (uint32_t)g * 256u, base + (uint32_t)((i * NW + wave) * 1024));
    // (every wave copies the same 64 sums: equal instruction counts)
    dma4s(xoff, xbase_s + (uint32_t)g * 4u, base + XO);
  };

  // The main loop and epilogue on token tiles of TM: MS tiles of TM tokens
  // x NS tiles of TM weight rows per wave (TM * NS = 64), NSUB = MS * TM / 16
  // subtiles in the ring.
  auto run = [&](auto tm_c, auto ms_c) {
    GTRACE(const unsigned long long t1 = __builtin_amdgcn_s_memtime());
    constexpr int TM = decltype(tm_c)::value, MS = decltype(ms_c)::value;
    constexpr int NS = 64 / TM, NSUB = MS * TM / 16, NSL = TM / 4;  // k-slices per group
    constexpr int NP = TM / 16;  // 32-k blocks of a row per lane
    constexpr int NQ = TM == 16 ? 1 : 4;  // row quads a lane holds of a tile
    using acc_t = typename std::conditional<TM == 16, f32x4, f32x16>::type;
    using nsub_t = std::integral_constant<int, NSUB>;
    constexpr int STAGE = Gm::stage(NSUB), STAGES = Gm::stages(NSUB);
    constexpr uint32_t BO = NSUB * Gm::A_SUB, SO = BO + Gm::B_STAGE, XO = SO + BN * 4;
    constexpr int PER = NSUB + Gm::B_DMA + 2;  // DMA instructions per wave and group
    issue(nsub_t(), 0, lds0);
    if (STAGES > 2 && G > 1) issue(nsub_t(), 1, lds0 + STAGE);
    // lane (Q, rl): row rl of a tile, 32-k blocks NP * Q'.. of the group: slice
    // s of TM = 16 is nibble pair s of block Q; slice s = 4 p + j of TM = 32
    // is nibble pair j of block 2 p + Q
    const int rl = lane & (TM - 1), Q = lane / TM;
    auto blk = [&](int p) { return TM == 16 ? Q : 2 * p + Q; };
    // B-rows of the wave's NS row tiles: brow0 + brow(ns); the tiles' LDS
    // addresses differ by constants (bswz depends on the row's low 4 bits)
    auto brow = [](int ns) {
      return MODE == 0 ? (ns < NS / 2 ? ns * TM : COLS + (ns - NS / 2) * TM) : ns * TM;
    };
    const int brow0 = (MODE == 0 ? wn * 32 : wn * 64) + rl;
    const uint32_t soffl = (uint32_t)(brow0 * 4);
    uint32_t boffl[NP], aoffl[NSL];
#pragma unroll
    for (int p = 0; p < NP; ++p) boffl[p] = (uint32_t)(brow0 * 64 + ((blk(p) ^ bswz(rl)) << 4));
#pragma unroll
    for (int s = 0; s < NSL; ++s)
      aoffl[s] = (uint32_t)(rl * 256 + (((4 * blk(s >> 2) + (s & 3)) ^ aswz(rl)) << 4));
    // the half of a row's scale dword that holds group 0's scale (odd G: every
    // other row; the same for all row tiles, whose rows differ by even numbers)
    uint32_t ssh = ((uint32_t)(brow0 * G) & 1u) * 16u;
    uint32_t magic;
    asm volatile("v_mov_b32 %0, 0x41C041C0" : "=v"(magic));
    // acc and sprev start at zero, so the scale step of "group -1" adds
    // +0 * +0 to tot's +0 and leaves it unchanged (no branch in the loop)
    acc_t tot[MS][NS], acc[MS][NS];
    float sg[NS], sprev[NS];
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) {
      sprev[ns] = 0.f;
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int i = 0; i < 4 * NQ; ++i) tot[ms][ns][i] = acc[ms][ns][i] = 0.f;
    }
    auto scale_step = [&]() {
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int ms = 0; ms < MS; ++ms) tot[ms][ns] += sprev[ns] * acc[ms][ns];
    };
    // One barrier per group.  At the top of iteration g every wave has
    // issued all its MFMAs of group g-1 (they may still be executing) and
    // has read its last fragment of stage g-1, so after the barrier a DMA may
    // overwrite that stage: group g+1 (2 stages) or g+2 (3 stages).
    int si = 0, sf = STAGES - 1;  // stages of group g and of the group to fill
    for (int g = 0; g < G; ++g) {
      // this thread's DMA of group g has landed (at 3 stages group g+1's,
      // issued after it, may be in flight)
      if (STAGES > 2 && g + 1 < G)
        wait_vm<PER>();
      else
        wait_vm<0>();
      block_barrier();  // and every thread's
      if (g + STAGES - 1 < G) issue(nsub_t(), g + STAGES - 1, lds0 + (uint32_t)(sf * STAGE));
      const uint8_t *st = lds + si * STAGE;
      // this wave's raw B chunks and scales, and the scale step of group g-1
      u32x4 bx[NS][NP];
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int ns = 0; ns < NS; ++ns)
          bx[ns][p] = *(const u32x4 *)(st + boffl[p] + BO + brow(ns) * 64);
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
        sg[ns] = scale_to_f32<SD>((uint16_t)(*(const uint32_t *)(st + soffl + SO + brow(ns) * 4) >> ssh));
      ssh ^= 16u;
      scale_step();
      // group sums (-24 sum_k a): the first k-slice accumulates onto them
      acc_t c0[MS];
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
          const f32x4 v = *(const f32x4 *)(st + XO + (ms * TM + 8 * i + 4 * Q) * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) c0[ms][4 * i + r] = v[r];
        }
      // A fragments one k-slice ahead, and each row tile's B operand of slice
      // s+1 unpacked right after its last use in slice s, so the unpacking
      // issues between MFMAs; the scheduling barrier after each slice keeps
      // the compiler from hoisting all reads to the top (spills)
      u32x4 af[2][MS], bf[NS];
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) af[0][ms] = *(const u32x4 *)(st + aoffl[0] + ms * TM * 256);
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) bf[ns] = nib_slice3(bx[ns][0], 0, magic);
#pragma unroll
      for (int s = 0; s < NSL; ++s) {
        if (s + 1 < NSL) {
#pragma unroll
          for (int ms = 0; ms < MS; ++ms)
            af[(s + 1) & 1][ms] = *(const u32x4 *)(st + aoffl[(s + 1) % NSL] + ms * TM * 256);
        }
#pragma unroll
        for (int ns = 0; ns < NS; ++ns) {
#pragma unroll
          for (int ms = 0; ms < MS; ++ms)
            acc[ms][ns] = mfma_bf16<TM>(af[s & 1][ms], bf[ns], s == 0 ? c0[ms] : acc[ms][ns]);
          if (s + 1 < NSL) bf[ns] = nib_slice3(bx[ns][((s + 1) / 4) % NP], (s + 1) & 3, magic);
        }
        // slice 0 also holds the scale step's fmas: left to the compiler
        if (s > 0) {
#pragma unroll
          for (int i = 0; i < NS * MS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            if (s + 1 < NSL) {
              __builtin_amdgcn_sched_group_barrier(0x002, 8 / MS, 0);  // VALU
              if (i < MS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            } else {
              __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) sprev[ns] = sg[ns];
      si = si + 1 == STAGES ? 0 : si + 1;
      sf = sf + 1 == STAGES ? 0 : sf + 1;
    }
    scale_step();
    wait_vm<0>();  // no DMA into the ring remains in flight
    block_barrier();  // every wave's last read of the ring precedes the staging below
    GTRACE(if (tid == 0 && lb < 16384) {
      const int o = (MODE * 16384 + lb) * 4;
      g_gtrace[o] = t0;
      g_gtrace[o + 1] = t1;
      g_gtrace[o + 2] = __builtin_amdgcn_s_memtime();
    });

    // ---- epilogue -------------------------------------------------------
    // A lane holds quad i (4 consecutive tokens) of tile (ms, ns): rows
    // ms * TM + 8 i + 4 Q + [0, 4), column ns * TM + rl.  Results are staged
    // in the (now idle) LDS ring and leave as 16-byte row chunks.  The lanes
    // of a column pair trade halves so that each stores whole dwords (the
    // lower lane tokens 0 and 1 of the quad, the upper 2 and 3): 2-byte LDS
    // stores cost several times a dword store.  Branch-free: the selects are
    // plain values and v_perm_b32 takes a per-lane selector.
    if constexpr (MODE == 0) {
      constexpr int OST = COLS * 2 + 16;  // staged row stride, bytes
      static_assert(BM * OST <= Gm::RING, "staging exceeds the ring");
      // columns k and k + 4 of a 32-column block are neighbours in MFMA order
      // (perm32_pos), and live in lanes rl and rl ^ 4
      const bool hi4 = (rl & 4) != 0;
      const uint32_t sel0 = pair_sel(hi4, 0), sel1 = pair_sel(hi4, 1);
      auto stage = [&](auto fast) {
#pragma unroll
        for (int ns = 0; ns < NS / 2; ++ns) {
          // within a 32-aligned block of columns, MFMA order is block-local
          const int p = perm32_pos(wn * 32 + ns * TM + (rl & ~4));  // the pair's even position
#pragma unroll
          for (int ms = 0; ms < MS; ++ms)
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
              float f[4];
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const float gv = tot[ms][ns][4 * i + r], uv = tot[ms][ns + NS / 2][4 * i + r];
                f[r] = decltype(fast)::value ? silu_mul_fast(gv, uv) : silu_mul(gv, uv);
              }
              const uint32_t p01 = bf16x2_bits(f[0], f[1]), p23 = bf16x2_bits(f[2], f[3]);
              const uint32_t send = hi4 ? p01 : p23, own = hi4 ? p23 : p01;
              // lane ^ 4 inside each group of 32 lanes (ds_swizzle bit mode)
              const uint32_t recv = (uint32_t)__builtin_amdgcn_ds_swizzle((int)send, 0x101F);
              const int row0 = ms * TM + 8 * i + 4 * Q + (hi4 ? 2 : 0);
              *(uint32_t *)(lds + row0 * OST + p * 2) = __builtin_amdgcn_perm(recv, own, sel0);
              *(uint32_t *)(lds + (row0 + 1) * OST + p * 2) = __builtin_amdgcn_perm(recv, own, sel1);
            }
        }
      };
      if (NSUB > 2 && a.T >= GEMM_MIN_T)
        stage(std::true_type());
      else
        stage(std::false_type());
      __syncthreads();
      uint16_t *dst = shared ? a.act_s : a.act;
      float *as = shared ? a.asum_s : a.asum;
      constexpr int CPR = COLS / 8;  // 16-byte chunks per row
      static_assert(CPR == 16, "a DPP row of lanes holds one act row");
      constexpr int NST = NSUB * 16 * CPR / THREADS;
      u32x4 out[NST];  // every LDS read before the (predicated) stores
#pragma unroll
      for (int i = 0; i < NST; ++i) {
        const int idx = tid + i * THREADS;
        out[i] = *(const u32x4 *)(lds + (idx / CPR) * OST + (idx % CPR) * 16);
      }
#pragma unroll
      for (int i = 0; i < NST; ++i) {
        const int idx = tid + i * THREADS, row = idx / CPR, c = idx % CPR;
        if (row < mcnt) *(u32x4 *)(dst + (size_t)(pos0 + row) * N + nb * COLS + c * 8) = out[i];
        // the row's sum over this block's 128 columns (one k-group of down)
        float v = 0.f;
#pragma unroll
        for (int d = 0; d < 4; ++d)
          v += __uint_as_float(out[i][d] << 16) + __uint_as_float(out[i][d] & 0xFFFF0000u);
        v = row16_sum(v);
        if (c == 0 && row < mcnt) as[(size_t)(pos0 + row) * (N / COLS) + nb] = -GEMM_NIB_OFFSET * v;
      }
    } else {
      constexpr int OST = BN * 2 + 16;
      static_assert(BM * OST <= Gm::RING, "staging exceeds the ring");
      // neighbouring columns live in lanes rl and rl ^ 1
      const bool odd = (rl & 1) != 0;
      const uint32_t sel0 = pair_sel(odd, 0), sel1 = pair_sel(odd, 1);
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) {
        const int cl = wn * 64 + TM * ns + (rl & ~1);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
          for (int i = 0; i < NQ; ++i) {
            const acc_t &v = tot[ms][ns];
            const uint32_t p01 = bf16x2_bits(v[4 * i], v[4 * i + 1]);
            const uint32_t p23 = bf16x2_bits(v[4 * i + 2], v[4 * i + 3]);
            const uint32_t send = odd ? p01 : p23, own = odd ? p23 : p01;
            const uint32_t recv =
                (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send, 0xB1, 0xF, 0xF, false);  // lane ^ 1
            const int row0 = ms * TM + 8 * i + 4 * Q + (odd ? 2 : 0);
            *(uint32_t *)(lds + row0 * OST + cl * 2) = __builtin_amdgcn_perm(recv, own, sel0);
            *(uint32_t *)(lds + (row0 + 1) * OST + cl * 2) = __builtin_amdgcn_perm(recv, own, sel1);
          }
      }
      __syncthreads();
      constexpr int CPR = BN / 8;
      constexpr int NST = NSUB * 16 * CPR / THREADS;
      u32x4 out[NST];  // every LDS read before the (predicated) stores
#pragma unroll
      for (int i = 0; i < NST; ++i) {
        const int idx = tid + i * THREADS;
        out[i] = *(const u32x4 *)(lds + (idx / CPR) * OST + (idx % CPR) * 16);
      }
#pragma unroll
      for (int i = 0; i < NST; ++i) {
        const int idx = tid + i * THREADS, row = idx / CPR, c = idx % CPR;
        const int col = nb * BN + c * 8;
        if (row < mcnt && col < N) {
          const size_t orow = shared ? (size_t)a.T * a.k + pos0 + row : (size_t)(pos0 + row);
          *(u32x4 *)(a.o + orow * a.H + col) = out[i];
        }
      }
    }
  };
  // 33 to 64 tokens: 2 x 2 tiles of 32 (a third subtile's missing partner
  // costs MFMAs but no copy; its rows are never stored); 17 to 32: 1 x 2; up
  // to 16: the 16-wide tiles
  using std::integral_constant;
  if (nms > 2)
    run(integral_constant<int, 32>(), integral_constant<int, 2>());
  else if (nms > 1)
    run(integral_constant<int, 32>(), integral_constant<int, 1>());
  else
    run(integral_constant<int, 16>(), integral_constant<int, 1>());
}

// One block per item.  The items a launch's blocks take are XCD-contiguous
// (xcd_remap over the device's item count, so every XCD gets an equal share
// whatever the host's tile bound), which keeps the column blocks of one
// expert tile, and the tiles of one expert, on one XCD: they share A rows and
// weights through that L2.
template <int SD, int MODE, int WN>
__global__ __launch_bounds__(64 * WN, 2) void k_expert_gemm(GemmArgs a) {
  const int n_items = *a.n_tiles * a.n_nblk;
  if ((int)blockIdx.x >= n_items) return;
  const int lb = xcd_remap(blockIdx.x, n_items);
  gemm_item<SD, MODE, WN>(a, lb, a.tiles[lb / a.n_nblk]);
  GTRACE(__syncthreads(); if (threadIdx.x == 0 && lb < 16384) g_gtrace[(MODE * 16384 + lb) * 4 + 3] =
             __builtin_amdgcn_s_memtime());
}

// ---------------------------------------------------------------------------
// Router logits for prefill: approx[t][e] = sum_k x[t][k] * w[e][k] (+ bias)
// on bf16 MFMA, fp32 accumulation.  Block tile: BM tokens x BN experts, 4 waves
// as 2 (tokens) x 2 (experts).  K streams through an LDS ring of ST stages in
// 64-wide steps (x rows and w rows, 128 bytes each, 16-byte chunk c of row r
// stored at c ^ (r & 7)).  The blocks after the GEMM tiles compute ||w_e||
// (used only as the bound of the canonical refine).
//
// A block is a serial chain of H / 64 steps, each a barrier, the DMA issue, the
// LDS reads and the MFMAs of one wave per SIMD, so a step costs what its tile
// moves (64 x 128: 0.62 us, 64 x 64: 0.41, 32 x 64: 0.30) and a deeper ring
// changes nothing (3 and 6 stages: 20.2, 20.6 us).  Hence the smallest tile whose
// items still have a CU each, and the largest, which reads the least, once none
// has.  us with 64 x 128 always -> now: E512 H2048 T512 19.5 -> 10.4 (32 x 64),
// T1024 20.1 -> 11.2, T1500 20.5 -> 13.6 (64 x 64; 32 x 64: 15.9), T2048 20.9 ->
// 14.9, T4096 23.0 -> 22.1 (64 x 128; 64 x 64: 24.9, 32 x 64: 29.6); E96 H2560 T301
// 24.4 -> 12.0.
// ---------------------------------------------------------------------------
constexpr int RG_BK = 64;
constexpr int RG_FILL = 256;  // items that leave no CU idle
constexpr int RG_NORM_ROWS = 16;                // experts per norm block

template <int BM, int BN, int ST>
struct RouterGeo {
  static constexpr int A = BM * RG_BK * 2, STAGE = A + BN * RG_BK * 2;  // bytes
  static constexpr int DMA = STAGE / (256 * 16);                       // per thread per stage
  static constexpr int LDS = ST * STAGE;
  static_assert((ST - 2) * DMA < 64, "vmcnt");
};

// all but the newest N * D of this wave's DMAs done (n <= N, wave-uniform)
template <int D, int N>
__device__ __forceinline__ void wait_stages(int n) {
  if constexpr (N > 0) {
    if (n < N) return wait_stages<D, N - 1>(n);
  }
  wait_vm<N * D>();
}

template <int BM, int BN, int ST>
__global__ __launch_bounds__(256) void k_router_gemm(const uint16_t *__restrict__ x,
                                                     const uint16_t *__restrict__ rw,
                                                     const float *__restrict__ bias,
                                                     float *__restrict__ approx,
                                                     float *__restrict__ wnorm, int T, int H,
                                                     int E, int n_mt, int n_nt,
                                                     uint32_t *__restrict__ zbuf, int zwords) {
  using Rg = RouterGeo<BM, BN, ST>;
  constexpr int MS = BM / 32, NS = BN / 32;  // 16-row MFMA tiles per wave
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n_items = n_mt * n_nt;
  if ((int)blockIdx.x >= n_items) {
    // ---- the dispatch counts and masks k_select fills next start at zero --
    const int nb = (int)gridDim.x - n_items, b = (int)blockIdx.x - n_items;
    for (int i = b * 256 + tid; i < zwords; i += nb * 256) zbuf[i] = 0u;
    // ---- row norms: wave w takes rows e0 + 4w .. e0 + 4w + 3 -------------
    const int e0 = ((int)blockIdx.x - n_items) * RG_NORM_ROWS + wave * 4;
    for (int r = 0; r < 4; ++r) {
      const int e = e0 + r;
      if (e >= E) break;
      const uint16_t *row = rw + (size_t)e * H;
      float ss = 0.0f;
      for (int c = lane; c < (H >> 3); c += 64) {
        const u32x4 v = *(const u32x4 *)(row + 8 * c);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const float lo = __uint_as_float(v[d] << 16), hi = __uint_as_float(v[d] & 0xFFFF0000u);
          ss = __builtin_fmaf(lo, lo, ss);
          ss = __builtin_fmaf(hi, hi, ss);
        }
      }
      for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
      if (lane == 0) wnorm[e] = sqrtf(ss);
    }
    return;
  }
  const int lb = xcd_remap(blockIdx.x, n_items);
  const int mt = lb / n_nt, nt = lb % n_nt;  // the n_nt expert tiles of a token tile share an XCD
  const int t0 = mt * BM, e0 = nt * BN;
  const int wm = wave & 1, wn = wave >> 1;
  const int m16 = lane & 15, q = lane >> 4;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

  // DMA sources: slot s = (i*4 + wave)*64 + lane; row s/8, stored chunk s%8
  const uint8_t *src[Rg::DMA];
#pragma unroll
  for (int i = 0; i < Rg::DMA; ++i) {
    const int sl = (i * 4 + wave) * 64 + lane;
    const int r = sl >> 3, c = (sl & 7) ^ (r & 7);
    if (r < BM) {
      src[i] = (const uint8_t *)(x + (size_t)min(t0 + r, T - 1) * H) + c * 16;
    } else {
      src[i] = (const uint8_t *)(rw + (size_t)min(e0 + r - BM, E - 1) * H) + c * 16;
    }
  }
  auto issue = [&](int g) {
    const uint32_t base = lds0 + (uint32_t)(g % ST) * Rg::STAGE;
#pragma unroll
    for (int i = 0; i < Rg::DMA; ++i)
      dma16(src[i] + g * (RG_BK * 2), base + (uint32_t)((i * 4 + wave) * 1024));
  };
  const int G = H / RG_BK;
  for (int g = 0; g < min(ST - 1, G); ++g) issue(g);
  f32x4 acc[MS][NS];
#pragma unroll
  for (int ms = 0; ms < MS; ++ms)
#pragma unroll
    for (int ns = 0; ns < NS; ++ns) acc[ms][ns] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int g = 0; g < G; ++g) {
    // stage g is there for every wave, and stage g - 1 read by every wave: its
    // place takes stage g + ST - 1
    wait_stages<Rg::DMA, ST - 2>(min(ST - 2, G - 1 - g));
    block_barrier();
    if (g + ST - 1 < G) issue(g + ST - 1);
    const uint8_t *sa = lds + (g % ST) * Rg::STAGE, *sb = sa + Rg::A;
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {  // two 32-wide MFMA steps
      u32x4 af[MS], bf[NS];
#pragma unroll
      for (int ms = 0; ms < MS; ++ms) {
        const int r = wm * (BM / 2) + ms * 16 + m16;
        af[ms] = *(const u32x4 *)(sa + r * 128 + (((4 * s2 + q) ^ (r & 7)) << 4));
      }
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) {
        const int r = wn * (BN / 2) + ns * 16 + m16;
        bf[ns] = *(const u32x4 *)(sb + r * 128 + (((4 * s2 + q) ^ (r & 7)) << 4));
      }
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int ns = 0; ns < NS; ++ns) acc[ms][ns] = mfma_bf16_16x16x32(af[ms], bf[ns], acc[ms][ns]);
    }
  }
  // lane (q, m16) of tile (ms, ns): tokens wm BM/2 + 16 ms + 4 q + r, expert wn BN/2 + 16 ns + m16
#pragma unroll
  for (int ns = 0; ns < NS; ++ns) {
    const int e = e0 + wn * (BN / 2) + ns * 16 + m16;
    if (e >= E) continue;
    const float b = bias ? bias[e] : 0.0f;
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = t0 + wm * (BM / 2) + ms * 16 + 4 * q + r;
        if (t < T) approx[(size_t)t * E + e] = bias ? acc[ms][ns][r] + b : acc[ms][ns][r];
      }
  }
}

template <int WN>
hipError_t launch_geo(int mode, int scale_dtype, GemmArgs a, int max_tiles, hipStream_t s) {
  using Gm = Geo<WN>;
  const int Nmax = mode == 0 ? (a.I > a.Is ? a.I : a.Is) : a.H;
  a.n_nblk = mode == 0 ? (Nmax + Gm::COLS - 1) / Gm::COLS : (Nmax + Gm::BN - 1) / Gm::BN;
  const long grid = (long)max_tiles * a.n_nblk;
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  // the group sums of act: MODE 0 writes one per COLS = 128 columns
  static_assert(Gm::COLS == 128, "one act sum per k-group");
  constexpr size_t lds = Gm::RING;
  static_assert(2 * lds <= 160 * 1024, "two blocks per CU");
  void (*kern)(GemmArgs);
  if (mode == 0)
    kern = scale_dtype == AINFER_SCALE_FP16 ? k_expert_gemm<AINFER_SCALE_FP16, 0, WN>
                                            : k_expert_gemm<AINFER_SCALE_BF16, 0, WN>;
  else
    kern = scale_dtype == AINFER_SCALE_FP16 ? k_expert_gemm<AINFER_SCALE_FP16, 1, WN>
                                            : k_expert_gemm<AINFER_SCALE_BF16, 1, WN>;
  kern<<<(unsigned)grid, Gm::THREADS, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_router_gemm(const void *x, const void *rw, const float *bias, float *approx,
                              float *wnorm, int T, int H, int E, uint32_t *zbuf, int zwords,
                              hipStream_t s) {
  if (T <= 0) return hipSuccess;
  if (H % RG_BK) return hipErrorInvalidValue;
  const int n_norm = (E + RG_NORM_ROWS - 1) / RG_NORM_ROWS;
  auto launch = [&](auto kern, int bm, int bn, int lds) {
    const int n_mt = (T + bm - 1) / bm, n_nt = (E + bn - 1) / bn;
    kern<<<(unsigned)(n_mt * n_nt + n_norm), 256, lds, s>>>(
        (const uint16_t *)x, (const uint16_t *)rw, bias, approx, wnorm, T, H, E, n_mt, n_nt,
        zbuf, zbuf ? zwords : 0);
  };
  const long m32 = (T + 31) / 32, m64 = (T + 63) / 64, n64 = (E + 63) / 64;
  if (m32 * n64 <= RG_FILL)
    launch(k_router_gemm<32, 64, 4>, 32, 64, RouterGeo<32, 64, 4>::LDS);
  else if (m64 * n64 <= RG_FILL)
    launch(k_router_gemm<64, 64, 4>, 64, 64, RouterGeo<64, 64, 4>::LDS);
  else
    launch(k_router_gemm<64, 128, 3>, 64, 128, RouterGeo<64, 128, 3>::LDS);
  return hipGetLastError();
}

// Both GEMM modes of one forward must use the same geometry (MODE 1 reads
// the act partial sums MODE 0 wrote).
hipError_t launch_expert_gemm(int mode, int scale_dtype, GemmArgs a, int max_tiles,
                              hipStream_t s) {
  if (max_tiles <= 0) return hipSuccess;
  return launch_geo<GEMM_WN>(mode, scale_dtype, a, max_tiles, s);
}

// ---------------------------------------------------------------------------
// MFMA-rate probe: every wave issues ITERS x 16 independent
// v_mfma_f32_16x16x32_bf16 (16 accumulator tiles) with NV independent fp32
// FMAs after each, so the rate it reports is the ceiling of a main loop that
// spends NV VALU instructions per MFMA.  One block per CU of 64 * 4 * WPS
// threads (WPS waves per SIMD).  The results are stored only when iters < 0,
// which never holds, so nothing is written and nothing is optimised away.
// ---------------------------------------------------------------------------
namespace {
template <int NV>
__global__ void k_mfma_probe(float *sink, int iters) {
  f32x4 acc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 a, b;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a[i] = 0x3F803F80u + threadIdx.x + i;
    b[i] = 0x3F803F80u + 3u * threadIdx.x + i;
  }
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (float)threadIdx.x * 0.001f + (float)i;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      acc[m] = mfma_bf16_16x16x32(a, b, acc[m]);
#pragma unroll
      for (int j = 0; j < NV; ++j) v[j & 7] = __builtin_fmaf(v[j & 7], 1.0001f, 0.5f);
    }
  }
  if (iters < 0) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) s += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
#pragma unroll
    for (int i = 0; i < 8; ++i) s += v[i];
    sink[threadIdx.x] = s;
  }
}
}  // namespace

extern "C" int ainfer_moe_mfma_probe(int32_t valu_per_mfma, int32_t waves_per_simd, int32_t iters,
                                     void *stream, float *tflops) {
  if (!tflops || iters <= 0 || iters > (1 << 20) || waves_per_simd < 1 || waves_per_simd > 4 ||
      valu_per_mfma < 0 || valu_per_mfma > 4)
    return AINFER_ERR_ARG;
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return AINFER_ERR_HIP;
  const hipStream_t s = (hipStream_t)stream;
  const dim3 grid((unsigned)cus), block(256u * (unsigned)waves_per_simd);
  auto launch = [&]() {
    switch (valu_per_mfma) {
      case 0: k_mfma_probe<0><<<grid, block, 0, s>>>(nullptr, iters); break;
      case 1: k_mfma_probe<1><<<grid, block, 0, s>>>(nullptr, iters); break;
      case 2: k_mfma_probe<2><<<grid, block, 0, s>>>(nullptr, iters); break;
      case 3: k_mfma_probe<3><<<grid, block, 0, s>>>(nullptr, iters); break;
      case 4: k_mfma_probe<4><<<grid, block, 0, s>>>(nullptr, iters); break;
      default: return false;
    }
    return true;
  };
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return AINFER_ERR_HIP;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return AINFER_ERR_HIP;
  }
  int rc = 0;
  float ms = 0.f;
  if (!launch()) {
    rc = AINFER_ERR_ARG;
  } else if (hipEventRecord(e0, s) != hipSuccess || !launch() || hipEventRecord(e1, s) != hipSuccess ||
             hipEventSynchronize(e1) != hipSuccess || hipEventElapsedTime(&ms, e0, e1) != hipSuccess ||
             hipGetLastError() != hipSuccess) {
    rc = AINFER_ERR_HIP;
  } else {
    const double flop = (double)cus * 4 * waves_per_simd * iters * 16 * (2.0 * 16 * 16 * 32);
    *tflops = (float)(flop / (ms * 1e-3) / 1e12);
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}
