// moe_gemm_w4a8.hip - the layer's expert GEMVs in W4A8 from 2 tokens on
// (w4a8_gemm_at, moe_internal.h), as a grouped int8 MFMA GEMM.
//
// Arithmetic: Int4Gemv's (tools/cmdlist/kernels.cpp:148-201) per (token,
// expert), bit for bit: the group dot gs = sum q * x exact in int32, its term
// float(gs) * s_w * s_x rounded product by product (no contraction), the
// terms added in group order from 0.
//
// The block, the ring and the tile shapes are moe_gemm.hip's: at most 64
// tokens x 256 weight rows (MODE 0: 128 gate and the matching 128 up rows),
// 4 waves of 64 rows, two blocks per CU, one 128-wide group per barrier.  A
// ring stage holds the int8 token rows (64 x 128 B), the raw INT4 rows, a
// dword per weight row with its scale, and per token row its scale and
// -8 x its code sum; three stages fit 80 KB at every tile height, so two
// groups are in flight.
//  - A nibble as a byte 8 + q is one v_bitop3 (even elements) or a shift and
//    one (odd); int32 accumulators start at -8 sum x, so they end at gs.
//    Activation codes are in W8 order (write_xperm): the 16 even elements of a
//    32-element block, then the 16 odd ones, the order those bytes come in.
//  - v_mfma_i32_32x32x32_i8 above 16 tokens, 16x16x64 up to 16.
//  - MODE 0's 128 columns are one quantization group of act: the epilogue
//    takes SiLU in fp32 (SiluMul, kernels.cpp:29-37), stages the rows in LDS
//    and writes the codes, scales and sums the down GEMM reads, so act never
//    goes to memory in fp32 and its quantization is no launch.
//
// Bound: the terms.  Each output takes a conversion, two products and an
// addition per group (256 VALU instructions per wave and group at 64 tokens,
// beside 48 of unpacking and 16 MFMAs), so full tiles are VALU-bound; at few
// tokens per expert the weights' stream is the bound.
#include <type_traits>

#include "moe_common.h"
#include "moe_internal.h"
#include "moe_gemm_parts.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = GEMM_MT, BN = 256, COLS = 128, NW = 4, THREADS = 256;
constexpr int B_STAGE = BN * 64;
// one ring stage at NSUB 16-token subtiles (a DMA instruction of the block
// moves 32 token rows)
constexpr int a_bytes(int nsub) { return nsub > 2 ? 64 * 128 : 32 * 128; }
constexpr int stage_bytes(int nsub) { return a_bytes(nsub) + B_STAGE + BN * 4 + 2 * BM * 4; }
constexpr int STAGES = 3;
constexpr int RING = STAGES * stage_bytes(4);
static_assert(2 * RING <= 160 * 1024, "two blocks per CU");

// A chunk swizzle: 16-byte chunk c (0..7) of token row r sits at c ^ a8swz(r),
// distinct over 8 consecutive rows (128 B, 32 banks) and over the rows of
// equal parity among 16 (256 B, 64 banks)
__device__ __forceinline__ int a8swz(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// D (TM x TM) += A B: 16 x 16 over 64 k, or 32 x 32 over 32 k
template <int TM, typename V>
__device__ __forceinline__ V mfma_i8(u32x4 a, u32x4 b, V c) {
  if constexpr (TM == 16)
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, a),
                                                 __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a),
                                                 __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

// bytes 8 + q of the even (o = 0) or odd elements of a packed 16-byte chunk
__device__ __forceinline__ u32x4 nib_bytes(u32x4 b, int o) {
  u32x4 r;
#pragma unroll
  for (int d = 0; d < 4; ++d) r[d] = ((b[d] >> (4 * o)) & 0x0F0F0F0Fu) ^ 0x08080808u;
  return r;
}

template <int SD, int MODE>
__device__ __forceinline__ void w8_item(const W8GemmArgs &a, const int lb, const int4 t) {
  // dynamic LDS: the ring; MODE 0's epilogue stages its rows there
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int nb = lb % a.n_nblk;
  const int e = t.x, pos0 = t.y, mcnt = t.z;
  const bool shared = e == a.E;
  const int N = MODE == 0 ? (shared ? a.Is : a.I) : a.H;
  const int K = MODE == 0 ? a.H : (shared ? a.Is : a.I);
  const int G = K >> 7;
  if (nb * (MODE == 0 ? COLS : BN) >= N) return;
  const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
  const int tid = tid_opaque();
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;

  // ---- per-lane DMA sources (moe_gemm.hip's, with int8 token rows) ---------
  const W8Rows &src = MODE == 0 ? a.x : (shared ? a.act_s : a.act);
  // MODE 0 routed rows are gathered by token; the others start at pos0
  const bool gather = MODE == 0 && !shared;
  const size_t row0 = gather ? 0 : (size_t)pos0;
  auto arow = [&](int r) {
    const int rr = min(r, mcnt - 1);
    return (uint32_t)(gather ? a.ptok[pos0 + rr] : rr);
  };
  uint32_t aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = i * 32 + wave * 8 + (lane >> 3);
    aoff[i] = arow(r) * (uint32_t)K + (uint32_t)(((lane & 7) ^ a8swz(r)) << 4);
  }
  const uint32_t xoff = arow(lane) * (uint32_t)G * 4u;
  const size_t rowb = (size_t)K / 2;
  uint64_t bbase[NW];
  uint32_t boff[NW];
  const uint8_t *w0 = shared ? a.ws0 : a.w0 + (size_t)e * N * rowb;
  const uint16_t *s0 = shared ? a.ss0 : a.s0 + (size_t)e * N * G;
  const uint8_t *w1 = w0;
  const uint16_t *s1 = s0;
  if (MODE == 0) {  // B-rows [0, COLS) gate, [COLS, 2 COLS) up
    w1 = shared ? a.ws1 : a.w1 + (size_t)e * N * rowb;
    s1 = shared ? a.ss1 : a.s1 + (size_t)e * N * G;
  }
  auto brow_of = [&](int r) { return min(MODE == 0 ? nb * COLS + r % COLS : nb * BN + r, N - 1); };
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int r = (i * NW + wave) * 16 + (lane >> 2);
    bbase[i] = sbase64((i * NW + wave) * 16 < COLS ? w0 : w1);
    boff[i] = (uint32_t)brow_of(r) * (uint32_t)rowb + (uint32_t)(((lane & 3) ^ bswz(r)) << 4);
  }
  // the aligned dword holding the row's scale of the group: rows are a
  // multiple of 128, so it never ends past the tensor
  const uint32_t soff = (uint32_t)(brow_of(wave * 64 + lane) * G) * 2u;
  const uint64_t abase = sbase64(src.q + row0 * K), xsbase = sbase64(src.s + row0 * G),
                 xcbase = sbase64(src.sum + row0 * G),
                 sbase = sbase64(wave * 64 < COLS ? s0 : s1);
  // DMA of group g into the ring stage at `base` (NW + 1 + A instructions + 2
  // per wave; every wave copies the same 64 row scales and sums)
  auto issue = [&](auto nsub_c, int g, uint32_t base) {
    constexpr int NSUB = decltype(nsub_c)::value;
    constexpr uint32_t BO = a_bytes(NSUB), SO = BO + B_STAGE, XO = SO + BN * 4, CO = XO + BM * 4;
#pragma unroll
    for (int i = 0; i < NW; ++i)
      dma16s(boff[i], bbase[i] + (uint32_t)g * 64u, base + BO + (uint32_t)((i * NW + wave) * 1024));
    dma4s((soff + 2u * (uint32_t)g) & ~3u, sbase, base + SO + (uint32_t)(wave * 256));
#pragma unroll
    for (int i = 0; i < (NSUB > 2 ? 2 : 1); ++i)
      dma16s(aoff[i], abase + (uint32_t)g * 128u, base + (uint32_t)((i * NW + wave) * 1024));
    dma4s(xoff, xsbase + (uint32_t)g * 4u, base + XO);
    dma4s(xoff, xcbase + (uint32_t)g * 4u, base + CO);
  };

  auto run = [&](auto tm_c, auto ms_c) {
    constexpr int TM = decltype(tm_c)::value, MS = decltype(ms_c)::value;
    constexpr int NS = 64 / TM, NSUB = MS * TM / 16, NP = TM / 16, NSL = 2 * NP;
    constexpr int NQ = TM == 16 ? 1 : 4;  // row quads a lane holds of a tile
    using iacc = typename std::conditional<TM == 16, i32x4, i32x16>::type;
    using facc = typename std::conditional<TM == 16, f32x4, f32x16>::type;
    using nsub_t = std::integral_constant<int, NSUB>;
    constexpr int STAGE = stage_bytes(NSUB);
    constexpr uint32_t BO = a_bytes(NSUB), SO = BO + B_STAGE, XO = SO + BN * 4, CO = XO + BM * 4;
    constexpr int PER = NW + 1 + (NSUB > 2 ? 2 : 1) + 2;  // DMA instructions per wave and group
    issue(nsub_t(), 0, lds0);
    if (G > 1) issue(nsub_t(), 1, lds0 + STAGE);
    // lane (Q, rl): row rl of a tile; block Q (TM = 16) or blocks 2 p + Q
    const int rl = lane & (TM - 1), Q = lane / TM;
    auto blk = [&](int p) { return TM == 16 ? Q : 2 * p + Q; };
    auto brow = [](int ns) {
      return MODE == 0 ? (ns < NS / 2 ? ns * TM : COLS + (ns - NS / 2) * TM) : ns * TM;
    };
    const int brow0 = (MODE == 0 ? wave * 32 : wave * 64) + rl;
    const uint32_t soffl = (uint32_t)(brow0 * 4);
    uint32_t boffl[NP], aoffl[NSL];
#pragma unroll
    for (int p = 0; p < NP; ++p) boffl[p] = (uint32_t)(brow0 * 64 + ((blk(p) ^ bswz(rl)) << 4));
#pragma unroll
    for (int s = 0; s < NSL; ++s)
      aoffl[s] = (uint32_t)(rl * 128 + (((2 * blk(s >> 1) + (s & 1)) ^ a8swz(rl)) << 4));
    uint32_t ssh = ((uint32_t)(brow0 * G) & 1u) * 16u;
    facc tot[MS][NS];
#pragma unroll
    for (int ms = 0; ms < MS; ++ms)
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int i = 0; i < 4 * NQ; ++i) tot[ms][ns][i] = 0.f;
    int si = 0, sf = STAGES - 1;  // stages of group g and of the group to fill
    for (int g = 0; g < G; ++g) {
      // group g has landed (g+1, issued after it, may be in flight); past the
      // barrier every wave is done with stage g-1, which group g+2 fills
      if (g + 1 < G)
        wait_vm<PER>();
      else
        wait_vm<0>();
      block_barrier();
      if (g + 2 < G) issue(nsub_t(), g + 2, lds0 + (uint32_t)(sf * STAGE));
      const uint8_t *st = lds + si * STAGE;
      u32x4 bx[NS][NP];
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int p = 0; p < NP; ++p)
          bx[ns][p] = *(const u32x4 *)(st + boffl[p] + BO + brow(ns) * 64);
      u32x4 af[MS][NSL];
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int s = 0; s < NSL; ++s)
          af[ms][s] = *(const u32x4 *)(st + aoffl[s] + ms * TM * 128);
      iacc c0[MS];  // -8 sum of the row's codes
#pragma unroll
      for (int ms = 0; ms < MS; ++ms)
#pragma unroll
        for (int i = 0; i < NQ; ++i) {
          const i32x4 v = *(const i32x4 *)(st + CO + (ms * TM + 8 * i + 4 * Q) * 4);
#pragma unroll
          for (int r = 0; r < 4; ++r) c0[ms][4 * i + r] = v[r];
        }
      float sg[NS];
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
        sg[ns] = scale_to_f32<SD>((uint16_t)(*(const uint32_t *)(st + soffl + SO + brow(ns) * 4) >> ssh));
      ssh ^= 16u;
      iacc acc[MS][NS];
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int s = 0; s < NSL; ++s) {
          const u32x4 b = nib_bytes(bx[ns][s >> 1], s & 1);
#pragma unroll
          for (int ms = 0; ms < MS; ++ms)
            acc[ms][ns] = mfma_i8<TM>(af[ms][s], b, s == 0 ? c0[ms] : acc[ms][ns]);
        }
      // the terms, rounded as the reference rounds them
#pragma unroll
      for (int ns = 0; ns < NS; ++ns)
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
          for (int i = 0; i < NQ; ++i) {
            const f32x4 sx = *(const f32x4 *)(st + XO + (ms * TM + 8 * i + 4 * Q) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
#pragma clang fp contract(off)
              const float term = (float)acc[ms][ns][4 * i + r] * sg[ns] * sx[r];
              tot[ms][ns][4 * i + r] = tot[ms][ns][4 * i + r] + term;
            }
          }
      si = si + 1 == STAGES ? 0 : si + 1;
      sf = sf + 1 == STAGES ? 0 : sf + 1;
    }

    // ---- epilogue: a lane holds rows ms * TM + 8 i + 4 Q + r, column
    // ns * TM + rl ------------------------------------------------------------
    if constexpr (MODE == 1) {
      float *o = a.o + (size_t)((shared ? a.T * a.k : 0) + pos0) * a.H;
#pragma unroll
      for (int ns = 0; ns < NS; ++ns) {
        const int col = nb * BN + wave * 64 + ns * TM + rl;
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
          for (int i = 0; i < 4 * NQ; ++i) {
            const int row = ms * TM + 8 * (i >> 2) + 4 * Q + (i & 3);
            if (row < mcnt && col < N) o[(size_t)row * a.H + col] = tot[ms][ns][i];
          }
      }
    } else {
      block_barrier();  // every wave's last read of the ring precedes the staging
      constexpr int OST = COLS + 4;  // staged row stride, floats
      static_assert(BM * OST * 4 <= RING, "staging exceeds the ring");
      float *stg = (float *)lds;
#pragma unroll
      for (int ns = 0; ns < NS / 2; ++ns)
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
          for (int i = 0; i < 4 * NQ; ++i) {
            const float gv = tot[ms][ns][i], uv = tot[ms][ns + NS / 2][i];
            stg[(ms * TM + 8 * (i >> 2) + 4 * Q + (i & 3)) * OST + wave * 32 + ns * TM + rl] =
                gv / (1.0f + expf(-gv)) * uv;
          }
      __syncthreads();
      // a half wave per row: the arithmetic of k_act_quant_i8 (max is exact,
      // so its order does not matter); lane l32 holds columns 4 l32 + [0, 4)
      const W8Rows &dst = shared ? a.act_s : a.act;
      const int l32 = tid & 31;
      for (int row = tid >> 5; row < mcnt; row += THREADS / 32) {
        const float4 v4 = *(const float4 *)(stg + row * OST + 4 * l32);
        const float v[4] = {v4.x, v4.y, v4.z, v4.w};
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float av = fabsf(v[i]);
          m = av > m ? av : m;
        }
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1)
          m = __uint_as_float(max(__float_as_uint(m), (uint32_t)__shfl_xor((int)__float_as_uint(m), o, 64)));
        float sc = m / 127.0f;
        sc = sc == 0.0f ? 1.0f : sc;
        int qi[4], qs = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float r = v[i] / sc;
          int q = (int)(r >= 0.0f ? r + 0.5f : r - 0.5f);
          qi[i] = q < -127 ? -127 : (q > 127 ? 127 : q);
          qs += qi[i];
        }
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) qs += __shfl_xor(qs, o, 64);
        // W8 order of the 32-element block l32 / 8: evens, then odds
        int8_t *qd = dst.q + (size_t)(pos0 + row) * N + nb * COLS + (l32 >> 3) * 32 + 2 * (l32 & 7);
        *(uint16_t *)qd = (uint16_t)((uint8_t)qi[0] | ((uint32_t)(uint8_t)qi[2] << 8));
        *(uint16_t *)(qd + 16) = (uint16_t)((uint8_t)qi[1] | ((uint32_t)(uint8_t)qi[3] << 8));
        if (l32 == 0) {
          dst.s[(size_t)(pos0 + row) * (N / COLS) + nb] = sc;
          dst.sum[(size_t)(pos0 + row) * (N / COLS) + nb] = -8 * qs;
        }
      }
    }
  };
  using std::integral_constant;
  if (mcnt > 32)
    run(integral_constant<int, 32>(), integral_constant<int, 2>());
  else if (mcnt > 16)
    run(integral_constant<int, 32>(), integral_constant<int, 1>());
  else
    run(integral_constant<int, 16>(), integral_constant<int, 1>());
}

template <int SD, int MODE>
__global__ __launch_bounds__(THREADS, 2) void k_w4a8_gemm(W8GemmArgs a) {
  const int n_items = *a.n_tiles * a.n_nblk;
  if ((int)blockIdx.x >= n_items) return;
  const int lb = xcd_remap(blockIdx.x, n_items);
  w8_item<SD, MODE>(a, lb, a.tiles[lb / a.n_nblk]);
}

}  // namespace

hipError_t launch_w4a8_gemm(int mode, int scale_dtype, W8GemmArgs a, int max_tiles,
                            hipStream_t s) {
  if (max_tiles <= 0) return hipSuccess;
  const int Nmax = mode == 0 ? (a.I > a.Is ? a.I : a.Is) : a.H;
  a.n_nblk = mode == 0 ? (Nmax + COLS - 1) / COLS : (Nmax + BN - 1) / BN;
  const long grid = (long)max_tiles * a.n_nblk;
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  void (*kern)(W8GemmArgs);
  if (mode == 0)
    kern = scale_dtype == AINFER_SCALE_FP16 ? k_w4a8_gemm<AINFER_SCALE_FP16, 0>
                                            : k_w4a8_gemm<AINFER_SCALE_BF16, 0>;
  else
    kern = scale_dtype == AINFER_SCALE_FP16 ? k_w4a8_gemm<AINFER_SCALE_FP16, 1>
                                            : k_w4a8_gemm<AINFER_SCALE_BF16, 1>;
  kern<<<(unsigned)grid, THREADS, RING, s>>>(a);
  return hipGetLastError();
}
