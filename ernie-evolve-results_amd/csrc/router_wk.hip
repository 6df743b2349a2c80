// Stage 1 for batches too small to fill the chip with whole-K tiles: the
// router GEMM with K split over the waves of a block.
//
// The fused kernel (route_fused.hip) gives a block 128 (64) tokens and all E
// experts, so a batch of T tokens runs on T / 128 of the 256 CUs and each of
// those streams the whole weight: at E = 256, H = 7168 the route took 91 us
// for any T from 1 to 4096.  Such a call is bound by what one CU can load
// (a DMA stream of 128-byte rows moves about 90 GB/s per CU here), so the
// tile is chosen for the fewest operand bytes per CU: BM tokens x BN experts
// with BM + BN as small as leaves at most one block per CU.  A block's four
// waves split K, each streaming its quarter through its own LDS ring by
// the gfx950 buffer_load ... lds DMA (8 rows of 128 bytes per instruction,
// XOR-swizzled 16-byte chunks); only the wave that fills a ring reads it, so
// the K loop has no barrier, and the ring is as deep as the LDS allows.
// The partial tiles meet in LDS and are added in K order.  A wave adds its quarter up in
// two chains, so that the sum is no further from 64 bits than with 8 K partitions in
// router_gemm.hip (relative error, E = 64, H = 8192, T = 128: one chain a wave 2.73e-7,
// two 1.89e-7, 8 partitions 1.92e-7; E = 64, H = 4096 1.92e-7, 1.36e-7, 1.40e-7).
// The blocks of one row tile are 8 apart in the grid: one XCD, whose L2 serves
// the row tile's x to all of them.
//
// Measured (MI355X; route = this GEMM + the scoring kernel, graph replay, us,
// the path it replaced first): E = 256, H = 7168: T = 16 88 / 11.2, 128 91 / 11.6,
// 1024 92 / 18.9, 4904 92 / 35.8, 8000 92 / 53.9, 16000 93 / 83.8; E = 128,
// H = 2048: T = 128 17.8 / 8.5, 4904 18.3 / 14.9; E = 64, H = 4096: T = 128
// 11.0 / 8.0.  GEMM alone at E = 256, H = 7168, T = 16: fragments loaded
// straight into registers (16 rows x 64 bytes per load instruction, so every
// four lanes touch four lines) 15.4 us, this ring 6.5; 8 waves x 2 stages 7.0,
// 4 waves x 3 stages 7.7.
//
// An fp32 weight (WF32) comes into the ring as fp32 and each lane splits its 8
// k into hi = bf16(w) and lo = bf16(w - hi) (the reference's wsplit_kernel,
// K:1786-1824); a logit is (sum of hi) + (sum of lo), each in K order.  That
// saves the split's launch, its [2E, H] copy and the partial sums: E = 64,
// H = 8192 T = 128 19.4 / 12.6, T = 3000 26.3 / 22.0; E = 256, H = 1024
// T = 128 16.8 / 8.9.
#include "moe_common.h"
#include <type_traits>

namespace moe {

namespace wk {
// word 3 of a gfx9 raw buffer resource (32-bit data format, no swizzle)
constexpr int kRsrcW3 = 0x00020000;
// fp32 chains that a logit's K is added up in, as many as K partitions in router_gemm.hip
constexpr int kChains = 8;
// an offset past every resource here: such a load writes zeros and moves nothing
constexpr int kPast = 0x7f000000;
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }
// 16 bytes per lane into LDS (1 KB per wave instruction)
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, char* l, int voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)l, 16, voff,
                                           0, 0, 0);
}
}  // namespace wk

// BM tokens x BN experts per block, NW waves with NS-stage rings; E % BN == 0.
// mtiles = ceil(T / BM); the grid rounds the row tiles up to a multiple of 8.
template <int BM, int BN, int NW, int NS, bool WF32>
__global__ __launch_bounds__(64 * NW) void router_wk_kernel(const __bf16* __restrict__ x,
                                                            const void* __restrict__ w, int T,
                                                            int H, int E, int mtiles,
                                                            float* __restrict__ out) {
  using namespace wk;
  constexpr int FM = BM / 16, FN = BN / 16;
  constexpr int WB = WF32 ? 4 : 2;       // bytes per weight element
  constexpr int NP = WF32 ? 2 : 1;       // hi and lo products
  constexpr int LD = BN + 4;             // row stride of a partial tile in LDS (floats)
  constexpr int WROWB = 64 * WB;         // weight bytes per row and stage
  constexpr int XB = BM * 128, STAGE_B = XB + BN * WROWB;
  constexpr int NQX = XB / 1024, NQ = STAGE_B / 1024;
  constexpr int RING_B = NW * NS * STAGE_B, PART_B = NW * BM * LD * 4;
  __shared__ __attribute__((aligned(1024))) char lds[RING_B > PART_B ? RING_B : PART_B];
  static_assert(sizeof(lds) <= 160 * 1024, "LDS");
  static_assert(kChains == NW || kChains == 2 * NW, "chains");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nt_n = E / BN;
  const int j8 = (int)blockIdx.x >> 3;
  const int nt = j8 % nt_n;
  const int mt = (j8 / nt_n) * 8 + ((int)blockIdx.x & 7);
  if (mt >= mtiles) return;
  const long long m0 = (long long)mt * BM;
  const int rows = T - m0 < BM ? (int)(T - m0) : BM;
  const int n0 = nt * BN;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(x + m0 * H), (short)0, rows * H * 2, kRsrcW3);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const char*)w + (long long)n0 * H * WB), (short)0, BN * H * WB, kRsrcW3);

  // this wave's K steps of 64: [u0, u1)
  const int U = H / 64;
  const int u0 = wave * U / NW, u1 = (wave + 1) * U / NW, n = u1 - u0;
  char* const ring = lds + wave * NS * STAGE_B;
  // Per-lane source of each DMA instruction of a stage: 16-byte chunk p of row r
  // goes to physical chunk p ^ swz(r), an fp32 weight row's 32-byte chunk c to
  // c ^ (r & 7).  Rows past T and steps past u1 lie past the resource (zeros),
  // so every step issues the same loads and the waits below are constants.
  int voff[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    if (q < NQX) {
      const int r = q * 8 + lane / 8;
      voff[q] = r * H * 2 + u0 * 128 + ((lane % 8) ^ swz(r)) * 16;
    } else if (!WF32) {
      const int r = (q - NQX) * 8 + lane / 8;
      voff[q] = r * H * 2 + u0 * 128 + ((lane % 8) ^ swz(r)) * 16;
    } else {
      const int r = (q - NQX) * 4 + lane / 16;  // 16 lanes of 16 B: 8 chunks of 32 B
      voff[q] = r * H * 4 + u0 * 256 + ((((lane % 16) >> 1) ^ (r & 7)) * 32) + (lane & 1) * 16;
    }
  }
  auto issue = [&](int u, int st) {
    const int kx = u < n ? u * 128 : kPast;
    const int kw = u < n ? u * WROWB : kPast;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      char* dst = ring + st * STAGE_B + q * 1024;
      if (q < NQX) dma16(rx, dst, voff[q] + kx);
      else dma16(rw, dst, voff[q] + kw);
    }
  };

  f32x4 acc[NP][FM][FN], tot[NP][FM][FN];  // tot: the chain before this one
#pragma unroll
  for (int st = 0; st < NS - 1; ++st) issue(st, st);
  const int fr = lane & 15, fc = lane >> 4;
  int slot = 0;
  // FIRST: of a chain, from a constant zero instead of cleared accumulators (route at
  // E = 128, H = 512, T = 8000: one chain a wave 12.7 us, two 13.2, two from the constant 12.6)
  auto step = [&]<bool FIRST>(std::bool_constant<FIRST>, int u) __attribute__((always_inline)) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    // stage u landed once at most the NS-2 later stages are outstanding; the
    // slot refilled now held step u-1, whose reads its MFMAs have consumed
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * NQ) : "memory");
    const int nslot = slot == 0 ? NS - 1 : slot - 1;
    issue(u + NS - 1, nslot);
    const char* sb = ring + slot * STAGE_B;
    slot = slot == NS - 1 ? 0 : slot + 1;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = kk * 4 + fc;
      bf16x8 av[FM];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int r = i * 16 + fr;
        av[i] = *reinterpret_cast<const bf16x8*>(sb + r * 128 + ((c ^ swz(r)) * 16));
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int r = j * 16 + fr;
        bf16x8 bh, bl;
        if constexpr (WF32) {
          const f32x4* pv = reinterpret_cast<const f32x4*>(sb + XB + r * WROWB + (c ^ (r & 7)) * 32);
          const f32x4 v0 = pv[0], v1 = pv[1];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = e < 4 ? v0[e & 3] : v1[e & 3];
            bh[e] = (__bf16)v;
            bl[e] = (__bf16)(v - (float)bh[e]);
          }
        } else {
          bh = *reinterpret_cast<const bf16x8*>(sb + XB + r * 128 + ((c ^ swz(r)) * 16));
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const bool z = FIRST && kk == 0;
          acc[0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[i], bh, z ? zero : acc[0][i][j],
                                                                 0, 0, 0);
          if constexpr (WF32)
            acc[1][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                av[i], bl, z ? zero : acc[1][i][j], 0, 0, 0);
        }
      }
    }
  };
  int u = 0;
  auto chain = [&](int end) __attribute__((always_inline)) {
    if (FM * FN >= 6 && u < end) {  // a third copy of the step costs the small tiles more
      step(std::true_type{}, u++);
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[p][i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    for (; u < end; ++u) step(std::false_type{}, u);
  };
  // An fp32 chain's error grows with its length: a wave with a quarter of K adds it up in
  // two (kChains).
  constexpr bool TWO = kChains > NW;
  if constexpr (TWO) {
    chain(n / 2);
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) tot[p][i][j] = acc[p][i][j];
  }
  chain(n);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past u1 have landed
  __syncthreads();  // every ring is read: the partial tiles may overwrite them
  float* const part = reinterpret_cast<float*>(lds);

  constexpr int NT = 64 * NW, NV = BM * BN / 4;  // 16-byte pieces of the tile
  constexpr int PER = (NV + NT - 1) / NT;
  f32x4 sum[PER];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    if (p > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          part[(wave * BM + i * 16 + fc * 4 + r) * LD + j * 16 + fr] =
              TWO ? tot[p][i][j][r] + acc[p][i][j][r] : acc[p][i][j][r];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int idx = threadIdx.x + q * NT;
      if (NV % NT != 0 && idx >= NV) continue;
      const int row = idx / (BN / 4), c4 = idx % (BN / 4);
      const float* s = part + row * LD + c4 * 4;
      f32x4 v = *reinterpret_cast<const f32x4*>(s);
#pragma unroll
      for (int g = 1; g < NW; ++g) v += *reinterpret_cast<const f32x4*>(s + g * BM * LD);
      sum[q] = p == 0 ? v : sum[q] + v;
    }
  }
  const bool vec = ((uintptr_t)out & 15u) == 0;  // moe_router_gemm takes 4-byte aligned logits
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int idx = threadIdx.x + q * NT;
    if (NV % NT != 0 && idx >= NV) continue;
    const int row = idx / (BN / 4), c4 = idx % (BN / 4);
    if (row >= rows) continue;
    float* o = out + (m0 + row) * E + n0 + c4 * 4;
    if (vec) {
      *reinterpret_cast<f32x4*>(o) = sum[q];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = sum[q][e];
    }
  }
}

template <int BM, int BN, int NW, int NS, bool WF32>
static hipError_t launch_wk(const __bf16* x, const void* w, int T, int H, int E, float* out,
                            hipStream_t s) {
  const int mt = (T + BM - 1) / BM;
  const dim3 grid((unsigned)((mt + 7) / 8 * 8 * (E / BN)));
  hipLaunchKernelGGL((router_wk_kernel<BM, BN, NW, NS, WF32>), grid, dim3(64 * NW), 0, s, x, w, T,
                     H, E, mt, out);
  return hipGetLastError();
}

namespace wk {
struct Tile {
  int bm, bn;
  hipError_t (*launch)(const __bf16*, const void*, int, int, int, float*, hipStream_t);
};
// The last two are the shared-ring kernel of router_gemm.hip (K in order, all of a
// block's waves on one tile), for batches of several rounds.
const Tile kTiles[] = {
    {16, 16, launch_wk<16, 16, 4, 4, false>}, {32, 16, launch_wk<32, 16, 4, 3, false>},
    {48, 16, launch_wk<48, 16, 4, 3, false>}, {32, 32, launch_wk<32, 32, 4, 3, false>},
    {48, 32, launch_wk<48, 32, 4, 3, false>}, {64, 32, launch_wk<64, 32, 4, 3, false>},
    {48, 64, launch_wk<48, 64, 4, 2, false>}, {64, 64, launch_wk<64, 64, 4, 2, false>},
    {80, 64, launch_wk<80, 64, 4, 2, false>}, {128, 64, launch_router_gemm_128x64},
    {128, 128, launch_router_gemm_128x128}};
const Tile kTilesF32[] = {{16, 16, launch_wk<16, 16, 8, 2, true>},
                          {32, 16, launch_wk<32, 16, 8, 2, true>},
                          {48, 16, launch_wk<48, 16, 8, 2, true>}};
constexpr int kCUs = 256;

// The tile of the least operand bytes per CU: rounds of blocks x operand rows
// per block (an fp32 weight row counts twice).  Measured for the GEMM alone over
// T = 1 .. 16384, E = 32 .. 256, H = 512 .. 8192: at 349 of 360 points the fastest tile
// or one within 5% of it, at worst 22% behind (E = 256, H = 8192, T = 10000: 128 x 128
// 69 us, 80 x 64 57).
static const Tile* pick(int T, int E, bool wf32) {
  const Tile* t = wf32 ? kTilesF32 : kTiles;
  const int n = (int)(wf32 ? sizeof(kTilesF32) : sizeof(kTiles)) / (int)sizeof(Tile);
  const Tile* best = nullptr;
  long long least = 0;
  for (int i = 0; i < n; ++i) {
    if (E % t[i].bn) continue;
    const long long blocks = (long long)((T + t[i].bm - 1) / t[i].bm) * (E / t[i].bn);
    const long long c = (blocks + kCUs - 1) / kCUs * (t[i].bm + (wf32 ? 2 : 1) * t[i].bn);
    if (!best || c < least) {
      best = t + i;
      least = c;
    }
  }
  return best;
}
}  // namespace wk

// Where it takes over (route times in us, the other path / this one):
//   E = 256, H = 7168 and E = 128, H = 2048 (the fused kernel's shapes): while
//     the fused kernel's tiles fill at most half (5/8) of the CUs: T = 16000 94 / 89,
//     18000 101 / 143; T = 10000 21.6 / 20.3, 12000 22.3 / 23.1.
//   elsewhere, against K split over blocks with the partial sums added by the
//     scoring kernel.  That path moves fewer operand bytes (larger tiles) but
//     writes and reads the partials; either is ahead as its tiles fill whole rounds:
//     E = 256, H = 4096 T = 4500 33.3 / 27.1, 6000 32.7 / 36.7, 7000 51.8 / 37.4,
//     10100 43.1 / 49.2, 12200 58.5 / 48.9; E = 64, H = 8192 T = 900 13.8 / 11.8,
//     2300 17.6 / 17.5.  The lines lie where the two met when the partitions were fewer
//     and the chains longer; past them this kernel is still as fast or faster up to
//     16000 tokens at H <= 4096 (E = 256, H = 4096 T = 13000 67.8 / 52.3, H = 1024
//     T = 16000 47.2 / 28.8; E = 64, H = 4096 T = 14000 27.7 / 26.8), and at H = 8192 up
//     to 3500 (E = 256 38.7 / 32.6; E = 64 19.7 / 18.6), not at E = 256,
//     H = 4096 T = 32768 (106 / 122).
//   E = 128 above 8192 tokens, where that path has one tile of 64 tokens and all
//     experts per 64 tokens and no K split: the 80 x 64 tiles up to 10240 (H = 4096
//     T = 9000 31.5 / 25.9).  From there the tiles are 128 x 64, above 16384 128 x 128.
//     They have the same operand bytes per CU (up to 16384 tokens) and lose or tie while
//     x stays in the 256 MB memory-side cache, except where H is short (H = 1024
//     T = 12200 20.5 / 17.4, 25000 25.5 / 25.1; H = 4096 T = 12200 32.9 / 34.4, 22000
//     49 / 47; H = 8192 T = 11000 49 / 56), and win beyond (H = 8192 T = 15000 76 / 58,
//     18000 124 / 98; H = 7168 T = 32768 138 / 115) unless the last of the 128-token
//     rounds is nearly empty (H = 8192 T = 45000 215 / 225).
//   fp32 weights, whose rows count twice: E = 64, H = 8192 T = 3070 25.7 / 21.7, 4000
//     28.2 / 30.7; E = 256, H = 4096 T = 700 27.0 / 16.3, 890 27.8 / 21.7; E = 32,
//     H = 4096 T = 6000 19.4 / 15.4, 7100 20.0 / 20.3, 8192 19.7 / 20.6.  At E >= 128 and
//     at H <= 1024 this kernel is ahead past the line too (E = 256, H = 4096 T = 1200
//     30.2 / 24.8; E = 128, H = 1024 T = 2600 24.9 / 14.0; E = 64, H = 512 T = 6000
//     17.3 / 11.8).
bool router_wk_use(int T, int H, int E, bool wf32) {
  if (T < 1 || E < 32 || H % 64 != 0 || H > 32768) return false;
  if (wf32) return (long long)T * E <= (H <= 4096 ? 229376 : 196608);
  if (E == 256 && H == 7168) return T <= 16384;
  if (E == 128 && H == 2048) return T <= 10240;
  if (E == 128 && T > 8192) {
    if (T <= 10240 || (H <= 2048 && T <= 16384)) return true;
    if ((long long)T * H <= 110ll << 20) return false;
    const int r = (T + 16383) / 16384;  // rounds of 64-token tiles, half as many of 128
    return r == 1 || 5 * ((r + 1) / 2) < 3 * r;
  }
  return H <= 4096 ? T <= 12288 : (long long)T * H <= 2560ll * 8192;
}

hipError_t launch_router_wk(const __bf16* x, const void* w, bool wf32, int T, int H, int E,
                            float* out, hipStream_t s) {
  const wk::Tile* t = wk::pick(T, E, wf32);
  return t ? t->launch(x, w, T, H, E, out, s) : hipErrorInvalidValue;
}

}  // namespace moe
