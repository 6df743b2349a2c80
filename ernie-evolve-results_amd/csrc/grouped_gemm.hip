// Expert grouped GEMM over the expert-contiguous rows the permute produces.
//
// Replaces the reference's CUTLASS grouped GEMMs (moe_gemm.h:66-95,
// moe_gemm.cu:616-650): group g owns rows [offs[g-1], offs[g]) of a
// (offs = inclusive group ends, offs[-1] = 0 -- exactly `offsets + 1` of
// moe_permute) and
//   plain : out[r, :] = a[r, :] . w[g]^T                     (grouped_mm)
//   swiglu: h[r, :]   = silu(a[r, :] . wg[g]^T) * (a[r, :] . wu[g]^T)
//           (grouped_mm_pair followed by silu*mul, fused into the epilogue)
// with a [M, K] bf16, w [G, N, K] bf16 (both K-contiguous), fp32 accumulate.
//
// Plan (the reference's plan_kernel builds per-group pointers for CUTLASS on
// the device; here it is one scan): tile_start[g] = sum over g' < g of
// ceil(m_g' / BM), on the device, so nothing waits for the host.  Up to 256
// groups every block scans the group ends itself (no plan launch); beyond,
// gg_plan_kernel writes tile_start into the workspace first.  The grid is
// sized by the bound sum ceil(m_g / BM) <= ceil(M / BM) + G; blocks past the
// last tile return at once.
//
// Tiles: 256 rows x 256 weight rows, 128-byte K steps (64 bf16 or 128 int8
// elements), staged in LDS by the gfx950 global_load_lds DMA in an XOR-swizzled
// 16-byte chunk layout, v_mfma_f32_16x16x32_bf16 or v_mfma_i32_16x16x64_i8.
// Eight waves in two groups of four (one wave of each per SIMD); a wave owns 64
// rows of each 128-row half of the tile and 32 weight rows of each half.
//
// K loop.  A K step is two half steps (the two row halves); each wave does, per
// half step, a load part (12 fragment reads, 4 DMA instructions) and 32 MFMAs,
// with a barrier after each, and the second group runs one barrier behind the
// first: while one group's MFMAs hold the matrix pipes the other reads
// fragments and issues loads.  The operand tile is recycled in quarters: the
// rows read in one half step are refilled in the next (every wave has waited for
// its reads before the barrier in between), for the step after next, so a load
// has three half steps to land and 96 of the 128 KB are in flight or in use.
// One 256 x 256 tile per CU.  Measured, dense 16384 x 16384 x 8192, counters and times of
// the same launches (share of cycles the MFMA units are busy x clock = rate): bf16 86% x
// 1.56 GHz = 1407 TFLOP/s, SwiGLU 85% x 1.74 = 1545, int8 78% x 1.81 = 2978 TOP/s; the
// library's bf16 GEMM 89% x 1.59 = 1482.  So 3 points of busy time are the schedule's, and
// the clock falls as the units are busier; 65536 x 8192 x 3584, where the start and end of
// a tile weigh more: bf16 79% x 1.77 = 1471, int8 65% x 1.92 = 2631.  The previous loop
// (both waves of a SIMD in step, the whole stage refilled at once) had bf16 1292, SwiGLU
// 1337, int8 2623 and, 65536 x 8192 x 3584, 1310 and 2268.
// The routed experts (64 experts, H = 8192, Ni = 3584, top-8, us): gate+up T = 16
// 1229 / 1122, 1024 1794 / 1340, 2048 2398 / 2070.  Tried and slower: four half steps
// of 16 MFMAs (5% instead of 13% gained), s_setprio around the MFMAs (-1%), the DMA issued
// between the MFMAs (-8%), the closing barrier 2 .. 12 MFMAs early (-8 .. -12%),
// 32x32x16 MFMAs (-13%).
//
// Tiles of at most 128 rows, where groups are small on average (bf16 and int8), are
// bound by their weight loads, and with few K steps by the start and end of a block: a
// CU holds one, so nothing else overlaps them.  All waves step together through a ring of
// three stages of up to 48 KB, one barrier a step; only the 16-row blocks that exist are
// computed and stored, from registers; a block can take two column tiles in a row
// (grouped_runs.h); and its tile is found by DPP scans.  Measured (us; experts of N x K
// weights, 128 x 512 tiles with a two-stage loop / 256-row tiles with the epilogue of 256
// rows / this): int8 128 experts 2048 x 512, 4 rows each 38 / 55 / 28, 40 rows
// 40 / 59 / 34; 64 experts SwiGLU 2048 x 1024, 16 rows 60 / 82 / 45; bf16 128 experts
// 1024 x 512, 16 rows 29 / 34 / 26; 64 experts SwiGLU 1024 x 1024, 4 rows 48 / 52 / 43;
// 8 experts SwiGLU 2048 x 4096, 16 rows 95 / 49 / 45.  Where the 128 x 512 tiles fill
// whole rounds of CUs and the weights' rows are a power of two apart they stay 3 .. 6%
// ahead: bf16 64 experts 4096 x 2048, 16 rows 188 / 206 / 196; SwiGLU 2048 x 4096, 40 rows
// 363 / 382 / 378; 128 experts 1024 x 512, 100 rows 33 / 40 / 34.4 (at worst 9%: 64 experts
// 4096 x 2048, 100 rows on average, 210 / - / 230).  Tried: four stages of
// 40 KB at up to 64 rows (no gain), two steps loaded at a time (-4%), other orders of the
// tiles over the XCDs (-2 .. -30%), row tiles of equal height instead of a last one with
// the rest (no gain: 2041 / 2018 .. 2027 at T = 2048).
//
// fp8 A: the DMA brings each wave's own 16 rows of e4m3fn bytes, and half a K step
// before they are read the wave writes them once as bf16(q * s) into the A tile
// (one tile is enough: its halves are refilled as above).  1708 / 1533 us at
// T = 1024, 5004 / 4341 at T = 4096 against a dequantisation pass with its own
// barrier in every step.
//
// Block ids are remapped so that each XCD runs a contiguous range of logical
// tiles, and inside a group the tiles go in 4 x 8 (row x column) super-tiles:
// the blocks running together on one XCD share A and weight slices in L2.
//
// swiglu: the first half of the weight rows is the gate, the second the up
// projection of the same 128 output columns, so both accumulators of a column
// sit in one lane and the epilogue forms h without an exchange.
//
// Identity shortcut (the reference's ident_a / ident_m): a group whose row
// count equals ident_m takes its A rows from ident_a (row i of the group =
// row i of ident_a) instead of a.
#include "grouped_runs.h"
#include "moe_common.h"
#include <cmath>
#include <utility>

namespace moe {

constexpr int kGgBM = 256, kGgBN = 256;  // rows and weight rows of a tile

// One workgroup of 1024 threads: inclusive scan of per-group tile counts.
__global__ __launch_bounds__(1024) void gg_plan_kernel(const int* __restrict__ offs, int G, int M,
                                                       int bm, int* __restrict__ tile_start) {
  __shared__ int part[16];
  __shared__ int carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int base = 0; base < G; base += 1024) {
    const int g = base + threadIdx.x;
    int tiles = 0;
    if (g < G) {
      const int lo = g > 0 ? min(max(offs[g - 1], 0), M) : 0;
      const int hi = min(max(offs[g], 0), M);
      tiles = hi > lo ? (hi - lo + bm - 1) / bm : 0;
    }
    // wave inclusive scan
    int v = tiles;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(v, o, 64);
      if (lane >= o) v += u;
    }
    if (lane == 63) part[wave] = v;
    __syncthreads();
    if (threadIdx.x < 16) {
      int p = part[threadIdx.x];
#pragma unroll
      for (int o = 1; o < 16; o <<= 1) {
        const int u = __shfl_up(p, o, 16);
        if ((threadIdx.x & 15) >= o) p += u;
      }
      part[threadIdx.x] = p;  // inclusive over waves
    }
    __syncthreads();
    const int incl = carry + (wave > 0 ? part[wave - 1] : 0) + v;
    if (g < G) tile_start[g + 1] = incl;
    if (g == 0) tile_start[0] = 0;
    __syncthreads();
    if (threadIdx.x == 1023) carry = incl;
    __syncthreads();
  }
  if (G == 0 && threadIdx.x == 0) tile_start[0] = 0;
}

// Up to kScanG groups a block finds its group itself: one wave-wide scan of
// the row-tile counts per 64 groups (a load or two from L2, shuffles and a
// ballot), instead of a separate plan launch and a binary search over its
// output (a chain of dependent loads at the start of every tile).
constexpr int kScanG = 256;

// Rows [lo, hi) of group gi, its ends clamped into [0, M]; empty past G.
__device__ __forceinline__ void group_rows(const int* __restrict__ offs, int gi, int G, int M,
                                           int& lo, int& hi) {
  lo = gi > 0 && gi < G ? min(max(offs[gi - 1], 0), M) : 0;
  hi = gi < G ? max(min(max(offs[gi], 0), M), lo) : lo;
}

// Inclusive wave scan by DPP moves (no LDS latency: it is on the way to a tile's first
// load): in rows of 16 lanes, then the row sums across rows.
__device__ __forceinline__ int wave_incl_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast15, 31
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

// silu(g) * u in fp32
__device__ __forceinline__ float swiglu(float g, float u) { return g / (1.0f + __expf(-g)) * u; }

// 16 e4m3fn bytes -> 16 bf16(q * s): exact fp8 -> fp32 conversion, one fp32
// multiply, and the gfx950 fp32 -> bf16 conversion (round to nearest even).
__device__ __forceinline__ void dequant16(u32x4 raw, float s, bf16x8& lo8, bf16x8& hi8) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[h], false);
    const f32x2 b = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[h], true);
    bf16x8& d = h < 2 ? lo8 : hi8;
    const int o = (h & 1) * 4;
    d[o + 0] = (__bf16)(a[0] * s);
    d[o + 1] = (__bf16)(a[1] * s);
    d[o + 2] = (__bf16)(b[0] * s);
    d[o + 3] = (__bf16)(b[1] * s);
  }
}

// Accumulator type and one MFMA of the K loop: bf16 16x16x32 (fp32 acc) or
// int8 16x16x64 (int32 acc, exact).  Both read 16 bytes per lane per operand.
typedef int i32x4 __attribute__((ext_vector_type(4)));
template <bool I8> struct AccOf { typedef f32x4 type; };
template <> struct AccOf<true> { typedef i32x4 type; };
template <bool I8>
__device__ __forceinline__ typename AccOf<I8>::type mfma_step(bf16x8 a, bf16x8 b,
                                                              typename AccOf<I8>::type c) {
  if constexpr (I8)
    return __builtin_amdgcn_mfma_i32_16x16x64_i8((i32x4)a, (i32x4)b, c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The A operand's row map (bf16 and int8 A) and the row / column scales of the
// int8 operands (unused by the bf16 and fp8 paths).
struct GgExtra {
  const float* a;      // int8: per row of a; fp8: [M, K/128]
  const int* a_idx;    // NULL, or [M]: operand row r is row a_idx[r] of a (data and scale)
  const float* ident;  // [ident_m] per row of ident_a
  const float* w0;     // [G, N] per weight row of w0
  const float* w1;     // [G, N] per weight row of w1 (SwiGLU up)
};

// The tiles of block blockIdx.x: false if it has none.  BM rows per tile.
struct GgTile {
  int g;      // group
  int gs;     // its first row
  int r0;     // first row of the tile
  int rlast;  // last row of the group
  int nt, nt1; // column tiles [nt, nt1)
  int rot;     // which of them comes first
  bool ident; // A rows from ident_a
};
// RUN: gg_run column tiles per block in short groups, by the real tile counts (up to
// kScanG groups, fewer than 2^15 row tiles; beyond, one).
template <int BM, bool RUN>
__device__ __forceinline__ bool gg_tile(const int* __restrict__ offs,
                                        const int* __restrict__ tile_start, int G, int M,
                                        int n_tiles, int KT, int ident_m,
                                        GgTile& out) {
  // XCD-aware order: hardware block b runs on XCD b % 8.  The grid is sized
  // by a bound on the tile count; the real count nreal is known here, and the
  // logical tiles [x*r, (x+1)*r), r = ceil(nreal / 8), all run on XCD x, so
  // every XCD gets an eighth of the real tiles.  (Spreading the bound instead
  // leaves the bound's surplus on the last XCD and up to a round more on the
  // others: the T = 2048 shared down projection, 256 tiles, took 305 us.)
  // Logical tiles are numbered group by group: group g owns
  // [gstart * n_tiles, (gstart + mtg) * n_tiles), gstart = tile_start[g]; with
  // runs a short group has as many as it has runs.
  const unsigned b = blockIdx.x;
  const int lane0 = threadIdx.x & 63;
  const bool runs = RUN && G <= kScanG;
  // row tiles of rows [lo, hi); with runs also, in the upper half, whether the group is
  // short
  auto tiles_of = [&](int lo, int hi) -> int {
    return (hi - lo + BM - 1) / BM + (runs && hi > lo && hi - lo <= 128 ? 1 << 16 : 0);
  };
  // total row tiles: from the plan (G > kScanG) or a scan of the group ends
  int total_rt = 0;
  int lo0 = 0, hi0 = 0, incl0 = 0, tiles0 = 0;  // groups 0..63, lane = group
  if (G <= kScanG) {
    for (int base = 0; base < G; base += 64) {
      int lo, hi;
      group_rows(offs, base + lane0, G, M, lo, hi);
      const int t = tiles_of(lo, hi);
      const int incl = wave_incl_scan(t);
      if (base == 0) {
        lo0 = lo;
        hi0 = hi;
        incl0 = incl;
        tiles0 = t;
      }
      total_rt += __builtin_amdgcn_readlane(incl, 63);
    }
  } else {
    total_rt = __builtin_amdgcn_readfirstlane(tile_start[G]);
  }
  int log = 0;
  unsigned nreal;
  if (runs) {
    log = gg_run(total_rt & 0xffff, total_rt >> 16, n_tiles, KT, (int)gridDim.x);
    nreal = gg_blocks(total_rt & 0xffff, total_rt >> 16, n_tiles, log);
  } else {
    nreal = (unsigned)total_rt * (unsigned)n_tiles;
  }
  const unsigned r = (nreal + 7u) >> 3;
  if ((b >> 3) >= r) return false;
  const unsigned l = (b & 7u) * r + (b >> 3);
  if (l >= nreal) return false;
  // group g of logical tile l: the first group whose inclusive count of logical tiles
  // exceeds l (groups without tiles never qualify); lt, and the counts compared with
  // it, are row tiles without runs
  const int lt = runs ? (int)l : (int)(l / (unsigned)n_tiles);
  auto count = [&](int t) { return runs ? gg_blocks(t & 0xffff, t >> 16, n_tiles, log) : t; };
  int g = 0, gstart = 0, mtg = 0, gs = 0, ge = 0;
  if (G <= 64) {
    const unsigned long long m = __ballot(lane0 < G && count(incl0) > lt);
    g = __ffsll((long long)m) - 1;
    mtg = __builtin_amdgcn_readlane(tiles0, g);
    gstart = __builtin_amdgcn_readlane(incl0, g) - mtg;
    gs = __builtin_amdgcn_readlane(lo0, g);
    ge = __builtin_amdgcn_readlane(hi0, g);
  } else if (G <= kScanG) {
    int carry = 0;
    for (int base = 0; base < G; base += 64) {
      int lo, hi;
      group_rows(offs, base + lane0, G, M, lo, hi);
      const int t = tiles_of(lo, hi);
      const int incl = wave_incl_scan(t) + carry;
      const unsigned long long m = __ballot(base + lane0 < G && count(incl) > lt);
      if (m) {
        const int L = __ffsll((long long)m) - 1;
        g = base + L;
        mtg = __builtin_amdgcn_readlane(t, L);
        gstart = __builtin_amdgcn_readlane(incl, L) - mtg;
        gs = __builtin_amdgcn_readlane(lo, L);
        ge = __builtin_amdgcn_readlane(hi, L);
        break;
      }
      carry = __builtin_amdgcn_readlane(incl, 63);
    }
  } else {
    // the last g with tile_start[g] <= lt
    int lo = 0, hi = G - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (tile_start[mid] <= lt) lo = mid; else hi = mid - 1;
    }
    g = __builtin_amdgcn_readfirstlane(lo);
    gstart = __builtin_amdgcn_readfirstlane(tile_start[g]);
    mtg = __builtin_amdgcn_readfirstlane(tile_start[g + 1]) - gstart;
    group_rows(offs, g, G, M, gs, ge);
  }
  int li = (int)l - (runs ? count(gstart) : gstart * n_tiles);
  const int rlast = ge - 1;  // last row of the group
  const bool ident = ident_m > 0 && ge - gs == ident_m;
  if (runs && mtg >> 16) {  // a run of a short group
    const int nt = li << log, nt1 = min((li + 1) << log, n_tiles);
    // Blocks start at different tiles of their runs: those that run together would
    // else all be at even tiles, whose addresses share memory channels (128 experts of
    // 4096 x 2048: 1022 us for 727).
    out = GgTile{g, gs, gs, rlast, nt, nt1, nt1 - nt == 2 ? li & 1 : 0, ident};
    return true;
  }
  // Inside a group, column blocks of kSuperN n-tiles, row tiles across each
  // block, n fastest: 32 consecutive tiles (one XCD's co-running blocks) are
  // 4 row tiles x 8 weight tiles, so each A slice and each weight slice of a
  // K step is fetched from HBM once and then reused from that XCD's L2.
  constexpr int kSuperN = 8;
  const int nblk = li / (mtg * kSuperN);
  const int rem = li - nblk * mtg * kSuperN;
  const int ncols = min(kSuperN, n_tiles - nblk * kSuperN);
  const int mt_local = rem / ncols;
  const int nt = nblk * kSuperN + rem % ncols;
  out = GgTile{g, gs, gs + mt_local * BM, rlast, nt, nt + 1, 0, ident};
  return true;
}

int grouped_gemm_n_tiles(int N, bool swiglu) {
  const int per = swiglu ? kGgBN / 2 : kGgBN;
  return (N + per - 1) / per;
}
enum GgType { kBf16, kInt8, kFp8 };  // A; the weights are bf16, int8, bf16

namespace gg {
constexpr int kHalf = 128 * 128;       // bytes of a half operand tile: 128 rows of 128 bytes
constexpr int kRaw = 128 * 64;         // fp8: the same half as e4m3fn bytes
// LDS map.  bf16 / int8: two K steps of B0, A0, B1, A1.  fp8: two K steps of
// B0, B1, one bf16 A tile, two K steps of raw A halves, the row scales.
template <GgType TY> __device__ constexpr int b_at(int buf, int y) {
  return TY == kFp8 ? (buf * 2 + y) * kHalf : (buf * 4 + 2 * y) * kHalf;
}
template <GgType TY> __device__ constexpr int a_at(int buf, int x) {
  return TY == kFp8 ? (4 + x) * kHalf : (buf * 4 + 2 * x + 1) * kHalf;
}
__device__ constexpr int raw_at(int buf, int x) { return 6 * kHalf + (buf * 2 + x) * kRaw; }
__device__ constexpr int sc_at(int buf, int x) { return 8 * kHalf + (buf * 2 + x) * 2048; }
// bf16 / int8 tiles of at most 128 rows: stages of B0, B1 and up to 128 rows of A
constexpr int kStages = 3, kRunMax = 2;
template <GgType TY, bool SHORT>
constexpr int kLds = TY == kFp8 ? 8 * kHalf + 8192
                   : SHORT      ? kStages * 3 * kHalf
                                : 8 * kHalf + (TY == kInt8 ? 2048 : 0);
// int8: the tile's row scales and column scales, past the operands
constexpr int kScales = 8 * kHalf;
static_assert(kStages * 3 * kHalf >= kScales + 2048, "LDS map");

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void dma16(const char* src, char* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ void dma4(const char* src, char* dst) {
  __builtin_amdgcn_global_load_lds((const void*)src,
                                   (__attribute__((address_space(3))) void*)dst, 4, 0, 0);
}
}  // namespace gg

// SHORT: tiles of at most 128 rows take the ring loop.
template <bool SWIGLU, GgType TY, bool SHORT>
__global__ __launch_bounds__(512) void grouped_gemm_kernel(
    const char* __restrict__ a, const char* __restrict__ ident_a, int ident_m,
    const char* __restrict__ w0, const char* __restrict__ w1, const int* __restrict__ offs,
    const int* __restrict__ tile_start, int G, int M, int N, int K, int n_tiles,
    unsigned short* __restrict__ out, GgExtra ex) {
  using namespace gg;
  constexpr bool I8 = TY == kInt8, F8 = TY == kFp8;
  constexpr int EL = I8 ? 1 : 2;       // bytes per weight element
  constexpr int BM = kGgBM;
  __shared__ __attribute__((aligned(1024))) char lds[kLds<TY, SHORT>];
  GgTile tile;
  const int KT = K * EL / 128;
  if (!gg_tile<BM, SHORT>(offs, tile_start, G, M, n_tiles, KT, ident_m, tile)) return;
  // wave-uniform: in SGPRs
  const int g = __builtin_amdgcn_readfirstlane(tile.g), gs = __builtin_amdgcn_readfirstlane(tile.gs);
  const int r0 = __builtin_amdgcn_readfirstlane(tile.r0);
  const int rlast = __builtin_amdgcn_readfirstlane(tile.rlast);
  const int nt = __builtin_amdgcn_readfirstlane(tile.nt);
  const int nt1 = __builtin_amdgcn_readfirstlane(tile.nt1);
  const int rot = __builtin_amdgcn_readfirstlane(tile.rot);
  const bool ident = tile.ident;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int fr = lane & 15, fc = lane >> 4;
  auto swz = [](int r) { return (r >> 1) & 7; };
  const long long rowb = (long long)K * EL;

  // DMA sources, advanced a K step by every issue.  Rows past the group and
  // weight rows past N are loaded (clamped), never stored.
  // B half y, instruction q of this wave: rows (wave*2 + q)*8 .. +8 of the half
  const char* bsrc[2][2];
  auto set_b = [&](int nt) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int r = (wave * 2 + q) * 8 + lane / 8, c = (lane & 7) ^ swz(r);
        const int wrow = SWIGLU ? nt * 128 + r : nt * 256 + y * 128 + r;
        bsrc[y][q] =
            (SWIGLU && y ? w1 : w0) + ((long long)g * N + min(wrow, N - 1)) * rowb + c * 16;
      }
  };
  // A half x: as B.  fp8: one instruction of 16 rows x 64 bytes, wave*16 .. +16, in
  // lane order (only this wave reads it), and the index of the lane's row scale
  // from the tile's first (fewer than 2^31 scales in all)
  constexpr int NA = F8 ? 1 : 2;
  const char* asrc[2][NA];
  unsigned sidx[2];
  const float* ssrc[2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int q = 0; q < NA; ++q) {
      const int r = F8 ? wave * 16 + lane / 4 : (wave * 2 + q) * 8 + lane / 8;
      const int c = F8 ? lane & 3 : (lane & 7) ^ swz(r);
      const int row = min(r0 + x * 128 + r, rlast);
      if constexpr (F8) {
        asrc[x][q] = a + (long long)row * K + c * 16;
        ssrc[x] = ex.a + (long long)r0 * (K / 128);
        sidx[x] = (unsigned)((row - r0) * (K / 128));
      } else {
        const int arow = (!ident && ex.a_idx) ? ex.a_idx[row] : row;
        asrc[x][q] = (ident ? ident_a + (long long)(row - gs) * rowb : a + (long long)arow * rowb) +
                     c * 16;
        ssrc[x] = nullptr;
        sidx[x] = 0;
      }
    }
  auto issue_b = [&](int y, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      dma16(bsrc[y][q], lds + b_at<TY>(buf, y) + (wave * 2 + q) * 1024);
      bsrc[y][q] += 128;
    }
  };
  auto issue_a = [&](int x, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NA; ++q) {
      dma16(asrc[x][q], lds + (F8 ? raw_at(buf, x) : a_at<TY>(buf, x)) + (wave * NA + q) * 1024);
      asrc[x][q] += F8 ? 64 : 128;
    }
  };
  auto issue_s = [&](int x, int sbuf) __attribute__((always_inline)) {
    dma4((const char*)(ssrc[x] + sidx[x]), lds + sc_at(sbuf, x) + wave * 256);
    ssrc[x] += 1;
  };
  // fp8: this wave's 16 rows of raw half x -> bf16(q * s) in the A tile.  Each
  // element is converted once per block, half a K step before it is read.
  auto convert = [&](int x, int buf, int sbuf) __attribute__((always_inline)) {
    if (r0 + x * 128 + wave * 16 > rlast) return;  // all past the group: never stored
    const float sc = *reinterpret_cast<const float*>(lds + sc_at(sbuf, x) + wave * 256 + lane * 4);
    const u32x4 raw =
        *reinterpret_cast<const u32x4*>(lds + raw_at(buf, x) + wave * 1024 + lane * 16);
    bf16x8 lo8, hi8;
    dequant16(raw, sc, lo8, hi8);
    const int r = wave * 16 + lane / 4, c = 2 * (lane & 3);
    char* d = lds + a_at<TY>(0, x) + r * 128;
    *reinterpret_cast<bf16x8*>(d + ((c ^ swz(r)) * 16)) = lo8;
    *reinterpret_cast<bf16x8*>(d + (((c + 1) ^ swz(r)) * 16)) = hi8;
  };

  using AccV = typename AccOf<I8>::type;
  AccV acc[2][2][4][2];  // [A half][B half][16-row block][16-column block]
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[x][y][i][j] = AccV{0, 0, 0, 0};
  bf16x8 fa[2][4], fb0[2][2][2], fb1[2][2];  // [kk][i]; B0: [step parity][kk][j]; B1: [kk][j]
  // fragment addresses: this wave's rows of a half, chunk kk*4 + fc
  int aoff[2], boff[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int c = ((kk * 4 + fc) ^ swz(fr)) * 16;
    aoff[kk] = (wm * 64 + fr) * 128 + c;
    boff[kk] = (wn * 32 + fr) * 128 + c;
  }
  auto read_a = [&](int x, int buf) __attribute__((always_inline)) {
    const char* p = lds + a_at<TY>(buf, x);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        fa[kk][i] = *reinterpret_cast<const bf16x8*>(p + aoff[kk] + i * 2048);
  };
  auto read_b = [&](bf16x8 (&fb)[2][2], int y, int buf) __attribute__((always_inline)) {
    const char* p = lds + b_at<TY>(buf, y);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        fb[kk][j] = *reinterpret_cast<const bf16x8*>(p + boff[kk] + j * 2048);
  };
  // a wave whose rows of a half all lie past the group skips its MFMAs
  const bool live0 = r0 + wm * 64 <= rlast, live1 = r0 + 128 + wm * 64 <= rlast;
  // the 32 MFMAs of a half step, between two barriers
  auto mma = [&](int x, const bf16x8 (&b0)[2][2], bool live) __attribute__((always_inline)) {
    barrier();
    if (live) {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acc[x][y][i][j] =
                  mfma_step<I8>(fa[kk][i], y ? fb1[kk][j] : b0[kk][j], acc[x][y][i][j]);
    }
    barrier();
  };

  const int rows = rlast + 1 - r0;  // of this tile, 256 if more
  // The block's column tiles over at most RA = 128 or 64 rows (a small group, or a
  // group's last tile): the loads bound them, so all waves step together through a
  // ring of three stages of RA rows of A and the 256 weight rows, one barrier a step,
  // two steps in flight, also across the end of a tile.  A wave has RA / 2 rows and
  // 64 weight rows (SwiGLU: 32 of each half).  Only 16-row blocks that hold rows are
  // loaded, read, multiplied and stored.  The MFMA operands are swapped, so a lane
  // ends with four neighbouring columns of a row (column fc*4 + e, row fr of a
  // 16 x 16 block); two column blocks exchanged between lanes make 16-byte stores, 64
  // bytes of a row per instruction.
  auto short_run = [&]<int RA>(std::integral_constant<int, RA>) __attribute__((always_inline)) {
    constexpr int NB = kStages, STAGE = 2 * kHalf + RA * 128, NI = RA / 32, NY = SWIGLU ? 1 : 2;
    constexpr int OUTC = SWIGLU ? 128 : 256;
    const int wr = wm * (RA / 2), wc = wn * (SWIGLU ? 32 : 64);
    constexpr int YB = SWIGLU ? 128 : 32;  // B rows between the wave's two blocks y
    const int nb = min(max((rows - wr + 15) >> 4, 0), NI);  // this wave's blocks with rows
    const int len = nt1 - nt, S = KT * len;
    auto tile_at = [&](int j) { return nt + (j + rot >= len ? j + rot - len : j + rot); };
    // int8: the row scale of row fr, the column scales of column fr for every tile
    float rs[NI], cs[kRunMax][2][2];
    if constexpr (I8) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int row = min(r0 + wr + i * 16 + fr, rlast);
        rs[i] = ident ? ex.ident[row - gs] : ex.a[ex.a_idx ? ex.a_idx[row] : row];
      }
#pragma unroll
      for (int c = 0; c < kRunMax; ++c)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int col =
                tile_at(min(c, len - 1)) * OUTC + (SWIGLU ? 0 : y * 32) + wc + j * 16 + fr;
            cs[c][y][j] = (SWIGLU && y ? ex.w1 : ex.w0)[(long long)g * N + min(col, N - 1)];
          }
    }
    const bool loads_a = wave * 16 < rows;
    int kin = 0, jin = 0;  // K step and tile of the next issue
    set_b(tile_at(0));
    auto issue = [&](int st) __attribute__((always_inline)) {
      char* d = lds + st * STAGE + wave * 2048;
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          dma16(bsrc[y][q], d + y * kHalf + q * 1024);
          bsrc[y][q] += 128;
        }
      if (loads_a) {
#pragma unroll
        for (int q = 0; q < NA; ++q) {
          dma16(asrc[0][q], d + 2 * kHalf + q * 1024);
          asrc[0][q] += 128;
        }
      }
      if (++kin == KT) {
        kin = 0;
        set_b(tile_at(++jin));
#pragma unroll
        for (int q = 0; q < NA; ++q) asrc[0][q] -= rowb;
      }
    };
    // a run shorter than the ring: the stages past it are loaded (weight rows are
    // clamped) and not read
#pragma unroll
    for (int q = 0; q < NB - 1; ++q) issue(q);
    int st_in = NB - 1, st = 0;
    if constexpr (I8) {  // the scales are here before the loop's own waits begin
#pragma unroll
      for (int i = 0; i < NI; ++i) asm volatile("" : "+v"(rs[i]));
#pragma unroll
      for (int c = 0; c < kRunMax; ++c)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int j = 0; j < 2; ++j) asm volatile("" : "+v"(cs[c][y][j]));
    }
    int ao[2], bo[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int c = ((kk * 4 + fc) ^ swz(fr)) * 16;
      ao[kk] = 2 * kHalf + (wr + fr) * 128 + c;
      bo[kk] = (wc + fr) * 128 + c;
    }
    auto product = [&](int y, int i, int j, int e) -> float {
      if constexpr (I8)
        return (float)acc[0][y][i][j][e] * (rs[i] * __shfl(cs[0][y][j], fc * 4 + e, 64));
      else
        return acc[0][y][i][j][e];
    };
    int kt = 0, jt = 0;
    for (int u = 0; u < S; ++u) {
      // this wave's part of the step landed once at most the next one is outstanding
      // (stores count too: then it waits for more); the barrier makes that true for
      // every wave, and every wave is past its reads of the stage refilled now
      const int rem = S - 1 - u;
      if (rem == 0) wait_vm<0>();
      else if (loads_a) wait_vm<6>();
      else wait_vm<4>();
      barrier();
      if (rem >= NB - 1) issue(st_in);
      const char* p = lds + st * STAGE;
      if (nb > 0) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            fb0[0][kk][j] = *reinterpret_cast<const bf16x8*>(p + bo[kk] + j * 2048);
            fb1[kk][j] = *reinterpret_cast<const bf16x8*>(p + YB * 128 + bo[kk] + j * 2048);
          }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          if (i >= nb) break;
#pragma unroll
          for (int kk = 0; kk < 2; ++kk)
            fa[kk][i] = *reinterpret_cast<const bf16x8*>(p + ao[kk] + i * 2048);
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          if (i >= nb) break;
#pragma unroll
          for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
              for (int j = 0; j < 2; ++j)
                acc[0][y][i][j] =
                    mfma_step<I8>(y ? fb1[kk][j] : fb0[0][kk][j], fa[kk][i], acc[0][y][i][j]);
        }
      }
      st = st == NB - 1 ? 0 : st + 1;
      st_in = st_in == NB - 1 ? 0 : st_in + 1;
      if (++kt < KT) continue;
      kt = 0;  // the tile is complete
      const int c0 = tile_at(jt++) * OUTC + wc;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (i >= nb) break;
        const int rl = wr + i * 16 + fr;
        unsigned short* o = out + (long long)(r0 + rl) * N;
#pragma unroll
        for (int y = 0; y < NY; ++y) {
          unsigned short v[2][4];
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              v[j][e] = (unsigned short)f2bf(
                  SWIGLU ? swiglu(product(0, i, j, e), product(1, i, j, e)) : product(y, i, j, e));
          if ((N & 7) == 0) {
            // lanes of odd fc give column block 0 and take column block 1
            u32x4 pk;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const auto sw = __builtin_amdgcn_permlane16_swap(
                  (unsigned)v[0][2 * h] | (unsigned)v[0][2 * h + 1] << 16,
                  (unsigned)v[1][2 * h] | (unsigned)v[1][2 * h + 1] << 16, false, false);
              pk[h] = sw[0];
              pk[2 + h] = sw[1];
            }
            const int col = c0 + y * 32 + (fc & 1) * 16 + (fc >> 1) * 8;
            if (rl < rows && col < N) *reinterpret_cast<u32x4*>(o + col) = pk;
          } else {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int col = c0 + y * 32 + j * 16 + fc * 4 + e;
                if (rl < rows && col < N) o[col] = v[j][e];
              }
          }
        }
      }
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[0][y][i][j] = AccV{0, 0, 0, 0};
      if constexpr (I8) {
#pragma unroll
        for (int c = 0; c + 1 < kRunMax; ++c)
#pragma unroll
          for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int j = 0; j < 2; ++j) cs[c][y][j] = cs[c + 1][y][j];
      }
    }
  };
  if constexpr (SHORT) {
    if (rows <= 64) {
      short_run(std::integral_constant<int, 64>{});
      return;
    }
    if (rows <= 128) {
      short_run(std::integral_constant<int, 128>{});
      return;
    }
  }
  {
    set_b(nt);
    if constexpr (I8) {
      // The scales land under the K loop: 256 row scales (waves 0 .. 3), then the 256
      // column scales in B row order.  As loads at the epilogue's start (36 a lane, behind
      // the row indexes) nothing hid them, and short K was slower than with 128 x 512 tiles
      // (256 rows an expert on average, weights N x K, us, 128 x 512 tiles / loads there /
      // this: 64 experts 1024 x 512 30.4 / 31.4 / 27.0, 200 rows 20.1 / 20.5 / 18.2;
      // 64 experts SwiGLU 512 x 1024 43.4 / 43.0 / 38.1; 32 experts SwiGLU 3584 x 8192
      // 677 / 575 / 562).
      const int i = (wave & 3) * 64 + lane;
      const float* src;
      if (wave < 4) {
        const int row = min(r0 + i, rlast);
        src = ident ? ex.ident + (row - gs) : ex.a + (ex.a_idx ? ex.a_idx[row] : row);
      } else {
        const int col = SWIGLU ? nt * 128 + (i & 127) : nt * 256 + i;
        src = (SWIGLU && i >= 128 ? ex.w1 : ex.w0) + (long long)g * N + min(col, N - 1);
      }
      dma4((const char*)src, lds + kScales + wave * 256);
    }
    issue_b(0, 0);
    issue_a(0, 0);
    if constexpr (F8) issue_s(0, 0);
    issue_b(1, 0);
    issue_a(1, 0);
    if constexpr (F8) issue_s(1, 0);
    if (KT > 1) {
      issue_b(0, 1);
      issue_a(0, 1);
      issue_b(1, 1);
      if constexpr (F8) {
        issue_a(1, 1);
        wait_vm<6>();  // step 0 landed
      } else {
        wait_vm<8>();  // B0, A0 and B1 of step 0 landed
      }
    } else {
      wait_vm<2>();  // not fp8 (K % 128 == 0): all but A1
    }
    barrier();
    read_b(fb0[0], 0, 0);
    if constexpr (F8) convert(0, 0, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
    if (wm == 1) barrier();  // half a step behind the other group from here on
    // P: parity of the step; rem: steps after it; sb (fp8): scale buffer of the step
    auto step = [&]<int P>(std::integral_constant<int, P>, int rem, int sb)
                    __attribute__((always_inline)) {
      read_a(0, P);
      read_b(fb1, 1, P);
      if constexpr (F8) {
        convert(1, P, sb);
        // per half step B0 + raw A0 or B1 + raw A1 (3 loads), in even steps a scale
        // too: what the next half needs was issued two half steps ago
        if (rem >= 2) {
          issue_b(0, P);
          issue_a(0, P);
          if (P == 0) issue_s(0, sb ^ 1);
          wait_vm<7>();
        } else if (P == 0) {
          wait_vm<3>();
        } else {
          wait_vm<0>();
        }
      } else {
        // in flight after the loads that the next half needs (A1 of this step, B0 of
        // the next): A0 and B1 of the next step and the two elements issued here
        if (rem >= 2) {
          issue_a(1, P ^ 1);
          issue_b(0, P);
          wait_vm<8>();
        } else if (rem == 1) {
          issue_a(1, P ^ 1);
          wait_vm<6>();
        } else {
          wait_vm<0>();
        }
      }
      mma(0, fb0[P], live0);
      read_a(1, P);
      read_b(fb0[P ^ 1], 0, P ^ 1);  // past the last step: not used
      if constexpr (F8) {
        if (rem >= 1) convert(0, P ^ 1, P == 0 ? sb : sb ^ 1);
        if (rem >= 2) {
          issue_b(1, P);
          issue_a(1, P);
          if (P == 0) issue_s(1, sb ^ 1);
          wait_vm<P == 0 ? 8 : 6>();
        } else {
          wait_vm<0>();
        }
      } else if (rem >= 2) {
        issue_a(0, P);
        issue_b(1, P);
        wait_vm<8>();
      } else {
        wait_vm<2>();  // rem 1: A1 of the last step may still be in flight
      }
      mma(1, fb0[P], live1);
    };
    int sb = 0;
    for (int kt = 0; kt < KT; kt += 2) {
      step(std::integral_constant<int, 0>{}, KT - 1 - kt, sb);
      if (F8 || kt + 1 < KT) step(std::integral_constant<int, 1>{}, KT - 2 - kt, sb);
      if (F8) sb ^= 1;
    }
    if (wm == 0) barrier();
  }

  // ---- epilogue: element e of a 16 x 16 block is row fc*4 + e, column fr.
  // SwiGLU: B half 0 is the gate, half 1 the up product of the same columns.
  // int8: value = float(acc) * (row scale * column scale).
  constexpr int OUTC = SWIGLU ? 128 : 256, NY = SWIGLU ? 1 : 2;
  auto colof = [&](int y, int j) { return y * 128 + wn * 32 + j * 16 + fr; };
  auto rowof = [&](int x, int i, int e) { return x * 128 + wm * 64 + i * 16 + fc * 4 + e; };
  float cs[2][2];
  f32x4 rs[2][4];
  if constexpr (I8) {
    const float* sc = reinterpret_cast<const float*>(lds + kScales);
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int j = 0; j < 2; ++j) cs[y][j] = sc[256 + colof(y, j)];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) rs[x][i] = *reinterpret_cast<const f32x4*>(sc + rowof(x, i, 0));
  }
  auto product = [&](int x, int y, int i, int j, int e) -> float {
    if constexpr (I8) return (float)acc[x][y][i][j][e] * (rs[x][i][e] * cs[y][j]);
    else return acc[x][y][i][j][e];
  };
  auto value = [&](int x, int y, int i, int j, int e) -> float {
    if constexpr (SWIGLU) return swiglu(product(x, 0, i, j, e), product(x, 1, i, j, e));
    else return product(x, y, i, j, e);
  };
  if ((N & 7) == 0) {
    // the bf16 tile through LDS (16-byte chunk c of row rl at c ^ 2*((rl >> 2) & 3):
    // the four row groups of one write land in distinct banks), then whole
    // 16-byte chunks of output rows
    constexpr int RCH = OUTC / 8;
    unsigned short* ct = reinterpret_cast<unsigned short*>(lds);
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int rl = rowof(x, i, e), sw = 2 * ((rl >> 2) & 3);
#pragma unroll
          for (int y = 0; y < NY; ++y)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const int cl = colof(y, j);
              ct[rl * OUTC + (((cl >> 3) ^ sw) << 3) + (cl & 7)] =
                  (unsigned short)f2bf(value(x, y, i, j, e));
            }
        }
    __syncthreads();
    const int c0 = nt * OUTC;
    for (int q = threadIdx.x; q < BM * RCH; q += 512) {
      const int rl = q / RCH, c = q % RCH;
      const int row = r0 + rl, col = c0 + c * 8;
      if (row > rlast || col >= N) continue;
      const u32x4 v =
          *reinterpret_cast<const u32x4*>(ct + rl * OUTC + ((c ^ (2 * ((rl >> 2) & 3))) << 3));
      *reinterpret_cast<u32x4*>(out + (long long)row * N + col) = v;
    }
    return;
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = r0 + rowof(x, i, e);
        if (row > rlast) continue;
#pragma unroll
        for (int y = 0; y < NY; ++y)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int col = nt * OUTC + colof(y, j);
            if (col < N) out[(long long)row * N + col] = (unsigned short)f2bf(value(x, y, i, j, e));
          }
      }
}

template <GgType TY>
static hipError_t launch_gg(const void* a, const void* ident_a, int ident_m, const void* w0,
                            const void* w1, const int32_t* offs, int G, int M, int N, int K,
                            bool swiglu, void* out, int32_t* tile_start, hipStream_t s,
                            GgExtra ex) {
  if (G > kScanG) {
    hipLaunchKernelGGL(gg_plan_kernel, dim3(1), dim3(1024), 0, s, offs, G, M, kGgBM, tile_start);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (M == 0 || N == 0 || G == 0) return hipSuccess;
  const int n_tiles = grouped_gemm_n_tiles(N, swiglu);
  // Groups of at most 128 rows on average: the kernel with the ring loop for short
  // tiles.  The one without it keeps 0.3 .. 0.6% at T = 8192 (whole layer 10.31 /
  // 10.36 ms; it needs 256 registers).
  constexpr bool kRing = TY != kFp8;
  constexpr int EL = TY == kInt8 ? 1 : 2;
  const bool ring = kRing && (long long)M <= 128ll * G;
  // Runs are chosen here as if the rows reached groups at random and all were short, and
  // again by every block for the real counts, as far as this grid holds them.  Above 96
  // rows on average some random group is long: its blocks would open another round of
  // two-tile ones (bf16, 128 experts, 1024 x 1024, 100 rows: 64 / 86 us).
  const int reach = (int)(G * (1.0 - std::exp(-(double)M / G)) + 0.5);
  const int log = ring && G <= kScanG && (long long)M <= 96ll * G
                      ? gg_run(reach, reach, n_tiles, K * EL / 128, 0x7fffffff)
                      : 0;
  const long long blocks = gg_grid(M, G, n_tiles, log);
  const dim3 grid((unsigned)((blocks + 7) / 8 * 8)), blk(512);
#define MOE_GG(SW, SH)                                                                         \
  hipLaunchKernelGGL((grouped_gemm_kernel<SW, TY, SH>), grid, blk, 0, s, (const char*)a,        \
                     (const char*)ident_a, ident_m, (const char*)w0,                           \
                     (const char*)(swiglu ? w1 : w0), offs, tile_start, G, M, N, K, n_tiles,   \
                     (unsigned short*)out, ex)
  if (swiglu) {
    if (ring) MOE_GG(true, kRing);
    else MOE_GG(true, false);
  } else {
    if (ring) MOE_GG(false, kRing);
    else MOE_GG(false, false);
  }
#undef MOE_GG
  return hipGetLastError();
}

// tile_start: [G+1] ints of workspace.  offs: inclusive group ends (device).
// a_scales == NULL: a is bf16.  Else a is e4m3fn bytes with one fp32 scale per
// row and 128-wide K block ([M, K/128]).  a_rows (bf16 A only; may be NULL):
// operand row r is row a_rows[r] of a.
hipError_t launch_grouped_gemm(const void* a, const float* a_scales, const int32_t* a_rows,
                               const void* ident_a, int ident_m, const void* w0, const void* w1,
                               const int32_t* offs, int G, int M, int N, int K, bool swiglu,
                               void* out, int32_t* tile_start, hipStream_t s) {
  if (a_scales)
    return launch_gg<kFp8>(a, ident_a, ident_m, w0, w1, offs, G, M, N, K, swiglu, out, tile_start,
                           s, GgExtra{a_scales, nullptr, nullptr, nullptr, nullptr});
  return launch_gg<kBf16>(a, ident_a, ident_m, w0, w1, offs, G, M, N, K, swiglu, out, tile_start,
                          s, GgExtra{nullptr, a_rows, nullptr, nullptr, nullptr});
}

// int8 A and weights, int32 accumulation, 128-wide K steps (LDS rows of 128
// bytes as in bf16).
hipError_t launch_grouped_gemm_i8(const void* a, const float* a_rs, const int32_t* a_rs_idx,
                                  const void* ident_a, const float* ident_rs, int ident_m,
                                  const void* w0, const float* w0s, const void* w1,
                                  const float* w1s, const int32_t* offs, int G, int M, int N, int K,
                                  bool swiglu, void* out, int32_t* tile_start, hipStream_t s) {
  return launch_gg<kInt8>(a, ident_a, ident_m, w0, w1, offs, G, M, N, K, swiglu, out, tile_start,
                          s, GgExtra{a_rs, a_rs_idx, ident_rs, w0s, swiglu ? w1s : w0s});
}

}  // namespace moe
