// bf16 GEMM with both operands K-contiguous, fed into LDS by buffer loads
// (buffer_load_dwordx4 ... lds, gfx950).
//
// Operand tiles (rows x 64 k) live in LDS as 128-byte rows without padding. The 16-byte
// chunk c of row R sits at physical chunk c ^ swz(R), swz(R) = (R & 7) ^ ((R >> 3) & 1),
// so the 16 consecutive rows a quarter-wave fragment read touches cover all 64 banks.
// Each load instruction moves one 1 KB block of whole rows: lane l writes physical chunk
// l % 8 of row l / 8, so it fetches the logical chunk the swizzle puts there.
//
// Operand addressing: a tile's rows start at a per-tile buffer descriptor base (scalar
// registers); each load's per-lane byte offset (row within the tile, swizzled chunk) is
// computed once per kernel and the stage's k position is added to it. The descriptor's
// record count ends at the operand's last row, so rows past the operand extent, and
// chunks past the end of its last row, load as zeros; their outputs are never stored.
//
// A ring of NS LDS stages (two, three or four), software-pipelined inside a wave
// (pipe_stage). A stage is four k16 steps; the fragments of step n+1 are read from LDS
// between the MFMAs of step n (two register sets), and the last step of a stage reads the
// first fragments of the next one, after the one barrier of the stage: this wave's loads of
// the next stage have landed (vmcnt) and its reads of this stage are done (lgkmcnt), so
// behind the barrier the next stage is visible and this one's space is free. The loads of
// stage kt+NS go out between the MFMAs of stage kt's last step; with SPLIT (256x256 tiles,
// two stages) half of them between those of stage kt+1's first step. A tile's last stage
// loads, reads and waits for nothing (run like the others, on empty descriptors, it cost
// contractions of one to six stages 5-8%). The order is
// pinned by scheduling barriers: left to itself the compiler reads a step's fragments into
// the registers of the step before, after its MFMAs, so a wave alternates between waiting
// for LDS and computing. Same products, same k order, so the same bits as the unpipelined
// loop; 256x256 tiles 4096x3072x4096 with B MN-major 131 -> 104 us (785 -> 994 TFLOP/s),
// both MN-major 137 -> 104 us, K-major 8192x4096x3072 210 -> 169 us. By the
// counters (8192x4096x3072 in 256x256 tiles) the matrix cores are busy 0.78 of the clocks
// in which a CU holds a block and the LDS reads 0.31, so the LDS port does not bound it;
// the rest is the stage barrier and its waits, 0.14 of the launch without a block (first
// loads, epilogue, last round), and a clock that falls to 1.8 GHz under this load.
// The barrier is a bare s_barrier with compiler-only memory clobbers: a fenced
// __syncthreads would wait for every load in flight.
//
// The MFMA runs with the operands swapped (B rows as the 32-row "A" input), so each lane
// ends with 4 consecutive output columns of one row per 4 accumulators; the epilogue
// writes them as one 8-byte (bf16) or 16-byte (fp32) store.
//
// Ragged contraction groups start at the 64-aligned k below the group's first row, so
// every 128-byte piece of a K-major row a stage loads is one whole cache line (from an
// 8-aligned start each piece straddled two lines: 20-25% slower weight gradients); k
// outside [kmin, kend) is zeroed in the fragments of a tile's first and last stage.
//
// MN-major operands (stored [K][rows], rows contiguous: the B of x @ V and acts @ U, both
// operands of a weight gradient x^T @ g). A stage of such an operand holds its 64 k-rows
// of R = BM (or BN) elements, 2R bytes each; the 16-byte chunk c of k-row r sits at
// physical chunk c ^ (4 * (r & 3)). One 1 KB load moves 1024 / 2R whole k-rows (lane l
// writes physical chunk l % (R / 8) of k-row l / (R / 8)). Fragments come out of LDS
// already transposed by ds_read_b64_tr_b16: within each 16-lane group, output lane
// 4a + b receives element b of the 8 bytes read by source lanes a, a + 4, a + 8, a + 12.
// Source lane 16g + 4e + a reads k-row 8 (g >> 1) + 4h + e (h = 0, 1: the fragment's two
// halves), elements 16 (g & 1) + 4a .. + 3 of the fragment's 32 rows, so output lane l
// holds rows l & 31 at k 8 (l >> 5) + 4h .. + 3: the same fragment the K-major path reads
// with one ds_read_b128. The four k-rows one 16-lane group reads (r & 3 = e = 0..3) sit in
// four distinct 64-byte bank groups, so a half-wave's 256 bytes are conflict-free.
#pragma once

#include <type_traits>

#include "pd_common.hpp"

namespace pd {

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((address_space(3))) void lds_void_t;

enum GemmMode { MODE_DENSE = 0, MODE_GROUPED = 1, MODE_GROUPED_K = 2, MODE_BATCHED = 3, MODE_SPLITK = 4 };

struct GemmArgs {
  int64_t M, N, K;
  const bf16_t* A;
  int64_t lda;
  const bf16_t* B;
  int64_t ldb;
  void* C;
  int64_t ldc;
  float alpha, beta;
  const int32_t* offsets;  // [E+1] group offsets (grouped modes)
  int E;
  int64_t strideB;  // elements between consecutive groups' B (GROUPED, BATCHED)
  int64_t strideC;  // elements between consecutive groups' C (GROUPED_K, BATCHED)
  int64_t strideA;  // elements between consecutive batches' A (BATCHED; 0 = shared)
  // Grouped modes: a second problem of identical shape and group offsets in the same
  // launch (gridDim.z doubles; the upper half uses A2/B2/C2). NULL = one problem.
  const bf16_t* A2;
  const bf16_t* B2;
  void* C2;
};

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2): give
// XCD x a contiguous range [x*q + min(x, r), ...) of the linear tile order (q, r =
// total / 8, total % 8) so tiles that share operand panels share an L2.
__device__ inline int64_t xcd_contiguous(int64_t L, int64_t total) {
  const int64_t x = L & 7, q = total >> 3, r = total & 7;
  return x * q + (x < r ? x : r) + (L >> 3);
}

// Number of BM-row tiles of group g (0 past the last group or for empty groups).
__device__ inline int group_tiles(const int32_t* __restrict__ off, int g, int E, int BMv) {
  if (g >= E) return 0;
  const int sz = off[g + 1] - off[g];
  return sz > 0 ? (sz + BMv - 1) / BMv : 0;
}

__device__ inline int wave_incl_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

// XCD-aware order for dense launches: XCD-contiguous ranges, then groups of 8 row
// tiles walked column by column.
__device__ inline void dense_tile(int& my, int& nx) {
  const int gx = gridDim.x, gy = gridDim.y;
  const int total = gx * gy;
  int L = blockIdx.y * gx + blockIdx.x;
  if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
  const int GROUP = 8;
  const int g = L / (GROUP * gx);
  const int first = g * GROUP;
  const int gm = gy - first < GROUP ? gy - first : GROUP;
  const int within = L - g * GROUP * gx;
  my = first + within % gm;
  nx = within / gm;
}

// One block's output tile: rows [m0, M) of the block's problem (M is an absolute bound),
// columns from n0, contraction [kbeg, kend), and the operand/output bases.
struct TileJob {
  int64_t m0, n0, M, kbeg, kend;
  const bf16_t* A;
  const bf16_t* B;
  void* C;
  int prob;    // 0, or 1 for the second problem of a paired launch
  int64_t lin;  // GROUPED: the tile's index within its problem, < (J / BM + E) * ceil(N / BN)
  int e;        // GROUPED / GROUPED_K: the tile's group (expert); 0 otherwise
};

// Maps this block to its tile (the four problem mappings); false = no work.
template <int BM, int BN, int MODE, typename TC>
__device__ inline bool map_tile(const GemmArgs& p, int lane, TileJob& t) {
  t.M = p.M;
  t.A = p.A;
  t.B = p.B;
  t.C = p.C;
  t.kbeg = 0;
  t.kend = p.K;
  t.prob = 0;
  t.lin = 0;
  t.e = 0;
  if (MODE == MODE_DENSE) {
    int my, nx;
    dense_tile(my, nx);
    t.m0 = (int64_t)my * BM;
    t.n0 = (int64_t)nx * BN;
  } else if (MODE == MODE_GROUPED) {
    // Row tiles are enumerated over all groups in order. Every wave scans the groups'
    // tile counts 64 at a time (lane = group); the grid has a few spare rows of blocks,
    // so the XCD remap runs over the tiles that exist. With E <= 64 one load of the
    // offsets serves the count, the lookup and the group's row range.
    const int64_t gx = gridDim.x;
    const int64_t lin = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gx + blockIdx.x;
    int e = -1, before = 0, tile = 0;
    int64_t off = 0, end = 0;
    auto pick = [&](int64_t per) -> bool {  // this block's (problem, column, row tile)
      if (lin >= per * gridDim.z) return false;
      int64_t lr = xcd_contiguous(lin, per * gridDim.z);
      if (lr >= per) {  // second problem of a paired launch
        lr -= per;
        t.A = p.A2;
        t.B = p.B2;
        t.C = p.C2;
        t.prob = 1;
      }
      t.n0 = (lr % gx) * BN;
      t.lin = lr;
      tile = (int)(lr / gx);
      return true;
    };
    if (p.E <= 64) {
      const bool in = lane < p.E;
      const int lo = in ? p.offsets[lane] : 0, hi = in ? p.offsets[lane + 1] : 0;
      const int nt = in && hi > lo ? (hi - lo + BM - 1) / BM : 0;
      const int incl = wave_incl_scan(nt, lane);
      if (!pick((int64_t)__shfl(incl, 63, 64) * gx)) return false;
      const unsigned long long hit = __ballot(incl > tile);
      if (!hit) return false;
      const int ln = __ffsll(hit) - 1;
      e = ln;
      before = __shfl(incl - nt, ln, 64);
      off = __shfl(lo, ln, 64);
      end = __shfl(hi, ln, 64);
    } else {
      int real = 0;
      for (int g0 = 0; g0 < p.E; g0 += 64)
        real += __shfl(wave_incl_scan(group_tiles(p.offsets, g0 + lane, p.E, BM), lane), 63, 64);
      if (!pick((int64_t)real * gx)) return false;
      for (int g0 = 0, base = 0; g0 < p.E; g0 += 64) {
        const int nt = group_tiles(p.offsets, g0 + lane, p.E, BM);
        const int incl = wave_incl_scan(nt, lane);
        const unsigned long long hit = __ballot(base + incl > tile);
        if (hit) {
          const int ln = __ffsll(hit) - 1;
          e = g0 + ln;
          before = base + __shfl(incl - nt, ln, 64);
          break;
        }
        base += __shfl(incl, 63, 64);
      }
      if (e < 0) return false;
      off = p.offsets[e];
      end = p.offsets[e + 1];
    }
    t.M = end < p.M ? end : p.M;  // absolute row bound, clamped to J
    t.m0 = off + (int64_t)(tile - before) * BM;
    if (t.m0 < 0) return false;
    t.B += (int64_t)e * p.strideB;
    t.e = e;
  } else if (MODE == MODE_SPLITK) {
    // a dense tile, over the contraction slice blockIdx.z of gridDim.z equal slices of
    // p.strideA k each (a multiple of 64); slice z writes its partial sum to
    // C + z * strideC (the caller adds the slices in order)
    int my, nx;
    dense_tile(my, nx);
    t.m0 = (int64_t)my * BM;
    t.n0 = (int64_t)nx * BN;
    t.kbeg = (int64_t)blockIdx.z * p.strideA;
    t.kend = t.kbeg + p.strideA < p.K ? t.kbeg + p.strideA : p.K;
    t.C = (TC*)p.C + (int64_t)blockIdx.z * p.strideC;
  } else if (MODE == MODE_BATCHED) {
    // blockIdx.z = batch; each operand advances by its own stride (0 = shared)
    const int64_t z = blockIdx.z;
    t.m0 = (int64_t)blockIdx.y * BM;
    t.n0 = (int64_t)blockIdx.x * BN;
    t.A = p.A + z * p.strideA;
    t.B = p.B + z * p.strideB;
    t.C = (TC*)p.C + z * p.strideC;
  } else {
    const int64_t gx = gridDim.x, gxy = gx * gridDim.y;
    const int64_t lin = ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gx + blockIdx.x;
    const int64_t lr = xcd_contiguous(lin, gxy * gridDim.z);
    int e = (int)(lr / gxy);
    if (e >= p.E) {  // second problem of a paired launch (gridDim.z = 2E)
      e -= p.E;
      t.A = p.A2;
      t.B = p.B2;
      t.C = p.C2;
      t.prob = 1;
    }
    t.m0 = (lr % gxy) / gx * BM;
    t.n0 = (lr % gx) * BN;
    t.kbeg = p.offsets[e] < 0 ? 0 : p.offsets[e];
    t.kend = p.offsets[e + 1] < p.K ? p.offsets[e + 1] : p.K;  // clamped to J
    if (t.kend < t.kbeg) t.kend = t.kbeg;
    t.C = (TC*)t.C + (int64_t)e * p.strideC;
    t.e = e;
  }
  return t.m0 < t.M && t.n0 < p.N;
}

// SPLIT: the loads of a stage go out in two halves; NS: LDS stages (see the top of this
// file).
template <int BM_, int BN_, int WM_, int WN_, bool SPLIT_, int NS_ = 2>
struct DtlCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, NS = NS_, BK = 64;
  static constexpr int NW = WM_ * WN_, NT = NW * 64;
  static constexpr int WTM = BM_ / WM_, WTN = BN_ / WN_;  // wave tile
  static constexpr int TM = WTM / 32, TN = WTN / 32;
  static constexpr int ROWB = 128, RPI = 8;  // LDS row bytes, rows per 1 KB load
  static constexpr int KK = BK / 16;         // k16 MFMA steps per stage
  static constexpr int STAGE_BYTES = (BM_ + BN_) * ROWB;
  static constexpr int A_INSTS = BM_ / (RPI * NW), B_INSTS = BN_ / (RPI * NW);  // 1 KB loads per wave per stage
  static constexpr int INSTS = A_INSTS + B_INSTS;
  static constexpr int HALF = SPLIT_ ? INSTS / 2 : INSTS;  // loads in the first half
  static_assert(NW % 2 == 0, "the swizzle parity of a wave's rows must not depend on the load index");
  static_assert(BM_ % (RPI * NW) == 0 && BN_ % (RPI * NW) == 0, "every wave moves whole 1 KB row blocks");
  static_assert(TM >= 1 && TN >= 1 && WTM % 32 == 0 && WTN % 32 == 0, "wave tile is a multiple of 32x32");
  static_assert(NS >= 2 && NS * STAGE_BYTES <= 160 * 1024, "LDS");
  static __device__ __host__ int ring(int64_t kt) { return (int)((uint32_t)kt % (uint32_t)NS); }  // stage kt's space
  static_assert(NS == 2 || !SPLIT_, "split loads are written for two stages");
  // loads in flight that a stage's readers need not wait for: those of the later stages
  static constexpr int AHEAD = (NS - 2) * INSTS;
};

// s_waitcnt on the vector-memory counter only (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] |
// lgkmcnt[11:8] | vmcnt_hi[15:14]; expcnt and lgkmcnt at their maxima = no wait).
template <int N>
__device__ inline void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Waits until at most N of this wave's buffer loads are in flight and for its LDS operations
// (lgkmcnt = 0).
template <int N>
__device__ inline void wait_loads_and_lds() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
}

// A bare s_barrier: it orders the waves but waits for none of this wave's memory
// operations (gfx950 inserts no wait before s_barrier). It suffices where the LDS data
// the barrier publishes arrived by buffer-to-LDS loads already waited for (vmcnt), or
// where it only frees LDS whose reads this wave has consumed.
__device__ inline void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A barrier after which every LDS access (ds_read / ds_write) any wave made before it has
// completed: LDS written before it is visible to all, LDS read before it is free to
// overwrite. This wave's LDS operations complete first (lgkmcnt = 0; the gfx9 s_waitcnt
// fields vmcnt [3:0] + [15:14] and expcnt [6:4] stay at their maxima), then the s_barrier.
__device__ inline void lds_write_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Physical-chunk swizzle of LDS row R (see the top of this file).
__device__ inline int dtl_swz(int R) { return (R & 7) ^ ((R >> 3) & 1); }

__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline int64_t uni64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)(uint64_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// 128x128x64 tiles (64 KB of LDS, two blocks per CU): 8 waves of 32x64, or 4 waves of 64x64,
// which read 4 fragments for 4 MFMAs instead of 3 for 2 but leave fewer waves to cover a
// transposing read's or an epilogue's latency. K-major 8192x1024x768 17.6 (4 waves) against
// 18.6 us, both MN-major 768x4096x4096 51 (8 waves) against 55; loads in two halves: 60.
typedef DtlCfg<128, 128, 4, 2, false> CfgDtl;
typedef DtlCfg<128, 128, 2, 2, false> CfgDtlRA;
// The same tile with a four-stage ring (one block per CU), for launches of at most one block
// per CU over a long contraction: a lone block waits out the latency of loads issued only
// one stage ahead. 3001x768x4096 41.6 -> 31.3 us, 4096x1024x768 12.5 -> 11.1; with an
// MN-major operand (bound by its transposing reads) 52 -> 52, over K = 384 5.6 -> 6.3, and
// with more tiles than CUs the second block is worth more (8192x1024x768 17.6 -> 19.4).
typedef DtlCfg<128, 128, 4, 2, false, 4> CfgDtlDeep;
inline bool deep_ring(int64_t M, int64_t N, int64_t K) {
  return ((M + 127) / 128) * ((N + 127) / 128) <= 256 && K >= 768;
}
// 256x256x64 tiles, 8 waves (128 KB of LDS, one block per CU): fewer LDS bytes per MFMA.
typedef DtlCfg<256, 256, 2, 4, true> CfgDtlBig;
// The small tile of a launch: 4 waves where both operands are K-major and one product fills
// the grid, 8 elsewhere (batches and ragged groups of few rows: 53 x 712x64x208 9.0 against
// 9.9 us, 8 groups of 53 rows over 248 6.6 against 7.2). A dense product fills it from 7/8
// of a round of two blocks per CU on: below, CUs hold one block, 4 or 8 waves of it. 4 against
// 8 waves, us: 259 tiles (4688x808x2032) 32.1 / 30.0, 384 (8192x768x7168) 101.9 / 99.7, 496
// (7912x968x1464) 32.9 / 34.0, 512 (8192x1024x3072) 52.7 / 53.4.
template <int MODE, bool AMN, bool BMN>
using CfgDtlSmall = std::conditional_t<AMN || BMN || MODE == MODE_BATCHED, CfgDtl, CfgDtlRA>;
inline bool dense_fills(int64_t M, int64_t N) { return ((M + 127) / 128) * ((N + 127) / 128) >= 448; }

// Whether an output takes `big` 256x256 tiles (one block per CU) rather than `small` 128x128
// ones (two per CU): by the rounds of 256 big or 512 small tiles, a partial round costing
// 0.8 + 0.2 of its fill. A round of small tiles is half the products of a round of big ones
// and costs `small_round` of it. Big against small, us: 192 big tiles
// (4096x3072x4096) 101 / 117, 384 (8192x3072x4864) 238 / 248, 512 (65536x512x512) 46 / 60,
// 256 (65536x256x512) 28 / 31; 128 (8192x1024x768) 21.7 / 17.6, 48 (768x4096x4096) 91 / 51.
inline bool big_rounds(int64_t big, int64_t small, double small_round) {
  auto rounds = [](int64_t tiles, int64_t cap) {  // in fifths
    const int64_t full = tiles / cap, rem = tiles % cap;
    return 5.0 * full + (rem ? 4.0 + (double)rem / cap : 0.0);
  };
  return rounds(big, 256) <= small_round * rounds(small, 512);
}
inline int64_t tiles_up(int64_t x, int64_t n) { return (x + n - 1) / n; }
// One product: 0.66 over a long contraction, 0.58 up to K = 1024, where a lone block's ramp
// (first loads, epilogue) has nothing beside it. Over 370 drawn products 1.5% slower than the
// better tile each time with 0.64 throughout, 0.6% with these.
inline bool big_tiles(int64_t rows, int64_t N, int64_t K) {
  return big_rounds(tiles_up(rows, 256) * tiles_up(N, 256), tiles_up(rows, 128) * tiles_up(N, 128),
                    K <= 1024 ? 0.58 : 0.66);
}
// Two-segment and grouped products run beside another stream's in the steps, where the small
// tile's waves cost more than alone: 65536x512x256 in 42 groups takes 39.6 against 41.5 us
// alone, yet the MoE step's forward products 1.65 against 1.59 ms.
constexpr double SHARED_ROUND = 0.64;
// J rows in E groups whose sizes only the device knows: the rows' tiles plus
// half a tile per group for the ragged ends, and at least one per group (of any size: small
// groups are what a big tile wastes most on). Big against small, us: 1352 rows in 128 groups
// over 440 (N = 528) 34 / 23, 560 in 128 over 96 (N = 1528) 29 / 21, 50664 in 32 over 144 (N =
// 1968) 81 / 92.
inline bool big_tiles_grouped(int64_t J, int64_t E, int64_t N, int64_t problems = 1) {
  const int64_t groups = E < J ? E : J;
  auto tiles = [&](int64_t t) {
    const int64_t rows = tiles_up(J + groups * (t / 2), t);
    return problems * (rows > groups ? rows : groups) * tiles_up(N, t);
  };
  return big_rounds(tiles(256), tiles(128), SHARED_ROUND);
}

// The kernel addresses each operand through a 31-bit buffer record count (rows = M or N
// for a K-major operand; for an MN-major one, K plus the 128 k-rows a last stage may
// reach past it).
inline bool dtl_fits(int64_t rows_a, int64_t lda, int64_t rows_b, int64_t ldb) {
  return rows_a * lda * 2 <= 0x7FFFFFFF && rows_b * ldb * 2 <= 0x7FFFFFFF;
}
inline bool dtl_fits_mn(int64_t K, int64_t ld) { return (K + 128) * ld * 2 <= 0x7FFFFFFF; }

// Record count (bytes) of a raw buffer descriptor, clamped to the 31-bit range (the
// launchers keep every operand below 2 GiB).
__device__ inline int32_t buf_bytes(int64_t bytes) {
  return bytes > 0x7FFFFFFF ? 0x7FFFFFFF : (bytes < 0 ? 0 : (int32_t)bytes);
}

// A wave's 1 KB loads of one operand tile: the lane's byte offset of load 0 relative to the
// tile's first row (K-major) or column (MN-major) at k = 0, and the step from load to load
// (one scalar: NW row blocks further, so the swizzle of the lane's chunk is the same).
// K-major: lane l fills physical chunk l % 8 of row l / 8 of the block, i.e. logical chunk
// (l % 8) ^ swz(row); the block of load q starts at row (q * NW + wave) * 8, so swz's
// parity bit is wave & 1 for every q. MN-major (R elements per k-row): load q covers k-rows
// (q * NW + wave) * RPL .. + RPL - 1; lane l fills physical chunk l % CPR of k-row l / CPR.
struct LaneOff {
  uint32_t off, step;
};
template <bool MN, int R, int NW>
__device__ inline LaneOff dtl_offsets(int64_t ld, int wave, int lane) {
  if constexpr (MN) {
    static_assert(R >= 128 && R <= 512, "an MN-major tile row is 256..1024 bytes");
    constexpr int CPR = R / 8, RPL = 1024 / (2 * R);
    static_assert(NW * RPL % 4 == 0, "the swizzle (k-row & 3) must not depend on the load index");
    const int row = wave * RPL + lane / CPR, c = (lane % CPR) ^ (4 * (row & 3));
    return {(uint32_t)((row * ld + c * 8) * 2), (uint32_t)uni((int)(NW * RPL * ld * 2))};
  } else {
    const int rsub = lane >> 3, c = (lane & 7) ^ rsub ^ (wave & 1);
    return {(uint32_t)(((wave * 8 + rsub) * ld + c * 8) * 2), (uint32_t)uni((int)(NW * 8 * ld * 2))};
  }
}

// LDS byte offset (within the operand's stage region, kk = 0, first half) of the
// transposing reads of fragment i of an MN-major tile of R elements per k-row; wave_r =
// the wave tile's first element within the block tile (a multiple of 32).
template <int R>
__device__ inline int mn_frag_off(int wave_r, int i, int lane) {
  constexpr int RB = 2 * R;
  const int g = lane >> 4, e = (lane >> 2) & 3, a = lane & 3;
  const int c = ((wave_r >> 3) + 4 * i) ^ (4 * e);
  return (8 * (g >> 1) + e) * RB + (c + 2 * (g & 1) + (a >> 1)) * 16 + (a & 1) * 8;
}

typedef short v4i16_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16_t* lds_v4i16_ptr;

// One fragment (rows lane & 31, k 8 (lane >> 5) .. + 7 of k16 step kk): MN: two transposing
// 8-byte reads; K-major: one 16-byte read at the lane's swizzled chunk coff.
template <bool MN, int R>
__device__ inline bf16x8 frag_load(const char* st, int off, int kk, int coff) {
  if constexpr (MN) {
    constexpr int RB = 2 * R;
    const char* q = st + off + kk * 16 * RB;
    const v4i16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(q));
    const v4i16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16_ptr)(q + 4 * RB));
    return bf16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  } else {
    return *(const bf16x8*)(st + off + coff);
  }
}

// A wave's fragment offsets within a stage (A region first, then B), per operand layout.
template <class CFG, bool AMN, bool BMN>
struct FragOffs {
  int a[CFG::TM], b[CFG::TN];
  int sw;
  __device__ inline FragOffs(int wm, int wn, int lane) {
    sw = dtl_swz(lane & 31);  // K-major fragment rows sit at multiples of 32 plus lane & 31
#pragma unroll
    for (int i = 0; i < CFG::TM; ++i)
      a[i] = AMN ? mn_frag_off<CFG::BM>(wm * CFG::WTM, i, lane) : (wm * CFG::WTM + i * 32 + (lane & 31)) * CFG::ROWB;
#pragma unroll
    for (int j = 0; j < CFG::TN; ++j)
      b[j] = CFG::BM * CFG::ROWB +
             (BMN ? mn_frag_off<CFG::BN>(wn * CFG::WTN, j, lane) : (wn * CFG::WTN + j * 32 + (lane & 31)) * CFG::ROWB);
  }
};

// Loads LO .. HI-1 of a stage of one operand at byte offset koff (the stage's k position)
// within each row. The descriptor spans [base, base + bytes) (stride 0); the whole offset
// goes in the per-lane register so the record-count check covers it (bytes = 0: zeros).
template <int NW, int LO, int HI>
__device__ inline void dtl_issue(char* dst, const bf16_t* base, int32_t bytes, LaneOff lo, uint32_t koff, int wave) {
  if constexpr (LO < HI) {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(base), (short)0, bytes, 0x00020000);
#pragma unroll
    for (int q = LO; q < HI; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void_t*)(dst + (q * NW + wave) * 8 * 128), 16,
                                               lo.off + (koff + q * lo.step), 0, 0, 0);
  }
}

// Loads LO .. HI-1 of a stage, counted over A's and then B's, into stage space st.
template <class CFG, int LO, int HI>
__device__ inline void dtl_issue_ab(char* st, const bf16_t* a, int32_t abytes, LaneOff offa, uint32_t ka,
                                    const bf16_t* b, int32_t bbytes, LaneOff offb, uint32_t kb, int wave) {
  constexpr int NA = CFG::A_INSTS;
  dtl_issue<CFG::NW, (LO < NA ? LO : NA), (HI < NA ? HI : NA)>(st, a, abytes, offa, ka, wave);
  dtl_issue<CFG::NW, (LO > NA ? LO - NA : 0), (HI > NA ? HI - NA : 0)>(st + CFG::BM * CFG::ROWB, b, bbytes, offb, kb, wave);
}

__device__ inline void mask_frag(bf16x8& v, int64_t k, int64_t kmin, int64_t kend) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (k + e < kmin || k + e >= kend) v[e] = 0;
}

template <typename TC>
__device__ inline void store4(TC* C, int64_t idx, const float* v, float alpha, float beta);
template <>
__device__ inline void store4<float>(float* C, int64_t idx, const float* v, float alpha, float beta) {
  float4 o = {alpha * v[0], alpha * v[1], alpha * v[2], alpha * v[3]};
  if (beta != 0.f) {
    const float4 c = *(const float4*)(C + idx);
    o.x += beta * c.x;
    o.y += beta * c.y;
    o.z += beta * c.z;
    o.w += beta * c.w;
  }
  *(float4*)(C + idx) = o;
}
template <>
__device__ inline void store4<bf16_t>(bf16_t* C, int64_t idx, const float* v, float alpha, float beta) {
  float o[4] = {alpha * v[0], alpha * v[1], alpha * v[2], alpha * v[3]};
  if (beta != 0.f) {
    const uint2 c = *(const uint2*)(C + idx);
    o[0] += beta * bf16_to_f32((bf16_t)(c.x & 0xFFFF));
    o[1] += beta * bf16_to_f32((bf16_t)(c.x >> 16));
    o[2] += beta * bf16_to_f32((bf16_t)(c.y & 0xFFFF));
    o[3] += beta * bf16_to_f32((bf16_t)(c.y >> 16));
  }
  uint2 w;
  w.x = pack_bf16x2(o[0], o[1]);
  w.y = pack_bf16x2(o[2], o[3]);
  *(uint2*)(C + idx) = w;
}

template <typename TC>
__device__ inline void store1(TC* C, int64_t idx, float v, float beta);
template <>
__device__ inline void store1<float>(float* C, int64_t idx, float v, float beta) {
  C[idx] = beta != 0.f ? v + beta * C[idx] : v;
}
template <>
__device__ inline void store1<bf16_t>(bf16_t* C, int64_t idx, float v, float beta) {
  C[idx] = f32_to_bf16(beta != 0.f ? v + beta * bf16_to_f32(C[idx]) : v);
}

// The fragments of one k16 step.
template <class CFG>
struct Frags {
  bf16x8 a[CFG::TM], b[CFG::TN];
};

template <class CFG, bool AMN, bool BMN>
__device__ inline void read_frags(const char* st, const FragOffs<CFG, AMN, BMN>& fo, int lane, int kk,
                                  Frags<CFG>& f) {
  const int coff = ((2 * kk + (lane >> 5)) ^ fo.sw) << 4;
#pragma unroll
  for (int j = 0; j < CFG::TN; ++j) f.b[j] = frag_load<BMN, CFG::BN>(st, fo.b[j], kk, coff);
#pragma unroll
  for (int i = 0; i < CFG::TM; ++i) f.a[i] = frag_load<AMN, CFG::BM>(st, fo.a[i], kk, coff);
}

// Zeroes the fragments' k outside [kmin, kend); k = the step's first.
template <class CFG>
__device__ inline void mask_frags(Frags<CFG>& f, int lane, int64_t k, int64_t kmin, int64_t kend) {
  const int64_t kf = k + (lane >> 5) * 8;
#pragma unroll
  for (int i = 0; i < CFG::TM; ++i) mask_frag(f.a[i], kf, kmin, kend);
#pragma unroll
  for (int j = 0; j < CFG::TN; ++j) mask_frag(f.b[j], kf, kmin, kend);
}

template <class CFG>
__device__ inline void dtl_mfma(const bf16x8 (&af)[CFG::TM], const bf16x8 (&bfr)[CFG::TN],
                                f32x16 (&acc)[CFG::TM][CFG::TN]) {
#pragma unroll
  for (int i = 0; i < CFG::TM; ++i)
#pragma unroll
    for (int j = 0; j < CFG::TN; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[j], af[i], acc[i][j], 0, 0, 0);
}

// Scheduling order of a step: after each of its MFMAS MFMAs, an equal share of its READS LDS
// reads (sched_group_barrier mask 0x100) and LOADS buffer loads (0x020).
template <int MFMAS, int READS, int LOADS>
__device__ inline void spread_step() {
#pragma unroll
  for (int m = 0; m < MFMAS; ++m) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if ((m + 1) * READS / MFMAS > m * READS / MFMAS)
      __builtin_amdgcn_sched_group_barrier(0x100, (READS + MFMAS - 1) / MFMAS, 0);
    if (LOADS > 0 && (m + 1) * LOADS / MFMAS > m * LOADS / MFMAS)
      __builtin_amdgcn_sched_group_barrier(0x020, (LOADS + MFMAS - 1) / MFMAS, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
}

// The stage's four k16 steps (see the top of this file). Before: f[0] holds the stage's
// step 0. read(kk, f): the stage's step kk; read_next(f): the next stage's step 0;
// issue(ahead, half): that half of the loads of the stage `ahead` stages
// on (NS stages, AHEAD loads of the later ones left in flight); mfma(kk, f):
// step kk's products. MFMAS, READS: a step's MFMAs and LDS reads; LOADS0, LOADS3: the loads issued in steps 0 and 3.
// LAST: the tile's last stage, after which nothing is loaded, read or waited for.
template <int MFMAS, int READS, int LOADS0, int LOADS3, int NS, int AHEAD, bool LAST, class F, class Read, class ReadNext,
          class Issue, class Mfma>
__device__ inline void pipe_stage(F (&f)[2], Read&& read, ReadNext&& read_next, Issue&& issue, Mfma&& mfma) {
  read(1, f[1]);
  if constexpr (!LAST) issue(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
  mfma(0, f[0]);
  spread_step<MFMAS, READS, LAST ? 0 : LOADS0>();
  read(2, f[0]);
  mfma(1, f[1]);
  spread_step<MFMAS, READS, 0>();
  read(3, f[1]);
  mfma(2, f[0]);
  spread_step<MFMAS, READS, 0>();
  if constexpr (LAST) {
    mfma(3, f[1]);
  } else {
    wait_loads_and_lds<AHEAD>();
    lds_barrier();
    read_next(f[0]);
    issue(std::integral_constant<int, NS>{}, std::integral_constant<int, 0>{});
    mfma(3, f[1]);
    spread_step<MFMAS, READS, LOADS3>();
  }
}

template <class CFG, typename TC>
__device__ inline void dtl_epilogue(const GemmArgs& p, const TileJob& t, int wm, int wn, int lane,
                                    f32x16 (&acc)[CFG::TM][CFG::TN]) {
  TC* C = (TC*)t.C;
  const bool vec = (p.ldc & 3) == 0 && ((uintptr_t)C & (4 * sizeof(TC) - 1)) == 0;
#pragma unroll
  for (int i = 0; i < CFG::TM; ++i) {
    const int64_t row = t.m0 + wm * CFG::WTM + i * 32 + (lane & 31);
    if (row >= t.M) continue;
#pragma unroll
    for (int j = 0; j < CFG::TN; ++j) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int64_t col = t.n0 + wn * CFG::WTN + j * 32 + 8 * g + 4 * (lane >> 5);
        const float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        if (vec && col + 3 < p.N) {
          store4<TC>(C, row * p.ldc + col, v, p.alpha, p.beta);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < p.N) store1<TC>(C, row * p.ldc + col + e, p.alpha * v[e], p.beta);
        }
      }
    }
  }
}

// A tile written through LDS: the accumulators go to a row-major LDS image (rows padded
// by 16 bytes, so the 32 rows one write instruction touches spread over the banks), then
// every lane stores 16 contiguous bytes and each instruction covers whole output rows.
// Straight from the MFMA layout a store instruction writes 16 (bf16) or 32 (fp32) bytes
// into each of 32 rows; through LDS the tile's 128-byte lines are written whole, which
// measured 13-25% faster on the grouped products with bf16 outputs. The image holds
// BM / PASSES rows at a time (the stage ring is the space); in pass q the waves whose
// rows fall in it write. Values are rounded as the register path rounds them: the bf16
// image holds round(alpha * acc) (so beta must be 0), the fp32 image alpha * acc, to
// which the store pass adds beta * C.
template <class CFG, int ES>
struct StagedStore {
  static constexpr int RSB = CFG::BN * ES + 16;  // LDS bytes per image row
  static constexpr int RING = CFG::NS * CFG::STAGE_BYTES;
  static constexpr int PASSES = CFG::BM * RSB <= RING           ? 1
                                : CFG::BM / 2 * RSB <= RING     ? 2
                                : CFG::BM / 4 * RSB <= RING     ? 4
                                                                : 0;
  static constexpr int ROWS = PASSES ? CFG::BM / PASSES : 0;
  static constexpr bool OK = PASSES > 0 && ROWS % CFG::WTM == 0;  // a wave's rows fall in one pass
};

// Pass q of the staged image: the waves whose rows fall in it write alpha * acc (bf16
// rounded for ES == 2) into the row-major LDS image; a barrier before (the k loop's last
// reads, or the previous pass's reads of the image, are done) and after (the image is
// complete).
template <class CFG, int ES>
__device__ inline void staged_image_pass(float alpha, int q, int wm, int wn, int lane,
                                         f32x16 (&acc)[CFG::TM][CFG::TN], char* smem) {
  typedef StagedStore<CFG, ES> SS;
  lds_write_barrier();
  const int r0 = wm * CFG::WTM - q * SS::ROWS;
  if (r0 >= 0 && r0 < SS::ROWS) {
#pragma unroll
    for (int i = 0; i < CFG::TM; ++i) {
      char* rowp = smem + (r0 + i * 32 + (lane & 31)) * SS::RSB;
#pragma unroll
      for (int j = 0; j < CFG::TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int c = wn * CFG::WTN + j * 32 + 8 * g + 4 * (lane >> 5);
          const float v0 = alpha * acc[i][j][4 * g], v1 = alpha * acc[i][j][4 * g + 1];
          const float v2 = alpha * acc[i][j][4 * g + 2], v3 = alpha * acc[i][j][4 * g + 3];
          if constexpr (ES == 2) {
            *(uint2*)(rowp + c * 2) = uint2{pack_bf16x2(v0, v1), pack_bf16x2(v2, v3)};
          } else {
            *(float4*)(rowp + c * 4) = float4{v0, v1, v2, v3};
          }
        }
    }
  }
  lds_write_barrier();
}

template <class CFG, typename TC>
__device__ inline void dtl_epilogue_staged(const GemmArgs& p, const TileJob& t, int wm, int wn, int tid,
                                           f32x16 (&acc)[CFG::TM][CFG::TN], char* smem) {
  constexpr int ES = sizeof(TC);
  typedef StagedStore<CFG, ES> SS;
  constexpr int EPC = 16 / ES;              // elements per 16-byte chunk
  constexpr int CPR = CFG::BN / EPC;        // chunks per output row
  constexpr int RPP = CFG::NT / CPR;        // rows one pass of the block's stores covers
  static_assert(CFG::NT % CPR == 0 && SS::ROWS % RPP == 0, "store passes");
  const int lane = tid & 63, rr = tid / CPR, cc = tid % CPR;
  TC* C = (TC*)t.C;
  const int64_t col = t.n0 + cc * EPC;
#pragma unroll
  for (int q = 0; q < SS::PASSES; ++q) {
    staged_image_pass<CFG, ES>(p.alpha, q, wm, wn, lane, acc, smem);
#pragma unroll
    for (int r = rr; r < SS::ROWS; r += RPP) {
      const int64_t row = t.m0 + q * SS::ROWS + r;
      if (row >= t.M || col >= p.N) continue;
      if constexpr (ES == 2) {
        *(uint4*)(C + row * p.ldc + col) = *(const uint4*)(smem + r * SS::RSB + cc * 16);
      } else {
        float4 o = *(const float4*)(smem + r * SS::RSB + cc * 16);
        if (p.beta != 0.f) {
          const float4 c = *(const float4*)(C + row * p.ldc + col);
          o.x += p.beta * c.x;
          o.y += p.beta * c.y;
          o.z += p.beta * c.z;
          o.w += p.beta * c.w;
        }
        *(float4*)(C + row * p.ldc + col) = o;
      }
    }
  }
}

// The epilogue is a policy: EPI::run(p, args, tile, wm, wn, tid, acc, smem) runs after the
// k loop with the LDS stage buffers still owned by the k loop (a policy that reuses
// them starts with a barrier); the block's LDS is max(stages, EPI::LDS_BYTES). EpiStore
// writes C = alpha * acc + beta * C: with 16-byte aligned rows and N a whole number of
// 16-byte chunks (and beta == 0 for a bf16 C) through the staged store, otherwise
// straight from the registers.
struct EpiStore {
  static constexpr int LDS_BYTES = 0;
  struct Args {};
  template <class CFG, typename TC>
  __device__ static void run(const GemmArgs& p, const Args&, const TileJob& t, int wm, int wn, int tid,
                             f32x16 (&acc)[CFG::TM][CFG::TN], char* smem) {
    constexpr int EPC = 16 / sizeof(TC);
    if constexpr (StagedStore<CFG, sizeof(TC)>::OK) {
      if ((sizeof(TC) == 4 || p.beta == 0.f) && p.ldc % EPC == 0 && p.N % EPC == 0 && ((uintptr_t)t.C & 15) == 0) {
        dtl_epilogue_staged<CFG, TC>(p, t, wm, wn, tid, acc, smem);
        return;
      }
    }
    dtl_epilogue<CFG, TC>(p, t, wm, wn, tid & 63, acc);
  }
};

// KEDGE: some stages cover k outside [kmin, kend) and are masked (ragged contraction
// groups, or K % 64 != 0). Only a tile's first and last stage can be such stages, so they
// are peeled off the main loop, which then has a single body: a branch between a masked
// and a plain stage inside the loop makes the compiler shuttle the accumulators between
// AGPRs and VGPRs on every iteration.
//
// AMN / BMN: A (or B) is MN-major, stored [K][M] (or [K][N]) with leading dimension lda
// (ldb) between k-rows.
template <class CFG, typename TC, int MODE, bool KEDGE, class EPI = EpiStore, bool AMN = false, bool BMN = false>
__global__ __launch_bounds__(CFG::NT) void k_gemm_dtl(GemmArgs p, typename EPI::Args ea) {
  constexpr int BM = CFG::BM, BN = CFG::BN, TM = CFG::TM, TN = CFG::TN, NW = CFG::NW;
  constexpr int BK = CFG::BK;
  constexpr int LDS = CFG::NS * CFG::STAGE_BYTES > EPI::LDS_BYTES ? CFG::NS * CFG::STAGE_BYTES : EPI::LDS_BYTES;
  __shared__ __attribute__((aligned(1024))) char smem[LDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int wm = wave / CFG::WN, wn = wave % CFG::WN;

  TileJob t;
  if (!map_tile<BM, BN, MODE, TC>(p, lane, t)) return;
  // every tile field is wave-uniform; say so, so the descriptors stay in scalar registers
  const int64_t m0 = uni64(t.m0), n0 = uni64(t.n0);
  const int64_t kmin = uni64(t.kbeg), kend = uni64(t.kend);
  const int64_t kbeg = kmin & ~(int64_t)63;
  const int64_t nk = kend > kmin ? (kend - kbeg + BK - 1) / BK : 0;
  // a K-major tile starts at its first row, an MN-major one at its first column; either
  // descriptor ends at the operand's end (rows past M / N, or k-rows past K, load zeros;
  // an MN-major tile's columns past M / N only feed outputs that are never stored)
  const bf16_t* abase = (const bf16_t*)uni64((int64_t)(AMN ? t.A + m0 : t.A + m0 * p.lda));
  const bf16_t* bbase = (const bf16_t*)uni64((int64_t)(BMN ? t.B + n0 : t.B + n0 * p.ldb));
  const int32_t abytes = buf_bytes(AMN ? (p.K * p.lda - m0) * 2 : (p.M - m0) * p.lda * 2);
  const int32_t bbytes = buf_bytes(BMN ? (p.K * p.ldb - n0) * 2 : (p.N - n0) * p.ldb * 2);
  const LaneOff offa = dtl_offsets<AMN, BM, NW>(p.lda, wave, lane), offb = dtl_offsets<BMN, BN, NW>(p.ldb, wave, lane);
  // a stage's k position as a byte offset: along the row (K-major) or down k-rows (MN)
  const uint32_t kstep_a = AMN ? (uint32_t)(p.lda * 2) : 2u, kstep_b = BMN ? (uint32_t)(p.ldb * 2) : 2u;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // half h of the loads of stage kt (none past the last stage: its descriptors are empty)
  auto issue = [&](int64_t kt, auto h) {
    constexpr int LO = decltype(h)::value ? CFG::HALF : 0, HI = decltype(h)::value ? CFG::INSTS : CFG::HALF;
    const uint32_t kpos = (uint32_t)(kbeg + kt * BK);
    const bool in = kt < nk;
    dtl_issue_ab<CFG, LO, HI>(smem + CFG::ring(kt) * CFG::STAGE_BYTES, abase, uni(in ? abytes : 0), offa,
                              kpos * kstep_a, bbase, uni(in ? bbytes : 0), offb, kpos * kstep_b, wave);
  };
#pragma unroll
  for (int st = 0; st < CFG::NS - 1; ++st) {
    issue(st, std::integral_constant<int, 0>{});
    issue(st, std::integral_constant<int, 1>{});
  }
  issue(CFG::NS - 1, std::integral_constant<int, 0>{});

  const FragOffs<CFG, AMN, BMN> fo(wm, wn, lane);
  Frags<CFG> f[2];
  wait_vmcnt<CFG::AHEAD + CFG::HALF>();
  lds_barrier();
  read_frags<CFG>(smem, fo, lane, 0, f[0]);
  constexpr int READS = TM * (AMN ? 2 : 1) + TN * (BMN ? 2 : 1);
  auto stage = [&](int64_t kt, auto edge, auto last) {
    const char* st = smem + CFG::ring(kt) * CFG::STAGE_BYTES;
    const char* nx = smem + CFG::ring(kt + 1) * CFG::STAGE_BYTES;
    pipe_stage<TM * TN, READS, CFG::INSTS - CFG::HALF, CFG::HALF, CFG::NS, CFG::AHEAD, decltype(last)::value>(
        f, [&](int kk, Frags<CFG>& g) { read_frags<CFG>(st, fo, lane, kk, g); },
        [&](Frags<CFG>& g) { read_frags<CFG>(nx, fo, lane, 0, g); },
        [&](auto ahead, auto h) { issue(kt + decltype(ahead)::value, h); },
        [&](int kk, Frags<CFG>& g) {
          if (decltype(edge)::value) mask_frags<CFG>(g, lane, kbeg + kt * BK + kk * 16, kmin, kend);
          dtl_mfma<CFG>(g.a, g.b, acc);
        });
  };
  if (KEDGE && nk > 1) stage(0, std::true_type{}, std::false_type{});
  for (int64_t kt = KEDGE; kt < nk - 1; ++kt) stage(kt, std::false_type{}, std::false_type{});
  if (nk > 0) stage(nk - 1, std::integral_constant<bool, KEDGE>{}, std::true_type{});
  wait_vmcnt<0>();  // the empty loads past the last stage still write their zeros
  EPI::template run<CFG, TC>(p, ea, t, wm, wn, tid, acc, smem);
}

// Two products of one shape in one block, P1 = A @ B^T and P2 = A2 @ B2^T (dense, every
// operand K-contiguous with the same lda / ldb), for epilogues that need both tiles of the
// same (row, column) block at once. EPI::run(p, ea, tile, wm, wn, tid, acc1, acc2, smem).
// SHARED_B (the caller guarantees B2 == B): one k loop, a stage holding A | B | A2, so B's
// rows and fragments are read once for both. Otherwise one k loop after the other through
// the same ring of A | B stages: both products side by side would need 128x128 tiles for
// their stages to fit (2048 x 16759 x 768 twice with the KL epilogue: 186 against 150 us;
// with two stages instead of three 167).
template <class CFG, bool KEDGE, class EPI, bool SHARED_B = false>
__global__ __launch_bounds__(CFG::NT) void k_gemm_dtl_dual(GemmArgs p, typename EPI::Args ea) {
  constexpr int BM = CFG::BM, BN = CFG::BN, TM = CFG::TM, TN = CFG::TN, NW = CFG::NW;
  constexpr int BK = CFG::BK, ROWB = CFG::ROWB;
  static_assert(CFG::HALF == CFG::INSTS && (!SHARED_B || CFG::NS == 2), "loads in one go; two stages of A | B | A2");
  constexpr int SB = (SHARED_B ? 2 * BM + BN : BM + BN) * ROWB, NS = CFG::NS;
  constexpr int LDS = NS * SB > EPI::template lds_bytes<CFG>() ? NS * SB : EPI::template lds_bytes<CFG>();
  static_assert(LDS <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) char smem[LDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int wm = wave / CFG::WN, wn = wave % CFG::WN;

  TileJob t;
  if (!map_tile<BM, BN, MODE_DENSE, float>(p, lane, t)) return;
  const int64_t m0 = uni64(t.m0), n0 = uni64(t.n0), K = p.K;
  const int64_t nk = (K + BK - 1) / BK;
  const bf16_t* abase = (const bf16_t*)uni64((int64_t)(p.A + m0 * p.lda));
  const bf16_t* a2base = (const bf16_t*)uni64((int64_t)(p.A2 + m0 * p.lda));
  const bf16_t* bbase = (const bf16_t*)uni64((int64_t)(p.B + n0 * p.ldb));
  const bf16_t* b2base = (const bf16_t*)uni64((int64_t)(p.B2 + n0 * p.ldb));
  const int32_t abytes = buf_bytes((p.M - m0) * p.lda * 2), bbytes = buf_bytes((p.N - n0) * p.ldb * 2);
  const LaneOff offa = dtl_offsets<false, BM, NW>(p.lda, wave, lane);
  const LaneOff offb = dtl_offsets<false, BN, NW>(p.ldb, wave, lane);

  f32x16 acc[TM][TN], acc2[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = acc2[i][j][v] = 0.f;
  const FragOffs<CFG, false, false> fo(wm, wn, lane);

  if constexpr (SHARED_B) {
    auto issue = [&](int64_t kt, auto h) {  // none past the last stage
      if (decltype(h)::value) return;
      char* st = smem + (int)(kt & 1) * SB;
      const uint32_t koff = (uint32_t)(kt * BK * 2);
      const int32_t ab = uni(kt < nk ? abytes : 0), bb = uni(kt < nk ? bbytes : 0);
      dtl_issue<NW, 0, CFG::A_INSTS>(st, abase, ab, offa, koff, wave);
      dtl_issue<NW, 0, CFG::B_INSTS>(st + BM * ROWB, bbase, bb, offb, koff, wave);
      dtl_issue<NW, 0, CFG::A_INSTS>(st + (BM + BN) * ROWB, a2base, ab, offa, koff, wave);
    };
    constexpr int LOADS = 2 * CFG::A_INSTS + CFG::B_INSTS;
    struct F2 {
      Frags<CFG> x;
      bf16x8 a2[TM];
    } f[2];
    auto read = [&](const char* st, int kk, F2& g) {
      read_frags<CFG>(st, fo, lane, kk, g.x);
      const int coff = ((2 * kk + (lane >> 5)) ^ fo.sw) << 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) g.a2[i] = frag_load<false, BM>(st, fo.a[i] + (BM + BN) * ROWB, kk, coff);
    };
    issue(0, std::integral_constant<int, 0>{});
    issue(1, std::integral_constant<int, 0>{});
    wait_vmcnt<LOADS>();
    lds_barrier();
    read(smem, 0, f[0]);
    auto stage = [&](int64_t kt, auto edge, auto last) {
      const char* st = smem + (int)(kt & 1) * SB;
      const char* nx = smem + (int)(~kt & 1) * SB;
      pipe_stage<2 * TM * TN, 2 * TM + TN, 0, LOADS, 2, 0, decltype(last)::value>(
          f, [&](int kk, F2& g) { read(st, kk, g); }, [&](F2& g) { read(nx, 0, g); },
          [&](auto ahead, auto h) { issue(kt + decltype(ahead)::value, h); },
          [&](int kk, F2& g) {
            if (decltype(edge)::value) {
              const int64_t kf = kt * BK + kk * 16;
              mask_frags<CFG>(g.x, lane, kf, 0, K);
#pragma unroll
              for (int i = 0; i < TM; ++i) mask_frag(g.a2[i], kf + (lane >> 5) * 8, 0, K);
            }
            dtl_mfma<CFG>(g.x.a, g.x.b, acc);
            dtl_mfma<CFG>(g.a2, g.x.b, acc2);
          });
    };
    for (int64_t kt = 0; kt < nk - 1; ++kt) stage(kt, std::false_type{}, std::false_type{});
    stage(nk - 1, std::integral_constant<bool, KEDGE>{}, std::true_type{});
  } else {
    auto issue = [&](int64_t kt, auto h) {  // stages nk .. 2 nk - 1 are the second product's
      if (decltype(h)::value) return;
      const bool s1 = kt < nk, in = kt < 2 * nk;
      const uint32_t koff = (uint32_t)((s1 ? kt : kt - nk) * BK * 2);
      dtl_issue_ab<CFG, 0, CFG::INSTS>(smem + CFG::ring(kt) * SB,
                                       (const bf16_t*)uni64((int64_t)(s1 ? abase : a2base)), uni(in ? abytes : 0), offa,
                                       koff, (const bf16_t*)uni64((int64_t)(s1 ? bbase : b2base)),
                                       uni(in ? bbytes : 0), offb, koff, wave);
    };
    Frags<CFG> f[2];
#pragma unroll
    for (int st = 0; st < NS; ++st) issue(st, std::integral_constant<int, 0>{});
    wait_vmcnt<CFG::AHEAD + CFG::INSTS>();
    lds_barrier();
    read_frags<CFG>(smem, fo, lane, 0, f[0]);
    auto stage = [&](int64_t kt, int64_t k0, auto edge, auto last, f32x16 (&ac)[TM][TN]) {
      const char* st = smem + CFG::ring(kt) * SB;
      const char* nx = smem + CFG::ring(kt + 1) * SB;
      pipe_stage<TM * TN, TM + TN, 0, CFG::INSTS, NS, CFG::AHEAD, decltype(last)::value>(
          f, [&](int kk, Frags<CFG>& g) { read_frags<CFG>(st, fo, lane, kk, g); },
          [&](Frags<CFG>& g) { read_frags<CFG>(nx, fo, lane, 0, g); },
          [&](auto ahead, auto h) { issue(kt + decltype(ahead)::value, h); },
          [&](int kk, Frags<CFG>& g) {
            if (decltype(edge)::value) mask_frags<CFG>(g, lane, k0 + kk * 16, 0, K);
            dtl_mfma<CFG>(g.a, g.b, ac);
          });
    };
    const std::false_type no{};
    for (int64_t kt = 0; kt < nk - KEDGE; ++kt) stage(kt, 0, no, no, acc);
    if constexpr (KEDGE) stage(nk - 1, (nk - 1) * BK, std::true_type{}, no, acc);
    for (int64_t kt = nk; kt < 2 * nk - 1; ++kt) stage(kt, 0, no, no, acc2);
    stage(2 * nk - 1, (nk - 1) * BK, std::integral_constant<bool, KEDGE>{}, std::true_type{}, acc2);
  }
  wait_vmcnt<0>();  // the empty loads past the last stage still write their zeros
  EPI::template run<CFG>(p, ea, t, wm, wn, tid, acc, acc2, smem);
}

// Two contractions into one accumulator, C = rs (.) (A1 @ op(B1)) + A2 @ op(B2): the
// k loop runs over A1's K1 columns, then A2's K2 (p.K), with rs, the per-row scale of
// the first product, applied to the accumulators in between. Every lane's 16 accumulators
// of a 32x32 MFMA tile sit in one output row, so the scale is one multiply per register.
// rs(t) = routed(t) ? (delta ? delta[t] : 0) : 1, routed(t) = !route || route[t] (delta
// bf16, or fp32 through delta_f): the
// blend weight of the target output x @ W^T in the masked linear (and of its cotangent).
// A1 and A2 are K-contiguous, K1 and K2 at least 1 (KEDGE: not both multiples of 64);
// B1MN / B2MN: the B operand is MN-major. The LDS stage ring
// runs straight through the segment boundary, so the second product's first stages
// load while the first product's last stage is consumed.
// MODE_GROUPED (job space of routed experts): rows are jobs sorted by expert, each B is an
// expert-major [E, N, K] stack (B1 advances by strideB1 per expert, B2 by p.strideB), an
// optional second problem of the same shape runs in the same launch (A1b, B1b with p.A2,
// p.B2, p.C2), and the row scale is per token, rs(row) = rs_tok[sort_idx[row] / k] (the
// second problem's from rs_tok2).
struct KcatArgs {
  const bf16_t* A1;
  int64_t lda1;
  const bf16_t* B1;
  int64_t ldb1;
  int64_t K1;
  const bf16_t* delta;
  const uint8_t* route;
  const bf16_t* A1b = nullptr;
  const bf16_t* B1b = nullptr;
  int64_t strideB1 = 0;
  const float* rs_tok = nullptr;
  const float* rs_tok2 = nullptr;
  const int32_t* sort_idx = nullptr;
  int k = 1;
  const float* delta_f = nullptr;  // fp32 per-row delta (dense mode; preferred over `delta`)
};

template <class CFG, typename TC, bool B1MN, bool B2MN, bool KEDGE, class EPI = EpiStore, int MODE = MODE_DENSE>
__global__ __launch_bounds__(CFG::NT) void k_gemm_dtl_kcat(GemmArgs p, KcatArgs q, typename EPI::Args ea) {
  constexpr int BM = CFG::BM, BN = CFG::BN, TM = CFG::TM, TN = CFG::TN, NW = CFG::NW;
  constexpr int BK = CFG::BK;
  constexpr int LDS = CFG::NS * CFG::STAGE_BYTES > EPI::LDS_BYTES ? CFG::NS * CFG::STAGE_BYTES : EPI::LDS_BYTES;
  __shared__ __attribute__((aligned(1024))) char smem[LDS];
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  const int wm = wave / CFG::WN, wn = wave % CFG::WN;

  TileJob t;
  if (!map_tile<BM, BN, MODE, TC>(p, lane, t)) return;
  const int64_t m0 = uni64(t.m0), n0 = uni64(t.n0);
  const int64_t K1 = q.K1, K2 = p.K;
  const int64_t nk1 = (K1 + BK - 1) / BK, nk = nk1 + (K2 + BK - 1) / BK;
  // the tile's segment-1 operands (its problem's, its expert's) and segment-2 operands
  // (map_tile placed t.A / t.B / t.C); selected by assignment, since a conditional over
  // the argument fields would take their address and move the arguments to scratch
  const bf16_t* A1 = q.A1;
  const bf16_t* B1 = q.B1;
  const float* rs_tok = q.rs_tok;
  if (t.prob) {
    A1 = q.A1b;
    B1 = q.B1b;
    rs_tok = q.rs_tok2;
  }
  B1 += (int64_t)t.e * q.strideB1;
  const bf16_t* a1 = (const bf16_t*)uni64((int64_t)(A1 + m0 * q.lda1));
  const bf16_t* b1 = (const bf16_t*)uni64((int64_t)(B1MN ? B1 + n0 : B1 + n0 * q.ldb1));
  const bf16_t* a2 = (const bf16_t*)uni64((int64_t)(t.A + m0 * p.lda));
  const bf16_t* b2 = (const bf16_t*)uni64((int64_t)(B2MN ? t.B + n0 : t.B + n0 * p.ldb));
  const int32_t a1bytes = buf_bytes((p.M - m0) * q.lda1 * 2), a2bytes = buf_bytes((p.M - m0) * p.lda * 2);
  const int32_t b1bytes = buf_bytes(B1MN ? (K1 * q.ldb1 - n0) * 2 : (p.N - n0) * q.ldb1 * 2);
  const int32_t b2bytes = buf_bytes(B2MN ? (K2 * p.ldb - n0) * 2 : (p.N - n0) * p.ldb * 2);
  const LaneOff oa1 = dtl_offsets<false, BM, NW>(q.lda1, wave, lane), ob1 = dtl_offsets<B1MN, BN, NW>(q.ldb1, wave, lane);
  const LaneOff oa2 = dtl_offsets<false, BM, NW>(p.lda, wave, lane), ob2 = dtl_offsets<B2MN, BN, NW>(p.ldb, wave, lane);
  const uint32_t ks1 = B1MN ? (uint32_t)(q.ldb1 * 2) : 2u, ks2 = B2MN ? (uint32_t)(p.ldb * 2) : 2u;

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // one issue path whose operands are selected value by value
  auto issue = [&](int64_t kt, auto h) {
    constexpr int LO = decltype(h)::value ? CFG::HALF : 0, HI = decltype(h)::value ? CFG::INSTS : CFG::HALF;
    const bool s1 = kt < nk1, in = kt < nk;
    const uint32_t kpos = (uint32_t)((s1 ? kt : kt - nk1) * BK);
    const LaneOff oa{s1 ? oa1.off : oa2.off, s1 ? oa1.step : oa2.step};
    const LaneOff ob{s1 ? ob1.off : ob2.off, s1 ? ob1.step : ob2.step};
    dtl_issue_ab<CFG, LO, HI>(smem + CFG::ring(kt) * CFG::STAGE_BYTES, (const bf16_t*)uni64((int64_t)(s1 ? a1 : a2)),
                              uni(in ? (s1 ? a1bytes : a2bytes) : 0), oa, kpos * 2,
                              (const bf16_t*)uni64((int64_t)(s1 ? b1 : b2)),
                              uni(in ? (s1 ? b1bytes : b2bytes) : 0), ob, kpos * (s1 ? ks1 : ks2), wave);
  };
#pragma unroll
  for (int st = 0; st < CFG::NS - 1; ++st) {
    issue(st, std::integral_constant<int, 0>{});
    issue(st, std::integral_constant<int, 1>{});
  }
  issue(CFG::NS - 1, std::integral_constant<int, 0>{});

  const FragOffs<CFG, false, B1MN> fo1(wm, wn, lane);
  const FragOffs<CFG, false, B2MN> fo2(wm, wn, lane);
  Frags<CFG> f[2];
  wait_vmcnt<CFG::AHEAD + CFG::HALF>();
  lds_barrier();
  read_frags<CFG>(smem, fo1, lane, 0, f[0]);
  // stage kt of a segment whose fragments sit at fo, the next stage's at fon; its k range
  // starts at k0 and ends at kend
  auto stage = [&](int64_t kt, const auto& fo, const auto& fon, int64_t k0, int64_t kend, auto edge, auto reads,
                   auto last) {
    const char* st = smem + CFG::ring(kt) * CFG::STAGE_BYTES;
    const char* nx = smem + CFG::ring(kt + 1) * CFG::STAGE_BYTES;
    pipe_stage<TM * TN, decltype(reads)::value, CFG::INSTS - CFG::HALF, CFG::HALF, CFG::NS, CFG::AHEAD,
               decltype(last)::value>(
        f, [&](int kk, Frags<CFG>& g) { read_frags<CFG>(st, fo, lane, kk, g); },
        [&](Frags<CFG>& g) { read_frags<CFG>(nx, fon, lane, 0, g); },
        [&](auto ahead, auto h) { issue(kt + decltype(ahead)::value, h); },
        [&](int kk, Frags<CFG>& g) {
          if (decltype(edge)::value) mask_frags<CFG>(g, lane, k0 + kk * 16, 0, kend);
          dtl_mfma<CFG>(g.a, g.b, acc);
        });
  };
  constexpr std::integral_constant<int, TM + TN * (B1MN ? 2 : 1)> r1{};
  constexpr std::integral_constant<int, TM + TN * (B2MN ? 2 : 1)> r2{};
  // segment 1; its last stage reads segment 2's first fragments (KEDGE: and masks its k tail)
  constexpr bool LAST1 = KEDGE || B1MN != B2MN;
  const std::false_type no{};
  for (int64_t kt = 0; kt < nk1 - LAST1; ++kt) stage(kt, fo1, fo1, kt * BK, K1, no, r1, no);
  if constexpr (LAST1) stage(nk1 - 1, fo1, fo2, (nk1 - 1) * BK, K1, std::integral_constant<bool, KEDGE>{}, r1, no);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t row = m0 + wm * CFG::WTM + i * 32 + (lane & 31);
    float rs = 1.f;
    if (rs_tok) rs = row < t.M ? rs_tok[q.sort_idx[row] / q.k] : 0.f;
    else if (row < p.M && (!q.route || q.route[row]))
      rs = q.delta_f ? q.delta_f[row] : (q.delta ? bf16_to_f32(q.delta[row]) : 0.f);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] *= rs;
  }
  // segment 2
  for (int64_t kt = nk1; kt < nk - 1; ++kt) stage(kt, fo2, fo2, (kt - nk1) * BK, K2, no, r2, no);
  stage(nk - 1, fo2, fo2, (nk - 1 - nk1) * BK, K2, std::integral_constant<bool, KEDGE>{}, r2, std::true_type{});
  wait_vmcnt<0>();  // the empty loads past the last stage still write their zeros
  EPI::template run<CFG, TC>(p, ea, t, wm, wn, tid, acc, smem);
}

template <class CFG, class EPI, typename TC, bool BMN>
inline void launch_epi_cfg(const GemmArgs& a, const typename EPI::Args& ea, hipStream_t s) {
  const dim3 grid((unsigned)((a.N + CFG::BN - 1) / CFG::BN), (unsigned)((a.M + CFG::BM - 1) / CFG::BM));
  if (a.K % CFG::BK)
    hipLaunchKernelGGL((k_gemm_dtl<CFG, TC, MODE_DENSE, true, EPI, false, BMN>), grid, dim3(CFG::NT), 0, s, a, ea);
  else
    hipLaunchKernelGGL((k_gemm_dtl<CFG, TC, MODE_DENSE, false, EPI, false, BMN>), grid, dim3(CFG::NT), 0, s, a, ea);
}

// Dense C = A [M, K] @ B^T (B stored [N, K], both K-contiguous, lda/ldb % 8 == 0, 16-byte
// aligned; BMN: B stored [K, N]) with the epilogue policy EPI (its Args carry everything
// beyond C's tile; EPI::BIG_OK: it takes 256x256 tiles too).
template <class EPI, typename TC, bool BMN = false>
inline int launch_dense_epi(const GemmArgs& a, const typename EPI::Args& ea, hipStream_t s, const char* what) {
  if (a.M * a.lda * 2 > 0x7FFFFFFF || !(BMN ? dtl_fits_mn(a.K, a.ldb) : a.N * a.ldb * 2 <= 0x7FFFFFFF))
    return fail(PD_EUNSUPPORTED, std::string(what) + ": operands of 2 GiB or more");
  if ((a.M + CfgDtl::BM - 1) / CfgDtl::BM > 65535 || (a.N + CfgDtl::BN - 1) / CfgDtl::BN > 65535)
    return fail(PD_EUNSUPPORTED, std::string(what) + ": too large");
  if (EPI::BIG_OK && big_tiles(a.M, a.N, a.K)) launch_epi_cfg<CfgDtlBig, EPI, TC, BMN>(a, ea, s);
  else if (!BMN && deep_ring(a.M, a.N, a.K)) launch_epi_cfg<CfgDtlDeep, EPI, TC, BMN>(a, ea, s);
  else launch_epi_cfg<CfgDtl, EPI, TC, BMN>(a, ea, s);
  return check_launch(what);
}

template <class CFG, class EPI, typename TC, bool B1MN, bool B2MN>
inline void launch_kcat_cfg(const GemmArgs& a, const KcatArgs& q, const typename EPI::Args& ea, hipStream_t s) {
  const dim3 grid((unsigned)((a.N + CFG::BN - 1) / CFG::BN), (unsigned)((a.M + CFG::BM - 1) / CFG::BM));
  if (a.K % CFG::BK || q.K1 % CFG::BK)
    hipLaunchKernelGGL((k_gemm_dtl_kcat<CFG, TC, B1MN, B2MN, true, EPI>), grid, dim3(CFG::NT), 0, s, a, q, ea);
  else
    hipLaunchKernelGGL((k_gemm_dtl_kcat<CFG, TC, B1MN, B2MN, false, EPI>), grid, dim3(CFG::NT), 0, s, a, q, ea);
}

// C = rs (.) (A1 @ op(B1)) + A2 @ op(B2) (k_gemm_dtl_kcat) with the epilogue policy EPI.
template <class EPI, typename TC, bool B1MN, bool B2MN>
inline int launch_kcat_epi(const GemmArgs& a, const KcatArgs& q, const typename EPI::Args& ea, hipStream_t s,
                           const char* what) {
  if (a.M * a.lda * 2 > 0x7FFFFFFF || a.M * q.lda1 * 2 > 0x7FFFFFFF ||
      !(B1MN ? dtl_fits_mn(q.K1, q.ldb1) : a.N * q.ldb1 * 2 <= 0x7FFFFFFF) ||
      !(B2MN ? dtl_fits_mn(a.K, a.ldb) : a.N * a.ldb * 2 <= 0x7FFFFFFF))
    return fail(PD_EUNSUPPORTED, std::string(what) + ": operands of 2 GiB or more");
  if ((a.M + CfgDtlRA::BM - 1) / CfgDtlRA::BM > 65535 || (a.N + CfgDtlRA::BN - 1) / CfgDtlRA::BN > 65535)
    return fail(PD_EUNSUPPORTED, std::string(what) + ": too large");
  if (big_rounds(tiles_up(a.M, 256) * tiles_up(a.N, 256), tiles_up(a.M, 128) * tiles_up(a.N, 128), SHARED_ROUND) &&
      EPI::LDS_BYTES <= 2 * CfgDtlBig::STAGE_BYTES)
    launch_kcat_cfg<CfgDtlBig, EPI, TC, B1MN, B2MN>(a, q, ea, s);
  else if (!B1MN && !B2MN && deep_ring(a.M, a.N, a.K + q.K1))
    launch_kcat_cfg<CfgDtlDeep, EPI, TC, B1MN, B2MN>(a, q, ea, s);
  else
    launch_kcat_cfg<CfgDtl, EPI, TC, B1MN, B2MN>(a, q, ea, s);
  return check_launch(what);
}

}  // namespace pd
