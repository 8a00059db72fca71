// GEMM kernels for the masked-component path (gfx950), v_mfma_f32_32x32x16_bf16.
//
// bf16 products run on the buffer-fed kernel of pd_gemm_dtl.hpp in every operand layout
// (an MN-contiguous operand is transposed on its way out of LDS): 128x128x64 tiles in 4 or
// 8 waves, two blocks per CU, or 256x256 tiles, one block per CU, by the rounds of each an
// output takes (`big_tiles`).
//
// Operands beyond the buffer kernel's 31-bit addressing: the register-staged kernel
// below. LDS holds both operands
// K-contiguous ([rows][BK+8]; the 144-byte row stride makes a wave's 16-byte fragment
// reads of 16 consecutive rows hit 16 distinct 4-bank groups); an operand whose global
// layout is MN-contiguous is transposed in registers (4 k-rows x 8 elements per thread)
// on its way into LDS. Two tile configurations:
//   BIG   256x256x64, 8 waves (2x4), 128x64 per wave (4x2 MFMA tiles), 144 KB LDS
//   SMALL 128x128x64, 4 waves (2x2), 64x64 per wave, for grids the big tile leaves
//         under-occupied (fewer than ~200 tiles on 256 CUs).
//
// Dense launches use an XCD-aware tile order: workgroups are dispatched round-robin
// over the 8 XCDs, so the linear id is remapped so each XCD's share is a compact
// 8-row-grouped region (fewer distinct A/B panels per XCD-local L2).
//
// Four problem mappings share the kernels:
//   DENSE     C = alpha*op(A)@op(B) + beta*C                  (x@V, acts@U, transposes)
//   GROUPED   out[rows_e] = lhs[rows_e] @ rhs[e], ragged rows  (pd/routed/experts.py:326-348)
//   GROUPED_K out[e] = lhs[rows_e]^T @ dout[rows_e]            (pd/routed/experts.py:209-280)
//   BATCHED   C[z] = op(A[z]) @ op(B[z]), per-operand strides  (per-block einsums,
//                                                              pd/core/linear_plan.py:149-160)
// Group offsets live on the device; blocks locate their group by scanning them, so no
// host synchronization is needed.
#include <algorithm>

#include "pd_gemm_dtl.hpp"

namespace pd {

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;

constexpr int BK = 64, LDS_PAD = 8, LDS_STRIDE = BK + LDS_PAD;

template <int BM_, int BN_, int WM_, int WN_>
struct TileCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int NT = WM_ * WN_ * 64;
  static constexpr int TM = BM_ / WM_ / 32, TN = BN_ / WN_ / 32;
  static constexpr int LDS_ELEMS = (BM_ + BN_) * LDS_STRIDE;
};
typedef TileCfg<256, 256, 2, 4> CfgBig;
typedef TileCfg<128, 128, 2, 2> CfgSmall;

// Loads one operand tile (ROWS x BK, rows = M or N index) into registers.
// KMAJ: global is [rows][K] (K contiguous): 16-byte chunks, 8 per row.
// !KMAJ: global is [K][rows] (rows contiguous): groups of 4 k-rows x 8 rows.
template <bool KMAJ, int ROWS, int NT>
struct TileLoader {
  static constexpr int NCH = KMAJ ? ROWS * BK / 8 / NT : (BK / 4) * (ROWS / 8) / NT;
  static constexpr int NV = KMAJ ? NCH : 4 * NCH;
  static_assert(NCH >= 1, "tile too small for the thread count");
  bf16x8 v[NV];
  // kmin: elements with k < kmin are zeroed (ragged-K groups whose tiles start at an
  // 8-aligned k below the group's first row); chunks are 8-aligned so loads stay 16 B.
  __device__ inline void load(const bf16_t* __restrict__ g, int64_t ld, int64_t row0, int64_t nrows, int64_t k0,
                              int64_t kmax, int tid, int64_t kmin = 0) {
    if (KMAJ) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        int id = tid + NT * i;
        int r = id >> 3, kc = id & 7;
        int64_t gr = row0 + r, gk = k0 + kc * 8;
        if (gr < nrows && gk < kmax) {
          v[i] = *(const bf16x8*)(g + gr * ld + gk);
          if (gk < kmin || gk + 8 > kmax) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
              if (gk + e < kmin || gk + e >= kmax) v[i][e] = 0;
          }
        } else {
          v[i] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        int id = tid + NT * i;
        int rc = id % (ROWS / 8), kg = id / (ROWS / 8);
        int64_t gr = row0 + rc * 8;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          int64_t gk = k0 + kg * 4 + q;
          if (gr < nrows && gk < kmax && gk >= kmin)
            v[4 * i + q] = *(const bf16x8*)(g + gk * ld + gr);
          else
            v[4 * i + q] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        }
      }
    }
  }
  __device__ inline void store(bf16_t* __restrict__ lds, int tid) {
    if (KMAJ) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        int id = tid + NT * i;
        int r = id >> 3, kc = id & 7;
        *(bf16x8*)(lds + r * LDS_STRIDE + kc * 8) = v[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        int id = tid + NT * i;
        int rc = id % (ROWS / 8), kg = id / (ROWS / 8);
        // v[4i+q][e]: k-row q, element e (row rc*8+e). Write row rc*8+e with its 4 k values.
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          bf16x4 w = {v[4 * i][e], v[4 * i + 1][e], v[4 * i + 2][e], v[4 * i + 3][e]};
          *(bf16x4*)(lds + (rc * 8 + e) * LDS_STRIDE + kg * 4) = w;
        }
      }
    }
  }
};

template <class CFG, bool A_KMAJ, bool B_KMAJ, typename TC, int MODE>
__global__ __launch_bounds__(CFG::NT) void k_gemm_bf16(GemmArgs p) {
  constexpr int BM = CFG::BM, BN = CFG::BN, NT = CFG::NT, TM = CFG::TM, TN = CFG::TN;
  constexpr int WTM = BM / CFG::WM, WTN = BN / CFG::WN;  // wave tile
  __shared__ __attribute__((aligned(16))) bf16_t lds[2][CFG::LDS_ELEMS];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / CFG::WN, wn = wave % CFG::WN;

  TileJob t;
  if (!map_tile<BM, BN, MODE, TC>(p, lane, t)) return;
  const int64_t M = t.M, N = p.N, m0 = t.m0, n0 = t.n0, kend = t.kend;
  int64_t kbeg = t.kbeg;
  const bf16_t* A = t.A;
  const bf16_t* B = t.B;
  TC* C = (TC*)t.C;

  TileLoader<A_KMAJ, BM, NT> la;
  TileLoader<B_KMAJ, BN, NT> lb;
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // K-major operands read 16-byte chunks, so a ragged group's K walk starts at the
  // 8-aligned k below its first row and the loaders zero k < kmin.
  const int64_t kmin = kbeg;
  if (MODE == MODE_GROUPED_K && (A_KMAJ || B_KMAJ)) kbeg &= ~(int64_t)7;
  const int64_t nk = (kend - kbeg + BK - 1) / BK;
  if (nk > 0) {
    la.load(A, p.lda, m0, M, kbeg, kend, tid, kmin);
    lb.load(B, p.ldb, n0, N, kbeg, kend, tid, kmin);
    la.store(lds[0], tid);
    lb.store(lds[0] + BM * LDS_STRIDE, tid);
    __syncthreads();
  }
  for (int64_t kt = 0; kt < nk; ++kt) {
    const int s = kt & 1;
    const bool more = kt + 1 < nk;
    if (more) {
      int64_t k0 = kbeg + (kt + 1) * BK;
      la.load(A, p.lda, m0, M, k0, kend, tid, kmin);
      lb.load(B, p.ldb, n0, N, k0, kend, tid, kmin);
    }
    const bf16_t* As = lds[s] + (wm * WTM + (lane & 31)) * LDS_STRIDE + (lane >> 5) * 8;
    const bf16_t* Bs = lds[s] + (BM + wn * WTN + (lane & 31)) * LDS_STRIDE + (lane >> 5) * 8;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 af[TM], bfr[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) af[i] = *(const bf16x8*)(As + i * 32 * LDS_STRIDE + kk * 16);
#pragma unroll
      for (int j = 0; j < TN; ++j) bfr[j] = *(const bf16x8*)(Bs + j * 32 * LDS_STRIDE + kk * 16);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
    if (more) {
      la.store(lds[s ^ 1], tid);
      lb.store(lds[s ^ 1] + BM * LDS_STRIDE, tid);
    }
    __syncthreads();
  }

  // epilogue: lane holds column (lane&31) and rows 8*(v/4) + 4*(lane>>5) + (v&3)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      int64_t col = n0 + wn * WTN + j * 32 + (lane & 31);
      if (col >= N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        int64_t row = m0 + wm * WTM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (row < M) store1<TC>(C, row * p.ldc + col, p.alpha * acc[i][j][v], p.beta);
      }
    }
}

// fp32 GEMM on the fp32 matrix cores (v_mfma_f32_32x32x2_f32), any operand layout;
// blockIdx.z = batch, each operand advancing by its own stride (0 = shared).
//
// Every wave computes a 32x32 output tile from 32x16 A and 16x32 B chunks it streams
// through a private LDS slice: coalesced loads along whichever dimension is contiguous,
// stored k-major so each MFMA operand read is one conflict-free float per lane; the next
// chunk's loads are in flight (registers) while the current chunk's MFMAs run. Two block
// forms of 4 waves:
//   KW > 1  one 32x32 tile per block of KW waves, the contraction cut into KW consecutive
//           k ranges (multiples of 16), the waves' partial tiles added in wave order
//           through LDS: for small outputs over long contractions (the toy targets' weight
//           gradients, e.g. 1000x100 over 2048 rows), which would otherwise leave most
//           CUs idle (KW = 8 from K = 1024 on, else 4);
//   KW = 1  a 64x64 tile per block of 4 waves, each one 32x32 quarter over the whole
//           contraction.
// Either way the summation order is fixed: results are deterministic, no workspace.
constexpr int FT = 32, FK = 16;
template <int KW, bool TA, bool TB>
__global__ __launch_bounds__(KW > 1 ? 64 * KW : 256) void k_gemm_f32(int64_t M, int64_t N, int64_t K, const float* __restrict__ A,
                                                  int64_t lda, const float* __restrict__ B, int64_t ldb,
                                                  float* __restrict__ C, int64_t ldc, float alpha, float beta,
                                                  int64_t sA, int64_t sB, int64_t sC) {
  constexpr bool SPLIT = KW > 1;
  constexpr int NWV = SPLIT ? KW : 4, NT = 64 * NWV;
  __shared__ float As[NWV][FK][FT], Bs[NWV][FK][FT];  // [wave][k][m or n]
  __shared__ float red[SPLIT ? KW : 1][SPLIT ? FT * FT : 1];
  A += (int64_t)blockIdx.z * sA;
  B += (int64_t)blockIdx.z * sB;
  C += (int64_t)blockIdx.z * sC;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int64_t bt = SPLIT ? FT : 2 * FT;
  const int64_t m0 = (int64_t)blockIdx.y * bt + (SPLIT ? 0 : (w >> 1) * FT);
  const int64_t n0 = (int64_t)blockIdx.x * bt + (SPLIT ? 0 : (w & 1) * FT);
  int64_t kb = 0, ke = K;
  if (SPLIT) {
    const int64_t kq = (K + KW * FK - 1) / (KW * FK) * FK;  // each wave's k range, a multiple of FK
    kb = (int64_t)w * kq;
    ke = kb + kq < K ? kb + kq : K;
  }
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  // a lane's 8 loads of a chunk: along k (K-contiguous rows: row l/2, k (l%2)*8 + e) or
  // along m / n (MN-contiguous k-rows: k l/4, column (l%4)*8 + e)
  const int r_k = lane >> 1, c_k = (lane & 1) * 8, r_mn = lane >> 2, c_mn = (lane & 3) * 8;
  float ra[8], rb[8];
  uint32_t okm = 0;  // bit e: ra[e] in range; bit 8 + e: rb[e]
  // out-of-range elements load the operand's first element (always valid) and are zeroed
  // when stored to LDS: no branches, and nothing waits for the loads until the next
  // chunk's stores, so all 16 loads are in flight during this chunk's MFMAs
  auto load = [&](int64_t k0) {
    okm = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int64_t off;
      bool ok;
      if constexpr (!TA) {  // A [M, K]
        const int64_t m = m0 + r_k, k = k0 + c_k + e;
        ok = m < M && k < ke;
        off = m * lda + k;
      } else {  // A [K, M]
        const int64_t k = k0 + r_mn, m = m0 + c_mn + e;
        ok = m < M && k < ke;
        off = k * lda + m;
      }
      ra[e] = A[ok ? off : 0];
      okm |= (uint32_t)ok << e;
      if constexpr (TB) {  // B [N, K]
        const int64_t n = n0 + r_k, k = k0 + c_k + e;
        ok = n < N && k < ke;
        off = n * ldb + k;
      } else {  // B [K, N]
        const int64_t k = k0 + r_mn, n = n0 + c_mn + e;
        ok = n < N && k < ke;
        off = k * ldb + n;
      }
      rb[e] = B[ok ? off : 0];
      okm |= (uint32_t)ok << (8 + e);
    }
  };
  if (kb < ke) load(kb);
  for (int64_t k0 = kb; k0 < ke; k0 += FK) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float av = (okm >> e) & 1u ? ra[e] : 0.f, bv = (okm >> (8 + e)) & 1u ? rb[e] : 0.f;
      if constexpr (!TA) As[w][c_k + e][r_k] = av;
      else As[w][r_mn][c_mn + e] = av;
      if constexpr (TB) Bs[w][c_k + e][r_k] = bv;
      else Bs[w][r_mn][c_mn + e] = bv;
    }
    if (k0 + FK < ke) load(k0 + FK);  // in flight during this chunk's MFMAs
    // the slice is this wave's alone: its LDS writes and reads stay in program order
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < FK; kk += 2)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[w][kk + (lane >> 5)][lane & 31], Bs[w][kk + (lane >> 5)][lane & 31],
                                                 acc, 0, 0, 0);
    asm volatile("" ::: "memory");
  }
  // lane holds column lane & 31, rows 8 (v / 4) + 4 (lane / 32) + v % 4 of its tile
  if constexpr (SPLIT) {
#pragma unroll
    for (int v = 0; v < 16; ++v) red[w][(8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * FT + (lane & 31)] = acc[v];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FT * FT / NT; ++q) {
      const int i = q * NT + tid, r = i / FT, c = i % FT;
      float sum = red[0][i];
#pragma unroll
      for (int x = 1; x < KW; ++x) sum += red[x][i];
      const int64_t gr = m0 + r, gc = n0 + c;
      if (gr < M && gc < N) C[gr * ldc + gc] = alpha * sum + (beta != 0.f ? beta * C[gr * ldc + gc] : 0.f);
    }
  } else {
    const int64_t gc = n0 + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t gr = m0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (gr < M && gc < N) C[gr * ldc + gc] = alpha * acc[v] + (beta != 0.f ? beta * C[gr * ldc + gc] : 0.f);
    }
  }
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// fp32 GEMM, direct form: the MFMA operands go from memory straight into registers, no
// LDS stage. Within each 16-k batch the two lane halves take different k: half h supplies
// k = kc + 8h + s on MFMA step s (the two k slots of v_mfma_f32_32x32x2_f32), so
//   an MN-contiguous operand is one coalesced dword per lane and step (32 consecutive
//     floats per half);
//   a K-contiguous operand is 8 consecutive floats per lane, loaded 4, 2 or 1 at a time
//     (`vec`: A's width + 16 times B's): as many as divide K, so that each run lies wholly
//     inside or outside the k range, and as every row's start is aligned to. Each such load
//     touches one cache line per lane, so it costs the same at any width.
// Every load goes through a buffer descriptor and is issued without a branch: an element
// outside the matrix or the wave's k range gets an offset past the descriptor's end, which
// the hardware returns as 0. Behind a branch the compiler has to assume that the loads were
// not issued and waits for every load in flight before each batch's MFMAs. F32_AHEAD batches
// are in flight: these launches hold one or two blocks per CU, so the load latency is what
// bounds them; a third batch was slower (104 registers against 75, so two blocks of 8 waves
// per CU against three): ResidualMLP step 222 against 210 us, 895x961x1521 with both
// transposed 81 against 76. A contraction of one or two batches per wave issues just those:
// loads past its range cost the address unit as much as data.
// Block forms as in k_gemm_f32 (KW waves splitting the contraction of a 32x32 tile, or 4
// waves of a 64x64 tile); the summation order is fixed. Each operand must span fewer than
// 2^31 bytes (checked on the host). 2048x1000 over 50, both K-contiguous at row stride 50,
// 17.6 us in dword loads (and a 3.6 us copy before it), 14.5 in 8-byte loads; the whole
// residual-MLP step 296 -> 210 us with the grouped launches below.
constexpr int F32_AHEAD = 2;

template <int KW, bool TA, bool TB>
__device__ inline void f32_direct_tile(const F32Prod& p, int bm, int bn, int kbeg, int kend, int32_t bytes_a,
                                       int32_t bytes_b, int vec, float alpha, float beta, float (*red)[FT * FT]) {
  constexpr bool SPLIT = KW > 1;
  constexpr int NWV = SPLIT ? KW : 4, NT = 64 * NWV, S = 8, D = F32_AHEAD;
  const float *A = p.A, *B = p.B, *Cin = p.Cin;
  float* C = p.C;
  const int64_t M = p.M, N = p.N, ldc = p.ldc;
  // the wave index as a scalar, so that a batch's position is one and each load's offset is
  // one lane register plus a scalar
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5;
  const int64_t bt = SPLIT ? FT : 2 * FT;
  const int64_t m0 = bm * bt + (SPLIT ? 0 : (w >> 1) * FT);
  const int64_t n0 = bn * bt + (SPLIT ? 0 : (w & 1) * FT);
  int kb = kbeg, ke = kend;
  if (SPLIT) {
    const int kq = (kend - kbeg + KW * FK - 1) / (KW * FK) * FK;
    kb = kbeg + w * kq;
    ke = kb + kq < ke ? kb + kq : ke;
  }
  const uint32_t m = (uint32_t)(m0 + (lane & 31)), n = (uint32_t)(n0 + (lane & 31));
  const uint32_t sta = TA ? (uint32_t)p.lda : 1u, stb = TB ? 1u : (uint32_t)p.ldb;  // elements from k to k + 1
  const auto rsa = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), (short)0, bytes_a, 0x00020000);
  const auto rsb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), (short)0, bytes_b, 0x00020000);
  // byte offset of the lane's element at k = 8h, and 8h itself: past any range for a row
  // outside the matrix
  const uint32_t oa = ((TA ? m : m * (uint32_t)p.lda) + h * S * sta) * 4u;
  const uint32_t ob = ((TB ? n * (uint32_t)p.ldb : n) + h * S * stb) * 4u;
  const int ha = m < M ? h * S : INT32_MAX, hb = n < N ? h * S : INT32_MAX;
  // offsets of in-range elements are < 2^31; 2^31 is past every descriptor's end
  auto load1 = [&](auto width, float (&x)[S], const auto& rs, uint32_t o, uint32_t st, int hs, int kc) {
    constexpr int W = decltype(width)::value;
#pragma unroll
    for (int s = 0; s < S; s += W) {
      const uint32_t off = hs < ke - kc - s ? o + (uint32_t)(kc + s) * st * 4u : 1u << 31;
      if constexpr (W == 1) {
        x[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
      } else {
        uint32_t u[W];  // a bit cast of a vector's element itself reads element 0
        if constexpr (W == 2) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
          u[0] = v[0], u[1] = v[1];
        } else {
          const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
          u[0] = v[0], u[1] = v[1], u[2] = v[2], u[3] = v[3];
        }
#pragma unroll
        for (int e = 0; e < W; ++e) x[s + e] = __builtin_bit_cast(float, u[e]);
      }
    }
  };
  auto load = [&](auto wa, auto wb, float (&a)[S], float (&b)[S], int kc) {
    load1(wa, a, rsa, oa, sta, ha, kc);
    load1(wb, b, rsb, ob, stb, hb, kc);
  };
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  auto contract = [&](auto wa, auto wb) {
    float a[D][S], b[D][S];
    auto mfma = [&](int d) {
#pragma unroll
      for (int s = 0; s < S; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[d][s], b[d][s], acc, 0, 0, 0);
    };
    if (ke - kb <= 2 * FK) {  // at most two batches: both in flight, none past the range
      if (kb >= ke) return;
      load(wa, wb, a[0], b[0], kb);
      if (ke - kb > FK) load(wa, wb, a[1], b[1], kb + FK);
      mfma(0);
      if (ke - kb > FK) mfma(1);
      return;
    }
#pragma unroll
    for (int d = 0; d < D; ++d) load(wa, wb, a[d], b[d], kb + d * FK);
    int kc = kb;
    for (; kc + D * FK < ke; kc += D * FK) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        mfma(d);
        load(wa, wb, a[d], b[d], kc + (d + D) * FK);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (kc + d * FK >= ke) return;
      mfma(d);
    }
  };
  typedef std::integral_constant<int, 1> W1;
  typedef std::integral_constant<int, 2> W2;
  typedef std::integral_constant<int, 4> W4;
  auto with_b = [&](auto wa) {
    if constexpr (TB) {
      if ((vec >> 4) == 4) return contract(wa, W4{});
      if ((vec >> 4) == 2) return contract(wa, W2{});
    }
    contract(wa, W1{});
  };
  const int va = vec & 15;
  if (TA || va == 1) with_b(W1{});
  else if (va == 4) with_b(W4{});
  else with_b(W2{});
  auto put = [&](int64_t gr, int64_t gc, float sum) {
    const int64_t i = gr * ldc + gc;
    float v = alpha * sum + (beta != 0.f ? beta * Cin[i] : 0.f);
    if (p.post == 1) v = fmaxf(v, 0.f);
    else if (p.post == 2) v = Cin[i] > 0.f ? v : 0.f;
    C[i] = v;
  };
  // lane holds column lane & 31, rows 8 (v / 4) + 4 (lane / 32) + v % 4 of its tile
  if constexpr (SPLIT) {
#pragma unroll
    for (int v = 0; v < 16; ++v) red[w][(8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * FT + (lane & 31)] = acc[v];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < FT * FT / NT; ++q) {
      const int i = q * NT + tid, r = i / FT, c = i % FT;
      float sum = red[0][i];
#pragma unroll
      for (int x = 1; x < KW; ++x) sum += red[x][i];
      const int64_t gr = m0 + r, gc = n0 + c;
      if (gr < M && gc < N) put(gr, gc, sum);
    }
  } else {
    const int64_t gc = n0 + (lane & 31);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int64_t gr = m0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
      if (gr < M && gc < N) put(gr, gc, acc[v]);
    }
  }
}

template <int KW, bool TA, bool TB>
__global__ __launch_bounds__(KW > 1 ? 64 * KW : 256, KW > 1 ? 4 : 3) void k_gemm_f32_direct(F32Prod p, float alpha, float beta,
                                                                           int64_t sA, int64_t sB, int64_t sC,
                                                                           int32_t bytes_a, int32_t bytes_b, int vec) {
  __shared__ float red[KW > 1 ? KW : 1][KW > 1 ? FT * FT : 1];
  p.A += (int64_t)blockIdx.z * sA;
  p.B += (int64_t)blockIdx.z * sB;
  p.C += (int64_t)blockIdx.z * sC;
  p.Cin += (int64_t)blockIdx.z * sC;
  f32_direct_tile<KW, TA, TB>(p, (int)blockIdx.y, (int)blockIdx.x, 0, (int)p.K, bytes_a, bytes_b, vec, alpha, beta,
                              (float(*)[FT * FT])red);
}

struct F32Group {
  F32Prod p[F32_GROUP];
  int32_t bytes_a[F32_GROUP], bytes_b[F32_GROUP], vec[F32_GROUP], tiles_n[F32_GROUP], first[F32_GROUP + 1];
  int32_t n, splits;
};

// Several small products in one launch: a block of KW waves takes one 32x32 tile of one
// product, or one contraction slice of it.
template <int KW, bool TA>
__global__ __launch_bounds__(64 * KW) void k_gemm_f32_group(F32Group g) {
  __shared__ float red[KW][FT * FT];
  int i = 0;
  while (i + 1 < g.n && (int)blockIdx.x >= g.first[i + 1]) ++i;
  F32Prod p = g.p[i];
  const int u = (int)blockIdx.x - g.first[i], t = u / g.splits, sl = u % g.splits;
  const int K = (int)p.K, kq = (K + g.splits * FK - 1) / (g.splits * FK) * FK;
  const int kb = sl * kq, ke = kb + kq < K ? kb + kq : K;  // kb >= ke: a slab of zeros
  p.C += (int64_t)sl * p.M * p.N;
  const int bm = t / g.tiles_n[i], bn = t % g.tiles_n[i];
  const float beta = p.Cin && p.post < 2 ? 1.f : 0.f;
  if (p.tb) f32_direct_tile<KW, TA, true>(p, bm, bn, kb, ke, g.bytes_a[i], g.bytes_b[i], g.vec[i], 1.f, beta, red);
  else f32_direct_tile<KW, TA, false>(p, bm, bn, kb, ke, g.bytes_a[i], g.bytes_b[i], g.vec[i], 1.f, beta, red);
}

// Bytes the operands span (>= 0), and the floats per load of each (`vec` of f32_direct_tile).
struct F32Span {
  int64_t a, b;
  int vec;
  bool fits;
};
static F32Span f32_span(const F32Prod& p, int64_t sA = 0, int64_t sB = 0) {
  // no contraction reads nothing: the last-row formulas would be negative at K = 0 where a
  // k-row is padded, and a negative record count is one past 2^31, inside which the loads'
  // out-of-range offset lies
  const int64_t ea = p.K == 0 ? 0 : 4 * (p.ta ? (p.K - 1) * p.lda + p.M : (p.M - 1) * p.lda + p.K);
  const int64_t eb = p.K == 0 ? 0 : 4 * (p.tb ? (p.N - 1) * p.ldb + p.K : (p.K - 1) * p.ldb + p.N);
  auto width = [&](const float* x, int64_t ld, int64_t stride) {
    auto by = [&](int w) { return p.K % w == 0 && ld % w == 0 && stride % w == 0 && (uintptr_t)x % (4 * w) == 0; };
    return by(4) ? 4 : by(2) ? 2 : 1;
  };
  const int vec = (p.ta ? 1 : width(p.A, p.lda, sA)) | (p.tb ? width(p.B, p.ldb, sB) : 1) << 4;
  return {ea, eb, vec, ea < (int64_t(1) << 31) && eb < (int64_t(1) << 31)};
}

// The fp32 block form. Whole-contraction 64x64 tiles once they alone give >= 512 blocks
// (direct form up to K = 256, the LDS-staged one beyond), else 32x32 tiles with the
// contraction split over waves: the direct form with 16 waves from K = 512 on, else 8.
// The LDS-staged form also serves operands of 2^31 bytes or more.
static bool f32_big(int64_t M, int64_t N, int64_t batch) { return cdiv(M, 2 * FT) * cdiv(N, 2 * FT) * batch >= 512; }

template <bool TA, bool TB>
static bool launch_f32_direct(const F32Prod& p, int64_t batch, float alpha, float beta, int64_t sA, int64_t sB,
                              int64_t sC, hipStream_t s) {
  const F32Span sp = f32_span(p, sA, sB);
  const bool big = f32_big(p.M, p.N, batch);
  if (!sp.fits || (big && p.K > 256)) return false;
  const int64_t t = big ? 2 * FT : FT;
  const dim3 grid((unsigned)cdiv(p.N, t), (unsigned)cdiv(p.M, t), (unsigned)batch);
#define PD_FD(KW_)                                                                                                   \
  hipLaunchKernelGGL((k_gemm_f32_direct<KW_, TA, TB>), grid, dim3(KW_ > 1 ? 64 * KW_ : 256), 0, s, p, alpha, beta, sA, \
                     sB, sC, (int32_t)sp.a, (int32_t)sp.b, sp.vec)
  if (big) PD_FD(1);
  else if (p.K >= 512) PD_FD(16);
  else PD_FD(8);
#undef PD_FD
  return true;
}

template <bool TA, bool TB>
static void launch_gemm_f32_l(int64_t batch, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                              const float* B, int64_t ldb, float* C, int64_t ldc, float alpha, float beta, int64_t sA,
                              int64_t sB, int64_t sC, hipStream_t s) {
  const F32Prod p{M, N, K, A, lda, TA, B, ldb, TB, C, ldc, C, 0};
  if (launch_f32_direct<TA, TB>(p, batch, alpha, beta, sA, sB, sC, s)) return;
  const dim3 g32((unsigned)cdiv(N, FT), (unsigned)cdiv(M, FT), (unsigned)batch);
  const dim3 g64((unsigned)cdiv(N, 2 * FT), (unsigned)cdiv(M, 2 * FT), (unsigned)batch);
  if (f32_big(M, N, batch))
    hipLaunchKernelGGL((k_gemm_f32<1, TA, TB>), g64, dim3(256), 0, s, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA,
                       sB, sC);
  else if (K >= 1024)
    hipLaunchKernelGGL((k_gemm_f32<8, TA, TB>), g32, dim3(512), 0, s, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA,
                       sB, sC);
  else
    hipLaunchKernelGGL((k_gemm_f32<4, TA, TB>), g32, dim3(256), 0, s, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA,
                       sB, sC);
}

static void launch_gemm_f32(int64_t batch, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda, int ta,
                            const float* B, int64_t ldb, int tb, float* C, int64_t ldc, float alpha, float beta,
                            int64_t sA, int64_t sB, int64_t sC, hipStream_t s) {
  if (ta && tb) launch_gemm_f32_l<true, true>(batch, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA, sB, sC, s);
  else if (ta) launch_gemm_f32_l<true, false>(batch, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA, sB, sC, s);
  else if (tb) launch_gemm_f32_l<false, true>(batch, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA, sB, sC, s);
  else launch_gemm_f32_l<false, false>(batch, M, N, K, A, lda, B, ldb, C, ldc, alpha, beta, sA, sB, sC, s);
}

bool gemm_f32_direct(const F32Prod& p, hipStream_t s) {
  if (cdiv(p.M, FT) > 65535 || cdiv(p.N, FT) > 65535) return false;  // pd_gemm refuses it
  const float beta = p.Cin && p.post < 2 ? 1.f : 0.f;
  if (p.ta) return p.tb ? launch_f32_direct<true, true>(p, 1, 1.f, beta, 0, 0, 0, s)
                        : launch_f32_direct<true, false>(p, 1, 1.f, beta, 0, 0, 0, s);
  return p.tb ? launch_f32_direct<false, true>(p, 1, 1.f, beta, 0, 0, 0, s)
              : launch_f32_direct<false, false>(p, 1, 1.f, beta, 0, 0, 0, s);
}

bool gemm_f32_group(const F32Prod* p, int n, int splits, hipStream_t s) {
  F32Group g{};
  g.n = n;
  g.splits = splits;
  int64_t blocks = 0;
  for (int i = 0; i < n; ++i) {
    const F32Span sp = f32_span(p[i]);
    if (!sp.fits || p[i].ta != p[0].ta) return false;
    g.p[i] = p[i];
    g.bytes_a[i] = (int32_t)sp.a;
    g.bytes_b[i] = (int32_t)sp.b;
    g.vec[i] = sp.vec;
    g.tiles_n[i] = (int32_t)cdiv(p[i].N, FT);
    g.first[i] = (int32_t)blocks;
    blocks += cdiv(p[i].M, FT) * g.tiles_n[i] * splits;
    if (blocks >= (int64_t(1) << 31)) return false;
  }
  g.first[n] = (int32_t)blocks;
  // partial sums at most as long as the single products': 16 waves over a long contraction,
  // 8 over the slices of a transposed A's
#define PD_FG(KW_, TA_) hipLaunchKernelGGL((k_gemm_f32_group<KW_, TA_>), dim3((unsigned)blocks), dim3(64 * KW_), 0, s, g)
  if (p[0].ta) PD_FG(8, true);
  else if (p[0].K >= 512) PD_FG(16, false);
  else PD_FG(8, false);
#undef PD_FG
  return true;
}

__global__ void k_zero_tail_rows(const int32_t* __restrict__ offsets, int E, int64_t J, int64_t width, int out_bytes,
                                 void* __restrict__ out) {
  int64_t start = offsets[E];
  if (start < 0) start = 0;
  int64_t n = (J - start) * width;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    if (out_bytes == 4)
      ((float*)out)[start * width + i] = 0.f;
    else
      ((bf16_t*)out)[start * width + i] = 0;
  }
}

template <class CFG, int MODE>
static int launch_bf16(const GemmArgs& a, bool a_kmaj, bool b_kmaj, int c_dtype, dim3 grid, hipStream_t s) {
#define PD_L(AK, BKM, TC) \
  hipLaunchKernelGGL((k_gemm_bf16<CFG, AK, BKM, TC, MODE>), grid, dim3(CFG::NT), 0, s, a)
  if (c_dtype == PD_DTYPE_F32) {
    if (a_kmaj && b_kmaj) PD_L(true, true, float);
    else if (a_kmaj) PD_L(true, false, float);
    else if (b_kmaj) PD_L(false, true, float);
    else PD_L(false, false, float);
  } else {
    if (a_kmaj && b_kmaj) PD_L(true, true, bf16_t);
    else if (a_kmaj) PD_L(true, false, bf16_t);
    else if (b_kmaj) PD_L(false, true, bf16_t);
    else PD_L(false, false, bf16_t);
  }
#undef PD_L
  return check_launch("pd_gemm bf16");
}

// host-side validation of a bf16 operand: contiguous dim a multiple of 8 elements,
// leading dim a multiple of 8, 16-byte aligned base.
static bool bf16_operand_ok(const void* ptr, int64_t ld, int64_t contig_extent) {
  return aligned16(ptr) && ld % 8 == 0 && contig_extent % 8 == 0;
}

// The big tile needs enough tiles to occupy the 256 CUs; otherwise use the small one.
static bool use_big_tile(int64_t M, int64_t N) { return cdiv(M, 256) * cdiv(N, 256) >= 192; }

template <class CFG, int MODE, bool AMN = false, bool BMN = false>
static int launch_dtl(const GemmArgs& a, int c_dtype, bool kedge, dim3 grid, hipStream_t s) {
#define PD_L(TC, KE) \
  hipLaunchKernelGGL((k_gemm_dtl<CFG, TC, MODE, KE, EpiStore, AMN, BMN>), grid, dim3(CFG::NT), 0, s, a, EpiStore::Args{})
  if (c_dtype == PD_DTYPE_F32) {
    if (kedge) PD_L(float, true);
    else PD_L(float, false);
  } else {
    if (kedge) PD_L(bf16_t, true);
    else PD_L(bf16_t, false);
  }
#undef PD_L
  return check_launch("pd_gemm bf16 (buffer-fed)");
}

// Any operand layout through the buffer-fed kernel (a_kmaj / b_kmaj: K-contiguous), in 256x256
// (`big`) or 128x128 tiles.
template <int MODE, bool BIG_OK>
static int launch_dtl_any(const GemmArgs& a, bool a_kmaj, bool b_kmaj, int c_dtype, bool kedge, bool big,
                          unsigned batch, hipStream_t s) {
  const int64_t t = BIG_OK && big ? 256 : 128;
  const dim3 grid((unsigned)cdiv(a.N, t), (unsigned)cdiv(a.M, t), batch);
#define PD_L(AMN, BMN)                                                                              \
  {                                                                                                 \
    if constexpr (BIG_OK)                                                                           \
      if (big) return launch_dtl<CfgDtlBig, MODE, AMN, BMN>(a, c_dtype, kedge, grid, s);            \
    if constexpr (MODE == MODE_DENSE && !(AMN) && !(BMN)) {                                         \
      if (deep_ring(a.M, a.N, a.K)) return launch_dtl<CfgDtlDeep, MODE>(a, c_dtype, kedge, grid, s); \
      if (!dense_fills(a.M, a.N)) return launch_dtl<CfgDtl, MODE>(a, c_dtype, kedge, grid, s);      \
    }                                                                                               \
    return launch_dtl<CfgDtlSmall<MODE, AMN, BMN>, MODE, AMN, BMN>(a, c_dtype, kedge, grid, s);     \
  }
  if (a_kmaj && b_kmaj) PD_L(false, false)
  if (a_kmaj) PD_L(false, true)
  if (b_kmaj) PD_L(true, false)
  PD_L(true, true)
#undef PD_L
}

// Every operand of the buffer-fed kernel within its 31-bit addressing range.
static bool dtl_fits_any(int64_t M, int64_t N, int64_t K, int64_t lda, bool a_kmaj, int64_t ldb, bool b_kmaj) {
  return (a_kmaj ? M * lda * 2 <= 0x7FFFFFFF : dtl_fits_mn(K, lda)) &&
         (b_kmaj ? N * ldb * 2 <= 0x7FFFFFFF : dtl_fits_mn(K, ldb));
}

}  // namespace pd

using namespace pd;

extern "C" {

int pd_gemm(int dtype, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, int trans_a, const void* B,
            int64_t ldb, int trans_b, void* C, int64_t ldc, int c_dtype, float alpha, float beta, void* stream) {
  if (M < 0 || N < 0 || K < 0 || !A || !B || !C) return fail(PD_EINVAL, "pd_gemm: bad args");
  if (M == 0 || N == 0) return PD_OK;
  hipStream_t s = (hipStream_t)stream;
  if (cdiv(M, FT) > 65535 || cdiv(N, FT) > 65535) return fail(PD_EUNSUPPORTED, "pd_gemm: too large");
  if (dtype == PD_DTYPE_F32) {
    if (c_dtype != PD_DTYPE_F32) return fail(PD_EINVAL, "pd_gemm: fp32 path writes fp32");
    launch_gemm_f32(1, M, N, K, (const float*)A, lda, trans_a, (const float*)B, ldb, trans_b, (float*)C, ldc, alpha,
                    beta, 0, 0, 0, s);
    return check_launch("pd_gemm f32");
  }
  if (dtype != PD_DTYPE_BF16) return fail(PD_EINVAL, "pd_gemm: dtype");
  bool a_kmaj = !trans_a, b_kmaj = trans_b;
  if (!bf16_operand_ok(A, lda, a_kmaj ? K : M) || !bf16_operand_ok(B, ldb, b_kmaj ? K : N))
    return fail(PD_EUNSUPPORTED, "pd_gemm: bf16 operands need 16B alignment and contiguous dims / ld % 8 == 0");
  GemmArgs a{M, N, K, (const bf16_t*)A, lda, (const bf16_t*)B, ldb, C, ldc, alpha, beta, nullptr, 0, 0, 0};
  if (dtl_fits_any(M, N, K, lda, a_kmaj, ldb, b_kmaj))
    return launch_dtl_any<MODE_DENSE, true>(a, a_kmaj, b_kmaj, c_dtype, K % 64 != 0, big_tiles(M, N, K), 1, s);
  if (use_big_tile(M, N))
    return launch_bf16<CfgBig, MODE_DENSE>(a, a_kmaj, b_kmaj, c_dtype,
                                           dim3((unsigned)cdiv(N, 256), (unsigned)cdiv(M, 256)), s);
  return launch_bf16<CfgSmall, MODE_DENSE>(a, a_kmaj, b_kmaj, c_dtype,
                                           dim3((unsigned)cdiv(N, 128), (unsigned)cdiv(M, 128)), s);
}

int pd_gemm_strided_batched(int dtype, int64_t batch, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                            int64_t stride_a, int trans_a, const void* B, int64_t ldb, int64_t stride_b, int trans_b,
                            void* C, int64_t ldc, int64_t stride_c, int c_dtype, float alpha, float beta,
                            void* stream) {
  if (batch < 0 || M < 0 || N < 0 || K < 0 || stride_a < 0 || stride_b < 0 || stride_c < 0 || !A || !B || !C)
    return fail(PD_EINVAL, "pd_gemm_strided_batched: bad args");
  if (batch == 0 || M == 0 || N == 0) return PD_OK;
  hipStream_t s = (hipStream_t)stream;
  if (batch > 65535 || cdiv(M, FT) > 65535 || cdiv(N, FT) > 65535)
    return fail(PD_EUNSUPPORTED, "pd_gemm_strided_batched: too large");
  if (dtype == PD_DTYPE_F32) {
    if (c_dtype != PD_DTYPE_F32) return fail(PD_EINVAL, "pd_gemm_strided_batched: fp32 path writes fp32");
    launch_gemm_f32(batch, M, N, K, (const float*)A, lda, trans_a, (const float*)B, ldb, trans_b, (float*)C, ldc,
                    alpha, beta, stride_a, stride_b, stride_c, s);
    return check_launch("pd_gemm_strided_batched f32");
  }
  if (dtype != PD_DTYPE_BF16) return fail(PD_EINVAL, "pd_gemm_strided_batched: dtype");
  bool a_kmaj = !trans_a, b_kmaj = trans_b;
  if (!bf16_operand_ok(A, lda, a_kmaj ? K : M) || !bf16_operand_ok(B, ldb, b_kmaj ? K : N) || stride_a % 8 ||
      stride_b % 8)
    return fail(PD_EUNSUPPORTED,
                "pd_gemm_strided_batched: bf16 operands need 16B alignment, ld and batch strides % 8 == 0");
  GemmArgs a{M, N, K, (const bf16_t*)A, lda, (const bf16_t*)B, ldb, C, ldc, alpha, beta, nullptr, 0, stride_b,
             stride_c, stride_a};
  if (dtl_fits_any(M, N, K, lda, a_kmaj, ldb, b_kmaj))
    return launch_dtl_any<MODE_BATCHED, false>(a, a_kmaj, b_kmaj, c_dtype, K % 64 != 0, false, (unsigned)batch, s);
  return launch_bf16<CfgSmall, MODE_BATCHED>(
      a, a_kmaj, b_kmaj, c_dtype, dim3((unsigned)cdiv(N, 128), (unsigned)cdiv(M, 128), (unsigned)batch), s);
}

int pd_grouped_gemm(const void* lhs, const void* rhs, const int32_t* offsets, int64_t J, int E, int64_t K, int64_t N,
                    int trans_rhs, void* out, int out_dtype, void* stream) {
  return pd::grouped_gemm(lhs, rhs, offsets, J, E, K, N, trans_rhs, out, out_dtype, stream, true);
}

}  // extern "C"

namespace pd {

int grouped_gemm(const void* lhs, const void* rhs, const int32_t* offsets, int64_t J, int E, int64_t K, int64_t N,
                 int trans_rhs, void* out, int out_dtype, void* stream, bool zero_tail) {
  if (J < 0 || E <= 0 || K <= 0 || N <= 0 || !lhs || !rhs || !offsets || !out)
    return fail(PD_EINVAL, "pd_grouped_gemm: bad args");
  if (J == 0) return PD_OK;
  bool b_kmaj = trans_rhs != 0;
  if (!bf16_operand_ok(lhs, K, K) || !bf16_operand_ok(rhs, b_kmaj ? K : N, b_kmaj ? K : N))
    return fail(PD_EUNSUPPORTED, "pd_grouped_gemm: K and N must be multiples of 8 with 16B-aligned bases");
  hipStream_t s = (hipStream_t)stream;
  // zero rows past sum(group_sizes) (ragged_dot leaves them 0)
  if (zero_tail)
    hipLaunchKernelGGL(k_zero_tail_rows, dim3(256), dim3(256), 0, s, offsets, E, J, N,
                       out_dtype == PD_DTYPE_F32 ? 4 : 2, out);
  GemmArgs a{J, N, K, (const bf16_t*)lhs, K, (const bf16_t*)rhs, b_kmaj ? K : N, out, N, 1.f, 0.f, offsets, E,
             K * N, 0};
  int64_t max_tiles = cdiv(J, CfgSmall::BM) + E;
  if (max_tiles > 65535) return fail(PD_EUNSUPPORTED, "pd_grouped_gemm: too many rows");
  dim3 grid((unsigned)cdiv(N, CfgSmall::BN), (unsigned)max_tiles);
  static_assert(CfgDtlRA::BM == CfgSmall::BM && CfgDtlRA::BN == CfgSmall::BN, "one grid shape for both kernels");
  const bool kedge = K % 64 != 0;
  if (b_kmaj && dtl_fits(J, K, N, K)) {
    if (big_tiles_grouped(J, E, N))
      return launch_dtl<CfgDtlBig, MODE_GROUPED>(a, out_dtype, kedge,
                                                 dim3((unsigned)cdiv(N, 256), (unsigned)(cdiv(J, 256) + E)), s);
    return launch_dtl<CfgDtl, MODE_GROUPED>(a, out_dtype, kedge, grid, s);
  }
  if (!b_kmaj && dtl_fits(J, K, 0, 0) && dtl_fits_mn(K, N))  // each expert's rhs stored [K][N]
    return launch_dtl<CfgDtl, MODE_GROUPED, false, true>(a, out_dtype, kedge, grid, s);
  return launch_bf16<CfgSmall, MODE_GROUPED>(a, true, b_kmaj, out_dtype, grid, s);
}

// ---------------------------------------------------------------- split contraction
// Slices: enough (tiles x slices >= 512, two blocks per CU) when the output has fewer than
// 384 128x128 tiles, each slice at least 512 deep, at most 16 slices; or the caller's
// count (`splits` > 0).
static int64_t splitk_slice(int64_t M, int64_t N, int64_t K, int splits_req = 0) {
  if (splits_req > 0) return splits_req < 2 || K < 2 * 64 ? 0 : cdiv(cdiv(K, splits_req), 64) * 64;
  const int64_t tiles = cdiv(M, CfgDtlRA::BM) * cdiv(N, CfgDtlRA::BN);
  if (tiles >= 384 || K < 1024) return 0;
  int64_t splits = std::min<int64_t>(std::min<int64_t>(cdiv(512, tiles), K / 512), 16);
  if (splits < 2) return 0;
  return cdiv(cdiv(K, splits), 64) * 64;
}

size_t gemm_splitk_ws_bytes(int64_t M, int64_t N, int64_t K, int splits) {
  const int64_t kc = splitk_slice(M, N, K, splits);
  return kc ? (size_t)cdiv(K, kc) * M * N * sizeof(float) : 0;
}

// C[m, n] = sum_z part[z][m, n] (+ beta * C), slices added in order; 4 columns per thread.
template <typename TC>
__global__ __launch_bounds__(256) void k_splitk_reduce(const float* __restrict__ part, int64_t M, int64_t N,
                                                       int splits, TC* __restrict__ C, int64_t ldc, float beta) {
  const int64_t n4 = N / 4, total = M * n4;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t m = i / n4, c = (i % n4) * 4;
    float4 acc = *(const float4*)(part + m * N + c);
    for (int z = 1; z < splits; ++z) {
      const float4 v = *(const float4*)(part + ((int64_t)z * M + m) * N + c);
      acc.x += v.x;
      acc.y += v.y;
      acc.z += v.z;
      acc.w += v.w;
    }
    const float o[4] = {acc.x, acc.y, acc.z, acc.w};
    store4<TC>(C, m * ldc + c, o, 1.f, beta);
  }
}

int gemm_splitk(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, int trans_a, const void* B, int64_t ldb,
                int trans_b, void* C, int64_t ldc, int c_dtype, float beta, void* ws, size_t ws_bytes, void* stream,
                int splits_req) {
  const int64_t kc = splitk_slice(M, N, K, splits_req);
  if (!kc || N % 4 || ldc % 4 || !aligned16(C))
    return pd_gemm(PD_DTYPE_BF16, M, N, K, A, lda, trans_a, B, ldb, trans_b, C, ldc, c_dtype, 1.f, beta, stream);
  const bool a_kmaj = !trans_a, b_kmaj = trans_b;
  if (!bf16_operand_ok(A, lda, a_kmaj ? K : M) || !bf16_operand_ok(B, ldb, b_kmaj ? K : N) ||
      !dtl_fits_any(M, N, K, lda, a_kmaj, ldb, b_kmaj))
    return fail(PD_EUNSUPPORTED, "gemm_splitk: operands");
  const int splits = (int)cdiv(K, kc);
  if (!ws || ws_bytes < (size_t)splits * M * N * sizeof(float)) return fail(PD_EWORKSPACE, "gemm_splitk: scratch");
  hipStream_t s = (hipStream_t)stream;
  GemmArgs a{M, N, K, (const bf16_t*)A, lda, (const bf16_t*)B, ldb, ws, N, 1.f, 0.f, nullptr, 0, 0, M * N, kc};
  int rc = launch_dtl_any<MODE_SPLITK, false>(a, a_kmaj, b_kmaj, PD_DTYPE_F32, K % 64 != 0, false, (unsigned)splits, s);
  if (rc) return rc;
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(M * N / 4, 256), 8192));
  if (c_dtype == PD_DTYPE_F32)
    hipLaunchKernelGGL(k_splitk_reduce<float>, dim3(blocks), dim3(256), 0, s, (const float*)ws, M, N, splits,
                       (float*)C, ldc, beta);
  else
    hipLaunchKernelGGL(k_splitk_reduce<bf16_t>, dim3(blocks), dim3(256), 0, s, (const float*)ws, M, N, splits,
                       (bf16_t*)C, ldc, beta);
  return check_launch("gemm_splitk reduce");
}

int gemm_nt_splitk(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, const void* Bt, int64_t ldb, void* C,
                   int64_t ldc, int c_dtype, float beta, void* ws, size_t ws_bytes, void* stream) {
  return gemm_splitk(M, N, K, A, lda, 0, Bt, ldb, 1, C, ldc, c_dtype, beta, ws, ws_bytes, stream);
}

int grouped_gemm_pair(const void* lhs1, const void* rhsT1, void* out1, const void* lhs2, const void* rhsT2, void* out2,
                      const int32_t* offsets, int64_t J, int E, int64_t K, int64_t N, int out_dtype, void* stream) {
  if (J < 0 || E <= 0 || K <= 0 || N <= 0 || !lhs1 || !rhsT1 || !out1 || !lhs2 || !rhsT2 || !out2 || !offsets)
    return fail(PD_EINVAL, "grouped_gemm_pair: bad args");
  if (J == 0) return PD_OK;
  if (!bf16_operand_ok(lhs1, K, K) || !bf16_operand_ok(rhsT1, K, K) || !bf16_operand_ok(lhs2, K, K) ||
      !bf16_operand_ok(rhsT2, K, K))
    return fail(PD_EUNSUPPORTED, "grouped_gemm_pair: K must be a multiple of 8 with 16B-aligned bases");
  GemmArgs a{J, N, K, (const bf16_t*)lhs1, K, (const bf16_t*)rhsT1, K, out1, N, 1.f, 0.f, offsets, E, K * N, 0, 0,
             (const bf16_t*)lhs2, (const bf16_t*)rhsT2, out2};
  if (cdiv(J, CfgDtlRA::BM) + E > 65535) return fail(PD_EUNSUPPORTED, "grouped_gemm_pair: too many rows");
  if (!dtl_fits(J, K, N, K)) return fail(PD_EUNSUPPORTED, "grouped_gemm_pair: operands of 2 GiB or more");
  if (big_tiles_grouped(J, E, N, 2))
    return launch_dtl<CfgDtlBig, MODE_GROUPED>(
        a, out_dtype, K % CfgDtlBig::BK != 0,
        dim3((unsigned)cdiv(N, CfgDtlBig::BN), (unsigned)(cdiv(J, CfgDtlBig::BM) + E), 2), (hipStream_t)stream);
  return launch_dtl<CfgDtlRA, MODE_GROUPED>(
      a, out_dtype, K % CfgDtlRA::BK != 0,
      dim3((unsigned)cdiv(N, CfgDtlRA::BN), (unsigned)(cdiv(J, CfgDtlRA::BM) + E), 2), (hipStream_t)stream);
}

int grouped_gemm_kcat(const void* lhs1, const void* rhs1, int64_t K1, const void* lhs2, const void* rhs2, int64_t K2,
                      void* out, const float* rs, const void* lhs1b, const void* rhs1b, const void* lhs2b,
                      const void* rhs2b, void* outb, const float* rs2, const int32_t* sort_idx, int k,
                      const int32_t* offsets, int64_t J, int E, int64_t N, void* stream) {
  const bool pair = lhs1b != nullptr;
  if (J < 0 || E <= 0 || E > 65535 || K1 <= 0 || K2 <= 0 || N <= 0 || k <= 0 || !lhs1 || !rhs1 || !lhs2 || !rhs2 ||
      !out || !rs || !sort_idx || !offsets || (pair && (!rhs1b || !lhs2b || !rhs2b || !outb)))
    return fail(PD_EINVAL, "grouped_gemm_kcat: bad args");
  if (J == 0) return PD_OK;
  const void* ops[8] = {lhs1, rhs1, lhs2, rhs2, pair ? lhs1b : lhs1, pair ? rhs1b : rhs1, pair ? lhs2b : lhs2,
                        pair ? rhs2b : rhs2};
  for (int i = 0; i < 8; ++i)
    if (!bf16_operand_ok(ops[i], (i & 2) ? K2 : K1, (i & 2) ? K2 : K1))
      return fail(PD_EUNSUPPORTED, "grouped_gemm_kcat: K1, K2 must be multiples of 8 with 16B-aligned bases");
  if (!aligned16(out) || (pair && !aligned16(outb)) || N % 8)
    return fail(PD_EUNSUPPORTED, "grouped_gemm_kcat: N % 8 and 16B-aligned outputs");
  if (!dtl_fits(J, K1, N, K1) || !dtl_fits(J, K2, N, K2))
    return fail(PD_EUNSUPPORTED, "grouped_gemm_kcat: operands of 2 GiB or more");
  if (cdiv(J, CfgDtlRA::BM) + E > 65535) return fail(PD_EUNSUPPORTED, "grouped_gemm_kcat: too many rows");
  GemmArgs a{J, N, K2, (const bf16_t*)lhs2, K2, (const bf16_t*)rhs2, K2, out, N, 1.f, 0.f, offsets, E, K2 * N, 0, 0,
             pair ? (const bf16_t*)lhs2b : nullptr, pair ? (const bf16_t*)rhs2b : nullptr, pair ? outb : nullptr};
  KcatArgs q{(const bf16_t*)lhs1, K1, (const bf16_t*)rhs1, K1, K1, nullptr, nullptr};
  q.A1b = pair ? (const bf16_t*)lhs1b : nullptr;
  q.B1b = pair ? (const bf16_t*)rhs1b : nullptr;
  q.strideB1 = K1 * N;
  q.rs_tok = rs;
  q.rs_tok2 = rs2 ? rs2 : rs;
  q.sort_idx = sort_idx;
  q.k = k;
#define PD_L(CFG, KE)                                                                                            \
  hipLaunchKernelGGL((k_gemm_dtl_kcat<CFG, bf16_t, false, false, KE, EpiStore, MODE_GROUPED>),                    \
                     dim3((unsigned)cdiv(N, CFG::BN), (unsigned)(cdiv(J, CFG::BM) + E), pair ? 2u : 1u),          \
                     dim3(CFG::NT), 0, (hipStream_t)stream, a, q, EpiStore::Args{})
  const bool ke = K1 % 64 || K2 % 64;
  if (big_tiles_grouped(J, E, N, pair ? 2 : 1)) {
    if (ke) PD_L(CfgDtlBig, true);
    else PD_L(CfgDtlBig, false);
  } else {
    if (ke) PD_L(CfgDtl, true);
    else PD_L(CfgDtl, false);
  }
#undef PD_L
  return check_launch("grouped_gemm_kcat");
}

int grouped_gemm_dw_pair(const void* lhs1, const void* dout1, void* out1, const void* lhs2, const void* dout2,
                         void* out2, const int32_t* offsets, int64_t J, int E, int64_t K, int64_t N, int out_dtype,
                         void* stream) {
  if (J < 0 || E <= 0 || K <= 0 || N <= 0 || !lhs1 || !dout1 || !out1 || !lhs2 || !dout2 || !out2 || !offsets)
    return fail(PD_EINVAL, "grouped_gemm_dw_pair: bad args");
  if (!bf16_operand_ok(lhs1, K, K) || !bf16_operand_ok(dout1, N, N) || !bf16_operand_ok(lhs2, K, K) ||
      !bf16_operand_ok(dout2, N, N))
    return fail(PD_EUNSUPPORTED, "grouped_gemm_dw_pair: K and N must be multiples of 8 with 16B-aligned bases");
  if (2 * (int64_t)E > 65535 || cdiv(K, CfgDtlRA::BM) > 65535) return fail(PD_EUNSUPPORTED, "grouped_gemm_dw_pair: size");
  if (!dtl_fits_mn(J, K) || !dtl_fits_mn(J, N))
    return fail(PD_EUNSUPPORTED, "grouped_gemm_dw_pair: operands of 2 GiB or more");
  // both operands MN-major (their rows are the contraction's jobs), 128x128 tiles
  GemmArgs a{K, N, J, (const bf16_t*)lhs1, K, (const bf16_t*)dout1, N, out1, N, 1.f, 0.f, offsets, E, 0, K * N, 0,
             (const bf16_t*)lhs2, (const bf16_t*)dout2, out2};
  dim3 grid((unsigned)cdiv(N, CfgDtlRA::BN), (unsigned)cdiv(K, CfgDtlRA::BM), (unsigned)(2 * E));
  return launch_dtl<CfgDtl, MODE_GROUPED_K, true, true>(a, out_dtype, true, grid, (hipStream_t)stream);
}

}  // namespace pd

extern "C" {

int pd_grouped_gemm_dw(const void* lhs, const void* dout, const int32_t* offsets, int64_t J, int E, int64_t K,
                       int64_t N, void* out, int out_dtype, void* stream) {
  if (J < 0 || E <= 0 || K <= 0 || N <= 0 || !lhs || !dout || !offsets || !out)
    return fail(PD_EINVAL, "pd_grouped_gemm_dw: bad args");
  if (!bf16_operand_ok(lhs, K, K) || !bf16_operand_ok(dout, N, N))
    return fail(PD_EUNSUPPORTED, "pd_grouped_gemm_dw: K and N must be multiples of 8 with 16B-aligned bases");
  if (E > 65535 || cdiv(K, CfgSmall::BM) > 65535) return fail(PD_EUNSUPPORTED, "pd_grouped_gemm_dw: E or K too large");
  // out[e] (M=K_in x N) = lhs[rows_e]^T (A stored [J,K]: M-contiguous) @ dout[rows_e] ([J,N])
  GemmArgs a{K, N, J, (const bf16_t*)lhs, K, (const bf16_t*)dout, N, out, N, 1.f, 0.f, offsets, E, 0, K * N};
  dim3 grid((unsigned)cdiv(N, CfgSmall::BN), (unsigned)cdiv(K, CfgSmall::BM), (unsigned)E);
  static_assert(CfgDtlRA::BM == CfgSmall::BM && CfgDtlRA::BN == CfgSmall::BN, "one grid shape for both kernels");
  if (dtl_fits_mn(J, K) && dtl_fits_mn(J, N))  // both operands MN-major: rows of lhs / dout are k
    return launch_dtl<CfgDtl, MODE_GROUPED_K, true, true>(a, out_dtype, true, grid, (hipStream_t)stream);
  return launch_bf16<CfgSmall, MODE_GROUPED_K>(a, false, false, out_dtype, grid, (hipStream_t)stream);
}

int pd_grouped_gemm_dw_kmajor(const void* lhsT, const void* doutT, const int32_t* offsets, int64_t J, int E,
                              int64_t K, int64_t N, void* out, int out_dtype, void* stream) {
  if (J < 0 || E <= 0 || K <= 0 || N <= 0 || !lhsT || !doutT || !offsets || !out)
    return fail(PD_EINVAL, "pd_grouped_gemm_dw_kmajor: bad args");
  if (!bf16_operand_ok(lhsT, J, J) || !bf16_operand_ok(doutT, J, J))
    return fail(PD_EUNSUPPORTED, "pd_grouped_gemm_dw_kmajor: J must be a multiple of 8 with 16B-aligned bases");
  if (E > 65535 || cdiv(K, CfgDtl::BM) > 65535) return fail(PD_EUNSUPPORTED, "pd_grouped_gemm_dw_kmajor: size");
  // (J == 0: every group has an empty k range, no loads are issued, out = 0)
  // out[e] (M=K x N) = lhsT[:, rows_e] (A stored [K, J]: K-major) @ doutT[:, rows_e]^T (B stored [N, J])
  GemmArgs a{K, N, J, (const bf16_t*)lhsT, J, (const bf16_t*)doutT, J, out, N, 1.f, 0.f, offsets, E, 0, K * N};
  if (!dtl_fits(K, J, N, J)) return fail(PD_EUNSUPPORTED, "pd_grouped_gemm_dw_kmajor: operands of 2 GiB or more");
  dim3 grid((unsigned)cdiv(N, CfgDtlRA::BN), (unsigned)cdiv(K, CfgDtlRA::BM), (unsigned)E);
  return launch_dtl<CfgDtlRA, MODE_GROUPED_K>(a, out_dtype, true, grid, (hipStream_t)stream);
}

}  // extern "C"
