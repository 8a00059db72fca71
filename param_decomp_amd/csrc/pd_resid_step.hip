// The ResidMLP toy decomposition step as one native call (gfx950, fp32).
//
//   target   r_0 = x W_E; per layer hid = relu(r W_in^T), r += hid W_out^T; out = r W_U
//                                                     pd/targets/resid_mlp.py:266-333
//   masked   the same with every mlp_in / mlp_out decomposed, site output
//            ((a V) (.) m) U (site_forward, pd/core/decomposed_linear.py:142-175;
//            the masked forward pd/targets/resid_mlp.py:336-390)
//   CI       paper-form gate per component on the clean input's a V, lower / upper leaky
//            hard sigmoids, m = lower + (1 - lower) u with fp32 Threefry draws per site
//            (pd/core/masking.py:148-167)
//   loss     recon_coeff mse(out, clean) + imp_coeff sum_sites sum_c mean_b upper^p
//            (pd/targets/resid_mlp.py:411-418; the paper's L_p), fwd + bwd
//
// The products run on the library's fp32 MFMA GEMM. Each site's CI gate, squashing, mask
// draw, masked activations and imp-min term form one column-mapped pass (one lane per
// component over RM_ROWS rows), and its backward (mask pullback into both a V operands,
// squashing and gate pullbacks, gate-parameter partials) another; the partials are added
// over row chunks in a fixed order. Relus and residual sums are the products' epilogues,
// independent small products share a launch. At the 1-layer benchmark shape (2048 x 1000, C =
// 100) that is 22 launches and 210 us per step (31 and 296 with one launch per product, relu,
// copy and weight gradient), against about 90 launches for the same step composed from the
// library's primitives.
#include <algorithm>
#include <vector>

#include "pd_common.hpp"

namespace pd {

static constexpr int RM_COLS = 64;   // components per block of the site passes
static constexpr int RM_WAVES = 4;   // waves per block, each RM_ROWS / RM_WAVES of its rows
static constexpr int RM_ROWS = 8;    // rows per block of the site passes
static constexpr int RM_GATE = 49;  // gate-parameter gradient slots per component

struct RmGate {
  const float *w_in, *b_in, *w_out, *b_out;  // [C,16], [C,16], [C,16], [C]
  uint32_t k0, k1;                           // the site's mask key
};

__device__ inline float rm_pow(float b, float p) { return p == 2.f ? b * b : (p == 1.f ? b : powf(b, p)); }
__device__ inline float rm_dpow(float b, float p) {
  return p == 2.f ? 2.f * b : (p == 1.f ? 1.f : p * powf(b, p - 1.f));
}

// Forward of one site: g = gate(hg) (kept in g_raw for the backward), lower / upper, the
// fp32 uniform u of element (t, c) of the site's [B, C] draw, acts = ha (lower + (1 -
// lower) u), and the block's sum of upper^p. Block = 64 components x RM_ROWS rows, wave w
// taking rows RM_ROWS / RM_WAVES w .. (sums added in wave order). hg is the clean input's a V (the gate
// input); ha the masked input's (the same array at the first mlp_in).
__global__ __launch_bounds__(RM_COLS * RM_WAVES) void k_rm_site_fwd(const float* __restrict__ hg,
                                                                    const float* __restrict__ ha, int64_t B, int C,
                                                                    RmGate gt, int layout, float p,
                                                                    float* __restrict__ g_raw,
                                                                    float* __restrict__ acts,
                                                                    float* __restrict__ imp_part) {
  __shared__ float red[RM_WAVES];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = blockIdx.x * RM_COLS + lane;
  constexpr int WR = RM_ROWS / RM_WAVES;
  const int64_t r0 = (int64_t)blockIdx.y * RM_ROWS + wv * WR, r1 = r0 + WR < B ? r0 + WR : B;
  float imp = 0.f;
  if (c < C) {
    float wi[16], bi[16], wo[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      wi[j] = gt.w_in[c * 16 + j];
      bi[j] = gt.b_in[c * 16 + j];
      wo[j] = gt.w_out[c * 16 + j];
    }
    const float bo = gt.b_out[c];
    const int64_t n = B * C;
    for (int64_t t = r0; t < r1; ++t) {
      const int64_t i = t * C + c;
      const float hv = hg[i];
      float g = bo;
#pragma unroll
      for (int j = 0; j < 16; ++j) g = fmaf(wo[j], gelu_only<true>(fmaf(wi[j], hv, bi[j])), g);
      g_raw[i] = g;
      const float lo = lower_fwd(g);
      imp += rm_pow(upper_fwd(g), p);
      const float u = draw_uniform(gt.k0, gt.k1, i, n, PD_DTYPE_F32, layout);
      acts[i] = ha[i] * (lo + (1.f - lo) * u);
    }
  }
  imp = wave_sum(imp);
  if (lane == 0) red[wv] = imp;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = red[0];
#pragma unroll
    for (int k = 1; k < RM_WAVES; ++k) t += red[k];
    imp_part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = t;
  }
}

// Backward of one site from d_acts: the mask pullback d_ha = d_acts m (onto the masked
// input's a V), and dg = lower_vjp(g, d_acts ha (1 - u)) + upper_vjp(g, imp_scale d upper^p)
// pulled back through the gate onto hg (d_hg) and into the lane's gate-parameter sums,
// written per row chunk to partial [chunk][49][C] (the block's waves added in row order).
// With d_hg == d_ha (the gate and the mask read the same a V) the two pullbacks are
// written summed.
__global__ __launch_bounds__(RM_COLS * RM_WAVES) void k_rm_site_bwd(
    const float* __restrict__ d_acts, const float* __restrict__ hg, const float* __restrict__ ha,
    const float* __restrict__ g_raw, int64_t B, int C, RmGate gt, int layout, float p, float imp_scale, float* d_ha,
    float* d_hg, float* __restrict__ partial) {
  __shared__ float red[RM_WAVES - 1][RM_GATE][RM_COLS];  // waves 1.. hand their sums to wave 0
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, c = blockIdx.x * RM_COLS + lane;
  constexpr int WR = RM_ROWS / RM_WAVES;
  const int64_t r0 = (int64_t)blockIdx.y * RM_ROWS + wv * WR, r1 = r0 + WR < B ? r0 + WR : B;
  const bool ok = c < C, same = d_ha == d_hg;
  float wi[16], bi[16], wo[16], a_wi[16], a_bi[16], a_wo[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    wi[j] = ok ? gt.w_in[c * 16 + j] : 0.f;
    bi[j] = ok ? gt.b_in[c * 16 + j] : 0.f;
    wo[j] = ok ? gt.w_out[c * 16 + j] : 0.f;
    a_wi[j] = a_bi[j] = a_wo[j] = 0.f;
  }
  float a_bo = 0.f;
  const int64_t n = B * C;
  for (int64_t t = r0; t < r1 && ok; ++t) {
    const int64_t i = t * C + c;
    const float hv = hg[i], av = ha[i], g = g_raw[i], da = d_acts[i];
    const float lo = lower_fwd(g);
    const float u = draw_uniform(gt.k0, gt.k1, i, n, PD_DTYPE_F32, layout);
    const float dmask = da * (lo + (1.f - lo) * u);
    const float dg = lower_vjp(g, da * av * (1.f - u)) + upper_vjp(g, imp_scale * rm_dpow(upper_fwd(g), p));
    float dh = 0.f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const GeluOut go = gelu_and_grad<true>(fmaf(wi[j], hv, bi[j]));
      const float dz = dg * wo[j] * go.grad;
      dh = fmaf(dz, wi[j], dh);
      a_wi[j] = fmaf(dz, hv, a_wi[j]);
      a_bi[j] += dz;
      a_wo[j] = fmaf(dg, go.gelu, a_wo[j]);
    }
    a_bo += dg;
    if (same) {
      d_ha[i] = dmask + dh;
    } else {
      d_ha[i] = dmask;
      d_hg[i] = dh;
    }
  }
  // the block's sum in wave order (the rows' order), by wave 0
  if (wv > 0) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      red[wv - 1][j][lane] = a_wi[j];
      red[wv - 1][16 + j][lane] = a_bi[j];
      red[wv - 1][32 + j][lane] = a_wo[j];
    }
    red[wv - 1][48][lane] = a_bo;
  }
  __syncthreads();
  if (wv > 0 || !ok) return;
#pragma unroll
  for (int k = 0; k < RM_WAVES - 1; ++k) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      a_wi[j] += red[k][j][lane];
      a_bi[j] += red[k][16 + j][lane];
      a_wo[j] += red[k][32 + j][lane];
    }
    a_bo += red[k][48][lane];
  }
  float* pp = partial + (int64_t)blockIdx.y * RM_GATE * C;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    pp[(int64_t)j * C + c] = a_wi[j];
    pp[(int64_t)(16 + j) * C + c] = a_bi[j];
    pp[(int64_t)(32 + j) * C + c] = a_wo[j];
  }
  pp[(int64_t)48 * C + c] = a_bo;
}

// Every site's gate-parameter gradients: the row-chunk partials of slot q of component c
// added in chunk order into the flat gradient buffer (w_in [C,16] | b_in | w_out | b_out
// after the site's dV and dU; every site spans (D + M + 49) C floats).
__global__ void k_rm_gate_reduce(const float* __restrict__ partial, int64_t chunks, int C, int D, int M, int nsites,
                                 float* __restrict__ grads) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = (int64_t)RM_GATE * C;
  if (idx >= per * nsites) return;
  const int s = (int)(idx / per);
  const int64_t rem = idx % per, q = rem / C, c = rem % C;
  const float acc = pd_ordered_sum(partial + (int64_t)s * chunks * per + rem, chunks, per);
  float* g = grads + ((int64_t)s * (D + M + RM_GATE) + D + M) * C;
  if (q < 48) g[(q / 16) * C * 16 + c * 16 + q % 16] = acc;
  else g[48 * C + c] = acc;
}

// relu in place; and the relu pullback d *= (y > 0) in place.
__global__ void k_rm_relu(float* __restrict__ a, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    a[i] = fmaxf(a[i], 0.f);
}
__global__ void k_rm_relu_bwd(float* __restrict__ d, const float* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    d[i] = y[i] > 0.f ? d[i] : 0.f;
}

// d_out = scale (out - clean) (scale = recon_coeff 2 / n) and each block's sum of squares.
static constexpr int RM_REC_BLOCKS = 256;
__global__ __launch_bounds__(256) void k_rm_recon(const float* __restrict__ out, const float* __restrict__ clean,
                                                  int64_t n, float scale, float* __restrict__ d_out,
                                                  float* __restrict__ rec_part) {
  __shared__ float red[4];
  float acc = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float e = out[i] - clean[i];
    d_out[i] = scale * e;
    acc = fmaf(e, e, acc);
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) rec_part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// losses = {recon_coeff recon + imp_coeff imp, recon, imp}: recon = sum(rec_part) / n,
// imp = sum(imp_part) / B (one block, partials added in order per thread, then in
// thread order).
__global__ void k_rm_losses(const float* __restrict__ rec_part, int n_rec, const float* __restrict__ imp_part,
                            int64_t n_imp, double inv_n, double inv_b, float recon_coeff, float imp_coeff,
                            float* __restrict__ losses) {
  __shared__ double sr[256], si[256];
  double r = 0.0, m = 0.0;
  for (int64_t i = threadIdx.x; i < n_rec; i += blockDim.x) r += rec_part[i];
  for (int64_t i = threadIdx.x; i < n_imp; i += blockDim.x) m += imp_part[i];
  sr[threadIdx.x] = r;
  si[threadIdx.x] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double R = 0.0, I = 0.0;
    for (int k = 0; k < (int)blockDim.x; ++k) {
      R += sr[k];
      I += si[k];
    }
    const double recon = R * inv_n, imp = I * inv_b;
    losses[0] = (float)(recon_coeff * recon + imp_coeff * imp);
    losses[1] = (float)recon;
    losses[2] = (float)imp;
  }
}

struct RmDims {
  int64_t B;
  int F, D, M, C, L;
  int nsites() const { return 2 * L; }
  int din(int s) const { return s % 2 ? M : D; }
  int dout(int s) const { return s % 2 ? D : M; }
  int64_t chunks() const { return cdiv(B, RM_ROWS); }
  int64_t cblocks() const { return cdiv(C, RM_COLS); }
};

// The flat gradient buffer: per site dV [din, C] | dU [C, dout] | gate (w_in | b_in |
// w_out | b_out), sites in order (layers.l.mlp_in, layers.l.mlp_out).
struct RmGradLayout {
  std::vector<int64_t> dV, dU, gate;
  int64_t total = 0;
  explicit RmGradLayout(const RmDims& D) {
    for (int s = 0; s < D.nsites(); ++s) {
      dV.push_back(total);
      total += (int64_t)D.din(s) * D.C;
      dU.push_back(total);
      total += (int64_t)D.C * D.dout(s);
      gate.push_back(total);
      total += (int64_t)RM_GATE * D.C;
    }
  }
};

struct RmArena {
  char* base;
  size_t off = 0;
  float* take(int64_t n) {
    float* p = base ? (float*)(base + off) : nullptr;
    off += ((size_t)n * sizeof(float) + 255) & ~(size_t)255;
    return p;
  }
};

struct RmWork {
  std::vector<float*> r, rm, hidc, hid, hg, ha, graw, acts;  // per layer (r, rm: L + 1) / per site
  float *clean, *out, *d_out, *d_r, *d_r2, *d_acts, *d_hid, *rec_part, *imp_part, *gpart, *wpart;
  float *d_ha[2], *d_hg[2];  // mlp_in's, mlp_out's: a layer's weight gradients are taken together
  int splits;                // contraction slices of the weight gradients, 0: one product at a time
  size_t bytes;
};

// A layer's weight gradients (up to 6 products over the batch) run in one launch, each
// contraction cut into slices of at least 256 rows, as many as give the chip four blocks
// per CU; their slabs are added in order afterwards. One at a time each took 16 us however
// small its output: 16 waves of one CU walking the whole batch. Outputs that fill the chip by
// themselves stay single products. At 2048 rows, D = 1000, C = 100, M = 50 (280 tiles, 4 slices):
// 81 us in five launches, 31 in two.
// What bounds them now is L2: a 32x32 tile of one wave reads 512 bytes per MFMA.
static int rm_splits(const RmDims& D) {
  const int64_t tm = cdiv(D.M, 32), tc = cdiv(D.C, 32), td = cdiv(D.D, 32);
  const int64_t tiles = (D.L > 1 ? 3 : 2) * td * tc + 3 * tm * tc;
  if (tiles > 1024) return 0;
  return (int)std::max<int64_t>(1, std::min<int64_t>({D.B / 256, cdiv(1024, tiles), 16}));
}

// Sums of consecutive [n] slabs, in order: the weight gradients' contraction slices.
struct RmSums {
  const float* src[4];
  float* dst[4];
  int64_t n[4], first[5];
  int32_t slabs[4];
};
__global__ __launch_bounds__(256) void k_rm_sum_slabs(RmSums a) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  int q = 0;
  while (q < 3 && i >= a.first[q + 1]) ++q;
  i -= a.first[q];
  const int64_t n = a.n[q];
  if (i >= n) return;
  const float* src = a.src[q] + i;
  float sum = src[0];
  for (int x = 1; x < a.slabs[q]; ++x) sum += src[x * n];
  a.dst[q][i] = sum;
}

static RmWork rm_layout(const RmDims& D, char* base) {
  RmArena A{base};
  RmWork W;
  const int64_t B = D.B;
  for (int l = 0; l <= D.L; ++l) {
    W.r.push_back(A.take(B * D.D));
    W.rm.push_back(l == 0 ? W.r[0] : A.take(B * D.D));  // the masked pass starts from the same r_0
  }
  for (int l = 0; l < D.L; ++l) {
    W.hidc.push_back(A.take(B * D.M));
    W.hid.push_back(A.take(B * D.M));
  }
  for (int s = 0; s < D.nsites(); ++s) {
    W.hg.push_back(A.take(B * D.C));
    W.ha.push_back(s == 0 ? W.hg[0] : A.take(B * D.C));  // mlp_in of layer 0 reads r_0 in both passes
    W.graw.push_back(A.take(B * D.C));
    W.acts.push_back(A.take(B * D.C));
  }
  W.clean = A.take(B * D.F);
  W.out = A.take(B * D.F);
  W.d_out = A.take(B * D.F);
  W.d_r = A.take(B * D.D);
  W.d_r2 = A.take(B * D.D);
  W.d_acts = A.take(B * D.C);
  for (int q = 0; q < 2; ++q) {
    W.d_ha[q] = A.take(B * D.C);
    W.d_hg[q] = A.take(B * D.C);
  }
  W.d_hid = A.take(B * D.M);
  W.rec_part = A.take(RM_REC_BLOCKS);
  W.imp_part = A.take((int64_t)D.nsites() * D.chunks() * D.cblocks());
  W.gpart = A.take((int64_t)D.nsites() * D.chunks() * RM_GATE * D.C);
  W.splits = rm_splits(D);
  W.wpart = A.take(W.splits * (int64_t)D.C * (3 * (int64_t)D.D + 3 * (int64_t)D.M));
  W.bytes = A.off;
  return W;
}

static unsigned rm_ew_blocks(int64_t n) { return (unsigned)std::min<int64_t>(cdiv(n, 256), 4096); }

}  // namespace pd

using namespace pd;

extern "C" {

size_t pd_resid_mlp_step_workspace_size(int64_t B, int F, int D, int M, int C, int L) {
  if (B <= 0 || F <= 0 || D <= 0 || M <= 0 || C <= 0 || L <= 0) return 0;
  return rm_layout(RmDims{B, F, D, M, C, L}, nullptr).bytes;
}

int64_t pd_resid_mlp_step_grads_size(int D, int M, int C, int L) {
  if (D <= 0 || M <= 0 || C <= 0 || L <= 0) return 0;
  return RmGradLayout(RmDims{1, 1, D, M, C, L}).total;
}

int pd_resid_mlp_step(int64_t B, int F, int D, int M, int C, int L, const float* x, const float* W_E,
                      const float* W_U, const float* const* W_in, const float* const* W_out, const float* const* V,
                      const float* const* U, const float* const* gates, uint32_t draw_k0, uint32_t draw_k1,
                      int layout, float p, float imp_coeff, float recon_coeff, float* grads, float* losses,
                      float* out, void* workspace, size_t workspace_bytes, void* stream) {
  const char* what = "pd_resid_mlp_step";
  if (B <= 0 || F <= 0 || D <= 0 || M <= 0 || C <= 0 || L <= 0 || !x || !W_E || !W_U || !W_in || !W_out || !V ||
      !U || !gates || !grads || !losses || !workspace)
    return fail(PD_EINVAL, std::string(what) + ": bad args");
  if (layout != PD_LAYOUT_PARTITIONABLE && layout != PD_LAYOUT_ORIGINAL)
    return fail(PD_EINVAL, std::string(what) + ": unknown counter layout");
  if (!(p > 0.f)) return fail(PD_EINVAL, std::string(what) + ": p > 0");
  if (B * (int64_t)std::max({F, D, M, C}) >= (int64_t(1) << 31))
    return fail(PD_EUNSUPPORTED, std::string(what) + ": B * width must stay below 2^31");
  const RmDims Dm{B, F, D, M, C, L};
  const int ns = Dm.nsites();
  for (int l = 0; l < L; ++l)
    if (!W_in[l] || !W_out[l]) return fail(PD_EINVAL, std::string(what) + ": null target weight");
  for (int s = 0; s < ns; ++s) {
    if (!V[s] || !U[s]) return fail(PD_EINVAL, std::string(what) + ": null component weight");
    for (int q = 0; q < 4; ++q)
      if (!gates[4 * s + q]) return fail(PD_EINVAL, std::string(what) + ": null gate parameter");
  }
  if (workspace_bytes < rm_layout(Dm, nullptr).bytes) return fail(PD_EWORKSPACE, std::string(what) + ": workspace too small");
  RmWork W = rm_layout(Dm, (char*)workspace);
  if (out) W.out = out;
  hipStream_t s = (hipStream_t)stream;
  const RmGradLayout G(Dm);

  // the sites' mask keys: mask_key = split(draw_key)[0], site key = fold_in(mask_key, site)
  uint32_t halves[4];
  split2(draw_k0, draw_k1, layout, halves);
  std::vector<RmGate> gt(ns);
  for (int i = 0; i < ns; ++i) {
    gt[i] = RmGate{gates[4 * i], gates[4 * i + 1], gates[4 * i + 2], gates[4 * i + 3], 0u, (uint32_t)i};
    threefry2x32(halves[0], halves[1], gt[i].k0, gt[i].k1);
  }

  int rc;
  auto gemm = [&](int64_t m, int64_t nn, int64_t k, const float* a, int64_t lda, int ta, const float* b, int64_t ldb,
                  int tb, float* c, int64_t ldc, float beta) {
    return pd_gemm(PD_DTYPE_F32, m, nn, k, a, lda, ta, b, ldb, tb, c, ldc, PD_DTYPE_F32, 1.f, beta, s);
  };
  auto prod = [&](int64_t m, int64_t nn, int64_t k, const float* a, int ta, const float* b, int tb, float* c,
                  const float* cin = nullptr, int post = 0) {
    return F32Prod{m, nn, k, a, ta ? m : k, ta, b, tb ? k : nn, tb, c, nn, cin, post};
  };
  // One product with its Cin / post in the epilogue; where the direct form does not take it,
  // as separate passes.
  auto fused = [&](const F32Prod& q) {
    if (gemm_f32_direct(q, s)) return (int)PD_OK;
    const bool add = q.Cin && q.post < 2;
    if (add && q.Cin != q.C)
      hipMemcpyAsync(q.C, q.Cin, (size_t)q.M * q.N * sizeof(float), hipMemcpyDeviceToDevice, s);
    if (int e = gemm(q.M, q.N, q.K, q.A, q.lda, q.ta, q.B, q.ldb, q.tb, q.C, q.ldc, add ? 1.f : 0.f)) return e;
    const int64_t n = q.M * q.N;
    if (q.post == 1) hipLaunchKernelGGL(k_rm_relu, dim3(rm_ew_blocks(n)), dim3(256), 0, s, q.C, n);
    if (q.post == 2) hipLaunchKernelGGL(k_rm_relu_bwd, dim3(rm_ew_blocks(n)), dim3(256), 0, s, q.C, q.Cin, n);
    return (int)PD_OK;
  };
  // Two independent products over the same rows: in one launch while both outputs are small
  // (fewer than 1024 32x32 tiles together, four blocks of 8 waves per CU), else one by one.
  auto two = [&](const F32Prod& x, const F32Prod& y) {
    const F32Prod q[2] = {x, y};
    if (cdiv(x.M, 32) * (cdiv(x.N, 32) + cdiv(y.N, 32)) < 1024 && gemm_f32_group(q, 2, 1, s)) return (int)PD_OK;
    const int e = fused(x);
    return e ? e : fused(y);
  };
  const dim3 sgrid((unsigned)Dm.cblocks(), (unsigned)Dm.chunks());
  const int64_t nsite_blocks = Dm.chunks() * Dm.cblocks();

  // ---- clean pass: r_{l+1} = r_l + relu(r_l W_in^T) W_out^T; the gate inputs a V
  if ((rc = fused(prod(B, D, F, x, 0, W_E, 0, W.r[0])))) return rc;
  for (int l = 0; l < L; ++l) {
    if ((rc = two(prod(B, M, D, W.r[l], 0, W_in[l], 1, W.hidc[l], nullptr, 1),
                  prod(B, C, D, W.r[l], 0, V[2 * l], 0, W.hg[2 * l]))))
      return rc;
    if ((rc = fused(prod(B, D, M, W.hidc[l], 0, W_out[l], 1, W.r[l + 1], W.r[l])))) return rc;
    if ((rc = fused(prod(B, C, M, W.hidc[l], 0, V[2 * l + 1], 0, W.hg[2 * l + 1])))) return rc;
  }

  // ---- masked pass
  auto site_fwd = [&](int si) {
    hipLaunchKernelGGL(k_rm_site_fwd, sgrid, dim3(RM_COLS * RM_WAVES), 0, s, W.hg[si], W.ha[si], B, C, gt[si], layout, p,
                       W.graw[si], W.acts[si], W.imp_part + si * nsite_blocks);
  };
  for (int l = 0; l < L; ++l) {
    const int si = 2 * l, so = 2 * l + 1;
    if (l > 0 && (rc = fused(prod(B, C, D, W.rm[l], 0, V[si], 0, W.ha[si])))) return rc;
    site_fwd(si);
    if ((rc = fused(prod(B, M, C, W.acts[si], 0, U[si], 0, W.hid[l], nullptr, 1)))) return rc;
    if ((rc = fused(prod(B, C, M, W.hid[l], 0, V[so], 0, W.ha[so])))) return rc;
    site_fwd(so);
    if ((rc = fused(prod(B, D, C, W.acts[so], 0, U[so], 0, W.rm[l + 1], W.rm[l])))) return rc;
  }
  // the target's output is first needed here, beside the masked one
  if ((rc = two(prod(B, F, D, W.r[L], 0, W_U, 0, W.clean), prod(B, F, D, W.rm[L], 0, W_U, 0, W.out)))) return rc;
  const int64_t nout = B * F;
  hipLaunchKernelGGL(k_rm_recon, dim3(RM_REC_BLOCKS), dim3(256), 0, s, W.out, W.clean, nout,
                     recon_coeff * 2.f / (float)nout, W.d_out, W.rec_part);
  if ((rc = check_launch(what))) return rc;

  // ---- backward: d_r is the masked residual's cotangent
  if ((rc = fused(prod(B, D, F, W.d_out, 0, W_U, 1, W.d_r)))) return rc;
  const float imp_scale = imp_coeff / (float)B;
  auto site_bwd = [&](int si, float* d_ha, float* d_hg) {
    hipLaunchKernelGGL(k_rm_site_bwd, sgrid, dim3(RM_COLS * RM_WAVES), 0, s, W.d_acts, W.hg[si], W.ha[si], W.graw[si], B, C,
                       gt[si], layout, p, imp_scale, d_ha, d_hg, W.gpart + (int64_t)si * Dm.chunks() * RM_GATE * C);
  };
  // A layer's weight gradients; q[i + 1] adds into q[i]'s output where both have the same C.
  auto weight_grads = [&](const F32Prod* q, int n) {
    F32Prod parts[F32_GROUP];
    RmSums sums{};
    int outs = 0;
    int64_t total = 0;
    float* part = W.wpart;
    for (int i = 0; i < n; ++i) {
      const int64_t mn = q[i].M * q[i].N;
      parts[i] = q[i];
      parts[i].C = part;
      if (i == 0 || q[i].C != q[i - 1].C) {
        sums.src[outs] = part;
        sums.dst[outs] = q[i].C;
        sums.n[outs] = mn;
        sums.first[outs++] = total;
        total += mn;
      }
      sums.slabs[outs - 1] += W.splits;
      part += W.splits * mn;
    }
    sums.first[4] = total;
    if (W.splits && gemm_f32_group(parts, n, W.splits, s)) {
      hipLaunchKernelGGL(k_rm_sum_slabs, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, s, sums);
      return (int)PD_OK;
    }
    for (int i = 0; i < n; ++i)
      if (int e = gemm(q[i].M, q[i].N, q[i].K, q[i].A, q[i].lda, 1, q[i].B, q[i].ldb, 0, q[i].C, q[i].ldc,
                       i && q[i].C == q[i - 1].C ? 1.f : 0.f))
        return e;
    return (int)PD_OK;
  };
  for (int l = L - 1; l >= 0; --l) {
    const int si = 2 * l, so = 2 * l + 1;
    // mlp_out: its output adds into the residual
    if ((rc = fused(prod(B, C, D, W.d_r, 0, U[so], 1, W.d_acts)))) return rc;
    site_bwd(so, W.d_ha[1], W.d_hg[1]);
    if ((rc = fused(prod(B, M, C, W.d_ha[1], 0, V[so], 1, W.d_hid, W.hid[l], 2)))) return rc;
    // mlp_in
    if ((rc = fused(prod(B, C, M, W.d_hid, 0, U[si], 1, W.d_acts)))) return rc;
    const bool shared = W.ha[si] == W.hg[si];
    site_bwd(si, W.d_ha[0], shared ? W.d_ha[0] : W.d_hg[0]);
    const F32Prod dw[F32_GROUP] = {
        prod(C, D, B, W.acts[so], 1, W.d_r, 0, grads + G.dU[so]),
        prod(M, C, B, W.hid[l], 1, W.d_ha[1], 0, grads + G.dV[so]),
        prod(M, C, B, W.hidc[l], 1, W.d_hg[1], 0, grads + G.dV[so]),
        prod(C, M, B, W.acts[si], 1, W.d_hid, 0, grads + G.dU[si]),
        prod(D, C, B, W.rm[l], 1, W.d_ha[0], 0, grads + G.dV[si]),
        prod(D, C, B, W.r[l], 1, W.d_hg[0], 0, grads + G.dV[si])};
    if ((rc = weight_grads(dw, shared ? 5 : 6))) return rc;
    if (l > 0) {  // the residual cotangent below this layer
      if ((rc = fused(prod(B, D, C, W.d_ha[0], 0, V[si], 1, W.d_r2, W.d_r)))) return rc;
      std::swap(W.d_r, W.d_r2);
    }
  }
  const int64_t gslots = (int64_t)ns * RM_GATE * C;
  hipLaunchKernelGGL(k_rm_gate_reduce, dim3((unsigned)cdiv(gslots, 256)), dim3(256), 0, s, W.gpart, Dm.chunks(), C,
                     D, M, ns, grads);
  hipLaunchKernelGGL(k_rm_losses, dim3(1), dim3(256), 0, s, W.rec_part, RM_REC_BLOCKS, W.imp_part,
                     (int64_t)ns * nsite_blocks, 1.0 / (double)nout, 1.0 / (double)B, recon_coeff, imp_coeff, losses);
  return check_launch(what);
}

}  // extern "C"
