// Triangle attention (starting / ending node), forward and backward.
//
// Forward, in the module's frame (the transposed pair for the ending node):
//   LN (two-pass) + fused pair-bias projection  -> xn h16, bias[H][M] (log2 e)
//   GEMM xn . [Wq|Wk|Wv|Wg]  (q scaled by D^-1/2 log2 e, +gating_b)  -> qkvg
//   flash attention (mask per row/key, bias per head)               -> o, og, lse
//   GEMM og . Wo + bo, fused residual + shared dropout (+ transposed write)
// Backward replays nothing: the save-set holds LN stats, bias, qkvg, o, lse.
// It runs on the cotangent times the module's scale s (ct_scale): loaded so
// by the first GEMM, divided out by the LayerNorm backward that ends it.
//   GEMM (tbl * dout) . Wo^T, the scale applied as A is loaded (transposed
//        read for the ending node), epilogue through the gate -> dO, dG, Dsum
//   attention backward                    -> dq|dk|dv, d(bias)
//   GEMM dqkvg . [Wq|Wk|Wv|Wg]^T          -> d(xn)
//   LN backward (+ d(bias) . W2d^T) accumulated into din
// Reference: modules.py:675-734 (TriangleAttention), :313-400 (Attention),
// accel.py:13-24 (logit clip); native/triattn_body.cuh:647-1488 (TriAttn).
#include "gemm.h"
#include "lnproj.h"
#include "modules.h"
#include <cmath>
#include <mutex>
#include <string>

namespace bc2n {

namespace {

template <class A>
struct TriAttnSave {
  float *mean, *rstd, *lse;
  h16* bias;
  h16 *qkvg, *o;
  TriAttnSave(A& a, int N, int C, int H) {
    const size_t M = (size_t)N * N;
    mean = a.template take<float>(M);
    rstd = a.template take<float>(M);
    bias = a.template take<h16>((size_t)H * M);
    lse = a.template take<float>((size_t)H * M);
    qkvg = a.template take<h16>(M * 4 * C);
    o = a.template take<h16>(M * C);
  }
};

// ---------------------------------------------------------------------------
// The backward's end in one kernel (C = 128 or 64 channels, H = 4 bias heads):
//   dy  = dqkvg . Wcat^T                       (K = 4C)
//   din = dout + LN'(dy + sum_h dbias_h w2d_h)  (the input LayerNorm's backward)
// with the bias gradient's per-chunk partials added here, in chunk order (the
// sums of the attention backward's reduction, which is not launched).
//
// A workgroup owns 16 RT rows.  Everything it reads -- its rows of dqkvg, x and
// dout, the partials -- is requested before the first wait, and the product
// then waits on weight fragments alone (32 output columns a wave, four K steps
// ahead, one contiguous 1 KB a fragment).  The 128 x 128 GEMM tile with this
// epilogue (same sums, same order) walks K in eight steps of exposed loads
// behind a prologue for the partials, in 32 workgroups at N = 64: 17 us there
// and at N = 128, against 5 and 11 here.
struct DxArgs {
  const h16 *dqkvg, *W;  // [M][4C]; dx_frags
  const float *x, *ln_g, *mean, *rstd, *dres, *dbias, *wb, *gmul;
  float* out;
  long M;
  int nt, nch;  // nt: the transposed pair's rows when > 0; nch: partials [nch][H][M]
};

// Fragment (n32 * 4C/32 + ks) * 2 + jj, lane 16 g + c: column 32 n32 + 16 jj + c
// of Wcat^T at k = 32 ks + 8 g + e.
std::vector<h16> dx_frags(const std::vector<float>& cat, int C) {  // cat: [C][4C]
  std::vector<h16> f((size_t)C * 4 * C);
  size_t o = 0;
  for (int n32 = 0; n32 < C / 32; ++n32)
    for (int ks = 0; ks < 4 * C / 32; ++ks)
      for (int jj = 0; jj < 2; ++jj)
        for (int l = 0; l < 64; ++l)
          for (int e = 0; e < 8; ++e)
            f[o++] = (h16)cat[(size_t)(32 * n32 + 16 * jj + (l & 15)) * 4 * C + 32 * ks + 8 * (l >> 4) + e];
  return f;
}

template <int C, int RT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RT == 2 ? 4 : 3, 4))) void
triattn_dx_kernel(DxArgs a) {
  constexpr int H = 4, K = 4 * C, KS = K / 32, BM = 16 * RT, LDX = K + 8, LDT = C + 4;
  constexpr int WC = C / 32, TI = RT * WC / 4;  // column waves, row tiles a wave
  constexpr int GK = 4, NG = KS / GK;           // K steps a fragment group, groups
  constexpr int LPR = C / 8, RPP = 256 / LPR, PASS = BM / RPP;
  static_assert(RT * WC % 4 == 0 && BM % RPP == 0 && LDT * 4 <= LDX * 2, "tile split");
  __shared__ __attribute__((aligned(16))) char smem[BM * LDX * 2];
  __shared__ __attribute__((aligned(16))) float wbs[C * H], dbs[BM * H];
  h16* xs = reinterpret_cast<h16*>(smem);
  float* T = reinterpret_cast<float*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wc = w % WC, wr = w / WC;
  const long M = a.M, m0 = (long)blockIdx.x * BM;
  const int fr = tid / LPR, c0 = (tid % LPR) * 8;

  // rows past M read row M - 1 and store nothing
  constexpr int XP = BM * K / 8 / 256;
  h16x8 av[XP];
#pragma unroll
  for (int p = 0; p < XP; ++p) {
    const int it = tid + 256 * p;
    av[p] = ld8(a.dqkvg + min(m0 + it / (K / 8), M - 1) * K + (it % (K / 8)) * 8);
  }
  float xv[PASS][8], dr[PASS][8], mu[PASS], rs[PASS];
  long src[PASS];
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const long m = min(m0 + p * RPP + fr, M - 1);
    src[p] = ln_src_row(m, a.nt) * C + c0;
    ld_f8(a.x + src[p], xv[p]);
    ld_f8(a.dres + src[p], dr[p]);
    mu[p] = a.mean[m];
    rs[p] = a.rstd[m];
  }
  for (int i = tid; i < C * H; i += 256) wbs[i] = a.wb[i];
  if (tid < BM * H) {
    // dbs[r][h]: the partials in chunk order, sixteen loads in flight
    const int r = tid % BM, h = tid / BM;
    const long cs = (long)H * M;
    const float* p = a.dbias + (long)h * M + min(m0 + r, M - 1);
    float s = 0.f;
    int c = 0;
    for (; c + 16 <= a.nch; c += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = p[(c + u) * cs];
#pragma unroll
      for (int u = 0; u < 16; ++u) s += v[u];
    }
    for (; c + 4 <= a.nch; c += 4) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = p[(c + u) * cs];
#pragma unroll
      for (int u = 0; u < 4; ++u) s += v[u];
    }
    for (; c < a.nch; ++c) s += p[c * cs];
    dbs[r * H + h] = s;
  }
  h16x8 bf[2][GK][2];
  auto load_b = [&](int grp, h16x8 (&b)[GK][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < GK; ++k)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
        b[k][jj] = ld8(a.W + ((long)((wc * KS + grp * GK + k) * 2 + jj) * 64 + lane) * 8);
  };
  load_b(0, bf[0]);
#pragma unroll
  for (int p = 0; p < XP; ++p) {
    const int it = tid + 256 * p;
    st8(xs + it / (K / 8) * LDX + (it % (K / 8)) * 8, av[p]);
  }
  __syncthreads();

  f32x4 acc[TI][2];
#pragma unroll
  for (int i = 0; i < TI; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int grp = 0; grp < NG; ++grp) {
    if (grp + 1 < NG) load_b(grp + 1, bf[(grp + 1) & 1]);
#pragma unroll
    for (int k = 0; k < GK; ++k)
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const h16x8 xf = ld8(xs + ((wr * TI + i) * 16 + l16) * LDX + (grp * GK + k) * 32 + 8 * g);
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) acc[i][jj] = mfma16x16x32(bf[grp & 1][k][jj], xf, acc[i][jj]);
      }
  }
  __syncthreads();  // every wave is done with xs, which T overlays
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
      *reinterpret_cast<f32x4*>(T + ((wr * TI + i) * 16 + l16) * LDT + 32 * wc + 16 * jj + 4 * g) = acc[i][jj];
  float gm[8];
  ld_f8(a.ln_g + c0, gm);
  const float gs = *a.gmul;
#pragma unroll
  for (int e = 0; e < 8; ++e) gm[e] *= gs;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PASS; ++p) {
    const int r = p * RPP + fr;
    if (m0 + r >= M) continue;  // a row's lanes leave together
    float gv[8];
    ld_f8(T + r * LDT + c0, gv);
    float db[H];
#pragma unroll
    for (int h = 0; h < H; ++h) db[h] = dbs[r * H + h];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) gv[e] += db[h] * wbs[(c0 + e) * H + h];
    float sg = 0.f, sgx = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      xv[p][e] = (xv[p][e] - mu[p]) * rs[p];
      gv[e] *= gm[e];
      sg += gv[e];
      sgx += gv[e] * xv[p][e];
    }
    sg = group_sum<LPR>(sg) * (1.f / C);
    sgx = group_sum<LPR>(sgx) * (1.f / C);
#pragma unroll
    for (int e = 0; e < 8; ++e) dr[p][e] += rs[p] * (gv[e] - sg - xv[p][e] * sgx);
    st_f8(a.out + src[p], dr[p]);
  }
}

// C = 128: up to 144 rows a CU (N = 192: 21.6 us against the GEMM's 25.6); past
// that both run at the memory's rate and the GEMM's loads, spread over its K
// steps, keep it busier (N = 224 29 against 26, 512 150 against 142).
bool triattn_dx_fits(int C, long M) { return C == 64 || M <= 144L * device_cus(); }

void triattn_dx(hipStream_t st, int C, const DxArgs& a) {
  auto go = [&](auto c, auto rt) {
    constexpr int RT = decltype(rt)::value;
    const long nwg = (a.M + 16 * RT - 1) / (16 * RT);
    hipLaunchKernelGGL((triattn_dx_kernel<decltype(c)::value, RT>), dim3((unsigned)nwg), dim3(256), 0,
                       st, a);
  };
  using std::integral_constant;
  if (C == 128) go(integral_constant<int, 128>(), integral_constant<int, 2>());
  // 64 rows beyond: N = 416 49 us against 55
  else if (a.M > 144L * device_cus()) go(integral_constant<int, 64>(), integral_constant<int, 4>());
  else go(integral_constant<int, 64>(), integral_constant<int, 2>());
}

}  // namespace

TriAttnW triattn_weights(WeightStore& ws, const std::string& P) {
  TriAttnW w;
  const HostTensor& qw = ws.host(P + "attention/query_w");
  if (qw.shape.size() != 3) throw std::runtime_error("triattn: query_w must be [C,H,D]");
  w.C = qw.shape[0];
  w.H = qw.shape[1];
  w.D = qw.shape[2];
  const int C = w.C, HD = w.H * w.D;
  if (HD != C) throw std::runtime_error("triattn: H*D must equal C");
  w.ln_g = ws.f32(P + "query_norm/scale");
  w.ln_b = ws.f32(P + "query_norm/offset");
  w.w2d = ws.f32(P + "feat_2d_weights");
  const char* parts[4] = {"attention/query_w", "attention/key_w", "attention/value_w",
                          "attention/gating_w"};
  auto cat = [&]() {
    std::vector<float> c((size_t)C * 4 * HD);
    for (int p = 0; p < 4; ++p) {
      const HostTensor& t = ws.host(P + parts[p]);
      for (int r = 0; r < C; ++r)
        for (int j = 0; j < HD; ++j) c[(size_t)r * 4 * HD + p * HD + j] = t.data[(size_t)r * HD + j];
    }
    return c;
  };
  const bool rows = (C == 128 || C == 64) && w.H == 4;  // the row-tile kernels' widths
  // the dX product's GEMM reads it at the row kernels' C = 128 too, at large M
  if (!rows || C == 128) w.wqkvg = ws.derived<h16>("triattn.wqkvg:" + P, [&] { return to_h16(cat()); });
  const HostTensor& ow = ws.host(P + "attention/output_w");  // [H,D,C]
  if (rows) {
    w.wqkvg_frag = ws.derived<h16>("triattn.wqkvg_frag:" + P, [&] {
      const std::vector<float> c = cat();  // [C][4HD]
      return proj_frags(4 * HD, C, 0, [&](int n, int k) { return c[(size_t)k * 4 * HD + n]; });
    });
    w.dx_frag = ws.derived<h16>("triattn.dx_frag:" + P, [&] { return dx_frags(cat(), C); });
    w.wo_frag = ws.derived<h16>("triattn.wo_frag:" + P, [&] {
      return proj_frags(C, HD, C, [&](int n, int k) { return ow.data[(size_t)k * C + n]; });
    });
    w.wo_bfrag = ws.derived<h16>("triattn.wo_bfrag:" + P, [&] {
      return proj_frags(HD, C, 0, [&](int n, int k) { return ow.data[(size_t)n * C + k]; });
    });
  } else {  // the GEMMs' forms
    w.wqkvg_t = ws.derived<h16>("triattn.wqkvg_t:" + P, [&] {
      std::vector<float> c = cat();
      return transpose_h16(c.data(), C, 4 * HD);
    });
    w.wo = ws.derived<h16>("triattn.wo:" + P, [&] { return to_h16(ow.data); });
    w.wo_t = ws.derived<h16>("triattn.wo_t:" + P, [&] { return transpose_h16(ow.data.data(), HD, C); });
  }
  w.bqkvg = ws.derived<float>("triattn.bqkvg:" + P, [&] {
    std::vector<float> b((size_t)4 * HD, 0.f);
    const HostTensor& gb = ws.host(P + "attention/gating_b");
    for (int j = 0; j < HD; ++j) b[3 * HD + j] = gb.data[j];
    return b;
  });
  w.bo = ws.f32(P + "attention/output_b");
  return w;
}

size_t triattn_save_bytes(int N, int C, int H) {
  Sizer s;
  TriAttnSave<Sizer> plan(s, N, C, H);
  (void)plan;
  return s.off;
}

static void triattn_check(const TriAttnW& w, int N) {
  if (N <= 0 || N % 32 != 0) throw std::runtime_error("triattn: N must be a positive multiple of 32");
  if (w.D != 32 && w.D != 16) throw std::runtime_error("triattn: head width 16 or 32 only");
}


// The forward with its scratch (og [M][HD] and, without the row kernels' weights,
// xn [M][C], binary16) supplied.
static void triattn_fwd_with(hipStream_t st, const TriAttnW& w, bool per_column, int N,
                             const float* pair_in, const float* mask, const float* tbl,
                             float* pair_out, void* save, h16* xn, h16* og) {
  const int C = w.C, H = w.H, HD = w.H * w.D;
  const long M = (long)N * N;
  Carver cv(save);
  TriAttnSave<Carver> sv(cv, N, C, H);
  const float qscale = LOG2E / std::sqrt((float)w.D);
  if (w.wqkvg_frag) {
    lnproj::Args la{};
    la.M = M; la.nt = per_column ? N : 0; la.bn = N; la.nout = 4 * HD;
    la.x = pair_in; la.g = w.ln_g; la.b = w.ln_b; la.wb = w.w2d; la.bscale = LOG2E;
    // xn stays on chip: the backward's LayerNorm term reads pair_in, mean and rstd
    la.xn = nullptr; la.mean = sv.mean; la.rstd = sv.rstd; la.bias = sv.bias; la.W = w.wqkvg_frag;
    KTimed kt(BC2N_TN(C, "triattn.ln_qkvg"), st);
    const EpiScaledCols cols(sv.qkvg, 4L * HD, w.bqkvg, qscale, HD);
    if (C == 128) lnproj::launch<lnproj::In::LN, 128, 4, false>(st, la, cols);
    else lnproj::launch<lnproj::In::LN, 64, 4, false>(st, la, cols);
  } else {
    {
      KTimed kt(BC2N_TN(C, "triattn.ln_fwd"), st);
      ln_fwd_f32(st, pair_in, M, C, per_column ? N : 0, w.ln_g, w.ln_b, xn, sv.mean, sv.rstd,
                 false, H, w.w2d, sv.bias, LOG2E);
    }
    GemmArgs g1;
    g1.M = (int)M; g1.N = 4 * HD; g1.K = C;
    g1.A = xn; g1.a_sm = C; g1.a_sk = 1;
    g1.B = w.wqkvg_t; g1.b_sn = C; g1.b_sk = 1;
    gemm<128, 128>(st, g1, EpiScaledCols(sv.qkvg, 4L * HD, w.bqkvg, qscale, HD),
                   BC2N_TN(C, "triattn.gemm_qkvg"));
  }

  AttnArgs a;
  a.R = N; a.H = H; a.N = N; a.D = w.D;
  a.qkvg = sv.qkvg; a.ld = 4L * HD;
  a.mask = mask;
  a.mask_sr = per_column ? 1 : N;
  a.mask_sk = per_column ? N : 1;
  a.bias = sv.bias;
  a.o = sv.o; a.og = og; a.ldo = HD;
  a.lse = sv.lse;
  attn_fwd(st, a);

  const EpiResidualRows res(pair_in, pair_out, w.bo, tbl, N, C, per_column);
  if (w.wo_frag) {
    lnproj::Args la{};
    la.M = M; la.nout = C; la.xn = og; la.W = w.wo_frag;
    KTimed kt(BC2N_TN(C, "triattn.gemm_out"), st);
    if (C == 128) lnproj::launch<lnproj::In::ROWS, 128, 0, false>(st, la, res);
    else lnproj::launch<lnproj::In::ROWS, 64, 0, false>(st, la, res);
    return;
  }
  GemmArgs g2;
  g2.M = (int)M; g2.N = C; g2.K = HD;
  g2.A = og; g2.a_sm = HD; g2.a_sk = 1;
  g2.B = w.wo_t; g2.b_sn = HD; g2.b_sk = 1;
  gemm<128, 128>(st, g2, res, BC2N_TN(C, "triattn.gemm_out"));
}

void triattn_fwd(hipStream_t st, const TriAttnW& w, bool per_column, int N,
                 const float* pair_in, const float* mask, const float* tbl,
                 float* pair_out, void* save) {
  triattn_check(w, N);
  nonnull(pair_in, "triattn pair_in"); nonnull(mask, "triattn mask");
  nonnull(pair_out, "triattn pair_out"); nonnull(save, "triattn save");
  const int C = w.C, HD = w.H * w.D;
  const long M = (long)N * N;
  Arena& ar = arena();
  std::lock_guard<std::recursive_mutex> lk(ar.lock());
  const size_t nxn = w.wqkvg_frag ? 0 : (size_t)M * C;  // the row kernel keeps xn on chip
  ar.reset(st, nxn * 2 + (size_t)M * HD * 2 + 1024);
  h16* xn = nxn ? ar.take_n<h16>(nxn) : nullptr;
  h16* og = ar.take_n<h16>((size_t)M * HD);
  triattn_fwd_with(st, w, per_column, N, pair_in, mask, tbl, pair_out, save, xn, og);
}

// ------------------------------------------------- the allocation-free variant
// Its scratch (xn and og of triattn_fwd_with, xn's part counted in the limit
// whether the path uses it or not) is this file-scope device array: one copy
// per GPU, allocated with the code object, held until the process ends.  Host
// code never passes `scratch` itself (its host-side name is a stand-in, not a
// device address): the first call on each device looks up the device address
// with hipGetSymbolAddress and keeps it per device.  Calls on one GPU share the
// array, so calls that overlap on one GPU race.
static __device__ __align__(256) unsigned char scratch[TRIATTN_NOALLOC_SCRATCH_BYTES];

static void* scratch_ptr() {
  static std::mutex mu;
  static void* per_dev[64] = {};
  int dev = 0;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= 64) throw std::runtime_error("triattn noalloc: device index out of range");
  std::lock_guard<std::mutex> lk(mu);
  if (!per_dev[dev]) {
    void* p = nullptr;
    hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    per_dev[dev] = p;
  }
  return per_dev[dev];
}

void triattn_fwd_noalloc(hipStream_t st, const TriAttnW& w, bool per_column, int N,
                         const float* pair_in, const float* mask, const float* tbl,
                         float* pair_out, void* save) {
  triattn_check(w, N);
  nonnull(pair_in, "triattn pair_in"); nonnull(mask, "triattn mask");
  nonnull(pair_out, "triattn pair_out"); nonnull(save, "triattn save");
  const int C = w.C, HD = w.H * w.D;
  const size_t M = (size_t)N * N;
  const size_t xn_bytes = (M * C * sizeof(h16) + 255) & ~size_t(255);
  if (xn_bytes + M * HD * sizeof(h16) > TRIATTN_NOALLOC_SCRATCH_BYTES)
    throw std::invalid_argument(
        "triattn_fwd_noalloc: N = " + std::to_string(N) + " needs " +
        std::to_string(xn_bytes + M * HD * sizeof(h16)) + " bytes of scratch; the static scratch holds " +
        std::to_string(TRIATTN_NOALLOC_SCRATCH_BYTES) + " (N <= 256 at C = 128)");
  char* base = static_cast<char*>(scratch_ptr());
  h16* xn = reinterpret_cast<h16*>(base);
  h16* og = reinterpret_cast<h16*>(base + xn_bytes);
  triattn_fwd_with(st, w, per_column, N, pair_in, mask, tbl, pair_out, save, xn, og);
}

void triattn_bwd(hipStream_t st, const TriAttnW& w, bool per_column, int N,
                 const float* pair_in, const float* mask, const float* tbl,
                 const void* save, const float* dout, float* din, CtScale cs) {
  triattn_check(w, N);
  nonnull(pair_in, "triattn pair_in"); nonnull(mask, "triattn mask"); nonnull(save, "triattn save");
  nonnull(dout, "triattn dout"); nonnull(din, "triattn din");
  const int C = w.C, H = w.H, HD = w.H * w.D;
  const long M = (long)N * N;
  Carver cv(const_cast<void*>(save));
  TriAttnSave<Carver> sv(cv, N, C, H);
  AttnBwdArgs b;
  b.rows_per_chunk = attn_rows_per_chunk(N, N, H, w.D);
  const int nch = attn_bwd_nchunk(N, b.rows_per_chunk);
  Arena& ar = arena();
  std::lock_guard<std::recursive_mutex> lk(ar.lock());
  cs = module_scale_lazy(st, cs, dout, M * C);
  // the row kernel below reduces a scale still in partials; the GEMM does not
  const float* sc = w.wo_bfrag ? cs.sc : ct_scale_now(st, cs);
  b.dbias_deferred = w.dx_frag != nullptr;  // the dX product's kernel adds the partials
  const bool sum = nch == 1 || !b.dbias_deferred;  // the whole gradient: one partial, or the reduction's
  Sizer need;
  need.take<h16>((size_t)M * HD);           // dO
  need.take<float>((size_t)H * M);           // Dsum
  need.take<h16>((size_t)M * 4 * HD);       // dqkvg
  need.take<float>((size_t)nch * H * M);     // dbias partials
  if (sum) need.take<float>((size_t)H * M);  // dbias
  if (!w.dx_frag) need.take<float>((size_t)M * C);  // dxn
  ar.reset(st, need.off);
  b.dO = ar.take_n<h16>((size_t)M * HD);
  b.nDsum = ar.take_n<float>((size_t)H * M);
  b.dqkvg = ar.take_n<h16>((size_t)M * 4 * HD);
  b.dbias_part = ar.take_n<float>((size_t)nch * H * M);
  b.dbias = sum ? ar.take_n<float>((size_t)H * M) : nullptr;
  float* dxn = w.dx_frag ? nullptr : ar.take_n<float>((size_t)M * C);

  // d(og) = (tbl * dout) . Wo^T, the dropout scale applied as A is loaded;
  // the epilogue continues through the gate (dO, dG, Dsum)
  auto gate = [&](auto eg) {
    eg.qkvg = sv.qkvg; eg.ld = 4L * HD; eg.o = sv.o; eg.dO = b.dO; eg.dqkvg = b.dqkvg;
    eg.nDsum = b.nDsum; eg.HD = HD; eg.H = H; eg.D = w.D; eg.Ntok = N;
    return eg;
  };
  if (w.wo_bfrag) {
    lnproj::Args la{};
    la.M = M; la.nt = per_column ? N : 0; la.bn = N; la.nout = HD;
    la.x = dout; la.tbl = tbl; la.sc = cs; la.W = w.wo_bfrag;
    KTimed kt(BC2N_TN(C, "triattn.gemm_dout"), st);
    const auto eg = gate(EpiGateBwdT<true>{});
    if (C == 128) lnproj::launch<lnproj::In::SCALED, 128, 0, false>(st, la, eg);
    else lnproj::launch<lnproj::In::SCALED, 64, 0, false>(st, la, eg);
  } else {
    GemmArgs g1;
    g1.M = (int)M; g1.N = HD; g1.K = C;
    g1.a_sm = C; g1.a_sk = 1;
    g1.B = w.wo; g1.b_sn = C; g1.b_sk = 1;
    gemm<64, 128>(st, g1, gate(EpiGateBwd{}), BC2N_TN(C, "triattn.gemm_dout"),
                  ALoadScaledRows{dout, tbl, N, C, per_column, sc});
  }
  b.gate_done = true;

  AttnArgs& a = b.f;
  a.R = N; a.H = H; a.N = N; a.D = w.D;
  a.qkvg = sv.qkvg; a.ld = 4L * HD;
  a.mask = mask;
  a.mask_sr = per_column ? 1 : N;
  a.mask_sk = per_column ? N : 1;
  a.bias = sv.bias;
  a.o = sv.o; a.og = nullptr; a.ldo = HD;
  a.lse = sv.lse;
  b.scale = 1.f / std::sqrt((float)w.D);
  attn_bwd(st, b);

  if (w.dx_frag && triattn_dx_fits(C, M)) {
    DxArgs d{};
    d.dqkvg = b.dqkvg; d.W = w.dx_frag; d.M = M; d.nt = per_column ? N : 0;
    d.x = pair_in; d.ln_g = w.ln_g; d.mean = sv.mean; d.rstd = sv.rstd; d.dres = dout; d.out = din;
    d.dbias = nch == 1 ? b.dbias : b.dbias_part; d.nch = nch;
    d.wb = w.w2d; d.gmul = sc + 1;
    KTimed kt(BC2N_TN(C, "triattn.gemm_dx_ln"), st);
    triattn_dx(st, C, d);
    return;
  }
  GemmArgs g2;
  g2.M = (int)M; g2.N = C; g2.K = 4 * HD;
  g2.A = b.dqkvg; g2.a_sm = 4L * HD; g2.a_sk = 1;
  g2.B = w.wqkvg; g2.b_sn = 4L * HD; g2.b_sk = 1;
  if (C == 128 && H == 4) {
    // the input LayerNorm's backward (with the pair-bias projection's term, its
    // per-chunk partials added in the epilogue) and the residual add
    const float* dbp = nch == 1 ? b.dbias : b.dbias_part;
    gemm<128, 128>(st, g2,
                   EpiLnBwd<4>(pair_in, w.ln_g, sv.mean, sv.rstd, dout, din, M, per_column ? N : 0,
                               dbp, w.w2d, sc + 1, nch),
                   BC2N_TN(C, "triattn.gemm_dx_ln"));
    return;
  }
  gemm<128, 128>(st, g2, EpiStore<float>{dxn, C, 0, nullptr, C}, BC2N_TN(C, "triattn.gemm_dx"));

  KTimed kt(BC2N_TN(C, "triattn.ln_bwd"), st);
  ln_bwd_f32(st, dxn, pair_in, M, C, per_column ? N : 0, w.ln_g, sv.mean, sv.rstd, din, true,
             H, b.dbias, w.w2d, dout, sc + 1);
}

}  // namespace bc2n
