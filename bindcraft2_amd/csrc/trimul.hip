// Triangle multiplication (outgoing 'ikc,jkc->ijc' / incoming 'kjc,kic->ijc'),
// AF2's fused-projection form, forward and backward.
//
// Forward:
//   LN (fast variance) -> xn h16
//   GEMM xn . Wcat  (Wcat = [proj|gate] channel pairs interleaved in 16-wide
//        blocks, then gating_linear), fused epilogue:
//          a = mask * proj * sigmoid(gate)   -> left/right planes [I][N*N] h16
//          g_out = sigmoid(gating_linear)  -> [M][C] h16
//        (xn is kept; the backward recomputes the proj/gate pre-activations)
//   batched MFMA GEMM over the I channels (plane layouts pick out/in)  -> T f32
//     (kept in f32: a sum of N products has no range bound binary16 holds)
//   centre LN (fast variance) reading the channel-major T            -> Tn h16
//   GEMM Tn . Wo + bo, fused: o kept, out = in + tbl * (o * g_out)
// Backward: the exact reverse with the contraction's two transposed GEMMs; the
// projection's gradient comes from a GEMM that recomputes the pre-activations
// from xn and turns them, with d(left|right), into the [proj|gate] columns of
// d(cat) in its epilogue.  The backward runs on the cotangent times the
// module's scale s (ct_scale), applied as the output projection's backward
// loads it and divided out by the input LayerNorm's backward at the end.
// Reference: modules.py:1044-1088 (_fused_triangle_multiplication), :909-919
// (fast-variance LN); native/trimul_body.cuh:1183-1796 (TriMul).
#include "gemm.h"
#include "lnproj.h"
#include "modules.h"

namespace bc2n {

namespace {

// GEMM column of projection channel ch (0..2I) and of its gate.
__host__ __device__ inline int col_proj(int ch) { return (ch / 16) * 32 + ch % 16; }
__host__ __device__ inline int col_gate(int ch) { return (ch / 16) * 32 + 16 + ch % 16; }

// Projection epilogue.  Tiles of the [proj|gate] columns (n0 < 4I) run in
// column mode: the thread of a proj column reads its gate column (16 to the
// right, same tile) from LDS and writes 8 consecutive m of the channel-major
// planes: a = mask * proj * sigmoid(gate) into left/right.  Tiles of
// gating_linear columns run in row mode: g_out[m][c] = sigmoid(acc + b).
struct EpiTrimulProj {
  static constexpr bool kHasCol = true;
  h16 *left, *right;   // [I][M]
  h16* gout;           // [M][C]
  const float *bp, *bg, *bgl, *mask;
  long M;
  int I, C;
  __device__ __forceinline__ bool col_mode(int n0) const { return n0 < 4 * I; }
  __device__ __forceinline__ void col(int, int m, int n, const float (&v)[8], const float* tp,
                                      int ldt) const {
    if ((n & 31) >= 16) return;  // gate column: done by its projection column
    const int ch = (n >> 5) * 16 + (n & 15);
    const float bpv = bp[ch], bgv = bg[ch];
    float mk[8];
    ld_f8(mask + m, mk);
    float pv[8], gv[8], av[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      pv[e] = v[e] + bpv;
      gv[e] = tp[e * ldt + 16] + bgv;
      av[e] = mk[e] * pv[e] * sigmoidf_(gv[e]);
    }
    if (ch < I) st_h8f(left + (long)ch * M + m, av);
    else st_h8f(right + (long)(ch - I) * M + m, av);
  }
  // 8 rows m.. of projection column n and of its gate (lnproj.h)
  __device__ __forceinline__ void cols(long m, int n, float (&pv)[8], const float (&gv)[8]) const {
    const int ch = (n >> 5) * 16 + (n & 15);
    const float bpv = bp[ch], bgv = bg[ch];
    float mk[8];
    ld_f8(mask + m, mk);
#pragma unroll
    for (int e = 0; e < 8; ++e) pv[e] = mk[e] * (pv[e] + bpv) * sigmoidf_(gv[e] + bgv);
    st_h8f((ch < I ? left + (long)ch * M : right + (long)(ch - I) * M) + m, pv);
  }
  __device__ __forceinline__ void row(int, int m, int n, const float (&v)[8]) const {
    const int c = n - 4 * I;
    if (c < 0 || c >= C) return;
    float bb[8], x[8];
    ld_f8(bgl + c, bb);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = sigmoidf_(v[e] + bb[e]);
    st_h8f(gout + (long)m * C + c, x);
  }
};

// o = acc + bo (kept, h16); out[m] = in[m] + tbl[(m%nt)*C+c] * o * g_out
struct EpiTrimulOut : EpiRows {
  const float* in;
  float* out;
  const float* bo;
  const h16* gout;
  h16* osave;
  const float* tbl;
  int nt, C;
  EpiTrimulOut(const float* i, float* o, const float* b, const h16* g, h16* os, const float* t,
               int n, int c)
      : in(i), out(o), bo(b), gout(g), osave(os), tbl(t), nt(n), C(c) {}
  struct Pre {
    float bb[8], tt[8], r[8];
    h16x8 gv;
  };
  __device__ __forceinline__ void load(long m, int n, Pre& p, int) const {
    const long o = m * C + n;
    ld_f8(bo + n, p.bb);
    p.gv = ld8(gout + o);
    if (tbl) ld_f8(tbl + (long)((int)m % nt) * C + n, p.tt);
    ld_f8(in + o, p.r);
  }
  __device__ __forceinline__ void row(long m, int n, const float (&v)[8], Pre& p, int) const {
    const long o = m * C + n;
    float ov[8], gv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) ov[e] = v[e] + p.bb[e];
    st_h8f(osave + o, ov);
#pragma unroll
    for (int e = 0; e < 8; ++e) gv[e] = (float)p.gv[e] * ov[e];
    if (tbl) {
#pragma unroll
      for (int e = 0; e < 8; ++e) gv[e] *= p.tt[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) p.r[e] += gv[e];
    st_f8(out + o, p.r);
  }
  __device__ __forceinline__ void row(int, int m, int n, const float (&v)[8]) const {
    Pre p;
    load(m, n, p, 4);
    row((long)m, n, v, p, 4);
  }
};

template <class A>
struct TriMulSave {
  float *mean, *rstd, *cmean, *crstd, *T;
  h16 *xn, *left, *right, *gout, *osave;
  TriMulSave(A& a, int N, int C, int I) {
    const size_t M = (size_t)N * N;
    mean = a.template take<float>(M);
    rstd = a.template take<float>(M);
    cmean = a.template take<float>(M);
    crstd = a.template take<float>(M);
    T = a.template take<float>(M * I);
    xn = a.template take<h16>(M * C);
    left = a.template take<h16>(M * I);
    right = a.template take<h16>(M * I);
    gout = a.template take<h16>(M * C);
    osave = a.template take<h16>(M * C);
  }
};

// Backward of the projection, as the epilogue of the GEMM xn . Wcat[:, :4I]
// that recomputes the [proj|gate] pre-activations.  Column pass: the thread of
// a proj column takes its gate column (16 to the right) from the staged tile
// and d(left|right) for 8 consecutive m (channel-major), and rewrites both
// columns of the tile with
//   dproj = da * mask * s,  dgate = da * mask * p * s(1-s),  s = sigmoid(gate);
// row pass: the rewritten tile goes to the row-major d(cat) columns.
struct EpiTrimulProjBwd {
  static constexpr bool kHasCol = true;
  static constexpr bool kTwoPhase = true;
  const h16 *dl, *dr;  // [I][M]
  const float *bp, *bg, *mask;
  h16* dcat;           // [M][ldcat]
  long M;
  int I, ldcat;
  __device__ __forceinline__ bool col_mode(int) const { return true; }
  __device__ __forceinline__ void col(int, int m, int n, const float (&v)[8], float* tp,
                                      int ldt) const {
    if ((n & 31) >= 16) return;  // gate column: done by its projection column
    const int ch = (n >> 5) * 16 + (n & 15);
    const float bpv = bp[ch], bgv = bg[ch];
    float mk[8], da[8];
    ld_f8(mask + m, mk);
    ld_h8f((ch < I ? dl + (long)ch * M : dr + (long)(ch - I) * M) + m, da);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float pv = v[e] + bpv;
      const float sg = sigmoidf_(tp[e * ldt + 16] + bgv);
      const float a = da[e] * mk[e];
      tp[e * ldt] = a * sg;
      tp[e * ldt + 16] = a * pv * sg * (1.f - sg);
    }
  }
  __device__ __forceinline__ void row(int, int m, int n, const float (&v)[8]) const {
    st_h8f(dcat + (long)m * ldcat + n, v);
  }
};

// A loader of the output-projection backward GEMM: d = s*tbl*dout (s = *mul,
// the cotangent scale); A = d*g_out (the GEMM operand) and, as a side output,
// dcat[m][off + c] = d * o * g(1-g)   (gating_linear pre-activation grad).
struct ALoadTrimulOut {
  static constexpr bool kDirect = false;
  static constexpr bool kSide = true;
  const float* dout;
  const float* tbl;
  const h16* gout;
  const h16* osave;
  h16* dcat;
  int C, ldcat, off, nt;
  const float* mul;
  __device__ __forceinline__ h16x8 operator()(int, int m, int k) const {
    const long i = (long)m * C + k;
    float d[8], gv[8], ov[8];
    ld_f8(dout + i, d);
    const float sm = *mul;
    if (tbl) {
      float t[8];
      ld_f8(tbl + (long)(m % nt) * C + k, t);
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] *= t[e] * sm;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) d[e] *= sm;
    }
    ld_h8f(gout + i, gv);
    ld_h8f(osave + i, ov);
    h16x8 a, dc;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a[e] = f2h_sat(d[e] * gv[e]);
      dc[e] = f2h_sat(d[e] * ov[e] * gv[e] * (1.f - gv[e]));
    }
    st8(dcat + (long)m * ldcat + off + k, dc);
    return a;
  }
};

// The centre LayerNorm's backward fused into the d(tn) product (I = C): the
// staged tile of d(tn) rows is the dy of ln_bwd_cm, normalised with the same
// sums in the same order (eight parts a row, C / 8 consecutive channels each),
// and written channel-major in binary16, so d(tn) never reaches memory.  A
// lane is a row and a wave one or two parts, so that the channel-major T is
// read (before the product) and dT written 64 or 32 rows of a channel at a
// time; the parts' sums meet in LDS.
template <int C_>
struct EpiCmLnBwd : EpiRows {
  static constexpr int C = C_, P = 8, CPL = C / P;
  const float *x, *gamma, *mean, *rstd;  // x: channel-major [C][M]
  h16* dx;                               // channel-major [C][M]
  long M;
  struct Tile {
    float x[2 * CPL], mu, rs;
  };
  template <int BM>
  static constexpr int parts() { return P * BM / 256; }  // a thread's parts
  template <int BM>
  __device__ __forceinline__ void load(long m0, Tile& t, int tid) const {
    const long m = min(m0 + tid % BM, M - 1);  // rows past M: never stored
#pragma unroll
    for (int k = 0; k < parts<BM>(); ++k)
#pragma unroll
      for (int e = 0; e < CPL; ++e)
        t.x[k * CPL + e] = x[(long)((tid / BM + 256 / BM * k) * CPL + e) * M + m];
    t.mu = mean[m];
    t.rs = rstd[m];
  }
  template <int BM>
  __device__ __forceinline__ void tile(long m0, const float* T, int ldt, int tid, Tile& t) const {
    __shared__ float red[2][P][BM];
    const int r = tid % BM;
    float g[parts<BM>() * CPL];
#pragma unroll
    for (int k = 0; k < parts<BM>(); ++k) {
      const int part = tid / BM + 256 / BM * k;
      float sg = 0.f, sgx = 0.f;
#pragma unroll
      for (int e0 = 0; e0 < CPL; e0 += 4) {
        const float4 d = *reinterpret_cast<const float4*>(T + r * ldt + part * CPL + e0);
        const float dv[4] = {d.x, d.y, d.z, d.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = k * CPL + e0 + q;
          t.x[i] = (t.x[i] - t.mu) * t.rs;
          g[i] = dv[q] * gamma[part * CPL + e0 + q];
          sg += g[i];
          sgx += g[i] * t.x[i];
        }
      }
      red[0][part][r] = sg;
      red[1][part][r] = sgx;
    }
    __syncthreads();
    auto total = [&](int q) {  // group_sum<8>'s pairs
      float v[P];
#pragma unroll
      for (int p = 0; p < P; ++p) v[p] = red[q][p][r];
      return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    };
    const float sg = total(0) / C, sgx = total(1) / C;
    if (m0 + r >= M) return;
#pragma unroll
    for (int k = 0; k < parts<BM>(); ++k)
#pragma unroll
      for (int e = 0; e < CPL; ++e) {
        const int i = k * CPL + e;
        dx[(long)((tid / BM + 256 / BM * k) * CPL + e) * M + m0 + r] =
            f2h_sat(t.rs * (g[i] - sg - t.x[i] * sgx));
      }
  }
};

// ---------------------------------------------------------------------------
// The backward's tail in one kernel (I = C, C = 128 or 64):
//
//   P   = xn . Wcat[:, :4I]                    (recompute, K = C)
//   d(cat)[:, :4I] from P, d(left|right), mask (the EpiTrimulProjBwd formulas)
//   dy  = d(cat) . Wcat^T                      (K = 4I + C; the last C columns
//                                               of d(cat) come from memory)
//   din = dout + LN'(dy)                       (the input LayerNorm's backward)
//
// A workgroup owns 16 RT rows: its xn tile (k order permuted inside 32-blocks,
// below) and its d(left|right) tile (channel-major, as in memory) are in LDS
// before the first product, so the chunk loop waits on memory for weight
// fragments alone, and those are loaded a chunk ahead.  The [proj|gate]
// columns are made and consumed 128 at a time.  The four waves split the
// columns of both products over all rows (every weight fragment is read once
// a workgroup, straight from memory, one contiguous 1 KB a wave):
//
//  GEMM1, transposed (the weights as the first MFMA operand): wave w makes
//    the chunk's 32-column block w, 16 proj columns and their 16 gates, and
//    ends with row l%16 and columns 4g..4g+3 of both, so d(cat) is formed in
//    registers, with d(left|right) from one transposed LDS read (channels
//    4g..4g+3 of row l%16).  The 8 values {proj 4g..4g+3, gate 4g..4g+3} are
//    one k-slot set of a 32-deep MFMA step: one 16-byte LDS store, one
//    16-byte read as GEMM2's operand.
//  GEMM2, transposed: wave w accumulates C / 4 output channels.
//
// Both products' K order and the row sums' order are those of the kernel this
// one replaced (128 rows a workgroup, the waves splitting rows, the weights
// streamed through LDS in ten barriers), whose bits it keeps.  That one was a
// chain of ten exposed prefetches in too few workgroups: 32 us at N = 128
// (128 workgroups) and 45 us at N = 224.
template <int C_, int RT_>
struct Tail {
  static constexpr int C = C_, I = C_, NC = 4 * I + C, RT = RT_, BM = 16 * RT;
  static constexpr int KS = C / 32;         // GEMM1's 32-deep steps
  static constexpr int NPG = 4 * I / 128;   // chunks of [proj|gate] columns
  static constexpr int JJ = C / 64;         // 16-channel output tiles a wave
  static constexpr int LDX = C + 8, LDH = 128 + 8, LDT = C + 4;
  static constexpr int LDD = BM % 32 == 16 ? BM : BM + 16;  // 16 mod 32: transposed reads
  static constexpr int XS = BM * LDX * 2, HS = BM * LDH * 2, T = BM * LDT * 4;
  static constexpr int MAIN = XS + HS > T ? XS + HS : T;  // xs, hs; the f32 output tile over both
  static constexpr int DS = 2 * I * LDD * 2;
};

struct TailArgs {
  const h16* xn;       // [M][C]
  const h16 *w1, *w2;  // tail_frags1 / tail_frags2
  const h16 *dl, *dr;  // [I][M]
  const h16* dcg;      // [M][C]: d(cat)'s gating_linear columns
  const float *bp, *bg, *mask;
  const float *x, *ln_g, *mean, *rstd, *dres;
  const float* gmul;   // inverse cotangent scale (device scalar)
  float* out;
  long M;
};

// The k order of the LDS tiles and weight fragments: inside a 32-block lane
// group g's 8 values are k = {4g..4g+3, 16+4g..16+4g+3}.
__host__ __device__ inline int tail_k(int g, int e) { return e < 4 ? 4 * g + e : 12 + 4 * g + e; }

// 8 consecutive k (k8 % 8 == 0) of one row into its permuted 32-block.
__device__ __forceinline__ void tail_put(h16* row, int k8, h16x8 v) {
  const int q = (k8 >> 3) & 3;
  h16* p = row + (k8 & ~31) + 16 * (q & 1) + 4 * (q >> 1);
  *reinterpret_cast<h16x4*>(p) = h16x4{v[0], v[1], v[2], v[3]};
  *reinterpret_cast<h16x4*>(p + 8) = h16x4{v[4], v[5], v[6], v[7]};
}

template <int C_, int RT_>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void trimul_tail_kernel(
    TailArgs a) {
  using K = Tail<C_, RT_>;
  constexpr int C = K::C, I = K::I, RT = K::RT, BM = K::BM, JJ = K::JJ, KS = K::KS;
  __shared__ __attribute__((aligned(16))) char smem[K::MAIN];
  __shared__ __attribute__((aligned(16))) h16 ds[2 * I * K::LDD];
  __shared__ __attribute__((aligned(16))) float bps[2 * I], bgs[2 * I];
  h16* xs = reinterpret_cast<h16*>(smem);
  h16* hs = reinterpret_cast<h16*>(smem + K::XS);
  float* T = reinterpret_cast<float*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long M = a.M, nwg = (M + BM - 1) / BM;
  // neighbours share lines of d(left|right)'s planes: one XCD a range of rows
  const long blk = xcd_block(nwg);
  if (blk >= nwg) return;
  const long m0 = blk * BM;

  h16x8 b1[KS][2], b2[4][JJ];
  auto load_b1 = [&](int j) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        b1[ks][q] = ld8(a.w1 + ((long)(((j * 4 + w) * 2 + q) * KS + ks) * 64 + lane) * 8);
  };
  auto load_b2 = [&](int j, int nb) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int jj = 0; jj < JJ; ++jj)
        if (b < nb) b2[b][jj] = ld8(a.w2 + ((long)(((j * 4 + b) * 4 + w) * JJ + jj) * 64 + lane) * 8);
  };
  // a [BM][C] tile, 16 bytes a piece; rows past M read row M - 1 (their
  // results are never stored)
  constexpr int XP = (BM * C / 8 + 255) / 256;
  auto load_rows = [&](const h16* src, h16x8 (&v)[XP]) {
#pragma unroll
    for (int p = 0; p < XP; ++p) {
      const int it = min(tid + 256 * p, BM * C / 8 - 1);
      v[p] = ld8(src + min(m0 + it / (C / 8), M - 1) * C + (it % (C / 8)) * 8);
    }
  };
  auto put_rows = [&](const h16x8 (&v)[XP]) {
#pragma unroll
    for (int p = 0; p < XP; ++p) {
      const int it = tid + 256 * p;
      if (it < BM * C / 8) tail_put(xs + it / (C / 8) * K::LDX, (it % (C / 8)) * 8, v[p]);
    }
  };

  // front: every load of both tiles before the first store
  float mk[RT];
  h16x8 xv[XP];
  {
    constexpr int DP = (2 * I * (BM / 8) + 255) / 256;
    h16x8 dv[DP];
    load_rows(a.xn, xv);
#pragma unroll
    for (int p = 0; p < DP; ++p) {
      const int it = min(tid + 256 * p, 2 * I * (BM / 8) - 1), ch = it / (BM / 8);
      const h16* plane = ch < I ? a.dl + (long)ch * M : a.dr + (long)(ch - I) * M;
      dv[p] = ld8(plane + min(m0 + (it % (BM / 8)) * 8, M - 8));
    }
    float bpv = 0.f, bgv = 0.f;
    if (tid < 2 * I) {
      bpv = a.bp[tid];
      bgv = a.bg[tid];
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) mk[i] = a.mask[min(m0 + i * 16 + l16, M - 1)];
    load_b1(0);
    load_b2(0, 4);
    put_rows(xv);
#pragma unroll
    for (int p = 0; p < DP; ++p) {
      const int it = tid + 256 * p;
      if (it < 2 * I * (BM / 8)) st8(ds + it / (BM / 8) * K::LDD + (it % (BM / 8)) * 8, dv[p]);
    }
    if (tid < 2 * I) {
      bps[tid] = bpv;
      bgs[tid] = bgv;
    }
  }
  __syncthreads();

  f32x4 acc2[RT][JJ];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj) acc2[i][jj] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int j = 0; j < K::NPG; ++j) {
    // GEMM1: proj and gate columns of channels 16 (4j + w) + 4g + r, row i*16 + l16
    f32x4 acc1[RT][2];
#pragma unroll
    for (int i = 0; i < RT; ++i) acc1[i][0] = acc1[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const h16x8 xf = ld8(xs + (i * 16 + l16) * K::LDX + ks * 32 + 8 * g);
#pragma unroll
        for (int q = 0; q < 2; ++q) acc1[i][q] = mfma16x16x32(b1[ks][q], xf, acc1[i][q]);
      }
    if (j + 1 < K::NPG) load_b1(j + 1);
    else load_rows(a.dcg, xv);  // the gating_linear columns take xs next
    // d(proj) = a * sigmoid(gate), d(gate) = a * proj * s (1 - s), a = d(act) * mask
    const int ch = 16 * (4 * j + w) + 4 * g;
    const float4 p4 = *reinterpret_cast<const float4*>(bps + ch);
    const float4 g4 = *reinterpret_cast<const float4*>(bgs + ch);
    const float bpv[4] = {p4.x, p4.y, p4.z, p4.w}, bgv[4] = {g4.x, g4.y, g4.z, g4.w};
    h16x8 f[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const h16x4 da = gemm_tr4(ds, K::LDD, 16 * (4 * j + w), i * 16, lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pv = acc1[i][0][r] + bpv[r];
        const float sg = sigmoidf_(acc1[i][1][r] + bgv[r]);
        const float ad = (float)da[r] * mk[i];
        f[i][r] = f2h_sat(ad * sg);
        f[i][4 + r] = f2h_sat(ad * pv * sg * (1.f - sg));
      }
    }
    if (j > 0) __syncthreads();  // the previous chunk's GEMM2 is done with hs
#pragma unroll
    for (int i = 0; i < RT; ++i) st8(hs + (i * 16 + l16) * K::LDH + 32 * w + 8 * g, f[i]);
    __syncthreads();
    if (j == K::NPG - 1) put_rows(xv);  // every wave is past its last read of xn
    // GEMM2: output channels 16 (JJ w + jj) + 4g + r of row i*16 + l16
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const h16x8 af = ld8(hs + (i * 16 + l16) * K::LDH + b * 32 + 8 * g);
#pragma unroll
        for (int jj = 0; jj < JJ; ++jj) acc2[i][jj] = mfma16x16x32(b2[b][jj], af, acc2[i][jj]);
      }
    load_b2(j + 1, j + 1 < K::NPG ? 4 : KS);
  }
  __syncthreads();  // the gating_linear columns are in xs

  // the LayerNorm's rows, behind the last product: lane part g of row `row`
  // takes channels 16j + 4g + r
  constexpr int NP = (4 * BM + 255) / 256;  // passes of 64 rows
  float4 xr[NP][C / 16], dr[NP][C / 16];
  float mu[NP], rs[NP];
  const int part = tid & 3;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const long m = min(m0 + p * 64 + (tid >> 2), M - 1);
#pragma unroll
    for (int j = 0; j < C / 16; ++j) {
      xr[p][j] = *reinterpret_cast<const float4*>(a.x + m * C + 16 * j + 4 * part);
      dr[p][j] = *reinterpret_cast<const float4*>(a.dres + m * C + 16 * j + 4 * part);
    }
    mu[p] = a.mean[m];
    rs[p] = a.rstd[m];
  }
#pragma unroll
  for (int b = 0; b < KS; ++b)
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const h16x8 af = ld8(xs + (i * 16 + l16) * K::LDX + b * 32 + 8 * g);
#pragma unroll
      for (int jj = 0; jj < JJ; ++jj) acc2[i][jj] = mfma16x16x32(b2[b][jj], af, acc2[i][jj]);
    }
  __syncthreads();  // every wave is done with xs and hs, which T overlays
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int jj = 0; jj < JJ; ++jj)
      *reinterpret_cast<f32x4*>(T + (i * 16 + l16) * K::LDT + 16 * (JJ * w + jj) + 4 * g) = acc2[i][jj];
  __syncthreads();

  // ---- LayerNorm backward + residual, four lanes a row
  const float gs = *a.gmul;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int row = p * 64 + (tid >> 2);
    const long m = m0 + row;
    if (row >= BM || m >= M) continue;  // the row's four lanes leave together
    float xh[C / 16][4], gg[C / 16][4];
    float sg = 0.f, sgx = 0.f;
#pragma unroll
    for (int j = 0; j < C / 16; ++j) {
      const int c = 16 * j + 4 * part;
      const float4 dy = *reinterpret_cast<const float4*>(T + row * K::LDT + c);
      const float4 gm = *reinterpret_cast<const float4*>(a.ln_g + c);
      const float xa[4] = {xr[p][j].x, xr[p][j].y, xr[p][j].z, xr[p][j].w};
      const float ga[4] = {gm.x, gm.y, gm.z, gm.w}, da[4] = {dy.x, dy.y, dy.z, dy.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        xh[j][r] = (xa[r] - mu[p]) * rs[p];
        gg[j][r] = da[r] * (ga[r] * gs);
        sg += gg[j][r];
        sgx += gg[j][r] * xh[j][r];
      }
    }
    sg = group_sum<4>(sg) * (1.f / C);
    sgx = group_sum<4>(sgx) * (1.f / C);
#pragma unroll
    for (int j = 0; j < C / 16; ++j) {
      float4 o;
      o.x = dr[p][j].x + rs[p] * (gg[j][0] - sg - xh[j][0] * sgx);
      o.y = dr[p][j].y + rs[p] * (gg[j][1] - sg - xh[j][1] * sgx);
      o.z = dr[p][j].z + rs[p] * (gg[j][2] - sg - xh[j][2] * sgx);
      o.w = dr[p][j].w + rs[p] * (gg[j][3] - sg - xh[j][3] * sgx);
      *reinterpret_cast<float4*>(a.out + m * C + 16 * j + 4 * part) = o;
    }
  }
}

template <int C>
void trimul_tail(hipStream_t st, const TailArgs& a) {
  constexpr int RT = 3;
  const long nwg = (a.M + 16 * RT - 1) / (16 * RT);
  hipLaunchKernelGGL((trimul_tail_kernel<C, RT>), dim3(xcd_grid(nwg)), dim3(256), 0, st, a);
}

// The tail's weight fragments, 64 lanes x 8 binary16 each, lane 16 g + c, from
// Wcat [C][NC]: GEMM1's ((j*4 + w)*2 + q)*KS + ks holds column 128j + 32w + 16q
// + c at k = 32 ks + tail_k(g, e); GEMM2's (b*4 + w)*JJ + jj holds channel
// 16 (JJ w + jj) + c at k = 32b + tail_k(g, e).
std::vector<h16> tail_frags1(const std::vector<float>& cat, int C) {
  const int NC = 5 * C, KS = C / 32;
  std::vector<h16> f((size_t)4 * C * C);
  size_t o = 0;
  for (int jwq = 0; jwq < 4 * C / 16; ++jwq)
    for (int ks = 0; ks < KS; ++ks)
      for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e)
          f[o++] = (h16)cat[(size_t)(32 * ks + tail_k(l >> 4, e)) * NC + 16 * jwq + (l & 15)];
  return f;
}
std::vector<h16> tail_frags2(const std::vector<float>& cat, int C) {
  const int NC = 5 * C;
  std::vector<h16> f((size_t)NC * C);
  size_t o = 0;
  for (int b = 0; b < NC / 32; ++b)
    for (int wj = 0; wj < C / 16; ++wj)
      for (int l = 0; l < 64; ++l)
        for (int e = 0; e < 8; ++e)
          f[o++] = (h16)cat[(size_t)(16 * wj + (l & 15)) * NC + 32 * b + tail_k(l >> 4, e)];
  return f;
}

}  // namespace

TriMulW trimul_weights(WeightStore& ws, const std::string& P) {
  TriMulW w;
  const HostTensor& pw = ws.host(P + "projection/weights");  // [C, 2I]
  w.C = pw.shape[0];
  w.I = pw.shape[1] / 2;
  const int C = w.C, I = w.I, NC = 4 * I + C;
  if (I % 16 != 0 || C % 64 != 0) throw std::runtime_error("trimul: widths must be multiples of 16/64");
  w.ln_g = ws.f32(P + "left_norm_input/scale");
  w.ln_b = ws.f32(P + "left_norm_input/offset");
  w.cn_g = ws.f32(P + "center_norm/scale");
  w.cn_b = ws.f32(P + "center_norm/offset");
  w.bp = ws.f32(P + "projection/bias");
  w.bg = ws.f32(P + "gate/bias");
  w.bgl = ws.f32(P + "gating_linear/bias");
  w.bo = ws.f32(P + "output_projection/bias");
  // Wcat [C][NC] in GEMM column order
  auto cat = [&]() {
    const HostTensor& gw = ws.host(P + "gate/weights");
    const HostTensor& lw = ws.host(P + "gating_linear/weights");
    std::vector<float> c((size_t)C * NC);
    for (int r = 0; r < C; ++r) {
      for (int ch = 0; ch < 2 * I; ++ch) {
        c[(size_t)r * NC + col_proj(ch)] = pw.data[(size_t)r * 2 * I + ch];
        c[(size_t)r * NC + col_gate(ch)] = gw.data[(size_t)r * 2 * I + ch];
      }
      for (int j = 0; j < C; ++j) c[(size_t)r * NC + 4 * I + j] = lw.data[(size_t)r * C + j];
    }
    return c;
  };
  const HostTensor& ow = ws.host(P + "output_projection/weights");  // [I, C]
  if (I == C && (C == 128 || C == 64)) {  // the row-tile kernels' widths and forms
    w.wcat_frag = ws.derived<h16>("trimul.wcat_frag:" + P, [&] {
      const std::vector<float> c = cat();  // [C][NC]
      return proj_frags(NC, C, 4 * I, [&](int n, int k) { return c[(size_t)k * NC + n]; });
    });
    w.tail_w1 = ws.derived<h16>("trimul.tail_w1:" + P, [&] { return tail_frags1(cat(), C); });
    w.tail_w2 = ws.derived<h16>("trimul.tail_w2:" + P, [&] { return tail_frags2(cat(), C); });
    w.wo_frag = ws.derived<h16>("trimul.wo_frag:" + P, [&] {
      return proj_frags(C, I, 0, [&](int n, int k) { return ow.data[(size_t)k * C + n]; });
    });
    w.wo_bfrag = ws.derived<h16>("trimul.wo_bfrag:" + P, [&] {
      return proj_frags(I, C, 0, [&](int n, int k) { return ow.data[(size_t)n * C + k]; });
    });
  } else {  // the GEMMs'
    w.wcat = ws.derived<h16>("trimul.wcat:" + P, [&] { return to_h16(cat()); });
    w.wcat_t = ws.derived<h16>("trimul.wcat_t:" + P, [&] {
      std::vector<float> c = cat();
      return transpose_h16(c.data(), C, NC);
    });
    w.wo = ws.derived<h16>("trimul.wo:" + P, [&] { return to_h16(ow.data); });
    w.wo_t = ws.derived<h16>("trimul.wo_t:" + P, [&] { return transpose_h16(ow.data.data(), I, C); });
  }
  return w;
}

size_t trimul_save_bytes(int N, int C, int I) {
  Sizer s;
  TriMulSave<Sizer> plan(s, N, C, I);
  (void)plan;
  return s.off;
}

static void trimul_check(int N) {
  if (N <= 0 || N % 32 != 0) throw std::runtime_error("trimul: N must be a positive multiple of 32");
}

// One batched contraction (operands described by `g`, one channel plane per
// batch entry): the dedicated kernel for N <= 256, the tiled GEMM beyond, in
// 128 x 128 tiles (64 x 64 tiles read every operand row of a plane from 8
// tiles: 1 GB of L2 traffic per contraction at N = 512).
template <class OutT>
static void contract(hipStream_t st, const GemmArgs& g, OutT* C, const char* name) {
  {
    KTimed kt(name, st);
    float* cf = nullptr;
    h16* cb = nullptr;
    if constexpr (sizeof(OutT) == 4) cf = C;
    else cb = C;
    if (trimul_contract(st, g.M, g.batch, g.A, g.a_sk == 1, g.B, g.b_sk == 1, cf, cb)) return;
  }
  gemm<128, 128>(st, g, EpiStore<OutT>{C, g.N, (long)g.M * g.N, nullptr, g.N}, name);
}

// Contraction operand layouts for one channel plane (row-major N x N).
static void contraction_fwd(hipStream_t st, bool outgoing, int N, int I, const h16* L,
                            const h16* R, float* T) {
  const long M = (long)N * N;
  GemmArgs g;
  g.M = N; g.N = N; g.K = N; g.batch = I;
  if (outgoing) {  // T[i][j] = sum_k L[i][k] R[j][k]
    g.A = L; g.a_sm = N; g.a_sk = 1;
    g.B = R; g.b_sn = N; g.b_sk = 1;
  } else {         // T[i][j] = sum_k R[k][i] L[k][j]
    g.A = R; g.a_sm = 1; g.a_sk = N;
    g.B = L; g.b_sn = 1; g.b_sk = N;
  }
  g.a_sb = M; g.b_sb = M;
  contract<float>(st, g, T, BC2N_TN(I, "trimul.contract_fwd"));
}

void trimul_fwd(hipStream_t st, const TriMulW& w, bool outgoing, int N, const float* pair_in,
                const float* mask, const float* tbl, float* pair_out, void* save) {
  trimul_check(N);
  nonnull(pair_in, "trimul pair_in"); nonnull(mask, "trimul mask");
  nonnull(pair_out, "trimul pair_out"); nonnull(save, "trimul save");
  const int C = w.C, I = w.I, NC = 4 * I + C;
  const long M = (long)N * N;
  Carver cv(save);
  TriMulSave<Carver> sv(cv, N, C, I);
  Arena& ar = arena();
  std::lock_guard<std::recursive_mutex> lk(ar.lock());
  h16* xn = sv.xn;
  h16* tn = nullptr;  // the row kernel keeps it on chip
  if (!w.wo_frag) {
    ar.reset(st, (size_t)M * I * 2 + 1024);
    tn = ar.take_n<h16>((size_t)M * I);
  }
  const EpiTrimulProj proj{sv.left, sv.right, sv.gout, w.bp, w.bg, w.bgl, mask, M, I, C};
  if (w.wcat_frag) {
    lnproj::Args la{};
    la.M = M; la.nt = 0; la.bn = N; la.nout = NC;
    la.x = pair_in; la.g = w.ln_g; la.b = w.ln_b;
    la.xn = xn; la.mean = sv.mean; la.rstd = sv.rstd; la.W = w.wcat_frag;
    KTimed kt(BC2N_TN(C, "trimul.ln_proj"), st);
    if (C == 128) lnproj::launch<lnproj::In::LN, 128, 0, true>(st, la, proj);
    else lnproj::launch<lnproj::In::LN, 64, 0, true>(st, la, proj);
  } else {
    {
      KTimed kt(BC2N_TN(C, "trimul.ln_fwd"), st);
      ln_fwd_f32(st, pair_in, M, C, 0, w.ln_g, w.ln_b, xn, sv.mean, sv.rstd, true, 0, nullptr,
                 nullptr);
    }
    GemmArgs g1;
    g1.M = (int)M; g1.N = NC; g1.K = C;
    g1.A = xn; g1.a_sm = C; g1.a_sk = 1;
    g1.B = w.wcat_t; g1.b_sn = C; g1.b_sk = 1;
    gemm<128, 128>(st, g1, proj, BC2N_TN(C, "trimul.gemm_proj"));
  }
  contraction_fwd(st, outgoing, N, I, sv.left, sv.right, sv.T);
  const EpiTrimulOut out(pair_in, pair_out, w.bo, sv.gout, sv.osave, tbl, N, C);
  if (w.wo_frag) {
    // the centre norm and the output projection in one kernel: the normalised
    // rows stay on chip (the same statistics and binary16 rows as ln_fwd_cm)
    lnproj::Args la{};
    la.M = M; la.nout = C; la.x = sv.T; la.g = w.cn_g; la.b = w.cn_b;
    la.mean = sv.cmean; la.rstd = sv.crstd; la.W = w.wo_frag;
    KTimed kt(BC2N_TN(C, "trimul.ln_out"), st);
    if (C == 128) lnproj::launch<lnproj::In::CM, 128, 0, true>(st, la, out);
    else lnproj::launch<lnproj::In::CM, 64, 0, true>(st, la, out);
    return;
  }
  {
    KTimed kt(BC2N_TN(C, "trimul.ln_center"), st);
    ln_fwd_cm(st, sv.T, M, I, w.cn_g, w.cn_b, tn, sv.cmean, sv.crstd, true);
  }
  GemmArgs g2;
  g2.M = (int)M; g2.N = C; g2.K = I;
  g2.A = tn; g2.a_sm = I; g2.a_sk = 1;
  g2.B = w.wo_t; g2.b_sn = I; g2.b_sk = 1;
  gemm<128, 128>(st, g2, out, BC2N_TN(C, "trimul.gemm_out"));
}

void trimul_bwd(hipStream_t st, const TriMulW& w, bool outgoing, int N, const float* pair_in,
                const float* mask, const float* tbl, const void* save, const float* dout,
                float* din, CtScale cs) {
  trimul_check(N);
  nonnull(pair_in, "trimul pair_in"); nonnull(mask, "trimul mask"); nonnull(save, "trimul save");
  nonnull(dout, "trimul dout"); nonnull(din, "trimul din");
  const int C = w.C, I = w.I, NC = 4 * I + C;
  const long M = (long)N * N;
  Carver cv(const_cast<void*>(save));
  TriMulSave<Carver> sv(cv, N, C, I);
  Arena& ar = arena();
  std::lock_guard<std::recursive_mutex> lk(ar.lock());
  cs = module_scale_lazy(st, cs, dout, M * C);
  // I = C = 128 or 64: the tail kernel keeps d(cat)'s [proj|gate] columns on
  // chip; only its gating_linear columns ([M][C]) go through memory
  const bool fused = w.tail_w1 != nullptr;
  // the row kernel below reduces a scale still in partials; the GEMM does not
  const float* sc = fused ? cs.sc : ct_scale_now(st, cs);
  const int ldcat = fused ? C : NC, off = fused ? 0 : 4 * I;
  Sizer need;
  need.take<h16>((size_t)M * ldcat);  // dcat
  if (!fused) need.take<float>((size_t)M * I);  // dTn
  need.take<h16>((size_t)M * I);   // dT
  need.take<h16>((size_t)M * I);   // dL
  need.take<h16>((size_t)M * I);   // dR
  if (!fused) need.take<float>((size_t)M * C);  // dxn
  ar.reset(st, need.off);
  h16* dcat = ar.take_n<h16>((size_t)M * ldcat);
  float* dtn = fused ? nullptr : ar.take_n<float>((size_t)M * I);
  h16* dT = ar.take_n<h16>((size_t)M * I);
  h16* dL = ar.take_n<h16>((size_t)M * I);
  h16* dR = ar.take_n<h16>((size_t)M * I);
  float* dxn = fused ? nullptr : ar.take_n<float>((size_t)M * C);

  // d(tn) = (tbl*dout*g_out) . Wo^T, the operand built as the product loads
  // it, which also writes the gating_linear columns of dcat
  if (fused) {
    // the centre norm's backward in the epilogue: dT straight from d(tn)
    lnproj::Args la{};
    la.M = M; la.bn = N; la.nout = I; la.x = dout; la.tbl = tbl; la.sc = cs;
    la.gout = sv.gout; la.osave = sv.osave; la.dcat = dcat; la.W = w.wo_bfrag;
    KTimed kt(BC2N_TN(C, "trimul.gemm_dout_ln"), st);
    auto go = [&](auto ep) {
      ep.x = sv.T; ep.gamma = w.cn_g; ep.mean = sv.cmean; ep.rstd = sv.crstd; ep.dx = dT; ep.M = M;
      lnproj::launch<lnproj::In::GATED, decltype(ep)::C, 0, false>(st, la, ep);
    };
    if (C == 128) go(EpiCmLnBwd<128>{});
    else go(EpiCmLnBwd<64>{});
  } else {
    GemmArgs g1;
    g1.M = (int)M; g1.N = I; g1.K = C;
    g1.a_sm = C; g1.a_sk = 1;
    g1.B = w.wo; g1.b_sn = C; g1.b_sk = 1;
    gemm<64, 128>(st, g1, EpiStore<float>{dtn, I, 0, nullptr, I}, BC2N_TN(C, "trimul.gemm_dout"),
                  ALoadTrimulOut{dout, tbl, sv.gout, sv.osave, dcat, C, ldcat, off, N, sc});
    KTimed kt(BC2N_TN(C, "trimul.ln_center_bwd"), st);
    ln_bwd_cm(st, dtn, sv.T, M, I, w.cn_g, sv.cmean, sv.crstd, dT);
  }
  {
    GemmArgs a, b;
    a.M = N; a.N = N; a.K = N; a.batch = I; a.a_sb = M; a.b_sb = M;
    b = a;
    if (outgoing) {
      // dL[i][k] = sum_j dT[i][j] R[j][k]
      a.A = dT; a.a_sm = N; a.a_sk = 1;
      a.B = sv.right; a.b_sn = 1; a.b_sk = N;
      // dR[j][k] = sum_i dT[i][j] L[i][k]
      b.A = dT; b.a_sm = 1; b.a_sk = N;
      b.B = sv.left; b.b_sn = 1; b.b_sk = N;
    } else {
      // dL[k][j] = sum_i R[k][i] dT[i][j]
      a.A = sv.right; a.a_sm = N; a.a_sk = 1;
      a.B = dT; a.b_sn = 1; a.b_sk = N;
      // dR[k][i] = sum_j L[k][j] dT[i][j]
      b.A = sv.left; b.a_sm = N; b.a_sk = 1;
      b.B = dT; b.b_sn = N; b.b_sk = 1;
    }
    bool one = false;
    if (N <= 256) {
      KTimed kt(BC2N_TN(C, "trimul.contract_bwd"), st);
      one = trimul_contract_pair(st, N, I, a.A, a.B, dL, b.A, b.a_sk == 1, b.B, b.b_sk == 1, dR);
    }
    if (!one) {
      contract<h16>(st, a, dL, BC2N_TN(C, "trimul.contract_bwd"));
      contract<h16>(st, b, dR, BC2N_TN(C, "trimul.contract_bwd"));
    }
  }
  if (fused) {
    TailArgs t;
    t.xn = sv.xn; t.w1 = w.tail_w1; t.w2 = w.tail_w2;
    t.dl = dL; t.dr = dR; t.dcg = dcat;
    t.bp = w.bp; t.bg = w.bg; t.mask = mask;
    t.x = pair_in; t.ln_g = w.ln_g; t.mean = sv.mean; t.rstd = sv.rstd; t.dres = dout;
    t.gmul = sc + 1;
    t.out = din; t.M = M;
    KTimed kt(BC2N_TN(C, "trimul.tail_bwd"), st);
    if (C == 128) trimul_tail<128>(st, t);
    else trimul_tail<64>(st, t);
    return;
  }
  {
    GemmArgs g;
    g.M = (int)M; g.N = 4 * I; g.K = C;
    g.A = sv.xn; g.a_sm = C; g.a_sk = 1;
    g.B = w.wcat_t; g.b_sn = C; g.b_sk = 1;
    gemm<128, 128>(st, g, EpiTrimulProjBwd{dL, dR, w.bp, w.bg, mask, dcat, M, I, NC},
                   BC2N_TN(C, "trimul.proj_bwd"));
  }
  GemmArgs g2;
  g2.M = (int)M; g2.N = C; g2.K = NC;
  g2.A = dcat; g2.a_sm = NC; g2.a_sk = 1;
  g2.B = w.wcat; g2.b_sn = NC; g2.b_sk = 1;
  if (C == 128) {
    // the input LayerNorm's backward and the residual add in the epilogue
    gemm<128, 128>(st, g2,
                   EpiLnBwd<0>(pair_in, w.ln_g, sv.mean, sv.rstd, dout, din, M, 0, nullptr,
                               nullptr, sc + 1),
                   BC2N_TN(C, "trimul.gemm_dx_ln"));
    return;
  }
  gemm<128, 128>(st, g2, EpiStore<float>{dxn, C, 0, nullptr, C}, BC2N_TN(C, "trimul.gemm_dx"));
  KTimed kt(BC2N_TN(C, "trimul.ln_bwd"), st);
  ln_bwd_f32(st, dxn, pair_in, M, C, 0, w.ln_g, sv.mean, sv.rstd, din, true, 0, nullptr, nullptr,
             dout, sc + 1);
}

}  // namespace bc2n
