// The pair track's K = C products (C = 128 or 64 channels) with what comes
// before and after them: a workgroup builds BM = 16 RT binary16 rows in LDS --
// the LayerNorm of f32 rows, the centre norm of a channel-major tensor, stored
// rows, or scaled cotangent rows -- and multiplies them by an nout x C weight
// matrix, 32 output columns a wave at a time.  Weight fragments come straight
// from memory (proj_frags order, one contiguous 1 KB a wave) a chunk ahead.
//
// The results go from the MFMA registers to the epilogue: no staging tile and,
// after the rows are in LDS, no barrier, so the waves run their chunks apart
// and one's stores overlap another's products.
//
//  row columns: the weights are the first MFMA operand, so a lane ends with
//    one row and, the fragments' columns being interleaved (proj_frags), 8
//    consecutive columns of it; four lanes cover a row's 32 columns.
//  column columns (channel-major outputs; EpiCols): the rows are the first
//    operand, so a lane ends with one column -- a projection (first fragment)
//    and its gate (second) -- and, the LDS rows being interleaved in 32-row
//    blocks (lds_row), 8 consecutive rows of it; four lanes cover 32 rows.
//
// Either way a store is 16 or 32 bytes a lane and 64 or 128 a row or channel.
// With each chunk's f32 tile staged through LDS instead (two barriers and 50 KB
// of LDS traffic a chunk, 48-row workgroups in more than one round) triangle
// attention's LayerNorm + q|k|v|g took 30 us a launch at N = 224 and 11 at 64,
// trimul's LayerNorm + projections 33 and 11.
#pragma once
#include "gemm.h"
#include "kernels.h"

namespace bc2n {

// B operand of an nout x K product (K = 64 or 128, nout % 32 == 0) in fragment
// order: fragment (n32 * 2 + jj) * (K / 32) + ks holds, at lane 16 g + c, the 8
// values B(n, 32 ks + 8 g + e), e = 0..7.  Its column n is, within 32-column
// block n32, 16 jj + c for columns below `cols` (column mode), and 8 (c / 4) +
// 4 jj + c % 4 above (row mode: MFMA row 4g + r of fragments 0 and 1 are
// columns 8g + r and 8g + 4 + r).
template <class B>
std::vector<h16> proj_frags(int nout, int K, int cols, B b) {
  std::vector<h16> f((size_t)nout * K);
  size_t o = 0;
  for (int n32 = 0; n32 < nout / 32; ++n32)
    for (int jj = 0; jj < 2; ++jj)
      for (int ks = 0; ks < K / 32; ++ks)
        for (int l = 0; l < 64; ++l)
          for (int e = 0; e < 8; ++e) {
            const int c = l & 15;
            const int n = 32 * n32 + (32 * n32 < cols ? 16 * jj + c : 8 * (c >> 2) + 4 * jj + (c & 3));
            f[o++] = (h16)b(n, 32 * ks + 8 * (l >> 4) + e);
          }
  return f;
}

namespace lnproj {
enum class In {
  LN,      // LayerNorm of f32 rows x (transposed read when nt > 0), xn kept when not null
  CM,      // centre norm of the channel-major x [C][M] (ln_fwd_cm's sums in its order)
  ROWS,    // the binary16 rows xn as they are
  SCALED,  // binary16(s * tbl * x) (transposed read when nt > 0)
  GATED,   // binary16(s * tbl * x * gout); dcat = s * tbl * x * osave * gout (1 - gout)
};

struct Args {
  long M;
  int nt, bn, nout;  // nt: transposed read (ending node) when > 0; bn: residues (M = bn^2)
  const float* x;
  const float *g, *b, *wb;  // LayerNorm scale, offset; bias weights [C][H]
  float bscale;
  h16* xn;
  float *mean, *rstd;
  h16* bias;  // [H][M] binary16 in score-fragment order
  const h16* W;
  // SCALED, GATED: dropout table [bn][C] or null, the cotangent scale
  const float* tbl;
  CtScale sc;
  const h16 *gout, *osave;  // GATED
  h16* dcat;
};

// LDS position of row r of the tile and back, where an epilogue has columns:
// inside a 32-row block, MFMA row 4g + k of 16-row tiles 0 and 1 are rows
// 8g + k and 8g + 4 + k.  In order otherwise.
template <bool COLS>
__host__ __device__ constexpr int lds_row(int r) {
  return COLS ? (r & ~31) + ((r >> 2) & 1) * 16 + ((r >> 3) & 3) * 4 + (r & 3) : r;
}
template <bool COLS>
__host__ __device__ constexpr int row_of(int p) {
  return COLS ? (p & ~31) + ((p >> 2) & 3) * 8 + ((p >> 4) & 1) * 4 + (p & 3) : p;
}

// An epilogue with operands of its own (nout == C) declares struct Pre,
// load(m, n, pre, d) and row(m, n, v, pre, d), for columns n..n+3 and
// n+d..n+d+3 of a row: the loads of all of a lane's rows are then in flight
// together.  With kQuads its weights are in column-mode order and d is 16.
template <class E, class = void>
struct has_pre : std::false_type {};
template <class E>
struct has_pre<E, std::void_t<typename E::Pre>> : std::true_type {};

template <class E, class = void>
struct quads : std::false_type {};
template <class E>
struct quads<E, std::void_t<decltype(E::kQuads)>> : std::bool_constant<E::kQuads> {};

template <class E, class = void>
struct has_tile : std::false_type {};
template <class E>
struct has_tile<E, std::void_t<typename E::Tile>> : std::true_type {};

// An epilogue with a Tile (nout == C: a row-wise reduction over the columns)
// takes the f32 tile whole, staged in LDS, with operands it loaded beforehand.

// WC waves side by side over the columns, 4 / WC row groups (WC = 2 where nout
// is 64).  64-row tiles with a front of their own keep three waves a SIMD: at
// four they spill (trimul's projections 48 registers: 50 us instead of 28 at
// N = 224).  Four waves are the most the others are given, for the registers'
// sake, but the centre norm's 32-row form is free to run at five, where its
// workgroups at N = 192 are one round (16.6 -> 15.5 us, N = 224 21.1 -> 20.5).
template <In IN, int RT>
constexpr int min_waves() {
  return RT >= 3 && (IN == In::LN || IN == In::CM || IN == In::GATED) ? 3 : 4;
}
template <In IN, int C, int RT, int WC, int H, bool FAST, class Epi>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(min_waves<IN, RT>(), IN == In::CM ? 8 : 4))) void
kernel(Args a, Epi epi) {
  constexpr int BM = 16 * RT, LDX = C + 8, KS = C / 32, TI = RT * WC / 4;
  constexpr int LPR = C / 8, RPP = 256 / LPR, PASS = BM / RPP;  // lanes a row, rows a pass
  constexpr bool TILE = has_tile<Epi>::value;
  constexpr bool ONE = TILE || has_pre<Epi>::value;  // one chunk of columns
  constexpr int LDT = C + (TILE ? 4 : 1);
  constexpr int XB = BM * LDX * 2, TB = IN == In::CM || TILE ? BM * LDT * 4 : 0;
  static_assert(RT * WC % 4 == 0 && BM % RPP == 0 && (BM % 32 == 0 || !Epi::kHasCol), "tile split");
  __shared__ __align__(16) char smem[XB > TB ? XB : TB];
  h16* xs = reinterpret_cast<h16*>(smem);
  float* T = reinterpret_cast<float*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wc = w % WC, wr = w / WC;
  // consecutive workgroups on consecutive XCDs: one front through memory.  (A
  // contiguous range of rows an XCD, eight fronts a power of two apart, is 5 to
  // 10% slower at N = 416 and 512.)
  const long M = a.M, m0 = (long)blockIdx.x * BM;

  h16x8 bf[KS][2];
  auto load_b = [&](int j) {
    const int n32 = min(j * WC + wc, a.nout / 32 - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
        bf[ks][jj] = ld8(a.W + ((long)((n32 * 2 + jj) * KS + ks) * 64 + lane) * 8);
  };

  const int fr = tid / LPR, l = tid % LPR, c0 = l * 8;  // front: row of a pass, lane in it, channels
  if constexpr (IN == In::ROWS) {
    h16x8 ob[PASS];
#pragma unroll
    for (int p = 0; p < PASS; ++p)
      ob[p] = ld8(a.xn + min(m0 + p * RPP + fr, M - 1) * C + c0);  // rows past M: never stored
    load_b(0);
#pragma unroll
    for (int p = 0; p < PASS; ++p) st8(xs + lds_row<Epi::kHasCol>(p * RPP + fr) * LDX + c0, ob[p]);
  } else if constexpr (IN == In::CM) {
    // the [C][BM] tile through T, then the rows over it: eight lanes a row
    static_assert(H == 0, "centre norm: no bias heads");
    load_b(0);
#pragma unroll 8
    for (int i = tid; i < C * (BM / 4); i += 256) {
      const int c = i / (BM / 4), q = (i % (BM / 4)) * 4;
      const float4 v4 = *reinterpret_cast<const float4*>(a.x + (long)c * M + min(m0 + q, M - 4));  // M % 4 == 0
      T[(q + 0) * LDT + c] = v4.x;
      T[(q + 1) * LDT + c] = v4.y;
      T[(q + 2) * LDT + c] = v4.z;
      T[(q + 3) * LDT + c] = v4.w;
    }
    __syncthreads();
    constexpr int P = 8, CPL = C / P, NR = BM / (256 / P);
    h16x8 ob[NR][CPL / 8];
    const int part = tid % P;
#pragma unroll
    for (int rb = 0; rb < NR; ++rb) {
      const int r = rb * (256 / P) + tid / P;
      const long m = m0 + r;
      float v[CPL];
      float s = 0.f, s2 = 0.f;
#pragma unroll
      for (int e = 0; e < CPL; ++e) {
        v[e] = T[r * LDT + part * CPL + e];
        s += v[e];
        s2 += v[e] * v[e];
      }
      s = group_sum<P>(s);
      const float mu = s / C;
      float var;
      if (FAST) {
        var = group_sum<P>(s2) / C - mu * mu;
      } else {
        float d2 = 0.f;
#pragma unroll
        for (int e = 0; e < CPL; ++e) { const float d = v[e] - mu; d2 += d * d; }
        var = group_sum<P>(d2) / C;
      }
      const float rs = rsqrtf(var + LN_EPS);
#pragma unroll
      for (int e0 = 0; e0 < CPL; e0 += 8)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int c = part * CPL + e0 + e;
          ob[rb][e0 / 8][e] = (h16)((v[e0 + e] - mu) * rs * a.g[c] + a.b[c]);
        }
      if (part == 0 && m < M) {
        a.mean[m] = mu;
        a.rstd[m] = rs;
      }
    }
    __syncthreads();  // every row is out of T, which xs overlays
#pragma unroll
    for (int rb = 0; rb < NR; ++rb)
#pragma unroll
      for (int e8 = 0; e8 < CPL / 8; ++e8)
        st8(xs + lds_row<Epi::kHasCol>(rb * (256 / P) + tid / P) * LDX + part * CPL + e8 * 8, ob[rb][e8]);
  } else if constexpr (IN == In::SCALED || IN == In::GATED) {
    // two passes' loads in flight at a time (a register budget for four waves)
    constexpr int PF = PASS < 2 ? PASS : 2;
    CtLoad cl;
    cl.load(a.sc, tid);
    float sm = 0.f;
    load_b(0);
#pragma unroll
    for (int p0 = 0; p0 < PASS; p0 += PF) {
      float v[PF][8], t[PF][8];
      h16x8 go[IN == In::GATED ? PF : 1], os[IN == In::GATED ? PF : 1];
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const long m = min(m0 + (p0 + p) * RPP + fr, M - 1);
        ld_f8(a.x + ln_src_row(m, a.nt) * C + c0, v[p]);
        if (a.tbl) ld_f8(a.tbl + (long)((int)m % a.bn) * C + c0, t[p]);
        if constexpr (IN == In::GATED) {
          go[p] = ld8(a.gout + m * C + c0);
          os[p] = ld8(a.osave + m * C + c0);
        }
      }
      if (p0 == 0) sm = cl.scale(a.sc, tid, blockIdx.x == 0);
#pragma unroll
      for (int p = 0; p < PF; ++p) {
        const int r = (p0 + p) * RPP + fr;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[p][e] *= a.tbl ? t[p][e] * sm : sm;
        h16x8 o;
        if constexpr (IN == In::SCALED) {
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = f2h_sat(v[p][e]);
        } else {
          h16x8 dc;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float gv = (float)go[p][e], ov = (float)os[p][e];
            o[e] = f2h_sat(v[p][e] * gv);
            dc[e] = f2h_sat(v[p][e] * ov * gv * (1.f - gv));
          }
          if (m0 + r < M) st8(a.dcat + (m0 + r) * C + c0, dc);
        }
        st8(xs + lds_row<Epi::kHasCol>(r) * LDX + c0, o);
      }
    }
  } else {
    float v[PASS][8];
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
      const long m = min(m0 + p * RPP + fr, M - 1);  // rows past M: in bounds, unused
      ld_f8(a.x + ln_src_row(m, a.nt) * C + c0, v[p]);
    }
    float gm[8], bt[8], wv[8][H > 0 ? H : 1];
    ld_f8(a.g + c0, gm);
    ld_f8(a.b + c0, bt);
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int h = 0; h < H; ++h) wv[e][h] = a.wb[(c0 + e) * H + h];
    load_b(0);
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
      const int r = p * RPP + fr;
      const long m = m0 + r;
      float s = 0.f, s2 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s += v[p][e];
        s2 += v[p][e] * v[p][e];
      }
      const float mu = group_sum<LPR>(s) / C;
      float var;
      if constexpr (FAST) {
        var = group_sum<LPR>(s2) / C - mu * mu;
      } else {
        float d2 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = v[p][e] - mu;
          d2 += d * d;
        }
        var = group_sum<LPR>(d2) / C;
      }
      const float rs = rsqrtf(var + LN_EPS);
      float o[8];
      h16x8 ob;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o[e] = (v[p][e] - mu) * rs * gm[e] + bt[e];
        ob[e] = (h16)o[e];
      }
      float mine = 0.f;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        float q = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) q += o[e] * wv[e][h];
        q = group_sum<LPR>(q);
        if (l == h) mine = q;
      }
      if (m < M) {
        if (a.xn) st8(a.xn + m * C + c0, ob);
        if (l == 0) {
          a.mean[m] = mu;
          a.rstd[m] = rs;
        }
        if (H > 0 && l < H)
          a.bias[bias_frag_index(l, (int)(m / a.bn), (int)(m % a.bn), a.bn)] = (h16)(mine * a.bscale);
      }
      st8(xs + lds_row<Epi::kHasCol>(r) * LDX + c0, ob);
    }
  }
  __syncthreads();

  const int nch = ONE ? 1 : (a.nout + 32 * WC - 1) / (32 * WC);
#pragma unroll 1
  for (int j = 0; j < nch; ++j) {
    const int n0 = (j * WC + wc) * 32;
    if (n0 >= a.nout) break;  // wave-uniform; no barrier follows in a wave's loop
    f32x4 acc[TI][2];
#pragma unroll
    for (int i = 0; i < TI; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto product = [&](auto cols_c) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        // With column outputs the rows of every K step read ahead spill: their
        // second half waits for the first half's products (the 20 to 60 bytes of
        // scratch cost a launch about 1 us, trimul's projections).
        if (IN == In::LN && Epi::kHasCol && ks == KS / 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          const h16x8 xf = ld8(xs + ((wr * TI + i) * 16 + l16) * LDX + ks * 32 + 8 * g);
#pragma unroll
          for (int jj = 0; jj < 2; ++jj)
            acc[i][jj] = decltype(cols_c)::value ? mfma16x16x32(xf, bf[ks][jj], acc[i][jj])
                                                 : mfma16x16x32(bf[ks][jj], xf, acc[i][jj]);
        }
      }
      // unconditional (the last chunk reloads its own): a load under a branch
      // leaves the in-order memory counter unknown at the join
      if constexpr (!ONE) load_b(min(j + 1, nch - 1));
    };
    if constexpr (Epi::kHasCol) {
      if (epi.col_mode(n0)) {
        product(std::true_type{});
        // 8 rows of a projection column and of its gate a lane
#pragma unroll
        for (int b = 0; b < TI / 2; ++b) {
          const long m = m0 + wr * TI * 16 + b * 32 + 8 * g;
          if (m >= M) continue;  // M % 8 == 0
          float pv[8], gv[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            pv[e] = acc[2 * b + e / 4][0][e % 4];
            gv[e] = acc[2 * b + e / 4][1][e % 4];
          }
          epi.cols(m, n0 + l16, pv, gv);
        }
        continue;
      }
    }
    product(std::false_type{});
    auto row_m = [&](int i) { return m0 + row_of<Epi::kHasCol>((wr * TI + i) * 16 + l16); };
    if constexpr (TILE) {
      // one chunk of every column (nout == C): the f32 tile over xs
      typename Epi::Tile tl;
      epi.template load<BM>(m0, tl, tid);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        float* p = T + (row_m(i) - m0) * LDT + n0 + 8 * g;
        *reinterpret_cast<f32x4*>(p) = acc[i][0];
        *reinterpret_cast<f32x4*>(p + 4) = acc[i][1];
      }
      __syncthreads();
      epi.template tile<BM>(m0, T, LDT, tid, tl);
    } else if constexpr (has_pre<Epi>::value) {
      constexpr bool Q = quads<Epi>::value;
      const int n = n0 + (Q ? 4 : 8) * g;
      typename Epi::Pre pre[TI];
#pragma unroll
      for (int i = 0; i < TI; ++i) epi.load(min(row_m(i), M - 1), n, pre[i], Q ? 16 : 4);
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const long m = row_m(i);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[i][e / 4][e % 4];
        if (m < M) epi.row(m, n, v, pre[i], Q ? 16 : 4);
      }
    } else {
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const long m = row_m(i);
        if (m >= M) continue;  // a row's four lanes leave together
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[i][e / 4][e % 4];
        epi.row(0, (int)m, n0 + 8 * g, v);
      }
    }
  }
}

// Rows a workgroup.  32 rows fill the chip at small M and, having the
// registers for four or more waves a SIMD, hide each other's loads; 64 rows
// read every weight fragment half as often.  Where the lines lie, C = 128, us
// a launch with 32 / 64 rows: LN at M = 16384 12 / 12, 65536 47 / 30, 262144
// 196 / 117 (trimul's); CM at M = 65536 26 / 27, 173056 84 / 80, 262144 132 /
// 122; GATED at M = 65536 21 / 21, 102400 40 / 37, 262144 106 / 98.  SCALED
// (14 / 17 at 50176, 79 / 77 at 262144) keeps 32; ROWS takes 48 beyond 32768
// (8.0 against 9.3 at 36864, 72 against 74 at 262144).  Triangle attention's LN
// takes 48 where 64-row workgroups come to one round and a little, or to much
// less than one (18.1 against 20.6 at 36864, 26.5 / 27.3 at 50176; 33 / 30 at 65536).
// From 448 rows a CU it takes 96: the 128 KB of weight fragments a workgroup reads
// from L2 serve half as many rows again (64 / 96 rows by events: 57.9 / 56.5 at
// 102400, 64.6 / 63.4 at 123904, 85.5 / 83.2 at 173056, 124 / 115 at 262144, 191 /
// 173 at 409600; with trimul's column outputs 125 / 152 at 262144).
template <In IN, int C, int H, bool FAST, class Epi>
void launch(hipStream_t st, const Args& a, const Epi& epi) {
  static_assert(H == 0 || H == 4, "bias heads 0 or 4");
  if (a.M <= 0 || a.M % 32 != 0 || a.nout % 32 != 0 || a.nout < 64 || !a.W ||
      ((has_tile<Epi>::value || has_pre<Epi>::value) && a.nout != C) ||
      (H > 0 && (long)a.bn * a.bn != a.M) ||
      ((IN == In::SCALED || IN == In::GATED) && (a.bn <= 0 || !a.sc.sc)))
    throw std::runtime_error("row projection: shape");
  auto go = [&](auto rt, auto wc) {
    constexpr int RT = decltype(rt)::value, WC = decltype(wc)::value;
    const long nwg = (a.M + 16 * RT - 1) / (16 * RT);
    hipLaunchKernelGGL((kernel<IN, C, RT, WC, H, FAST, Epi>), dim3((unsigned)nwg), dim3(256), 0, st,
                       a, epi);
  };
  using std::integral_constant;
  auto width = [&](auto rt) {
    if constexpr (C == 64 && ((has_tile<Epi>::value || has_pre<Epi>::value)))
      go(rt, integral_constant<int, 2>());  // nout is 64
    else
      go(rt, integral_constant<int, 4>());
  };
  const long per_cu = a.M / device_cus();
  if constexpr (IN == In::SCALED) {
    width(integral_constant<int, 2>());
  } else if constexpr (IN == In::ROWS) {
    if (C == 128 && per_cu > 128) {
      if constexpr (C == 128) width(integral_constant<int, 3>());
    } else {
      width(integral_constant<int, 2>());
    }
  } else {
    constexpr long tall = IN == In::LN ? 64 : IN == In::CM ? 512 : 288;
    if constexpr (C == 128 && IN == In::LN && !Epi::kHasCol) {
      if (per_cu > 112 && per_cu < 224) {
        width(integral_constant<int, 3>());
        return;
      }
      if (per_cu > 448) {
        width(integral_constant<int, 6>());
        return;
      }
    }
    if (per_cu >= tall) width(integral_constant<int, 4>());
    else width(integral_constant<int, 2>());
  }
}
}  // namespace lnproj
}  // namespace bc2n
