// FP64 Legendre contractions on v_mfma_f64_16x16x4_f64: rtrans_forward and
// rtrans_backward (src/submodules/mlegs_scalar_ops.f90:1852-2008), the same
// sums as legendre.hip's, term by term in the same order (bit for bit).
//
// Both are GEMMs whose A operand is the field (16 rows = the real and
// imaginary parts of 8 axial slices; element r of lane l of the accumulator is
// row l/16 + 4r, measured on gfx950, so A row i carries field column 4(i%4) +
// i/4 and that element is column 4(l/16) + r) and whose B operand is the table (16
// radial rows or points).  A workgroup of 8 waves takes KT slices of one column m.
//
// What bounds them: the FP64 MFMA (3.25 GFLOP, 45 us at the 72.6 TFLOP/s of a
// large product) and the field's two passes over HBM (240-270 MB, about 50 us)
// cost the same, so what counts is that neither waits for the other.
//  - The field chunk goes through LDS, shared by the eight waves; the table
//    goes from the XCD's L2 straight into the registers of the one wave that
//    uses it (512 bytes per KT / 8 MFMA of 64 cycles): no LDS traffic, and one
//    barrier per chunk (two buffers).
//  - LDS rows have a pitch of 2 KT + 2 doubles: the 16-byte writes of 8
//    consecutive radial points fall in different banks (a pitch of 16 modulo 64
//    doubles, good for the reads alone, made the writes 8-way conflicts: the
//    staging by itself took 72 us of a 256^3 launch, now 32).
//  - Output rows of both parities are put together in LDS and written as whole
//    columns, streaming.
// At 256^3, every column, in the first nine round trips of a field: forward 170 ->
// 122 us, backward 129 -> 105 us (kernels that stage the table in LDS, one wave per
// SIMD, before); 116 and 101 over 33 round trips.
#include "mlx_internal.h"

namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

// The slices of a launch: nf fields of nz axial slices each, slice s is slice
// s % nz of field s / nz.  A tile takes KT consecutive ones of one column m:
// the fields of a batch share its table, and a kit of few slices (a polar kit
// has one) fills a tile with several fields.
struct LegFields {
  const double2 *in[mlx::kZBatch];
  double2 *out[mlx::kZBatch];
  const double *ln[mlx::kZBatch];  // log coefficients (device), or null
};
// sizes, the radial grid and the decomposition: nyt slice tiles, nsp row
// splits, ncol columns with workgroups (npc of them computed), tpitch the
// table's row pitch
struct LegDims {
  int nrdim, npdim, nz, nf, nr, nrh, ne, nrc, npc, ncol, nyt, nsp, tpitch;
  const double *w, *lnx;
};

// Workgroup L -> column u, tile y: whole groups of 8 columns by xcd_map, the
// nyt tiles of the remaining columns spread over the XCDs (129 columns leave
// one, whose tiles on one XCD would run alone at the end; a launch of column 0
// alone would have one XCD of the eight).
__device__ inline void leg_map(int L, int ncol, int nyt, int &u, int &y) {
  const int full = ncol / kXcd * kXcd;
  if (L < full * nyt) {
    xcd_map(L, nyt, u, y);
    return;
  }
  L -= full * nyt;
  u = full + L / nyt;
  y = L % nyt;
}

// the slice pointers of a tile, column offset included; null past the end
template <int KT>
__device__ inline void leg_slices(const LegFields &f, const LegDims &d, int m, int k0, const double2 **si, double2 **so,
                                  const double **sl) {
  const int t = threadIdx.x, s = k0 + t;
  if (t < KT) {
    const bool ok = s < d.nf * d.nz;
    const int q = ok ? s / d.nz : 0;
    const size_t o = (size_t)(ok ? s % d.nz : 0) * d.nrdim * d.npdim + (size_t)d.nrdim * m;
    const double2 *in = f.in[0];
    double2 *out = f.out[0];
    const double *ln = f.ln[0];
#pragma unroll
    for (int j = 1; j < mlx::kZBatch; ++j)
      if (q == j) in = f.in[j], out = f.out[j], ln = f.ln[j];
    si[t] = ok ? in + o : nullptr;
    so[t] = ok ? out + o : nullptr;
    sl[t] = (ok && m == 0) ? ln : nullptr;
  }
  __syncthreads();
}

template <int KT>
__device__ inline void leg_zero(double2 *const *so, int r0, int r1) {
  const int span = r1 - r0;
  for (int idx = threadIdx.x; idx < (span > 0 ? span : 0) * KT; idx += 512) {
    double2 *o = so[idx / span];
    if (o) o[r0 + idx % span] = make_double2(0.0, 0.0);
  }
}

__device__ inline int arow(int i) { return 4 * (i & 3) + (i >> 2); }

// forward: out(2a+p, m, k) = sum_x P_p(a, x) fold_p(x, k), table pfg[m][p][x][a].
// A wave owns S tiles of 16 rows a of one parity (half the field reads of a
// wave that owns both); the workgroup the 64 S rows a from 64 S sp on.
// f.ln: column 0 of the input less ln lnx(x) (the log term's step of trans).
template <int KT, int S, int XC>
__global__ void __launch_bounds__(512) k_leg_fwd_f64m(LegFields f, LegDims d, const double *__restrict__ tab) {
  constexpr int NT = KT / 8, PC = 2 * KT + 2, NB = 2 * XC * PC, KS = XC / 4;
  constexpr int R = 128 * S, SPR = R + 1;  // output rows, their LDS pitch
  constexpr int NF = (XC * KT + 511) / 512;
  constexpr int NLDS = 2 * NB > 16 * SPR ? 2 * NB : 16 * SPR;
  __shared__ double Bs[NLDS];
  __shared__ const double2 *si[KT];
  __shared__ double2 *so[KT];
  __shared__ const double *sl[KT];
  int m, y;
  leg_map(blockIdx.x, d.ncol, d.nyt * d.nsp, m, y);
  const int sp = y % d.nsp, k0 = (y / d.nsp) * KT;
  const int nr = d.nr, nrh = d.nrh, nrdim = d.nrdim;
  const int nn = (m < d.npc && d.nrc > m) ? d.nrc - m : 0, Mmax = (nn + 1) / 2;
  const int a0 = 64 * S * sp;
  leg_slices<KT>(f, d, m, k0, si, so, sl);
  if (a0 >= Mmax) {  // an inactive column, or rows past its chop
    leg_zero<KT>(so, 2 * a0, sp == d.nsp - 1 ? nrdim : min(2 * a0 + R, nrdim));
    return;
  }
  // the waves' tiles turn with the slice tile: the short last tile of a column
  // then falls on another SIMD in each workgroup
  const int tid = threadIdx.x, lane = tid % 64, li = lane % 16, lk = lane / 16;
  const int wv = (tid / 64 + 2 * (k0 / KT)) % 8, p = wv & 1, tw = wv >> 1;
  const int left = d.nf * d.nz - k0;
  const int ntile = left >= KT ? NT : (left + 7) / 8;  // 16-column tiles in use
  const double *Tg = tab + ((size_t)m * 2 + p) * nrh * d.tpitch;
  doublex4 acc[S][NT];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[s][t] = doublex4{0.0, 0.0, 0.0, 0.0};
  double2 ra[NF], rb[NF];
  double rw[NF], bn[KS][S];
  auto fetch = [&](int x0) {
#pragma unroll
    for (int q = 0; q < NF; ++q) {
      const int idx = tid + 512 * q, x = idx % XC, kl = idx / XC, xg = x0 + x;
      ra[q] = rb[q] = make_double2(0.0, 0.0);
      rw[q] = 0.0;
      const double2 *col = idx < XC * KT ? si[kl] : nullptr;
      if (col && xg < nrh) {
        ra[q] = col[xg];
        rb[q] = col[nr - 1 - xg];
        rw[q] = d.w[xg];
        if (const double *ln = sl[kl]) {
          ra[q].x = __builtin_fma(-ln[0], d.lnx[xg], ra[q].x);
          rb[q].x = __builtin_fma(-ln[0], d.lnx[nr - 1 - xg], rb[q].x);
        }
      }
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int a = a0 + (tw + 4 * s) * 16;
#pragma unroll
      for (int k = 0; k < KS; ++k) {
        const int xg = x0 + 4 * k + lk;
        bn[k][s] = (xg < nrh && a < Mmax) ? Tg[(size_t)xg * d.tpitch + a + li] : 0.0;
      }
    }
  };
  fetch(0);
  int buf = 0;
  for (int x0 = 0; x0 < nrh; x0 += XC) {
#pragma unroll
    for (int q = 0; q < NF; ++q) {
      const int idx = tid + 512 * q, x = idx % XC, kl = idx / XC;
      if (idx < XC * KT) {
        const double2 u = ra[q], v = rb[q];
        const double wx = rw[q];
        double *b = &Bs[buf * NB + x * PC + 2 * kl];
        *reinterpret_cast<double2 *>(b) = make_double2((u.x + v.x) * wx, (u.y + v.y) * wx);
        *reinterpret_cast<double2 *>(b + XC * PC) = make_double2((u.x - v.x) * wx, (u.y - v.y) * wx);
      }
    }
    double b[KS][S];
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int s = 0; s < S; ++s) b[k][s] = bn[k][s];
    __syncthreads();
    if (x0 + XC < nrh) fetch(x0 + XC);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      double fa[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) fa[t] = Bs[buf * NB + (p * XC + 4 * k + lk) * PC + 16 * t + arow(li)];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (a0 + (tw + 4 * s) * 16 >= Mmax) continue;
#pragma unroll
        for (int t = 0; t < NT; ++t)
          if (t < ntile) acc[s][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[t], b[k][s], acc[s][t], 0, 0, 0);
      }
    }
    buf ^= 1;
  }
  // 8 slices at a time: rows of both parities into LDS, whole columns out
  double2 *st = reinterpret_cast<double2 *>(&Bs[0]);
  const int r0 = 2 * a0, rn = nrdim - r0 < R ? nrdim - r0 : R;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (t >= ntile) break;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        st[(2 * lk + h) * SPR + 2 * ((tw + 4 * s) * 16 + li) + p] =
            make_double2(acc[s][t][2 * h], acc[s][t][2 * h + 1]);
    __syncthreads();
    for (int idx = tid; idx < 8 * R; idx += 512) {
      const int r = idx % R, kl = idx / R;
      double2 *o = so[8 * t + kl];
      if (o && r < rn) st_nt(o + r0 + r, r0 + r < nn ? st[kl * SPR + r] : make_double2(0.0, 0.0));
    }
  }
  if (sp == d.nsp - 1) leg_zero<KT>(so, r0 + R, nrdim);  // rows past the tiles
}

// backward: f(x) = be + bo, f(-x) = be - bo, b_p(x, k) = sum_a P(x, 2a+p)
// e(2a+p, k), table ptab[m][n][x].  A wave owns 16 points x, both parities;
// the workgroup the 128 points from 128 sp on.  KT = 16 and chunks of 8 for
// every size: one kernel (32 slices take 90 us at 256^3 against 97, but 13.1
// against 11.4 at 128 x 64 x 64; round trips of one field).  f.ln: column 0 of the output plus ln lnx(x).
__global__ void __launch_bounds__(512) k_leg_bwd_f64m(LegFields f, LegDims d, const double *__restrict__ ptab) {
  constexpr int KT = 16, AC = 8, NT = KT / 8, PC = 2 * KT + 2, KS = AC / 4;
  // the even and odd rows' planes: 64 bytes apart modulo the banks
  constexpr int PL = AC * PC + 8;
  __shared__ double Es[2][2 * PL];
  __shared__ const double2 *si[KT];
  __shared__ double2 *so[KT];
  __shared__ const double *sl[KT];
  static_assert(2 * AC * KT <= 512, "one coefficient per thread and chunk");
  int m, y;
  leg_map(blockIdx.x, d.ncol, d.nyt * d.nsp, m, y);
  const int sp = y % d.nsp, k0 = (y / d.nsp) * KT;
  const int nr = d.nr, nrh = d.nrh, nrdim = d.nrdim;
  if (m >= d.npc && sp != 0) return;
  leg_slices<KT>(f, d, m, k0, si, so, sl);
  if (m >= d.npc) {
    leg_zero<KT>(so, 0, nrdim);
    return;
  }
  const int nn = d.nrc > m ? d.nrc - m : 0, Me = (nn + 1) / 2;
  const int tid = threadIdx.x, lane = tid % 64, wv = tid / 64, li = lane % 16, lk = lane / 16;
  const int xw = 128 * sp + 16 * wv, x = xw + li;
  const int left = d.nf * d.nz - k0;
  const int ntile = left >= KT ? NT : (left + 7) / 8;
  const double *P = ptab + (size_t)m * d.ne * nrh + x;
  doublex4 acc[NT][2];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t][0] = acc[t][1] = doublex4{0.0, 0.0, 0.0, 0.0};
  const int fr = tid % (2 * AC), fk = tid / (2 * AC);  // this thread's row and slice of a chunk
  const double2 *col = fk < KT ? si[fk] : nullptr;
  double2 rf;
  double bn[KS][2];
  auto fetch = [&](int a0) {
    rf = (col && 2 * a0 + fr < nn) ? col[2 * a0 + fr] : make_double2(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < KS; ++k)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int n = 2 * (a0 + 4 * k + lk) + p;
        bn[k][p] = (n < nn && x < nrh) ? P[(size_t)n * nrh] : 0.0;
      }
  };
  fetch(0);
  int buf = 0;
  for (int a0 = 0; a0 < Me; a0 += AC) {
    if (fk < KT) *reinterpret_cast<double2 *>(&Es[buf][(fr & 1) * PL + (fr >> 1) * PC + 2 * fk]) = rf;
    double b[KS][2];
#pragma unroll
    for (int k = 0; k < KS; ++k) b[k][0] = bn[k][0], b[k][1] = bn[k][1];
    __syncthreads();
    if (a0 + AC < Me) fetch(a0 + AC);
    if (xw < nrh) {
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int t = 0; t < NT; ++t)
            if (t < ntile)
              acc[t][p] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                  Es[buf][p * PL + (4 * k + lk) * PC + 16 * t + arow(li)], b[k][p], acc[t][p], 0, 0, 0);
    }
    buf ^= 1;
  }
  if (x < nrh) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int kl = 8 * t + 2 * lk + h;
        double2 *o = so[kl];
        if (!o) continue;
        const double er = acc[t][0][2 * h], ei = acc[t][0][2 * h + 1];
        const double qr = acc[t][1][2 * h], qi = acc[t][1][2 * h + 1];
        double2 hi = make_double2(er + qr, ei + qi), lo = make_double2(er - qr, ei - qi);
        if (const double *ln = sl[kl]) {
          hi.x = __builtin_fma(ln[0], d.lnx[x], hi.x);
          lo.x = __builtin_fma(ln[0], d.lnx[nr - 1 - x], lo.x);
        }
        o[x] = hi;
        o[nr - 1 - x] = lo;
      }
  }
  if (sp == 0) leg_zero<KT>(so, nr, nrdim);
}

// vec2tp's projection (:1387-1436): psi = -i m V.eo(ur) - D.oe(up), chi =
// i kv D.oe(ur) + m kv V.eo(up) - T.eo(uz), eo/oe the folds b(x) +- b(-x) chosen
// by the row parity; tables tg[m][p][x][a].  The five products accumulate apart
// and are combined at the end, in the order and with the roundings of the
// general kernel (k_v2t_f64): the kappa = 0 Laplacian systems solved afterwards
// amplify a change of rounding here by up to 1e9.
// Bound by the FP64 MFMA (9.0 GFLOP, 124 us at 256^3 with the de-aliasing
// limits): the even and odd waves share the six folds of the three fields (a
// workgroup of one parity read and folded all three for itself), the tables go
// from L2 into the registers of the wave that uses them, and the rows leave in
// whole columns: 387 -> 282 us.  One tile of 16 rows a wave: two would need 320
// accumulator registers.
// Only rows < nrchop - m are computed: the three rows of the radial offset are
// chopped afterwards by the reference.  Columns mbeg .. mend - 1.
// COL0: column 0 alone beside an FP32 launch of the others.  Its V products
// vanish; psi and chi are one chain each, of operands scaled when staged.
// Workgroup ks of ksplit contracts its share of the radial points and writes
// its partial sums to psi/chi + ks kstride (slice stride zso); a second kernel
// adds them.
struct V2tArgs {
  const double2 *f[3];  // ur, up, uz
  double2 *out[2];      // psi, chi
  const double *t[3];   // V, D, T
  const double *ak;
  int nrdim, npdim, nz, nr, nrh, nrc, npc, nzc, nzcu, nyt, nsp, zlo, zhi, mbeg, mend, tpitch, ksplit;
  size_t zso, kstride;
};
// Four waves (32 rows a, both parities) and 8 slices a workgroup for every size, held
// to the registers of four workgroups a CU: at 256^3 282 us, where eight waves and
// 32 slices (half the table and field reads from L2, one workgroup to a CU) take
// 316, 16 slices 321, and this tile without the bound 316.  150 x 120 x 90: 45 us
// (51 without the bound) against 76 with eight waves; one slice, 256 x 256: 25
// against 37 with 16 slices.
template <bool COL0>
__global__ void __launch_bounds__(256, 4) k_v2t_f64m(V2tArgs g) {
  constexpr int NW = 4, KT = 8, NTH = 64 * NW, NT = KT / 8, XC = 8, KS = XC / 4, PC = 2 * KT + 2, PL = XC * PC, NB = 6 * PL;
  constexpr int NP = NW / 2, R = 16 * NW, SPR = R + 1;  // output rows, their LDS pitch
  constexpr int NF = (XC * KT + NTH - 1) / NTH;
  constexpr int NLDS = 2 * NB > 16 * SPR ? 2 * NB : 16 * SPR;
  __shared__ double Bs[NLDS];
  int m, y;
  leg_map(blockIdx.x, g.mend - g.mbeg, g.nyt * g.nsp * g.ksplit, m, y);
  m += g.mbeg;
  const int sp = y % g.nsp, yt = (y / g.nsp) % g.nyt, ks = y / g.nsp / g.nyt;
  const int k0 = yt * KT, nr = g.nr, nrdim = g.nrdim, nz = g.nz;
  const int xshare = ((((g.nrh + XC - 1) / XC) + g.ksplit - 1) / g.ksplit) * XC;
  const int xb = ks * xshare, xe = min(xb + xshare, g.nrh);
  const size_t zs = (size_t)nrdim * g.npdim;
  // every workgroup writes all its rows: zeros in columns m >= npc, past the
  // chopped range, and in slices outside the chopped set or in zlo..zhi
  const int nn = (m < g.npc && g.nrc > m) ? g.nrc - m : 0, Mmax = (nn + 1) / 2;
  const int a0 = 16 * NP * sp, r0 = 2 * a0;
  const bool band_tile = k0 >= g.zlo && k0 + KT - 1 <= g.zhi;
  const bool active = a0 < Mmax && !band_tile;
  const int tid = threadIdx.x, lane = tid % 64, li = lane % 16, lk = lane / 16;
  const int wv = (tid / 64 + 2 * yt) % NW, p = wv & 1, tw = wv >> 1;
  const int at = a0 + 16 * tw;  // this wave's rows a
  const size_t tb = ((size_t)m * 2 + p) * g.nrh * g.tpitch + at + li;
  doublex4 acc[5][NT];
#pragma unroll
  for (int q = 0; q < 5; ++q)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[q][t] = doublex4{0.0, 0.0, 0.0, 0.0};
  double2 ra[NF][3], rb[NF][3];
  double bn[KS][3];
  static_assert(!COL0 || NF == 1, "column 0: one point per thread and chunk");
  const double kvs = (COL0 && k0 + tid / XC < nz) ? g.ak[k0 + tid / XC] : 0.0;
  auto fetch = [&](int x0) {
#pragma unroll
    for (int q = 0; q < NF; ++q) {
      const int idx = tid + NTH * q, x = x0 + idx % XC, kg = k0 + idx / XC;
      const bool ok = idx < XC * KT && x < xe && kg < nz;
      const size_t o = (size_t)kg * zs + (size_t)nrdim * m;
#pragma unroll
      for (int f = 0; f < 3; ++f) {
        ra[q][f] = ok ? g.f[f][o + x] : make_double2(0.0, 0.0);
        rb[q][f] = ok ? g.f[f][o + nr - 1 - x] : make_double2(0.0, 0.0);
      }
    }
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int x = x0 + 4 * k + lk;
#pragma unroll
      for (int f = 0; f < 3; ++f) bn[k][f] = (x < xe && at < Mmax) ? g.t[f][tb + (size_t)x * g.tpitch] : 0.0;
    }
  };
  if (active) {
    fetch(xb);
    int buf = 0;
    for (int x0 = xb; x0 < xe; x0 += XC) {
#pragma unroll
      for (int q = 0; q < NF; ++q) {
        const int idx = tid + NTH * q;
        if (idx < XC * KT) {
          double *b = &Bs[buf * NB + (idx % XC) * PC + 2 * (idx / XC)];
#pragma unroll
          for (int f = 0; f < 3; ++f) {
            const double2 u = ra[q][f], v = rb[q][f];
            double2 ev = make_double2(u.x + v.x, u.y + v.y), od = make_double2(u.x - v.x, u.y - v.y);
            if (COL0 && f == 0) {  // i kv ur
              ev = make_double2(-kvs * ev.y, kvs * ev.x);
              od = make_double2(-kvs * od.y, kvs * od.x);
            } else if (COL0) {  // -up, -uz
              ev = make_double2(-ev.x, -ev.y);
              od = make_double2(-od.x, -od.y);
            }
            *reinterpret_cast<double2 *>(b + 2 * f * PL) = ev;
            *reinterpret_cast<double2 *>(b + (2 * f + 1) * PL) = od;
          }
        }
      }
      double b[KS][3];
#pragma unroll
      for (int k = 0; k < KS; ++k)
#pragma unroll
        for (int f = 0; f < 3; ++f) b[k][f] = bn[k][f];
      __syncthreads();
      if (x0 + XC < xe) fetch(x0 + XC);
      if (at < Mmax) {
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const double *base = &Bs[buf * NB + (4 * k + lk) * PC + arow(li)];
          // V eo(ur), D oe(up), D oe(ur), V eo(up), T eo(uz)
#pragma unroll
          for (int q = 0; q < 5; ++q) {
            if ((COL0 || m == 0) && (q == 0 || q == 3)) continue;  // their factor is m
            const int fld = (q == 0 || q == 2) ? 0 : q == 4 ? 2 : 1;
            const int odd = (q == 0 || q >= 3) ? p : 1 - p;
            const int tbl = (q == 0 || q == 3) ? 0 : q == 4 ? 2 : 1;
            const int to = (COL0 && q == 2) ? 4 : q;  // chi's chain
            const double *pl = base + (2 * fld + odd) * PL;
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[to][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(pl[16 * t], b[k][tbl], acc[to][t], 0, 0, 0);
          }
        }
      }
      buf ^= 1;
    }
  }
  double2 *st = reinterpret_cast<double2 *>(&Bs[0]);
  const int rn = nrdim - r0 < R ? nrdim - r0 : R;
  const double mv = (double)m;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      double2 *out = g.out[o] + (size_t)ks * g.kstride + (size_t)nrdim * m;
      if (active) {
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          auto val = [&](int q) { return make_double2(acc[q][t][2 * h], acc[q][t][2 * h + 1]); };
          double2 A = val(0), B = val(1), C = val(2), Dd = val(3), E = val(4);
          if (m == 0) A = make_double2(0.0, 0.0), Dd = make_double2(0.0, 0.0);
          const int kg = k0 + 8 * t + 2 * lk + h;
          const double kv = kg < nz ? g.ak[kg] : 0.0;
          st[(2 * lk + h) * SPR + 32 * tw + 2 * li + p] =
              COL0 ? (o == 0 ? B : E)
              : o == 0 ? make_double2(mv * A.y - B.x, -mv * A.x - B.y)
                     : make_double2(-kv * C.y + mv * kv * Dd.x - E.x, kv * C.x + mv * kv * Dd.y - E.y);
        }
        __syncthreads();
      }
      for (int idx = tid; idx < 8 * R; idx += NTH) {
        const int r = idx % R, kl = idx / R, kg = k0 + 8 * t + kl;
        if (r >= rn || kg >= nz) continue;
        const bool keep =
            active && r0 + r < nn && (kg + 1 <= g.nzc || kg + 1 >= g.nzcu) && !(kg >= g.zlo && kg <= g.zhi);
        st_nt(out + (size_t)kg * g.zso + r0 + r, keep ? st[kl * SPR + r] : make_double2(0.0, 0.0));
      }
    }
  if (sp != g.nsp - 1) return;  // the last of the row-sharing workgroups zeroes the rest
  const int span = nrdim - r0 - R;
  for (int idx = tid; idx < (span > 0 ? span : 0) * KT; idx += NTH) {
    const int r = r0 + R + idx % span, kg = k0 + idx / span;
    if (kg < nz)
      for (int o = 0; o < 2; ++o)
        g.out[o][(size_t)ks * g.kstride + (size_t)nrdim * m + (size_t)kg * g.zso + r] = make_double2(0.0, 0.0);
  }
}

LegDims leg_dims(const KitDev &k, int nf, int npc, int ncol, int kt, int nsp) {
  LegDims d;
  d.nrdim = k.nrdim, d.npdim = k.npdim, d.nz = k.nzdim, d.nf = nf, d.nr = k.nr, d.nrh = k.nrh, d.ne = k.ne;
  d.nrc = k.nrchop, d.npc = npc, d.ncol = ncol, d.nyt = (nf * k.nzdim + kt - 1) / kt, d.nsp = nsp;
  d.tpitch = k.mfma_ap, d.w = k.w, d.lnx = k.lnx;
  return d;
}
LegFields leg_fields(const double2 *const *in, double2 *const *out, const double *const *ln, int nf) {
  if (nf < 1 || nf > mlx::kZBatch) MLX_THROW(MLX_E_ARG, "rtrans: at most kZBatch fields per launch");
  LegFields f;
  for (int q = 0; q < mlx::kZBatch; ++q) {
    const int j = q < nf ? q : 0;
    f.in[q] = in[j], f.out[q] = out[j], f.ln[q] = ln ? ln[j] : nullptr;
  }
  return f;
}

}  // namespace

namespace mlx {

// In place: one workgroup then reads all of a column's slices it writes, and
// has read them before it writes the first.
bool leg_inplace_ok(const KitDev &k) { return k.nrh <= 128 && (k.nrchop + 1) / 2 <= 128; }

// ncols > 0: columns m >= ncols are written as zero without being read
// (ztail = false: they get no workgroups and are left as they are)
void leg_forward_f64(mlx_ctx *c, const double2 *const *in, double2 *const *out, const double *const *ln, int nf,
                     int ncols, bool ztail) {
  const KitDev &k = c->kit;
  const int npc = (ncols > 0 && ncols < k.npchop) ? ncols : k.npchop, ncol = ztail ? k.npdim : npc;
  const LegFields f = leg_fields(in, out, ln, nf);
  const int M = (k.nrchop + 1) / 2;
  ProbeScope probe(c, MLX_PROBE_LEG_FWD, nf * leg_bytes(k, 0, 8, npc), nf * leg_flops(k, 0, npc));
  // 32 slices and 128 rows a workgroup where that still leaves two workgroups
  // to a CU; 16 slices and 64 rows below (round trips of one field: at 256^3 112 us
  // against 123 in the small tiles; at 128 x 64 x 64, 66 workgroups of the large
  // kind, 17.4 against 11.0)
  const LegDims big = leg_dims(k, nf, npc, ncol, 32, (M + 127) / 128);
  const bool inplace = in[0] == out[0];
  if (inplace && !leg_inplace_ok(k)) MLX_THROW(MLX_E_ARG, "rtrans_forward: in place past 256 radial points");
  if (npc * big.nyt * big.nsp >= 512 || (inplace && M > 64)) {
    probed_launch(probe, k_leg_fwd_f64m<32, 2, 8>, dim3(ncol * big.nyt * big.nsp), dim3(512), 0, c->stream, f, big,
                  (const double *)k.pfg64);
  } else {
    const LegDims d = leg_dims(k, nf, npc, ncol, 16, (M + 63) / 64);
    probed_launch(probe, k_leg_fwd_f64m<16, 1, 16>, dim3(ncol * d.nyt * d.nsp), dim3(512), 0, c->stream, f, d,
                  (const double *)k.pfg64);
  }
  HIPCHK(hipGetLastError());
}

void leg_backward_f64(mlx_ctx *c, const double2 *const *in, double2 *const *out, const double *const *ln, int nf,
                      int ncols, bool ztail) {
  const KitDev &k = c->kit;
  const int npc = (ncols > 0 && ncols < k.npchop) ? ncols : k.npchop, ncol = ztail ? k.npdim : npc;
  const LegFields f = leg_fields(in, out, ln, nf);
  ProbeScope probe(c, MLX_PROBE_LEG_BWD, nf * leg_bytes(k, 0, 8, npc), nf * leg_flops(k, 0, npc));
  const LegDims d = leg_dims(k, nf, npc, ncol, 16, (k.nrh + 127) / 128);
  if (in[0] == out[0] && d.nsp > 1) MLX_THROW(MLX_E_ARG, "rtrans_backward: in place past 256 radial points");
  probed_launch(probe, k_leg_bwd_f64m, dim3(ncol * d.nyt * d.nsp), dim3(512), 0, c->stream, f, d, (const double *)k.pf);
  HIPCHK(hipGetLastError());
}

// the projection's columns mbeg .. mend - 1 on stream s (arguments as
// k_v2t_f64m's); every entry of those columns is written
void v2t_f64(mlx_ctx *c, hipStream_t s, const double2 *ur, const double2 *up, const double2 *uz, double2 *psi,
             double2 *chi, int npc, int zlo, int zhi, int mbeg, int mend, int ksplit, size_t zso, size_t kstride) {
  const KitDev &k = c->kit;
  const int M = (k.nrchop + 1) / 2;
  V2tArgs g;
  g.f[0] = ur, g.f[1] = up, g.f[2] = uz, g.out[0] = psi, g.out[1] = chi;
  g.t[0] = k.tVg64, g.t[1] = k.tDg64, g.t[2] = k.tTg64, g.ak = k.ak;
  g.nrdim = k.nrdim, g.npdim = k.npdim, g.nz = k.nzdim, g.nr = k.nr, g.nrh = k.nrh, g.nrc = k.nrchop, g.npc = npc;
  g.nzc = k.chopzl, g.nzcu = k.chopzu, g.zlo = zlo, g.zhi = zhi, g.mbeg = mbeg, g.mend = mend;
  g.tpitch = k.mfma_ap, g.ksplit = ksplit, g.zso = zso, g.kstride = kstride;
  g.nyt = (k.nzdim + 7) / 8, g.nsp = (M + 31) / 32;
  const dim3 grid((mend - mbeg) * g.nyt * g.nsp * ksplit);
  if (ksplit > 1) {
    if (mbeg != 0 || mend != 1) MLX_THROW(MLX_E_ARG, "vec2tp: radial shares of column 0 only");
    hipLaunchKernelGGL(k_v2t_f64m<true>, grid, dim3(256), 0, s, g);
  } else {
    hipLaunchKernelGGL(k_v2t_f64m<false>, grid, dim3(256), 0, s, g);
  }
  HIPCHK(hipGetLastError());
}

}  // namespace mlx
