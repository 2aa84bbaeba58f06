// phi and z Fourier transforms of the field, FP64, in LDS.
//
// Replaces horizontal_fft_forward/backward and vertical_fft_forward/backward
// (src/submodules/mlegs_scalar_ops.f90:1567-1848), which call FFTE's
// dzfft2d/zdfft2d/zfft1d per row.  Conventions kept from the reference:
//   phi forward : real row f_0..f_{np-1} packed as e(i, j) = f_{2j} + i f_{2j+1}
//                 -> C_m = (1/np) sum_t f_t e^{-2 pi i m t/np}, m = 0..np/2
//   phi backward: f_t = sum_m C_m e^{+2 pi i m t/np} (Hermitian), packed back;
//                 column np/2+1 (scratch in the reference) is written as 0
//   z forward   : (1/nz) sum e^{-2 pi i jk/nz};  z backward: sum e^{+...}
//   every row (including radial padding) and every column is transformed.
//
// Design: one workgroup owns TI consecutive radial rows i of one (k) plane
// (phi) or one (j) column (z), the line index fastest (coalesced global
// access, conflict-free LDS).  The powers of two from 16 to 256 take the
// four-step kernels (k_fft4, k_fft4_cross), other lengths the grouped Stockham
// kernels (k_fftg, k_fftg_cross); both read a line element from HBM once, straight into
// registers, and write it once.  The real-to-complex phi transform is a
// complex FFT of length np/2 plus the even/odd untangling step.  HBM-bound for
// large fields, launch-bound for small ones: up to kZBatch fields share a launch.
#include <algorithm>
#include <cmath>

#include "mlx_internal.h"

namespace {

constexpr int kThreads = 256;

// The fields of a launch (one per blockIdx.z), and rscale of each
struct FftFields {
  const double2 *in[mlx::kZBatch];
  double2 *out[mlx::kZBatch];
  int rs[mlx::kZBatch];
};

struct Cx {
  double x, y;
};
__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double2 cmuli(double2 a, double s) { return make_double2(-s * a.y, s * a.x); }  // i*s*a
// a w with its roundings written out: which product a contraction leaves
// rounded must not depend on the code around it (the solves behind the
// projection amplify a last bit by up to 1e9)
__device__ __forceinline__ double2 twmul(double2 a, double2 w) {
  return make_double2(__builtin_fma(a.x, w.x, -(a.y * w.y)), __builtin_fma(a.y, w.x, a.x * w.y));
}

// DFT of size R on v with sign sg (-1 forward, +1 inverse)
template <int R>
__device__ inline void dft(double2 *v, double sg);

template <>
__device__ inline void dft<2>(double2 *v, double) {
  double2 a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <>
__device__ inline void dft<4>(double2 *v, double sg) {
  double2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
  double2 b0 = cadd(v[1], v[3]), b1 = csub(v[1], v[3]);
  double2 ib1 = cmuli(b1, sg);  // (sg*i) * (v1 - v3)
  v[0] = cadd(a0, b0);
  v[2] = csub(a0, b0);
  v[1] = cadd(a1, ib1);
  v[3] = csub(a1, ib1);
}
template <>
__device__ inline void dft<3>(double2 *v, double sg) {
  const double c1 = -0.5, s1 = sg * 0.86602540378443864676;
  double2 t1 = cadd(v[1], v[2]), d = csub(v[1], v[2]);
  double2 t2 = make_double2(__builtin_fma(c1, t1.x, v[0].x), __builtin_fma(c1, t1.y, v[0].y));
  v[0] = cadd(v[0], t1);
  v[1] = make_double2(__builtin_fma(-s1, d.y, t2.x), __builtin_fma(s1, d.x, t2.y));
  v[2] = make_double2(__builtin_fma(s1, d.y, t2.x), __builtin_fma(-s1, d.x, t2.y));
}
template <>
__device__ inline void dft<5>(double2 *v, double sg) {
  const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
  const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
  auto f = [](double a, double b, double c) { return __builtin_fma(a, b, c); };
  double2 a14 = cadd(v[1], v[4]), b14 = csub(v[1], v[4]);
  double2 a23 = cadd(v[2], v[3]), b23 = csub(v[2], v[3]);
  double2 r1 = make_double2(f(c2, a23.x, f(c1, a14.x, v[0].x)), f(c2, a23.y, f(c1, a14.y, v[0].y)));
  double2 r2 = make_double2(f(c1, a23.x, f(c2, a14.x, v[0].x)), f(c1, a23.y, f(c2, a14.y, v[0].y)));
  double2 i1 = make_double2(f(s2, b23.x, s1 * b14.x), f(s2, b23.y, s1 * b14.y));
  double2 i2 = make_double2(f(s2, b14.x, -(s1 * b23.x)), f(s2, b14.y, -(s1 * b23.y)));
  double2 j1 = cmuli(i1, sg), j2 = cmuli(i2, sg);
  v[0] = make_double2(v[0].x + a14.x + a23.x, v[0].y + a14.y + a23.y);
  v[1] = cadd(r1, j1);
  v[4] = csub(r1, j1);
  v[2] = cadd(r2, j2);
  v[3] = csub(r2, j2);
}

// ---------------------------------------------------------------------------
// Fast path for the lengths N = N1 * N2 = 16 to 256 (powers of two): four-step
// FFT.  Stage 1 loads x[n2 + N2 n1] of a line straight into registers, runs
// the N1-point DFT over n1 there and applies W_N^{n2 k1}; one LDS exchange;
// stage 2 runs the N2-point DFT over n2 and writes X[k1 + N1 k2].  A
// workgroup owns TI consecutive rows (lines) of one column (z) or plane (phi),
// so every global access is a run of TI consecutive complex numbers.
// The real phi transform adds its even/odd untangling (forward) or tangling
// (backward) through a second LDS exchange.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr double c16(int q) {
  // cos(2 pi q / 16), q = 0..7
  return q == 0 ? 1.0 : q == 1 ? 0.92387953251128675613 : q == 2 ? 0.70710678118654752440
       : q == 3 ? 0.38268343236508977173 : q == 4 ? 0.0 : q == 5 ? -0.38268343236508977173
       : q == 6 ? -0.70710678118654752440 : -0.92387953251128675613;
}
__host__ __device__ constexpr double s16(int q) {
  // sin(2 pi q / 16), q = 0..7
  return q == 0 ? 0.0 : q == 1 ? 0.38268343236508977173 : q == 2 ? 0.70710678118654752440
       : q == 3 ? 0.92387953251128675613 : q == 4 ? 1.0 : q == 5 ? 0.92387953251128675613
       : q == 6 ? 0.70710678118654752440 : 0.38268343236508977173;
}
__host__ __device__ constexpr int bitrev(int i, int n) {
  int r = 0;
  for (int b = 1; b < n; b <<= 1) {
    r = (r << 1) | (i & 1);
    i >>= 1;
  }
  return r;
}

// in-register radix-2 DIT DFT of size N (N <= 16), sign sg of the exponent
// FP32 storage of physical fields (two floats per packed entry)
typedef float mlx_fv2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void st_nt_f32(double2 *base, size_t idx, double2 x) {
  const mlx_fv2 v = {(float)x.x, (float)x.y};
  __builtin_nontemporal_store(v, reinterpret_cast<mlx_fv2 *>(base) + idx);
}
__device__ __forceinline__ double2 ld_nt_f32(const double2 *base, size_t idx) {
  const mlx_fv2 v = __builtin_nontemporal_load(reinterpret_cast<const mlx_fv2 *>(base) + idx);
  return make_double2((double)v.x, (double)v.y);
}

template <int N>
__device__ __forceinline__ void dft_reg(double2 *v, double sg) {
  double2 t[N];
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = v[bitrev(i, N)];
#pragma unroll
  for (int len = 2; len <= N; len <<= 1) {
    const int h = len / 2;
#pragma unroll
    for (int i0 = 0; i0 < N; i0 += len) {
#pragma unroll
      for (int j = 0; j < h; ++j) {
        const double2 a = t[i0 + j];
        double2 b = t[i0 + j + h];
        if (j != 0) {
          const int q = j * (16 / len);
          const double cw = c16(q), sw = sg * s16(q);
          b = make_double2(b.x * cw - b.y * sw, b.x * sw + b.y * cw);
        }
        t[i0 + j] = make_double2(a.x + b.x, a.y + b.y);
        t[i0 + j + h] = make_double2(a.x - b.x, a.y - b.y);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = t[i];
}

__device__ __forceinline__ double2 twid(const double2 *tw, int idx, double sg) {
  double2 w = tw[idx];
  if (sg > 0) w.y = -w.y;
  return w;
}

// ---------------------------------------------------------------------------
// Any length N = 2^a 3^b 5^c up to 512: a Stockham FFT of radix 4, 2, 3 and 5
// passes (the plan's order), up to two passes of product <= 16 at a time in
// registers.  A group of passes that starts with ns transformed takes item j <
// N / NG to the NG elements j + i N / NG; its outputs go to (j / ns) ns NG +
// j % ns + e ns.  Between groups the lines go through LDS (two buffers); the
// first group reads HBM, the last one writes it.  The passes' arithmetic and
// its order are those of single passes through LDS (one pass, two barriers and
// an LDS round trip each), which this replaces, bit for bit: us a field at 150 x
// 120 x 90 (lengths 60 and 90), phi back 20.8 -> 18.7, phi forward 20.8 -> 10.2,
// z 20.5 -> 7.3; phi back at 64 x 48 x 32 (24) 9.9 -> 1.5 (six fields a launch).
// ---------------------------------------------------------------------------
struct FftGroups {
  int n, ng, til;     // length, groups, log2 of the rows per tile
  int type[5], ns[5]; // 16 R1 + R2 of each group (R2 = 1: a single pass), transformed before it
};

// keeps a value as it is rounded here: no contraction into what follows
__device__ __forceinline__ double2 rounded(double2 x) {
  asm volatile("" : "+v"(x.x), "+v"(x.y));
  return x;
}

template <int R1, int R2, class LD, class ST>
__device__ __forceinline__ void fft_group(int N, int ns, int til, const double2 *tw, double sg, LD ld, ST st) {
  constexpr int NG = R1 * R2;
  const int M = N / NG, s1 = N / (ns * R1), s2 = N / (ns * NG);
  const int TI = 1 << til;
  for (int b = threadIdx.x; b < (M << til); b += blockDim.x) {
    const int l = b & (TI - 1), j = b >> til;
    const int jq = j / ns, k = j - jq * ns;
    double2 v[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) v[i] = ld(j + i * M, l);
    double2 u[NG];  // u[r + R1 q]: output r of first-pass butterfly q
#pragma unroll
    for (int q = 0; q < R2; ++q) {
      double2 t[R1];
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        t[r] = v[q + r * R2];
        if (r > 0) {
          double2 w = tw[r * k * s1];
          if (sg > 0) w.y = -w.y;
          t[r] = twmul(t[r], w);
        }
      }
      dft<R1>(t, sg);
#pragma unroll
      for (int r = 0; r < R1; ++r) u[r + R1 * q] = t[r];
    }
    if constexpr (R2 > 1) {
#pragma unroll
      for (int r = 0; r < R1; ++r) {
        double2 t[R2];
        const int k2 = k + r * ns;
#pragma unroll
        for (int q = 0; q < R2; ++q) {
          t[q] = u[r + R1 * q];
          if (q > 0) {
            double2 w = tw[q * k2 * s2];
            if (sg > 0) w.y = -w.y;
            t[q] = twmul(t[q], w);
          }
        }
        dft<R2>(t, sg);
#pragma unroll
        for (int q = 0; q < R2; ++q) u[r + R1 * q] = t[q];
      }
    }
    const int base = jq * ns * NG + k;
#pragma unroll
    for (int e = 0; e < NG; ++e) st(base + e * ns, l, u[e]);
  }
}

template <class LD, class ST>
__device__ __forceinline__ void fft_group_of(int type, int N, int ns, int til, const double2 *tw, double sg, LD ld,
                                             ST st) {
  switch (type) {
    case 16 * 4 + 4: fft_group<4, 4>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 4 + 2: fft_group<4, 2>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 4 + 3: fft_group<4, 3>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 4 + 1: fft_group<4, 1>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 2 + 3: fft_group<2, 3>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 2 + 5: fft_group<2, 5>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 2 + 1: fft_group<2, 1>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 3 + 3: fft_group<3, 3>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 3 + 5: fft_group<3, 5>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 3 + 1: fft_group<3, 1>(N, ns, til, tw, sg, ld, st); break;
    case 16 * 1 + 1:  // length 1
      for (int l = threadIdx.x; l < (1 << til); l += blockDim.x) st(0, l, ld(0, l));
      break;
    default:  // (5, 1): groups_of makes no others
      fft_group<5, 1>(N, ns, til, tw, sg, ld, st);
      break;
  }
}

// All groups of one tile: ld0(n, l) the line elements, stN(n, l, v) takes the
// result.  A, B: two LDS buffers of N << til elements.
template <class LD, class ST>
__device__ __forceinline__ void fft_lines(const FftGroups &g, double2 *A, double2 *B, const double2 *tw, double sg,
                                          LD ld0, ST stN) {
  const int til = g.til, N = g.n;
  double2 *src = A, *dst = B;
  auto ldA = [&](int n, int l) { return src[(n << til) + l]; };
  auto stB = [&](int n, int l, double2 v) { dst[(n << til) + l] = v; };
  if (g.ng == 1) {
    fft_group_of(g.type[0], N, 1, til, tw, sg, ld0, stN);
    return;
  }
  fft_group_of(g.type[0], N, 1, til, tw, sg, ld0, stB);
  for (int i = 1; i < g.ng - 1; ++i) {
    __syncthreads();
    double2 *t = src;
    src = dst, dst = t;
    fft_group_of(g.type[i], N, g.ns[i], til, tw, sg, ldA, stB);
  }
  __syncthreads();
  src = dst;
  fft_group_of(g.type[g.ng - 1], N, g.ns[g.ng - 1], til, tw, sg, ldA, stN);
}

struct FftgArgs {
  FftGroups g;
  FftFields f;
  size_t es, gs;
  int nrow, act_nrc;
  const double2 *tw, *twh;
  double sg, scale;
  const double *r;
  int nr, mlim, zin_lo, zin_hi, zout_lo, zout_hi, pstride;
};

// C_m = E + W^m O, m = 0..N, scaled, from the N spectral values of a packed
// real line
__device__ __forceinline__ double2 untangle(double2 zm, double2 zc, double2 w, double scale) {
  // O = -i (zm - conj zc) / 2
  const double ox = 0.5 * (zm.y + zc.y), oy = -0.5 * (zm.x - zc.x);
  const double re = __builtin_fma(w.x, ox, -(oy * w.y)), im = __builtin_fma(w.x, oy, w.y * ox);
  return make_double2(__builtin_fma(0.5, zm.x + zc.x, re) * scale, __builtin_fma(0.5, zm.y - zc.y, im) * scale);
}

// MODE, PAIR, limits: as k_fft4.  MODE 2 reads the modes m and N - m of its
// inputs directly (the second time from the cache).
template <int MODE, bool PAIR>
__global__ void __launch_bounds__(kThreads) k_fftg(FftgArgs a) {
  extern __shared__ double2 lds[];
  const int N = a.g.n, til = a.g.til, TI = 1 << til;
  const int TH = PAIR ? TI / 2 : TI;  // input rows (or pairs) per tile
  const double2 *in = a.f.in[0];
  double2 *out = a.f.out[0];
  int rscale = a.f.rs[0];
#pragma unroll
  for (int q = 1; q < mlx::kZBatch; ++q)
    if (blockIdx.z == q) in = a.f.in[q], out = a.f.out[q], rscale = a.f.rs[q];
  const int i0 = blockIdx.x * TH;
  const size_t es = a.es, base = (size_t)blockIdx.y * a.gs;
  int rlim = a.nrow;
  if (a.act_nrc > 0) {
    const int v = a.act_nrc - (int)blockIdx.y;
    rlim = v < 0 ? 0 : (v < a.nrow ? v : a.nrow);
  }
  if (i0 >= rlim) return;  // the whole tile lies outside the active rows
  double2 *A = lds, *B = lds + ((size_t)N << til);
  if (MODE == 0) {
    auto ld = [&](int n, int l) {
      const bool skip = (n >= a.zin_lo && n <= a.zin_hi) || i0 + l >= rlim;
      return skip ? make_double2(0.0, 0.0) : ld_nt(&in[base + (size_t)n * es + i0 + l]);
    };
    auto st = [&](int n, int l, double2 v) {
      if (i0 + l < rlim && !(n >= a.zout_lo && n <= a.zout_hi))
        st_nt(&out[base + (size_t)n * es + i0 + l], make_double2(v.x * a.scale, v.y * a.scale));
    };
    fft_lines(a.g, A, B, a.tw, a.sg, ld, st);
  } else if (MODE == 1) {
    auto ld = [&](int n, int l) {
      const int i = i0 + l;
      double2 x = i < rlim ? ld_nt(&in[base + (size_t)n * es + i]) : make_double2(0.0, 0.0);
      if (rscale > 0 && i < a.nr) {
        const double rr = a.r[i];
        x = rounded(make_double2(x.x * rr, x.y * rr));
      }
      return x;
    };
    double2 *R = (a.g.ng & 1) ? B : A;  // not what the last group reads
    auto st = [&](int n, int l, double2 v) { R[(n << til) + l] = v; };
    fft_lines(a.g, A, B, a.tw, a.sg, ld, st);
    __syncthreads();
    for (int b = threadIdx.x; b < ((N + 1) << til); b += blockDim.x) {
      const int l = b & (TI - 1), m = b >> til;
      if (i0 + l >= rlim) continue;
      const double2 zm = R[((m == N ? 0 : m) << til) + l], zc = R[((m == 0 ? 0 : N - m) << til) + l];
      st_nt(&out[base + (size_t)m * es + i0 + l], untangle(zm, zc, a.twh[m], a.scale));
    }
  } else {
    const float4 *pin = reinterpret_cast<const float4 *>(in);
    const size_t npd = a.gs / es;
    auto mode = [&](int m, int l) {
      double2 v = make_double2(0.0, 0.0);
      if (m >= a.mlim) return v;
      if (PAIR) {
        const int x = i0 + (l & (TH - 1));
        if (x >= rlim) return v;
        const float4 p = pin[((size_t)blockIdx.y * npd + m) * a.pstride + x];
        const double ex = p.x, ey = p.y, ox = p.z, oy = p.w;
        return l < TH ? make_double2(ex + ox, ey + oy) : make_double2(ex - ox, ey - oy);
      }
      return i0 + l < rlim ? in[base + (size_t)m * es + i0 + l] : v;
    };
    auto ld = [&](int n, int l) {
      double2 cm = mode(n, l), cc = mode(N - n, l);
      if (n == 0) cm.y = 0.0, cc.y = 0.0;  // imaginary parts of DC and Nyquist are ignored
      cc.y = -cc.y;
      const double2 E = cadd(cm, cc);
      double2 w = a.twh[n];
      w.y = -w.y;
      const double2 O = twmul(csub(cm, cc), w);
      return rounded(make_double2(E.x - O.y, E.y + O.x));
    };
    // in place, every line of the tile has been read when the first value is
    // written: a barrier follows the first group (one group: a line is one
    // thread's, and its scratch column, element N, belongs to that thread too)
    auto st = [&](int n, int l, double2 v) {
      const int lx = PAIR ? (l & (TH - 1)) : l;
      if (i0 + lx >= rlim) return;
      const int i = (PAIR && l >= TH) ? a.nr - 1 - (i0 + lx) : i0 + lx;
      if (rscale < 0 && i < a.nr) {
        const double rr = a.r[i];
        v = make_double2(v.x / rr, v.y / rr);
      }
      st_nt(&out[base + (size_t)n * es + i], v);
      if (n == 0) st_nt(&out[base + (size_t)N * es + i], make_double2(0.0, 0.0));
    };
    fft_lines(a.g, A, B, a.tw, a.sg, ld, st);
  }
}

// MODE 0: complex transform (z); MODE 1: real forward (phi); MODE 2: real backward (phi)
// MODE 2: modes m >= mlim are taken as zero without being read.  MODE 0:
// line entries zin_lo..zin_hi are taken as zero without being read and
// outputs zout_lo..zout_hi are not written (their consumer does not read them)
// PAIR (MODE 2): the input is the backward radial contraction's float4
// (be, bo) per radial pair x < nrow at ((z npdim + m) pstride + x), npdim =
// gs / es (each line of pairs starts on a 256-byte boundary); a tile holds
// the pairs x0 .. x0 + TI/2 - 1 and synthesizes rows x = be + bo and
// nr - 1 - x = be - bo (formed in FP64 on load), rows < nr only.
// F32OUT (MODE 2): the output is stored in FP32 at f32_index (columns
// padded to 128-byte lines, half the bytes).
// gridDim.z > 1: the fields f.in[z] -> f.out[z] (same shape and limits, rscale
// f.rs[z]), one launch for all.
template <int N1, int N2, int TI, int NTH, int MODE, bool PAIR = false, bool F32OUT = false>
__global__ void __launch_bounds__(NTH) k_fft4(FftFields f, size_t es, size_t gs, int nrow,
                                                   int act_nrc, const double2 *tw, const double2 *twh, double sg,
                                                   double scale, const double *r, int nr, int mlim,
                                                   int zin_lo, int zin_hi, int zout_lo, int zout_hi,
                                                   int pstride) {
  constexpr int N = N1 * N2;
  const double2 *in = f.in[0];
  double2 *out = f.out[0];
  int rscale = f.rs[0];
  if (gridDim.z > 1) {
    in = f.in[blockIdx.z];
    out = f.out[blockIdx.z];
    rscale = f.rs[blockIdx.z];
  }
  constexpr int T1 = (TI * N2 + NTH - 1) / NTH;
  constexpr int T2 = (TI * N1 + NTH - 1) / NTH;
  constexpr bool HALF = (MODE == 0 && N == 256);
  __shared__ double2 buf[HALF ? TI * N / 2 : TI * N];
  __shared__ double2 nyq[MODE == 2 ? TI : 1];
  constexpr int TH = PAIR ? TI / 2 : TI;  // input rows (or pairs) per tile
  const int i0 = blockIdx.x * TH;
  const size_t base = (size_t)blockIdx.y * gs;
  int rlim = nrow;
  if (act_nrc > 0) {
    const int a = act_nrc - (int)blockIdx.y;
    rlim = a < 0 ? 0 : (a < nrow ? a : nrow);
  }
  if (i0 >= rlim) return;  // the whole tile lies outside the active rows
  const int tid = threadIdx.x;

  if (MODE == 2 && PAIR) {
    // stage 0 from radial pairs: tile rows l (x) and TH + l (nr - 1 - x)
    const float4 *pin = reinterpret_cast<const float4 *>(in);
    for (int b = tid; b < TH * (N + 1); b += NTH) {
      const int l = b % TH, m = b / TH, x = i0 + l;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      // an ordinary load: the pairs were just written and are read from the cache
      if (x < rlim && m < mlim) v = pin[((size_t)blockIdx.y * (gs / es) + m) * pstride + x];
      const double ex = v.x, ey = v.y, ox = v.z, oy = v.w;
      const double2 hi = make_double2(ex + ox, ey + oy), lo = make_double2(ex - ox, ey - oy);
      if (m < N) {
        buf[m * TI + l] = hi;
        buf[m * TI + TH + l] = lo;
      } else {
        nyq[l] = hi;
        nyq[TH + l] = lo;
      }
    }
    __syncthreads();
  } else if (MODE == 2) {
    // stage 0: C_m, m = 0..N, into LDS (C_N apart)
    for (int b = tid; b < TI * (N + 1); b += NTH) {
      const int l = b % TI, m = b / TI, i = i0 + l;
      const double2 v = (i < rlim && m < mlim) ? ld_nt(&in[base + (size_t)m * es + i]) : make_double2(0.0, 0.0);
      if (m < N) buf[m * TI + l] = v;
      else nyq[l] = v;
    }
    __syncthreads();
  }

  // stage 1
  double2 y1[T1][N1];
#pragma unroll
  for (int t = 0; t < T1; ++t) {
    const int b = tid + t * NTH;
    if (b < TI * N2) {
      const int l = b % TI, n2 = b / TI, i = i0 + l;
      double2 v[N1];
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
        const int j = n2 + N2 * n1;
        if (MODE == 2) {
          double2 cm = buf[j * TI + l];
          double2 cc = (j == 0) ? nyq[l] : buf[(N - j) * TI + l];
          if (j == 0) { cm.y = 0.0; cc.y = 0.0; }  // imaginary parts of DC and Nyquist are ignored
          cc.y = -cc.y;
          const double2 E = cadd(cm, cc);
          double2 w = twh[j];
          w.y = -w.y;
          const double2 O = cmul(csub(cm, cc), w);
          v[n1] = make_double2(E.x - O.y, E.y + O.x);
        } else {
          const bool zin = MODE == 0 && j >= zin_lo && j <= zin_hi;
          double2 x = (i < rlim && !zin) ? ld_nt(&in[base + (size_t)j * es + i]) : make_double2(0.0, 0.0);
          if (MODE == 1 && rscale > 0 && i < nr) {
            const double rr = r[i];
            x = make_double2(x.x * rr, x.y * rr);
          }
          v[n1] = x;
        }
      }
      dft_reg<N1>(v, sg);
#pragma unroll
      for (int k1 = 1; k1 < N1; ++k1) {
        const int q = (n2 * k1) & (N - 1);
        if (q) v[k1] = cmul(v[k1], twid(tw, q, sg));
      }
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) y1[t][k1] = v[k1];
    }
  }
  if (MODE == 2) __syncthreads();  // stage 0 data fully consumed
  double2 y2[T2][N2];
  if (HALF) {
    // the exchange in two halves through TI N doubles: real parts, then
    // imaginary parts
    double *bd = reinterpret_cast<double *>(buf);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();
#pragma unroll
      for (int t = 0; t < T1; ++t) {
        const int b = tid + t * NTH;
        if (b < TI * N2) {
          const int l = b % TI, n2 = b / TI;
#pragma unroll
          for (int k1 = 0; k1 < N1; ++k1) bd[(k1 * N2 + n2) * TI + l] = h ? y1[t][k1].y : y1[t][k1].x;
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < T2; ++t) {
        const int b = tid + t * NTH;
        if (b < TI * N1) {
          const int l = b % TI, k1 = b / TI;
#pragma unroll
          for (int n2 = 0; n2 < N2; ++n2) {
            if (h) y2[t][n2].y = bd[(k1 * N2 + n2) * TI + l];
            else y2[t][n2].x = bd[(k1 * N2 + n2) * TI + l];
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < T2; ++t)
      if (tid + t * NTH < TI * N1) dft_reg<N2>(y2[t], sg);
  } else {
#pragma unroll
    for (int t = 0; t < T1; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N2) {
        const int l = b % TI, n2 = b / TI;
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) buf[(k1 * N2 + n2) * TI + l] = y1[t][k1];
      }
    }
    __syncthreads();

    // stage 2
#pragma unroll
    for (int t = 0; t < T2; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N1) {
        const int l = b % TI, k1 = b / TI;
#pragma unroll
        for (int n2 = 0; n2 < N2; ++n2) y2[t][n2] = buf[(k1 * N2 + n2) * TI + l];
        dft_reg<N2>(y2[t], sg);
      }
    }
  }
  if (MODE == 0 || MODE == 2) {
#pragma unroll
    for (int t = 0; t < T2; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N1) {
        const int l = b % TI, k1 = b / TI;
        // the output row of tile row l (PAIR: pair x = i0 + l % TH)
        const int lx = PAIR ? l % TH : l;
        const int i = (PAIR && l >= TH) ? nr - 1 - (i0 + lx) : i0 + lx;
        if (i0 + lx < rlim) {
          double dv = 1.0;
          if (MODE == 2 && rscale < 0 && i < nr) dv = r[i];
#pragma unroll
          for (int k2 = 0; k2 < N2; ++k2) {
            const int ko = k1 + N1 * k2;
            if (MODE == 0 && ko >= zout_lo && ko <= zout_hi) continue;
            double2 x = y2[t][k2];
            if (MODE == 0) x = make_double2(x.x * scale, x.y * scale);
            else if (dv != 1.0) x = make_double2(x.x / dv, x.y / dv);
            if (F32OUT) st_nt_f32(out, f32_index(blockIdx.y, ko, i, es, gs / es), x);
            else st_nt(&out[base + (size_t)ko * es + i], x);
          }
          if (MODE == 2 && k1 == 0) {
            if (F32OUT) st_nt_f32(out, f32_index(blockIdx.y, N, i, es, gs / es), make_double2(0.0, 0.0));
            else st_nt(&out[base + (size_t)N * es + i], make_double2(0.0, 0.0));
          }
        }
      }
    }
    return;
  }
  // MODE 1: natural order into LDS, then C_m = E + W^m O, m = 0..N, scaled 1/np
  __syncthreads();
#pragma unroll
  for (int t = 0; t < T2; ++t) {
    const int b = tid + t * NTH;
    if (b < TI * N1) {
      const int l = b % TI, k1 = b / TI;
#pragma unroll
      for (int k2 = 0; k2 < N2; ++k2) buf[(k1 + N1 * k2) * TI + l] = y2[t][k2];
    }
  }
  __syncthreads();
  for (int b = tid; b < TI * (N + 1); b += NTH) {
    const int l = b % TI, m = b / TI, i = i0 + l;
    const double2 zm = buf[(m % N) * TI + l];
    double2 zc = buf[((N - m) % N) * TI + l];
    zc.y = -zc.y;
    const double2 E = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
    const double2 D = make_double2(0.5 * (zm.x - zc.x), 0.5 * (zm.y - zc.y));
    const double2 O = make_double2(D.y, -D.x);  // -i * D
    const double2 C = cadd(E, cmul(twh[m], O));
    if (i < rlim) st_nt(&out[base + (size_t)m * es + i], make_double2(C.x * scale, C.y * scale));
  }
}

// Forward phi transform of the three components of v x w, straight from the
// six physical (PPP, packed real) fields: vector_product
// (mlegs_scalar_ops.f90:1561-1566, here with the background axial flow ub
// added to v_z first, vortical_flow_3d.f90:381) followed by the first step
// of vector_projection (:1320-1336: r v_r, r v_phi and v_z to PFP).  Stage 1
// of the four-step transform forms the products while loading, so each
// input is read once and no physical product field is written.  Rows
// i >= nr give zero products, as vector_product leaves them.
// F32IN: the six velocity and vorticity fields are stored in FP32 at
// f32_index (ub, the background flow, stays FP64).
template <int N1, int N2, int TI, int NTH, bool F32IN = false>
__global__ void __launch_bounds__(NTH) k_fft4_cross(double2 *o0, double2 *o1, double2 *o2, const double2 *v0,
                                                         const double2 *v1, const double2 *v2, const double2 *w0,
                                                         const double2 *w1, const double2 *w2, const double2 *ub,
                                                         size_t es, size_t gs, int nrow, const double2 *tw,
                                                         const double2 *twh, double scale, const double *r, int nr,
                                                         double *ln0, double *ln1, double *ln2, int mmax) {
  constexpr int N = N1 * N2;
  constexpr int T1 = (TI * N2 + NTH - 1) / NTH;
  constexpr int T2 = (TI * N1 + NTH - 1) / NTH;
  const double sg = -1.0;
  __shared__ double2 buf[TI * N];
  const int i0 = blockIdx.x * TI;
  const size_t base = (size_t)blockIdx.y * gs;
  // the products carry no log term
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    if (ln0) ln0[0] = 0.0;
    if (ln1) ln1[0] = 0.0;
    if (ln2) ln2[0] = 0.0;
  }
  if (i0 >= nrow) return;
  const int tid = threadIdx.x;

  // stage 1, all three components
  double2 y1[3][T1][N1];
#pragma unroll
  for (int t = 0; t < T1; ++t) {
    const int b = tid + t * NTH;
    if (b < TI * N2) {
      const int l = b % TI, n2 = b / TI, i = i0 + l;
      double2 c0[N1], c1[N1], c2[N1];
      const double rr = (i < nr) ? r[i] : 0.0;
#pragma unroll
      for (int n1 = 0; n1 < N1; ++n1) {
        const int j = n2 + N2 * n1;
        const double2 z2 = make_double2(0.0, 0.0);
        double2 a1 = z2, a2 = z2, a3 = z2, b1 = z2, b2 = z2, b3 = z2;
        if (i < nr) {
          const size_t o = base + (size_t)j * es + i;
          if (F32IN) {
            const size_t o32 = f32_index(blockIdx.y, j, i, es, gs / es);
            a1 = ld_nt_f32(v0, o32);
            a2 = ld_nt_f32(v1, o32);
            a3 = ld_nt_f32(v2, o32);
            b1 = ld_nt_f32(w0, o32);
            b2 = ld_nt_f32(w1, o32);
            b3 = ld_nt_f32(w2, o32);
          } else {
            a1 = ld_nt(&v0[o]);
            a2 = ld_nt(&v1[o]);
            a3 = ld_nt(&v2[o]);
            b1 = ld_nt(&w0[o]);
            b2 = ld_nt(&w1[o]);
            b3 = ld_nt(&w2[o]);
          }
          if (ub) {
            const double2 u = ld_nt(&ub[o]);
            a3 = make_double2(a3.x + u.x, a3.y + u.y);
          }
        }
        const double2 pr = make_double2(a2.x * b3.x - a3.x * b2.x, a2.y * b3.y - a3.y * b2.y);
        const double2 pp = make_double2(a3.x * b1.x - a1.x * b3.x, a3.y * b1.y - a1.y * b3.y);
        c2[n1] = make_double2(a1.x * b2.x - a2.x * b1.x, a1.y * b2.y - a2.y * b1.y);
        c0[n1] = make_double2(pr.x * rr, pr.y * rr);
        c1[n1] = make_double2(pp.x * rr, pp.y * rr);
      }
      dft_reg<N1>(c0, sg);
      dft_reg<N1>(c1, sg);
      dft_reg<N1>(c2, sg);
#pragma unroll
      for (int k1 = 1; k1 < N1; ++k1) {
        const int q = (n2 * k1) & (N - 1);
        if (q) {
          const double2 w = twid(tw, q, sg);
          c0[k1] = cmul(c0[k1], w);
          c1[k1] = cmul(c1[k1], w);
          c2[k1] = cmul(c2[k1], w);
        }
      }
#pragma unroll
      for (int k1 = 0; k1 < N1; ++k1) {
        y1[0][t][k1] = c0[k1];
        y1[1][t][k1] = c1[k1];
        y1[2][t][k1] = c2[k1];
      }
    }
  }
#pragma unroll
  for (int comp = 0; comp < 3; ++comp) {
    double2 *out = comp == 0 ? o0 : comp == 1 ? o1 : o2;
    if (comp > 0) __syncthreads();  // the previous component's untangling has read buf
#pragma unroll
    for (int t = 0; t < T1; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N2) {
        const int l = b % TI, n2 = b / TI;
#pragma unroll
        for (int k1 = 0; k1 < N1; ++k1) buf[(k1 * N2 + n2) * TI + l] = y1[comp][t][k1];
      }
    }
    __syncthreads();
    double2 y2[T2][N2];
#pragma unroll
    for (int t = 0; t < T2; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N1) {
        const int l = b % TI, k1 = b / TI;
#pragma unroll
        for (int n2 = 0; n2 < N2; ++n2) y2[t][n2] = buf[(k1 * N2 + n2) * TI + l];
        dft_reg<N2>(y2[t], sg);
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T2; ++t) {
      const int b = tid + t * NTH;
      if (b < TI * N1) {
        const int l = b % TI, k1 = b / TI;
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) buf[(k1 + N1 * k2) * TI + l] = y2[t][k2];
      }
    }
    __syncthreads();
    // C_m = E + W^m O, m = 0..N, scaled 1/np
    for (int b = tid; b < TI * (N + 1); b += NTH) {
      const int l = b % TI, m = b / TI, i = i0 + l;
      const double2 zm = buf[(m % N) * TI + l];
      double2 zc = buf[((N - m) % N) * TI + l];
      zc.y = -zc.y;
      const double2 E = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      const double2 D = make_double2(0.5 * (zm.x - zc.x), 0.5 * (zm.y - zc.y));
      const double2 O = make_double2(D.y, -D.x);  // -i * D
      const double2 C = cadd(E, cmul(twh[m], O));
      if (i < nrow && m < mmax) st_nt(&out[base + (size_t)m * es + i], make_double2(C.x * scale, C.y * scale));
    }
  }
}

// k_fft4_cross for any length (FP64 fields): component blockIdx.z of the
// product per workgroup, formed while loading the first group
struct CrossArgs {
  FftGroups g;
  double2 *o[3];
  const double2 *v[3], *w[3], *ub;
  double *ln[3];
  size_t es, gs;
  int nrow, nr, mmax;
  const double2 *tw, *twh;
  double scale;
  const double *r;
};
__global__ void __launch_bounds__(kThreads) k_fftg_cross(CrossArgs a) {
  extern __shared__ double2 lds[];
  const int N = a.g.n, til = a.g.til, TI = 1 << til;
  // the three components of a tile 8 workgroups apart: on one XCD, at about
  // the same time, so that its L2 serves two of the three reads of each field
  const int comp = blockIdx.x % 24 / 8, i0 = (blockIdx.x / 24 * 8 + blockIdx.x % 8) * TI;
  const size_t es = a.es, base = (size_t)blockIdx.y * a.gs;
  // the products carry no log term
  if (i0 == 0 && blockIdx.y == 0 && threadIdx.x == 0 && a.ln[comp]) a.ln[comp][0] = 0.0;
  if (i0 >= a.nrow) return;
  double2 *A = lds, *B = lds + ((size_t)N << til);
  // components of v x w: (2,3), (3,1), (1,2)
  const int p = comp == 0 ? 1 : comp == 1 ? 2 : 0, q = comp == 0 ? 2 : comp == 1 ? 0 : 1;
  auto ld = [&](int n, int l) {
    const int i = i0 + l;
    if (i >= a.nr) return make_double2(0.0, 0.0);
    const size_t o = base + (size_t)n * es + i;
    double2 ap = a.v[p][o], aq = a.v[q][o];
    const double2 bp = a.w[p][o], bq = a.w[q][o];
    if (a.ub && (p == 2 || q == 2)) {
      const double2 u = a.ub[o];
      if (p == 2) ap = rounded(make_double2(ap.x + u.x, ap.y + u.y));
      if (q == 2) aq = rounded(make_double2(aq.x + u.x, aq.y + u.y));
    }
    double2 c = make_double2(__builtin_fma(ap.x, bq.x, -(aq.x * bp.x)), __builtin_fma(ap.y, bq.y, -(aq.y * bp.y)));
    if (comp < 2) {
      const double rr = a.r[i];
      c = rounded(make_double2(c.x * rr, c.y * rr));
    }
    return c;
  };
  double2 *R = (a.g.ng & 1) ? B : A;
  auto st = [&](int n, int l, double2 v) { R[(n << til) + l] = v; };
  fft_lines(a.g, A, B, a.tw, -1.0, ld, st);
  __syncthreads();
  for (int b = threadIdx.x; b < (a.mmax << til); b += blockDim.x) {
    const int l = b & (TI - 1), m = b >> til;
    if (i0 + l >= a.nrow) continue;
    const double2 zm = R[((m == N ? 0 : m) << til) + l], zc = R[((m == 0 ? 0 : N - m) << til) + l];
    st_nt(&a.o[comp][base + (size_t)m * es + i0 + l], untangle(zm, zc, a.twh[m], a.scale));
  }
}

// Tiles of ti rows leave the card less than two workgroups to a CU: small
// tiles (128 or 256 bytes of a line) then, each with the threads its items
// need.  One slice of 128 x 128 is 4 workgroups of 32 rows: the fused product
// takes 14.5 us there and 11.3 in tiles of 8, the phi transforms 8.2 and 7.1;
// one slice of 256 x 256 15.9 against 15.1.  With two workgroups to a CU the
// large tiles' longer lines are as fast or faster.
bool few_tiles(int nrow, int ti, int nwg) { return (nrow + ti - 1) / ti * nwg < 512; }

// grid_y: columns or planes (y) and fields (z) of the launch; false when N is
// no length of the four-step kernels
template <int MODE, bool PAIR = false, bool F32OUT = false>
bool launch_fft4(mlx_ctx *c, ProbeScope &ps, int N, dim3 grid_y, const FftFields &f, size_t es, size_t gs, int nrow,
                 int act_nrc, const double2 *tw, const double2 *twh, double sg, double scale, int mlim = 1 << 30,
                 int zin_lo = 1, int zin_hi = 0, int zout_lo = 1, int zout_hi = 0, int pstride = 0) {
  const KitDev &k = c->kit;
// NTH_ threads; small grids take TS_ rows a tile and TS_ max(N1, N2) threads
#define MLX_FFT4_(N1_, N2_, TI_, NTH_)                                                                             \
  do {                                                                                                             \
    constexpr int TH_ = PAIR ? TI_ / 2 : TI_;                                                                      \
    dim3 grid((nrow + TH_ - 1) / TH_, grid_y.y, grid_y.z);                                                         \
    probed_launch(ps, k_fft4<N1_, N2_, TI_, NTH_, MODE, PAIR, F32OUT>, grid, dim3(NTH_), 0, c->stream, f, es, gs, \
                  nrow, act_nrc, tw, twh, sg, scale, k.r, k.nr, mlim, zin_lo, zin_hi, zout_lo, zout_hi, pstride);  \
    return true;                                                                                                   \
  } while (0)
#define MLX_FFT4(N1_, N2_, TI_, TS_)                                                                               \
  do {                                                                                                             \
    if (few_tiles(PAIR ? 2 * nrow : nrow, TI_, grid_y.y * grid_y.z)) MLX_FFT4_(N1_, N2_, TS_, TS_ * N2_);          \
    MLX_FFT4_(N1_, N2_, TI_, kThreads);                                                                            \
  } while (0)
  switch (N) {
    case 16: MLX_FFT4(4, 4, 64, 16);
    case 32: MLX_FFT4(4, 8, 64, 8);
    case 64: MLX_FFT4(8, 8, 32, 8);
    case 128: MLX_FFT4(8, 16, 16, 8);
    case 256:
      if (MODE == 0) MLX_FFT4_(16, 16, 16, kThreads);  // 64 KiB of LDS
      MLX_FFT4_(16, 16, 8, kThreads);                  // the real modes also hold the Nyquist column
    default: return false;
  }
#undef MLX_FFT4
#undef MLX_FFT4_
}

// the pairs of passes that fft_group_of has a kernel for
constexpr bool pair_built(int r1, int r2) {
  return r1 == 4 ? r2 <= 4 : (r1 == 2 || r1 == 3) && (r2 == 3 || r2 == 5);
}

// The groups of a plan: the two whose larger one is the smallest (the most
// lines in flight: a group of NG elements is one thread's), or, where two
// groups of at most 16 do not cover the length, pairs of passes in turn.  Rows
// per tile: as many as leave nwg workgroups per row of tiles to fill the card
// twice, within 24 KB a buffer; at least 8 (one line of 128 bytes) where the
// buffers allow.
FftGroups groups_of(const FftPlan &pl, int nrow, int nwg) {
  FftGroups g;
  g.n = pl.n;
  g.ng = 0;
  int ns = 1;
  auto add = [&](int p, int n) {
    if (g.ng == 5) MLX_THROW(MLX_E_ARG, "fft: length above 512 is not supported");
    const int r1 = pl.radix[p], r2 = n > 1 ? pl.radix[p + 1] : 1;
    g.type[g.ng] = 16 * r1 + r2;
    g.ns[g.ng++] = ns;
    ns *= r1 * r2;
  };
  auto size = [&](int p, int n) {
    if (n < 1 || n > 2 || (n == 2 && !pair_built(pl.radix[p], pl.radix[p + 1]))) return 1 << 30;
    return pl.radix[p] * (n > 1 ? pl.radix[p + 1] : 1);
  };
  int cut = 0, best = 17;
  for (int p = 1; p < pl.npass; ++p) {
    const int m = std::max(size(0, p), size(p, pl.npass - p));
    if (m < best) best = m, cut = p;
  }
  if (pl.npass == 0) {
    g.type[0] = 17, g.ns[0] = 1, g.ng = 1;
  } else if (cut > 0) {
    add(0, cut);
    add(cut, pl.npass - cut);
  } else {
    for (int p = 0; p < pl.npass;) {
      const int n = (p + 1 < pl.npass && size(p, 2) <= 16) ? 2 : 1;
      add(p, n);
      p += n;
    }
  }
  g.til = 5;
  while (g.til > 3 && (((size_t)pl.n << g.til) > 1536 || ((nrow + (1 << g.til) - 1) >> g.til) * nwg < 512)) --g.til;
  while (g.til > 2 && ((size_t)pl.n << g.til) > 2048) --g.til;
  return g;
}
// threads of a workgroup: one per item of the group with the most, up to kThreads
unsigned group_threads(const FftGroups &g) {
  int most = 1;
  for (int i = 0; i < g.ng; ++i) most = std::max(most, g.n / ((g.type[i] / 16) * (g.type[i] % 16)));
  const int t = ((most << g.til) + 63) / 64 * 64;
  return t < kThreads ? t : kThreads;
}

template <int MODE, bool PAIR = false>
void launch_fftg(mlx_ctx *c, ProbeScope &ps, const FftPlan &pl, dim3 grid_y, const FftFields &f, size_t es, size_t gs,
                 int nrow, int act_nrc, const double2 *tw, const double2 *twh, double sg, double scale,
                 int mlim = 1 << 30, int zin_lo = 1, int zin_hi = 0, int zout_lo = 1, int zout_hi = 0,
                 int pstride = 0) {
  const KitDev &k = c->kit;
  FftgArgs a;
  a.g = groups_of(pl, PAIR ? 2 * nrow : nrow, grid_y.y * grid_y.z);
  a.f = f, a.es = es, a.gs = gs, a.nrow = nrow, a.act_nrc = act_nrc, a.tw = tw, a.twh = twh, a.sg = sg;
  a.scale = scale, a.r = k.r, a.nr = k.nr, a.mlim = mlim, a.zin_lo = zin_lo, a.zin_hi = zin_hi;
  a.zout_lo = zout_lo, a.zout_hi = zout_hi, a.pstride = pstride;
  const int th = PAIR ? (1 << a.g.til) / 2 : 1 << a.g.til;
  const dim3 grid((nrow + th - 1) / th, grid_y.y, grid_y.z);
  probed_launch(ps, k_fftg<MODE, PAIR>, grid, dim3(group_threads(a.g)), (unsigned)(2 * sizeof(double2) * pl.n << a.g.til),
                c->stream, a);
}

FftFields one_field(double2 *out, const double2 *in, int rs) {
  FftFields f;
  for (int q = 0; q < mlx::kZBatch; ++q) f.in[q] = in, f.out[q] = out, f.rs[q] = rs;
  return f;
}

bool pow2_line(int N) { return N == 16 || N == 32 || N == 64 || N == 128 || N == 256; }

}  // namespace

namespace mlx {

bool fft_f32_rows(const KitDev &k) { return k.np > 1 && pow2_line(k.nph); }

void fft_phi_batch(mlx_ctx *c, double2 *const *out, const double2 *const *in, int nf, int dir, const int *rscale,
                   int mlim, bool phys_rows) {
  const KitDev &k = c->kit;
  if (k.np <= 1 || nf <= 0) return;
  if (k.nph > 512) MLX_THROW(MLX_E_ARG, "fft_phi: np/2 above 512 is not supported");
  if (nf > kZBatch) MLX_THROW(MLX_E_ARG, "fft_phi: at most kZBatch fields per launch");
  // packed reals in, nph+1 modes out (or back): nr rows x nz slices
  const double nread = (mlim > 0 && mlim < k.nph + 1) ? mlim : k.nph + 1;
  ProbeScope probe(c, MLX_PROBE_FFT_PHI, 16.0 * nf * k.nr * k.nz * (dir > 0 ? nread + k.nph : 2.0 * k.nph + 1),
                   2.5 * nf * k.np * std::log2((double)k.np) * k.nr * k.nz);
  const size_t plane = (size_t)k.nrdim * k.npdim;
  const dim3 gy(1, k.nzdim, nf);
  FftFields f;
  for (int q = 0; q < kZBatch; ++q) {
    const int j = q < nf ? q : 0;
    f.in[q] = in[j], f.out[q] = out[j], f.rs[q] = rscale ? rscale[j] : 0;
  }
  if (dir < 0) {
    if (!launch_fft4<1>(c, probe, k.nph, gy, f, k.nrdim, plane, k.nrdim, 0, k.tw_nph, k.tw_half, -1.0, 1.0 / k.np))
      launch_fftg<1>(c, probe, k.plan_nph, gy, f, k.nrdim, plane, k.nrdim, 0, k.tw_nph, k.tw_half, -1.0, 1.0 / k.np);
  } else {
    const int rows = phys_rows ? k.nr : k.nrdim, ml = mlim > 0 ? mlim : 1 << 30;
    if (!launch_fft4<2>(c, probe, k.nph, gy, f, k.nrdim, plane, rows, 0, k.tw_nph, k.tw_half, +1.0, 1.0, ml))
      launch_fftg<2>(c, probe, k.plan_nph, gy, f, k.nrdim, plane, rows, 0, k.tw_nph, k.tw_half, +1.0, 1.0, ml);
  }
  HIPCHK(hipGetLastError());
}

void fft_phi(mlx_ctx *c, double2 *out, const double2 *in, int dir, int rscale, int mlim, bool phys_rows) {
  fft_phi_batch(c, &out, &in, 1, dir, &rscale, mlim, phys_rows);
}

// The backward phi transform of the radial pairs that leg_backward_pairs_f32
// writes: rows x and nr - 1 - x (x < nr / 2) of the PPP output, rows >= nr
// left as they are.  mlim: modes m >= mlim are taken as zero.
void fft_phi_pairs(mlx_ctx *c, double2 *out, const float4 *pairs, int rscale, int mlim, bool f32out) {
  const KitDev &k = c->kit;
  if (k.np <= 1 || k.nph > 512 || (k.nr & 1)) MLX_THROW(MLX_E_ARG, "fft_phi: radial pairs need 1 < np/2 <= 512");
  if (f32out && !fft_f32_rows(k)) MLX_THROW(MLX_E_ARG, "fft_phi: FP32 rows need a power-of-two np/2");
  const double nread = (mlim > 0 && mlim < k.nph + 1) ? mlim : k.nph + 1;
  ProbeScope probe(c, MLX_PROBE_FFT_PHI, 8.0 * k.nr * k.nz * nread + (f32out ? 8.0 : 16.0) * k.nr * k.nz * k.nph,
                   2.5 * k.np * std::log2((double)k.np) * k.nr * k.nz);
  const size_t plane = (size_t)k.nrdim * k.npdim;
  const FftFields f = one_field(out, reinterpret_cast<const double2 *>(pairs), rscale);
  const int ml = mlim > 0 ? mlim : 1 << 30;
  const dim3 gy(1, k.nzdim, 1);
  if (f32out)
    launch_fft4<2, true, true>(c, probe, k.nph, gy, f, k.nrdim, plane, k.nrh, 0, k.tw_nph, k.tw_half, +1.0, 1.0, ml, 1,
                               0, 1, 0, pair_stride(k));
  else if (!launch_fft4<2, true>(c, probe, k.nph, gy, f, k.nrdim, plane, k.nrh, 0, k.tw_nph, k.tw_half, +1.0, 1.0, ml,
                                 1, 0, 1, 0, pair_stride(k)))
    launch_fftg<2, true>(c, probe, k.plan_nph, gy, f, k.nrdim, plane, k.nrh, 0, k.tw_nph, k.tw_half, +1.0, 1.0, ml, 1,
                         0, 1, 0, pair_stride(k));
  HIPCHK(hipGetLastError());
}

void fft_phi_cross(mlx_ctx *c, double2 *o0, double2 *o1, double2 *o2, const double2 *v0, const double2 *v1,
                   const double2 *v2, const double2 *w0, const double2 *w1, const double2 *w2, const double2 *ub,
                   double *ln0, double *ln1, double *ln2, int mmax, bool f32in) {
  const KitDev &k = c->kit;
  const int N = k.nph;
  if (mmax <= 0 || mmax > N + 1) mmax = N + 1;
  if (k.np <= 1 || N > 512) MLX_THROW(MLX_E_ARG, "fft_phi: the fused product needs 1 < np/2 <= 512");
  if (f32in && !fft_f32_rows(k)) MLX_THROW(MLX_E_ARG, "fft_phi: FP32 rows need a power-of-two np/2");
  const size_t plane = (size_t)k.nrdim * k.npdim;
  // six physical fields (FP32 or FP64) and ub read (rows < nr), three PFP
  // fields written
  ProbeScope probe(c, MLX_PROBE_PHI_CROSS, k.nr * k.nz * ((f32in ? 48.0 : 96.0) * N + 16.0 * N + 48.0 * mmax),
                   3.0 * 2.5 * k.np * std::log2((double)k.np) * k.nr * k.nz + 18.0 * k.nr * k.np * k.nz);
#define MLX_FFTX_(N1_, N2_, TI_, NTH_)                                                                          \
  do {                                                                                                          \
    dim3 grid((k.nrdim + TI_ - 1) / TI_, k.nzdim);                                                              \
    if (f32in)                                                                                                  \
      probed_launch(probe, k_fft4_cross<N1_, N2_, TI_, NTH_, true>, grid, dim3(NTH_), 0, c->stream, o0, o1, o2, v0, \
                    v1, v2, w0, w1, w2, ub, (size_t)k.nrdim, plane, k.nrdim, k.tw_nph, k.tw_half, 1.0 / k.np, k.r, \
                    k.nr, ln0, ln1, ln2, mmax);                                                                 \
    else                                                                                                        \
      probed_launch(probe, k_fft4_cross<N1_, N2_, TI_, NTH_, false>, grid, dim3(NTH_), 0, c->stream, o0, o1, o2, \
                    v0, v1, v2, w0, w1, w2, ub, (size_t)k.nrdim, plane, k.nrdim, k.tw_nph, k.tw_half, 1.0 / k.np, \
                    k.r, k.nr, ln0, ln1, ln2, mmax);                                                            \
  } while (0)
// a small tile of 32 points has the large one's thread pattern (one item each
// in stage 2, none idle): the compiler then fuses the same products, and a
// slice's result does not depend on the tile
#define MLX_FFTX(N1_, N2_, TI_, TS_, NS_)                                                                       \
  do {                                                                                                          \
    if (few_tiles(k.nrdim, TI_, k.nzdim)) MLX_FFTX_(N1_, N2_, TS_, NS_);                                        \
    else MLX_FFTX_(N1_, N2_, TI_, kThreads);                                                                    \
  } while (0)
  switch (N) {
    case 16: MLX_FFTX(4, 4, 64, 16, 64); break;
    case 32: MLX_FFTX(4, 8, 64, 16, 64); break;
    case 64: MLX_FFTX(8, 8, 32, 8, 64); break;
    case 128: MLX_FFTX(8, 16, 16, 8, 128); break;
    case 256: MLX_FFTX_(16, 16, 8, kThreads); break;
    default: {
      CrossArgs a;
      a.g = groups_of(k.plan_nph, k.nrdim, 3 * k.nzdim);
      a.o[0] = o0, a.o[1] = o1, a.o[2] = o2, a.v[0] = v0, a.v[1] = v1, a.v[2] = v2;
      a.w[0] = w0, a.w[1] = w1, a.w[2] = w2, a.ub = ub, a.ln[0] = ln0, a.ln[1] = ln1, a.ln[2] = ln2;
      a.es = k.nrdim, a.gs = plane, a.nrow = k.nrdim, a.nr = k.nr, a.mmax = mmax, a.tw = k.tw_nph, a.twh = k.tw_half;
      a.scale = 1.0 / k.np, a.r = k.r;
      const int ti = 1 << a.g.til;
      const int nt = (k.nrdim + ti - 1) / ti;
      probed_launch(probe, k_fftg_cross, dim3((nt + 7) / 8 * 24, k.nzdim), dim3(group_threads(a.g)),
                    (unsigned)(2 * sizeof(double2) * N << a.g.til), c->stream, a);
    }
  }
#undef MLX_FFTX
#undef MLX_FFTX_
  HIPCHK(hipGetLastError());
}

void fft_z_batch(mlx_ctx *c, double2 *const *e, int nf, int dir, double ncol, int act_nrc, int ncols, int zin_lo,
                 int zin_hi, int zout_lo, int zout_hi) {
  const KitDev &k = c->kit;
  if (k.nz <= 1 || nf <= 0) return;
  if (k.nz > 512) MLX_THROW(MLX_E_ARG, "fft_z: nz above 512 is not supported");
  if (nf > kZBatch) MLX_THROW(MLX_E_ARG, "fft_z: at most kZBatch fields per launch");
  if (ncols <= 0 || ncols > k.npdim) ncols = k.npdim;
  auto span = [&](int lo, int hi) {
    lo = lo < 0 ? 0 : lo;
    hi = hi > k.nz - 1 ? k.nz - 1 : hi;
    return hi >= lo ? hi - lo + 1 : 0;
  };
  // entries read and written per line (the skipped ranges neither)
  ProbeScope probe(c, MLX_PROBE_FFT_Z,
                   16.0 * nf * ncol * (2.0 * k.nz - span(zin_lo, zin_hi) - span(zout_lo, zout_hi)),
                   5.0 * nf * k.nz * std::log2((double)k.nz) * ncol);
  FftFields f;
  for (int q = 0; q < kZBatch; ++q) f.in[q] = f.out[q] = e[q < nf ? q : 0], f.rs[q] = 0;
  const size_t zs = (size_t)k.nrdim * k.npdim;
  const double sg = dir < 0 ? -1.0 : 1.0, sc = dir < 0 ? 1.0 / k.nz : 1.0;
  const dim3 gy(1, ncols, nf);
  if (!launch_fft4<0>(c, probe, k.nz, gy, f, zs, k.nrdim, k.nrdim, act_nrc, k.tw_nz, nullptr, sg, sc, 1 << 30, zin_lo,
                      zin_hi, zout_lo, zout_hi))
    launch_fftg<0>(c, probe, k.plan_nz, gy, f, zs, k.nrdim, k.nrdim, act_nrc, k.tw_nz, nullptr, sg, sc, 1 << 30,
                   zin_lo, zin_hi, zout_lo, zout_hi);
  HIPCHK(hipGetLastError());
}

void fft_z(mlx_ctx *c, double2 *e, int dir, double ncol, int act_nrc, int ncols, int zin_lo, int zin_hi,
           int zout_lo, int zout_hi) {
  fft_z_batch(c, &e, 1, dir, ncol, act_nrc, ncols, zin_lo, zin_hi, zout_lo, zout_hi);
}

}  // namespace mlx
