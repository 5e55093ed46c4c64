// facg_batch.hip -- FACG() (Gfix/FACG.c:238-392) for many small lattices of
// one shape in a single launch: one workgroup owns one lattice and runs its
// whole gauge fixing -- theta test, steepest-descent start, Polak-Ribiere
// CG with Fourier acceleration and the three-probe line search, GLU's
// continuation below 1e3 acc and its 123456789 sentinel -- with workgroup
// barriers only.  No workgroup waits for another, so the launch needs no
// grid-wide synchronisation and every workgroup ends when its own lattice
// stops.
//
// On a small lattice the iteration of the context path is bound by the
// latency of its eight dependent launches (an 8^4 iteration takes 34 us, of
// which the bytes account for a few); here one launch carries every
// iteration of hundreds of lattices.
//
// Arithmetic is FP64 throughout.  The caller's links (GLU's layout, fixed
// in place) are copied at the start into device scratch as the first two
// columns of each link in structure-of-arrays planes, the layout the
// context path streams, and written back in GLU's layout at the end with
// the third column completed.  The fields in, sn and in_old (4 packed
// complex fields each, Gfix/FACG.c:57-60) live in the same scratch, sn
// twice: the CG update is formed inside the line-search probes, which
// write the new direction beside the old one.
// The Fourier acceleration transforms each axis (extents up to 16) on
// pencils in registers, by an FFT of the extent's prime factors: the x, y, z
// transforms of each time slice
// staged in LDS, the t transforms with the p^2 factor between them, so
// three passes over the fields.  Reductions are workgroup sums in a fixed order.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "../../include/glu_gfix.h"
#include "gfix_ctx.h"

using namespace gfix;

namespace {

constexpr int kMaxWgWaves = 8;  // workgroups of up to 512 threads
constexpr int kMaxExtent = 16;
constexpr double kCgTolB = 5e-11;     // CG_TOL, Headers/GLU_definitions.h:449-455
constexpr double kPl1 = 0.15, kPl2 = 0.30;  // Gfix/line_search.c:34-35
// scratch per site of each lattice, in complex numbers: the links'
// columns 0 and 1 (24), the fields in, in_old and two of sn (4 each)
constexpr long long kScratchPerSite = 40;
constexpr int kMaxSegments = 100;  // continuation segments; GLU does not bound them

// mL, mS: multipliers for division by the extents and strides (CDNA has
// no integer divide instruction; a division by a runtime value expands to
// a few dozen instructions, 64-bit ones to many more): for 2 <= d and
// x < 2^32 / d, x / d == umulhi(x, floor((2^32 - 1) / d) + 1).  Lattices
// of at most 16^4 sites keep every quotient here in that range.
struct BGeo {
  int L[4];
  long long S[4];
  long long V;
  unsigned mL[4], mS[4];  // mS[0] unused (S[0] = 1)
};

__device__ __forceinline__ unsigned bquot(unsigned x, unsigned m) { return __umulhi(x, m); }

__device__ __forceinline__ void bcoords(const BGeo &g, long long i, int x[4]) {
  unsigned r = (unsigned)i;
#pragma unroll
  for (int mu = 0; mu < 4; mu++) {
    const unsigned q = bquot(r, g.mL[mu]);
    x[mu] = (int)(r - q * (unsigned)g.L[mu]);
    r = q;
  }
}
__device__ __forceinline__ long long bfwd(const BGeo &g, long long i, const int x[4], int mu) {
  return x[mu] < g.L[mu] - 1 ? i + g.S[mu] : i - (long long)(g.L[mu] - 1) * g.S[mu];
}
__device__ __forceinline__ long long bbwd(const BGeo &g, long long i, const int x[4], int mu) {
  return x[mu] > 0 ? i - g.S[mu] : i + (long long)(g.L[mu] - 1) * g.S[mu];
}

// GLU's layout: link (i, mu) is 9 complex numbers, row-major
__device__ __forceinline__ const double2 *glu_link(const double2 *U, long long i, int mu) { return U + (i * 4 + mu) * 9; }

// The solve works on a copy of the links in scratch: columns 0 and 1 of
// link (i, mu) as 6 planes of V complex numbers, element k of direction mu
// at ((mu * 6 + k) V + i), so a wave's loads of one element are one
// contiguous run; column 2 is completed on every load, as the context
// path stores and completes its links
constexpr int kCol01[6] = {0, 1, 3, 4, 6, 7};
__device__ __forceinline__ su3<double> bload(const double2 *__restrict__ Uc, long long V, long long i, int mu) {
  su3<double> m;
#pragma unroll
  for (int k = 0; k < 6; k++) m.e[kCol01[k]] = ld<double>(Uc + (mu * 6 + k) * V + i);
  complete_col2(m);
  return m;
}
__device__ __forceinline__ void bstore(double2 *__restrict__ Uc, long long V, long long i, int mu, const su3<double> &m) {
#pragma unroll
  for (int k = 0; k < 6; k++) st<double>(Uc + (mu * 6 + k) * V + i, m.e[kCol01[k]]);
}

__device__ __forceinline__ su3<double> bgauge(const double2 *__restrict__ F, long long V, long long i, double al) {
  auto f = [&](long long k) { return ld<double>(F + k); };
  return gauge_matrix<double>(f(i), f(V + i), f(2 * V + i), f(3 * V + i), al);
}

// workgroup sum of NV values, fixed order, the result in every thread
template <int WG, int NV> __device__ void wg_sum(double (&v)[NV], double (*sh)[kMaxWgWaves]) {
  const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    const double s = wave_sum(v[k]);
    if (lane == 0) sh[k][w] = s;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double s = 0.0;
    for (int j = 0; j < WG / kWave; j++) s += sh[k][j];
    v[k] = s;
  }
  __syncthreads();
}

// Delta and its packing into F (Gfix/FACG.c:38-73); returns sum tr Delta^2
template <int WG> __device__ __forceinline__ double bderiv(const double2 *__restrict__ U, double2 *__restrict__ F, const BGeo &g,
                         double (*sh)[kMaxWgWaves]) {
  double v[1] = {0.0};
  for (long long i = threadIdx.x; i < g.V; i += WG) {
    int x[4];
    bcoords(g, i, x);
    DerivAcc<double> d;
    for (int mu = 0; mu < 4; mu++) d.add(bload(U, g.V, i, mu), bload(U, g.V, bbwd(g, i, x, mu), mu));
    v[0] += d.store(F, g.V, i);
  }
  wg_sum<WG, 1>(v, sh);
  return v[0];
}

// The DFT of N <= 16 numbers in registers (unnormalised; twiddles tw[k] =
// exp(-2 pi i k / NT) with NT a multiple of N, sign -1 forward): decimation
// in time by the smallest prime factor R, every index a compile-time
// constant.  The R-point sums of an odd R take the inputs q and R - q
// together, which share their cosines and, up to sign, their sines.  Direct
// sums, N products per number with two table reads each, took a third of an
// iteration wherever an extent is no power of two: 96 lattices of 6x10x12x9
// 0.81 -> 0.57 ms per iteration, 64 of 12^4 2.76 -> 1.76.
constexpr int small_factor(int n) {
  for (int r = 2; r < n; r++)
    if (n % r == 0) return r;
  return n;
}
template <int N, int NT, int ST>
__device__ __forceinline__ void reg_dft(const cx<double> (&in)[kMaxExtent], int first, cx<double> (&out)[N], int sign,
                                        const double2 *tw) {
  if constexpr (N == 1) {
    out[0] = in[first];
  } else {
    constexpr int R = small_factor(N), M = N / R;
    cx<double> sub[R][M];
#pragma unroll
    for (int r = 0; r < R; r++) reg_dft<M, NT, ST * R>(in, first + ST * r, sub[r], sign, tw);
    auto w = [&](int k) {  // exp(sign 2 pi i k / N)
      const double2 t = tw[k * (NT / N)];
      return mk<double>(t.x, sign < 0 ? t.y : -t.y);
    };
#pragma unroll
    for (int k = 0; k < M; k++) {
      cx<double> v[R];
      v[0] = sub[0][k];
#pragma unroll
      for (int r = 1; r < R; r++) v[r] = k > 0 ? cmul(sub[r][k], w(r * k)) : sub[r][k];
      if constexpr (R == 2) {
        out[k] = cadd(v[0], v[1]);
        out[k + M] = csub(v[0], v[1]);
      } else {
        constexpr int H = (R - 1) / 2;
        cx<double> a[H + 1], b[H + 1], y0 = v[0];
#pragma unroll
        for (int q = 1; q <= H; q++) {
          a[q] = cadd(v[q], v[R - q]);
          b[q] = csub(v[q], v[R - q]);
          y0 = cadd(y0, a[q]);
        }
        out[k] = y0;
#pragma unroll
        for (int m = 1; m <= H; m++) {
          cx<double> A = v[0], B = mk<double>(0.0, 0.0);
#pragma unroll
          for (int q = 1; q <= H; q++) {
            const cx<double> c = w((q * m) % R * M);  // exp(sign 2 pi i q m / R)
            A = mk<double>(A.re + c.re * a[q].re, A.im + c.re * a[q].im);
            B = mk<double>(B.re + c.im * b[q].re, B.im + c.im * b[q].im);
          }
          out[k + M * m] = mk<double>(A.re - B.im, A.im + B.re);  // A + i B
          out[k + M * (R - m)] = mk<double>(A.re + B.im, A.im - B.re);
        }
      }
    }
  }
}
template <int N>
__device__ __forceinline__ void fft_reg(cx<double> (&a)[kMaxExtent], int sign, const double2 *tw) {
  cx<double> y[N];
  reg_dft<N, N, 1>(a, 0, y, sign, tw);
#pragma unroll
  for (int k = 0; k < N; k++) a[k] = y[k];
}

// f(integral constant N) for the run-time extent N in 2..16
template <typename F> __device__ __forceinline__ void with_extent(int N, F f) {
  switch (N) {
    case 2: f(std::integral_constant<int, 2>{}); return;
    case 3: f(std::integral_constant<int, 3>{}); return;
    case 4: f(std::integral_constant<int, 4>{}); return;
    case 5: f(std::integral_constant<int, 5>{}); return;
    case 6: f(std::integral_constant<int, 6>{}); return;
    case 7: f(std::integral_constant<int, 7>{}); return;
    case 8: f(std::integral_constant<int, 8>{}); return;
    case 9: f(std::integral_constant<int, 9>{}); return;
    case 10: f(std::integral_constant<int, 10>{}); return;
    case 11: f(std::integral_constant<int, 11>{}); return;
    case 12: f(std::integral_constant<int, 12>{}); return;
    case 13: f(std::integral_constant<int, 13>{}); return;
    case 14: f(std::integral_constant<int, 14>{}); return;
    case 15: f(std::integral_constant<int, 15>{}); return;
    default: f(std::integral_constant<int, 16>{}); return;
  }
}

// one pencil of N numbers in registers: ld(j) reads input j, st(k, v)
// writes output k; every input is read before the first output is written,
// so a pencil may be transformed in place
template <typename Ld, typename St>
__device__ __forceinline__ void pencil_dft(int N, int sign, const double2 *tw, Ld ld, St st) {
  with_extent(N, [&](auto n) {
    constexpr int M = decltype(n)::value;
    cx<double> a[kMaxExtent];
#pragma unroll
    for (int j = 0; j < M; j++) a[j] = ld(j);
    fft_reg<M>(a, sign, tw);
#pragma unroll
    for (int k = 0; k < M; k++) st(k, a[k]);
  });
}

// The x, y and z transforms of the time slices of the fields (slabs of
// Lx Ly Lz sites, contiguous in F) run in LDS, as many slabs at a time as
// the stage holds: the slabs cross HBM once for the three axes instead of
// three times.  Each axis is transformed by pencil_dft on whole pencils
// in registers, in place.  Every x pencil is
// padded by one number in LDS (site (x, y, r) at x + (Lx + 1)(y + Ly r)),
// so that a wave's threads, one pencil each, read and write at a stride
// that spreads over the LDS banks.  The stage holds 9216 complex numbers
// (144 KiB) with 512 threads, whose workgroup holds a CU alone, and 4608
// with fewer, whose workgroups share a CU: a padded slab of 16^3 sites, the
// largest, fits either.
template <int WG> constexpr int stage_cx() { return WG >= 512 ? 9216 : 4608; }
static_assert((kMaxExtent + 1) * kMaxExtent * kMaxExtent <= stage_cx<128>());

// x, y, z transforms of the 4 T slabs of the 4 fields; the z sums are
// written straight back to F
template <int WG>
__device__ __forceinline__ void bdft_xyz(double2 *__restrict__ F, const BGeo &g, int sign,
                                         const double2 (*tw)[kMaxExtent], double2 *__restrict__ lds) {
  const int Lx = g.L[0], Ly = g.L[1], Lz = g.L[2], s3 = (int)g.S[3], sxy = (int)g.S[2];
  const int px = Lx + 1, per = stage_cx<WG>() / (px * Ly * Lz), nslab = 4 * g.L[3];
  for (int s0 = 0; s0 < nslab; s0 += per) {
    const int npts = min(per, nslab - s0) * s3;
    double2 *src = F + (long long)s0 * s3;  // slab (f, t) starts at (f T + t) s3
    for (int p = threadIdx.x; p < npts; p += WG) lds[p + (int)bquot((unsigned)p, g.mL[0])] = src[p];
    __syncthreads();
    // x: pencil q at q px, stride 1
    for (int q = threadIdx.x; q < npts / Lx; q += WG) {
      double2 *b = lds + q * px;
      pencil_dft(Lx, sign, tw[0], [&](int j) { return ld<double>(b + j); },
                 [&](int k, cx<double> v) { st<double>(b + k, v); });
    }
    __syncthreads();
    // y: pencil q = x + Lx r (r = z + Lz s, s the slab of the round) at
    // x + px Ly r, stride px
    for (int q = threadIdx.x; q < npts / Ly; q += WG) {
      const int r = (int)bquot((unsigned)q, g.mL[0]);
      double2 *b = lds + (q - r * Lx) + px * Ly * r;
      pencil_dft(Ly, sign, tw[1], [&](int j) { return ld<double>(b + j * px); },
                 [&](int k, cx<double> v) { st<double>(b + k * px, v); });
    }
    __syncthreads();
    // z: pencil q = x + Lx y + Lx Ly s at x + px (y + Ly Lz s), stride
    // px Ly, into F at s s3 + x + Lx y, stride Lx Ly
    for (int q = threadIdx.x; q < npts / Lz; q += WG) {
      const int sl = (int)bquot((unsigned)q, g.mS[2]), xy = q - sl * sxy;
      const int y = (int)bquot((unsigned)xy, g.mL[0]), x = xy - y * Lx;
      const double2 *b = lds + x + px * (y + Ly * Lz * sl);
      double2 *o = src + (long long)sl * s3 + xy;
      pencil_dft(Lz, sign, tw[2], [&](int j) { return ld<double>(b + j * px * Ly); },
                 [&](int k, cx<double> v) { st<double>(o + (long long)k * sxy, v); });
    }
    __syncthreads();  // the stage is free for the next round, F complete
  }
}

// along t, on pencils in registers: forward, x MAX / p^2, backward -- the
// middle of the Fourier acceleration in one pass
template <int WG>
__device__ __forceinline__ void bdft_t_scale(double2 *__restrict__ F, const BGeo &g, const double2 (*tw)[kMaxExtent]) {
  const long long S = g.S[3], V = g.V;
  const double mx = 4.0 * 4 / (double)V;
  with_extent(g.L[3], [&](auto n) {
    constexpr int N = decltype(n)::value;
    for (unsigned p = threadIdx.x; p < 4 * S; p += WG) {
      const unsigned f = bquot(p, g.mS[3]), q = p - f * (unsigned)S;
      const long long base = (long long)f * V + q;
      int x[4];
      bcoords(g, q, x);
      const double kxyz = tw[0][x[0]].x + tw[1][x[1]].x + tw[2][x[2]].x;
      cx<double> a[kMaxExtent];
#pragma unroll
      for (int j = 0; j < N; j++) a[j] = ld<double>(F + base + j * S);
      fft_reg<N>(a, -1, tw[3]);
#pragma unroll
      for (int k = 0; k < N; k++) {
        const double kc = kxyz + tw[3][k].x;  // sum of cos(2 pi n_mu / L_mu), mu in order
        const double fac = mx / ((kc == 4.0) ? 1.0 : 2.0 * (4.0 - kc));
        a[k] = mk<double>(a[k].re * fac, a[k].im * fac);
      }
      fft_reg<N>(a, +1, tw[3]);
#pragma unroll
      for (int k = 0; k < N; k++) st<double>(F + base + k * S, a[k]);
    }
  });
  __syncthreads();
}

// forward transform, x MAX / p^2 (p^2(0) := 1, MAX = 4 ND / V), backward
// transform: Gfix/FACG.c:77-95 with Gfix/Landau.c:275-284
template <int WG>
__device__ __forceinline__ void bfourier_accelerate(double2 *__restrict__ F, const BGeo &g,
                                                    const double2 (*tw)[kMaxExtent], double2 *__restrict__ lds) {
  // (one copy of each transform's code for both directions)
#pragma unroll 1
  for (int sign = -1; sign <= 1; sign += 2) {
    bdft_xyz<WG>(F, g, sign, tw, lds);
    if (sign < 0) bdft_t_scale<WG>(F, g, tw);
  }
}

// <in, in> and <in, in - old> in GLU's trace metric (Gfix/FACG.c:99-178)
template <int WG> __device__ __forceinline__ void bpr_sums(const double2 *__restrict__ F, const double2 *__restrict__ O, const BGeo &g, double out[2],
                         double (*sh)[kMaxWgWaves]) {
  double v[2] = {0.0, 0.0};
  const long long V = g.V;
  for (long long i = threadIdx.x; i < V; i += WG) {
    const cx<double> z0 = ld<double>(F + i), o0 = ld<double>(O + i);
    const double zr = z0.re, zi = z0.im, tr = zr - o0.re, ti = zi - o0.im;
    double s1 = 2.0 * (zr * zr + zi * zi + zr * zi);
    double s2 = 2.0 * (zr * tr + zi * ti) + zr * ti + zi * tr;
    for (int f = 1; f < 4; f++) {
      const cx<double> z = ld<double>(F + f * V + i), o = ld<double>(O + f * V + i);
      s1 += 2.0 * (z.re * z.re + z.im * z.im);
      s2 += 2.0 * (z.re * (z.re - o.re) + z.im * (z.im - o.im));
    }
    v[0] += s1;
    v[1] += s2;
  }
  wg_sum<WG, 2>(v, sh);
  out[0] = v[0];
  out[1] = v[1];
}

// functional probes at 0, PL1, PL2 along the packed direction D
// (Gfix/line_search.c:274-341): each link is loaded once for the three
// probes.  The direction loop stays rolled: unrolled, the compiler hoists
// the loads of all four links and their neighbours' gauge matrices and
// spills.
template <int WG> __device__ __forceinline__ void bprobes(const double2 *__restrict__ U, const double2 *__restrict__ D, const BGeo &g, double out[3],
                        double (*sh)[kMaxWgWaves]) {
  double v[3] = {0.0, 0.0, 0.0};
  const long long V = g.V;
  for (long long i = threadIdx.x; i < V; i += WG) {
    int x[4];
    bcoords(g, i, x);
    // the site's gauge matrices are rebuilt from its four field values in
    // every direction rather than held across the loop: fewer registers
    // live (34 -> 24 spilled at 512 threads), the same values
    const cx<double> f0 = ld<double>(D + i), f1 = ld<double>(D + V + i), f2 = ld<double>(D + 2 * V + i),
                     f3 = ld<double>(D + 3 * V + i);
    double acc1 = 0.0, acc2 = 0.0;
#pragma unroll 1
    for (int mu = 0; mu < 4; mu++) {
      const su3<double> u = bload(U, V, i, mu);
      v[0] += u.e[0].re + u.e[4].re + u.e[8].re;
      cx<double> au1[6], au2[6];
      ab_rows01<double>(gauge_matrix<double>(f0, f1, f2, f3, kPl1), u, au1);
      ab_rows01<double>(gauge_matrix<double>(f0, f1, f2, f3, kPl2), u, au2);
      const long long f = bfwd(g, i, x, mu);
      acc1 += retrace_rows01_dag<double>(au1, bgauge(D, V, f, kPl1));
      acc2 += retrace_rows01_dag<double>(au2, bgauge(D, V, f, kPl2));
    }
    v[1] += acc1;
    v[2] += acc2;
  }
  wg_sum<WG, 3>(v, sh);
  for (int k = 0; k < 3; k++) out[k] = v[k];
}

// bprobes along the new direction sn + beta... : D = I + beta S formed
// where it is read (at each site and its forward neighbours, with the
// arithmetic of the CG update), and each site's own value written to N,
// the next direction -- the CG update folded into the probes.  S is only
// read here, so no thread waits for another's update.
template <int WG>
__device__ __forceinline__ void bprobes_cg(const double2 *__restrict__ U, const double2 *__restrict__ I,
                                           const double2 *__restrict__ S, double2 *__restrict__ N, double beta,
                                           const BGeo &g, double out[3], double (*sh)[kMaxWgWaves]) {
  double v[3] = {0.0, 0.0, 0.0};
  const long long V = g.V;
  auto dir = [&](long long k) {
    const double2 a = I[k], s = S[k];
    return make_double2(a.x + beta * s.x, a.y + beta * s.y);
  };
  for (long long i = threadIdx.x; i < V; i += WG) {
    int x[4];
    bcoords(g, i, x);
    const double2 d0 = dir(i), d1 = dir(V + i), d2 = dir(2 * V + i), d3 = dir(3 * V + i);
    N[i] = d0;
    N[V + i] = d1;
    N[2 * V + i] = d2;
    N[3 * V + i] = d3;
    const cx<double> f0 = mk<double>(d0.x, d0.y), f1 = mk<double>(d1.x, d1.y), f2 = mk<double>(d2.x, d2.y),
                     f3 = mk<double>(d3.x, d3.y);
    double acc1 = 0.0, acc2 = 0.0;
#pragma unroll 1
    for (int mu = 0; mu < 4; mu++) {
      const su3<double> u = bload(U, V, i, mu);
      v[0] += u.e[0].re + u.e[4].re + u.e[8].re;
      cx<double> au1[6], au2[6];
      ab_rows01<double>(gauge_matrix<double>(f0, f1, f2, f3, kPl1), u, au1);
      ab_rows01<double>(gauge_matrix<double>(f0, f1, f2, f3, kPl2), u, au2);
      const long long f = bfwd(g, i, x, mu);
      const double2 n0 = dir(f), n1 = dir(V + f), n2 = dir(2 * V + f), n3 = dir(3 * V + f);
      const cx<double> g0 = mk<double>(n0.x, n0.y), g1 = mk<double>(n1.x, n1.y), g2 = mk<double>(n2.x, n2.y),
                       g3 = mk<double>(n3.x, n3.y);
      acc1 += retrace_rows01_dag<double>(au1, gauge_matrix<double>(g0, g1, g2, g3, kPl1));
      acc2 += retrace_rows01_dag<double>(au2, gauge_matrix<double>(g0, g1, g2, g3, kPl2));
    }
    v[1] += acc1;
    v[2] += acc2;
  }
  wg_sum<WG, 3>(v, sh);
  for (int k = 0; k < 3; k++) out[k] = v[k];
}

// U_mu(x) <- g(x) U_mu(x) g(x + mu)^dag with g from D at step alpha, in
// place: g depends on D only, and each link is written by its own site
// (Gfix/line_search.c:60-97)
template <int WG> __device__ __forceinline__ void begauge(double2 *__restrict__ U, const double2 *__restrict__ D, const BGeo &g, double alpha) {
  for (long long i = threadIdx.x; i < g.V; i += WG) {
    int x[4];
    bcoords(g, i, x);
    const su3<double> A = bgauge(D, g.V, i, alpha);
#pragma unroll 1
    for (int mu = 0; mu < 4; mu++)
      bstore(U, g.V, i, mu, gtransform<double>(A, bload(U, g.V, i, mu), bgauge(D, g.V, bfwd(g, i, x, mu), alpha)));
  }
  __syncthreads();
}

__device__ __forceinline__ void swap_fields(double2 *&a, double2 *&b) {
  double2 *t = a;
  a = b;
  b = t;
}

// begauge and bderiv in one pass: U' = g U g^dag in place, the packed Delta
// of U' into F, the sum of tr Delta^2 returned.  The lattice is walked in
// chunks of one site per thread, in the order of the sites.  A backward
// neighbour's U' comes from LDS if the neighbour is in the chunk (along t,
// where few are, from memory), from memory if its chunk is done, and is
// otherwise (at the lower edges) formed here from the old link, which nobody
// replaces before the barrier at the chunk's end.
// The old links are read once and the new ones written once, where a second
// pass for the derivative read them again and moved its partial sums twice:
// 2500 -> 2000 bytes per site and iteration.  Iteration of 512 lattices of
// 8^4 0.90 -> 0.82 ms, of 96 of 6x10x12x9 0.571 -> 0.560, of 256 of 10^4 1.25
// -> 1.13, of 64 of 16^4 5.58 -> 5.16.  A barrier per direction, which needs
// a third of the LDS, drains the loads four times as often: 0.83 and 0.577
// for the first two.
template <int WG>
__device__ __forceinline__ double begauge_deriv(double2 *__restrict__ U, const double2 *__restrict__ D,
                                                double2 *__restrict__ F, const BGeo &g, double alpha,
                                                double (*sh)[kMaxWgWaves], double2 *__restrict__ buf) {
  static_assert(3 * 6 * WG <= stage_cx<WG>());
  double v[1] = {0.0};
  const long long V = g.V;
  const int tid = threadIdx.x;
  for (long long base = 0; base < V; base += WG) {
    const long long i = base + tid;
    const bool on = i < V;
    int x[4] = {0, 0, 0, 0};
    su3<double> A;
    DerivAcc<double> d;
    if (on) {
      bcoords(g, i, x);
      A = bgauge(D, V, i, alpha);
#pragma unroll 1
      for (int mu = 0; mu < 4; mu++) {
        const su3<double> m = gtransform<double>(A, bload(U, V, i, mu), bgauge(D, V, bfwd(g, i, x, mu), alpha));
        bstore(U, V, i, mu, m);
        d.add_own(m);
        if (mu < 3) {
#pragma unroll
          for (int k = 0; k < 6; k++) st<double>(buf + (mu * 6 + k) * WG + tid, m.e[kCol01[k]]);
        }
      }
    }
    __syncthreads();
    if (on) {
#pragma unroll 1
      for (int mu = 0; mu < 4; mu++) {
        const long long xb = bbwd(g, i, x, mu), rel = xb - base;
        su3<double> m;
        if (rel >= WG) {
          m = gtransform<double>(bgauge(D, V, xb, alpha), bload(U, V, xb, mu), A);
        } else if (rel >= 0 && mu < 3) {
#pragma unroll
          for (int k = 0; k < 6; k++) m.e[kCol01[k]] = ld<double>(buf + (mu * 6 + k) * WG + rel);
          complete_col2(m);
        } else {
          m = bload(U, V, xb, mu);
        }
        d.add_bwd(m);
      }
      v[0] += d.store(F, V, i);
    }
    __syncthreads();  // the next chunk's old links and buf may be replaced
  }
  wg_sum<WG, 1>(v, sh);
  return v[0];
}

struct BTrace {
  double *rows;  // 3 per row
  long long cap, n;
  __device__ void rec(double th, double al, double be) {
    if (rows && n < cap && threadIdx.x == 0) {
      rows[3 * n] = th;
      rows[3 * n + 1] = al;
      rows[3 * n + 2] = be;
    }
    if (n < cap) n++;
  }
};

// FACG of lattice blockIdx.x: links U (GLU layout, V sites), scratch
// fields in, in_old and two of sn (4 V complex each).  Writes its iteration count (GLU's
// return value) and final theta.
template <int WG>
__global__ __launch_bounds__(WG, WG >= 256 ? 2 : 1) void k_facg_batch(double2 *const *__restrict__ lat, double2 *__restrict__ scratch,
                                                          BGeo g, int nlat, double gf, double acc,
                                                          long long max_iters, long long *iters_out,
                                                          double *theta_out, double *trace, long long trace_cap,
                                                          int keep_failed) {
  __shared__ double sh[3][kMaxWgWaves];
  __shared__ double2 tw[4][kMaxExtent];
  __shared__ double2 stage[stage_cx<WG>()];
  const int b = blockIdx.x;
  if (b >= nlat) return;
  const long long V = g.V;
  double2 *glu = lat[b];
  double2 *U = scratch + (long long)b * V * kScratchPerSite;  // the links, columns 0 and 1
  double2 *in = U + 24 * V, *sn = in + 4 * V, *old = in + 8 * V, *sn2 = in + 12 * V;
  for (long long j = threadIdx.x; j < 4 * V; j += WG) {
    const long long i = j >> 2;
    const int mu = (int)(j & 3);
    const double2 *p = glu_link(glu, i, mu);
#pragma unroll
    for (int k = 0; k < 6; k++) U[(mu * 6 + k) * V + i] = p[kCol01[k]];
  }
  for (int t = threadIdx.x; t < 4 * kMaxExtent; t += WG) {
    const int mu = t / kMaxExtent, k = t % kMaxExtent;
    const double a = 6.283185307179586 * (double)k / (double)g.L[mu];
    tw[mu][k] = make_double2(cos(a), -sin(a));
  }
  __syncthreads();
  BTrace tr{trace ? trace + (long long)b * trace_cap * 3 : nullptr, trace_cap, 0};
  const double norm = 1.0 / (3.0 * (double)V);  // GFNORM_LANDAU
  // theta_test_lin (FACG.c:349): 2 x the FA theta of the input links
  double theta = 2.0 * bderiv<WG>(U, in, g, sh) * norm;
  long long iters = 0;
  if (theta < acc) {
    if (threadIdx.x == 0) {
      iters_out[b] = 0;
      theta_out[b] = theta;
    }
    return;
  }
  // GLU's red[] slots carried into a continuation's SD start (FACG.c:249-265)
  double stale_theta = 0.0, stale_insum = 0.0, stale_probe[3] = {0.0, 0.0, 0.0};
  for (int seg = 0; seg < kMaxSegments; seg++) {
    // steepest-descent start
    theta = bderiv<WG>(U, in, g, sh) * norm + stale_theta;
    bfourier_accelerate<WG>(in, g, tw, stage);
    double pr[3];
    bprobes<WG>(U, in, g, pr, sh);
    double val[3];
    for (int k = 0; k < 3; k++) val[k] = -(pr[k] + stale_probe[k]);
    const double als[3] = {0.0, kPl1, kPl2};
    double alpha = approx_minimum(als, val);
    begauge<WG>(U, in, g, alpha);
    tr.rec(theta, alpha, 0.0);
    for (long long j = threadIdx.x; j < 4 * V; j += WG) sn[j] = in[j];
    // in_old <- in: the two buffers trade roles instead of copying, and
    // the next derivative is written into the other
    swap_fields(in, old);
    double s2[2];
    bpr_sums<WG>(old, old, g, s2, sh);  // <in, in> (sum_DER3)
    double inold = s2[0] + stale_insum;
    long long loc = 0;
    double insum = 0.0, probe[3] = {0.0, 0.0, 0.0};
    int did_ls = 0;
    double next = bderiv<WG>(U, in, g, sh) * norm;
    for (;;) {
      theta = next;
      bfourier_accelerate<WG>(in, g, tw, stage);
      bpr_sums<WG>(in, old, g, s2, sh);
      insum = s2[0];
      double beta = s2[1] / inold;
      if (beta < 0.0) beta = 0.0;
      if (theta < kCgTolB) beta = insum / inold;  // Fletcher-Reeves below CG_TOL
      inold = insum;
      if (theta > kCgTolB) {
        // sn <- in + beta sn inside the probes, into the other buffer
        bprobes_cg<WG>(U, in, sn, sn2, beta, g, probe, sh);
        swap_fields(sn, sn2);
        for (int k = 0; k < 3; k++) val[k] = -probe[k];
        alpha = approx_minimum(als, val);
        did_ls = 1;
      } else {
        for (long long j = threadIdx.x; j < 4 * V; j += WG) {
          const double2 a = in[j], s = sn[j];
          sn[j] = make_double2(a.x + beta * s.x, a.y + beta * s.y);
        }
        __syncthreads();
        alpha = gf;
        did_ls = 0;
      }
      swap_fields(in, old);  // in_old <- in
      next = begauge_deriv<WG>(U, sn, in, g, alpha, sh, stage) * norm;  // into `in`, which is free
      tr.rec(theta, alpha, beta);
      loc++;
      if (!(theta > acc && loc < max_iters)) break;
    }
    stale_theta = theta;
    stale_insum = insum;
    for (int k = 0; k < 3; k++) stale_probe[k] = did_ls ? probe[k] : 0.0;
    iters = loc;
    if (loc >= max_iters) {
      if (theta < 1e3 * acc) continue;  // continuation (FACG.c:372-378)
      iters = 123456789;
    }
    break;
  }
  if (iters == max_iters && !(theta < acc)) iters = 123456789;  // the segment bound ran out
  __syncthreads();
  // the fixed links back in GLU's layout, column 2 completed (a failed
  // lattice keeps its input when the caller restarts from it)
  for (long long j = threadIdx.x; j < 4 * V && !(keep_failed && iters == 123456789); j += WG) {
    const long long i = j >> 2;
    const int mu = (int)(j & 3);
    const su3<double> m = bload(U, V, i, mu);
    double2 *p = glu + (i * 4 + mu) * 9;
#pragma unroll
    for (int k = 0; k < 9; k++) st<double>(p + k, m.e[k]);
  }
  if (threadIdx.x == 0) {
    iters_out[b] = iters;
    theta_out[b] = theta;
  }
}

}  // namespace

// the shape and sizes one launch takes, checked before any device work
static int batch_geometry(const size_t dims[4], size_t nlat, size_t max_iters, BGeo *g) {
  if (!dims) return gfix_fail(-1, "glu_gfix_facg_batch: null argument");
  if (nlat > 65535) return gfix_fail(-1, "glu_gfix_facg_batch: %zu lattices exceed the 65535 of one launch", nlat);
  if (max_iters == 0) return gfix_fail(-1, "max_iters must be positive");
  long long V = 1;
  for (int mu = 0; mu < 4; mu++) {
    if (dims[mu] < 2 || dims[mu] > (size_t)kMaxExtent)
      return gfix_fail(-1, "glu_gfix_facg_batch: extent %zu outside 2..%d", dims[mu], kMaxExtent);
    g->L[mu] = (int)dims[mu];
    g->S[mu] = V;
    V *= (long long)dims[mu];
  }
  g->V = V;
  // division multipliers (extents are at least 2, strides past the first too)
  auto mul = [](long long d) { return (unsigned)(0xFFFFFFFFull / (unsigned long long)d) + 1u; };
  for (int mu = 0; mu < 4; mu++) {
    g->mL[mu] = mul(g->L[mu]);
    g->mS[mu] = mu ? mul(g->S[mu]) : 0u;
  }
  return 0;
}

// FACG of nlat lattices of one shape whose links (GLU's layout, device
// memory) are at lat[k], a host array of device pointers, on a stream of
// its own; with keep_failed, a lattice that returns 123456789 keeps its
// input links
int facg_batch_run(const size_t dims[4], size_t nlat, double *const *lat, double gf_tune, double accuracy,
                   size_t max_iters, size_t *iters, double *theta, double *trace, size_t trace_cap,
                   int keep_failed) {
  if (!lat || !iters || !theta) return gfix_fail(-1, "glu_gfix_facg_batch: null argument");
  BGeo g{};
  if (int rc = batch_geometry(dims, nlat, max_iters, &g)) return rc;
  if (nlat == 0) return 0;
  const long long V = g.V;
  for (size_t k = 0; k < nlat; k++)
    if (!lat[k]) return gfix_fail(-1, "glu_gfix_facg_batch: null links of lattice %zu", k);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return gfix_fail(-3, "no HIP device: the gauge-fixing library has no CPU path");
  double2 *scratch = nullptr, **d_lat = nullptr;
  long long *d_it = nullptr;
  double *d_th = nullptr, *d_tr = nullptr;
  hipStream_t st = nullptr;
  int rc = 0;
  const size_t tcap = trace ? trace_cap : 0;
  if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) {
    st = nullptr;
    rc = gfix_fail(-2, "glu_gfix_facg_batch: stream creation failed");
  } else if (hipMalloc(&scratch, nlat * (size_t)V * kScratchPerSite * sizeof(double2)) != hipSuccess ||
      hipMalloc(&d_lat, nlat * sizeof(double2 *)) != hipSuccess ||
      hipMalloc(&d_it, nlat * sizeof(long long)) != hipSuccess || hipMalloc(&d_th, nlat * sizeof(double)) != hipSuccess ||
      (tcap && hipMalloc(&d_tr, nlat * tcap * 3 * sizeof(double)) != hipSuccess)) {
    rc = gfix_fail(-2, "glu_gfix_facg_batch: scratch allocation failed");
  } else if (hipMemcpyAsync(d_lat, lat, nlat * sizeof(double2 *), hipMemcpyHostToDevice, st) != hipSuccess) {
    rc = gfix_fail(-2, "glu_gfix_facg_batch: pointer upload failed");
  } else {
    // threads per lattice: 512 unless GLU_GFIX_BATCH_WG picks 128 or 256
    // (512 8^4 lattices: 9350, 8940 and 7080 configs/s at 512, 256 and 128
    // before the update took in the derivative; 10180 at 512 since)
    int wg = 512;
    if (const char *e = getenv("GLU_GFIX_BATCH_WG")) wg = atoi(e);
    auto launch = [&](auto kernel, int threads) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)nlat), dim3(threads), 0, st, (double2 *const *)d_lat, scratch, g,
                         (int)nlat, gf_tune, accuracy, (long long)max_iters, d_it, d_th, d_tr, (long long)tcap,
                         keep_failed);
    };
    if (wg == 128)
      launch(k_facg_batch<128>, 128);
    else if (wg == 256)
      launch(k_facg_batch<256>, 256);
    else
      launch(k_facg_batch<512>, 512);
    std::vector<long long> it(nlat);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(it.data(), d_it, nlat * sizeof(long long), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipMemcpyAsync(theta, d_th, nlat * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
        (tcap && hipMemcpyAsync(trace, d_tr, nlat * tcap * 3 * sizeof(double), hipMemcpyDeviceToHost, st) !=
                     hipSuccess) ||
        hipStreamSynchronize(st) != hipSuccess) {
      rc = gfix_fail(-2, "glu_gfix_facg_batch failed: %s", hipGetErrorString(hipGetLastError()));
    } else {
      for (size_t k = 0; k < nlat; k++) iters[k] = (size_t)it[k];
    }
  }
  // teardown: nothing to undo if a free fails
  if (st) (void)hipStreamSynchronize(st);
  if (scratch) (void)hipFree(scratch);
  if (d_lat) (void)hipFree(d_lat);
  if (d_it) (void)hipFree(d_it);
  if (d_th) (void)hipFree(d_th);
  if (d_tr) (void)hipFree(d_tr);
  if (st) (void)hipStreamDestroy(st);
  return rc;
}

extern "C" int glu_gfix_facg_batch(const size_t dims[4], size_t nlat, double *links_dev, double gf_tune,
                                   double accuracy, size_t max_iters, size_t *iters, double *theta, double *trace,
                                   size_t trace_cap) {
  if (!links_dev || !iters || !theta) return gfix_fail(-1, "glu_gfix_facg_batch: null argument");
  BGeo g{};
  if (int rc = batch_geometry(dims, nlat, max_iters, &g)) return rc;
  if (nlat == 0) return 0;
  const size_t V = (size_t)g.V;
  std::vector<double *> lat(nlat);
  for (size_t k = 0; k < nlat; k++) lat[k] = links_dev + k * V * 72;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return gfix_fail(-3, "no HIP device: the gauge-fixing library has no CPU path");
  // the links may still be in flight on any of the caller's streams
  if (hipDeviceSynchronize() != hipSuccess)
    return gfix_fail(-2, "glu_gfix_facg_batch: device synchronisation failed: %s", hipGetErrorString(hipGetLastError()));
  return facg_batch_run(dims, nlat, lat.data(), gf_tune, accuracy, max_iters, iters, theta, trace, trace_cap, 0);
}
