// fft_kernels.hip -- LDS-staged mixed-radix (2, 3, 4, 5, 7, 8) complex FFT
// along one or two lattice axes per pass, batched over every pencil of the 4
// packed fields, with the p^2 preconditioner fused into the last forward
// axis.
//
// This replaces the FFTW transforms of Gfix/FACG.c:77-95 (Landau, 4D) and
// Gfix/CFACG.c:70-89 (Coulomb, 3D per time slice): forward transform,
// multiply by psq = MAX / p^2 (Gfix/Landau.c:278-284), backward transform,
// both unnormalised.
//
// A workgroup stages pencils in LDS, runs a Stockham auto-sort sequence of
// radix stages on them, and writes them back.  Pencils along x are contiguous rows; along y, z, t consecutive
// pencils are consecutive addresses, so loads and stores are coalesced in
// both cases.  Twiddles come from a per-axis table computed on the host.
#include "gfix_kernels.h"

namespace gfix {

template <typename T, int R> __device__ __forceinline__ void dft_small(cx<T> (&v)[R], int sign) {
  if constexpr (R == 2) {
    const cx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const cx<T> a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
    const cx<T> c = cadd(v[1], v[3]), d = csub(v[1], v[3]);
    // forward: y1 = b - i d, y3 = b + i d ; backward swaps
    const cx<T> id = sign < 0 ? mk<T>(d.im, -d.re) : mk<T>(-d.im, d.re);
    v[0] = cadd(a, c);
    v[2] = csub(a, c);
    v[1] = cadd(b, id);
    v[3] = csub(b, id);
  } else if constexpr (R == 8) {
    // two 4-point DFTs of the even and odd inputs, combined with the
    // eighth roots of unity e^{sign i pi k / 4}
    cx<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft_small<T, 4>(e, sign);
    dft_small<T, 4>(o, sign);
    const T h = T(0.70710678118654752440);
    const T sg = sign < 0 ? T(-1) : T(1);
    cx<T> w[4];
    w[0] = o[0];
    w[1] = mk<T>(h * (o[1].re - sg * o[1].im), h * (o[1].im + sg * o[1].re));  // * h (1 + i sg)
    w[2] = mk<T>(-sg * o[2].im, sg * o[2].re);                                 // * i sg
    w[3] = mk<T>(-h * (o[3].re + sg * o[3].im), h * (sg * o[3].re - o[3].im)); // * h (-1 + i sg)
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = cadd(e[k], w[k]);
      v[k + 4] = csub(e[k], w[k]);
    }
  } else if constexpr (R == 5 || R == 7) {
    // the odd primes GLU's extents may contain
    constexpr double c5[5] = {1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475,
                              0.30901699437494745};
    constexpr double s5[5] = {0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731,
                              -0.9510565162951535};
    constexpr double c7[7] = {1.0, 0.6234898018587336, -0.22252093395631434, -0.9009688679024191,
                              -0.9009688679024191, -0.22252093395631434, 0.6234898018587336};
    constexpr double s7[7] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.43388373911755823,
                              -0.43388373911755823, -0.9749279121818236, -0.7818314824680298};
    if constexpr (sizeof(T) == 8) {
      // the inputs q and R - q share their cosines and, up to sign, their
      // sines: half the products and registers of the plain sums, which
      // FP32 keeps (its rounding decides the FP32 phase's trajectory)
      constexpr int H = (R - 1) / 2;
      cx<T> a[H + 1], b[H + 1], y0 = v[0];
#pragma unroll
      for (int q = 1; q <= H; q++) {
        a[q] = cadd(v[q], v[R - q]);
        b[q] = cscale(csub(v[q], v[R - q]), (T)sign);
        y0 = cadd(y0, a[q]);
      }
#pragma unroll
      for (int m = 1; m <= H; m++) {
        cx<T> A = v[0], B = mk<T>(T(0), T(0));
#pragma unroll
        for (int q = 1; q <= H; q++) {
          const int k = (q * m) % R;
          A = cadd(A, cscale(a[q], (T)(R == 5 ? c5[k] : c7[k])));
          B = cadd(B, cscale(b[q], (T)(R == 5 ? s5[k] : s7[k])));
        }
        v[m] = mk<T>(A.re - B.im, A.im + B.re);  // A + i B
        v[R - m] = mk<T>(A.re + B.im, A.im - B.re);
      }
      v[0] = y0;
      return;
    }
    cx<T> y[R];
#pragma unroll
    for (int m = 0; m < R; m++) {
      cx<T> acc = v[0];
#pragma unroll
      for (int q = 1; q < R; q++) {
        const int k = (q * m) % R;
        const T c = (T)(R == 5 ? c5[k] : c7[k]), sn = (T)(sign * (R == 5 ? s5[k] : s7[k]));
        acc = cadd(acc, cmul(v[q], mk<T>(c, sn)));
      }
      y[m] = acc;
    }
#pragma unroll
    for (int m = 0; m < R; m++) v[m] = y[m];
  } else if constexpr (R == 3) {
    const T c1 = T(-0.5), s1 = T(sign) * T(0.86602540378443864676);
    const cx<T> a = v[0], b = v[1], c = v[2];
    const cx<T> sbc = cadd(b, c), dbc = csub(b, c);
    v[0] = cadd(a, sbc);
    const cx<T> m = mk<T>(a.re + c1 * sbc.re, a.im + c1 * sbc.im);
    // i s1 (b - c)
    const cx<T> r = mk<T>(-s1 * dbc.im, s1 * dbc.re);
    v[1] = cadd(m, r);
    v[2] = csub(m, r);
  }
}

constexpr int kFftThreads = 256;

// ---------------------------------------------------------------------------
// Any extents: one or two axes of a tile per pass, plans at run time
// ---------------------------------------------------------------------------
// The pass for extents without a compile-time kernel below: it transforms
// the two axes of an x-y plane, the z and t axes of a column (forward z, t,
// x p^2, backward t, z), or one axis, so that a lattice of any extents goes
// through three passes over the fields like the common ones.  The tile sits
// in LDS twice and every stage reads one copy and writes the other: one
// barrier a stage, no values held across it, so a stage may have any number
// of butterflies per thread.  Indices come from multipliers (the GPU has no
// integer divide), and a stage's twiddle index q k N / (Ns R) is below N by
// construction.  The arithmetic of a pencil is that of the compile-time
// kernels: the same radix plan, twiddles and p^2 order.
// On 20x28x10x36 in FP64 a Fourier acceleration took seven single-axis
// passes of 30 us, bound by integer division; the three passes here take
// 21 us each, bound by the issue of index and LDS instructions (FP32 takes
// 17; a copy at 5.2 TB/s would take 5).
struct AnyStage {
  int R, Ns, nbf, tstep;
  unsigned mNs;
};
struct AnyAxis {
  int N, nst;
  AnyStage st[8];
  const double2 *tw;
};
// pencils of one axis in the tile: pencil j at (j % PJ) SJ + (j / PJ) PS,
// its points SN apart
struct AnyPencils {
  int P, SN, SJ, PJ, PS;
  unsigned mP, mPJ;
};
// what a tile is: m x-y planes (two axes), m neighbouring x-y sites' z-t
// planes (two axes), m contiguous rows or m neighbouring pencils (one axis).
// A template argument: a tile layout chosen at run time inside the kernel
// left the compiler with a load address that one of the layouts never set.
enum { ANY_PLANE = 0, ANY_COLUMN = 1, ANY_ROW = 2, ANY_AXIS = 3 };
constexpr int any_axes(int lay) { return lay == ANY_PLANE || lay == ANY_COLUMN ? 2 : 1; }
struct AnyPass {
  AnyAxis ax[2];
  AnyPencils pe[2];
  int mode;
  int m;            // planes, x-y sites or pencils per tile
  int ld;           // LDS row length
  int elems, pool;  // tile elements, LDS elements of one copy
  unsigned mRow;    // division of an element index by the memory row
  unsigned mZ;      // by the column's NZ
  long long S, St;  // memory strides of the axes
};

inline unsigned any_mul(unsigned d) { return 0x80000000u / d + 1u; }
// n / d for n d < 2^31, m = any_mul(d), d >= 1
__device__ __forceinline__ unsigned any_div(unsigned n, unsigned m) { return __umulhi(2u * n, m); }

template <typename T, int R>
__device__ __forceinline__ void any_stage(const vec2<T> *src, vec2<T> *dst, const AnyPencils &pe,
                                          const AnyStage &sg, const vec2<T> *tw, const int sign) {
  const int total = sg.nbf * pe.P, Ns = sg.Ns;
  for (int w = threadIdx.x; w < total; w += blockDim.x) {
    const int b = (int)any_div((unsigned)w, pe.mP), j = w - b * pe.P;
    const int g = pe.PJ == pe.P ? 0 : (int)any_div((unsigned)j, pe.mPJ);
    const int jo = (j - g * pe.PJ) * pe.SJ + g * pe.PS;
    const int h = (int)any_div((unsigned)b, sg.mNs), k = b - h * Ns;
    cx<T> v[R];
#pragma unroll
    for (int q = 0; q < R; q++) v[q] = ld<T>(src + (b + q * sg.nbf) * pe.SN + jo);
    if (Ns > 1) {
      const int kt = k * sg.tstep;
#pragma unroll
      for (int q = 1; q < R; q++) {
        cx<T> t = ld<T>(tw + q * kt);
        if (sign > 0) t.im = -t.im;
        v[q] = cmul(v[q], t);
      }
    }
    dft_small<T, R>(v, sign);
    const int out = h * Ns * R + k;
#pragma unroll
    for (int q = 0; q < R; q++) st<T>(dst + (out + q * Ns) * pe.SN + jo, v[q]);
  }
  __syncthreads();
}

// element e of a tile: its offset in memory and in LDS
template <int LAY> __device__ __forceinline__ void any_place(const AnyPass &p, int e, long long &mem, int &lds) {
  const int r = (int)any_div((unsigned)e, p.mRow);
  if constexpr (LAY == ANY_COLUMN) {  // (j, z, t): e = j + m (z + NZ t)
    const int t = (int)any_div((unsigned)r, p.mZ), NZ = p.ax[0].N;
    mem = (e - r * p.m) + (long long)(r - t * NZ) * p.S + (long long)t * p.St;
    lds = t * p.ld + (e - t * NZ * p.m);
  } else if constexpr (LAY == ANY_AXIS) {  // (j, n): e = j + m n
    mem = (e - r * p.m) + (long long)r * p.S;
    lds = r * p.ld + (e - r * p.m);
  } else {  // rows of N contiguous elements, one LDS column each
    mem = e;
    lds = (e - r * p.ax[0].N) * p.ld + r;
  }
}

// mode: 0 forward, 1 backward, 2 forward, x p^2, backward.  blockIdx.y is
// the field, blockIdx.z a batch slice (Coulomb: one time slice)
template <typename T, int LAY, int POOL, int NTHR>
__global__ __launch_bounds__(NTHR) void k_fft_any(vec2<T> *__restrict__ F, long long fstride, AnyPass p, PsqInfo ps,
                                                 const Ctrl *__restrict__ ctrl, long long slice_len,
                                                 const int *__restrict__ slice_done,
                                                 const int *__restrict__ slice_map) {
  constexpr int NAX = any_axes(LAY);
  if (ctrl && ctrl->done) return;
  // batch row blockIdx.z is time slice zs (the rows of running slices only)
  const int zs = slice_map ? slice_map[blockIdx.z] : (int)blockIdx.z;
  if (slice_done && slice_done[zs]) return;
  __shared__ vec2<T> pool[POOL];
  int cur = 0, alt = p.pool;
  const int tw0 = 2 * p.pool;  // the twiddles of axis 0, then of axis 1
#pragma unroll
  for (int x = 0; x < NAX; x++)
    for (int k = threadIdx.x; k < p.ax[x].N; k += NTHR) {
      const double2 w = p.ax[x].tw[k];
      st<T>(pool + tw0 + x * p.ax[0].N + k, mk<T>((T)w.x, (T)w.y));
    }
  // neighbouring tiles share cache lines: each XCD gets a contiguous run
  const unsigned nb = gridDim.x;
  const unsigned tile = (nb & 7u) ? blockIdx.x : (blockIdx.x & 7u) * (nb >> 3) + (blockIdx.x >> 3);
  long long first;  // first site of the tile
  if constexpr (LAY == ANY_COLUMN) {
    first = (long long)tile * p.m;
  } else if constexpr (LAY == ANY_AXIS) {
    const unsigned p0 = tile * (unsigned)p.m, q = p0 / (unsigned)p.S;
    first = (long long)(p0 - q * (unsigned)p.S) + (long long)q * p.S * p.ax[0].N;
  } else {
    first = (long long)tile * p.elems;
  }
  vec2<T> *base = F + (long long)blockIdx.y * fstride + (long long)zs * slice_len + first;
  // four loads in flight per thread before their LDS stores; past the end
  // the last element is stored again
  for (int e0 = threadIdx.x; e0 < p.elems; e0 += 4 * NTHR) {
    vec2<T> v[4];
    int lds[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      long long mem;
      any_place<LAY>(p, min(e0 + k * NTHR, p.elems - 1), mem, lds[k]);
      v[k] = base[mem];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) pool[lds[k]] = v[k];
  }
  __syncthreads();
  // the axes in order: forward 0, 1; backward 1, 0; mode 2 both in turn
  const int steps = p.mode == 2 ? 2 * NAX : NAX;
#pragma unroll 1
  for (int i = 0; i < steps; i++) {
    const bool back = p.mode == 1 || i >= NAX;
    const int x = NAX == 1 ? 0 : (back ? (p.mode == 1 ? NAX : 2 * NAX) - 1 - i : i);
    if (i == NAX) {
      // p^2 with the zero mode set to 1 (Geometry/geometry.c:170-186), the
      // cos of x, y, z, t added in that order
      for (int e = threadIdx.x; e < p.elems; e += NTHR) {
        long long mem;
        int lds;
        any_place<LAY>(p, e, mem, lds);
        unsigned r = (unsigned)(first + mem);
        double kcos = 0.0;
        for (int mu = 0; mu < ps.D; mu++) {
          const unsigned q = __umulhi(r, ps.dm[mu]) >> ps.ds[mu];
          kcos += ps.cosv[ps.off[mu] + (int)(r - q * (unsigned)ps.L[mu])];
          r = q;
        }
        const double p2 = (kcos == (double)ps.D) ? 1.0 : 2.0 * ((double)ps.D - kcos);
        const T f = (T)(ps.max / p2);
        const cx<T> z = ld<T>(pool + cur + lds);
        st<T>(pool + cur + lds, mk<T>(z.re * f, z.im * f));
      }
      __syncthreads();
    }
    const AnyAxis &ax = p.ax[x];
    const AnyPencils pe = p.pe[x];
    const vec2<T> *tw = pool + tw0 + x * p.ax[0].N;
    for (int s = 0; s < ax.nst; s++) {
      const AnyStage sg = ax.st[s];
      const vec2<T> *src = pool + cur;
      vec2<T> *dst = pool + alt;
      const int sign = back ? +1 : -1;
      // In FP32 the compiler fuses the products of the radix-5 and radix-7
      // sums by whether it knows the sign; the axis p^2 is applied on is
      // transformed back with a known one, as it always has been, so that an
      // FP32 trajectory keeps its rounding
      if (sizeof(T) == 4 && i == NAX && (sg.R == 5 || sg.R == 7)) {
        if (sg.R == 5)
          any_stage<T, 5>(src, dst, pe, sg, tw, +1);
        else
          any_stage<T, 7>(src, dst, pe, sg, tw, +1);
      } else {
        switch (sg.R) {
          case 2: any_stage<T, 2>(src, dst, pe, sg, tw, sign); break;
          case 3: any_stage<T, 3>(src, dst, pe, sg, tw, sign); break;
          case 4: any_stage<T, 4>(src, dst, pe, sg, tw, sign); break;
          case 5: any_stage<T, 5>(src, dst, pe, sg, tw, sign); break;
          case 7: any_stage<T, 7>(src, dst, pe, sg, tw, sign); break;
          default: any_stage<T, 8>(src, dst, pe, sg, tw, sign); break;
        }
      }
      const int t = cur;
      cur = alt;
      alt = t;
    }
  }
  for (int e = threadIdx.x; e < p.elems; e += NTHR) {
    long long mem;
    int lds;
    any_place<LAY>(p, e, mem, lds);
    base[mem] = pool[cur + lds];
  }
}

// ---------------------------------------------------------------------------
// Compile-time specialisation for the common extents: N, P and the radix
// plan are constants, so every index, modulo and loop bound folds away.
// Each thread keeps one pencil for the whole pass (P divides the block), the
// twiddles sit in LDS, and the p^2 factor of the fused pass is the pencil's
// cos sum plus one table entry per element.
// ---------------------------------------------------------------------------
struct RadPlan {
  int n;
  int r[8];
};
// radix 8 first: two stages where radix 4/2 needs three (N = 32, 64), so
// one LDS round trip and two barriers fewer per pass
constexpr RadPlan make_plan(int N) {
  RadPlan p{0, {0, 0, 0, 0, 0, 0, 0, 0}};
  while (N % 8 == 0) {
    p.r[p.n++] = 8;
    N /= 8;
  }
  while (N % 4 == 0) {
    p.r[p.n++] = 4;
    N /= 4;
  }
  if (N % 2 == 0) {
    p.r[p.n++] = 2;
    N /= 2;
  }
  while (N % 3 == 0) {
    p.r[p.n++] = 3;
    N /= 3;
  }
  return p;
}
constexpr int fast_P(int N) {
  int p = 1;
  while (p * 2 <= 2048 / N && p * 2 <= 256) p *= 2;
  return p;
}

// element n of pencil j at lds[n * SN + (j % PJ) * SJ + (j / PJ) * PS]:
// pencils come in groups of PJ (one group per plane of a multi-plane tile)
template <typename T, int N, int P, int R, int Ns, int SN, int SJ, int PJ = P, int PS = 0>
__device__ __forceinline__ void fast_stage(vec2<T> *lds, const cx<T> *twl, int sign) {
  constexpr int nbf = N / R, total = nbf * P, tstep = N / (Ns * R);
  constexpr int items = (total + kFftThreads - 1) / kFftThreads;
  cx<T> v[items][R];
#pragma unroll
  for (int it = 0; it < items; it++) {
    const int w = threadIdx.x + it * kFftThreads;
    if (total % kFftThreads == 0 || w < total) {
      const int j = w % P, b = w / P, k = b % Ns;
      const int jo = (j % PJ) * SJ + (j / PJ) * PS;
#pragma unroll
      for (int q = 0; q < R; q++) v[it][q] = ld<T>(lds + (b + q * nbf) * SN + jo);
      if constexpr (Ns > 1) {
#pragma unroll
        for (int q = 1; q < R; q++) {
          cx<T> t = twl[(q * k * tstep) % N];
          if (sign > 0) t.im = -t.im;
          v[it][q] = cmul(v[it][q], t);
        }
      }
      dft_small<T, R>(v[it], sign);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < items; it++) {
    const int w = threadIdx.x + it * kFftThreads;
    if (total % kFftThreads == 0 || w < total) {
      const int j = w % P, b = w / P, k = b % Ns;
      const int jo = (j % PJ) * SJ + (j / PJ) * PS;
      const int out = (b / Ns) * Ns * R + k;
#pragma unroll
      for (int q = 0; q < R; q++) st<T>(lds + (out + q * Ns) * SN + jo, v[it][q]);
    }
  }
  __syncthreads();
}

template <typename T, int N, int P, int S_, int Ns, int SN = P + 1, int SJ = 1, int PJ = P, int PS = 0>
__device__ __forceinline__ void fast_run(vec2<T> *lds, const cx<T> *twl, int sign) {
  constexpr RadPlan pl = make_plan(N);
  if constexpr (S_ < pl.n) {
    constexpr int R = pl.r[S_];
    fast_stage<T, N, P, R, Ns, SN, SJ, PJ, PS>(lds, twl, sign);
    fast_run<T, N, P, S_ + 1, Ns * R, SN, SJ, PJ, PS>(lds, twl, sign);
  }
}

// both in-plane axes of NPL consecutive x-y planes in one pass: the planes
// (contiguous in memory) are staged as lds[x * (NPL NY + 1) + p NY + y]; the
// x transform runs on the NPL NY pencils (p, y) with stride NPL NY + 1
// between points, the y transform on the NPL NX pencils (p, x) with stride
// 1; the row length NPL NY + 1 is odd, so both access patterns are
// bank-conflict free.  With two 32 x 32 planes per workgroup every thread
// is busy in every stage (one plane leaves half of them idle in the
// radix-8 stages).
template <typename T, int NX, int NY, int NPL>
__global__ __launch_bounds__(kFftThreads) void k_fft_xy(vec2<T> *__restrict__ F, long long fstride,
                                                       const double2 *__restrict__ twx,
                                                       const double2 *__restrict__ twy, int mode,
                                                       const Ctrl *__restrict__ ctrl, long long slice_len,
                                                       const int *__restrict__ slice_done,
    const int *__restrict__ slice_map) {
  constexpr int LD = NPL * NY + 1, NE = NX * NY, NT = NPL * NE;
  if (ctrl && ctrl->done) return;
  // batch row blockIdx.z is time slice zs (the rows of running slices only)
  const int zs = slice_map ? slice_map[blockIdx.z] : (int)blockIdx.z;
  if (slice_done && slice_done[zs]) return;
  __shared__ vec2<T> lds[NX * LD];
  __shared__ cx<T> tx[NX], ty[NY];
  for (int k = threadIdx.x; k < NX; k += kFftThreads) tx[k] = mk<T>((T)twx[k].x, (T)twx[k].y);
  for (int k = threadIdx.x; k < NY; k += kFftThreads) ty[k] = mk<T>((T)twy[k].x, (T)twy[k].y);
  vec2<T> *base =
      F + (long long)blockIdx.y * fstride + (long long)zs * slice_len + (long long)blockIdx.x * NT;
  // element e of the tile: plane e / NE, row (e % NE) / NX, column e % NX
#pragma unroll 4
  for (int e = threadIdx.x; e < NT; e += kFftThreads) lds[(e % NX) * LD + e / NX] = base[e];
  __syncthreads();
  const int sign = mode == 1 ? +1 : -1;
  fast_run<T, NX, NPL * NY, 0, 1, LD, 1>(lds, tx, sign);
  fast_run<T, NY, NPL * NX, 0, 1, 1, LD, NX, NY>(lds, ty, sign);
#pragma unroll 4
  for (int e = threadIdx.x; e < NT; e += kFftThreads) base[e] = lds[(e % NX) * LD + e / NX];
}

// ---- launches of the run-time pass
// extents with compile-time kernels keep their radix order (8 first)
static bool fast_extent(int N) {
  for (int n : {4, 6, 8, 12, 16, 24, 32, 48, 64, 96})
    if (n == N) return true;
  return false;
}
// axes of 48 and 96 points stay with their compile-time passes in FP32: the
// three-stage kernels round some products differently, and an FP32
// trajectory follows the rounding.  It costs little: an FP32 iteration takes
// 282, 465, 1058 and 3807 us on 48x12x12x96, 24^3x96, 32^3x96 and 48^3x96,
// where the run-time passes take 298, 500, 1140 and 4235, and 105 and 76 on
// 16^3x48 and 10^3x48, where they take 102 and 71
template <typename T> static bool any_keeps_rounding(const FftAxis &ax) {
  return sizeof(T) == 8 || (ax.N != 48 && ax.N != 96);
}
static AnyAxis any_axis_plan(const FftAxis &ax) {
  AnyAxis a{};
  a.N = ax.N;
  a.tw = ax.tw;
  const RadPlan fast = make_plan(ax.N);
  const bool f = fast_extent(ax.N);
  a.nst = f ? fast.n : ax.nst;
  int Ns = 1;
  for (int s = 0; s < a.nst; s++) {
    const int R = f ? fast.r[s] : ax.rad[s];
    a.st[s] = AnyStage{(unsigned short)R, (unsigned short)Ns, (unsigned short)(ax.N / R),
                       (unsigned short)(ax.N / (Ns * R)), any_mul((unsigned)Ns)};
    Ns *= R;
  }
  return a;
}
static AnyPencils any_pencils(int P, int SN, int SJ, int PJ, int PS) {
  return AnyPencils{P, SN, SJ, PJ, PS, any_mul((unsigned)P), any_mul((unsigned)PJ)};
}
// LDS of a workgroup in complex numbers: 40, 80 and 160 KB in FP64 (4, 2
// and 1 workgroups per CU), half of that in FP32
constexpr int kAnyPool[3] = {2560, 5120, 10000};

// the largest divisor m of n whose tile (need(m) LDS numbers) fits `pool`
// and leaves at least `least` tiles; 0 if not even m = 1 fits
template <typename Need> static int any_split(long long n, int pool, long long least, Need need) {
  int best = 0;
  for (int m = 1; m <= n && m <= 256; m++) {
    if (n % m) continue;
    if (need(m) > pool) break;
    if (m > 1 && n / m < least) break;
    best = m;
  }
  return best;
}

// Two axes that both have compile-time passes: does the run-time pass over
// both pay?  It saves launches, one of a plane's two or two of a column's
// three, but its run-time plan costs more per number, so it may pay up to a
// volume only.  The lines, in sites (4 fields), lie where the times of a
// whole iteration cross (us with single axes / with the run-time pass):
//  - x-y planes of up to 64x64 points pay at any volume (32x64x32x32 1128 /
//    1070 in FP64, 834 / 838 in FP32), larger ones to 2^21 (48x96x16x16 674 /
//    630, 48x96x24x24 1420 / 1437);
//  - z-t columns in tiles several sites wide pay at any volume in FP64
//    (32^2x8x64 253 / 247, 48^2x24^2 688 / 682), to 2^19 in FP32 (230 / 225,
//    529 / 537);
//  - columns in tiles one site wide, whose loads are runs of one number, pay
//    to 2^18 in FP64 (16^3x48 110 / 103, 8^2x64^2 183 / 176, 16^2x32x48 199 /
//    201, 32^3x96 1575 / 1694, 48^3x96 5.56 / 6.31 ms) and 2^17 in FP32
//    (8^2x64x32 89 / 88, 16^2x32^2 124 / 124, 48^2x24x64 1325 / 1467).
static bool any_pays(const FftAxis &a, const FftAxis &b, long long numbers, long long sites) {
  return !fast_extent(a.N) || !fast_extent(b.N) || numbers <= 4 * sites;
}

template <typename T, int LAY>
static void launch_any(void *F, long long fstride, int nfield, const AnyPass &p, unsigned tiles, const PsqInfo &ps,
                       const Ctrl *ctrl, hipStream_t s, int nslice, long long slice_len, const int *slice_done,
                       const int *slice_map) {
  const int need = 2 * p.pool + p.ax[0].N + (any_axes(LAY) > 1 ? p.ax[1].N : 0);
  const dim3 grid(tiles, nfield, nslice);
  if (need <= kAnyPool[0])
    hipLaunchKernelGGL((k_fft_any<T, LAY, kAnyPool[0], 256>), grid, dim3(256), 0, s, (vec2<T> *)F, fstride, p, ps, ctrl,
                       slice_len, slice_done, slice_map);
  else if (need <= kAnyPool[1])
    hipLaunchKernelGGL((k_fft_any<T, LAY, kAnyPool[1], 512>), grid, dim3(512), 0, s, (vec2<T> *)F, fstride, p, ps, ctrl,
                       slice_len, slice_done, slice_map);
  else
    hipLaunchKernelGGL((k_fft_any<T, LAY, kAnyPool[2], 512>), grid, dim3(512), 0, s, (vec2<T> *)F, fstride, p, ps, ctrl,
                       slice_len, slice_done, slice_map);
}

// Tiles a pass is split into at least.  Per pass on 28x36x42x32 FP64: 85 us
// with 256 or 512 tiles, 90 with 1024, 84 with 2048; on 20x28x10x36 21.3, 23
// and 25 us with 512, 1024 and 2048, and 12x12x12x24 11.4 us with up to 512,
// 13 above
constexpr long long kAnyTiles = 512;

// x-y planes of any extents (false when a plane does not fit the LDS)
template <typename T>
static bool any_plane(void *F, long long fstride, int nfield, const FftAxis &ax, const FftAxis &ay, int mode,
                      const Ctrl *ctrl, hipStream_t s, long long nplane, int nslice, long long slice_len,
                      const int *slice_done, const int *slice_map) {
  const int NX = ax.N, NY = ay.N;
  auto need = [&](int m) { return 2 * NX * ((m * NY) | 1) + NX + NY; };
  if (!any_keeps_rounding<T>(ax) || !any_keeps_rounding<T>(ay)) return false;
  if ((long long)NX * NY > kAnyPool[2] || need(1) > kAnyPool[2]) return false;
  if (NX * NY > 4096 && !any_pays(ax, ay, nfield * nslice * nplane * NX * NY, 1 << 21)) return false;
  int m = any_split(nplane, kAnyPool[0], kAnyTiles / ((long long)nfield * nslice) + 1, need);
  if (!m) m = 1;
  AnyPass p{};
  p.mode = mode;
  p.m = m;
  p.ld = (m * NY) | 1;
  p.elems = m * NX * NY;
  p.pool = NX * p.ld;
  p.mRow = any_mul((unsigned)NX);
  p.S = 1;
  p.ax[0] = any_axis_plan(ax);
  p.ax[1] = any_axis_plan(ay);
  p.pe[0] = any_pencils(m * NY, p.ld, 1, m * NY, 0);   // x pencil (plane, y)
  p.pe[1] = any_pencils(m * NX, 1, p.ld, NX, NY);      // y pencil (plane, x)
  launch_any<T, ANY_PLANE>(F, fstride, nfield, p, (unsigned)(nplane / m), PsqInfo{}, ctrl, s, nslice, slice_len, slice_done,
                slice_map);
  return true;
}

// z-t columns of any extents, m neighbouring x-y sites per tile.  The
// smallest LDS pool that holds a column: longer runs in a larger pool were
// no faster (36x36x36x40 FP64: 127 us per pass with runs of 16 B, 128 with
// 64), the columns of one XCD share the lines in its L2
template <typename T>
static bool any_column(void *F, long long V, int nfield, const FftAxis &ax, const FftAxis &ay, const FftAxis &az,
                       const FftAxis &at, const PsqInfo &ps, const Ctrl *ctrl, hipStream_t s, bool launch) {
  const int NZ = az.N, NT = at.N;
  const long long nxy = (long long)ax.N * ay.N;
  auto need = [&](int m) { return 2 * NT * ((m * NZ) | 1) + NZ + NT; };
  if (!any_keeps_rounding<T>(az) || !any_keeps_rounding<T>(at)) return false;
  if ((long long)NZ * NT > kAnyPool[2] || need(1) > kAnyPool[2]) return false;
  int m = 0;
  for (int k = 0; k < 3 && !m; k++) m = any_split(nxy, kAnyPool[k], kAnyTiles / nfield, need);
  if ((sizeof(T) == 4 || m == 1) &&
      !any_pays(az, at, nfield * V, sizeof(T) == 8 ? 1 << 18 : m == 1 ? 1 << 17 : 1 << 19))
    return false;
  if (!launch) return true;
  AnyPass p{};
  p.mode = 2;
  p.m = m;
  p.ld = (m * NZ) | 1;
  p.elems = m * NZ * NT;
  p.pool = NT * p.ld;
  p.mRow = any_mul((unsigned)m);
  p.mZ = any_mul((unsigned)NZ);
  p.S = nxy;
  p.St = nxy * NZ;
  p.ax[0] = any_axis_plan(az);
  p.ax[1] = any_axis_plan(at);
  p.pe[0] = any_pencils(m * NT, m, 1, m, p.ld);       // z pencil (t, j)
  p.pe[1] = any_pencils(m * NZ, p.ld, 1, m * NZ, 0);  // t pencil (z, j)
  launch_any<T, ANY_COLUMN>(F, V, nfield, p, (unsigned)(nxy / m), ps, ctrl, s, 1, 0, nullptr, nullptr);
  return true;
}

// one axis of any extent: m pencils per tile, neighbours in memory (m
// divides the stride, so a tile never straddles two pencil rows)
template <typename T>
static void any_single(void *F, long long fstride, int nfield, const FftAxis &ax, int mode, const PsqInfo &ps,
                       const Ctrl *ctrl, hipStream_t s, int nslice, long long slice_len, const int *slice_done,
                       const int *slice_map) {
  const int N = ax.N;
  auto need = [&](int m) { return 2 * N * (m | 1) + N; };
  const long long n = ax.S == 1 ? ax.npencil : ax.S;
  int m = any_split(n, kAnyPool[0], 1, need);
  if (!m) m = 1;  // N up to 2048: 3 N numbers fit the largest pool
  AnyPass p{};
  p.mode = mode;
  p.m = m;
  p.ld = m | 1;
  p.elems = m * N;
  p.pool = N * p.ld;
  p.mRow = any_mul((unsigned)(ax.S == 1 ? N : m));
  p.S = ax.S;
  p.ax[0] = any_axis_plan(ax);
  p.pe[0] = any_pencils(m, p.ld, 1, m, 0);
  const unsigned tiles = (unsigned)(ax.npencil / m);
  if (ax.S == 1)
    launch_any<T, ANY_ROW>(F, fstride, nfield, p, tiles, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
  else
    launch_any<T, ANY_AXIS>(F, fstride, nfield, p, tiles, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
}

template <typename T, int N>
static bool try_xy(void *F, long long fstride, int nfield, const FftAxis &ax, const FftAxis &ay, int mode,
                   const Ctrl *ctrl, hipStream_t s, long long nplane, int nslice, long long slice_len,
                   const int *slice_done, const int *slice_map) {
  if (ax.N != N || ay.N != N) return false;
  if (sizeof(T) * 2 * N * (N + 1) > 48 * 1024) return false;
  // two planes per tile in FP32 where a plane has at most 1024 points (the
  // tile's row e / NX runs over (plane, y)); in FP64 the doubled tile
  // halves the workgroups an LDS holds and gained nothing at 32 x 32
  constexpr int NPL = (sizeof(T) == 4 && N * N <= 1024) ? 2 : 1;
  if (NPL == 2 && nplane % 2 == 0)
    hipLaunchKernelGGL((k_fft_xy<T, N, N, NPL>), dim3((unsigned)(nplane / 2), nfield, nslice), dim3(kFftThreads),
                       0, s, (vec2<T> *)F, fstride, ax.tw, ay.tw, mode, ctrl, slice_len, slice_done, slice_map);
  else
    hipLaunchKernelGGL((k_fft_xy<T, N, N, 1>), dim3((unsigned)nplane, nfield, nslice), dim3(kFftThreads), 0, s,
                       (vec2<T> *)F, fstride, ax.tw, ay.tw, mode, ctrl, slice_len, slice_done, slice_map);
  return true;
}

template <typename T>
bool launch_fft_xy(void *F, long long fstride, int nfield, const FftAxis &ax, const FftAxis &ay, int mode,
                   const Ctrl *ctrl, hipStream_t s, long long nplane, int nslice, long long slice_len,
                   const int *slice_done, const int *slice_map) {
  return try_xy<T, 8>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map) ||
         try_xy<T, 16>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map) ||
         try_xy<T, 24>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map) ||
         try_xy<T, 32>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map) ||
         try_xy<T, 48>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map) ||
         any_plane<T>(F, fstride, nfield, ax, ay, mode, ctrl, s, nplane, nslice, slice_len, slice_done, slice_map);
}
template bool launch_fft_xy<double>(void *, long long, int, const FftAxis &, const FftAxis &, int, const Ctrl *,
                                    hipStream_t, long long, int, long long, const int *, const int *);
template bool launch_fft_xy<float>(void *, long long, int, const FftAxis &, const FftAxis &, int, const Ctrl *,
                                   hipStream_t, long long, int, long long, const int *, const int *);

// The z and t axes of the 4D transform in one LDS residency: forward z,
// forward t, x p^2, backward t, backward z, for PX consecutive x values of
// one y (a "column" of z-t planes), after the forward x-y plane pass and
// before the backward one.  Three passes over the fields per Fourier
// acceleration instead of five.  The pencils' arithmetic is that of the
// single-axis passes (same radix plan, twiddles and p^2 summation order).
// Element (j, z, t) of the column sits at lds[t RZ + z PX + j]; a t row is
// padded to RZ = NZ PX + 1 entries.  Workgroups are dealt to the 8 XCDs
// round-robin; logical block l = (b % 8) nb/8 + b / 8 gives each XCD a
// contiguous run of columns, so the x groups sharing a cache line are
// fetched into one L2.
template <typename T, int NZ, int NT, int PX>
__global__ __launch_bounds__(kFftThreads) void k_fft_zt(vec2<T> *__restrict__ F, long long V, int Lx, int Ly,
                                                       const double2 *__restrict__ twz,
                                                       const double2 *__restrict__ twt, PsqInfo ps,
                                                       const Ctrl *__restrict__ ctrl) {
  constexpr int RZ = NZ * PX + 1, NE = NZ * NT * PX;
  if (ctrl && ctrl->done) return;
  __shared__ vec2<T> lds[NT * RZ];
  __shared__ cx<T> tz[NZ], tt[NT];
  for (int k = threadIdx.x; k < NZ; k += kFftThreads) tz[k] = mk<T>((T)twz[k].x, (T)twz[k].y);
  for (int k = threadIdx.x; k < NT; k += kFftThreads) tt[k] = mk<T>((T)twt[k].x, (T)twt[k].y);
  // logical block -> (field, y, x group); gridDim.x is a multiple of 8
  const unsigned nb = gridDim.x, b = blockIdx.x;
  const unsigned l = (b & 7u) * (nb >> 3) + (b >> 3);
  const int ngx = Lx / PX;
  const unsigned cols = (unsigned)(ngx * Ly);
  const int field = (int)(l / cols), col = (int)(l % cols);
  const int xg = col % ngx, y = col / ngx;
  const long long Sz = (long long)Lx * Ly, St = Sz * NZ;
  vec2<T> *base = F + (long long)field * V + (long long)xg * PX + (long long)y * Lx;
  // the column's loads are all issued before any is stored to LDS: with
  // runs of only PX elements per (z, t) row the pass is bound by the bytes
  // each thread keeps in flight
  if constexpr (NE % kFftThreads == 0) {
    constexpr int K = NE / kFftThreads;
    vec2<T> r[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int e = threadIdx.x + k * kFftThreads;
      const int j = e % PX, z = (e / PX) % NZ, t = e / (PX * NZ);
      r[k] = base[j + z * Sz + t * St];
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
      const int e = threadIdx.x + k * kFftThreads;
      const int j = e % PX, z = (e / PX) % NZ, t = e / (PX * NZ);
      lds[t * RZ + z * PX + j] = r[k];
    }
  } else {
    for (int e = threadIdx.x; e < NE; e += kFftThreads) {
      const int j = e % PX, z = (e / PX) % NZ, t = e / (PX * NZ);
      lds[t * RZ + z * PX + j] = base[j + z * Sz + t * St];
    }
  }
  __syncthreads();
  // forward z: pencil (j, t) at j + t RZ, points PX apart
  fast_run<T, NZ, PX * NT, 0, 1, PX, 1, PX, RZ>(lds, tz, -1);
  // forward t: pencil (j, z) at z PX + j, points RZ apart
  fast_run<T, NT, PX * NZ, 0, 1, RZ, 1>(lds, tt, -1);
  // p^2 = 2 (4 - sum cos) with p^2(0) := 1 (Geometry/geometry.c:170-186),
  // the cos of x, y, z, t added in that order
  const double *cx_ = ps.cosv + ps.off[0], *cy_ = ps.cosv + ps.off[1];
  const double *cz_ = ps.cosv + ps.off[2], *ct_ = ps.cosv + ps.off[3];
#pragma unroll 4
  for (int e = threadIdx.x; e < NE; e += kFftThreads) {
    const int j = e % PX, z = (e / PX) % NZ, t = e / (PX * NZ);
    double kc = 0.0;
    kc += cx_[xg * PX + j];
    kc += cy_[y];
    kc += cz_[z];
    const double kcos = kc + ct_[t];
    const double p2 = (kcos == 4.0) ? 1.0 : 2.0 * (4.0 - kcos);
    const T f = (T)(ps.max / p2);
    const int a = t * RZ + z * PX + j;
    const cx<T> v = ld<T>(lds + a);
    st<T>(lds + a, mk<T>(v.re * f, v.im * f));
  }
  __syncthreads();
  fast_run<T, NT, PX * NZ, 0, 1, RZ, 1>(lds, tt, +1);
  fast_run<T, NZ, PX * NT, 0, 1, PX, 1, PX, RZ>(lds, tz, +1);
#pragma unroll 8
  for (int e = threadIdx.x; e < NE; e += kFftThreads) {
    const int j = e % PX, z = (e / PX) % NZ, t = e / (PX * NZ);
    base[j + z * Sz + t * St] = lds[t * RZ + z * PX + j];
  }
}

// x values (pencils) of a z-t column per workgroup: variant 0 the largest
// power of two whose tile fits 40 KiB of LDS (2 in FP32, 1 in FP64 at
// 32 x 64), variant 1 half of it, variant 2 twice it where the tile stays
// within 96 KiB (gfx950 gives a workgroup up to 160 KiB)
template <typename T, int NZ, int NT> constexpr int zt_px(int v) {
  constexpr int bytes = NZ * NT * (int)sizeof(vec2<T>);
  int p = 1;
  while (p * 2 * bytes <= 40 * 1024 && p < 8) p *= 2;
  if (v == 1) return p > 1 ? p / 2 : p;
  if (v == 2) return (2 * p * NZ + 1) * NT * (int)sizeof(vec2<T>) <= 98304 ? 2 * p : p;
  return p;
}

template <typename T, int NZ, int NT, int PX>
static bool zt_go(void *F, long long V, int nfield, const FftAxis &ax, const FftAxis &ay, const FftAxis &az,
                  const FftAxis &at, const PsqInfo &ps, const Ctrl *ctrl, hipStream_t s, bool launch) {
  if (ax.N % PX) return false;
  const long long nb = (long long)(ax.N / PX) * ay.N * nfield;
  if (nb % 8 || nb > (1ll << 30)) return false;
  if (!launch) return true;
  hipLaunchKernelGGL((k_fft_zt<T, NZ, NT, PX>), dim3((unsigned)nb), dim3(kFftThreads), 0, s, (vec2<T> *)F, V,
                     ax.N, ay.N, az.tw, at.tw, ps, ctrl);
  return true;
}

template <typename T, int NZ, int NT>
static bool try_zt(void *F, long long V, int nfield, const FftAxis &ax, const FftAxis &ay, const FftAxis &az,
                   const FftAxis &at, const PsqInfo &ps, const Ctrl *ctrl, hipStream_t s, bool launch, int v) {
  if (az.N != NZ || at.N != NT) return false;
  if (v == 1) return zt_go<T, NZ, NT, zt_px<T, NZ, NT>(1)>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch);
  if (v == 2) return zt_go<T, NZ, NT, zt_px<T, NZ, NT>(2)>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch);
  return zt_go<T, NZ, NT, zt_px<T, NZ, NT>(0)>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch);
}

template <typename T>
bool launch_fft_zt(void *F, long long V, int nfield, const FftAxis &ax, const FftAxis &ay, const FftAxis &az,
                   const FftAxis &at, const PsqInfo &ps, const Ctrl *ctrl, hipStream_t s, bool launch, int v) {
  if (ps.D != 4) return false;
  return try_zt<T, 8, 8>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch, v) ||
         try_zt<T, 16, 16>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch, v) ||
         try_zt<T, 16, 32>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch, v) ||
         try_zt<T, 24, 48>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch, v) ||
         try_zt<T, 32, 64>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch, v) ||
         (v == 0 && any_column<T>(F, V, nfield, ax, ay, az, at, ps, ctrl, s, launch));
}
template bool launch_fft_zt<double>(void *, long long, int, const FftAxis &, const FftAxis &, const FftAxis &,
                                    const FftAxis &, const PsqInfo &, const Ctrl *, hipStream_t, bool, int);
template bool launch_fft_zt<float>(void *, long long, int, const FftAxis &, const FftAxis &, const FftAxis &,
                                   const FftAxis &, const PsqInfo &, const Ctrl *, hipStream_t, bool, int);

template <typename T, int N, int P>
__global__ __launch_bounds__(kFftThreads) void k_fft_fast(vec2<T> *__restrict__ F, long long fstride, long long S,
                                                         long long npencil, const double2 *__restrict__ tw, int mode,
                                                         PsqInfo ps, const Ctrl *__restrict__ ctrl,
                                                         long long slice_len, const int *__restrict__ slice_done,
    const int *__restrict__ slice_map) {
  constexpr int LD = P + 1, TOT = N * P;
  static_assert(LD > 0, "");
  static_assert(kFftThreads % P == 0, "a pencil per thread needs P | threads");
  if (ctrl && ctrl->done) return;
  // batch row blockIdx.z is time slice zs (the rows of running slices only)
  const int zs = slice_map ? slice_map[blockIdx.z] : (int)blockIdx.z;
  if (slice_done && slice_done[zs]) return;
  __shared__ vec2<T> lds[N * LD];
  __shared__ cx<T> twl[N];
  for (int k = threadIdx.x; k < N; k += kFftThreads) twl[k] = mk<T>((T)tw[k].x, (T)tw[k].y);
  vec2<T> *base = F + (long long)blockIdx.y * fstride + (long long)zs * slice_len;
  const long long p0 = (long long)blockIdx.x * P;
  // this thread's pencil and first element (strided axes)
  const int jt = threadIdx.x % P, n0 = threadIdx.x / P;
  constexpr int nstep = kFftThreads / P;
  const long long pt = p0 + jt;
  const bool valid = pt < npencil;
  long long a0 = 0;
  if (S != 1 && valid) a0 = (pt % S) + (pt / S) * S * N;
  if (S == 1) {
    const long long lim = (npencil - p0) * N;  // elements left in this chunk
    const vec2<T> *src = base + p0 * N;
    for (int idx = threadIdx.x; idx < TOT; idx += kFftThreads)
      if (idx < lim) lds[(idx % N) * LD + idx / N] = src[idx];
  } else if (valid) {
#pragma unroll 4
    for (int n = n0; n < N; n += nstep) lds[n * LD + jt] = base[a0 + (long long)n * S];
  }
  __syncthreads();
  if (mode == 1)
    fast_run<T, N, P, 0, 1>(lds, twl, +1);
  else
    fast_run<T, N, P, 0, 1>(lds, twl, -1);
  if (mode == 2) {
    // p^2 = 2 (D - sum cos) with p^2(0) := 1 (Geometry/geometry.c:170-186);
    // the fused axis is the last of the D, so its cos enters the sum last
    double kc = 0.0;
    long long r = a0;
    for (int mu = 0; mu < ps.D - 1; mu++) {
      kc += ps.cosv[ps.off[mu] + (int)(r % ps.L[mu])];
      r /= ps.L[mu];
    }
    const double *cl = ps.cosv + ps.off[ps.D - 1];
    if (valid && S != 1) {
#pragma unroll 4
      for (int n = n0; n < N; n += nstep) {
        const double kcos = kc + cl[n];
        const double p2 = (kcos == (double)ps.D) ? 1.0 : 2.0 * ((double)ps.D - kcos);
        const T f = (T)(ps.max / p2);
        const cx<T> z = ld<T>(lds + n * LD + jt);
        st<T>(lds + n * LD + jt, mk<T>(z.re * f, z.im * f));
      }
    }
    __syncthreads();
    fast_run<T, N, P, 0, 1>(lds, twl, +1);
  }
  if (S == 1) {
    const long long lim = (npencil - p0) * N;
    vec2<T> *dst = base + p0 * N;
    for (int idx = threadIdx.x; idx < TOT; idx += kFftThreads)
      if (idx < lim) dst[idx] = lds[(idx % N) * LD + idx / N];
  } else if (valid) {
#pragma unroll 4
    for (int n = n0; n < N; n += nstep) base[a0 + (long long)n * S] = lds[n * LD + jt];
  }
}

// pencils per workgroup of variant v: the default fast_P(N), half of it,
// or twice it where the LDS tile stays within 64 KB
template <typename T, int N> constexpr int variant_P(int v) {
  constexpr int P0 = fast_P(N);
  if (v == 1) return P0 > 1 ? P0 / 2 : P0;
  if (v == 2) return (2 * P0 <= kFftThreads && N * (2 * P0 + 1) * (int)sizeof(vec2<T>) <= 65536) ? 2 * P0 : P0;
  return P0;
}

template <typename T, int N, int P>
static void run_fast(void *F, long long fstride, int nfield, const FftAxis &ax, int mode, const PsqInfo &ps,
                     const Ctrl *ctrl, hipStream_t s, int nslice, long long slice_len, const int *slice_done, const int *slice_map) {
  const unsigned nb = (unsigned)((ax.npencil + P - 1) / P);
  hipLaunchKernelGGL((k_fft_fast<T, N, P>), dim3(nb, nfield, nslice), dim3(kFftThreads), 0, s, (vec2<T> *)F,
                     fstride, ax.S, ax.npencil, ax.tw, mode, ps, ctrl, slice_len, slice_done, slice_map);
}

template <typename T, int N>
static bool try_fast(void *F, long long fstride, int nfield, const FftAxis &ax, int mode, const PsqInfo &ps,
                     const Ctrl *ctrl, hipStream_t s, int nslice, long long slice_len, const int *slice_done, const int *slice_map) {
  if (ax.N != N) return false;
  // the fused p^2 pass runs on a strided axis (it is always the last one)
  if (mode == 2 && ax.S == 1) return false;
  if (ax.pv == 1)
    run_fast<T, N, variant_P<T, N>(1)>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
  else if (ax.pv == 2)
    run_fast<T, N, variant_P<T, N>(2)>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
  else
    run_fast<T, N, variant_P<T, N>(0)>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
  return true;
}

template <typename T>
void launch_fft_axis(void *F, long long fstride, int nfield, const FftAxis &ax, int mode, const PsqInfo &ps,
                     const Ctrl *ctrl, hipStream_t s, int nslice, long long slice_len, const int *slice_done, const int *slice_map) {
  if (try_fast<T, 4>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 6>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 8>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 12>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 16>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 24>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 32>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 48>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 64>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map) ||
      try_fast<T, 96>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map))
    return;
  any_single<T>(F, fstride, nfield, ax, mode, ps, ctrl, s, nslice, slice_len, slice_done, slice_map);
}
template void launch_fft_axis<double>(void *, long long, int, const FftAxis &, int, const PsqInfo &, const Ctrl *,
                                      hipStream_t, int, long long, const int *, const int *);
template void launch_fft_axis<float>(void *, long long, int, const FftAxis &, int, const PsqInfo &, const Ctrl *,
                                     hipStream_t, int, long long, const int *, const int *);

}  // namespace gfix
