// landau_kernels.hip -- site-parallel streaming kernels of the Landau
// FACG/FASD iteration: derivative + theta, Polak-Ribiere sums, CG update,
// three-probe line search, gauge update, control kernels, and the
// link (re)packing / measurement kernels around them.
//
// One thread per lattice site, 256-thread blocks, SoA planes (coalesced),
// FP64 per-block partial sums reduced by a single-block kernel in a fixed
// order (bitwise reproducible, independent of what else runs on the GPU).
#include "gfix_kernels.h"

namespace gfix {

// ---------------------------------------------------------------------------
// derivative: Gfix/lin_derivs.c:75-193 + packing Gfix/FACG.c:38-73
// ---------------------------------------------------------------------------
// Delta(x) and its packing: DerivAcc (gfix_device.h)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_deriv(const vec2<T> *__restrict__ U, vec2<T> *__restrict__ F,
                                                 double *__restrict__ part, Geo g, const Ctrl *__restrict__ ctrl) {
  if (ctrl && ctrl->done) return;
  const long long V = g.V;
  const unsigned lb = logical_block(g);
  const long long i = (long long)lb * blockDim.x + threadIdx.x;
  double loc[1] = {0.0};
  if (i < V) {
    int x[4];
    coords(g, i, x);
    DerivAcc<T> d;
#pragma unroll
    for (int mu = 0; mu < kND; mu++)
      d.add(load_link<T>(U, mu, i, V), load_link<T>(U, mu, nb_bwd(g, i, x, mu), V));
    loc[0] = d.store(F, V, i);
  }
  block_sum_store<1>(loc, part + lb);
}

// ---------------------------------------------------------------------------
// trace-metric sums of the packed field: Gfix/FACG.c:99-178
//   s1 = <in, in>,  s2 = <in, in - old>
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_pr_sums(const vec2<T> *__restrict__ F, const vec2<T> *__restrict__ O,
                                                   double *__restrict__ part, long long V,
                                                   const Ctrl *__restrict__ ctrl) {
  if (ctrl && ctrl->done) return;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  double v[2] = {0.0, 0.0};
  if (i < V) {
    double s1 = 0.0, s2 = 0.0;
    const cx<T> z0t = ld<T>(F + i), o0t = ld<T>(O + i);
    const double zr = z0t.re, zi = z0t.im, tr = zr - (double)o0t.re, ti = zi - (double)o0t.im;
    s1 += 2.0 * (zr * zr + zi * zi + zr * zi);
    s2 += 2.0 * (zr * tr + zi * ti);
    s2 += zr * ti + zi * tr;
#pragma unroll
    for (int f = 1; f < 4; f++) {
      const cx<T> z = ld<T>(F + f * V + i), o = ld<T>(O + f * V + i);
      const double ar = z.re, ai = z.im;
      s1 += 2.0 * (ar * ar + ai * ai);
      s2 += 2.0 * (ar * (ar - (double)o.re) + ai * (ai - (double)o.im));
    }
    v[0] = s1;
    v[1] = s2;
  }
  block_sum_store<2>(v, part + 2 * blockIdx.x);
}

// Small lattices (up to kSmallBlocks partial rows) run without the
// single-block finalisers of the PR sums and of the line search: every block
// of the kernel that needs beta or the step adds the partial rows itself, in
// the order of final_sum, and block 0 writes the scalars, none of which the
// kernel's other blocks read.  At 8^4 a finaliser took 3 to 4 us of an
// iteration's 47.  The line: one row for each thread of a block.  Iteration
// with and without the small-lattice kernels (FP64 / mixed, us): 4^4 41 / 41
// and 52 / 52, 8^4 34 / 42 and 47 / 56, 12^4 58 / 63 and 69 / 76, 14^4 73 /
// 78 and 81 / 89, 16^4 71 / 70 and 72 / 73: at 16^4 every CU has its
// wavefronts without the split and the gain ends.
constexpr long long kSmallBlocks = 256;
// one row a thread; a row may be kept as the 4 sums of its block's waves
template <int NV>
__device__ __forceinline__ void small_sum(const double *__restrict__ part, long long nb, int sub, double (&out)[NV]) {
  __shared__ double sh[NV][kBlock / kWave];
  const int b = threadIdx.x;
#pragma unroll
  for (int k = 0; k < NV; k++) {
    double v = 0.0;
    if (b < nb) {
      if (sub == 1)
        v = part[(long long)b * NV + k];
      else
        for (int j = 0; j < 4; j++) v += part[((long long)b * 4 + j) * NV + k];
    }
    v = wave_sum(v);
    if (threadIdx.x % kWave == 0) sh[k][threadIdx.x / kWave] = v;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; k++) {
    out[k] = 0.0;
    for (int j = 0; j < kBlock / kWave; j++) out[k] += sh[k][j];
  }
}

// beta: Polak-Ribiere clipped at 0, Fletcher-Reeves below CG_TOL
// (Gfix/FACG.c:306-313)
__device__ __forceinline__ double pr_beta(const Ctrl *ctrl, double insum, double sc) {
  double beta = sc / ctrl->inold;
  if (beta < 0.0) beta = 0.0;
  if (ctrl->theta < ctrl->cg_tol) beta = insum / ctrl->inold;
  if (ctrl->switch_theta > 0.0) {  // safeguards of the mixed FP32 phase
    if ((ctrl->sg_mode & 1) && ctrl->sg_uphill) beta = 0.0;
    if ((ctrl->sg_mode & 2) && beta > ctrl->beta_cap) beta = ctrl->beta_cap;
  }
  return beta;
}
__device__ __forceinline__ void pr_record(Ctrl *ctrl, double insum, double sc, double beta) {
  ctrl->insum = insum;  // becomes inold with the step (ls_record)
  ctrl->sum_conj = sc;
  ctrl->beta = beta;
}

// sn = in + beta sn (Gfix/FACG.c:315-323).  GLU's old = in needs no copy:
// the fused update writes the next derivative into the field buffer that
// held in_old, and the host swaps the two, so `in` becomes in_old in place.
// nb > 0: beta comes from the nb partial rows of the PR sums.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg_update(const vec2<T> *__restrict__ F, vec2<T> *__restrict__ sn,
                                                     long long n4, Ctrl *ctrl, const double *__restrict__ part,
                                                     long long nb) {
  if (ctrl->done) return;
  double b;
  if (nb > 0) {
    double s[2];
    small_sum<2>(part, nb, 1, s);
    b = pr_beta(ctrl, s[0], s[1]);
    if (blockIdx.x == 0 && threadIdx.x == 0) pr_record(ctrl, s[0], s[1], b);
  } else {
    b = ctrl->beta;
  }
  const T beta = (T)b;
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < n4; j += (long long)gridDim.x * blockDim.x) {
    const cx<T> a = ld<T>(F + j), b = ld<T>(sn + j);
    st<T>(sn + j, mk<T>(a.re + beta * b.re, a.im + beta * b.im));
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_copy(const vec2<T> *__restrict__ F, vec2<T> *__restrict__ a, long long n4,
                                                const Ctrl *__restrict__ ctrl) {
  if (ctrl->done) return;
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < n4; j += (long long)gridDim.x * blockDim.x)
    a[j] = F[j];
}

template <typename T>
__device__ __forceinline__ su3<T> gauge_at(const vec2<T> *__restrict__ F, long long V, long long i, T alpha) {
  return gauge_matrix<T>(ld<T>(F + i), ld<T>(F + V + i), ld<T>(F + 2 * V + i), ld<T>(F + 3 * V + i), alpha);
}

// ---------------------------------------------------------------------------
// line search probes: Gfix/line_search.c:274-341 (probes PL1 = 0.15,
// PL2 = 0.30 at :34-35).  Skipped (no partials) when theta <= CG_TOL unless
// forced (the SD start always searches).  The probes are evaluations of the
// functional, so they are computed in FP64 whatever the storage type: in
// FP32 the rounding of the reunitarised probe matrices biases the O(12 V)
// sums by more than the differences the parabola fit needs.
//
// Bound by FP64 issue (about 2500 instructions a site).  Both probes are
// taken in one pass: the links and the neighbours' fields are loaded and
// converted once, and no third column of a link or a neighbour's matrix is
// formed (retrace_cols).  In FP64 the two matrices of a site share their
// inner products (ProbeSite); the FP32 phase builds each by Gram-Schmidt and
// sums over 8 x 4 x 4 x 2 tiles, because its trajectory follows the rounding
// of the step.  It runs at 2 waves per SIMD (218 VGPRs, 184 in FP32): the
// two probes' chains fill the issue slots, where one probe at a time at 3
// waves took 253 us and capped at 4 waves, spilling, 795.  32^3x64: 242 us
// in FP64 (388 with the matrices shared through LDS on tiles, 306 with one
// probe at a time and three-column traces), 238 from FP32 links (281 on LDS
// tiles); the bytes alone would take 180 and 90.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ su3<double> gauge_at64(const vec2<T> *__restrict__ F, long long V, long long i,
                                                  double alpha) {
  auto f = [&](long long k) {
    const cx<T> z = ld<T>(F + k);
    return mk<double>((double)z.re, (double)z.im);
  };
  return gauge_matrix<double>(f(i), f(V + i), f(2 * V + i), f(3 * V + i), alpha);
}

// the four packed field values at a site, in FP64
template <typename T>
__device__ __forceinline__ void field_at(const vec2<T> *__restrict__ F, long long V, long long i, cx<double> (&f)[4]) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const cx<T> z = ld<T>(F + k * V + i);
    f[k] = mk<double>((double)z.re, (double)z.im);
  }
}
// columns 0 and 1 of the two probe matrices of one site
__device__ __forceinline__ void probe_cols(const cx<double> (&f)[4], cx<double> (&c)[2][6], double) {
  ProbeSite s;
  s.set(f[0], f[1], f[2], f[3]);
  s.cols(0.15, c[0]);
  s.cols(0.30, c[1]);
}
__device__ __forceinline__ void probe_cols(const cx<double> (&f)[4], cx<double> (&c)[2][6], float) {
#pragma unroll
  for (int pr = 0; pr < 2; pr++) {
    const su3<double> m = gauge_cols01<double>(f[0], f[1], f[2], f[3], pr == 0 ? 0.15 : 0.30);
    c[pr][0] = m.e[0], c[pr][1] = m.e[3], c[pr][2] = m.e[6];
    c[pr][3] = m.e[1], c[pr][4] = m.e[4], c[pr][5] = m.e[7];
  }
}
// site of thread t of block lb: in FP32 a block owns an 8 x 4 x 4 x 2 tile
__device__ __forceinline__ long long probe_site(const Geo &g, unsigned lb, unsigned t, double) {
  return (long long)lb * kBlock + t;
}
__device__ __forceinline__ long long probe_site(const Geo &g, unsigned lb, unsigned t, float) {
  const unsigned nx = (unsigned)g.L[0] / 8, ny = (unsigned)g.L[1] / 4, nz = (unsigned)g.L[2] / 4;
  const unsigned by = lb / nx, bz = by / ny, bt = bz / nz;
  const long long x = (lb - by * nx) * 8 + (t & 7u), y = (by - bz * ny) * 4 + (t >> 3 & 3u);
  const long long z = (bz - bt * nz) * 4 + (t >> 5 & 3u), tt = bt * 2 + (t >> 7);
  return x + g.S[1] * y + g.S[2] * z + g.S[3] * tt;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_line_search(const vec2<T> *__restrict__ U, const vec2<T> *__restrict__ F,
                                                       double *__restrict__ part, Geo g,
                                                       const Ctrl *__restrict__ ctrl, int force) {
  if (ctrl->done) return;
  if (!force && !(ctrl->theta > ctrl->cg_tol)) return;
  const long long V = g.V;
  const unsigned lb = logical_block(g);
  const long long i = probe_site(g, lb, threadIdx.x, T(0));
  double v[3] = {0.0, 0.0, 0.0};
  if (i < V) {
    int x[4];
    coords(g, i, x);
    cx<double> A[2][6];
    {
      cx<double> f[4];
      field_at<T>(F, V, i, f);
      probe_cols(f, A, T(0));
    }
#pragma unroll 1
    for (int mu = 0; mu < kND; mu++) {
      cx<double> u[6], f[4], B[2][6];
      load_cols<T>(U, mu, i, V, u);
      field_at<T>(F, V, nb_fwd(g, i, x, mu), f);
      // Re tr u, its third diagonal entry conj(U00 U11 - U10 U01)
      v[0] += u[0].re + u[4].re + (u[0].re * u[4].re - u[0].im * u[4].im) -
              (u[1].re * u[3].re - u[1].im * u[3].im);
      probe_cols(f, B, T(0));
#pragma unroll
      for (int pr = 0; pr < 2; pr++) {
        cx<double> a2[3], M[6];
        third_col(A[pr], a2);
        mul_cols01(A[pr], a2, u, M);
        v[1 + pr] += retrace_cols(M, B[pr]);
      }
    }
  }
  block_sum_store<3>(v, part + 3 * lb);
}

// FP32 links of a shape the tiles do not divide, or where the autotuner finds
// this form the faster one: one probe at a time, the traces from the rows of
// A u (again for the rounding of the step).  On a thermalised 32^3x64 it takes
// 186 us in contiguous order, the tiles 197; untuned contexts keep the tiles,
// whose rounding their trajectories follow
__device__ __forceinline__ su3<double> promote(const su3<float> &m) {
  su3<double> d;
#pragma unroll
  for (int k = 0; k < 9; k++) d.e[k] = mk<double>((double)m.e[k].re, (double)m.e[k].im);
  return d;
}
__global__ __launch_bounds__(kBlock) void k_line_search_rows(const float2 *__restrict__ U, const float2 *__restrict__ F,
                                                       double *__restrict__ part, Geo g,
                                                       const Ctrl *__restrict__ ctrl, int force) {
  if (ctrl->done) return;
  if (!force && !(ctrl->theta > ctrl->cg_tol)) return;
  const long long V = g.V;
  const unsigned lb = logical_block(g);
  const long long i = (long long)lb * blockDim.x + threadIdx.x;
  double v[3] = {0.0, 0.0, 0.0};
  if (i < V) {
    int x[4];
    coords(g, i, x);
    // one probe at a time keeps a single probe matrix per site live (the
    // link loads of the second probe hit the caches)
#pragma unroll 1
    for (int pr = 1; pr <= 2; pr++) {
      const double al = pr == 1 ? 0.15 : 0.30;
      const su3<double> A = gauge_at64<float>(F, V, i, al);
      double acc = 0.0;
#pragma unroll 1
      for (int mu = 0; mu < kND; mu++) {
        // rows 0, 1 of A u first: the link is dead while the neighbour's
        // matrix is built, which keeps the register peak lower
        cx<double> au[6];
        {
          const su3<double> u = promote(load_link<float>(U, mu, i, V));
          if (pr == 1) v[0] += u.e[0].re + u.e[4].re + u.e[8].re;
          ab_rows01<double>(A, u, au);
        }
        acc += retrace_rows01_dag<double>(au, gauge_at64<float>(F, V, nb_fwd(g, i, x, mu), al));
      }
      v[pr] = acc;
    }
  }
  block_sum_store<3>(v, part + 3 * lb);
}

// The probes of a small lattice: one wave per direction of 64 sites, so that
// a lattice of fewer sites than the GPU has lanes runs four times the waves,
// each a quarter of the chain.  The sites of a block of k_line_search (or
// k_line_search_rows) are four workgroups here, whose three sums stay
// separate in part; the terms and the order of their addition are the same.
// 8^4: 4.3 us, 9.0 with one thread per site.
enum { PROBE_COLS = 0, PROBE_ROWS = 1 };
template <typename T, int KIND>
__global__ __launch_bounds__(kBlock) void k_line_search_small(const vec2<T> *__restrict__ U,
                                                             const vec2<T> *__restrict__ F, double *__restrict__ part,
                                                             Geo g, const Ctrl *__restrict__ ctrl, int force) {
  if (ctrl->done) return;
  if (!force && !(ctrl->theta > ctrl->cg_tol)) return;
  __shared__ double sh[3][4][kWave];
  const long long V = g.V;
  const unsigned lb = blockIdx.x >> 2, w = blockIdx.x & 3u;
  const int lane = threadIdx.x % kWave, mu = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const long long i = KIND == PROBE_ROWS ? (long long)lb * kBlock + w * kWave + lane
                                         : probe_site(g, lb, w * kWave + lane, T(0));
  double v[3] = {0.0, 0.0, 0.0};
  if (i < V) {
    int x[4];
    coords(g, i, x);
    if constexpr (KIND == PROBE_ROWS) {
      // the loops of k_line_search_rows, one direction long: which product
      // of a sum is fused depends on what shares a basic block with it, and
      // the FP32 schedule keeps that kernel's rounding
      int end = mu + 1;
      asm("" : "+s"(end));
#pragma unroll 1
      for (int pr = 1; pr <= 2; pr++) {
        const double al = pr == 1 ? 0.15 : 0.30;
        const su3<double> A = gauge_at64<T>(F, V, i, al);
        double acc = 0.0;
#pragma unroll 1
        for (int d = mu; d < end; d++) {
          cx<double> au[6];
          {
            const su3<double> u = promote(load_link<float>(U, d, i, V));
            if (pr == 1) v[0] += u.e[0].re + u.e[4].re + u.e[8].re;
            ab_rows01<double>(A, u, au);
          }
          acc += retrace_rows01_dag<double>(au, gauge_at64<T>(F, V, nb_fwd(g, i, x, d), al));
        }
        v[pr] = acc;
      }
    } else {
      cx<double> f[4], u[6], A[2][6], B[2][6];
      field_at<T>(F, V, i, f);
      probe_cols(f, A, T(0));
      load_cols<T>(U, mu, i, V, u);
      field_at<T>(F, V, nb_fwd(g, i, x, mu), f);
      v[0] = u[0].re + u[4].re + (u[0].re * u[4].re - u[0].im * u[4].im) - (u[1].re * u[3].re - u[1].im * u[3].im);
      probe_cols(f, B, T(0));
#pragma unroll
      for (int pr = 0; pr < 2; pr++) {
        cx<double> a2[3], M[6];
        third_col(A[pr], a2);
        mul_cols01(A[pr], a2, u, M);
        v[1 + pr] = retrace_cols(M, B[pr]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 3; k++) sh[k][mu][lane] = v[k];
  __syncthreads();
  if (mu < 3) {  // wave k adds sum k: the directions in order, then the sites
    double s = 0.0;
    for (int d = 0; d < 4; d++) s += sh[mu][d][lane];
    s = wave_sum(s);
    if (lane == 0) part[3 * (long long)blockIdx.x + mu] = s;
  }
}

// ---------------------------------------------------------------------------
// U_mu(x) <- g(x) U_mu(x) g(x+mu)^dagger: Gfix/line_search.c:60-97.
// With G != null the site transform is also accumulated in FP64,
// G(x) <- g(x) G(x) with g rebuilt in FP64 from the same field values: the
// mixed schedule keeps the FP64 links untouched during the FP32 phase and
// replays G on them exactly at the switch.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_egauge(vec2<T> *__restrict__ U, const vec2<T> *__restrict__ F,
                                                  double2 *__restrict__ G, Geo g, const Ctrl *__restrict__ ctrl,
                                                  int fixed_step) {
  if (ctrl->done) return;
  const long long V = g.V;
  const long long i = (long long)logical_block(g) * blockDim.x + threadIdx.x;
  if (i >= V) return;
  const double alpha = fixed_step ? ctrl->gf_alpha : ctrl->alpha;
  int x[4];
  coords(g, i, x);
  const su3<T> A = gauge_at<T>(F, V, i, (T)alpha);
#pragma unroll
  for (int mu = 0; mu < kND; mu++) {
    const su3<T> B = gauge_at<T>(F, V, nb_fwd(g, i, x, mu), (T)alpha);
    const su3<T> u = load_link<T>(U, mu, i, V);
    su3<T> n = gtransform<T>(A, u, B);
    // FP32 links are kept on SU(3): unchecked, FP32 rounding of the columns
    // feeds back through the completed third column over hundreds of updates
    if (sizeof(T) == 4) gram_reunit<T>(n);
    store_link<T>(U, mu, i, V, n);
  }
  if (G) {
    const su3<double> A64 = gauge_at64<T>(F, V, i, alpha);
    store_link<double>(G, 0, i, V, mul_cols<double>(A64, load_link<double>(G, 0, i, V)));
  }
}

// the step of an iteration from its probe sums: parabola vertex
// (Gfix/line_search.c:274-341), or GF_TUNE below CG_TOL
__device__ __forceinline__ bool ls_runs(const Ctrl *ctrl, int force) { return force || (ctrl->theta > ctrl->cg_tol); }
struct LsStep {
  double alpha, probe[3];
  int uphill;
};
__device__ __forceinline__ LsStep ls_step(const Ctrl *ctrl, const double (&s)[3], bool do_ls, int force, double pl1,
                                          double pl2) {
  LsStep r{ctrl->gf_alpha, {0.0, 0.0, 0.0}, 0};
  if (!do_ls) return r;
  double val[3];
  for (int k = 0; k < 3; k++) {
    const double tot = s[k] + (ctrl->sd_start ? ctrl->stale_probe[k] : 0.0);
    r.probe[k] = tot;
    val[k] = -tot;
  }
  const double al[3] = {0.0, pl1, pl2};
  r.alpha = approx_minimum(al, val);
  // mixed FP32 phase: the functional rises along the direction
  const int sg = ctrl->switch_theta > 0.0 && !force ? ctrl->sg_mode : 0;
  r.uphill = sg && val[1] > val[0];
  if ((sg & 4) && r.uphill) r.alpha = 0.0;
  return r;
}
__device__ __forceinline__ void ls_record(Ctrl *ctrl, const LsStep &r, bool do_ls, int force) {
  ctrl->upd++;  // the gauge update that follows will run
  if (do_ls)
    for (int k = 0; k < 3; k++) ctrl->probe[k] = r.probe[k];
  ctrl->alpha = r.alpha;
  ctrl->did_ls = do_ls;
  ctrl->sg_uphill = r.uphill;  // the forced search of an SD start clears it
  if (force) return;
  ctrl->inold = ctrl->insum;  // beta has been taken
}

// ---------------------------------------------------------------------------
// The gauge update of one CG iteration fused with the derivative of the
// next (Gfix/FACG.c:325-334 followed by :276-280).  The update is out of
// place, Uin -> Uout: each site also forms its backward links
// U'_mu(x - mu) = g(x - mu) U_mu(x - mu) g(x)^dag from the old links, with
// the arithmetic of the site that stores them, and the old links of the
// neighbours must stay readable meanwhile.  The derivative of the updated
// links then costs no second pass over them.  D is the search direction;
// Fout (the buffer of in_old, which this iteration no longer needs)
// receives the packed derivative and part its theta partials; the host
// then swaps the link buffers and the field buffers Fin <-> Fout.  Past
// convergence the launch does nothing: the control block counts the
// updates that ran (Ctrl::upd), and the host undoes the swaps of those
// that did not once the batch has ended.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kBlock) void k_egauge_deriv(const vec2<T> *__restrict__ Uin, vec2<T> *__restrict__ Uout,
                                                        const vec2<T> *__restrict__ D, double2 *__restrict__ G,
                                                        vec2<T> *__restrict__ Fin, vec2<T> *__restrict__ Fout,
                                                        double *__restrict__ part, Geo g, const Ctrl *__restrict__ ctrl) {
  if (ctrl->done) return;
  const long long V = g.V;
  const unsigned lb = logical_block(g);
  const long long i = (long long)lb * blockDim.x + threadIdx.x;
  double loc[1] = {0.0};
  if (i < V) {
    const double alpha = ctrl->alpha;
    int x[4];
    coords(g, i, x);
    const su3<T> A = gauge_at<T>(D, V, i, (T)alpha);
    DerivAcc<T> d;
#pragma unroll 1
    for (int mu = 0; mu < kND; mu++) {
      const su3<T> B = gauge_at<T>(D, V, nb_fwd(g, i, x, mu), (T)alpha);
      su3<T> n = gtransform<T>(A, load_link<T>(Uin, mu, i, V), B);
      if (sizeof(T) == 4) gram_reunit<T>(n);
      store_link<T>(Uout, mu, i, V, n);
      const long long xb = nb_bwd(g, i, x, mu);
      const su3<T> C = gauge_at<T>(D, V, xb, (T)alpha);
      su3<T> sb = gtransform<T>(C, load_link<T>(Uin, mu, xb, V), A);
      if (sizeof(T) == 4) gram_reunit<T>(sb);
      d.add(n, sb);
    }
    loc[0] = d.store(Fout, V, i);
    if (G) {
      const su3<double> A64 = gauge_at64<T>(D, V, i, alpha);
      store_link<double>(G, 0, i, V, mul_cols<double>(A64, load_link<double>(G, 0, i, V)));
    }
  }
  block_sum_store<1>(loc, part + lb);
}

// k_egauge_deriv on a small lattice: one wave per direction of 64 sites (see
// k_line_search_small), each thread one link, its backward link and their
// terms of the divergence, which wave 0 adds in the order of DerivAcc.  nb >
// 0: the step comes from the probe partials probe[12 nb] of the line search.
// 8^4: 7.4 us, 12 with one thread per site.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_egauge_deriv_small(const vec2<T> *__restrict__ Uin,
                                                              vec2<T> *__restrict__ Uout,
                                                              const vec2<T> *__restrict__ D, double2 *__restrict__ G,
                                                              vec2<T> *__restrict__ Fout, double *__restrict__ part,
                                                              Geo g, Ctrl *ctrl, const double *__restrict__ probe,
                                                              long long nb) {
  if (ctrl->done) return;
  __shared__ T sh[10][4][kWave];
  double alpha;
  if (nb > 0) {
    const bool do_ls = ls_runs(ctrl, 0);
    double s[3] = {0.0, 0.0, 0.0};
    if (do_ls) small_sum<3>(probe, nb, 4, s);
    const LsStep r = ls_step(ctrl, s, do_ls, 0, 0.15, 0.30);
    alpha = r.alpha;
    if (blockIdx.x == 0 && threadIdx.x == 0) ls_record(ctrl, r, do_ls, 0);
  } else {
    alpha = ctrl->alpha;
  }
  const long long V = g.V;
  const int lane = threadIdx.x % kWave, mu = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const long long i = (long long)blockIdx.x * kWave + lane;
  if (i < V) {
    int x[4];
    coords(g, i, x);
    const su3<T> A = gauge_at<T>(D, V, i, (T)alpha);
    const su3<T> B = gauge_at<T>(D, V, nb_fwd(g, i, x, mu), (T)alpha);
    su3<T> n = gtransform<T>(A, load_link<T>(Uin, mu, i, V), B);
    if (sizeof(T) == 4) gram_reunit<T>(n);
    store_link<T>(Uout, mu, i, V, n);
    const long long xb = nb_bwd(g, i, x, mu);
    const su3<T> C = gauge_at<T>(D, V, xb, (T)alpha);
    su3<T> sb = gtransform<T>(C, load_link<T>(Uin, mu, xb, V), A);
    if (sizeof(T) == 4) gram_reunit<T>(sb);
    const DerivTerms<T> t(n, sb);
#pragma unroll
    for (int k = 0; k < 10; k++) sh[k][mu][lane] = t.v[k];
    if (G && mu == 3) {
      const su3<double> A64 = gauge_at64<T>(D, V, i, alpha);
      store_link<double>(G, 0, i, V, mul_cols<double>(A64, load_link<double>(G, 0, i, V)));
    }
  }
  __syncthreads();
  if (mu == 0) {
    double s = 0.0;
    if (i < V) s = deriv_sum<T>([&](int m, int k) { return sh[k][m][lane]; }).store(Fout, V, i);
    s = wave_sum(s);
    if (lane == 0) part[blockIdx.x] = s;
  }
}

// ---------------------------------------------------------------------------
// single-block finalisers (fixed summation order)
// ---------------------------------------------------------------------------
// sub = 4: a row is kept as the 4 sums of its block's waves
template <int NV>
__device__ __forceinline__ void final_sum(const double *__restrict__ part, long long nb, double (&out)[NV],
                                          int sub = 1) {
  __shared__ double sh[NV][1024 / kWave];
  double v[NV];
#pragma unroll
  for (int k = 0; k < NV; k++) v[k] = 0.0;
  for (long long b = threadIdx.x; b < nb; b += blockDim.x)
#pragma unroll
    for (int k = 0; k < NV; k++) {
      double r = 0.0;
      if (sub == 1)
        r = part[b * NV + k];
      else
        for (int j = 0; j < 4; j++) r += part[(b * 4 + j) * NV + k];
      v[k] += r;
    }
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
    for (int j = 0; j < (int)(blockDim.x / kWave); j++) s += sh[k][j];
    out[k] = s;
  }
}

// theta = sum / (NC V): GFNORM_LANDAU, Headers/GLU_definitions.h:427
__global__ void k_fin_theta(const double *__restrict__ part, long long nb, Ctrl *ctrl, double norm, int sub) {
  if (ctrl->done) return;
  double s[1];
  final_sum<1>(part, nb, s, sub);
  if (threadIdx.x == 0) {
    double th = s[0] * norm;
    if (ctrl->sd_start) th += ctrl->stale_theta;  // GLU's stale red[5] slots
    ctrl->theta = th;
  }
}

__global__ void k_fin_pr(const double *__restrict__ part, long long nb, Ctrl *ctrl) {
  if (ctrl->done) return;
  double s[2];
  final_sum<2>(part, nb, s);
  if (threadIdx.x == 0) pr_record(ctrl, s[0], s[1], pr_beta(ctrl, s[0], s[1]));
}

// end of the SD start: inold = sum_DER3 (+ GLU's stale red[3] slots)
__global__ void k_fin_sd(const double *__restrict__ part, long long nb, Ctrl *ctrl) {
  if (ctrl->done) return;
  double s[2];
  final_sum<2>(part, nb, s);
  if (threadIdx.x == 0) {
    ctrl->inold = s[0] + ctrl->stale_insum;
    ctrl->beta = 0.0;
    if (ctrl->trace_n < ctrl->trace_cap) ctrl->trace_n++;  // row already written
    ctrl->sd_start = 0;
    ctrl->stale_insum = 0.0;
    ctrl->stale_theta = 0.0;
    ctrl->stale_probe[0] = ctrl->stale_probe[1] = ctrl->stale_probe[2] = 0.0;
  }
}

__global__ void k_fin_ls(const double *__restrict__ part, long long nb, Ctrl *ctrl, double *trace, int force,
                         double pl1, double pl2, int sub) {
  if (ctrl->done) return;
  const bool do_ls = ls_runs(ctrl, force);
  double s[3] = {0.0, 0.0, 0.0};
  if (do_ls) final_sum<3>(part, nb, s, sub);
  if (threadIdx.x == 0) {
    ls_record(ctrl, ls_step(ctrl, s, do_ls, force, pl1, pl2), do_ls, force);
    if (ctrl->sd_start && trace && ctrl->trace_n < ctrl->trace_cap) {
      double *r = trace + 3 * ctrl->trace_n;
      r[0] = ctrl->theta;
      r[1] = ctrl->alpha;
      r[2] = 0.0;
    }
  }
}

// end of a loop iteration: count, record, stop test (Gfix/FACG.c:331-334);
// returns the done flag
__device__ int iter_end_body(Ctrl *ctrl, double *trace, int fasd) {
  if (fasd) {
    ctrl->alpha = ctrl->gf_alpha;
    ctrl->beta = 0.0;
  }
  const double theta = ctrl->theta;
  const long long iters = ctrl->iters + 1;
  ctrl->iters = iters;
  ctrl->total++;
  if (trace && ctrl->trace_n < ctrl->trace_cap) {
    double *r = trace + 3 * ctrl->trace_n;
    r[0] = theta;
    r[1] = ctrl->alpha;
    r[2] = ctrl->beta;
    ctrl->trace_n++;
  }
  ctrl->stale_insum = ctrl->insum;
  ctrl->stale_theta = theta;
  for (int k = 0; k < 3; k++) ctrl->stale_probe[k] = ctrl->did_ls ? ctrl->probe[k] : 0.0;
  int done = !(theta > ctrl->acc && iters < ctrl->max_iters);
  if (ctrl->switch_theta > 0.0) {  // mixed FP32 phase: the switch to FP64
    const double tmin = ctrl->theta_min;
    if (theta < tmin) ctrl->theta_min = theta;
    const bool stalled = ctrl->stall_factor > 0.0 && tmin < ctrl->stall_theta && theta > ctrl->stall_factor * tmin;
    if (theta < ctrl->switch_theta || stalled) {
      ctrl->switched = stalled && !(theta < ctrl->switch_theta) ? 2 : 1;
      done = 1;
    }
  }
  ctrl->done = done;
  return done;
}

__global__ void k_iter_end(Ctrl *ctrl, double *trace, int fasd) {
  if (ctrl->done) return;
  iter_end_body(ctrl, trace, fasd);
}

// The end of a CG iteration and the theta of the next one in one launch:
// the stop test on theta_k, then, unless it stopped, theta_k+1 from the
// partials of the fused update + derivative (as k_fin_theta; the SD start
// is over, so no stale slots enter).  A stopped run keeps the theta it
// tested, and the derivative it left is taken again if a segment resumes.
__global__ void k_fin_iter(const double *__restrict__ part, long long nb, Ctrl *ctrl, double *trace, double norm,
                           int sub) {
  if (ctrl->done) return;
  double s[1];
  final_sum<1>(part, nb, s, sub);
  if (threadIdx.x == 0 && !iter_end_body(ctrl, trace, 0)) ctrl->theta = s[0] * norm;
}

// plain sum of nb partials into *out (fixed order)
__global__ void k_sum_part(const double *__restrict__ part, long long nb, double *out) {
  double s[1];
  final_sum<1>(part, nb, s);
  if (threadIdx.x == 0) *out = s[0];
}

__global__ void k_begin_segment(Ctrl *ctrl, int sd) {
  ctrl->done = 0;
  ctrl->iters = 0;
  ctrl->sd_start = sd;
  ctrl->did_ls = 0;
}

// ---------------------------------------------------------------------------
// layout conversion: GLU AoS double[V][4][18] <-> device column planes
// ---------------------------------------------------------------------------
// A workgroup moves 64 sites through LDS, one wave per direction: the
// sites' 36 KB of GLU's layout are read or written as one contiguous run and
// each plane as runs of 1 KB.  A site takes 37 complex numbers in LDS (36
// used), so that the lanes of a wave, one site each, spread over the banks.
// Bound by memory, 960 B a site: on 32^3x64 unpacking took 837 us with one
// thread writing a site's 576 B by itself (2.4 TB/s), packing 452; now about
// 390 each, a copy's rate.
constexpr int kPackSites = 64;
constexpr int kPackLds = 37;
// the caller's links are doubles: 8-byte aligned
struct GluCx {
  double re, im;
};
__global__ __launch_bounds__(kBlock) void k_pack(const GluCx *__restrict__ aos, double2 *__restrict__ U,
                                                long long V, long long site0, long long nsite) {
  __shared__ double2 sh[kPackSites * kPackLds];
  const long long s0 = (long long)blockIdx.x * kPackSites;
  const int n = (int)(nsite - s0 < kPackSites ? nsite - s0 : kPackSites);
  const GluCx *src = aos + s0 * 36;
  // all loads in flight before the first is stored; past the end the last
  // number is stored again
  GluCx v[9];
#pragma unroll
  for (int k = 0; k < 9; k++) v[k] = src[min((int)threadIdx.x + k * kBlock, n * 36 - 1)];
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const int e = min((int)threadIdx.x + k * kBlock, n * 36 - 1);
    sh[e / 36 * kPackLds + e % 36] = make_double2(v[k].re, v[k].im);
  }
  __syncthreads();
  const int s = threadIdx.x % kPackSites, mu = threadIdx.x / kPackSites;
  if (s >= n) return;
  su3<double> m;
#pragma unroll
  for (int k = 0; k < 9; k++)
    if (k % 3 < 2) m.e[k] = ld<double>(sh + s * kPackLds + mu * 9 + k);
  store_link<double>(U, mu, site0 + s0 + s, V, m);
}

__global__ __launch_bounds__(kBlock) void k_unpack(const double2 *__restrict__ U, GluCx *__restrict__ aos,
                                                  long long V, long long site0, long long nsite) {
  __shared__ double2 sh[kPackSites * kPackLds];
  const long long s0 = (long long)blockIdx.x * kPackSites;
  const int n = (int)(nsite - s0 < kPackSites ? nsite - s0 : kPackSites);
  const int s = threadIdx.x % kPackSites, mu = threadIdx.x / kPackSites;
  if (s < n) {
    const su3<double> m = load_link<double>(U, mu, site0 + s0 + s, V);
#pragma unroll
    for (int k = 0; k < 9; k++) st<double>(sh + s * kPackLds + mu * 9 + k, m.e[k]);
  }
  __syncthreads();
  GluCx *dst = aos + s0 * 36;
#pragma unroll
  for (int k = 0; k < 9; k++) {
    const int e = threadIdx.x + k * kBlock, t = e / 36;
    const double2 v = sh[t * kPackLds + e % 36];
    if (t < n) dst[e] = GluCx{v.x, v.y};
  }
}

// FP64 links -> FP32 copy
__global__ __launch_bounds__(kBlock) void k_demote(const double2 *__restrict__ U, float2 *__restrict__ W, long long n) {
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (long long)gridDim.x * blockDim.x) {
    const double2 v = U[j];
    W[j] = make_float2((float)v.x, (float)v.y);
  }
}

// identity site transform (column planes of one "direction")
template <typename T>
__global__ __launch_bounds__(kBlock) void k_identity(vec2<T> *__restrict__ G, long long V) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  su3<T> m;
#pragma unroll
  for (int k = 0; k < 9; k++) m.e[k] = mk<T>(T(0), T(0));
  m.e[0].re = m.e[4].re = m.e[8].re = T(1);
  store_link<T>(G, 0, i, V, m);
}

// U_mu(x) <- G(x) U_mu(x) G(x+mu)^dagger in FP64 with the accumulated site
// transform reunitarised first (Gfix/gtrans.c:169-189)
__global__ __launch_bounds__(kBlock) void k_apply_gauge(double2 *__restrict__ U, const double2 *__restrict__ G,
                                                       Geo g) {
  const long long V = g.V;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  int x[4];
  coords(g, i, x);
  auto fetch = [&](long long s) {
    su3<double> d = load_link<double>(G, 0, s, V);
    gram_reunit<double>(d);
    return d;
  };
  const su3<double> A = fetch(i);
#pragma unroll
  for (int mu = 0; mu < kND; mu++) {
    const su3<double> B = fetch(nb_fwd(g, i, x, mu));
    const su3<double> u = load_link<double>(U, mu, i, V);
    store_link<double>(U, mu, i, V, gtransform<double>(A, u, B));
  }
}

// packed fields FP32 -> FP64 (the CG state crosses the precision switch)
__global__ __launch_bounds__(kBlock) void k_promote(const float2 *__restrict__ a, double2 *__restrict__ b, long long n) {
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (long long)gridDim.x * blockDim.x) {
    const float2 v = a[j];
    b[j] = make_double2(v.x, v.y);
  }
}

// reunitarise every link (Geometry/random_config.c:43-56)
__global__ __launch_bounds__(kBlock) void k_reunit(double2 *__restrict__ U, long long V, int nd) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  for (int mu = 0; mu < nd; mu++) {
    su3<double> m = load_link<double>(U, mu, i, V);
    gram_reunit<double>(m);
    store_link<double>(U, mu, i, V, m);
  }
}

// plaquette / link-trace partial sums: Field/plaqs_links.c:243-265, 399-448.
// Bound by the cache traffic of the neighbour links (1536 B a site, 384 of
// them from HBM): 438 us on 32^3x64, 124 on 24^3x48.  Products whose third
// columns or rows are completed would take 378 and 119, but are off by 1e-7
// a loop on links rounded to single precision
__global__ __launch_bounds__(kBlock) void k_measure(const double2 *__restrict__ U, double *__restrict__ part, Geo g) {
  const long long V = g.V;
  const unsigned lb = logical_block(g);
  const long long i = (long long)lb * blockDim.x + threadIdx.x;
  double v[3] = {0.0, 0.0, 0.0};  // plaquette sum, link trace, temporal trace
  double mx = -1e300;             // largest single-link trace
  if (i < V) {
    int x[4];
    coords(g, i, x);
    su3<double> u[4];
#pragma unroll
    for (int mu = 0; mu < 4; mu++) {
      u[mu] = load_link<double>(U, mu, i, V);
      const double r = retrace<double>(u[mu]);
      v[1] += r;
      if (mu == 3) v[2] += r;
      mx = r > mx ? r : mx;
    }
    const long long nb[4] = {nb_fwd(g, i, x, 0), nb_fwd(g, i, x, 1), nb_fwd(g, i, x, 2), nb_fwd(g, i, x, 3)};
#pragma unroll
    for (int mu = 1; mu < 4; mu++) {
      const long long t = nb[mu];
#pragma unroll
      for (int nu = 0; nu < mu; nu++)
        // Re tr(U_mu(x) U_nu(x+mu) U_mu(x+nu)^dag U_nu(x)^dag)
        v[0] += retrace_ab_cd_dag<double>(u[mu], load_link<double>(U, nu, t, V), u[nu],
                                          load_link<double>(U, mu, nb[nu], V));
    }
  }
  __shared__ double mxs[kBlock / kWave];
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) mx = fmax(mx, __shfl_down(mx, o, kWave));
  if (threadIdx.x % kWave == 0) mxs[threadIdx.x / kWave] = mx;
  block_sum_store<3>(v, part + 4 * lb);  // its barrier covers mxs
  if (threadIdx.x == 0) part[4 * lb + 3] = fmax(fmax(mxs[0], mxs[1]), fmax(mxs[2], mxs[3]));
}

// the sums and the maximum of nb rows of 4 partials (fixed order)
__global__ void k_fin_measure(const double *__restrict__ part, long long nb, double *out) {
  __shared__ double sh[4][1024 / kWave];
  double v[4] = {0.0, 0.0, 0.0, -1e300};
  for (long long b = threadIdx.x; b < nb; b += blockDim.x) {
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] += part[4 * b + k];
    v[3] = fmax(v[3], part[4 * b + 3]);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
#pragma unroll
    for (int k = 0; k < 3; k++) v[k] += __shfl_down(v[k], o, kWave);
    v[3] = fmax(v[3], __shfl_down(v[3], o, kWave));
  }
  if (threadIdx.x % kWave == 0)
    for (int k = 0; k < 4; k++) sh[k][threadIdx.x / kWave] = v[k];
  __syncthreads();
  if (threadIdx.x < 4) {
    double r = sh[threadIdx.x][0];
    for (int w = 1; w < 1024 / kWave; w++) r = threadIdx.x < 3 ? r + sh[threadIdx.x][w] : fmax(r, sh[threadIdx.x][w]);
    out[threadIdx.x] = r;
  }
}

// ---------------------------------------------------------------------------
// explicit instantiations + launch helpers
// ---------------------------------------------------------------------------
static inline unsigned nblk(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

template <typename T>
void launch_deriv(const void *U, void *F, double *part, const Geo &g, const Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_deriv<T>, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const vec2<T> *)U, (vec2<T> *)F, part, g,
                     ctrl);
}
template <typename T>
void launch_pr_sums(const void *F, const void *O, double *part, long long V, const Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_pr_sums<T>, dim3(nblk(V)), dim3(kBlock), 0, s, (const vec2<T> *)F, (const vec2<T> *)O, part,
                     V, ctrl);
}
template <typename T>
void launch_cg_update(const void *F, void *sn, long long V, Ctrl *ctrl, hipStream_t s, const double *part,
                      long long nb) {
  const long long n4 = 4 * V;
  const unsigned b = (unsigned)std::min<long long>(nblk(n4), 8192);
  hipLaunchKernelGGL(k_cg_update<T>, dim3(b), dim3(kBlock), 0, s, (const vec2<T> *)F, (vec2<T> *)sn, n4, ctrl, part,
                     nb);
}
template <typename T> void launch_copy(const void *F, void *a, long long V, const Ctrl *ctrl, hipStream_t s) {
  const long long n4 = 4 * V;
  const unsigned b = (unsigned)std::min<long long>(nblk(n4), 8192);
  hipLaunchKernelGGL(k_copy<T>, dim3(b), dim3(kBlock), 0, s, (const vec2<T> *)F, (vec2<T> *)a, n4, ctrl);
}
bool line_search_tiles(const Geo &g) { return !(g.L[0] % 8 || g.L[1] % 4 || g.L[2] % 4 || g.L[3] % 2); }
template <typename T>
void launch_line_search(const void *U, const void *F, double *part, const Geo &g, const Ctrl *ctrl, int force,
                        hipStream_t s, int rows) {
  if constexpr (sizeof(T) == 4) {
    Geo gt = g;
    if (rows || !line_search_tiles(g)) {
      hipLaunchKernelGGL(k_line_search_rows, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const float2 *)U,
                         (const float2 *)F, part, g, ctrl, force);
      return;
    }
    gt.xcd = g.xcd ? 1 : 0;  // tiles are numbered x fastest: plain or XCD-contiguous
    hipLaunchKernelGGL(k_line_search<T>, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const vec2<T> *)U,
                       (const vec2<T> *)F, part, gt, ctrl, force);
  } else {
    hipLaunchKernelGGL(k_line_search<T>, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const vec2<T> *)U,
                       (const vec2<T> *)F, part, g, ctrl, force);
  }
}
bool small_lattice(const Geo &g) { return nblk(g.V) <= kSmallBlocks; }
template <typename T>
void launch_line_search_small(const void *U, const void *F, double *part, const Geo &g, const Ctrl *ctrl, int force,
                              hipStream_t s, int rows) {
  const dim3 grid(4 * nblk(g.V)), blk(kBlock);
  if constexpr (sizeof(T) == 4) {
    if (rows || !line_search_tiles(g)) {
      hipLaunchKernelGGL((k_line_search_small<T, PROBE_ROWS>), grid, blk, 0, s, (const vec2<T> *)U,
                         (const vec2<T> *)F, part, g, ctrl, force);
      return;
    }
  }
  hipLaunchKernelGGL((k_line_search_small<T, PROBE_COLS>), grid, blk, 0, s, (const vec2<T> *)U, (const vec2<T> *)F,
                     part, g, ctrl, force);
}
template <typename T>
void launch_egauge_deriv_small(const void *Uin, void *Uout, const void *D, void *G, void *Fout, double *part,
                               const Geo &g, Ctrl *ctrl, const double *probe, long long nb, hipStream_t s) {
  hipLaunchKernelGGL(k_egauge_deriv_small<T>, dim3(4 * nblk(g.V)), dim3(kBlock), 0, s, (const vec2<T> *)Uin,
                     (vec2<T> *)Uout, (const vec2<T> *)D, (double2 *)G, (vec2<T> *)Fout, part, g, ctrl, probe, nb);
}
template <typename T>
void launch_egauge(void *U, const void *F, void *G, const Geo &g, const Ctrl *ctrl, int fixed, hipStream_t s) {
  hipLaunchKernelGGL(k_egauge<T>, dim3(nblk(g.V)), dim3(kBlock), 0, s, (vec2<T> *)U, (const vec2<T> *)F,
                     (double2 *)G, g, ctrl, fixed);
}
template <typename T>
void launch_egauge_deriv(const void *Uin, void *Uout, const void *D, void *G, void *Fin, void *Fout, double *part,
                         const Geo &g, const Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_egauge_deriv<T>, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const vec2<T> *)Uin, (vec2<T> *)Uout,
                     (const vec2<T> *)D, (double2 *)G, (vec2<T> *)Fin, (vec2<T> *)Fout, part, g, ctrl);
}
template <typename T> void launch_identity(void *G, long long V, hipStream_t s) {
  hipLaunchKernelGGL(k_identity<T>, dim3(nblk(V)), dim3(kBlock), 0, s, (vec2<T> *)G, V);
}

#define GFIX_INST(T)                                                                                          \
  template void launch_deriv<T>(const void *, void *, double *, const Geo &, const Ctrl *, hipStream_t);      \
  template void launch_pr_sums<T>(const void *, const void *, double *, long long, const Ctrl *, hipStream_t); \
  template void launch_cg_update<T>(const void *, void *, long long, Ctrl *, hipStream_t, const double *,      \
                                    long long);                                                               \
  template void launch_line_search_small<T>(const void *, const void *, double *, const Geo &, const Ctrl *,  \
                                            int, hipStream_t, int);                                           \
  template void launch_egauge_deriv_small<T>(const void *, void *, const void *, void *, void *, double *,    \
                                             const Geo &, Ctrl *, const double *, long long, hipStream_t);    \
  template void launch_copy<T>(const void *, void *, long long, const Ctrl *, hipStream_t);                    \
  template void launch_line_search<T>(const void *, const void *, double *, const Geo &, const Ctrl *, int,   \
                                      hipStream_t, int);                                                      \
  template void launch_egauge<T>(void *, const void *, void *, const Geo &, const Ctrl *, int, hipStream_t);  \
  template void launch_egauge_deriv<T>(const void *, void *, const void *, void *, void *, void *, double *,     \
                                       const Geo &, const Ctrl *, hipStream_t);                                   \
  template void launch_identity<T>(void *, long long, hipStream_t);
GFIX_INST(double)
GFIX_INST(float)

void launch_fin_theta(const double *part, long long nb, Ctrl *ctrl, double norm, hipStream_t s, int sub) {
  hipLaunchKernelGGL(k_fin_theta, dim3(1), dim3(1024), 0, s, part, nb, ctrl, norm, sub);
}
void launch_fin_pr(const double *part, long long nb, Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_fin_pr, dim3(1), dim3(1024), 0, s, part, nb, ctrl);
}
void launch_fin_sd(const double *part, long long nb, Ctrl *ctrl, hipStream_t s) {
  hipLaunchKernelGGL(k_fin_sd, dim3(1), dim3(1024), 0, s, part, nb, ctrl);
}
void launch_fin_ls(const double *part, long long nb, Ctrl *ctrl, double *trace, int force, double pl1, double pl2,
                   hipStream_t s, int sub) {
  hipLaunchKernelGGL(k_fin_ls, dim3(1), dim3(1024), 0, s, part, nb, ctrl, trace, force, pl1, pl2, sub);
}
void launch_fin_iter(const double *part, long long nb, Ctrl *ctrl, double *trace, double norm, hipStream_t s,
                     int sub) {
  hipLaunchKernelGGL(k_fin_iter, dim3(1), dim3(1024), 0, s, part, nb, ctrl, trace, norm, sub);
}
void launch_sum_part(const double *part, long long nb, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_sum_part, dim3(1), dim3(1024), 0, s, part, nb, out);
}
void launch_iter_end(Ctrl *ctrl, double *trace, int fasd, hipStream_t s) {
  hipLaunchKernelGGL(k_iter_end, dim3(1), dim3(1), 0, s, ctrl, trace, fasd);
}
void launch_begin_segment(Ctrl *ctrl, int sd, hipStream_t s) {
  hipLaunchKernelGGL(k_begin_segment, dim3(1), dim3(1), 0, s, ctrl, sd);
}
static unsigned pack_blocks(long long n) { return (unsigned)((n + kPackSites - 1) / kPackSites); }
void launch_pack(const double *aos, void *U, long long V, long long site0, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_pack, dim3(pack_blocks(n)), dim3(kBlock), 0, s, (const GluCx *)aos, (double2 *)U, V, site0, n);
}
void launch_unpack(const void *U, double *aos, long long V, long long site0, long long n, hipStream_t s) {
  hipLaunchKernelGGL(k_unpack, dim3(pack_blocks(n)), dim3(kBlock), 0, s, (const double2 *)U, (GluCx *)aos, V, site0,
                     n);
}
void launch_demote(const void *U, void *W, long long n, hipStream_t s) {
  const unsigned b = (unsigned)std::min<long long>(nblk(n), 16384);
  hipLaunchKernelGGL(k_demote, dim3(b), dim3(kBlock), 0, s, (const double2 *)U, (float2 *)W, n);
}
void launch_apply_gauge(void *U, const void *G, const Geo &g, hipStream_t s) {
  hipLaunchKernelGGL(k_apply_gauge, dim3(nblk(g.V)), dim3(kBlock), 0, s, (double2 *)U, (const double2 *)G, g);
}
void launch_promote(const void *a, void *b, long long n, hipStream_t s) {
  const unsigned bl = (unsigned)std::min<long long>(nblk(n), 16384);
  hipLaunchKernelGGL(k_promote, dim3(bl), dim3(kBlock), 0, s, (const float2 *)a, (double2 *)b, n);
}
void launch_reunit(void *U, long long V, int nd, hipStream_t s) {
  hipLaunchKernelGGL(k_reunit, dim3(nblk(V)), dim3(kBlock), 0, s, (double2 *)U, V, nd);
}
void launch_measure(const void *U, double *part, double *out, const Geo &g, hipStream_t s) {
  hipLaunchKernelGGL(k_measure, dim3(nblk(g.V)), dim3(kBlock), 0, s, (const double2 *)U, part, g);
  if (out)
    hipLaunchKernelGGL(k_fin_measure, dim3(1), dim3(1024), 0, s, part, (long long)nblk(g.V), out);
}

}  // namespace gfix
