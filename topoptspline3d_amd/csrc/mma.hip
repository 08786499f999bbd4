// mma.hip -- method of moving asymptotes (MMA::mma_t, optimization/mma_t.h:159-266,
// mma_t.cpp:18-51, mma_t.cu:15-807), FP64.
//
// The reference evaluates every vector expression of the primal-dual Newton iteration as
// its own kernel (dozens per step) and solves the (m+1)x(m+1) reduced system on the host.
// Here each n-length sweep of a Newton step is one fused grid-stride kernel over the whole
// GPU that also produces the step's reductions as fixed-order per-block partials, which one
// wave per column folds; the host reads the few scalars that steer the iteration.  It waits
// twice per Newton step: for the sums of the reduced system and the KKT residual at the
// current point (k_mma_point), and for the residuals of the line search (k_mma_trials: the
// step bound is taken on the device and the first kTrials halvings are tried together).  With
// a wait per sweep and trial, 5.3 a step, the 40 steps of the first update of 9537 coefficients
// spent more time between kernels than in them; a TO iteration at 128x64x64 went from 12.5 to
// 10.0 ms with two.
#include "tos_internal.hpp"

namespace tos {

constexpr int MMAX = 4;       // constraints supported
constexpr int kTrials = 4;    // line-search steps tried together
// columns of the reductions: sums first, then the maxima
constexpr int kkt_cols(int m) { return 6 + m; }                   // 3 sums, m proxies, 3 maxima
constexpr int point_cols(int m) { return m * m + m + kkt_cols(m); }
constexpr int MMA_CNT = 4 + kTrials * kkt_cols(MMAX);             // widest: step bound and trials
static_assert(MMA_CNT >= point_cols(MMAX), "reduction buffer");

struct MmaVecs {
  int n, m;
  double *x, *xmin, *xmax, *L, *U, *alpha, *beta, *lastdx, *xi, *eta;
  double *p, *q;  // (m+1) x n
  double *curx, *Dx, *G, *dlx, *dx, *dxi, *deta;
};

struct MmaSmall {  // scalars passed by value
  double lam[MMAX], dlam[MMAX];
  double eps, step, move;
};

// lambda at a trial step, rounded as the host rounds it (product, then sum)
__device__ __forceinline__ double mma_lam_at(double lam, double dlam, double step) {
#pragma clang fp contract(off)
  const double d = dlam * step;
  return lam + d;
}

__device__ __forceinline__ int64_t mtid() { return (int64_t)blockIdx.x * blockDim.x + threadIdx.x; }
__device__ __forceinline__ int64_t mstride() { return (int64_t)gridDim.x * blockDim.x; }

template <int CNT>
__device__ __forceinline__ void block_partials(double (&v)[CNT], const bool (&ismax)[CNT], double* partial) {
  __shared__ double sh[4][CNT];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    double a = v[i];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const double b = __shfl_down(a, o, 64);
      a = ismax[i] ? fmax(a, b) : a + b;
    }
    if (lane == 0) sh[wid][i] = a;
  }
  __syncthreads();
  if (threadIdx.x < CNT) {
    const int i = threadIdx.x;
    const double r = ismax[i] ? fmax(fmax(sh[0][i], sh[1][i]), fmax(sh[2][i], sh[3][i]))
                              : (sh[0][i] + sh[1][i]) + (sh[2][i] + sh[3][i]);
    partial[(int64_t)i * gridDim.x + blockIdx.x] = r;
  }
}

// p_i, q_i at the current x, the constraint proxies there (for b), then the subproblem
// start point (mma_subproblem_t::init mma_t.cu:15-118 and reset :702-713).
__global__ __launch_bounds__(256) void k_mma_pq(MmaVecs V, const double* __restrict__ df,
                                                const double* __restrict__ dg, double* partial) {
  const int n = V.n, m = V.m;
  double v[MMAX] = {0, 0, 0, 0};
  const bool mx[MMAX] = {false, false, false, false};
  for (int64_t j = mtid(); j < n; j += mstride()) {
    const double x = V.x[j], ux = V.U[j] - x, xl = x - V.L[j];
    const double r = 1e-5 / (V.xmax[j] - V.xmin[j]);
    for (int i = 0; i <= m; ++i) {
      const double d = i == 0 ? df[j] : dg[(int64_t)(i - 1) * n + j];
      const double dp = fmax(d, 0.0), dm = fmax(-d, 0.0);
      const double pv = ux * ux * (1.001 * dp + 0.001 * dm + r);
      const double qv = xl * xl * (0.001 * dp + 1.001 * dm + r);
      V.p[(int64_t)i * n + j] = pv;
      V.q[(int64_t)i * n + j] = qv;
      if (i > 0) v[i - 1] += pv / ux + qv / xl;
    }
    V.curx[j] = x;
    const double xn = 0.5 * (V.alpha[j] + V.beta[j]);
    V.x[j] = xn;
    V.xi[j] = fmax(1.0 / (xn - V.alpha[j]), 1.0);
    V.eta[j] = fmax(1.0 / (V.beta[j] - xn), 1.0);
  }
  block_partials<MMAX>(v, mx, partial);
}

// The current point (moved by S.step along the Newton direction first, unless 0) with the
// multipliers S.lam: Dx, delta_x and G there, the sums of the reduced system (mma_t.cu:358-395,
// solveLinearSystem :228-328), A11 = G Dx^-1 G^T in columns 0 .. m*m - 1 and b1's part
// G (delta_x / Dx) in the next m, and the n-length parts of the KKT residual (kkt_err
// mma_t.cu:574-678) in the rest: three sums of squares, the m proxies g_i, three maxima.
template <int M>
__global__ __launch_bounds__(256) void k_mma_point(MmaVecs V, MmaSmall S, double* partial) {
  const int n = V.n;
  constexpr int C = point_cols(M), K = M * M + M;
  double v[C];
  bool mx[C];
#pragma unroll
  for (int i = 0; i < C; ++i) { v[i] = 0; mx[i] = i >= C - 3; }
  for (int64_t j = mtid(); j < n; j += mstride()) {
    double X = V.x[j], XI = V.xi[j], ETA = V.eta[j];
    if (S.step != 0) {
      X = fma(V.dx[j], S.step, X);
      XI = fma(V.dxi[j], S.step, XI);
      ETA = fma(V.deta[j], S.step, ETA);
      V.x[j] = X; V.xi[j] = XI; V.eta[j] = ETA;
    }
    double pl = V.p[j], ql = V.q[j], pi[M], qi[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      pi[i] = V.p[(int64_t)(i + 1) * n + j];
      qi[i] = V.q[(int64_t)(i + 1) * n + j];
      pl += S.lam[i] * pi[i];
      ql += S.lam[i] * qi[i];
    }
    const double ux = V.U[j] - X, xl = X - V.L[j];
    const double xa = X - V.alpha[j], bx = V.beta[j] - X;
    const double psi = 2 * pl / (ux * ux * ux) + 2 * ql / (xl * xl * xl);
    const double Dx = psi + XI / xa + ETA / bx;
    const double phi = pl / (ux * ux) - ql / (xl * xl);
    const double dlx = -(S.eps / xa - S.eps / bx - phi);
    V.Dx[j] = Dx;
    V.dlx[j] = dlx;
    double Gi[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      Gi[i] = pi[i] / (ux * ux) - qi[i] / (xl * xl);
      V.G[(int64_t)i * n + j] = Gi[i];
      v[K + 3 + i] += pi[i] / ux + qi[i] / xl;
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
#pragma unroll
      for (int k = 0; k < M; ++k) v[i * M + k] += Gi[i] * (Gi[k] / Dx);
      v[M * M + i] += Gi[i] * (dlx / Dx);
    }
    const double rx = phi - XI + ETA, r1 = XI * xa - S.eps, r2 = ETA * bx - S.eps;
    v[K] += rx * rx; v[K + 1] += r1 * r1; v[K + 2] += r2 * r2;
    v[C - 3] = fmax(v[C - 3], fabs(rx));
    v[C - 2] = fmax(v[C - 2], fabs(r1));
    v[C - 1] = fmax(v[C - 1], fabs(r2));
  }
  block_partials<C>(v, mx, partial);
}

// Newton direction in x, xi, eta and the fraction-to-boundary bounds (mma_t.cu:302-317,
// :396-402)
template <int M>
__global__ __launch_bounds__(256) void k_mma_direction(MmaVecs V, MmaSmall S, double* partial) {
  const int n = V.n;
  double t[3] = {-1e300, -1e300, -1e300};
  const bool mx[3] = {true, true, true};
  const double cf = 1.0 / 0.99;
  for (int64_t j = mtid(); j < n; j += mstride()) {
    double dxv = -V.dlx[j] / V.Dx[j];
#pragma unroll
    for (int i = 0; i < M; ++i) dxv -= S.dlam[i] * V.G[(int64_t)i * n + j] / V.Dx[j];
    const double xa = V.x[j] - V.alpha[j], bx = V.beta[j] - V.x[j];
    const double dxi = S.eps / xa - dxv / xa * V.xi[j] - V.xi[j];
    const double deta = S.eps / bx + V.eta[j] / bx * dxv - V.eta[j];
    V.dx[j] = dxv;
    V.dxi[j] = dxi;
    V.deta[j] = deta;
    t[0] = fmax(t[0], -cf * (dxv / xa));
    t[1] = fmax(t[1], cf * (dxv / bx));
    t[2] = fmax(t[2], fmax(-cf * dxi / V.xi[j], -cf * deta / V.eta[j]));
  }
  block_partials<3>(t, mx, partial);
}

// folds the three bounds of k_mma_direction into out[0 .. 2] and the step into out[3]:
// 1 / max(x bounds, max(xi and eta bound, the scalars' bound sb))
__global__ __launch_bounds__(192) void k_mma_step(const double* __restrict__ partial, int nb, double sb,
                                                  double* __restrict__ out) {
  __shared__ double sh[3];
  const int c = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double s = -HUGE_VAL;
  for (int b = lane; b < nb; b += 64) s = fmax(s, partial[(int64_t)c * nb + b]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s = fmax(s, __shfl_xor(s, o, 64));
  if (lane == 0) sh[c] = out[c] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[3] = 1.0 / fmax(fmax(sh[0], sh[1]), fmax(sh[2], sb));
}

// n-length parts of the KKT residual at x + t dx for the steps t = scale * step[0] / 2^k,
// k < kTrials: columns k * kkt_cols(M) + (three sums of squares, proxies, three maxima)
template <int M>
__global__ __launch_bounds__(256) void k_mma_trials(MmaVecs V, MmaSmall S, const double* __restrict__ step,
                                                    double scale, double* partial) {
  const int n = V.n;
  constexpr int CK = kkt_cols(M), C = kTrials * CK;
  double t[kTrials], lam[kTrials][M];
  t[0] = scale * step[0];
#pragma unroll
  for (int k = 0; k < kTrials; ++k) {
    if (k > 0) t[k] = t[k - 1] / 2;
#pragma unroll
    for (int i = 0; i < M; ++i) lam[k][i] = mma_lam_at(S.lam[i], S.dlam[i], t[k]);
  }
  double v[C];
  bool mx[C];
#pragma unroll
  for (int i = 0; i < C; ++i) { v[i] = 0; mx[i] = i % CK >= CK - 3; }
  for (int64_t j = mtid(); j < n; j += mstride()) {
    const double x0 = V.x[j], xi0 = V.xi[j], eta0 = V.eta[j], dx = V.dx[j], dxi = V.dxi[j], deta = V.deta[j];
    const double U = V.U[j], L = V.L[j], al = V.alpha[j], be = V.beta[j], p0 = V.p[j], q0 = V.q[j];
    double pi[M], qi[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      pi[i] = V.p[(int64_t)(i + 1) * n + j];
      qi[i] = V.q[(int64_t)(i + 1) * n + j];
    }
#pragma unroll
    for (int k = 0; k < kTrials; ++k) {
      const double X = fma(dx, t[k], x0), XI = fma(dxi, t[k], xi0), ETA = fma(deta, t[k], eta0);
      double pl = p0, ql = q0;
#pragma unroll
      for (int i = 0; i < M; ++i) {
        pl += lam[k][i] * pi[i];
        ql += lam[k][i] * qi[i];
      }
      const double ux = U - X, xl = X - L;
      const double rx = pl / (ux * ux) - ql / (xl * xl) - XI + ETA;
      const double r1 = XI * (X - al) - S.eps, r2 = ETA * (be - X) - S.eps;
      double* w = v + k * CK;
      w[0] += rx * rx; w[1] += r1 * r1; w[2] += r2 * r2;
#pragma unroll
      for (int i = 0; i < M; ++i) w[3 + i] += pi[i] / ux + qi[i] / xl;
      w[CK - 3] = fmax(w[CK - 3], fabs(rx));
      w[CK - 2] = fmax(w[CK - 2], fabs(r1));
      w[CK - 1] = fmax(w[CK - 1], fabs(r2));
    }
  }
  block_partials<C>(v, mx, partial);
}

// asymptotes and move limits for the next iteration (adjust_asym mma_t.cu:164-226), after the
// last accepted Newton step S.step
__global__ __launch_bounds__(256) void k_mma_asym(MmaVecs V, MmaSmall S, double* partial) {
  const int n = V.n;
  double v[1] = {0};
  const bool mx[1] = {false};
  for (int64_t j = mtid(); j < n; j += mstride()) {
    const double xv = S.step != 0 ? fma(V.dx[j], S.step, V.x[j]) : V.x[j];
    V.x[j] = xv;
    const double d1 = xv - V.curx[j], d2 = V.lastdx[j];
    double gam = 1;
    if (d1 * d2 > 0) gam = 1.2;
    if (d1 * d2 < 0) gam = 0.7;
    const double st = V.xmax[j] - V.xmin[j];
    double al = xv - gam * (xv - d1 - V.L[j]);
    double au = xv + gam * (V.U[j] - xv + d1);
    al = fmin(fmax(al, xv - 10 * st), xv - 0.01 * st);
    au = fmin(fmax(au, xv + 0.01 * st), xv + 10 * st);
    V.L[j] = al;
    V.U[j] = au;
    double na = V.xmin[j];
    na = fmax(na, al + 0.1 * (xv - al));
    na = fmax(na, xv - S.move * st);
    double nb = V.xmax[j];
    nb = fmin(nb, au - 0.1 * (au - xv));
    nb = fmin(nb, xv + S.move * st);
    V.alpha[j] = na;
    V.beta[j] = nb;
    V.lastdx[j] = d1;
    v[0] += d1 * d1;
  }
  block_partials<1>(v, mx, partial);
}

// fold `cnt` columns of `nb` per-block partials in a fixed order: one 64-lane wave per
// column (grid = cnt), lane-strided partial sums, then a fixed butterfly
// (every `period` columns the last `nmax` are maxima)
__global__ __launch_bounds__(64) void k_mma_fold(const double* __restrict__ partial, int nb, int period, int nmax,
                                                 double* __restrict__ out) {
  const int c = blockIdx.x;
  const bool mx = c % period >= period - nmax;
  const int lane = threadIdx.x;
  const double* col = partial + (int64_t)c * nb;
  double s = lane < nb ? col[lane] : (mx ? -HUGE_VAL : 0.0);
  for (int b = lane + 64; b < nb; b += 64) {
    const double v = col[b];
    s = mx ? fmax(s, v) : s + v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double v = __shfl_xor(s, o, 64);
    s = mx ? fmax(s, v) : s + v;
  }
  if (lane == 0) out[c] = s;
}

}  // namespace tos
