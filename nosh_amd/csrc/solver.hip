// solver.hip -- the preconditioner (Chebyshev iteration with 2x2 block-Jacobi
// scaling, standing in for the MueLu AMG cycle of keo_regularized::apply,
// src/keo_regularized.cpp:88-165) and preconditioned MINRES (Paige-Saunders),
// the in-repo replacement of the Belos solver (the reference example selects
// Pseudo Block GMRES at examples/conf.xml:104 with its MINRES line :105
// commented out; J is symmetric and the preconditioner SPD, so MINRES solves
// the same systems with a short recurrence, tolerance and limit as :117-123).
//
// MINRES runs as a fixed sequence of fused kernels per iteration with every
// scalar of the Lanczos/Givens recurrences kept on the device:
//   A  the Givens step of the previous iteration, one Jacobian product
//      v = y/beta, u = J v - (beta/beta_old) r1, the partial sums of
//      alpha = <v,u>, and the previous iteration's update of the direction
//      vectors w and the solution x;
//   B  alpha, r_new = u - (alfa/beta) r2 and the first Chebyshev step on r_new;
//   C  the remaining Chebyshev steps, each one product with P; the last one
//      also forms the partial sums of beta^2 = <r_new, z>.
// Reductions are deterministic: partial sums per block, added in a fixed order
// by every block of the next kernel (A and B) while there are few of them
// (kFoldMax), else by a one-block kernel in between. The Givens state is then
// written by A's first block to the other of two records, since the other
// blocks still read the old one. The host only polls the `done` flag every
// few iterations, so iterations issued after convergence leave before their
// row products (seven of them at 96^3: 0.17 ms, where working through the
// products without storing them took 1.1); it counts the iterations it issues,
// which fixes every buffer rotation (r1/r2, w) until then.
// Vectors are FP64 or FP32 (template T); inner products, norms, recurrence
// scalars and the solution accumulator are always FP64.

#include <algorithm>

#include "kernels.hpp"
#include "minres_device.hpp"
#include "solver.hpp"

namespace nosh {
namespace {

constexpr int kBlock = 256;

// Most partial sums that the consuming kernel adds itself: 16 loads a thread,
// issued ahead of the row product. A separate one-block kernel costs 2.5-6 us
// and a launch. Newton step of 16 iterations with the line at 1000 / 2048 /
// 4096 sums: 300^2 square (1416 sums) 856 / 800 / 803 us, 400^2 (2513)
// 961 / 967 / 893 us, 60^3 cube (3547) 1687 / 1685 / 1651 us. At 96^3 (14 k
// sums) both ways take 5.65 ms, and every block's own sum reads 200 MB.
constexpr unsigned kFoldMax = 4096;

// Sum of v over the 256 threads of a block, in every thread (fixed order).
__device__ __forceinline__ double block_total(double v) {
  __shared__ double w[kBlock / 64];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  return (w[0] + w[1]) + (w[2] + w[3]);
}

__device__ __forceinline__ double thread_sum(const double* __restrict__ partials, int nb) {
  double v = 0.0;
#pragma unroll 8
  for (int i = threadIdx.x; i < nb; i += kBlock) v += partials[i];
  return v;
}

// Chebyshev coefficients of one solve: theta, then (c1, c2) of steps 1, 2, ...
// Worked out once by the first kernel of a chain (some ten dependent FP64
// divisions, 0.5 us, that every thread of every step used to do).
template <class T>
struct ChebArgs {
  int64_t n;
  SellView sv;  // split off-diagonal layout
  const V2<T>* pval;   // P off-diagonal values
  const T* pblk;       // P diagonal blocks (3 n)
  const double* bound; // max ratio from the rebuild
  double upper, ratio;
  int iters;           // Chebyshev iterations (0 = identity)
  V2<T>* r;            // residual (written by mode 2's first step)
  const V2<T>* r2;     // mode 2: the previous residual
  const V2<T>* u;      // mode 2: J v - (beta/oldb) r1
  V2<T>* D;            // the Chebyshev direction (FP32)
  MinresScalars* S;
  double* coef;
  const double* pa;    // partial sums of alfa, na of them (mode 2)
  int na, fold;        // fold: the first step adds them, else S->alfa holds the sum
  double* pb;          // partial sums of beta^2
};

// Chebyshev step 0 (z = D^{-1} r / theta), producing r first in mode 2.
// mode: 0 standalone preconditioner, 1 MINRES initialisation, 2 MINRES iteration.
template <class T>
__global__ __launch_bounds__(kBlock) void k_cheb_first(ChebArgs<T> a, int mode, V2<T>* zout) {
  MinresScalars* S = a.S;
  const int64_t row = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  double alfa = 0.0;
  if (mode == 2) {
    alfa = a.fold ? thread_sum(a.pa, a.na) : S->alfa;
    if (S->done) return;
    if (a.fold) alfa = block_total(alfa);
    if (a.fold && blockIdx.x == 0 && threadIdx.x == 0) {
      S->alfa = alfa;
      S->pending = 0;
    }
  } else {
    if (mode == 1 && S->done) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      const double hi = cheb_hi(a.bound, a.upper);
      a.coef[0] = 0.5 * (hi + hi / a.ratio);
      for (int j = 1; j < a.iters; ++j) {
        const Cheb c = cheb_coef(hi, a.ratio, j);
        a.coef[2 * j - 1] = c.c1;
        a.coef[2 * j] = c.c2;
      }
    }
  }
  double s2[1] = {0.0};
  if (row < a.n) {
    V2<T> rv;
    if (mode == 2) {
      const T c = T(alfa / S->beta);
      const V2<T> uu = a.u[row], r2v = a.r2[row];
      rv.x = uu.x - c * r2v.x;
      rv.y = uu.y - c * r2v.y;
      a.r[row] = rv;
    } else {
      rv = a.r[row];
    }
    V2<T> z;
    if (a.iters == 0) {
      z = rv;
    } else {
      double th = 0.0;
      if (mode == 2) {
        th = a.coef[0];
      } else {
        const double hi = cheb_hi(a.bound, a.upper);
        th = 0.5 * (hi + hi / a.ratio);
      }
      T o0, o1;
      dinv<T>(a.pblk[row], a.pblk[a.n + row], a.pblk[2 * a.n + row], rv.x, rv.y, &o0, &o1);
      z.x = o0 / T(th);
      z.y = o1 / T(th);
    }
    zout[row] = z;
    s2[0] = double(rv.x) * double(z.x) + double(rv.y) * double(z.y);
  }
  if (mode == 0 || a.iters > 1) return;
  block_partials<1>(s2, a.pb);
}

// Chebyshev step j >= 1: z_j = z_{j-1} + d_j, d_0 = z_0,
// d_j = c1 d_{j-1} + c2 D^{-1} (r - P z_{j-1}). In FP64 d_{j-1} is the
// difference of the last two z (z_{j-2} sits in z_j's buffer and is overwritten
// by its own thread), which saves a write (96^3: 3 % of a solve). In FP32 it is
// stored by the steps that have a next one, not to carry the rounding of z.
template <class T, int P>
__global__ __launch_bounds__(kBlock) void k_cheb_step(ChebArgs<T> a, int mode, int j,
                                                     const V2<T>* __restrict__ zin,
                                                     V2<T>* __restrict__ zout) {
  const MinresScalars* S = a.S;  // never null, if of no use in mode 0
  const RowBlock<T, P> rb(a.n, a.sv);
  if (S->done && mode != 0) return;
  const int64_t row = rb.row;
  V2<T> zi{}, rv{}, d{};
  T b0 = T(1), b1 = T(1), b2 = T(0);
  if (rb.owner) {
    zi = zin[row];
    rv = a.r[row];
    if (j > 1) d = sizeof(T) == 4 ? a.D[row] : zout[row];
    b0 = a.pblk[row], b1 = a.pblk[a.n + row], b2 = a.pblk[2 * a.n + row];
  }
  const T c1 = T(a.coef[2 * j - 1]), c2 = T(a.coef[2 * j]);
  const V2<T> acc = row_product<T, P>(rb, a.n, a.sv, a.pval, zin);
  double s2 = 0.0;
  if (rb.owner) {
    const T res0 = rv.x - (acc.x + b0 * zi.x + b2 * zi.y);
    const T res1 = rv.y - (acc.y + b2 * zi.x + b1 * zi.y);
    T u0, u1;
    dinv<T>(b0, b1, b2, res0, res1, &u0, &u1);
    if (j == 1) {
      d = zi;
    } else if (sizeof(T) == 8) {
      d.x = zi.x - d.x;
      d.y = zi.y - d.y;
    }
    d.x = c1 * d.x + c2 * u0;
    d.y = c1 * d.y + c2 * u1;
    V2<T> z;
    z.x = zi.x + d.x;
    z.y = zi.y + d.y;
    if (sizeof(T) == 4 && j != a.iters - 1) a.D[row] = d;
    zout[row] = z;
    s2 = double(rv.x) * double(z.x) + double(rv.y) * double(z.y);
  }
  if (mode == 0 || j != a.iters - 1) return;
  slice_partials(rb, s2, a.pb);
}

// beta^2 = sum of the partials of <r, z>: MINRES initialisation (mode 1) or
// the Givens step of the current iteration (mode 2).
__global__ __launch_bounds__(kFinThreads) void k_fin_beta(MinresScalars* S,
                                                          const double* __restrict__ partials,
                                                          int nb, int mode) {
  if (mode == 2 && S->done) return;
  const double v = fin_sum(partials, nb);
  if (threadIdx.x == 0) {
    if (mode == 1)
      init_update(S, v);
    else
      givens_update(S, v);
  }
}

__global__ __launch_bounds__(kFinThreads) void k_fin_alfa(MinresScalars* S,
                                                          const double* __restrict__ partials,
                                                          int nb) {
  if (S->done) return;
  const double v = fin_sum(partials, nb);
  if (threadIdx.x == 0) {
    S->alfa = v;
    S->pending = 0;
  }
}

template <class T>
struct MinresArgs {
  int64_t n;
  SellView sv;  // split off-diagonal layout
  const V2<T>* jval;
  const T* jblk;
  const V2<T>* y;  // preconditioned residual of the previous iteration
  V2<T>* v;
  V2<T>* u;
  V2<T>* W[3];     // direction vector k in W[k % 3]
  double2* x;
};

// Pending update of iteration k: w_k = (v_k - oldeps w_{k-2} - delta w_{k-1}) / gamma,
// x += phi w_k.
template <class T>
__device__ __forceinline__ void w_update(const V2<T>* w1p, const V2<T>* w2p, V2<T>* wk, double2* x,
                                         const MinresScalars& S, int64_t row, V2<T> vk) {
  const V2<T> w1 = w1p[row], w2 = w2p[row];
  const T oe = T(S.p_oldeps), de = T(S.p_delta), dn = T(S.p_denom);
  V2<T> w;
  w.x = (vk.x - oe * w1.x - de * w2.x) * dn;
  w.y = (vk.y - oe * w1.y - de * w2.y) * dn;
  wk[row] = w;
  double2 xv = x[row];
  xv.x += S.p_phi * double(w.x);
  xv.y += S.p_phi * double(w.y);
  x[row] = xv;
}

// Iteration `it` (from 0). Sin: the state of this iteration's start, or with
// nb > 0 the one before the Givens step whose nb partial sums are in pb, which
// is then taken here and stored in Sout.
template <class T, int P>
__global__ __launch_bounds__(kBlock) void k_minres_a(MinresArgs<T> a, int it, const V2<T>* r1,
                                                     const MinresScalars* Sin, MinresScalars* Sout,
                                                     const double* pb, int nb, double* pa) {
  __shared__ MinresScalars S;
  double sum = nb > 0 ? thread_sum(pb, nb) : 0.0;
  const RowBlock<T, P> rb(a.n, a.sv);
  if (Sin->done) {
    if (nb > 0 && blockIdx.x == 0 && threadIdx.x == 0) *Sout = *Sin;
    return;
  }
  const int64_t row = rb.row;
  const V2<T> acc = row_product<T, P>(rb, a.n, a.sv, a.jval, a.y);
  if (nb > 0) sum = block_total(sum);
  if (threadIdx.x == 0) {
    S = *Sin;
    if (nb > 0) {
      givens_update(&S, sum);
      if (blockIdx.x == 0) *Sout = S;
    }
  }
  __syncthreads();
  if (S.done) return;
  double s = 0.0;
  if (rb.owner) {
    if (it >= 1)
      w_update<T>(a.W[(it + 1) % 3], a.W[(it + 2) % 3], a.W[it % 3], a.x, S, row, a.v[row]);
    const V2<T> yi = a.y[row];
    const T b0 = a.jblk[row], b1 = a.jblk[a.n + row], b2 = a.jblk[2 * a.n + row];
    const T ib = T(1.0 / S.beta);
    V2<T> uu;
    uu.x = (acc.x + b0 * yi.x + b2 * yi.y) * ib;
    uu.y = (acc.y + b2 * yi.x + b1 * yi.y) * ib;
    if (it >= 1) {
      const T c = T(S.beta / S.oldb);
      const V2<T> rv = r1[row];
      uu.x -= c * rv.x;
      uu.y -= c * rv.y;
    }
    V2<T> vn;
    vn.x = yi.x * ib;
    vn.y = yi.y * ib;
    a.v[row] = vn;
    a.u[row] = uu;
    s = double(vn.x) * double(uu.x) + double(vn.y) * double(uu.y);
  }
  slice_partials(rb, s, pa);
}

// Applies the last pending w/x update, then psi += x when psi != nullptr.
template <class T>
__global__ __launch_bounds__(kBlock) void k_minres_flush(MinresArgs<T> a, const MinresScalars* S,
                                                         double2* psi) {
  const int64_t row = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (row >= a.n) return;
  if (S->pending) {
    const int k = S->it;
    w_update<T>(a.W[(k + 1) % 3], a.W[(k + 2) % 3], a.W[k % 3], a.x, *S, row, a.v[row]);
  }
  if (psi) {
    const double2 d = a.x[row];
    double2 p = psi[row];
    p.x += d.x;
    p.y += d.y;
    psi[row] = p;
  }
}

// r0 = r1 = scale * b (converted to T), x = 0, w_{-1} = w_0 = 0, and the state
// of a solve about to start.
template <class T>
__global__ void k_minres_setup(int64_t n, const double2* __restrict__ b, double scale,
                               V2<T>* R0, V2<T>* R1, V2<T>* W0, V2<T>* W2, double2* x,
                               MinresScalars* S, double rtol, int maxit) {
  const int64_t row = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (row == 0) {
    S->done = 0;
    S->it = 0;
    S->pending = 0;
    S->rtol = rtol;
    S->maxit = maxit;
    S->relres = 1.0;
  }
  if (row >= n) return;
  const double2 bv = b[row];
  V2<T> r;
  r.x = T(scale * bv.x);
  r.y = T(scale * bv.y);
  R0[row] = r;
  R1[row] = r;
  V2<T> z;
  z.x = T(0);
  z.y = T(0);
  W0[row] = z;
  W2[row] = z;
  x[row] = make_double2(0.0, 0.0);
}

template <class T>
__global__ void k_to_t(int64_t m, const double* __restrict__ a, T* __restrict__ b) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i < m) b[i] = T(a[i]);
}

}  // namespace

template <class T>
void MinresWork<T>::ensure(int64_t n_) {
  if (n == n_) return;
  n = n_;
  for (auto* b : {&Y, &Z2, &v, &u, &R0, &R1, &W0, &W1, &W2}) b->alloc(n);
  if (sizeof(T) == 4) D.alloc(n);
  x.alloc(n);
  partials.alloc(2 * size_t(grid_for(n, kSliceH) + 4));  // one per slice, whatever its waves
  if (!S.p) S.alloc(2);
  if (!Sh) NOSH_HIP(hipHostMalloc(reinterpret_cast<void**>(&Sh), sizeof(MinresScalars)));
  NOSH_HIP(hipStreamSynchronize(default_stream()));
}

template <class T>
MinresWork<T>::~MinresWork() {
  if (Sh) (void)hipHostFree(Sh);
}

template <class T>
static ChebArgs<T> cheb_args(const MeshCache& m, const PrecView<T>& P, MinresWork<T>& w) {
  const size_t nc = 2 * size_t(std::max(P.iters, 64));
  if (w.coef.n < nc) w.coef.alloc(nc);
  ChebArgs<T> a{};
  a.n = m.n;
  a.sv = sell_view(m);
  a.pval = P.val;
  a.pblk = P.blk;
  a.bound = P.bound;
  a.upper = P.upper;
  a.ratio = P.ratio;
  a.iters = P.iters;
  a.u = w.u.p;
  a.D = w.D.p;
  a.S = w.S.p;
  a.coef = w.coef.p;
  a.pa = w.partials.p;
  a.pb = w.partials.p + w.partials.n / 2;
  return a;
}

// Launches the Chebyshev chain so that the final z lands in `out`; returns
// the number of partial sums of beta^2 (modes 1 and 2).
template <class T>
static unsigned cheb_chain(const MeshCache& m, const ChebArgs<T>& a, int mode, V2<T>* out,
                           V2<T>* tmp, hipStream_t s) {
  const unsigned n1 = grid_for(m.n, kBlock), nb = row_blocks(m);
  const auto step = row_split(m) == 4 ? k_cheb_step<T, 4> : k_cheb_step<T, 2>;
  const int steps = a.iters < 1 ? 1 : a.iters;
  V2<T>* zb[2] = {out, tmp};
  int cur = (steps - 1) % 2;
  k_cheb_first<T><<<n1, kBlock, 0, s>>>(a, mode, zb[cur]);
  for (int j = 1; j < steps; ++j) {
    step<<<nb, kBlock, 0, s>>>(a, mode, j, zb[cur], zb[1 - cur]);
    cur = 1 - cur;
  }
  return steps > 1 ? row_slices(m) : n1;
}

template <class T>
void prec_apply(const MeshCache& m, const PrecView<T>& P, MinresWork<T>& w, const V2<T>* r,
                V2<T>* z, hipStream_t s) {
  ChebArgs<T> a = cheb_args(m, P, w);
  a.r = const_cast<V2<T>*>(r);  // read only in mode 0
  cheb_chain<T>(m, a, 0, z, w.Z2.p, s);
}

template <class T>
int minres_solve(const MeshCache& m, const JacView<T>& J, const PrecView<T>& P,
                 MinresWork<T>& w, const double* b, double b_scale, double rtol, int maxit,
                 double* psi_update, hipStream_t s, double* relres_out, int poll) {
  w.ensure(m.n);
  const unsigned n1 = grid_for(m.n, kBlock), nb = row_blocks(m), ns = row_slices(m);
  MinresScalars* S[2] = {w.S.p, w.S.p + 1};
  int cur = 0;  // the current state's record
  k_minres_setup<T><<<n1, kBlock, 0, s>>>(m.n, reinterpret_cast<const double2*>(b), b_scale,
                                          w.R0.p, w.R1.p, w.W0.p, w.W2.p, w.x.p, S[0], rtol,
                                          maxit);
  V2<T>* R[2] = {w.R0.p, w.R1.p};
  ChebArgs<T> ca = cheb_args(m, P, w);
  double* const pa = w.partials.p;
  ca.na = int(ns);
  ca.fold = ns <= kFoldMax;
  // y = M^{-1} b and beta1.
  ca.r = R[0];
  const unsigned nbeta = cheb_chain<T>(m, ca, 1, w.Y.p, w.Z2.p, s);
  k_fin_beta<<<1, kFinThreads, 0, s>>>(S[0], ca.pb, int(nbeta), 1);
  MinresArgs<T> ma{m.n, sell_view(m), J.val, J.blk, w.Y.p, w.v.p, w.u.p,
                   {w.W0.p, w.W1.p, w.W2.p}, w.x.p};
  const bool fold_beta = nbeta <= kFoldMax;
  const auto iter = row_split(m) == 4 ? k_minres_a<T, 4> : k_minres_a<T, 2>;
  int issued = 0;
  for (;;) {
    bool owed = false;  // the last iteration's Givens step is still to be taken
    for (int q = 0; q < poll && issued < maxit; ++q, ++issued) {
      iter<<<nb, kBlock, 0, s>>>(ma, issued, R[issued & 1], S[cur], S[1 - cur], ca.pb,
                                 owed ? int(nbeta) : 0, pa);
      if (owed) cur = 1 - cur;
      ca.S = S[cur];
      ca.r = R[issued & 1];
      ca.r2 = R[1 - (issued & 1)];
      if (!ca.fold) k_fin_alfa<<<1, kFinThreads, 0, s>>>(S[cur], pa, int(ns));
      cheb_chain<T>(m, ca, 2, w.Y.p, w.Z2.p, s);
      owed = fold_beta && q + 1 < poll && issued + 1 < maxit;
      if (!owed) k_fin_beta<<<1, kFinThreads, 0, s>>>(S[cur], ca.pb, int(nbeta), 2);
    }
    NOSH_HIP(hipMemcpyAsync(w.Sh, S[cur], sizeof(MinresScalars), hipMemcpyDeviceToHost, s));
    NOSH_HIP(hipStreamSynchronize(s));
    if (w.Sh->done || issued >= maxit) break;
  }
  k_minres_flush<T><<<n1, kBlock, 0, s>>>(ma, S[cur], reinterpret_cast<double2*>(psi_update));
  if (relres_out) *relres_out = w.Sh->relres;
  return w.Sh->it;
}

template <class T>
void convert_to(const double* a, T* b, int64_t m, hipStream_t s) {
  k_to_t<T><<<grid_for(m, kBlock), kBlock, 0, s>>>(m, a, b);
}

template struct MinresWork<double>;
template struct MinresWork<float>;
template void prec_apply<double>(const MeshCache&, const PrecView<double>&, MinresWork<double>&,
                                 const double2*, double2*, hipStream_t);
template void prec_apply<float>(const MeshCache&, const PrecView<float>&, MinresWork<float>&,
                                const float2*, float2*, hipStream_t);
template int minres_solve<double>(const MeshCache&, const JacView<double>&,
                                  const PrecView<double>&, MinresWork<double>&, const double*,
                                  double, double, int, double*, hipStream_t, double*, int);
template int minres_solve<float>(const MeshCache&, const JacView<float>&, const PrecView<float>&,
                                 MinresWork<float>&, const double*, double, double, int, double*,
                                 hipStream_t, double*, int);
template void convert_to<float>(const double*, float*, int64_t, hipStream_t);

}  // namespace nosh
