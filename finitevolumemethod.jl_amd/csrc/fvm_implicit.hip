// TR-BDF2 for small problems whose right-hand side is affine in u, and GMRES for small
// systems with an explicit sparse matrix, each in one launch.
//
// The reference integrates the tutorials' stiff problems with TRBDF2 and a KLU
// factorisation of the sparse Jacobian (solve.jl:167-183, jacobian_sparsity
// solve.jl:50-77).  When f(u) = J u + c (linear fluxes, sources affine in u,
// conditions constant in t), J is constant: the host package extracts it once
// from fvm_jvp probes over a colouring of jacobian_sparsity's pattern, and
// trbdf2_affine_kernel runs the whole integration: both stages' Newton iterations
// with restarted GMRES(m) on W = I - d h J (the Hessenberg least squares by Givens
// rotations), the W^-1-filtered error estimate, the step controller, the Dirichlet
// update and the saveat interpolation, with no host round trip.  For a nonlinear
// problem the host integrator keeps its loop and hands each linear system to
// gmres_kernel, J frozen at the step's start and extracted there the same way.
//
// Layout: one row per thread, one workgroup per CU, the workgroups resident together
// (cooperative launch).  Every vector of the integration is a register of its row's
// thread, the matrix row too, and the Krylov basis of a workgroup's rows lies in its
// LDS; a product publishes one vector to the grid and a Gram-Schmidt pass is one
// grid-wide sum (fvm_grid.hpp), so a Krylov step costs two exchanges of 1.5 to 2 us
// and about as much arithmetic, whatever n.  What bounds it is that latency: 6.0 ms for
// 805 Krylov steps and 139 Newton iterations on 10,000 rows, where the same loop in
// one workgroup of 1024 threads, its vectors in memory, took 55.5 ms (one CU's rate
// out of L2).
// The algorithm is the host integrator's (solve.py), step for step; reductions here
// sum in a different order, so results agree with it to the Krylov and Newton
// tolerances, not bit for bit.
#include <cmath>

#include "fvm_grid.hpp"

namespace {

using fvm::Grid;
using fvm::GridShared;

constexpr int kMaxRestart = 30;
constexpr int64_t kMaxN = 65536;
constexpr int kRows = 256;  // rows per workgroup: 256 workgroups at most
// One pass of classical Gram-Schmidt multiplies the basis's loss of orthogonality by
// |w| / |w'| (the vector's length before and after it; Giraud, Langou, Rozloznik & van
// den Eshof, Numer. Math. 101, 2005), so the loss is tracked and the pass repeated when
// it would exceed this part of the solve's own tolerance: at rtol 1e-3 and 10,000 rows
// no step needs the second pass, which taken always costs 15 %.
constexpr double kLossPart = 1e-3;

constexpr double kG = 0.58578643762690485;  // 2 - sqrt(2)

// J in ELL form (fvm_affine_op), column s of row i at [s n + i]
struct EllJ {
  int64_t n;
  int W;
  const int32_t* col;
  const double* val;
  const double* diag;
  const int32_t* orp;
  const int32_t* ocol;
  const double* oval;
};

template <int T>
struct Shared {
  GridShared<T> grid;
  double V[kMaxRestart + 1][T];  // the basis on this workgroup's rows
  double H[kMaxRestart + 1][kMaxRestart];
  double h[kMaxRestart + 1];
  double g[kMaxRestart + 1], cs[kMaxRestart], sn[kMaxRestart], y[kMaxRestart];
};

// The thread's row of J: W slots in registers (W > 0), or read from memory four at a
// time (W == 0: widths beyond the meshes').
template <int W>
struct Row {
  uint32_t c[W > 0 ? W : 1];  // grid_offset of the column
  double v[W > 0 ? W : 1];
  double diag;
  int o0, o1;
  __device__ __forceinline__ void load(const EllJ& J, int64_t i, bool active) {
    diag = active ? J.diag[i] : 0.0;
    o0 = active ? J.orp[i] : 0;
    o1 = active ? J.orp[i + 1] : 0;
#pragma unroll
    for (int s = 0; s < W; ++s) {
      c[s] = active ? fvm::grid_offset(J.col[s * J.n + i]) : 0;
      v[s] = active ? J.val[s * J.n + i] : 0.0;
    }
  }
};

// row i of J x for the vector published last, x this thread's entry of it
template <int W, int T>
__device__ __forceinline__ double row_J(const EllJ& J, const Row<W>& R, Grid<T>& G, int64_t i, bool active,
                                        double x) {
  double acc = 0.0;
  if constexpr (W > 0) {
    double xc[W];
    G.fetch(R.c, xc, active);
#pragma unroll
    for (int s = 0; s < W; ++s) acc += R.v[s] * xc[s];
  } else if (active) {
    for (int s0 = 0; s0 < J.W; s0 += 4) {
      uint32_t c[4];
      double v[4], xc[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bool on = s0 + s < J.W;
        c[s] = fvm::grid_offset(on ? J.col[(s0 + s) * J.n + i] : (int)i);
        v[s] = on ? J.val[(s0 + s) * J.n + i] : 0.0;
      }
      G.fetch(c, xc, true);
#pragma unroll
      for (int s = 0; s < 4; ++s) acc += v[s] * xc[s];
    }
  }
  for (int k = R.o0; k < R.o1; ++k) acc += J.oval[k] * G.fetch1(J.ocol[k]);
  return acc + R.diag * x;
}

template <int W, int T>
__device__ __forceinline__ double apply_J(const EllJ& J, const Row<W>& R, Grid<T>& G, int64_t i, bool active,
                                          double x) {
  G.publish(i, x, active);
  return row_J<W>(J, R, G, i, active, x);
}

// x = A^-1 b approximately, A = a I + bj J, restarted GMRES(m) from x = 0 (solve.py's
// gmres_device: stop when |r| <= rtol |b|), right-preconditioned by diag(scale) with
// scale this row's entry; returns the Arnoldi steps taken, or -1 when the grid gave up
template <int W, int T>
__device__ __forceinline__ int64_t gmres(Shared<T>& S, Grid<T>& G, const EllJ& J, const Row<W>& R, int64_t i,
                                         bool active, double a, double bj, double scale, double b, double& x,
                                         double rtol, int m, int64_t maxiter) {
  const int tid = threadIdx.x;
  x = 0.0;
  double bnorm = -1.0;
  int64_t total = 0;
  while (total < maxiter) {
    // r = b - A x (r = b while x is still zero)
    double r = b;
    if (bnorm >= 0.0) r = b - (a * x + bj * apply_J<W>(J, R, G, i, active, x));
    double rr;
    if (!G.sum1(r * r, &rr)) return -1;
    const double beta = sqrt(rr);
    if (bnorm < 0.0) {
      bnorm = beta;
      if (bnorm == 0.0) return 0;
    } else if (beta <= rtol * bnorm) {
      break;
    }
    double vj = r / beta;
    S.V[0][tid] = vj;
    if (tid == 0) S.g[0] = beta;
    int kd = 0;
    double loss = 0.0;
    double z = scale * vj;
    G.publish(i, z, active);
    for (int j = 0; j < m; ++j) {
      double w = a * z + bj * row_J<W>(J, R, G, i, active, z);
      double ww = 0.0;
#pragma nounroll
      for (int pass = 0; pass < 2; ++pass) {
        // w against the basis, and |w|^2 before the pass
        if (!G.sum(j + 2, [&](int q) { return (q <= j ? S.V[q][tid] : w) * w; })) return -1;
        double hh = 0.0;
#pragma unroll 4
        for (int q = 0; q <= j; ++q) {
          const double h = S.grid.tot[q];
          hh += h * h;
          w = w - h * S.V[q][tid];
        }
        const double w0 = S.grid.tot[j + 1];
        ww = w0 - hh;  // |w|^2 after it (Pythagoras)
        if (tid <= j) S.h[tid] = pass == 0 ? S.grid.tot[tid] : S.h[tid] + S.grid.tot[tid];
        __syncthreads();  // tot is free again, h written
        const double grown = (loss + 0x1p-52) * sqrt(w0 / ww);
        if (ww > 0.0 && grown <= kLossPart * rtol) {
          loss = fmax(loss, grown);
          break;
        }
      }
      const double hn = sqrt(fmax(ww, 0.0));
      vj = hn > 0.0 ? w / hn : 0.0;
      S.V[j + 1][tid] = vj;
      // the next basis vector goes out before the rotations decide whether it is needed:
      // they take about as long as its way (one that is not needed is not read, so its
      // half of the buffer may be written again at once)
      z = scale * vj;
      G.publish(i, z, active);
      if (tid == 0) {
        double hq = S.h[0];
#pragma nounroll
        for (int q = 0; q < j; ++q) {  // previous rotations
          const double o = S.h[q + 1];
          S.H[q][j] = S.cs[q] * hq + S.sn[q] * o;
          hq = -S.sn[q] * hq + S.cs[q] * o;
        }
        const double dd = sqrt(hq * hq + hn * hn);
        const double cs = dd == 0.0 ? 1.0 : hq / dd, sn = dd == 0.0 ? 0.0 : hn / dd;
        S.cs[j] = cs;
        S.sn[j] = sn;
        S.H[j][j] = dd;
        const double g = S.g[j];
        S.g[j + 1] = -sn * g;
        S.g[j] = cs * g;
      }
      __syncthreads();
      ++total;
      kd = j + 1;
      if (fabs(S.g[j + 1]) <= rtol * bnorm || total >= maxiter) break;
    }
    const double res = fabs(S.g[kd]);
    if (tid == 0) {  // back substitution
#pragma nounroll
      for (int q = kd - 1; q >= 0; --q) {
        double sum = S.g[q];
#pragma nounroll
        for (int p = q + 1; p < kd; ++p) sum -= S.H[q][p] * S.y[p];
        S.y[q] = sum / S.H[q][q];
      }
    }
    __syncthreads();
    double acc = 0.0;
#pragma unroll 4
    for (int q = 0; q < kd; ++q) acc = acc + S.y[q] * S.V[q][tid];
    x = x + scale * acc;
    if (res <= rtol * bnorm) break;
  }
  return total;
}

struct Trb {
  EllJ J;
  const double* c;
  int32_t n_dir;
  const int32_t* dir_idx;
  const double* dir_val;
  double* u;  // the state in and out
  uint64_t* grid;
  double t0, tf, dt, abstol, reltol;
  int64_t maxiters;
  double kappa, krtol;
  int max_newton, restart, smooth;
  int64_t n_save;
  const double* save_t;
  double* saves;
  double* stats;
};

template <int W, int T>
__global__ __launch_bounds__(T) void trbdf2_affine_kernel(Trb a) {
  __shared__ Shared<T> S;
  const int64_t n = a.J.n;
  const int64_t i = (int64_t)blockIdx.x * T + threadIdx.x;
  const bool active = i < n;
  Grid<T> G;
  G.open(a.grid, n, &S.grid);
  Row<W> R;
  R.load(a.J, i, active);
  const double ci = active ? a.c[i] : 0.0;
  double u = active ? a.u[i] : 0.0;
  bool held = false;  // a Dirichlet node (the last entry naming it wins)
  double held_at = 0.0;
  for (int k = 0; k < a.n_dir; ++k)
    if (a.dir_idx[k] == i) {
      held = true;
      held_at = a.dir_val[k];
    }
  const double d = kG / 2;
  const double TA = 1.0 / (kG * (2.0 - kG)), TB = -(1.0 - kG) * (1.0 - kG) / (kG * (2.0 - kG));
  const double TK = (3 * kG * kG - 4 * kG + 2) / (6 * (2.0 - kG));
  int64_t nf = 0, njvp = 0, naccept = 0, nreject = 0, nnewton = 0, nkrylov = 0, nfail = 0, ks = 0, it = 0;
  int retcode = 0;  // FVM_ODE_SUCCESS
  bool up = true;   // the grid's exchanges work
  double t = a.t0, dt = a.dt, eta_keep = 1.0;
  // sqrt(mean((e / (abstol + reltol max(|p|, |q|)))^2)), the integrators' error norm
  auto err_norm = [&](double e, double p, double q) {
    const double r = e / (a.abstol + a.reltol * fmax(fabs(p), fabs(q)));
    double s = 0.0;
    up = up && G.sum1(active ? r * r : 0.0, &s);
    return sqrt(s / (double)n);
  };
  double fn = 0.0;
  bool fresh = false;  // fn = f(u)
  while (t < a.tf && it < a.maxiters) {
    ++it;
    const double h = fmin(dt, a.tf - t), dh = d * h;
    // Three solves per step: stage 0, TR: z - d h f(z) = u + d h f_n, predictor
    // u + gamma h f_n; stage 1, BDF2: u1 - d h f(u1) = A z + B u, predictor
    // z + (1 - gamma) h f_gamma; each by Newton.  Stage 2: the error estimate through
    // W^-1.  One loop, so that the product and the Krylov solve are compiled once.
    double z = u, u1 = 0.0, fg = 0.0, f1 = 0.0, est = 0.0;
    bool ok = true;
#pragma nounroll
    for (int stage = fresh ? 0 : -1; stage < 3 && ok; ++stage) {
      double x = 0.0, fx = 0.0, rhs = 0.0;
      if (stage == -1) {
        x = u;
      } else if (stage == 0) {
        rhs = u + dh * fn;
        x = u + kG * h * fn;
      } else if (stage == 1) {
        rhs = TA * z + TB * u;
        x = z + (1.0 - kG) * h * fg;
      } else {
        if (!a.smooth) break;
      }
      double eta = fvm::ctrl_pow(fmax(eta_keep, 1e-16), 0.8), prev = -1.0;
      bool done = stage == -1;
      ok = done;
#pragma nounroll
      for (int itn = 0;; ++itn) {
        double b = est;
        if (stage < 2) {
          fx = apply_J<W>(a.J, R, G, i, active, x) + ci;
          ++nf;
          if (done || itn == a.max_newton) break;
          b = -1.0 * x + dh * fx + rhs;
        }
        double dx;
        const int64_t k = gmres<W, T>(S, G, a.J, R, i, active, 1.0, -dh, 1.0, b, dx, a.krtol, a.restart,
                                      20 * (int64_t)a.restart);
        up = up && k >= 0;
        if (!up) break;
        nkrylov += k;
        njvp += k + 1;
        if (stage == 2) {
          est = dx;
          ok = true;
          break;
        }
        x = x + dx;
        ++nnewton;
        const double ndz = err_norm(dx, u, x);
        if (!up || !isfinite(ndz)) break;
        if (prev >= 0.0) {
          const double theta = ndz / prev;
          if (theta >= 1.0) break;
          eta = theta / (1.0 - theta);
        }
        if (eta * ndz <= a.kappa || ndz == 0.0) done = ok = true;
        prev = ndz;
      }
      if (!ok) break;
      if (stage == -1) {
        fn = fx;
        fresh = true;
      } else if (stage == 0) {
        z = x;
        fg = fx;
        eta_keep = eta;
      } else if (stage == 1) {
        u1 = x;
        f1 = fx;
        eta_keep = eta;
        est = TK * h / kG * fn;
        est = est + -TK * h / (kG * (1 - kG)) * fg;
        est = est + TK * h / (1 - kG) * f1;
      }
    }
    if (!up) break;
    if (!ok) {
      ++nfail;
      ++nreject;
      dt = h / 4;
      if (dt < 1e-14 * fmax(1.0, fabs(t))) {
        retcode = 3;  // ConvergenceFailure
        break;
      }
      continue;
    }
    const double EEst = err_norm(est, u, u1);
    if (!up) break;
    if (!isfinite(EEst)) {
      retcode = 2;  // Unstable
      break;
    }
    if (EEst <= 1.0) {
      const double tn = t + h;
      while (ks < a.n_save && a.save_t[ks] <= tn + 1e-12 * fmax(1.0, fabs(tn))) {
        const double th = fmin(1.0, fmax(0.0, (a.save_t[ks] - t) / h));
        const double t2 = th * th, t3 = t2 * th;
        const double h00 = 2 * t3 - 3 * t2 + 1, h10 = t3 - 2 * t2 + th, h01 = -2 * t3 + 3 * t2, h11 = t3 - t2;
        double v = h00 * u;
        v = v + h10 * h * fn;
        v = v + h01 * u1;
        v = v + h11 * h * f1;
        if (active) a.saves[ks * n + i] = v;
        ++ks;
      }
      u = u1;
      t = tn;
      ++naccept;
      if (a.n_dir > 0) {  // the Dirichlet callback (values constant), then f(u) afresh
        if (held) u = held_at;
        fresh = false;
      } else {
        fn = f1;
      }
    } else {
      ++nreject;
    }
    const double q = 0.9 * fvm::ctrl_pow(fmax(EEst, 1e-10), -1.0 / 3.0);
    dt = h * fmin(5.0, fmax(0.2, q));
    if (dt < 1e-14 * fmax(1.0, fabs(t))) {  // the step collapsed: stop instead of creeping on
      retcode = 3;
      break;
    }
  }
  if (retcode == 0 && !(t >= a.tf)) retcode = 1;  // MaxIters
  if (active) a.u[i] = u;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    double* st = a.stats;
    st[0] = t;
    st[1] = (double)nf;
    st[2] = (double)njvp;
    st[3] = (double)naccept;
    st[4] = (double)nreject;
    st[5] = (double)nnewton;
    st[6] = (double)nkrylov;
    st[7] = (double)nfail;
    st[8] = (double)ks;
    st[9] = up ? (double)retcode : -1.0;
  }
}

// One linear solve of the host loop's Newton iterations: 9 Krylov steps on 2,867 rows
// take about 55 us with the cooperative launch's 20, where the host-driven GMRES took
// about a dozen launches and a synchronisation per Krylov step (107 us); the nonlinear
// TR-BDF2 solve of 61 x 47 nodes went from 85.8 to 12.0 ms.
struct Gm {
  EllJ J;
  double a, bj;
  int jacobi;
  const double* b;
  double* x;
  double rtol;
  int restart;
  int64_t maxiter;
  uint64_t* grid;
};

template <int W, int T>
__global__ __launch_bounds__(T) void gmres_kernel(Gm p) {
  __shared__ Shared<T> S;
  const int64_t i = (int64_t)blockIdx.x * T + threadIdx.x;
  const bool active = i < p.J.n;
  Grid<T> G;
  G.template open<true>(p.grid, p.J.n, &S.grid);
  Row<W> R;
  R.load(p.J, i, active);
  const double di = p.a + p.bj * R.diag;  // the row's diagonal entry
  const double scale = p.jacobi && fabs(di) > 1e-12 ? 1.0 / di : 1.0;
  double x;
  const int64_t k = gmres<W, T>(S, G, p.J, R, i, active, p.a, p.bj, scale, active ? p.b[i] : 0.0, x, p.rtol,
                                p.restart, p.maxiter);
  // no solution when the grid gave up: the host's norms of x see it at once
  if (active) p.x[i] = k < 0 ? __longlong_as_double(0x7ff8000000000000ll) : x;
  if (k > 0 && blockIdx.x == 0 && threadIdx.x == 0) p.grid[fvm::kGridUser] += (uint64_t)k;
  G.close();
}

// J in ELL form from its products with the colours' probe vectors: entry (slot, row) is
// the row's entry of the product with its column's colour (255: padding), the diagonal
// in slot W.
__global__ __launch_bounds__(256) void ell_from_probes(int64_t n, int W, const uint8_t* __restrict__ colour,
                                                       const double* __restrict__ jv, double* __restrict__ val,
                                                       double* __restrict__ diag) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  for (int s = 0; s <= W; ++s) {
    const int c = colour[s * n + i];
    const double v = c == 255 ? 0.0 : jv[c * n + i];
    if (s < W) val[s * n + i] = v;
    else diag[i] = v;
  }
}

EllJ ell_of(const fvm_affine_op* op) {
  EllJ J;
  J.n = op->n;
  J.W = op->width;
  J.col = op->d_col;
  J.val = op->d_val;
  J.diag = op->d_diag;
  J.orp = op->d_ovf_rp;
  J.ocol = op->d_ovf_col;
  J.oval = op->d_ovf_val;
  return J;
}

// kernel<W, kRows> for an operator of ELL width w: the widths of triangle meshes as
// compile-time constants, others at run time.
#define FVM_TRB_KERNEL(kernel, w)                            \
  ((w) == 4    ? (const void*)kernel<4, kRows>               \
   : (w) == 5  ? (const void*)kernel<5, kRows>               \
   : (w) == 6  ? (const void*)kernel<6, kRows>               \
   : (w) == 7  ? (const void*)kernel<7, kRows>               \
   : (w) == 8  ? (const void*)kernel<8, kRows>               \
   : (w) == 9  ? (const void*)kernel<9, kRows>               \
   : (w) == 10 ? (const void*)kernel<10, kRows>              \
               : (const void*)kernel<0, kRows>)

int64_t workgroups(int64_t n) { return (n + kRows - 1) / kRows; }

// FVM_ERR_STATE where the device does not hold the kernel's workgroups for n rows at once
int check_fits(const void* kernel, int64_t n, const char* who) {
  bool fits;
  FVM_HIP(fvm::grid_fits(kernel, kRows, workgroups(n), &fits));
  if (fits) return FVM_OK;
  fvm::set_error(std::string(who) + ": the device does not hold a workgroup per 256 unknowns at once");
  return FVM_ERR_STATE;
}

template <class Args>
hipError_t launch(const void* kernel, int64_t n, Args& a, hipStream_t s) {
  void* p[] = {&a};
  return hipLaunchCooperativeKernel(kernel, dim3((unsigned)workgroups(n)), dim3(kRows), p, 0, s);
}

int check_op(const fvm_affine_op* op, const char* who) {
  FVM_CHECK(op->n > 0 && op->n <= kMaxN, std::string(who) + ": 1 <= n <= 65536");
  FVM_CHECK(op->width >= 0 && op->d_col && op->d_val && op->d_diag && op->d_ovf_rp,
            std::string(who) + ": incomplete operator");
  return FVM_OK;
}

}  // namespace

extern "C" {

int fvm_trbdf2_affine(const fvm_affine_op* op, const fvm_trbdf2_opts* o, double* d_u, fvm_trbdf2_stats* st,
                      fvm_stream s) {
  FVM_CHECK(op && o && d_u && st, "fvm_trbdf2_affine: null argument");
  int rc = check_op(op, "fvm_trbdf2_affine");
  if (rc) return rc;
  FVM_CHECK(op->d_c, "fvm_trbdf2_affine: incomplete operator");
  FVM_CHECK(op->n_dirichlet == 0 || (op->d_dir_nodes && op->d_dir_values), "fvm_trbdf2_affine: Dirichlet lists");
  FVM_CHECK(o->krylov_restart >= 1 && o->krylov_restart <= kMaxRestart, "fvm_trbdf2_affine: restart 1..30");
  FVM_CHECK(o->max_newton >= 1 && o->abstol > 0 && o->reltol >= 0 && o->maxiters > 0 && o->tf >= o->t0 &&
                o->dt > 0,
            "fvm_trbdf2_affine: bad options");
  FVM_CHECK(o->n_save >= 0 && (o->n_save == 0 || (o->save_t && o->d_saves)), "fvm_trbdf2_affine: save times");
  const int64_t n = op->n;
  const void* const kernel = FVM_TRB_KERNEL(trbdf2_affine_kernel, op->width);
  if ((rc = check_fits(kernel, n, "fvm_trbdf2_affine"))) return rc;
  Trb a;
  a.J = ell_of(op);
  a.c = op->d_c;
  a.n_dir = op->n_dirichlet;
  a.dir_idx = op->d_dir_nodes;
  a.dir_val = op->d_dir_values;
  a.u = d_u;
  a.t0 = o->t0;
  a.tf = o->tf;
  a.dt = o->dt;
  a.abstol = o->abstol;
  a.reltol = o->reltol;
  a.maxiters = o->maxiters;
  a.kappa = o->newton_kappa;
  a.krtol = o->krylov_rtol;
  a.max_newton = o->max_newton;
  a.restart = o->krylov_restart;
  a.smooth = o->smooth_est;
  a.n_save = o->n_save;
  a.saves = o->d_saves;
  const size_t words = fvm::grid_words(n);
  double* base = nullptr;
  FVM_HIP(fvm::dev_alloc((void**)&base, sizeof(double) * (words + (size_t)o->n_save + 16)));
  a.grid = (uint64_t*)base;
  double* tail = base + words;
  a.save_t = tail;
  a.stats = tail + o->n_save;
  hipStream_t st_ = (hipStream_t)s;
  double r[10] = {0};
  hipError_t e = hipMemsetAsync(base, 0, sizeof(double) * words, st_);
  if (e == hipSuccess && o->n_save > 0)
    e = hipMemcpyAsync(tail, o->save_t, sizeof(double) * (size_t)o->n_save, hipMemcpyHostToDevice, st_);
  if (e == hipSuccess) e = launch(kernel, n, a, st_);
  if (e == hipSuccess) e = hipMemcpyAsync(r, a.stats, sizeof r, hipMemcpyDeviceToHost, st_);
  if (e == hipSuccess) e = hipStreamSynchronize(st_);
  (void)fvm::dev_free(base);
  if (e != hipSuccess) return fvm::hip_fail(e, "fvm_trbdf2_affine");
  if (r[9] < 0) {
    fvm::set_error("fvm_trbdf2_affine: the grid's exchange timed out");
    return FVM_ERR_HIP;
  }
  st->t = r[0];
  st->nf = (int64_t)r[1];
  st->njvp = (int64_t)r[2];
  st->naccept = (int64_t)r[3];
  st->nreject = (int64_t)r[4];
  st->nnewton = (int64_t)r[5];
  st->nkrylov = (int64_t)r[6];
  st->nnewton_fail = (int64_t)r[7];
  st->nsaved = (int64_t)r[8];
  st->retcode = (int32_t)r[9];
  return FVM_OK;
}

size_t fvm_gmres_work_bytes(int64_t n) { return sizeof(uint64_t) * fvm::grid_words(n > 0 ? n : 0); }

int fvm_gmres_ell(const fvm_affine_op* op, double a, double b, int32_t jacobi, const double* d_rhs, double* d_x,
                  double rtol, int32_t restart, int64_t maxiter, void* d_work, fvm_stream s) {
  FVM_CHECK(op && d_rhs && d_x && d_work, "fvm_gmres_ell: null argument");
  int rc = check_op(op, "fvm_gmres_ell");
  if (rc) return rc;
  FVM_CHECK(restart >= 1 && restart <= kMaxRestart, "fvm_gmres_ell: restart 1..30");
  FVM_CHECK(rtol > 0 && maxiter > 0, "fvm_gmres_ell: rtol and maxiter must be positive");
  const void* const kernel = FVM_TRB_KERNEL(gmres_kernel, op->width);
  if ((rc = check_fits(kernel, op->n, "fvm_gmres_ell"))) return rc;
  Gm g;
  g.J = ell_of(op);
  g.a = a;
  g.bj = b;
  g.jacobi = jacobi;
  g.b = d_rhs;
  g.x = d_x;
  g.rtol = rtol;
  g.restart = restart;
  g.maxiter = maxiter;
  g.grid = (uint64_t*)d_work;
  FVM_HIP(launch(kernel, g.J.n, g, (hipStream_t)s));
  return FVM_OK;
}

int fvm_ell_resident(int64_t n, int32_t* fits) {
  FVM_CHECK(fits, "fvm_ell_resident: null output");
  *fits = 0;
  if (n <= 0 || n > kMaxN) return FVM_OK;
  for (int w : {0, 4, 5, 6, 7, 8, 9, 10}) {
    bool a, b;
    FVM_HIP(fvm::grid_fits(FVM_TRB_KERNEL(trbdf2_affine_kernel, w), kRows, workgroups(n), &a));
    FVM_HIP(fvm::grid_fits(FVM_TRB_KERNEL(gmres_kernel, w), kRows, workgroups(n), &b));
    if (!a || !b) return FVM_OK;
  }
  *fits = 1;
  return FVM_OK;
}

int fvm_gmres_iterations(const void* d_work, int64_t* iterations, fvm_stream s) {
  FVM_CHECK(d_work && iterations, "fvm_gmres_iterations: null argument");
  uint64_t h[fvm::kGridHead];
  FVM_HIP(hipMemcpyAsync(h, d_work, sizeof h, hipMemcpyDeviceToHost, (hipStream_t)s));
  FVM_HIP(hipStreamSynchronize((hipStream_t)s));
  if (h[fvm::kGridFault]) {
    fvm::set_error("fvm_gmres_ell: the grid's exchange timed out");
    return FVM_ERR_HIP;
  }
  *iterations = (int64_t)h[fvm::kGridUser];
  return FVM_OK;
}

int fvm_jacobian_ell(fvm_ctx* ctx, int32_t n_colours, const double* const* d_probes, const uint8_t* d_colour,
                     int32_t width, const double* d_u, double t, double* d_products, double* d_val,
                     double* d_diag, fvm_stream s) {
  FVM_CHECK(ctx && d_probes && d_colour && d_u && d_products && d_val && d_diag, "fvm_jacobian_ell: null argument");
  FVM_CHECK(n_colours >= 1 && n_colours < 255 && width >= 1, "fvm_jacobian_ell: 1..254 colours and width >= 1");
  const int64_t n = ctx->m->N;
  for (int c = 0; c < n_colours; ++c) {
    FVM_CHECK(d_probes[c], "fvm_jacobian_ell: null probe");
    const int rc = fvm_jvp(ctx, d_u, d_probes[c], d_products + c * n, t, s);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(ell_from_probes, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)s, n, width,
                     d_colour, d_products, d_val, d_diag);
  FVM_HIP(hipGetLastError());
  return FVM_OK;
}

}  // extern "C"
