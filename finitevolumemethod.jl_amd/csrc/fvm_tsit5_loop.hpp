// The Tsit5 loop of fvm_ode_solve inside a kernel: stages, error norm, step control,
// saves and first same as last, for the one-launch forms (fvm_tsit5.hip,
// fvm_tsit5_mesh.hip).  Every element's arithmetic is the multi-kernel path's.
#pragma once
#include "fvm_ctrl.hpp"
#include "fvm_grid.hpp"
#include "fvm_tsit5.hpp"

namespace fvm {

constexpr int kBlk = 256;        // elements per partial sum of the error norm
constexpr int kDppShl4 = 0x104, kDppShl2 = 0x102, kDppShl1 = 0x101;

// Lane 0: the wave's sum in the order of shuffles down by 32, 16, 8, 4, 2, 1.
__device__ __forceinline__ double wave_tree(double x) {
  x = half_sums<32>(x, x);
  x = half_sums<16>(x, x);
  x += dpp<kDppRor8>(x);
  x += dpp<kDppShl4>(x);
  x += dpp<kDppShl2>(x);
  return x + dpp<kDppShl1>(x);
}

__device__ __forceinline__ double first_lane(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// ctrl_pow's operations with its divisions by small integers as Markstein's corrected
// products (div_rn: the same quotients bit for bit): 20 dependent divisions are 2 us of
// latency in a step of 7 us.
__device__ __forceinline__ double step_pow(double x, double p) {
  const double y = p * ctrl_log(x);
  const double k = floor(y / 0.69314718055994531 + 0.5);
  const double r = y - k * 0.69314718055994531;
  double e = 1.0;
#pragma unroll
  for (int i = 20; i >= 1; --i) e = 1.0 + div_rn(e * r, (double)i, 1.0 / (double)i);
  return ldexp(e, (int)k);
}

// One wave: p[q] = partial sum lane + 64 q of the nb that the grid's workgroups have put
// into the sums' words.
template <int T>
__device__ __forceinline__ void grid_parts(Grid<T>& G, int nb, double (&p)[4]) {
  const int lane = threadIdx.x & 63;
  const uint32_t P = G.sums();
#pragma nounroll
  for (unsigned spin = 0;; ++spin) {
    uint32_t stale = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (lane + 64 * j < nb) {
        const grid_pair w = grid_get(G.view, P + 16u * (lane + 64 * j));
        stale |= grid_stale(w, G.rtag);
        p[j] = grid_value(w);
      }
    if (__all(stale == 0)) break;
    if (G.waited_long(spin)) {
      if (lane == 0) G.give_up();
      break;
    }
  }
}

// row(r): the thread's r-th element, n or more for none; u_of(r): its state; k[0] = f on
// entry.  apply(x, out, t): out = f(x, t), x handed to the other threads first;
// norm_sum(q): the sum over the elements in the multi-kernel path's order;
// dirichlet(u, t): the element's state after the callback.  kRolled: apply stands once in
// a loop over the stages, for right-hand sides of much code.  up: false once the grid has
// given up.
template <int RPT, bool kRolled, class U, class Row, class Apply, class Norm, class Dir>
__device__ __forceinline__ void tsit5_loop(const Tsit5Loop& a, double (&k)[7][RPT], double (&un)[RPT], U u_of, Row row,
                                           Apply apply, Norm norm_sum, Dir dirichlet, const bool& up) {
  const int lane = threadIdx.x & 63;
  double t = a.t0, dt = a.dt, qold = 1e-4;
  int64_t it = a.it0, ks = a.ks0, naccept = 0, nreject = 0, nf = 0;
  int retcode = FVM_ODE_SUCCESS;
  int j0 = 1;  // kRolled: 0 when k[0] has to be formed first
  auto combine = [&](int j) {
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      double v = 1.0 * u_of(r);
#pragma unroll
      for (int i = 0; i < j; ++i) v = v + dt * a.A[j][i] * k[i][r];
      un[r] = v;
    }
  };
  while (t < a.tf && it < a.maxiters) {
    ++it;
    dt = fmin(dt, a.tf - t);
    if constexpr (kRolled) {
#pragma nounroll
      for (int j = j0; j < 7; ++j) {
        double f[RPT];
#pragma unroll
        for (int q = 0; q < 7; ++q)
          if (q == j) combine(q);
        apply(un, f, t + a.C[j] * dt);
#pragma unroll
        for (int q = 0; q < 7; ++q)
          if (q == j) {
#pragma unroll
            for (int r = 0; r < RPT; ++r) k[q][r] = f[r];
          }
      }
      nf += 6;
      j0 = 1;
    } else {
#pragma unroll
      for (int j = 1; j < 7; ++j) {
        combine(j);
        apply(un, k[j], t + a.C[j] * dt);
        ++nf;
      }
    }
    // the error norm: per element r = (sum_j dt bt_j k_j) / (abstol + reltol max(|u|, |unew|))
    double q2[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      double v = dt * a.Bt[0] * k[0][r];
#pragma unroll
      for (int j = 1; j < 7; ++j) v = v + dt * a.Bt[j] * k[j][r];
      const double sc = a.abstol + a.reltol * fmax(fabs(u_of(r)), fabs(un[r]));
      const double e = v / sc;
      q2[r] = row(r) < a.n ? e * e : 0.0;
    }
    const double EEst = sqrt(norm_sum(q2) / (double)a.n);
    if (!up) break;
    if (!isfinite(EEst)) {
      retcode = FVM_ODE_UNSTABLE;
      break;
    }
    // max(EEst, 1e-16)^(7/50) in the even lanes, qold^(2/25) in the odd ones
    const double pw = step_pow(lane & 1 ? qold : fmax(EEst, 1e-16), lane & 1 ? 2.0 / 25.0 : 7.0 / 50.0);
    const double pe = first_lane(pw), po = first_lane(dpp<kDppXor1>(pw));
    if (EEst <= 1.0) {
      const double tn = t + dt;
      while (ks < a.n_save && a.save_t[ks] <= tn + 1e-12 * fmax(1.0, fabs(tn))) {
        const double th = fmin(1.0, fmax(0.0, (a.save_t[ks] - t) / dt));
        const double t2 = th * th, t3 = t2 * th;
        const double h00 = 2 * t3 - 3 * t2 + 1;
        const double h10 = t3 - 2 * t2 + th;
        const double h01 = -2 * t3 + 3 * t2;
        const double h11 = t3 - t2;
        const double c0 = h00, c1 = h10 * dt, c2 = h01, c3 = h11 * dt;
#pragma unroll
        for (int r = 0; r < RPT; ++r) {
          const int64_t i = row(r);
          double v = c0 * u_of(r);
          v = v + c1 * k[0][r];
          v = v + c2 * un[r];
          v = v + c3 * k[6][r];
          if (i < a.n) a.saves[ks * a.n + i] = v;
        }
        ++ks;
      }
#pragma unroll
      for (int r = 0; r < RPT; ++r) u_of(r) = dirichlet(un[r], tn);
      t = tn;
      ++naccept;
      if (a.fsal && (!a.dirichlet || naccept >= 2)) {
#pragma unroll
        for (int r = 0; r < RPT; ++r) k[0][r] = k[6][r];
      } else if constexpr (kRolled) {
        j0 = 0;
        ++nf;
      } else {
        apply(un, k[0], t);
        ++nf;
      }
      double q = pe / po;
      q = fmin(5.0, fmax(0.1, q / 0.9));
      dt = dt / q;
      qold = fmax(EEst, 1e-4);
    } else {
      ++nreject;
      const double q = fmin(5.0, pe / 0.9);
      dt = dt / q;
    }
  }
  if (retcode == FVM_ODE_SUCCESS && !(t >= a.tf)) retcode = FVM_ODE_MAXITERS;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int64_t i = row(r);
    if (i < a.n) a.u_out[i] = u_of(r);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.stats[0] = t;
    a.stats[1] = (double)naccept;
    a.stats[2] = (double)nreject;
    a.stats[3] = (double)nf;
    a.stats[4] = (double)ks;
    a.stats[5] = up ? (double)retcode : -1.0;
  }
}

}  // namespace fvm
