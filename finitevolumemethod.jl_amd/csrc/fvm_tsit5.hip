// Tsit5 on a small ODE template du/dt = A u + b in one launch: the adaptive loop of
// fvm_ode_solve (fvm_ode.hip) with stages, products, error norm, step control, saveat
// and first same as last inside the kernel.
//
// Layout: each thread holds its rows in registers for the whole integration: the state,
// the seven stages, the row of A and b.  A stage hands the combined state to the other
// rows and gathers the row's neighbours; nothing else leaves the registers.  Two forms:
//   one workgroup (kLocal): up to five rows per thread, the state exchanged through LDS
//     (double buffered: one barrier per stage);
//   a resident grid: one row per thread, the state exchanged through fvm_grid.hpp's
//     words (1.3 to 2 us per stage, whatever n).
// Both are bound by latency: 11 us a step at 2,500 rows in one workgroup (six barriers
// and LDS gathers, the error norm's trees, the controller's power), 14 us at 2,601 rows
// and 20 us at 62,500 on the grid.  The same loop with its vectors in memory took 57 us a
// step at 2,500 rows in one workgroup, and about 80 us of launches a step above that.
// The 50 x 50 plate to t = 0.5 (88 steps): 4.92 -> 0.97 ms.
//
// Every element's arithmetic is the multi-kernel path's: the row products in
// sell_slice's order, the linear combinations with their terms left to right, the
// error norm summed in the order of that path's 512 x 256 grid, and the step
// controller's power fvm_ctrl.hpp's: the same states bit for bit.
#include <algorithm>
#include <cmath>

#include "fvm_grid.hpp"
#include "fvm_tsit5.hpp"

using namespace fvm;

namespace {

constexpr int kBlk = 256;        // elements per partial sum of the error norm
constexpr int kSlice = 64;       // rows per slice of the sliced ELL form
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

// The rows of one thread: W off-diagonal slots (padding: the row itself, value 0) as
// where to find the neighbour and value.  kLocal: two 16-bit LDS byte offsets per register,
// taken apart at every use (hoisted out of the loop they would fill the registers twice).
template <int W, int RPT, bool kLocal>
struct Rows {
  static constexpr int C = kLocal ? W / 2 : W;
  uint32_t c[RPT][C];
  double v[RPT][W], diag[RPT];
};

template <int T, int RPT, bool kLocal>
struct Lds {
  double X[kLocal ? 2 * T * RPT : 1];   // the exchanged state
  double u[kLocal ? T * RPT : 1], b[kLocal ? T * RPT : 1];
  double tree[RPT][T];
  double part[kLocal ? 64 : 1];
  GridShared<T> grid;
};

template <int W, int T, int RPT, bool kLocal>
__global__ __launch_bounds__(T) void tsit5_rows_kernel(SmallTsit5 a) {
  static_assert(W % 2 == 0 && (kLocal || RPT == 1) && T * RPT <= 8192, "layout");
  __shared__ Lds<T, RPT, kLocal> S;
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t n = a.n;
  const int64_t i0 = (int64_t)blockIdx.x * T + tid;  // the thread's rows: i0 + r T
  Grid<T> G;
  if (!kLocal) G.open(a.grid, n, &S.grid);
  int xbuf = 0;
  bool up = true;

  // the lane that holds each of the wave's rows inside its slice: the inverse of sl_perm
  auto slot_of = [&](int64_t i) {
    const int at = i < n ? (int)a.perm[i] : lane;
    return __builtin_amdgcn_ds_permute(at << 2, lane);
  };
  Rows<W, RPT, kLocal> R;
  double u0 = 0.0, b0 = 0.0;   // one row per thread: the state and b in registers
  double k[7][RPT], un[RPT];
  uint32_t longer = 0;         // slices with rows longer than the operator's W slots, bit r
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int64_t i = i0 + (int64_t)r * T, b = i / kSlice;
    const bool in = i < n;
    const int pos = slot_of(i);
#pragma unroll
    for (int s = 0; s < W; ++s) {
      const int e0 = in && s < a.W ? a.off[(a.W + 1) * b + s] : 0;
      const int e1 = in && s < a.W ? a.off[(a.W + 1) * b + s + 1] : 0;
      const bool on = e0 + pos < e1;
      const int c = on ? (a.eoff ? (int)i + (int)a.eoff[e0 + pos] : a.ecol[e0 + pos]) : (in ? (int)i : 0);
      if (!kLocal) R.c[r][s] = grid_offset(c);
      else if (s % 2 == 0) R.c[r][s / 2] = (uint32_t)c * 8u;
      else R.c[r][s / 2] |= (uint32_t)c << 19;
      R.v[r][s] = on ? a.eval[e0 + pos] : 0.0;
    }
    R.diag[r] = in ? a.diag[i] : 0.0;
    k[0][r] = in ? a.k0[i] : 0.0;
    (kLocal ? S.u[tid + r * T] : u0) = in ? a.u[i] : 0.0;
    (kLocal ? S.b[tid + r * T] : b0) = in ? a.b[i] : 0.0;
    if (__any(in && a.rem_ptr[b + 1] > a.rem_ptr[b])) longer |= 1u << r;
  }
  auto u_of = [&](int r) -> double& { return kLocal ? S.u[tid + r * T] : u0; };

  // out = A x + b on the thread's rows, x handed to the other rows first
  auto apply = [&](const double (&x)[RPT], double (&out)[RPT]) {
    double* const X = S.X + (kLocal ? xbuf * T * RPT : 0);
    if (kLocal) {
#pragma unroll
      for (int r = 0; r < RPT; ++r) X[tid + r * T] = x[r];
      xbuf ^= 1;
      __syncthreads();
    } else {
      G.publish(i0, x[0], i0 < n);
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      double xc[W];
      if constexpr (kLocal) {
#pragma unroll
        for (int s = 0; s < W; s += 2) {
          uint32_t w = R.c[r][s / 2];
          asm volatile("" : "+v"(w));
          xc[s] = *(const double*)((const char*)X + (w & 0xffffu));
          xc[s + 1] = *(const double*)((const char*)X + (w >> 16));
        }
      } else {
        G.fetch(R.c[r], xc, i0 < n);
      }
      double acc = 0.0;
#pragma unroll
      for (int s = 0; s < W; ++s) acc += R.v[r][s] * xc[s];
      if (longer & (1u << r)) {
        const int64_t i = i0 + (int64_t)r * T, b = i / kSlice;
        const int pos = slot_of(i);
        if (i < n) {
          int st = a.off[(a.W + 1) * b + a.W];
          for (int q = a.rem_ptr[b]; q < a.rem_ptr[b + 1]; ++q) {
            const int e = st + pos;
            if (e < a.rem_off[q]) {
              const int c = a.eoff ? (int)i + (int)a.eoff[e] : a.ecol[e];
              acc += a.eval[e] * (kLocal ? X[c] : G.fetch1(c));
            }
            st = a.rem_off[q];
          }
        }
      }
      acc += R.diag[r] * (kLocal ? X[tid + r * T] : x[r]);
      out[r] = acc + (kLocal ? S.b[tid + r * T] : b0);
      // rows one after the other: all rows' gathers at once would spill
      if (kLocal) __builtin_amdgcn_sched_barrier(0);
    }
  };

  // sum over the grid's rows of q[r], in the order of 512 workgroups of 256 threads
  // and their sum by one more: pairwise trees of 256 elements, then of the partial sums
  auto norm_sum = [&](const double (&q)[RPT]) -> double {
    const int lt = tid % kBlk;
#pragma unroll
    for (int r = 0; r < RPT; ++r) S.tree[r][tid] = q[r];
    __syncthreads();
    if (lt < 64) {
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        const double v = (S.tree[r][tid] + S.tree[r][tid + 128]) + (S.tree[r][tid + 64] + S.tree[r][tid + 192]);
        const double t = wave_tree(v);
        if (lt == 0) {
          if (kLocal) S.part[(tid + r * T) / kBlk] = t;
          else grid_put(G.view, G.sums() + 16u * (uint32_t)(i0 / kBlk), t, G.rtag);
        }
      }
    }
    double p[4] = {0.0, 0.0, 0.0, 0.0};  // partial sums lane, lane + 64, ...
    if (kLocal) {
      __syncthreads();
      if (lane < T * RPT / kBlk) p[0] = S.part[lane];
    } else {
      if (tid < 64) {
        const int nb = (int)((n + kBlk - 1) / kBlk);
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
    }
    const double t = wave_tree((p[0] + p[2]) + (p[1] + p[3]));
    if (kLocal) return first_lane(t);
    if (tid == 0) S.part[0] = t;
    __syncthreads();
    up = S.grid.fault == 0;
    return S.part[0];
  };

  double t = a.t0, dt = a.dt, qold = 1e-4;
  int64_t it = a.it0, ks = a.ks0, naccept = 0, nreject = 0, nf = 0;
  int retcode = FVM_ODE_SUCCESS;
  while (t < a.tf && it < a.maxiters) {
    ++it;
    dt = fmin(dt, a.tf - t);
#pragma unroll
    for (int j = 1; j < 7; ++j) {
#pragma unroll
      for (int r = 0; r < RPT; ++r) {
        double v = 1.0 * u_of(r);
#pragma unroll
        for (int i = 0; i < j; ++i) v = v + dt * a.A[j][i] * k[i][r];
        un[r] = v;
      }
      apply(un, k[j]);
      ++nf;
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
      q2[r] = i0 + (int64_t)r * T < n ? e * e : 0.0;
    }
    if (!kLocal) ++G.rtag;
    const double EEst = sqrt(norm_sum(q2) / (double)n);
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
          const int64_t i = i0 + (int64_t)r * T;
          double v = c0 * u_of(r);
          v = v + c1 * k[0][r];
          v = v + c2 * un[r];
          v = v + c3 * k[6][r];
          if (i < n) a.saves[ks * n + i] = v;
        }
        ++ks;
      }
#pragma unroll
      for (int r = 0; r < RPT; ++r) u_of(r) = un[r];
      t = tn;
      ++naccept;
      if (a.fsal) {
#pragma unroll
        for (int r = 0; r < RPT; ++r) k[0][r] = k[6][r];
      } else {
        apply(un, k[0]);
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
    const int64_t i = i0 + (int64_t)r * T;
    if (i < n) a.u_out[i] = u_of(r);
  }
  if (blockIdx.x == 0 && tid == 0) {
    a.stats[0] = t;
    a.stats[1] = (double)naccept;
    a.stats[2] = (double)nreject;
    a.stats[3] = (double)nf;
    a.stats[4] = (double)ks;
    a.stats[5] = up ? (double)retcode : -1.0;
  }
}

constexpr int kLocalT = 512, kGridT = 256;

template <int W, int RPT>
hipError_t run_local(SmallTsit5& a, hipStream_t s) {
  hipLaunchKernelGGL((tsit5_rows_kernel<W, kLocalT, RPT, true>), dim3(1), dim3(kLocalT), 0, s, a);
  return hipGetLastError();
}

template <int W, int T>
hipError_t run_grid(SmallTsit5& a, hipStream_t s) {
  void* args[] = {&a};
  return hipLaunchCooperativeKernel((const void*)tsit5_rows_kernel<W, T, 1, false>, dim3((unsigned)((a.n + T - 1) / T)),
                                    dim3(T), args, 0, s);
}

// rows per thread of the one-workgroup form, at most: what its registers hold
template <int W>
hipError_t run(SmallTsit5& a, bool local, hipStream_t s) {
  if (!local) return run_grid<W, kGridT>(a, s);
  const int rows = (int)((a.n + kLocalT - 1) / kLocalT);
  if (rows <= 2) return run_local<W, 2>(a, s);
  return rows <= 4 ? run_local<W, 4>(a, s) : run_local<W, W <= 6 ? 5 : 4>(a, s);
}

}  // namespace

namespace fvm {

int64_t tsit5_rows_local_max(int W) { return (int64_t)kLocalT * (W <= 6 ? 5 : 4); }

size_t tsit5_rows_grid_words(int64_t n) { return grid_words(n); }

hipError_t tsit5_rows(SmallTsit5& a, bool local, hipStream_t s) {
  if (a.W <= 6) return run<6>(a, local, s);
  if (a.W <= 8) return run<8>(a, local, s);
  return run<10>(a, local, s);
}

}  // namespace fvm
