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
#include "fvm_grid.hpp"
#include "fvm_tsit5.hpp"
#include "fvm_tsit5_loop.hpp"

using namespace fvm;

namespace {

constexpr int kSlice = 64;       // rows per slice of the sliced ELL form

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

// kLong: there are rows longer than the operator's W slots (hubs); a form of its own, for its
// registers (the others need 6 to 40 fewer without it, and spill none).
template <int W, int T, int RPT, bool kLocal, bool kLong>
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
  uint32_t longer = 0;         // kLong: slices with such rows, bit r
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
    if (kLong && __any(in && a.rem_ptr[b + 1] > a.rem_ptr[b])) longer |= 1u << r;
  }
  auto u_of = [&](int r) -> double& { return kLocal ? S.u[tid + r * T] : u0; };

  // out = A x + b on the thread's rows, x handed to the other rows first
  auto apply = [&](const double (&x)[RPT], double (&out)[RPT], double) {
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
      if (kLong && longer & (1u << r)) {
        const int64_t i = i0 + (int64_t)r * T, b = i / kSlice;
        const int pos = slot_of(i);
        if (i < n) {
          // eight entries' loads in flight (absent ones load entry 0), added in their order:
          // 20 steps with a hub of 300 on 661 rows 7.6 -> 2.5 ms (one by one against eight), on
          // 3,661 rows (the grid) 13.0 -> 4.8 ms; the multi-kernel loop takes 7.5
          constexpr int K = 8;
          int st = a.off[(a.W + 1) * b + a.W];
          const int q1 = a.rem_ptr[b + 1];
          for (int q = a.rem_ptr[b]; q < q1; q += K) {
            int e[K], c[K];
            double v[K], xc[K];
            uint32_t on = 0, o[K];
#pragma unroll
            for (int s = 0; s < K; ++s) {
              const int end = a.rem_off[q + s < q1 ? q + s : q1 - 1];
              const bool here = q + s < q1 && st + pos < end;
              on |= (uint32_t)here << s;
              e[s] = here ? st + pos : 0;
              st = end;
            }
            if (a.eoff) {
#pragma unroll
              for (int s = 0; s < K; ++s) c[s] = (int)i + (int)a.eoff[e[s]];
            } else {
#pragma unroll
              for (int s = 0; s < K; ++s) c[s] = a.ecol[e[s]];
            }
#pragma unroll
            for (int s = 0; s < K; ++s) v[s] = a.eval[e[s]];
#pragma unroll
            for (int s = 0; s < K; ++s) {
              if (!(on >> s & 1)) c[s] = (int)i;
              if (kLocal) xc[s] = X[c[s]];
              else o[s] = grid_offset(c[s]);
            }
            if constexpr (!kLocal) G.fetch(o, xc, true);
#pragma unroll
            for (int s = 0; s < K; ++s)
              if (on >> s & 1) acc += v[s] * xc[s];
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
    if (!kLocal) ++G.rtag;
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
      if (tid < 64) grid_parts(G, (int)((n + kBlk - 1) / kBlk), p);
    }
    const double t = wave_tree((p[0] + p[2]) + (p[1] + p[3]));
    if (kLocal) return first_lane(t);
    if (tid == 0) S.part[0] = t;
    __syncthreads();
    up = S.grid.fault == 0;
    return S.part[0];
  };

  auto row = [&](int r) { return i0 + (int64_t)r * T; };
  auto no_dirichlet = [](double x, double) { return x; };
  tsit5_loop<RPT, false>(a, k, un, u_of, row, apply, norm_sum, no_dirichlet, up);
}

constexpr int kLocalT = 512, kGridT = 256;

template <int W, int RPT, bool kLong>
hipError_t run_local(SmallTsit5& a, hipStream_t s) {
  hipLaunchKernelGGL((tsit5_rows_kernel<W, kLocalT, RPT, true, kLong>), dim3(1), dim3(kLocalT), 0, s, a);
  return hipGetLastError();
}

// (rows are longer than W slots only where W is the operators' most, kTsit5MaxW)
const void* grid_kernel(int W, bool long_rows) {
  if (W <= 6) return (const void*)tsit5_rows_kernel<6, kGridT, 1, false, false>;
  if (W <= 8) return (const void*)tsit5_rows_kernel<8, kGridT, 1, false, false>;
  if (!long_rows) return (const void*)tsit5_rows_kernel<kTsit5MaxW, kGridT, 1, false, false>;
  return (const void*)tsit5_rows_kernel<kTsit5MaxW, kGridT, 1, false, true>;
}
int64_t grid_wgs(int64_t n) { return (n + kGridT - 1) / kGridT; }

// rows per thread of the one-workgroup form, at most: what its registers hold
template <int W, bool kLong>
hipError_t run(SmallTsit5& a, hipStream_t s) {
  const int rows = (int)((a.n + kLocalT - 1) / kLocalT);
  if (rows <= 2) return run_local<W, 2, kLong>(a, s);
  return rows <= 4 ? run_local<W, 4, kLong>(a, s) : run_local<W, W <= 6 ? 5 : 4, kLong>(a, s);
}

}  // namespace

namespace fvm {

int64_t tsit5_rows_local_max(int W) { return (int64_t)kLocalT * (W <= 6 ? 5 : 4); }

int tsit5_run(Tsit5Loop& a, size_t words, uint64_t** grid, const fvm_ode_opts* o, const std::function<hipError_t()>& launch,
              fvm_ode_stats* st, hipStream_t s) {
  a.tf = o->tf;
  a.abstol = o->abstol;
  a.reltol = o->reltol;
  a.maxiters = o->maxiters;
  a.fsal = o->fsal;
  a.n_save = o->n_save;
  a.saves = o->d_saves;
  // exchange words of the grid forms, save times, 6 result slots
  double* dev = nullptr;
  FVM_HIP(dev_alloc((void**)&dev, sizeof(double) * (words + (size_t)o->n_save + 6)));
  *grid = (uint64_t*)dev;
  a.save_t = dev + words;
  a.stats = dev + words + o->n_save;
  hipError_t e = hipSuccess;
  if (words) e = hipMemsetAsync(dev, 0, sizeof(double) * words, s);
  if (e == hipSuccess && o->n_save > 0)
    e = hipMemcpyAsync(dev + words, o->save_t, sizeof(double) * (size_t)o->n_save, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = launch();
  const bool refused = e == hipErrorCooperativeLaunchTooLarge;
  double r[6] = {0, 0, 0, 0, 0, 0};
  if (e == hipSuccess) e = hipMemcpyAsync(r, a.stats, sizeof r, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)dev_free(dev);
  if (refused) {  // fewer resident workgroups than grid_fits was told: the multi-kernel loop
    (void)hipGetLastError();
    return FVM_ERR_STATE;
  }
  if (e != hipSuccess) return hip_fail(e, "fvm_ode_solve (one-launch Tsit5)");
  if (r[5] < 0) {
    set_error("fvm_ode_solve: the grid's exchange timed out");
    return FVM_ERR_HIP;
  }
  st->t = r[0];
  st->naccept += (int64_t)r[1];
  st->nreject += (int64_t)r[2];
  st->nf += (int64_t)r[3];
  st->nsaved = (int64_t)r[4];
  st->retcode = (int32_t)r[5];
  return FVM_OK;
}

size_t tsit5_rows_grid_words(int64_t n) { return grid_words(n); }

hipError_t tsit5_rows_fits(int64_t n, int W, bool long_rows, bool* fits) {
  return grid_fits(grid_kernel(W, long_rows), kGridT, grid_wgs(n), fits);
}

hipError_t tsit5_rows(SmallTsit5& a, bool local, hipStream_t s) {
  if (!local) {
    void* args[] = {&a};
    return hipLaunchCooperativeKernel(grid_kernel(a.W, a.long_rows), dim3((unsigned)grid_wgs(a.n)), dim3(kGridT), args, 0, s);
  }
  if (a.W <= 6) return run<6, false>(a, s);
  if (a.W <= 8) return run<8, false>(a, s);
  return a.long_rows ? run<kTsit5MaxW, true>(a, s) : run<kTsit5MaxW, false>(a, s);
}

}  // namespace fvm
