// Arguments of the one-launch Tsit5 loop over a small ODE template (fvm_tsit5.hip).
#pragma once
#include <functional>

#include "fvm_internal.hpp"

namespace fvm {

// What the loop itself takes (fvm_tsit5_loop.hpp).
struct Tsit5Loop {
  int64_t n;
  double t0, tf, dt;
  double abstol, reltol;
  int64_t maxiters, it0;
  int32_t fsal, dirichlet;
  int64_t n_save, ks0;
  const double* save_t;  // device copy
  double* saves;
  const double* k0;      // f(u) on entry
  const double* u;       // the state on entry
  double* u_out;
  double* stats;         // [0] t, [1] naccept, [2] nreject, [3] nf, [4] nsaved, [5] retcode
  double A[7][6], Bt[7], C[7];
};

// The options' part of a, its device memory (words of exchange memory, zeroed, to *grid
// before launch()), the launch and the results to st; FVM_ERR_STATE, nothing done, when the
// runtime refuses the grid.
int tsit5_run(Tsit5Loop& a, size_t words, uint64_t** grid, const fvm_ode_opts* o, const std::function<hipError_t()>& launch,
              fvm_ode_stats* st, hipStream_t s);

struct SmallTsit5 : Tsit5Loop {
  // the sliced ELL copy of A (fvm_template): W unrolled slots, one of ecol / eoff
  int W;
  const int32_t* off;
  const uint8_t* perm;
  const int32_t* rem_ptr;
  const int32_t* rem_off;
  const int32_t* ecol;
  const int16_t* eoff;
  const double* eval;
  const double* diag;
  const double* b;
  bool long_rows;    // some rows have more than W entries off the diagonal
  uint64_t* grid;    // the grid form's exchange memory, zeroed
};

constexpr int kTsit5MaxW = 10;            // unrolled slots of the operators, at most
constexpr int64_t kTsit5GridMax = 65536;  // rows of the grid form (256 workgroups of 256)
// rows of the one-workgroup form for an ELL width, at most
int64_t tsit5_rows_local_max(int W);
// 8-byte words of exchange memory of the grid form
size_t tsit5_rows_grid_words(int64_t n);
// whether the device holds the grid form's workgroups at once
hipError_t tsit5_rows_fits(int64_t n, int W, bool long_rows, bool* fits);
hipError_t tsit5_rows(SmallTsit5& a, bool local, hipStream_t s);

}  // namespace fvm
