// Smoothed-aggregation multigrid for the template operators M (fvm_amg.hip), as the
// preconditioner of the conjugate gradients in fvm_linalg.hip.
#pragma once
#include <vector>

#include "fvm_internal.hpp"

namespace fvm {

// A sparse matrix by rows: CSR (rp given), or kAmgRow places per row, cnt of them used.
constexpr int kAmgRow = 48;  // entries per row of a coarse operator, at most
constexpr int kAmgQ = 16;    // entries per row of Q, at most (the transposed lists' keys hold 4 bits of it)
// Rows of an operator, at most: the transposed lists' starts are int32, their keys row << 4 | slot.
constexpr int64_t kAmgMaxRows = INT32_MAX / kAmgQ;
static_assert(kAmgMaxRows * kAmgQ <= INT32_MAX && kAmgMaxRows < ((int64_t)1 << 28) && kAmgQ <= 16, "int32 lists");

struct AmgMat {
  int64_t n = 0;
  const int32_t* rp = nullptr;
  const int32_t* cnt = nullptr;
  const int32_t* col = nullptr;
  const double* val = nullptr;
  __device__ __forceinline__ int len(int64_t i) const { return rp ? rp[i + 1] - rp[i] : cnt[i]; }
  __device__ __forceinline__ int64_t at(int64_t i, int k) const { return rp ? (int64_t)rp[i] + k : i * kAmgRow + k; }
};

// One level and its transfer to the next.  Q = (I - S A) P, qcnt entries of row i at
// i qi + k qk (slot-major on the first level, where a thread takes a row, row-major on
// the others, where a group of lanes does), and its transpose by rows, values in FP32:
// the cycle only preconditions; s the smoothing weights.
struct AmgLevel {
  AmgMat A;
  double* s = nullptr;
  uint8_t* qcnt = nullptr;
  int32_t* qcol = nullptr;
  float* qv = nullptr;
  int64_t qi = 0, qk = 0;
  int64_t nc = 0;  // rows of the next level, 0: the coarsest
  int32_t* qtp = nullptr;
  int32_t* qti = nullptr;
  float* qtv = nullptr;
  double *b = nullptr, *x = nullptr;  // right-hand side and correction (levels > 0)
};

struct Amg {
  std::vector<AmgLevel> level;
  std::vector<void*> mem;
  double* inverse = nullptr;  // dense inverse of the coarsest operator, when it is small
  int tail = 0;               // first level of the one-workgroup tail kernel
  double seconds = 0.0;       // set-up time
  ~Amg();
};

// Sets up the hierarchy of M (n rows, CSR on the device); *out stays null where the
// operator does not coarsen.
int amg_build(int64_t n, const int32_t* rp, const int32_t* col, const double* val, Amg** out, hipStream_t s);
// The correction of the levels below the first from level 1's right-hand side b
// (which the caller has restricted into level[1].b): level[1].x.  Kernels return at
// once when *done is nonzero.
void amg_coarse(const Amg* a, const double* done, hipStream_t s);
}  // namespace fvm
