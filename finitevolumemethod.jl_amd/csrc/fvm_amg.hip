// Smoothed-aggregation multigrid (Vanek, Mandel & Brezina, Computing 56, 1996) for the
// template operators, set up and applied on the device.
//
// Jacobi-preconditioned CG needs a number of iterations that grows like the side of the
// mesh: 3,800 on 1000 x 1000 jittered nodes, with this preconditioner 44 (and the three
// Jacobi steps before it).  A solve there takes 9.2 ms instead of 158, the first one of a
// template 14.5 with the set-up (5 ms: half of it sorting and summing the first level's
// lists, bound by the latency of its gathers).
//
// Set-up, per level:
//   weights   s_i = 1.8 / sum_j |a_ij|: Jacobi with 0.9 of the inverse diagonal on an
//             M-matrix, and convergent for any symmetric positive definite A (the
//             eigenvalues of D^-1 A with D the row sums of |A| do not exceed 1)
//   strength  a_ij^2 > theta^2 a_ii a_jj
//   roots     a maximal independent set at distance 2 of the strong graph (Bell, Dalton &
//             Olson, SIAM J. Sci. Comput. 34, 2012), by rounds of neighbourhood maxima of
//             hashed priorities; its neighbours and theirs join: the aggregates
//   P = (I - 1.6 D_F^-1 F) P0, P0 the aggregates' indicator, F the strong entries; A P;
//   Q = P - S A P;
//   A_c = P^T (A P), a row per thread, its sum in a fixed order (the transposed lists
//             are sorted), so that the hierarchy is the same bit for bit every time.
// Cycle.  One V-cycle with a Jacobi sweep before and after the coarse correction,
//   x = S b;  x += P A_c^-1 P^T (b - A x);  x += S (b - A x),
// is, for symmetric A, x = S (2 b - A S b) + Q A_c^-1 Q^T b: one pass over Q^T on the way
// down and one over A and Q on the way up, instead of two products with A, a restriction
// and a prolongation.  Of an iteration's 200 us on 1000 x 1000, the first level's passes
// take 100 (up 40, the product p.M p 30, down 19, update 12; by their counters 148, 94, 47
// and 51 MB of HBM traffic: 3.7, 3.2, 2.4 and 4.5 TB/s), the levels below 65, the gaps
// between the 11 launches the rest.  Levels of at most kTailRows rows and the coarsest one's dense
// inverse run in one workgroup, in one launch: smaller launches cost 3 to 4 us each and
// hold next to no work.
#include "fvm_amg.hpp"

#include <algorithm>
#include <chrono>

using namespace fvm;

namespace {

constexpr int kB = 256;
constexpr int kDense = 128;       // rows of the densely inverted coarsest operator, at most
constexpr int kTailRows = 1024;   // rows of a level in the one-workgroup tail, at most
constexpr int kTailLevels = 6;
constexpr int kMisRounds = 8;
constexpr double kTheta = 0.08;
constexpr int kTailThreads = 1024;
constexpr double kWeight = 1.8, kWeightP = 1.6;

__device__ __forceinline__ int wave_max(int x) {
  for (int o = 32; o > 0; o >>= 1) x = max(x, __shfl_xor(x, o, 64));
  return x;
}
inline dim3 grid1(int64_t n) { return dim3((unsigned)((n + kB - 1) / kB)); }
__device__ __forceinline__ int64_t gid() { return (int64_t)blockIdx.x * blockDim.x + threadIdx.x; }

// the integer mixer lowbias32 (C. Wellons, hash-prospector, 2018)
__device__ __forceinline__ uint32_t hash32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  return x ^ (x >> 16);
}

__global__ __launch_bounds__(kB) void weights_kernel(AmgMat A, double* __restrict__ d, double* __restrict__ s) {
  const int64_t i = gid();
  if (i >= A.n) return;
  double l1 = 0.0, di = 0.0;
  const int m = A.len(i);
  for (int k = 0; k < m; ++k) {
    const int64_t e = A.at(i, k);
    const double v = A.val[e];
    l1 += fabs(v);
    if (A.col[e] == i) di = v;
  }
  d[i] = di;
  s[i] = l1 > 0.0 ? kWeight / l1 : 0.0;
}

// Bit k of mask[i]: entry k of row i is strong (the first 64 entries; further ones count
// as weak).  t: state (2 root, 1 undecided, 0 out) << 62 | priority << 32 | index.
__global__ __launch_bounds__(kB) void strong_kernel(AmgMat A, const double* __restrict__ d, double theta2,
                                                    uint64_t* __restrict__ mask, uint64_t* __restrict__ t) {
  const int64_t i = gid();
  if (i >= A.n) return;
  const int m = min(A.len(i), 64);
  uint64_t w = 0;
  const double di = d[i];
  for (int k = 0; k < m; ++k) {
    const int64_t e = A.at(i, k);
    const int c = A.col[e];
    const double v = A.val[e];
    if (c != i && v * v > theta2 * di * d[c]) w |= 1ull << k;
  }
  mask[i] = w;
  t[i] = ((uint64_t)(w ? 1 : 0) << 62) | ((uint64_t)(hash32((uint32_t)i) >> 2) << 32) | (uint64_t)i;
}

// the largest of in over the strong neighbourhood
__device__ __forceinline__ uint64_t strong_max(const AmgMat& A, uint64_t w, int64_t i,
                                               const uint64_t* __restrict__ in) {
  uint64_t m = in[i];
  while (w) {
    const int k = __builtin_ctzll(w);
    w &= w - 1;
    const uint64_t v = in[A.col[A.at(i, k)]];
    m = v > m ? v : m;
  }
  return m;
}

__global__ __launch_bounds__(kB) void mis_max_kernel(AmgMat A, const uint64_t* __restrict__ mask,
                                                     const uint64_t* __restrict__ t, uint64_t* __restrict__ t1) {
  const int64_t i = gid();
  if (i < A.n) t1[i] = strong_max(A, mask[i], i, t);
}

__global__ __launch_bounds__(kB) void mis_decide_kernel(AmgMat A, const uint64_t* __restrict__ mask,
                                                        const uint64_t* __restrict__ t1, uint64_t* __restrict__ t) {
  const int64_t i = gid();
  if (i >= A.n) return;
  const uint64_t own = t[i];
  if (own >> 62 != 1) return;
  const uint64_t m = strong_max(A, mask[i], i, t1);
  const uint64_t low = own & ~(3ull << 62);
  if (m == own) t[i] = (2ull << 62) | low;
  else if (m >> 62 == 2) t[i] = low;
}

// ---- exclusive scan of int32 (blocks of 1024, at most 1024 * 1024 * 2 elements per pass)
constexpr int kScan = 1024;
__device__ __forceinline__ int scan1024(int v, int* sh, int* total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh[w] = x;
  __syncthreads();
  if (w == 0) {
    int y = lane < 16 ? sh[lane] : 0;
    for (int o = 1; o < 16; o <<= 1) {
      const int z = __shfl_up(y, o, 64);
      if (lane >= o) y += z;
    }
    if (lane < 16) sh[16 + lane] = y;
  }
  __syncthreads();
  *total = sh[31];
  const int r = x - v + (w ? sh[16 + w - 1] : 0);
  __syncthreads();
  return r;
}
// kind 0: in as it is; kind 1: 1 where the tuple is a root
template <int KIND>
__device__ __forceinline__ int scan_in(const void* in, int64_t i, int64_t n) {
  if (i >= n) return 0;
  return KIND == 0 ? ((const int32_t*)in)[i] : (int)(((const uint64_t*)in)[i] >> 62 == 2);
}
template <int KIND>
__global__ __launch_bounds__(kScan) void scan_sums_kernel(int64_t n, const void* in, int32_t* __restrict__ sums) {
  __shared__ int sh[32];
  int tot;
  scan1024(scan_in<KIND>(in, gid(), n), sh, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}
// one workgroup: sums -> exclusive starts, their total in sums[nb]
__global__ __launch_bounds__(kScan) void scan_blocks_kernel(int nb, int32_t* __restrict__ sums) {
  __shared__ int sh[32];
  int base = 0;
  for (int b0 = 0; b0 < nb; b0 += kScan) {
    const int i = b0 + threadIdx.x;
    int tot;
    const int ex = scan1024(i < nb ? sums[i] : 0, sh, &tot);
    if (i < nb) sums[i] = base + ex;
    base += tot;
  }
  if (threadIdx.x == 0) sums[nb] = base;
}
template <int KIND>
__global__ __launch_bounds__(kScan) void scan_out_kernel(int64_t n, const void* in, const int32_t* __restrict__ sums,
                                                         int32_t* __restrict__ out) {
  __shared__ int sh[32];
  int tot;
  const int64_t i = gid();
  const int ex = scan1024(scan_in<KIND>(in, i, n), sh, &tot);
  if (i < n) out[i] = sums[blockIdx.x] + ex;
}

// ---- aggregates
__global__ __launch_bounds__(kB) void join_roots_kernel(AmgMat A, const uint64_t* __restrict__ mask,
                                                        const uint64_t* __restrict__ t,
                                                        const int32_t* __restrict__ id, int32_t* __restrict__ agg) {
  const int64_t i = gid();
  if (i >= A.n) return;
  if (t[i] >> 62 == 2) {
    agg[i] = id[i];
    return;
  }
  int best = -1;
  double bv = 0.0;
  for (uint64_t w = mask[i]; w; w &= w - 1) {
    const int64_t e = A.at(i, __builtin_ctzll(w));
    const int c = A.col[e];
    const double v = fabs(A.val[e]);
    if (t[c] >> 62 == 2 && v > bv) {
      bv = v;
      best = id[c];
    }
  }
  agg[i] = best;
}

__global__ __launch_bounds__(kB) void join_rest_kernel(AmgMat A, const uint64_t* __restrict__ mask,
                                                       const int32_t* __restrict__ agg1, int32_t* __restrict__ agg) {
  const int64_t i = gid();
  if (i >= A.n) return;
  int best = agg1[i];
  if (best < 0) {
    double bv = 0.0;
    for (uint64_t w = mask[i]; w; w &= w - 1) {
      const int64_t e = A.at(i, __builtin_ctzll(w));
      const int a = agg1[A.col[e]];
      const double v = fabs(A.val[e]);
      if (a >= 0 && v > bv) {
        bv = v;
        best = a;
      }
    }
  }
  agg[i] = best;
}

// P = P0 - 1.6 F / (row sums of |F|) P0, F the operator with its weak entries lumped into
// the diagonal (filtered: the coarse operators stay near 15 entries a row instead of 30,
// at 5 % more iterations).  Rows of kP places.
constexpr int kP = 8;
__global__ __launch_bounds__(kB) void prolong_kernel(AmgMat A, const uint64_t* __restrict__ mask,
                                                     const int32_t* __restrict__ agg, uint8_t* __restrict__ pcnt,
                                                     int32_t* __restrict__ pcol, double* __restrict__ pv) {
  const int64_t i = gid();
  if (i >= A.n) return;
  const uint64_t w = mask[i];
  const int m = A.len(i);
  double dF = 0.0, l1 = 0.0;
  for (int k = 0; k < m; ++k) {
    const double a = A.val[A.at(i, k)];
    if (k < 64 && (w >> k & 1)) l1 += fabs(a);
    else dF += a;
  }
  l1 += fabs(dF);
  const double f = l1 > 0.0 ? kWeightP / l1 : 0.0;
  int32_t* const c = pcol + i * kP;
  double* const v = pv + i * kP;
  int np = 0;
  auto add = [&](int key, double x) {
    for (int q = 0; q < np; ++q)
      if (c[q] == key) {
        v[q] += x;
        return;
      }
    if (np < kP) {
      c[np] = key;
      v[np] = x;
      ++np;
    } else {
      v[0] += x;  // no place left: the weight stays with the row's own aggregate
    }
  };
  if (agg[i] >= 0) add(agg[i], 1.0 - f * dF);
  for (uint64_t u = w; u; u &= u - 1) {
    const int64_t e = A.at(i, __builtin_ctzll(u));
    const int g = agg[A.col[e]];
    if (g >= 0) add(g, -f * A.val[e]);
  }
  pcnt[i] = (uint8_t)np;
}

// Sums by column of a group of kG lanes, in a hash table of SLOTS places in LDS (open
// addressing).  add() is called by the whole group with distinct columns in its active
// lanes, one call after the other, so each column's sum has a fixed order and needs no
// atomic addition.
constexpr int kG = 16;
template <int SLOTS, int NV>
struct Sums {
  int32_t* key;
  double* val;  // [NV][SLOTS]
  __device__ __forceinline__ void clear(int lane) {
    for (int k = lane; k < SLOTS; k += kG) {
      key[k] = -1;
#pragma unroll
      for (int q = 0; q < NV; ++q) val[q * SLOTS + k] = 0.0;
    }
    fence();
  }
  static __device__ __forceinline__ void fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  __device__ __forceinline__ void add(bool on, int c, int q, double x) {
    if (on) {
      uint32_t h = ((uint32_t)c * 2654435761u) >> 8 & (SLOTS - 1);
      for (int tries = 0; tries < SLOTS; ++tries) {
        const int old = atomicCAS(key + h, -1, c);
        if (old == -1 || old == c) {
          val[q * SLOTS + h] += x;
          break;
        }
        h = (h + 1) & (SLOTS - 1);
      }  // a full table: the entry is left out
    }
    fence();
  }
};

__device__ __forceinline__ int group_ballot(bool p) {
  return (int)(__ballot(p) >> (threadIdx.x & 63 & ~(kG - 1)) & 0xffffu);
}

// The row of A P, then q = p - s (A P) on its pattern (kAmgQ entries: P's own columns,
// then the others); counts the columns' entries.  A group of lanes per row.
__global__ __launch_bounds__(kB) void smooth_kernel(AmgMat A, const double* __restrict__ s,
                                                    const uint8_t* __restrict__ pcnt,
                                                    const int32_t* __restrict__ pcol, const double* __restrict__ pv,
                                                    uint8_t* __restrict__ qcnt, int32_t* __restrict__ qcol,
                                                    float* __restrict__ qv, int64_t qi, int64_t qk,
                                                    int32_t* __restrict__ tcol, double* __restrict__ tp,
                                                    double* __restrict__ tap, int32_t* __restrict__ count) {
  constexpr int SL = 64, GR = kB / kG;
  __shared__ int32_t key[GR * SL];
  __shared__ double val[GR * 2 * SL];
  const int lane = threadIdx.x % kG, g = threadIdx.x / kG;
  const int64_t i = gid() / kG;
  const bool row = i < A.n;
  Sums<SL, 2> T{key + g * SL, val + g * 2 * SL};
  T.clear(lane);
  const int np = row ? pcnt[i] : 0;
  T.add(lane < np, lane < np ? pcol[i * kP + lane] : 0, 1, lane < np ? pv[i * kP + lane] : 0.0);
  const int m = row ? A.len(i) : 0;
  const int mm = wave_max(m);
  for (int k0 = 0; k0 < mm; k0 += kG) {
    // entry k0 + lane of the row, then the entries one after the other
    const int64_t e = k0 + lane < m ? A.at(i, k0 + lane) : 0;
    const double a = k0 + lane < m ? A.val[e] : 0.0;
    const int j = k0 + lane < m ? A.col[e] : 0;
    const int pj = a != 0.0 ? pcnt[j] : 0;
    for (int k = 0; k < kG && k0 + k < mm; k += 4) {
      int c[4], on[4];
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int jj = __shfl(j, k + u, kG);
        on[u] = lane < __shfl(pj, k + u, kG);
        const double aa = __shfl(a, k + u, kG);
        c[u] = on[u] ? pcol[(int64_t)jj * kP + lane] : 0;
        v[u] = on[u] ? aa * pv[(int64_t)jj * kP + lane] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) T.add(on[u], c[u], 0, v[u]);
    }
  }
  const double si = row ? s[i] : 0.0;
  int at = 0;
  for (int own = 1; own >= 0; --own)
    for (int k0 = 0; k0 < SL; k0 += kG) {
      const int c = T.key[k0 + lane];
      const double p = T.val[SL + k0 + lane], ap = T.val[k0 + lane];
      const bool take = row && c >= 0 && (p != 0.0) == (own != 0);
      const int b = group_ballot(take);
      const int to = at + __popc(b & ((1 << lane) - 1));
      at += __popc(b);
      if (take && to < kAmgQ) {
        qcol[i * qi + to * qk] = c;
        qv[i * qi + to * qk] = (float)(p - si * ap);
        tcol[i * kAmgQ + to] = c;
        tp[i * kAmgQ + to] = p;
        tap[i * kAmgQ + to] = ap;
        atomicAdd(count + c, 1);
      }
    }
  if (row && lane == 0) qcnt[i] = (uint8_t)min(at, kAmgQ);
}

__global__ __launch_bounds__(kB) void zero_kernel(int64_t n, int32_t* __restrict__ p) {
  const int64_t i = gid();
  if (i < n) p[i] = 0;
}

// keys row << 4 | slot of the transposed lists, in no order yet (count runs back to 0)
__global__ __launch_bounds__(kB) void transpose_fill_kernel(int64_t n, const uint8_t* __restrict__ qcnt,
                                                            const int32_t* __restrict__ tcol,
                                                            const int32_t* __restrict__ qtp,
                                                            int32_t* __restrict__ count, uint32_t* __restrict__ key) {
  const int64_t i = gid() / kG;
  const int k = threadIdx.x % kG;
  if (i >= n || k >= qcnt[i]) return;
  const int c = tcol[i * kAmgQ + k];
  key[qtp[c] + atomicAdd(count + c, -1) - 1] = (uint32_t)i << 4 | (uint32_t)k;
}

// Lists of more than kListWave entries (the columns of a hub's aggregate) in ascending order: a
// workgroup looks at 1024 lists and sorts those it finds one after the other, by Batcher's
// bitonic network with every comparator ascending (the first step of a merge mirrored), so that
// places beyond the end act as infinities; in LDS up to kListLds entries.  m log^2 m steps by
// 1024 threads: a list in memory of 10^5 entries takes about 15,000 rounds, where one lane's
// insertion sort of a list that arrives in descending order takes 5 10^9 dependent steps.
constexpr int kListWave = 128, kListLds = 8192;
__global__ __launch_bounds__(1024) void transpose_sort_long_kernel(int64_t nc, const int32_t* __restrict__ qtp,
                                                                   uint32_t* __restrict__ key) {
  __shared__ uint32_t sh[kListLds];
  __shared__ int found[1024], n_found;
  const int tid = threadIdx.x;
  if (tid == 0) n_found = 0;
  __syncthreads();
  const int64_t c = gid();
  if (c < nc && qtp[c + 1] - qtp[c] > kListWave) found[atomicAdd(&n_found, 1)] = (int)c;
  __syncthreads();
  for (int f = 0; f < n_found; ++f) {
    const int k0 = qtp[found[f]], m = qtp[found[f] + 1] - k0;
    const bool lds = m <= kListLds;
    uint32_t* const a = lds ? sh : key + k0;
    if (lds)
      for (int i = tid; i < m; i += 1024) a[i] = key[k0 + i];
    __syncthreads();
    auto order = [&](int64_t i, int64_t j) {
      if (j >= m) return;
      const uint32_t x = a[i], y = a[j];
      if (x > y) {
        a[i] = y;
        a[j] = x;
      }
    };
    for (int64_t size = 2; size < 2 * (int64_t)m; size <<= 1) {
      const int64_t half = size >> 1;
      // pairs t of blocks of `size`; the last block's may lie beyond the end
      for (int64_t t = tid; t / half * size < m; t += 1024) order(t / half * size + t % half, t / half * size + size - 1 - t % half);
      __syncthreads();
      for (int64_t step = half >> 1; step > 0; step >>= 1) {
        for (int64_t t = tid; t / step * 2 * step < m; t += 1024) order(t / step * 2 * step + t % step, t / step * 2 * step + t % step + step);
        __syncthreads();
      }
    }
    if (lds)
      for (int i = tid; i < m; i += 1024) key[k0 + i] = a[i];
    __syncthreads();
  }
}

// each list in ascending order, and its values: a wave per list, two entries per lane up
// to kListWave (a bitonic network over e = lane + 64 r); longer ones are in order already
__global__ __launch_bounds__(kB) void transpose_sort_kernel(int64_t nc, const int32_t* __restrict__ qtp,
                                                            uint32_t* __restrict__ key, const float* __restrict__ qv,
                                                            int64_t qi, int64_t qk, int32_t* __restrict__ qti,
                                                            float* __restrict__ qtv) {
  const int64_t c = gid() / 64;
  const int lane = threadIdx.x & 63;
  if (c >= nc) return;
  const int k0 = qtp[c], m = qtp[c + 1] - k0;
  if (m <= kListWave) {
    uint32_t x[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) x[r] = lane + 64 * r < m ? key[k0 + lane + 64 * r] : 0xffffffffu;
    const int top = m > 64 ? 128 : 64;
    for (int size = 2; size <= top; size <<= 1) {
      if (size == 128) {  // step 64: the lane's own pair
        const uint32_t lo = min(x[0], x[1]), hi = max(x[0], x[1]);
        x[0] = lo;
        x[1] = hi;
      }
      for (int step = min(size >> 1, 32); step > 0; step >>= 1)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const uint32_t y = __shfl_xor(x[r], step, 64);
          const bool up = ((lane + 64 * r) & size) == 0;
          x[r] = (!(lane & step) == up) ? min(x[r], y) : max(x[r], y);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; ++r)
      if (lane + 64 * r < m) key[k0 + lane + 64 * r] = x[r];
  }
  for (int k = lane; k < m; k += 64) {
    const uint32_t x = key[k0 + k];
    const int64_t i = x >> 4, sl = x & 15u;
    qti[k0 + k] = (int32_t)i;
    qtv[k0 + k] = qv[i * qi + sl * qk];
  }
}

// A_c = P^T (A P): a group of lanes per coarse row, its fine rows one after the other
__global__ __launch_bounds__(64) void coarse_kernel(int64_t nc, const int32_t* __restrict__ qtp,
                                                    const uint32_t* __restrict__ key,
                                                    const uint8_t* __restrict__ qcnt,
                                                    const int32_t* __restrict__ tcol, const double* __restrict__ tp,
                                                    const double* __restrict__ tap, int32_t* __restrict__ cnt,
                                                    int32_t* __restrict__ col, double* __restrict__ val) {
  constexpr int SL = 128, GR = 64 / kG;
  __shared__ int32_t keys[GR * SL];
  __shared__ double vals[GR * SL];
  const int lane = threadIdx.x % kG, g = threadIdx.x / kG;
  const int64_t c = gid() / kG;
  const bool row = c < nc;
  Sums<SL, 1> T{keys + g * SL, vals + g * SL};
  T.clear(lane);
  const int k0 = row ? qtp[c] : 0, m = row ? qtp[c + 1] - k0 : 0;
  const int mm = wave_max(m);
  for (int b0 = 0; b0 < mm; b0 += kG) {
    const uint32_t x = b0 + lane < m ? key[k0 + b0 + lane] : 0u;
    const int64_t i = x >> 4;
    const double p = b0 + lane < m ? tp[i * kAmgQ + (x & 15u)] : 0.0;
    const int len = p != 0.0 ? qcnt[i] : 0;
    for (int k = 0; k < kG; k += 4) {
      if (!__any(__shfl(len, k, kG) | __shfl(len, k + 1, kG) | __shfl(len, k + 2, kG) | __shfl(len, k + 3, kG)))
        continue;
      int cc[4], on[4];
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t ii = __shfl((int)i, k + u, kG);
        const double pp = __shfl(p, k + u, kG);
        on[u] = lane < __shfl(len, k + u, kG);
        cc[u] = on[u] ? tcol[ii * kAmgQ + lane] : 0;
        v[u] = on[u] ? pp * tap[ii * kAmgQ + lane] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) T.add(on[u], cc[u], 0, v[u]);
    }
  }
  int at = 0;
  for (int own = 1; own >= 0; --own)  // the diagonal first
    for (int q = 0; q < SL; q += kG) {
      const int cc = T.key[q + lane];
      const bool take = row && cc >= 0 && (cc == c) == (own != 0);
      const int b = group_ballot(take);
      const int to = at + __popc(b & ((1 << lane) - 1));
      at += __popc(b);
      if (take && to < kAmgRow) {
        col[c * kAmgRow + to] = cc;
        val[c * kAmgRow + to] = T.val[q + lane];
      }
    }
  if (row && lane == 0) cnt[c] = min(at, kAmgRow);
}

// ---- the coarsest operator's inverse, by Gauss-Jordan in LDS (positive definite: no
// pivoting; a vanishing pivot's unknown is left out)
__global__ __launch_bounds__(1024) void invert_kernel(AmgMat A, double* __restrict__ inv) {
  __shared__ double a[kDense * kDense];
  __shared__ double rk[kDense], ck[kDense];
  const int n = (int)A.n, tid = threadIdx.x;
  for (int e = tid; e < n * n; e += 1024) a[e] = 0.0;
  __syncthreads();
  double top = 0.0;
  if (tid < n)
    for (int k = 0; k < A.len(tid); ++k) a[tid * n + A.col[A.at(tid, k)]] += A.val[A.at(tid, k)];
  __syncthreads();
  for (int k = 0; k < n; ++k) top = fmax(top, fabs(a[k * n + k]));
  for (int k = 0; k < n; ++k) {
    const double p = a[k * n + k];
    const double ip = fabs(p) > 1e-13 * top ? 1.0 / p : 0.0;
    __syncthreads();
    if (tid < n) {
      rk[tid] = a[k * n + tid];
      ck[tid] = a[tid * n + k];
    }
    __syncthreads();
    for (int e = tid; e < n * n; e += 1024) {
      const int i = e / n, j = e - i * n;
      double v;
      if (i == k) v = j == k ? ip : rk[j] * ip;
      else if (j == k) v = -ck[i] * ip;
      else v = a[e] - ck[i] * rk[j] * ip;
      a[e] = v;
    }
    __syncthreads();
  }
  for (int e = tid; e < n * n; e += 1024) inv[e] = a[e];
}

// ---- the cycle
struct View {  // a level as the cycle's kernels see it
  AmgMat A;
  const double* s;
  const uint8_t* qcnt;
  const int32_t* qcol;
  const float* qv;
  int64_t qi, qk;
  int64_t nc;
  const int32_t* qtp;
  const int32_t* qti;
  const float* qtv;
  double* b;
  double* x;
};

// The cycle's rows by `lanes` lanes each (8 to 64), every lane returning the row's value;
// four entries per lane and round, their loads in flight together.
constexpr int kLanes = 8;
__device__ __forceinline__ double lanes_sum(double v, int lanes) {
  for (int o = lanes >> 1; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
template <class Entry>
__device__ __forceinline__ double lanes_dot(int k, int k1, int lanes, Entry entry) {
  double v = 0.0;
  for (; k < k1; k += 4 * lanes) {
    int c[4];
    double a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      a[u] = 0.0;
      c[u] = -1;
      if (k + u * lanes < k1) entry(k + u * lanes, &c[u], &a[u], false);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (c[u] >= 0) entry(k, &c[u], &a[u], true);
#pragma unroll
    for (int u = 0; u < 4; ++u) v += a[u];
  }
  return v;
}
// s_i (2 b_i - (A S b)_i) + (Q e)_i
__device__ __forceinline__ double up_row(const View& L, int64_t i, int lane, int lanes, const double* b,
                                         const double* e) {
  const double ax = lanes_dot(lane, L.A.len(i), lanes, [&](int k, int* c, double* a, bool gather) {
    if (!gather) {
      *c = L.A.col[L.A.at(i, k)];
      *a = L.A.val[L.A.at(i, k)];
    } else {
      *a *= L.s[*c] * b[*c];
    }
  });
  double v = -L.s[i] * ax;
  if (e)
    v += lanes_dot(lane, L.qcnt[i], lanes, [&](int k, int* c, double* a, bool gather) {
      if (!gather) {
        *c = L.qcol[i * L.qi + k * L.qk];
        *a = (double)L.qv[i * L.qi + k * L.qk];
      } else {
        *a *= e[*c];
      }
    });
  return lanes_sum(v, lanes) + L.s[i] * 2.0 * b[i];
}
// (Q^T b)_c
__device__ __forceinline__ double down_row(const View& L, int64_t c, int lane, int lanes, const double* b) {
  const double v = lanes_dot(L.qtp[c] + lane, L.qtp[c + 1], lanes, [&](int k, int* i, double* a, bool gather) {
    if (!gather) {
      *i = L.qti[k];
      *a = (double)L.qtv[k];
    } else {
      *a *= b[*i];
    }
  });
  return lanes_sum(v, lanes);
}
// lanes per row of the tail kernel for n rows
__device__ __forceinline__ int tail_lanes(int n) { return n <= 16 ? 64 : n <= 32 ? 32 : n <= 64 ? 16 : kLanes; }

__global__ __launch_bounds__(kB) void down_kernel(View L, const double* __restrict__ b, double* __restrict__ out,
                                                  const double* __restrict__ done) {
  if (*done != 0.0) return;
  const int64_t c = gid() / kLanes;
  if (c >= L.nc) return;
  const double v = down_row(L, c, threadIdx.x % kLanes, kLanes, b);
  if (threadIdx.x % kLanes == 0) out[c] = v;
}

__global__ __launch_bounds__(kB) void up_kernel(View L, const double* __restrict__ e, const double* __restrict__ done) {
  if (*done != 0.0) return;
  const int64_t i = gid() / kLanes;
  if (i >= L.A.n) return;
  const double v = up_row(L, i, threadIdx.x % kLanes, kLanes, L.b, e);
  if (threadIdx.x % kLanes == 0) L.x[i] = v;
}

// The levels from the first of at most kTailRows rows to the coarsest and back, vectors
// in LDS.
struct Tail {
  int nl;
  View L[kTailLevels];
  const double* inverse;  // of the last level, or null: Jacobi sweeps there
};
__global__ __launch_bounds__(kTailThreads) void tail_kernel(Tail t, const double* __restrict__ done) {
  __shared__ double sb[2 * kTailRows], sx[2 * kTailRows];
  __shared__ double part[kTailThreads];
  if (*done != 0.0) return;
  const int tid = threadIdx.x;
  int off[kTailLevels + 1];
  off[0] = 0;
#pragma unroll
  for (int l = 0; l < kTailLevels; ++l) off[l + 1] = off[l] + (l < t.nl ? (int)t.L[l].A.n : 0);
  for (int i = tid; i < t.L[0].A.n; i += kTailThreads) sb[i] = t.L[0].b[i];
  __syncthreads();
#pragma unroll
  for (int l = 0; l < kTailLevels - 1; ++l) {
    if (l + 1 >= t.nl) break;
    const int nc = (int)t.L[l].nc, lanes = tail_lanes(nc);
    for (int c = tid / lanes; c < nc; c += kTailThreads / lanes) {
      const double v = down_row(t.L[l], c, tid % lanes, lanes, sb + off[l]);
      if (tid % lanes == 0) sb[off[l + 1] + c] = v;
    }
    __syncthreads();
  }
#pragma unroll
  for (int l = kTailLevels - 1; l >= 0; --l) {
    if (l >= t.nl) continue;
    const int n = (int)t.L[l].A.n;
    const double* const b = sb + off[l];
    double* const x = sx + off[l];
    if (l == t.nl - 1 && t.inverse) {
      // kTailThreads / n threads per row (at most kDense rows: at least 8)
      const int per = kTailThreads / kDense, r = tid / per, q = tid % per;
      double v = 0.0;
      if (r < n)
        for (int j = q; j < n; j += per) v += t.inverse[r * n + j] * b[j];
      part[tid] = v;
      __syncthreads();
      if (q == 0 && r < n) {
        double s = 0.0;
        for (int j = 0; j < per; ++j) s += part[tid + j];
        x[r] = s;
      }
    } else {
      const double* const e = l == t.nl - 1 ? nullptr : sx + off[l + 1];
      const int lanes = tail_lanes(n);
      for (int i = tid / lanes; i < n; i += kTailThreads / lanes) {
        const double v = up_row(t.L[l], i, tid % lanes, lanes, b, e);
        if (tid % lanes == 0) x[i] = v;
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < t.L[0].A.n; i += kTailThreads) t.L[0].x[i] = sx[i];
}

View view_of(const AmgLevel& l) {
  View v;
  v.A = l.A;
  v.s = l.s;
  v.qcnt = l.qcnt;
  v.qcol = l.qcol;
  v.qv = l.qv;
  v.qi = l.qi;
  v.qk = l.qk;
  v.nc = l.nc;
  v.qtp = l.qtp;
  v.qti = l.qti;
  v.qtv = l.qtv;
  v.b = l.b;
  v.x = l.x;
  return v;
}

// A block of device memory cut into 256-byte aligned pieces.
struct Arena {
  char* base = nullptr;
  size_t at = 0;
  template <class T>
  T* take(int64_t n) {
    T* p = (T*)(base + at);
    at += (sizeof(T) * (size_t)std::max<int64_t>(n, 1) + 255) & ~(size_t)255;
    return p;
  }
};

}  // namespace

namespace fvm {

Amg::~Amg() {
  for (void* p : mem) (void)hipFree(p);
}

int amg_build(int64_t n0, const int32_t* rp, const int32_t* col, const double* val, Amg** out, hipStream_t st) {
  *out = nullptr;
  if (n0 > kAmgMaxRows) return FVM_OK;
  const auto t0 = std::chrono::steady_clock::now();
  struct Guard {
    Amg* a;
    void* scratch = nullptr;
    ~Guard() {
      if (scratch) (void)hipFree(scratch);
      delete a;
    }
  } G{new Amg};
  Amg* const a = G.a;
  auto carve = [&](Arena& A, auto&& layout) -> int {  // sizes first, then one allocation
    layout(A);
    const size_t bytes = A.at;
    FVM_HIP(fvm::dev_malloc((void**)&A.base, bytes));
    A.at = 0;
    layout(A);
    return FVM_OK;
  };
  // work of one level, sized for the first
  uint64_t *mask, *t, *t1;
  double *d, *pv, *tp, *tap;
  int32_t *id, *agg1, *agg, *pcol, *tcol, *sums, *count;
  uint8_t* pcnt;
  Arena W;
  int rc = carve(W, [&](Arena& A) {
    mask = A.take<uint64_t>(n0);
    t = A.take<uint64_t>(n0);
    t1 = A.take<uint64_t>(n0);
    d = A.take<double>(n0);
    pv = A.take<double>(kP * n0);
    tp = A.take<double>(kAmgQ * n0);
    tap = A.take<double>(kAmgQ * n0);
    id = A.take<int32_t>(n0);
    agg1 = A.take<int32_t>(n0);
    agg = A.take<int32_t>(n0);
    pcol = A.take<int32_t>(kP * n0);
    tcol = A.take<int32_t>(kAmgQ * n0);
    sums = A.take<int32_t>(n0 / kScan + 2);
    count = A.take<int32_t>(n0);
    pcnt = A.take<uint8_t>(n0);
  });
  if (rc) return rc;
  G.scratch = W.base;

  AmgMat M;
  M.n = n0;
  M.rp = rp;
  M.col = col;
  M.val = val;
  double *lb = nullptr, *lx = nullptr;
  for (int lev = 0;; ++lev) {
    const int64_t n = M.n;
    AmgLevel L;
    L.A = M;
    L.b = lb;
    L.x = lx;
    Arena P;
    rc = carve(P, [&](Arena& A) {
      L.s = A.take<double>(n);
      L.qcnt = A.take<uint8_t>(n);
      L.qcol = A.take<int32_t>(kAmgQ * n);
      L.qv = A.take<float>(kAmgQ * n);
    });
    L.qi = lev == 0 ? 1 : kAmgQ;
    L.qk = lev == 0 ? n : 1;
    if (rc) return rc;
    a->mem.push_back(P.base);
    hipLaunchKernelGGL(weights_kernel, grid1(n), dim3(kB), 0, st, M, d, L.s);
    bool last = n <= kDense || lev >= 15;
    int32_t nc = 0;
    const int nb = (int)((n + kScan - 1) / kScan);
    if (!last) {
      hipLaunchKernelGGL(strong_kernel, grid1(n), dim3(kB), 0, st, M, d, kTheta * kTheta, mask, t);
      for (int r = 0; r < kMisRounds; ++r) {
        hipLaunchKernelGGL(mis_max_kernel, grid1(n), dim3(kB), 0, st, M, mask, t, t1);
        hipLaunchKernelGGL(mis_decide_kernel, grid1(n), dim3(kB), 0, st, M, mask, t1, t);
      }
      hipLaunchKernelGGL(scan_sums_kernel<1>, dim3(nb), dim3(kScan), 0, st, n, (const void*)t, sums);
      hipLaunchKernelGGL(scan_blocks_kernel, dim3(1), dim3(kScan), 0, st, nb, sums);
      hipLaunchKernelGGL(scan_out_kernel<1>, dim3(nb), dim3(kScan), 0, st, n, (const void*)t, sums, id);
      hipLaunchKernelGGL(join_roots_kernel, grid1(n), dim3(kB), 0, st, M, mask, t, id, agg1);
      hipLaunchKernelGGL(join_rest_kernel, grid1(n), dim3(kB), 0, st, M, mask, agg1, agg);
      hipLaunchKernelGGL(prolong_kernel, grid1(n), dim3(kB), 0, st, M, mask, agg, pcnt, pcol, pv);
      hipLaunchKernelGGL(zero_kernel, grid1(n), dim3(kB), 0, st, n, count);
      hipLaunchKernelGGL(smooth_kernel, grid1(n * kG), dim3(kB), 0, st, M, L.s, pcnt, pcol, pv, L.qcnt, L.qcol, L.qv,
                         L.qi, L.qk, tcol, tp, tap, count);
      FVM_HIP(hipMemcpyAsync(&nc, sums + nb, sizeof nc, hipMemcpyDeviceToHost, st));
      FVM_HIP(hipStreamSynchronize(st));
      last = nc == 0 || nc > 0.7 * n;
    }
    if (last) {
      a->level.push_back(L);
      break;
    }
    // the transposed lists and the next level's operator and vectors
    const int nbc = (nc + kScan - 1) / kScan;
    int32_t nq = 0;
    hipLaunchKernelGGL(scan_sums_kernel<0>, dim3(nbc), dim3(kScan), 0, st, (int64_t)nc, (const void*)count, sums);
    hipLaunchKernelGGL(scan_blocks_kernel, dim3(1), dim3(kScan), 0, st, nbc, sums);
    FVM_HIP(hipMemcpyAsync(&nq, sums + nbc, sizeof nq, hipMemcpyDeviceToHost, st));
    FVM_HIP(hipStreamSynchronize(st));
    L.nc = nc;
    int32_t *ccnt, *ccol;
    double* cval;
    uint32_t* key;
    Arena C;
    rc = carve(C, [&](Arena& A) {
      L.qtp = A.take<int32_t>((int64_t)nc + 1);
      L.qti = A.take<int32_t>(nq);
      L.qtv = A.take<float>(nq);
      key = A.take<uint32_t>(nq);
      ccnt = A.take<int32_t>(nc);
      ccol = A.take<int32_t>((int64_t)kAmgRow * nc);
      cval = A.take<double>((int64_t)kAmgRow * nc);
      lb = A.take<double>(nc);
      lx = A.take<double>(nc);
    });
    if (rc) return rc;
    a->mem.push_back(C.base);
    hipLaunchKernelGGL(scan_out_kernel<0>, dim3(nbc), dim3(kScan), 0, st, (int64_t)nc, (const void*)count, sums,
                       L.qtp);
    FVM_HIP(hipMemcpyAsync(L.qtp + nc, sums + nbc, sizeof nq, hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(transpose_fill_kernel, grid1(n * kG), dim3(kB), 0, st, n, L.qcnt, tcol, L.qtp, count, key);
    hipLaunchKernelGGL(transpose_sort_long_kernel, dim3((unsigned)((nc + 1023) / 1024)), dim3(1024), 0, st, (int64_t)nc,
                       L.qtp, key);
    hipLaunchKernelGGL(transpose_sort_kernel, grid1((int64_t)nc * 64), dim3(kB), 0, st, (int64_t)nc, L.qtp, key, L.qv,
                       L.qi, L.qk, L.qti, L.qtv);
    hipLaunchKernelGGL(coarse_kernel, dim3((unsigned)(((int64_t)nc * kG + 63) / 64)), dim3(64), 0, st, (int64_t)nc,
                       L.qtp, key, L.qcnt, tcol, tp, tap, ccnt, ccol, cval);
    a->level.push_back(L);
    M = AmgMat();
    M.n = nc;
    M.cnt = ccnt;
    M.col = ccol;
    M.val = cval;
  }
  FVM_HIP(hipGetLastError());
  const int nl = (int)a->level.size();
  if (nl < 2) return FVM_OK;  // no coarse level: nothing gained over Jacobi
  const AmgLevel& B = a->level[nl - 1];
  if (B.A.n <= kDense) {
    double* inv = nullptr;
    FVM_HIP(fvm::dev_malloc((void**)&inv, sizeof(double) * kDense * kDense));
    a->mem.push_back(inv);
    a->inverse = inv;
    hipLaunchKernelGGL(invert_kernel, dim3(1), dim3(1024), 0, st, B.A, inv);
  }
  a->tail = nl;
  int64_t rows = 0;
  while (a->tail > 1 && nl - a->tail < kTailLevels && a->level[a->tail - 1].A.n <= kTailRows &&
         rows + a->level[a->tail - 1].A.n <= 2 * kTailRows)
    rows += a->level[--a->tail].A.n;
  FVM_HIP(hipStreamSynchronize(st));
  a->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  G.a = nullptr;
  *out = a;
  return FVM_OK;
}

void amg_coarse(const Amg* a, const double* done, hipStream_t st) {
  const int nl = (int)a->level.size();
  for (int l = 1; l + 1 < nl && l < a->tail; ++l)
    hipLaunchKernelGGL(down_kernel, grid1(a->level[l].nc * kLanes), dim3(kB), 0, st, view_of(a->level[l]),
                       a->level[l].b, a->level[l + 1].b, done);
  if (a->tail < nl) {
    Tail t;
    t.nl = nl - a->tail;
    for (int l = 0; l < t.nl; ++l) t.L[l] = view_of(a->level[a->tail + l]);
    t.inverse = a->inverse;
    hipLaunchKernelGGL(tail_kernel, dim3(1), dim3(kTailThreads), 0, st, t, done);
  }
  for (int l = std::min(a->tail, nl) - 1; l >= 1; --l)
    hipLaunchKernelGGL(up_kernel, grid1(a->level[l].A.n * kLanes), dim3(kB), 0, st, view_of(a->level[l]),
                       l + 1 < nl ? a->level[l + 1].x : (const double*)nullptr, done);
}

}  // namespace fvm
