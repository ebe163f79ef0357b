// Exchange between the workgroups of one cooperative (all resident) grid, without
// leaving the kernel: published vectors and grid-wide sums.
//
// Every 8-byte word carries 4 bytes of payload and the 4-byte number of its exchange,
// so a reader polls the words themselves until the numbers match: a store and a load
// make one exchange, with no flag, fence or cache write-back between them (each word is
// one aligned 64-bit half of its access, seen whole).  The accesses are of agent scope,
// which every XCD's L2 passes on to memory.  Measured on MI355X: a sum over the grid takes
// 1.35 us on one workgroup, 1.7 us on 4 to 40, 1.8 us on 64 and 3.1 us on 256 (a counter
// barrier with the data stored beside it: 1.2, 1.5 to 2.1, 2.3 and 4.8 us), where a kernel
// boundary costs 2.6 us of launch and its own first loads.
//
// The buffers alternate between two halves by the exchange's parity, so a half is
// written again two exchanges later, when every reader must have been through it:
//   sums: no workgroup completes the next one before every workgroup has contributed,
//     that is, has read this one;
//   vectors: a kernel publishes at most two of them between two sums, or the pattern of
//     its gathers is symmetric (a row then publishes again only after it has read the
//     next vector's entries from every row that reads its own, which those rows
//     published after reading).
// Every workgroup adds the contributions in the same order, so all of them hold the same
// sums bit for bit and take the same branches.
//
// Polls are bounded: a workgroup that waits too long raises the grid's fault word,
// which ends every other wait too, and the kernel returns with an error.
#pragma once
#include "fvm_internal.hpp"

namespace fvm {

constexpr int kGridMaxSums = 32;    // values per grid-wide sum
constexpr int kGridMaxWgs = 256;    // workgroups of a grid (four per lane in a sum)
constexpr unsigned kGridSpin = 1u << 21;

// Device memory of the exchanges of a grid of nwg workgroups over vectors of n:
// header (words 0..7: next vector and sum numbers, fault, counters of the kernels),
// then the vector's words, then the sums'.  Zeroed before its first use.
enum { kGridVec = 0, kGridSum = 1, kGridFault = 2, kGridUser = 3, kGridHead = 8 };
__host__ __device__ inline size_t grid_words(int64_t n) { return kGridHead + 4 * (size_t)n + 4 * (size_t)kGridMaxSums * kGridMaxWgs; }

// The pair of words of one double, moved by one 16-byte access (half the requests of two
// 8-byte ones; each word still carries its own number), through a buffer descriptor:
// the base in scalar registers, a 32-bit offset per lane, agent scope.
typedef uint32_t grid_pair __attribute__((ext_vector_type(4)));  // lo, number, hi, number
constexpr int kAgentScope = 1 << 4;                   // cache policy: sc1
constexpr int kVolatile = (int)(1u << 31);
using grid_rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ grid_rsrc grid_view(uint64_t* mem, size_t words) {
  return __builtin_amdgcn_make_buffer_rsrc(mem, 0, (int)(8 * words), 0x00027000);
}
__device__ __forceinline__ void grid_put(grid_rsrc m, uint32_t off, double x, uint32_t tag) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const grid_pair p = {(uint32_t)u, tag, (uint32_t)(u >> 32), tag};
  __builtin_amdgcn_raw_buffer_store_b128(p, m, (int)off, 0, kAgentScope | kVolatile);
}
__device__ __forceinline__ grid_pair grid_get(grid_rsrc m, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(m, (int)off, 0, kAgentScope | kVolatile);
}
// 0 when both words are of exchange tag
__device__ __forceinline__ uint32_t grid_stale(grid_pair p, uint32_t tag) { return (p.y ^ tag) | (p.w ^ tag); }
__device__ __forceinline__ double grid_value(grid_pair p) {
  return __longlong_as_double((long long)((uint64_t)p.x | ((uint64_t)p.z << 32)));
}
__device__ __forceinline__ uint64_t grid_fault(const uint64_t* mem) {
  return __hip_atomic_load(mem + kGridFault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Cross-lane moves of a double in vector registers (a shuffle through the LDS unit
// takes over 100 cycles, six of them a tenth of an exchange): DPP within rows of 16
// lanes, and the half swaps of gfx950 across them.
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
  const uint64_t u = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, CTRL, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// x of this half of the 64 (32: W = 32) lanes plus x of the other half, for two values
// at once: the lower half returns the sum of a, the upper half that of b
template <int W>
__device__ __forceinline__ double half_sums(double a, double b) {
  const uint64_t ua = (uint64_t)__double_as_longlong(a), ub = (uint64_t)__double_as_longlong(b);
  uint32_t r[2][2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const uint32_t x = (uint32_t)(ua >> (32 * k)), y = (uint32_t)(ub >> (32 * k));
    const auto p = W == 32 ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                           : __builtin_amdgcn_permlane16_swap(x, y, false, false);
    r[k][0] = p[0];
    r[k][1] = p[1];
  }
  const double s = __longlong_as_double((long long)(((uint64_t)r[1][0] << 32) | r[0][0]));
  const double t = __longlong_as_double((long long)(((uint64_t)r[1][1] << 32) | r[0][1]));
  return s + t;
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140, kDppRor8 = 0x128;

// The sum over the wave, in every lane.
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp<kDppXor1>(x);
  x += dpp<kDppXor2>(x);
  x += dpp<kDppHalfMirror>(x);
  x += dpp<kDppMirror>(x);
  x = half_sums<16>(x, x);
  return half_sums<32>(x, x);
}

// Sums of 8 values per lane over the wave: three halving steps leave one of the
// values in each group of eight lanes (lane >> 3 selects which), three more fold the
// group.  Lanes 8 q .. 8 q + 7 (q < 8) hold sum q.
__device__ __forceinline__ double wave_sums8(const double* v) {
  const bool h3 = threadIdx.x & 8;
  double a[4], b[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) a[i] = half_sums<32>(v[i], v[i + 4]);
#pragma unroll
  for (int i = 0; i < 2; ++i) b[i] = half_sums<16>(a[i], a[i + 2]);
  double c = (h3 ? b[1] : b[0]) + dpp<kDppRor8>(h3 ? b[0] : b[1]);
  c += dpp<kDppXor1>(c);
  c += dpp<kDppXor2>(c);
  return c + dpp<kDppHalfMirror>(c);
}

// Byte offset of entry c of a published vector (grids of up to 65,536 rows: 1 MiB).
__device__ __forceinline__ uint32_t grid_offset(int c) { return (uint32_t)c * 16u; }

// One workgroup's side of the exchanges, T threads.
template <int T>
struct GridShared {
  double red[T / 64][kGridMaxSums];
  double tot[kGridMaxSums];
  int fault;
};

template <int T>
struct Grid {
  uint64_t* mem;
  grid_rsrc view;
  int64_t n;
  int nwg;
  uint32_t vtag, rtag;
  GridShared<T>* sh;

  // kAgain: memory that earlier kernels have used.  A fault of one of them stands: its exchange
  // numbers are unknown, so every workgroup gives up after its first sum.
  template <bool kAgain = false>
  __device__ __forceinline__ void open(uint64_t* m, int64_t n_, GridShared<T>* s) {
    mem = m;
    view = grid_view(m, grid_words(n_));
    n = n_;
    nwg = (int)gridDim.x;
    sh = s;
    vtag = __builtin_amdgcn_readfirstlane((uint32_t)m[kGridVec]);
    rtag = __builtin_amdgcn_readfirstlane((uint32_t)m[kGridSum]);
    if (threadIdx.x == 0) s->fault = kAgain ? grid_fault(m) != 0 : 0;
    __syncthreads();
  }
  // the numbers the next kernel on this memory starts from (every workgroup has read
  // the old ones: it has taken part in a sum since)
  __device__ __forceinline__ void close() {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      mem[kGridVec] = vtag;
      mem[kGridSum] = rtag;
    }
  }
  // byte offsets of the halves in use
  __device__ __forceinline__ uint32_t vec() const {
    return 8u * kGridHead + (vtag & 1 ? 16u * (uint32_t)n : 0u);
  }
  __device__ __forceinline__ uint32_t sums() const {
    return 8u * kGridHead + 32u * (uint32_t)n + (rtag & 1 ? 16u * kGridMaxSums * kGridMaxWgs : 0u);
  }
  __device__ __forceinline__ void give_up() {
    __hip_atomic_store(mem + kGridFault, (uint64_t)1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sh->fault = 1;
  }
  __device__ __forceinline__ bool waited_long(unsigned spin) const {
    return spin > kGridSpin || (spin > 1000 && grid_fault(mem));
  }

  // x is entry i of the next published vector (active: this thread has an entry)
  __device__ __forceinline__ void publish(int64_t i, double x, bool active) {
    ++vtag;
    if (active) grid_put(view, vec() + 16u * (uint32_t)i, x, vtag);
  }
  // the entries at off[0..K) (grid_offset) of the published vector, all loads in flight
  // together
  template <int K>
  __device__ __forceinline__ void fetch(const uint32_t (&off)[K], double (&x)[K], bool active) {
    if (!active) {
#pragma unroll
      for (int s = 0; s < K; ++s) x[s] = 0.0;
      return;
    }
    const uint32_t v = vec();
    grid_pair p[K];
#pragma nounroll
    for (unsigned spin = 0;; ++spin) {
      uint32_t stale = 0;
#pragma unroll
      for (int s = 0; s < K; ++s) p[s] = grid_get(view, v + off[s]);
#pragma unroll
      for (int s = 0; s < K; ++s) stale |= grid_stale(p[s], vtag);
      if (stale == 0) break;
      if (waited_long(spin)) {
        give_up();
        break;
      }
    }
#pragma unroll
    for (int s = 0; s < K; ++s) x[s] = grid_value(p[s]);
  }
  __device__ __forceinline__ double fetch1(int c) {
    const uint32_t off[1] = {grid_offset(c)};
    double x[1];
    fetch<1>(off, x, true);
    return x[0];
  }

  // sums over the grid of k <= kGridMaxSums values per thread; value(q) is called with
  // q < k.  The totals are in sh->tot[0..k) for every thread after the call; false when
  // the grid has given up.
  template <class F>
  __device__ __forceinline__ bool sum(int k, F value) {
    constexpr int NW = T / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int q0 = 0; q0 < k; q0 += 8) {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = q0 + q < k ? value(q0 + q) : 0.0;
      const double s = wave_sums8(v);
      if ((lane & 7) == 0) sh->red[wave][q0 + (lane >> 3)] = s;
    }
    __syncthreads();
    ++rtag;
    const uint32_t P = sums();
    if ((int)threadIdx.x < k) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < NW; ++w) s += sh->red[w][threadIdx.x];
      if (nwg > 1) grid_put(view, P + 16u * (threadIdx.x * kGridMaxWgs + blockIdx.x), s, rtag);
      else sh->tot[threadIdx.x] = s;
    }
    if (nwg > 1) {
      // wave w collects sums w, w + NW, ..., kQ of them per round of polls (a round trip
      // to memory each), 64 workgroups' contributions per load
      constexpr int kQ = 4, kG = kGridMaxWgs / 64;
      for (int q0 = wave; q0 < k; q0 += kQ * NW) {
        double x[kQ];
#pragma nounroll
        for (unsigned spin = 0;; ++spin) {
          grid_pair p[kQ][kG];
#pragma unroll
          for (int r = 0; r < kQ; ++r) {
            const uint32_t q = q0 + r * NW < k ? q0 + r * NW : q0;
#pragma unroll
            for (int g = 0; g < kG; ++g) {
              p[r][g] = grid_pair{0u, rtag, 0u, rtag};  // 0.0, arrived
              if (q0 + r * NW < k && lane + 64 * g < nwg)
                p[r][g] = grid_get(view, P + 16u * (q * kGridMaxWgs + lane + 64 * g));
            }
          }
          uint32_t stale = 0;
#pragma unroll
          for (int r = 0; r < kQ; ++r) {
            x[r] = 0.0;
#pragma unroll
            for (int g = 0; g < kG; ++g) {
              stale |= grid_stale(p[r][g], rtag);
              x[r] += grid_value(p[r][g]);
            }
          }
          if (__all(stale == 0)) break;
          if (waited_long(spin)) {
            if (lane == 0) give_up();
            break;
          }
        }
#pragma unroll
        for (int r = 0; r < kQ; ++r) {
          const double t = wave_sum(x[r]);
          if (lane == 0 && q0 + r * NW < k) sh->tot[q0 + r * NW] = t;
        }
      }
    }
    __syncthreads();
    return sh->fault == 0;
  }
  __device__ __forceinline__ bool sum1(double v, double* out) {
    const bool ok = sum(1, [&](int) { return v; });
    *out = sh->tot[0];  // written again only after the next sum's first barrier
    return ok;
  }
};

}  // namespace fvm
