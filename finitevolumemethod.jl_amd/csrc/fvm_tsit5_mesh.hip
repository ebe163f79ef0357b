// Tsit5 on fvm_eqs! of a mesh of up to 65,536 nodes in one launch: the adaptive loop of
// fvm_ode_solve (fvm_ode.hip), right-hand sides, Dirichlet callback and step control
// inside a resident grid, one block of 256 nodes per workgroup (MeshBlocks).
//
// Layout: a thread holds one node (state, seven stages) and up to two of the block's
// triangles (their records, rebuilt once) in registers, LDS
// the boundary items.  A stage hands the block's states to the neighbouring blocks through
// fvm_grid.hpp's words, forms the fluxes of the triangles that need none of theirs while
// those are on their way, then the others', into LDS, where every node sums its own.
// Triangles between blocks are formed in each: a sixth more fluxes, and no partial sums to
// exchange.  The exchange is what a stage waits for (2 us and more), then the fluxes' and
// sums' chains; the same loop as kernels was bound by about 20 launches a step: 63 steps
// at 62,451 nodes (D(u) quadratic) 7.0 -> 1.4 ms a solve, 1.3 ms of it this kernel (20 us
// a step); 10 steps at 1,600 nodes 1.38 -> 0.54 ms, at 144 nodes (one workgroup, no
// exchange) 0.90 -> 0.31 ms.  Every size it takes is the faster form.
//
// Every element's arithmetic is the multi-kernel path's (tri_fluxes, boundary_flux,
// NodeSum, finish_pre; the error norm in the order of the nodes' numbers, handed over
// once a step): the same states bit for bit.
#include <exception>

#include "fvm_internal.hpp"
#include "fvm_rhs_kernels.hpp"
#include "fvm_tsit5_loop.hpp"

using namespace fvm;
using namespace fvm_k;

namespace {

constexpr int kT = 512, NB = kBlockNodes, kRow = kBlockFlux;
static_assert(kBlockTris == kT && kBlockHalo == kT && kBlockItems == kT - NB && NB == kBlk, "one per thread");

struct MeshTsit5 : Tsit5Loop {
  KArgs p;
  MeshBlocks m;
  uint64_t* grid;
};

template <int FK>
struct MeshLds {
  double u[NB + kBlockHalo];   // states: the block's, the neighbours'
  double q[4 * kRow];          // fluxes (Q3, Q1, Q2, Q3) as in tile_kernel; first the coordinates
  double b[kBlockItems];       // boundary fluxes
  BItem<FK> item[kBlockItems];
  double tree[NB];
  double total;
  GridShared<kT> grid;
};

template <int FK>
__global__ __launch_bounds__(kT) void tsit5_mesh_kernel(MeshTsit5 a) {
  constexpr int NL = NB + kBlockHalo;
  static_assert(3 * NL <= 4 * kRow, "the coordinates fit in the flux rows");
  __shared__ MeshLds<FK> S;
  const int tid = threadIdx.x, lane = tid & 63, wg = blockIdx.x;
  const int64_t at = (int64_t)wg * NB + tid;  // the thread's node's position
  KArgs p = a.p;
  Grid<kT> G;
  // entries by position, then (the error norm's) by node
  const int64_t slots = (int64_t)gridDim.x * NB;
  G.open(a.grid, 2 * slots, &S.grid);
  const bool alone = gridDim.x == 1;
  bool up = true;

  // the node
  const int g = tid < NB ? a.m.node[at] : -1;
  const bool own = g >= 0;
  const int gs = own ? g : 0;
  const int code = own ? p.code[gs] : 3;
  const double V = own ? p.cv[gs] : 1.0;
  const int deg = own ? a.m.deg[at] : 0;
  const int rest = own ? a.m.more[at] : 0;
  const int bit = own ? a.m.bitem[at] : 0;
  uint4 ent = make_uint4(0, 0, 0, 0);
  if (own) ent = ((const uint4*)a.m.inc)[at];
  double u0 = own ? a.u[gs] : 0.0, k[7][1], un[1];
  k[0][0] = own ? a.k0[gs] : 0.0;
  // a node of a neighbouring block
  const int hp = a.m.halo[(int64_t)wg * kBlockHalo + tid];
  const bool halo = hp >= 0;
  const uint32_t hoff[1] = {grid_offset(halo ? hp : 0)};

  // the triangles' records
  double* const s_x = S.q;
  double* const s_y = S.q + NL;
  double* const s_D = S.q + 2 * NL;
  if (own) {
    s_x[tid] = p.x[g];
    s_y[tid] = p.y[g];
    if (FK == FVM_FLUX_D_NODAL) s_D[tid] = exp(p.log_d[g]);
  }
  if (halo) {
    const int h = a.m.node[hp];
    s_x[NB + tid] = p.x[h];
    s_y[NB + tid] = p.y[h];
    if (FK == FVM_FLUX_D_NODAL) s_D[NB + tid] = exp(p.log_d[h]);
  }
  __syncthreads();
  constexpr int ND = FK == FVM_FLUX_LINEAR ? 9 : 3;
  double P[2][P_COUNT], Ds[2][ND];
  int tri[2], loc[2];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int64_t lt = (int64_t)wg * 2 * kBlockTris + r * kT + tid;
    tri[r] = a.m.tri[lt];
    loc[r] = a.m.loc[lt];
    if (tri[r] < 0) continue;
    const int ia = loc[r] & 1023, ib = loc[r] >> 10 & 1023, ic = loc[r] >> 20 & 1023;
    rebuild_record<kGeo>(s_x[ia], s_y[ia], s_x[ib], s_y[ib], s_x[ic], s_y[ic], P[r]);
#pragma unroll
    for (int j = 0; j < ND; ++j) {
      if (FK == FVM_FLUX_D_NODAL) Ds[r][j] = s_D[j == 0 ? ia : (j == 1 ? ib : ic)];
      if (FK == FVM_FLUX_D_EDGE || FK == FVM_FLUX_LINEAR) Ds[r][j] = p.d_edge[j * p.T + tri[r]];
    }
  }
  // the boundary item
  const int iw = tid >= NB ? a.m.item[(int64_t)wg * kBlockItems + tid - NB] : -1;
  const int il = tid >= NB ? a.m.iloc[(int64_t)wg * kBlockItems + tid - NB] : 0;
  if (iw >= 0) {
    const int64_t Tt = p.badj[iw >> 1];
    S.item[tid - NB] = boundary_item<FK>(p, iw >> 1, iw & 1, p.tri[Tt], p.tri[p.T + Tt], p.tri[2 * p.T + Tt]);
  }
  __syncthreads();

  auto fluxes = [&](int r) {
    if (tri[r] < 0) return;
    const int ia = loc[r] & 1023, ib = loc[r] >> 10 & 1023, ic = loc[r] >> 20 & 1023;
    double Q[3];
    tri_fluxes<FK, M_RHS>(p, P[r], S.u[ia], S.u[ib], S.u[ic], 0.0, 0.0, 0.0, Ds[r][0], Ds[r][1], Ds[r][2], Ds[r], Q);
    const int lt = r * kT + tid;
    S.q[lt] = Q[2];
    S.q[kRow + lt] = Q[0];
    S.q[2 * kRow + lt] = Q[1];
    S.q[3 * kRow + lt] = Q[2];
  };
  // out = fvm_eqs!(x, ts) at the thread's node
  auto apply = [&](const double (&x)[1], double (&out)[1], double ts) {
    if (own) S.u[tid] = x[0];
    if (!alone) G.publish(at, x[0], own);
    p.t = ts;
    __syncthreads();
    fluxes(0);
    if (!alone) {
      double h[1];
      G.fetch(hoff, h, halo);
      if (halo) S.u[NB + tid] = h[0];
    }
    __syncthreads();
    fluxes(1);
    if (iw >= 0)
      S.b[tid - NB] = boundary_flux<FK>(p, S.item[tid - NB], S.u[il & 1023], S.u[il >> 10 & 1023], S.u[il >> 20 & 1023]);
    __syncthreads();
    out[0] = 0.0;
    if (!own) return;
    NodeSum sum;
    double qa[8], qb[8];
    const uint32_t e2[4] = {ent.x, ent.y, ent.z, ent.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int e = e2[j / 2] >> (16 * (j & 1)) & 0x7fff;
      qa[j] = S.q[e];
      qb[j] = S.q[e + kRow];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sum.add(j < deg, e2[j / 2] >> (16 * (j & 1)) & 0x8000, qa[j], qb[j]);
    for (int j0 = 8; j0 < deg; j0 += 8) {  // a hub's others, eight loads in flight
      int e[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) e[j] = j0 + j < deg ? a.m.rest[rest + j0 + j - 8] : 0;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        qa[j] = S.q[e[j] & 0x7fff];
        qb[j] = S.q[(e[j] & 0x7fff) + kRow];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) sum.add(j0 + j < deg, e[j] & 0x8000, qa[j], qb[j]);
    }
    double acc = sum.value();
    for (int j = 0; j < (bit & 255); ++j) acc = acc - S.b[(bit >> 8) + j];
    out[0] = finish_pre<FK, M_RHS>(p, g, acc, x[0], 0.0, code, V, 0.0);
  };

  // sum of q over the nodes, by their numbers (block b: nodes 256 b, ...)
  auto norm_sum = [&](const double (&q)[1]) -> double {
    ++G.rtag;
    if (alone) {
      if (tid < NB) S.tree[own ? g : tid] = own ? q[0] : 0.0;
    } else {
      G.publish(slots + gs, q[0], own);
      const bool in = tid < NB && at < a.n;
      const uint32_t off[1] = {grid_offset((int)(slots + (in ? at : 0)))};
      double x[1];
      G.fetch(off, x, in);
      if (tid < NB) S.tree[tid] = x[0];
    }
    __syncthreads();
    if (tid < 64) {
      const double v = (S.tree[tid] + S.tree[tid + 128]) + (S.tree[tid + 64] + S.tree[tid + 192]);
      const double t = wave_tree(v);
      double part[4] = {0.0, 0.0, 0.0, 0.0};
      if (alone) {
        part[0] = lane == 0 ? t : 0.0;
      } else {
        if (lane == 0) grid_put(G.view, G.sums() + 16u * (uint32_t)wg, t, G.rtag);
        grid_parts(G, (int)gridDim.x, part);
      }
      const double total = wave_tree((part[0] + part[2]) + (part[1] + part[3]));
      if (lane == 0) S.total = total;
    }
    __syncthreads();
    up = S.grid.fault == 0;
    return S.total;
  };
  auto row = [&](int) { return own ? (int64_t)g : a.n; };
  auto u_of = [&](int) -> double& { return u0; };
  auto dirichlet = [&](double x, double t) {
    if (!a.dirichlet || code != 1) return x;
    return eval_cond(p.C, p.fidx[g], p.x[g], p.y[g], t, x, p.C.node_g ? p.C.node_g[g] : 0.0);
  };
  tsit5_loop<1, true>(a, k, un, u_of, row, apply, norm_sum, dirichlet, up);
}

const void* kernel_of(int flux_kind) {
  switch (flux_kind) {
    case FVM_FLUX_D_POLY_U: return (const void*)tsit5_mesh_kernel<FVM_FLUX_D_POLY_U>;
    case FVM_FLUX_D_NODAL: return (const void*)tsit5_mesh_kernel<FVM_FLUX_D_NODAL>;
    case FVM_FLUX_LINEAR: return (const void*)tsit5_mesh_kernel<FVM_FLUX_LINEAR>;
    case FVM_FLUX_D_POWER: return (const void*)tsit5_mesh_kernel<FVM_FLUX_D_POWER>;
    default: return (const void*)tsit5_mesh_kernel<FVM_FLUX_D_EDGE>;
  }
}

}  // namespace

namespace fvm {

int problem_tsit5_small(const fvm_ctx* c, const fvm_ode_opts* o, const Tsit5Loop& start, fvm_ode_stats* st,
                        hipStream_t s) {
  const int64_t wgs = (c->m->N + NB - 1) / NB;
  if (wgs > kGridMaxWgs || o->n != c->m->N || c->flux_kind == FVM_FLUX_JIT) return FVM_ERR_STATE;
  const void* const kernel = kernel_of(c->flux_kind);
  bool fits;
  FVM_HIP(grid_fits(kernel, kT, wgs, &fits));
  if (!fits) return FVM_ERR_STATE;
  MeshBlocks m;
  int rc;
  try {
    rc = mesh_blocks(c->m, &m, s);
  } catch (const std::exception&) {  // no host memory
    rc = FVM_ERR_ALLOC;
  }
  if (rc == FVM_ERR_ALLOC || (rc == FVM_OK && m.n == 0)) return FVM_ERR_STATE;  // no (room for) lists
  if (rc != FVM_OK) return rc;
  MeshTsit5 a;
  static_cast<Tsit5Loop&>(a) = start;
  a.p = make_args(c);
  a.m = m;
  const size_t words = grid_words(2 * (int64_t)m.n * NB);
  auto launch = [&] {
    void* args[] = {&a};
    if (m.n == 1) return hipLaunchKernel(kernel, dim3(1), dim3(kT), args, 0, s);
    return hipLaunchCooperativeKernel(kernel, dim3((unsigned)m.n), dim3(kT), args, 0, s);
  };
  return tsit5_run(a, words, &a.grid, o, launch, st, s);
}

}  // namespace fvm
