// Lists of a device mesh that single paths read: the node incidences of node_kernel
// (fvm_rhs_kernels.hpp) and the node blocks of the one-launch Tsit5 (fvm_tsit5_mesh.hip).
//
// Both are made on the device from the mesh's incidence lists.  On the host, beside the mesh's
// uploads, they took a fifth of creating a mesh whether or not anything read them (16.0 -> 19.6 ms
// at 62,451 nodes, 1.07 -> 1.33 at 2,500).  Here the incidences are one kernel among the mesh's own
// (16.9 and 1.04 ms), and the blocks are made by the first solve that uses them: 0.4 ms at 62,451
// nodes, half of it blocks_kernel, whose threads follow chains of incidences (latency of dependent
// loads; it runs once per mesh).
#include <algorithm>
#include <vector>

#include "fvm_internal.hpp"

using namespace fvm;

namespace {

// The tile of a sorted triangle.
__device__ __forceinline__ int tile_of(const int32_t* __restrict__ start, int n, int s) {
  int lo = 0, hi = n;  // start[lo] <= s < start[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= s) lo = mid;
    else hi = mid;
  }
  return lo;
}

// ---- the per-node incidences of node_kernel
// A node's first block of eight is its own index, further ones stand after all nodes' (of
// node g from N + extra[g] on; extra null: no node has more than eight).
constexpr int kL = 8;
__global__ __launch_bounds__(256) void node_lists_kernel(int64_t N, int64_t T, const int32_t* __restrict__ tri,
                                                         const int32_t* __restrict__ start,
                                                         const int32_t* __restrict__ node_tri,
                                                         const int32_t* __restrict__ tile_tri_start, int n_tiles,
                                                         const int32_t* __restrict__ extra, int4* __restrict__ ent,
                                                         int32_t* __restrict__ next, int32_t* __restrict__ bed) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t g = q / kL;
  const int lane = (int)(q % kL);
  if (g >= N) return;
  const int k0 = start[g], deg = start[g + 1] - k0;
  const int blocks = deg > kL ? (deg + kL - 1) / kL : 1;
  for (int b = 0; b < blocks; ++b) {
    const int64_t at = b == 0 ? g : N + extra[g] + b - 1;
    int4 e = make_int4((int)g, (int)g, (int)g, -1);
    const int k = b * kL + lane;
    if (k < deg) {
      const int c = node_tri[k0 + k], s = c >> 2;
      const bool fresh = k > 0 && tile_of(tile_tri_start, n_tiles, s) !=
                                      tile_of(tile_tri_start, n_tiles, node_tri[k0 + k - 1] >> 2);
      e = make_int4(tri[s], tri[T + s], tri[2 * T + s], s << 3 | (int)fresh << 2 | (c & 3));
    }
    ent[at * kL + lane] = e;
    if (lane == 0) next[at] = b + 1 < blocks ? (int32_t)(N + extra[g] + b) : -1;
  }
  if (lane == 0) bed[g] = 0;
}
__global__ __launch_bounds__(256) void node_bed_kernel(int n_fix, const int32_t* __restrict__ fix_nodes,
                                                       const int32_t* __restrict__ fix_bedge_start,
                                                       int32_t* __restrict__ bed) {
  const int f = blockIdx.x * 256 + threadIdx.x;
  if (f < n_fix) bed[fix_nodes[f]] = fix_bedge_start[f] << 8 | (fix_bedge_start[f + 1] - fix_bedge_start[f]);
}

// ---- the blocks of the one-launch Tsit5
// Blocks are runs of the nodes in the order in which the triangles, sorted along a
// space-filling curve, first reach them (nodes of no triangle last): compact patches,
// whatever the numbering.
struct BlockArgs {
  int N, T, n_tiles, n_fix;
  const int32_t *tri, *start, *node_tri, *tile_tri_start, *fix_nodes, *fix_bedge_start, *fix_bedge, *badj;
  const int32_t* extra;  // per node its place in rest, null: no node has more than eight triangles
  // work: positions, nodes by position, tile of each triangle, fix entry of each node (-1: none),
  // sums of the scan, local id of a triangle for each of its vertices' blocks [3][T], halo id of
  // its vertex v in the block of its first vertex in that block w [3 v + w][T]
  int32_t *pos, *order, *tile, *fix, *sums, *at, *hid;
  // lists (MeshBlocks)
  uint16_t *inc, *rest;
  int32_t *node, *bitem, *deg, *more, *btri, *loc, *halo, *item, *iloc;
  int32_t* none;  // set when a block does not fit
};

__global__ __launch_bounds__(256) void block_setup_kernel(BlockArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < a.T) a.tile[i] = tile_of(a.tile_tri_start, a.n_tiles, i);
  if (i < a.N) a.fix[i] = -1;
  if (i == 0) *a.none = 0;
}

// Entry i < 3 T: vertex i % 3 of triangle i / 3, counted where its node is met first; then the
// nodes of no triangle.
__device__ __forceinline__ int first_meet(const BlockArgs& a, int i, int* g) {
  if (i < 3 * a.T) {
    *g = a.tri[(int64_t)(i % 3) * a.T + i / 3];
    return a.node_tri[a.start[*g]] == ((i / 3) << 2 | i % 3);
  }
  *g = i - 3 * a.T;
  return *g < a.N && a.start[*g] == a.start[*g + 1];
}

// exclusive sum over the workgroup's TH threads, and the whole
template <int TH>
__device__ __forceinline__ int exclusive(int x, int* sh, int* total) {
  const int t = threadIdx.x;
  sh[t] = x;
  __syncthreads();
  for (int o = 1; o < TH; o <<= 1) {
    const int y = t >= o ? sh[t - o] : 0;
    __syncthreads();
    sh[t] += y;
    __syncthreads();
  }
  *total = sh[TH - 1];
  const int r = sh[t] - x;
  __syncthreads();
  return r;
}

constexpr int kScanT = 1024;
__global__ __launch_bounds__(kScanT) void block_count_kernel(BlockArgs a) {
  __shared__ int sh[kScanT];
  const int i = blockIdx.x * kScanT + threadIdx.x;
  int g, total;
  exclusive<kScanT>(first_meet(a, i, &g), sh, &total);
  if (threadIdx.x == 0) a.sums[blockIdx.x] = total;
  if (i < a.n_fix) a.fix[a.fix_nodes[i]] = i;
}
__global__ __launch_bounds__(kScanT) void block_order_kernel(BlockArgs a) {
  __shared__ int sh[kScanT];
  int before, unused, g;
  exclusive<kScanT>((int)threadIdx.x < (int)blockIdx.x ? a.sums[threadIdx.x] : 0, sh, &before);  // at most kScanT workgroups
  const int i = blockIdx.x * kScanT + threadIdx.x;
  const int on = first_meet(a, i, &g);
  const int p = before + exclusive<kScanT>(on, sh, &unused);
  if (on) {
    a.pos[g] = p;
    a.order[p] = g;
  }
}

// One workgroup per block, a thread per node.  A triangle is listed by its vertex of the lowest
// position in the block, a neighbouring node by the first of its triangles that touches the block.
__global__ __launch_bounds__(kBlockNodes) void blocks_kernel(BlockArgs a) {
  constexpr int NB = kBlockNodes, NT = 2 * kBlockTris, NH = kBlockHalo, NI = kBlockItems;
  __shared__ int sh[NB];
  const int p = threadIdx.x, b = blockIdx.x, P = b * NB + p;
  const int64_t T = a.T;
  const int g = P < a.N ? a.order[P] : -1;
  const int k0 = g >= 0 ? a.start[g] : 0, k1 = g >= 0 ? a.start[g + 1] : 0;
  for (int i = p; i < NT; i += NB) {
    a.btri[b * NT + i] = -1;
    a.loc[b * NT + i] = 0;
  }
  for (int i = p; i < NH; i += NB) a.halo[b * NH + i] = -1;
  for (int i = p; i < NI; i += NB) {
    a.item[b * NI + i] = -1;
    a.iloc[b * NI + i] = 0;
  }
  a.node[P] = g;
  a.deg[P] = k1 - k0;
  a.more[P] = g >= 0 && a.extra ? a.extra[g] : 0;

  auto vertex = [&](int v, int s) { return a.tri[v * T + s]; };
  auto local = [&](int h) {
    const int q = a.pos[h] - b * NB;
    return q >= 0 && q < NB ? q : -1;
  };
  auto inside = [&](int s) {  // the lowest slot of a vertex in the block, 3: none
    for (int v = 0; v < 3; ++v)
      if (local(vertex(v, s)) >= 0) return v;
    return 3;
  };
  auto slot_of = [&](int s, int h) { return vertex(0, s) == h ? 0 : (vertex(1, s) == h ? 1 : 2); };
  // incidence c of this node lists its triangle: 1 inside the block, 2 across its border
  auto listed = [&](int c) {
    const int s = c >> 2;
    if ((c & 3) != slot_of(s, g)) return 0;
    bool whole = true;
    for (int v = 0; v < 3; ++v) {
      const int l = local(vertex(v, s));
      if (l < 0) whole = false;
      else if (l < p) return 0;
    }
    return whole ? 1 : 2;
  };
  auto first_touch = [&](int h) {  // the first incidence of h whose triangle touches the block
    for (int k = a.start[h]; k < a.start[h + 1]; ++k)
      if (inside(a.node_tri[k] >> 2) < 3) return (int)a.node_tri[k];
    return -1;
  };
  auto halo_slot = [&](int c) -> int32_t& {  // where the halo id of that incidence's node stands
    return a.hid[(3 * (c & 3) + inside(c >> 2)) * T + (c >> 2)];
  };
  auto id_of = [&](int h) {  // local id of a vertex, -1: not of the block's triangles
    const int l = local(h);
    if (l >= 0) return l;
    const int c = first_touch(h);
    return c < 0 ? -1 : NB + halo_slot(c);
  };
  auto vertices = [&](int s) { return id_of(vertex(0, s)) | id_of(vertex(1, s)) << 10 | id_of(vertex(2, s)) << 20; };
  auto give_up = [&] {
    if (p == 0) atomicOr(a.none, 1);
  };

  // every incidence of the block's nodes is one of its triangles', at most three of each
  int total;
  exclusive<NB>(k1 - k0 < 4 * NT ? k1 - k0 : 4 * NT, sh, &total);
  if (total > 3 * NT) return give_up();
  int n_in = 0, n_out = 0;
  for (int k = k0; k < k1; ++k) {
    const int l = listed(a.node_tri[k]);
    n_in += l == 1;
    n_out += l == 2;
  }
  const int before = exclusive<NB>(n_in | n_out << 16, sh, &total);  // at most 3 NT of each
  const int all_in = total & 0xffff, all_out = total >> 16;
  // inner triangles beyond their half of the list stand behind the others
  if (all_out + (all_in > kBlockTris ? all_in - kBlockTris : 0) > kBlockTris) return give_up();
  int in = before & 0xffff, out = before >> 16, n_halo = 0;
  for (int k = k0; k < k1; ++k) {
    const int c = a.node_tri[k], s = c >> 2, l = listed(c);
    if (!l) continue;
    int id;
    if (l == 1) {
      id = in < kBlockTris ? in : all_out + in;
      ++in;
    } else {
      id = kBlockTris + out++;
    }
    a.btri[b * NT + id] = s;
    for (int v = 0; v < 3; ++v) {
      const int h = vertex(v, s);
      if (local(h) >= 0) a.at[v * T + s] = id;
      else n_halo += first_touch(h) == (s << 2 | v);
    }
  }
  int h0 = exclusive<NB>(n_halo, sh, &total);
  if (total > NH) return give_up();
  for (int k = k0; k < k1; ++k) {
    const int c = a.node_tri[k], s = c >> 2;
    if (listed(c) != 2) continue;
    for (int v = 0; v < 3; ++v) {
      const int h = vertex(v, s);
      if (local(h) >= 0 || first_touch(h) != (s << 2 | v)) continue;
      a.halo[b * NH + h0] = a.pos[h];
      halo_slot(s << 2 | v) = h0++;
    }
  }
  __syncthreads();  // at, hid

  uint32_t e8[4] = {0, 0, 0, 0};
  int last = -1;
  for (int k = k0; k < k1; ++k) {
    const int c = a.node_tri[k], s = c >> 2, id = a.at[(c & 3) * T + s];
    if (listed(c)) a.loc[b * NT + id] = vertices(s);
    const bool fresh = k > k0 && a.tile[s] != last;
    last = a.tile[s];
    const uint32_t e = (uint32_t)((c & 3) * kBlockFlux + id) | (fresh ? 0x8000u : 0u);
    if (k - k0 < 8) e8[(k - k0) / 2] |= e << (16 * ((k - k0) & 1));
    else a.rest[a.more[P] + k - k0 - 8] = (uint16_t)e;
  }
  ((uint4*)a.inc)[P] = make_uint4(e8[0], e8[1], e8[2], e8[3]);

  const int f = g >= 0 ? a.fix[g] : -1;
  const int b0 = f >= 0 ? a.fix_bedge_start[f] : 0, nb = f >= 0 ? a.fix_bedge_start[f + 1] - b0 : 0;
  const int first = exclusive<NB>(nb < NI + 1 ? nb : NI + 1, sh, &total);
  if (total > NI) return give_up();  // (255 items of one node at most: a block of more has two nodes of them)
  a.bitem[P] = first << 8 | (nb < 256 ? nb : 255);
  if (nb > 255) atomicOr(a.none, 1);
  for (int q = 0; q < nb; ++q) {
    a.item[b * NI + first + q] = a.fix_bedge[b0 + q];
    const int v = vertices(a.badj[a.fix_bedge[b0 + q] >> 1]);
    a.iloc[b * NI + first + q] = v;
    if (v < 0) atomicOr(a.none, 1);  // a boundary edge beside a triangle without its node
  }
}

// A block of device memory cut into 256-byte aligned pieces.
struct Pieces {
  char* base = nullptr;
  size_t at = 0;
  template <class U>
  void take(U** p, int64_t n) {
    *p = (U*)(base + at);
    at += (sizeof(U) * (size_t)(n > 0 ? n : 1) + 255) & ~(size_t)255;
  }
};

int64_t max_degree(const fvm_mesh* m) {
  int64_t most = 0;
  for (int64_t g = 0; g < m->N; ++g) most = std::max<int64_t>(most, m->h_node_tri_start[g + 1] - m->h_node_tri_start[g]);
  return most;
}
constexpr int64_t kNodeDegree = 40, kBlockDegree = 200;

// extra[g]: units(degree) summed over the nodes before g; empty when no node has any
template <class F>
std::vector<int32_t> running(const fvm_mesh* m, F units, int64_t* total) {
  int64_t sum = 0;
  std::vector<int32_t> r;
  for (int64_t g = 0; g < m->N; ++g) sum += units(m->h_node_tri_start[g + 1] - m->h_node_tri_start[g]);
  *total = sum;
  if (sum == 0) return r;
  r.resize(m->N);
  sum = 0;
  for (int64_t g = 0; g < m->N; ++g) {
    r[g] = (int32_t)sum;
    sum += units(m->h_node_tri_start[g + 1] - m->h_node_tri_start[g]);
  }
  return r;
}

}  // namespace

namespace fvm {

// Queues the kernels on the null stream, as the mesh's geometry kernels.
int make_node_lists(fvm_mesh* m) {
  // one group of lanes adds a node's incidences, eight a round of about 1 us: with a hub the
  // tile kernels, which share its triangles among their workgroups, are faster (RHS, us, node
  // against tile kernels: 6.1 / 7.5 at a degree of 28, 7.0 / 6.9 at 40, 15 / 10 at 100, 126 / 16 at
  // 1,000, 525 / 25 at 4,000)
  if (max_degree(m) > kNodeDegree) return FVM_OK;
  for (int32_t f = 0; f < m->n_fix; ++f) {
    const int32_t b0 = m->h_fix_bedge_start[f];
    if (m->h_fix_bedge_start[f + 1] - b0 > 255 || b0 >= 1 << 23) return FVM_OK;  // the tile kernels
  }
  int64_t n_extra;
  const std::vector<int32_t> extra = running(m, [](int d) { return d > kL ? (d + kL - 1) / kL - 1 : 0; }, &n_extra);
  const int64_t N = m->N, blocks = N + n_extra;
  Pieces P;
  int32_t* d_extra = nullptr;
  auto cut = [&] {
    P.at = 0;
    P.take(&m->node_ent, kL * blocks);
    P.take(&m->node_next, blocks);
    P.take(&m->node_bed, N);
    P.take(&d_extra, (int64_t)extra.size());
  };
  cut();
  m->node_ent = nullptr;
  FVM_HIP(dev_malloc((void**)&P.base, P.at));
  cut();
  if (!extra.empty())
    FVM_HIP(hipMemcpy(d_extra, extra.data(), sizeof(int32_t) * extra.size(), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(node_lists_kernel, dim3((unsigned)((N * kL + 255) / 256)), dim3(256), 0, 0, N, m->T, m->tri,
                     m->node_tri_start, m->node_tri, m->tile_tri_start, m->n_tiles, extra.empty() ? nullptr : d_extra,
                     m->node_ent, m->node_next, m->node_bed);
  if (m->n_fix > 0)
    hipLaunchKernelGGL(node_bed_kernel, dim3((unsigned)((m->n_fix + 255) / 256)), dim3(256), 0, 0, m->n_fix,
                       m->fix_nodes, m->fix_bedge_start, m->node_bed);
  return FVM_OK;
}

// The lists of the blocks, made by the first call for this mesh; n = 0 when there are none.
int mesh_blocks(const fvm_mesh* m, MeshBlocks* out, hipStream_t s) {
  std::lock_guard<std::mutex> lock(m->blocks_mutex);
  if (!m->blocks_made) {
    const int64_t N = m->N, T = m->T, n = (N + kBlockNodes - 1) / kBlockNodes;
    // each triangle is in a block's list; a hub's thread adds its triangles alone, which holds up
    // every stage (20 steps with a hub of 100: 1.3 ms, the multi-kernel loop 2.5; 200: 2.1 / 2.6;
    // 300: 3.1 / 2.7)
    int64_t n_rest;
    if (N > 65536 || m->grouped || T > n * 2 * kBlockTris || max_degree(m) > kBlockDegree) {
      m->blocks_made = true;
      *out = m->blocks;
      return FVM_OK;
    }
    const std::vector<int32_t> extra = running(m, [](int d) { return d > 8 ? d - 8 : 0; }, &n_rest);
    struct Memory {
      void *work = nullptr, *lists = nullptr;
      ~Memory() {
        if (work) (void)dev_free(work);
        if (lists) (void)hipFree(lists);
      }
    } mem;
    BlockArgs a;
    a.N = (int)N;
    a.T = (int)T;
    a.n_tiles = m->n_tiles;
    a.n_fix = m->n_fix;
    a.tri = m->tri;
    a.start = m->node_tri_start;
    a.node_tri = m->node_tri;
    a.tile_tri_start = m->tile_tri_start;
    a.fix_nodes = m->fix_nodes;
    a.fix_bedge_start = m->fix_bedge_start;
    a.fix_bedge = m->fix_bedge;
    a.badj = m->badj;
    const int scan = (int)((3 * T + N + kScanT - 1) / kScanT);  // at most 832
    Pieces W, L;
    int32_t* d_extra;
    auto cut = [&] {
      W.at = L.at = 0;
      W.take(&a.pos, N);
      W.take(&a.order, N);
      W.take(&a.tile, T);
      W.take(&a.fix, N);
      W.take(&a.sums, scan);
      W.take(&a.at, 3 * T);
      W.take(&a.hid, 9 * T);
      W.take(&a.none, 1);
      W.take(&d_extra, (int64_t)extra.size());
      L.take(&a.inc, 8 * n * kBlockNodes);
      L.take(&a.node, n * kBlockNodes);
      L.take(&a.bitem, n * kBlockNodes);
      L.take(&a.deg, n * kBlockNodes);
      L.take(&a.more, n * kBlockNodes);
      L.take(&a.btri, n * 2 * kBlockTris);
      L.take(&a.loc, n * 2 * kBlockTris);
      L.take(&a.halo, n * kBlockHalo);
      L.take(&a.item, n * kBlockItems);
      L.take(&a.iloc, n * kBlockItems);
      L.take(&a.rest, n_rest);
    };
    cut();
    FVM_HIP(dev_alloc(&mem.work, W.at));
    FVM_HIP(dev_malloc(&mem.lists, L.at));
    W.base = (char*)mem.work;
    L.base = (char*)mem.lists;
    cut();
    a.extra = extra.empty() ? nullptr : d_extra;
    if (!extra.empty())
      FVM_HIP(hipMemcpyAsync(d_extra, extra.data(), sizeof(int32_t) * extra.size(), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(block_setup_kernel, dim3((unsigned)((std::max(N, T) + 255) / 256)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(block_count_kernel, dim3((unsigned)scan), dim3(kScanT), 0, s, a);
    hipLaunchKernelGGL(block_order_kernel, dim3((unsigned)scan), dim3(kScanT), 0, s, a);
    hipLaunchKernelGGL(blocks_kernel, dim3((unsigned)n), dim3(kBlockNodes), 0, s, a);
    int32_t none = 0;
    FVM_HIP(hipGetLastError());
    FVM_HIP(hipMemcpyAsync(&none, a.none, sizeof none, hipMemcpyDeviceToHost, s));
    FVM_HIP(hipStreamSynchronize(s));
    if (!none) {
      MeshBlocks& B = m->blocks;
      B.n = (int32_t)n;
      B.inc = a.inc;
      B.rest = a.rest;
      B.node = a.node;
      B.bitem = a.bitem;
      B.deg = a.deg;
      B.more = a.more;
      B.tri = a.btri;
      B.loc = a.loc;
      B.halo = a.halo;
      B.item = a.item;
      B.iloc = a.iloc;
      m->block_mem = mem.lists;
      mem.lists = nullptr;
    }
    m->blocks_made = true;
  }
  *out = m->blocks;
  return FVM_OK;
}

}  // namespace fvm

// For tests (not in fvm_hip.h): the mesh's blocks, 0: none, -1: not made yet.
extern "C" int64_t fvm_test_mesh_blocks(const fvm_mesh* m) { return m->blocks_made ? m->blocks.n : -1; }
