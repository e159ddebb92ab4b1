// Connected components of a graph held as CSR, edges taken in both directions.
//
// Reference: sparse/csgraph/_components.pyx:86-177 (find_components_sparse,
// an iterative DFS over CSR and CSC) and :15-81 (find_components, the dense
// crawl).  Both number components by their smallest vertex, in increasing
// order.  Here every vertex carries a label that only decreases, a union-find
// forest in which a label is never above its vertex: one pass over the edges
// joins the two ends' trees, hooking the larger root under the smaller with a
// compare-and-swap that only ever takes a root.  Labels may be read stale
// (another XCD's L2): a stale label is still one of the vertex's own tree, the
// swap fails on a root that is one no longer and returns its present label,
// and the join goes on from there.  So every edge is joined when the pass
// ends -- no second pass, and nothing for the host to read.  A component's
// smallest vertex is never hooked, so it ends as the root: labels are the
// components' smallest vertices, which rank into the reference's ids.
#include "rbg_common.hpp"

namespace rbg {

constexpr int CC_HOOKS = 2;  // hooking passes before the join (100 + 115 us; one: 56 + 296, three: 110 + 114)
constexpr int32_t CC_SMALL = 1024;  // vertices up to which they cost more than they save (n = 300: 45 us without, 80 with; 4096, 8 edges each: 448, 78)
constexpr int CC_STEPS = 64;  // of a compression before the last

// A first forest: each vertex under the first vertex of its row, if smaller
// (in a closed graph numbered parents first, a founder of its own).
static __global__ void k_cc_init(const int64_t* __restrict__ indptr, const int32_t* __restrict__ indices,
                                 int32_t* __restrict__ lab, int32_t n) {
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t e = indptr[v];
    const int32_t w = e < indptr[v + 1] ? indices[e] : (int32_t)v;
    lab[v] = w < (int32_t)v ? w : (int32_t)v;
  }
}

// A label through this workgroup's caches; may be stale (see above).
static __device__ inline int32_t cc_load(const int32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The root of x as far as the labels read tell; vertices on the way are moved
// up to their grandparents.
static __device__ inline int32_t cc_find(int32_t* lab, int32_t x) {
  int32_t p = cc_load(&lab[x]);
  while (p != x) {
    const int32_t g = cc_load(&lab[p]);
    if (g == p) return p;
    __hip_atomic_store(&lab[x], g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    x = g;
    p = cc_load(&lab[x]);
  }
  return x;
}

static __device__ inline void cc_join(int32_t* lab, int32_t a, int32_t b) {
  while (a != b) {
    const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
    const int32_t seen = atomicCAS(&lab[hi], hi, lo);
    if (seen == hi) return;
    a = cc_find(lab, seen);  // below hi: every turn lowers one end
    b = cc_find(lab, lo);
  }
}

// One entry of every row hooked, a thread per vertex: the larger of the two
// labels (roots, after a compression) under the smaller, without asking
// whether another hook came first -- the join pass makes every edge good.  A
// few such passes leave few trees, so that the join pass finds most of its
// edges settled at once; straight away its edges meet stale labels and queue
// up at the swap (300,007 vertices, 15 M edges: 1.94 ms against 0.24 ms for all launches; four rounds
// of hooking over every edge, each with a wait of the host, took 1.85 ms).
// Towards the end most edges hook the same root, and atomics on one address
// are served one by one: of a wave's hooks of one root only the smallest goes
// out, and only if it lowers the label as it stands.
static __global__ void k_cc_hook(const int64_t* __restrict__ indptr, const int32_t* __restrict__ indices, int32_t n,
                                 int32_t k, int32_t* lab) {
  const int lane = threadIdx.x & 63;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t v0 = blockIdx.x * (int64_t)blockDim.x + threadIdx.x - lane; v0 < n; v0 += stride) {
    const int64_t v = v0 + lane, e = v < n ? indptr[v] + k : 0;
    int32_t a = 0, b = 0;
    if (v < n && e < indptr[v + 1]) {
      a = cc_load(&lab[v]);
      b = cc_load(&lab[indices[e]]);
    }
    const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
    bool hook = a != b;
    const uint64_t hooks = __ballot(hook);
    if (hooks) {  // the first hooking lane's root
      const int lead = __ffsll((unsigned long long)hooks) - 1;
      const int32_t root = __builtin_amdgcn_readlane(hi, lead);
      const bool same = hook && hi == root;
      int32_t least = same ? lo : 0x7fffffff;
      for (int o = 32; o > 0; o >>= 1) {
        const int32_t q = __shfl_xor(least, o, 64);
        least = q < least ? q : least;
      }
      if (lane == lead && least < __hip_atomic_load(&lab[root], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&lab[root], least);
      hook = hook && !same;
    }
    if (hook && lo < __hip_atomic_load(&lab[hi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(&lab[hi], lo);
  }
}

// One wave per vertex v, a lane per edge (v, w).  Most edges end at the first
// comparison: w's label is v's root already.
static __global__ __launch_bounds__(256) void k_cc_join(const int64_t* __restrict__ indptr,
                                                        const int32_t* __restrict__ indices, int32_t n, int32_t* lab) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * 4;
  for (int64_t v = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); v < n; v += waves) {
    const int64_t e1 = indptr[v + 1];
    for (int64_t e = indptr[v] + lane; e < e1; e += 64) {
      const int32_t w = indices[e];
      const int32_t a = cc_load(&lab[v]);
      if (cc_load(&lab[w]) != a) cc_join(lab, cc_find(lab, a), cc_find(lab, w));
    }
  }
}

// Every vertex under its root, or `most` labels up its way: a first forest may
// be one long path (vertices in a row, each under the one before), whose walk
// to the root would be as long for the last of them.  64 a pass shorten the path
// 64 times a pass, and a vertex left on the way is under one of its own tree.
static __global__ void k_cc_compress(int32_t* lab, int32_t n, int32_t most) {
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n; v += (int64_t)gridDim.x * blockDim.x) {
    int32_t x = cc_load(&lab[v]), p = cc_load(&lab[x]);
    for (int32_t step = 1; p != x && step < most; step++) {
      x = p;
      p = cc_load(&lab[x]);
    }
    lab[v] = x;
  }
}

}  // namespace rbg

using namespace rbg;

extern "C" {

int rbg_components(const int64_t* indptr, const int32_t* indices, int32_t n, int32_t* labels, int32_t* flags,
                   int32_t* rounds, rbg_stream_t stream) {
  hipStream_t s = (hipStream_t)stream;
  if (n < 0 || (n > 0 && (!indptr || !labels || !flags))) return RBG_E_ARG;
  if (rounds) *rounds = 0;
  if (n == 0) return 0;
  const int grid = (int)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096);
  const int join_grid = (int)((n + 3) / 4 < 8192 ? (n + 3) / 4 : 8192);  // a wave per vertex
  hipLaunchKernelGGL(k_cc_init, dim3(grid), dim3(256), 0, s, indptr, indices, labels, n);
  RBG_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(256), 0, s, labels, n, CC_STEPS);
  RBG_CHECK_LAUNCH();
  for (int32_t r = 0; r < CC_HOOKS && n > CC_SMALL; r++) {
    hipLaunchKernelGGL(k_cc_hook, dim3(grid), dim3(256), 0, s, indptr, indices, n, 1 + r % 2, labels);
    RBG_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(256), 0, s, labels, n, CC_STEPS);
    RBG_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(k_cc_join, dim3(join_grid), dim3(256), 0, s, indptr, indices, n, labels);
  RBG_CHECK_LAUNCH();
  hipLaunchKernelGGL(k_cc_compress, dim3(grid), dim3(256), 0, s, labels, n, 0x7fffffff);
  RBG_CHECK_LAUNCH();
  if (rounds) *rounds = 1;
  return 0;
}

}  // extern "C"
