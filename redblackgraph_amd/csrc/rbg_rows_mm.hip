// Dense AVOS product C = A (x) B of operands with few entries (closures of
// pedigrees hold under 1% of their cells): the entries of both are gathered
// row by row, and row i of C takes A[i][k] (x) B[k][j] for the present pairs
// only, in place of the M K N terms of the blocked kernels (rbg_dense_mm.hip).
//
// Reference: redblack.c.src:554-700 (the 'ij,jk' einsum loop).  Terms with an
// absent operand are the loop's neutral ones.  The sum is order-free: in the encoding -1 -> 0,
// v -> v, absent -> all ones it is one unsigned min.
//
// Three launches, nothing read by the host:
//   scan  a wave per row of A and B: the row's entries and their number, and
//         the domain check of the blocked fast kernel (rbg_matmul_precheck_*);
//   plan  the number of present pairs;
//   rows  a workgroup per row of C: N cells in LDS, a wave per entry of A's
//         row, lanes over the entries of B's row, LDS atomic min.
// N = 8192 int32, W @ W of the closure of a 24-generation pedigree (0.56% of
// the cells): scan 123 us (0.54 GB, 4.4 TB/s), plan 8, rows 177, of which 35
// write C, about 90 wait for B's rows and the rest is the terms' arithmetic
// (all avos_product: 227; one of B's rows at a time: 267); 26.1 ms blocked.
#include "fw_kernels.hpp"

namespace rbg {

// Taken when the present pairs are at most 1 in ROWS_MM_PAIRS of the M K N
// terms, no row has more entries than a quarter of its length (or 64), no value
// is below -1, and the pairs take less time than the blocked kernels would
// (mm_limits).  Near the first line (both operands 12% full) it takes, against
// the blocked kernel (us): int32 63 / 277 at n = 512, 239 / 705 at 2048, 14640
// / 27490 at 8192; int64 2218 / 11120 at 4096.  Operands not taken pay for the
// scan in place of rbg_matmul_precheck_* (within 2%, n = 256 to 8192).
constexpr int64_t ROWS_MM_PAIRS = 64;
constexpr int ROWS_MM_NT = 256;
constexpr int ROWS_MM_LDS = 64 * 1024;
constexpr int ROWS_MM_COUNTERS = 16;  // pairs are summed in 16 words on lines of their own

enum : uint32_t {
  MM_INVALID = 1u << 31,  // a value below -1
  MM_DOMAIN = 1u << 30,   // outside the blocked fast kernel's domain
  MM_WIDE = 1u << 29,     // more entries than slots
  MM_COUNT = MM_WIDE - 1,
};

template <typename T>
struct MmList {
  uint32_t* head;  // entries | MM_* flags
  int32_t* col;    // row r's at [r * slots]
  T* val;
  int64_t slots;
};
template <typename T>
struct MmWork {
  unsigned long long* pairs;  // [16 * ROWS_MM_COUNTERS]
  MmList<T> a, b;
};

// a quarter of a row, and of rows up to 256 columns 64 or all
static inline int64_t mm_slots(int64_t cols) { return cols / 4 < 64 ? (cols < 64 ? cols : 64) : cols / 4; }

template <typename T>
static int64_t mm_layout(int64_t M, int64_t K, int64_t N, char* base, MmWork<T>* w) {
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += (bytes + 255) & ~(int64_t)255;
    return base + at;
  };
  auto list = [&](int64_t rows, int64_t cols) {
    const int64_t s = mm_slots(cols);
    char* head = take(4 * rows);
    char* col = take(4 * rows * s);
    char* val = take((int64_t)sizeof(T) * rows * s);
    return MmList<T>{(uint32_t*)head, (int32_t*)col, (T*)val, s};
  };
  char* pairs = take(8 * 16 * ROWS_MM_COUNTERS);
  const MmList<T> a = list(M, K), b = list(K, N);
  if (w) *w = MmWork<T>{(unsigned long long*)pairs, a, b};
  return o;
}

// The most present pairs for which the entries are faster, where the blocked
// fast kernel would follow (operands in its domain) and where the general one
// would, in ns of what was measured: here 2.5 + K / 100 a row of C and, on each
// of the workgroups that run at once, 3 a pair (4, and once for every part,
// where a row of C does not fit the LDS); there 50,000, 200 (int64 650; general
// 2,000 and 3,000) a k for every round of 256 tiles, and the operands'
// conversion.  Times (us, entries / blocked fast / general), int32: 10% full
// 2^18 x 64 x 64 924 / 490 / 838, 2^16 x 16 x 16 195 / 104 / 150, 2^13 x 32 x 64
// 61 / 97 / 151, 2^17 x 256 x 8 800 / 869 / 1281; 12% 300 x 1024 x 16000 800 /
// 600 / 4595; 10% 2000 x 500 x 40000 14500 / 2340 / 27100, 2% 767 / 2250 / 18300;
// 5% 64 x 64 x 262144 7290 / 256 / 677; 64 x 2^18 x 64 1910 / 65100 / 489000.
// `fits`: the entries may be faster also with operands in the domain, and their
// scan, a wave a row (2.3 ns a column), is no large part of the product.
struct MmLimits {
  int64_t cells, parts;  // of a row of C in LDS, and how often
  size_t lds;
  unsigned long long fast, general;
  bool fits;
};
template <typename T>
static MmLimits mm_limits(int64_t M, int64_t K, int64_t N) {
  MmLimits l;
  const int64_t fit = ROWS_MM_LDS / (int64_t)sizeof(T) - 16, V = 16 / (int64_t)sizeof(T);
  l.cells = N < fit ? N : fit;
  l.parts = (N + l.cells - 1) / l.cells;
  l.lds = (size_t)((l.cells + V - 1) / V * 16);
  const double a_cu = l.lds > 20 * 1024 ? 160 * 1024 / (double)l.lds : 8, slots = 256 * (double)(int)a_cu;
  const double few = (double)M * (double)K * (double)N / ROWS_MM_PAIRS;
  const double tiles = (double)((M + 127) / 128) * (double)((N + 127) / 128), rounds = tiles > 256 ? tiles / 256 : 1;
  const double cells = sizeof(T) * ((double)M * (double)K + (double)K * (double)N), out = sizeof(T) * (double)M * (double)N;
  auto most = [&](double blocked) {
    const double left = blocked - (2.5 + 0.01 * (double)K) * (double)M;
    const double p = left * ((double)M < slots ? (double)M : slots) / (l.parts > 1 ? 4.0 * (double)l.parts : 3.0);
    return p <= 0 ? 0ull : (unsigned long long)(p < few ? p : few);
  };
  const double fast = 50e3 + (sizeof(T) == 8 ? 650.0 : 200.0) * (double)K * rounds + (4 * cells + out) / 4000;
  l.fast = most(fast);
  l.general = most(50e3 + (sizeof(T) == 8 ? 3000.0 : 2000.0) * (double)K * rounds + (cells + out) / 4000);
  l.fits = l.fast != 0 && 2.3 * (double)(K > N ? K : N) < 0.15 * fast;
  return l;
}

// A row's entries in column order, by one wave: 16-byte loads, eight in
// flight per lane; vectors without an entry in the wave cost a test.
template <typename T>
__device__ inline void mm_scan_row(const T* __restrict__ x, int64_t cols, int64_t r, bool vec, MmList<T> l) {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int UN = 8;
  const int lane = threadIdx.x & 63;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int32_t* col = l.col + r * l.slots;
  T* val = l.val + r * l.slots;
  int64_t cnt = 0;
  bool invalid = false, domain = false;
  auto emit = [&](int64_t j, const T* v) {
    bool keep[V];
    int before = 0, total = 0;
#pragma unroll
    for (int c = 0; c < V; c++) {
      keep[c] = v[c] != 0;
      invalid |= v[c] < (T)-1;
      domain |= keep[c] && (j + c == r ? v[c] > (T)1 : v[c] == (T)1 || v[c] == (T)-1);
      const uint64_t m = __ballot(keep[c]);
      before += __popcll(m & below);
      total += __popcll(m);
    }
    int64_t p = cnt + before;
#pragma unroll
    for (int c = 0; c < V; c++)
      if (keep[c]) {
        if (p < l.slots) {
          col[p] = (int32_t)(j + c);
          val[p] = v[c];
        }
        p++;
      }
    cnt += total;
  };
  const int64_t nv = vec ? cols / V : 0;
  for (int64_t b = 0; b < nv; b += 64 * UN) {
    uint4 q[UN];
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int64_t k = b + 64 * u + lane;
      q[u] = k < nv ? ((const uint4*)x)[k] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (!__any((q[u].x | q[u].y | q[u].z | q[u].w) != 0)) continue;
      T v[V];
      if constexpr (V == 4) {
        v[0] = (T)q[u].x, v[1] = (T)q[u].y, v[2] = (T)q[u].z, v[3] = (T)q[u].w;
      } else {
        v[0] = (T)((uint64_t)q[u].x | (uint64_t)q[u].y << 32);
        v[1] = (T)((uint64_t)q[u].z | (uint64_t)q[u].w << 32);
      }
      emit((b + 64 * u + lane) * V, v);
    }
  }
  // the columns past the last whole vector, or all of an unaligned row
  for (int64_t b = nv * V; b < cols; b += 64 * UN) {
    T s[UN];
#pragma unroll
    for (int u = 0; u < UN; u++) {
      const int64_t j = b + 64 * u + lane;
      s[u] = j < cols ? x[j] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (!__any(s[u] != 0)) continue;
      T v[V] = {};
      v[0] = s[u];
      emit(b + 64 * u + lane, v);
    }
  }
  const uint32_t f = (__any(invalid) ? (uint32_t)MM_INVALID : 0u) | (__any(domain) ? (uint32_t)MM_DOMAIN : 0u) |
                     (cnt > l.slots ? (uint32_t)MM_WIDE : 0u);
  if (lane == 0) l.head[r] = (uint32_t)(cnt < l.slots ? cnt : l.slots) | f;
}

template <typename T>
static __global__ __launch_bounds__(NT) void k_mm_scan(const T* A, int64_t lda, bool veca, const T* B, int64_t ldb,
                                                      bool vecb, int64_t M, int64_t K, int64_t N, MmWork<T> w,
                                                      rbg_status* st) {
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) status_clear(st);
    if (threadIdx.x < ROWS_MM_COUNTERS) w.pairs[16 * threadIdx.x] = 0;
  }
  const int64_t q = blockIdx.x * (int64_t)(NT / 64) + threadIdx.x / 64;
  if (q < M)
    mm_scan_row<T>(A + q * lda, K, q, veca, w.a);
  else if (q - M < K)
    mm_scan_row<T>(B + (q - M) * ldb, N, q - M, vecb, w.b);
}

constexpr int MM_PLAN_NT = 1024;
template <typename T>
static __global__ __launch_bounds__(MM_PLAN_NT) void k_mm_plan(int64_t M, int64_t K, MmWork<T> w, rbg_status* st) {
  __shared__ unsigned long long sum;
  __shared__ uint32_t flags;
  if (threadIdx.x == 0) {
    sum = 0;
    flags = 0;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t r = blockIdx.x * (int64_t)(MM_PLAN_NT / 64) + threadIdx.x / 64;
  unsigned long long pairs = 0;
  uint32_t f = 0;
  if (r < K) f |= w.b.head[r];
  if (r < M) {
    const uint32_t h = w.a.head[r];
    f |= h;
    for (int64_t e = lane; e < (int64_t)(h & MM_COUNT); e += 64)
      pairs += w.b.head[w.a.col[r * w.a.slots + e]] & MM_COUNT;
  }
  for (int o = 32; o > 0; o >>= 1) pairs += __shfl_xor(pairs, o, 64);
  if (lane == 0) {
    if (pairs) atomicAdd(&sum, pairs);
    if (f & ~MM_COUNT) atomicOr(&flags, f & ~MM_COUNT);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (sum) atomicAdd(&w.pairs[16 * (blockIdx.x % ROWS_MM_COUNTERS)], sum);
    uint32_t s = 0;
    if (flags & (MM_INVALID | MM_DOMAIN)) s |= RBG_F_PRECOND_FAIL;
    if (flags & (MM_INVALID | MM_WIDE)) s |= RBG_F_CAPACITY;
    if (s & ~__hip_atomic_load(&st->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(&st->flags, s);
  }
}

// Row blockIdx.x of C.  `cells` of N in LDS at a time.  aux[5] = 1: written.
template <typename T>
static __global__ __launch_bounds__(ROWS_MM_NT) void k_mm_rows(MmWork<T> w, T* C, int64_t ldc, int64_t N, int64_t cells,
                                                              unsigned long long fast, unsigned long long general,
                                                              rbg_status* st) {
  using U = typename unsigned_of<T>::type;
  constexpr int V = 16 / (int)sizeof(T);
  extern __shared__ __align__(16) unsigned char lds[];
  U* acc = (U*)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  unsigned long long pairs = lane < ROWS_MM_COUNTERS ? w.pairs[16 * lane] : 0;
  for (int o = 8; o > 0; o >>= 1) pairs += __shfl_xor(pairs, o, 64);
  pairs = __shfl(pairs, 0, 64);
  // fast <= general; the flags are looked at apart: read for every comparison,
  // their latency comes before the sum of the pairs' (n = 8192: 179.7 -> 177.0 us)
  if (pairs > fast && (pairs > general || !(st->flags & RBG_F_PRECOND_FAIL))) return;
  if (st->flags & RBG_F_CAPACITY) return;
  if (tid == 0 && blockIdx.x == 0) st->aux[5] = 1;
  const int64_t i = blockIdx.x;
  const int count = (int)(w.a.head[i] & MM_COUNT);
  const int32_t* acol = w.a.col + i * w.a.slots;
  const T* aval = w.a.val + i * w.a.slots;
  int top = 0;
  for (int64_t j0 = 0; j0 < N; j0 += cells) {
    const int64_t n = N - j0 < cells ? N - j0 : cells;
    const bool whole = j0 == 0 && n == N;
    for (int64_t c = tid; c < (n + V - 1) / V; c += ROWS_MM_NT) ((uint4*)acc)[c] = make_uint4(~0u, ~0u, ~0u, ~0u);
    __syncthreads();
    // a wave's share of the row's entries: 64 at a time, their columns,
    // values and list lengths one per lane
    for (int e0 = (tid >> 6) * 64; e0 < count; e0 += ROWS_MM_NT) {
      const bool on = e0 + lane < count;
      const int k = on ? acol[e0 + lane] : 0;
      const T a = on ? aval[e0 + lane] : (T)0;
      const int len = on ? (int)(w.b.head[k] & MM_COUNT) : 0;
      const int here = count - e0 < 64 ? count - e0 : 64;
      // four of B's rows in flight; most have at most 64 entries
      // avos_product(ae, b) for operands >= -1 (ae is the wave's): a shift and
      // an add, an identity keeps the other operand or drops the term.  `top`:
      // the largest MSB sum, past width - 2 a term overflows.
      auto term = [&](T ae, int32_t c, T b) {
        U r;  // encoded
        if (ae == (T)1 || ae == (T)-1) {
          r = b > (T)1 ? (U)b : (b == ae ? (U)(ae == (T)1) : ~(U)0);
        } else {
          const int m = msb_u((U)b), sum = b > (T)1 ? m + msb_u((U)ae) : 0;
          top = sum > top ? sum : top;
          r = b > (T)1 ? ((U)(ae - 1) << m) + (U)b : (((ae & 1) != 0) == (b == (T)1) ? (U)ae : ~(U)0);
        }
        const int j = (int)(c - j0);
        if (r != ~(U)0 && (whole || (unsigned)j < (unsigned)n)) atomicMin(&acc[j], r);
      };
      for (int e = 0; e < here; e += 4) {
        int le[4];
        int64_t at[4];
        T ae[4], b[4];
        int32_t c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int q = e + u < here ? e + u : e;
          le[u] = e + u < here ? __builtin_amdgcn_readlane(len, q) : 0;
          at[u] = (int64_t)__builtin_amdgcn_readlane(k, q) * w.b.slots + lane;
          if constexpr (sizeof(T) == 4)
            ae[u] = (T)__builtin_amdgcn_readlane((int)a, q);
          else
            ae[u] = (T)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)a, q) |
                        (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)a >> 32), q) << 32);
          if (lane < le[u]) {
            c[u] = w.b.col[at[u]];
            b[u] = w.b.val[at[u]];
          }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (lane < le[u]) term(ae[u], c[u], b[u]);
          for (int t = 64 + lane; t < le[u]; t += 64) term(ae[u], w.b.col[at[u] + t - lane], w.b.val[at[u] + t - lane]);
        }
      }
    }
    __syncthreads();
    T* out = C + i * ldc + j0;
    if ((((uintptr_t)out) & 15) == 0) {
      for (int64_t c = tid; c < n / V; c += ROWS_MM_NT) {
        uint4 q = ((uint4*)acc)[c];
        if constexpr (V == 4) {
          q.x = (uint32_t)e_dec<int32_t>((int32_t)q.x), q.y = (uint32_t)e_dec<int32_t>((int32_t)q.y);
          q.z = (uint32_t)e_dec<int32_t>((int32_t)q.z), q.w = (uint32_t)e_dec<int32_t>((int32_t)q.w);
          ((uint4*)out)[c] = q;
        } else {
          const U* p = acc + c * V;
          ((ulonglong2*)out)[c] = make_ulonglong2((unsigned long long)e_dec<T>((T)p[0]),
                                                  (unsigned long long)e_dec<T>((T)p[1]));
        }
      }
      for (int64_t c = n / V * V + tid; c < n; c += ROWS_MM_NT) out[c] = e_dec<T>((T)acc[c]);
    } else {
      for (int64_t c = tid; c < n; c += ROWS_MM_NT) out[c] = e_dec<T>((T)acc[c]);
    }
    __syncthreads();
  }
  // a term that overflows: the general kernel keeps every event's rules
  if (__any(top > 8 * (int)sizeof(T) - 2) && lane == 0) atomicOr(&st->flags, (uint32_t)RBG_F_NEED_GENERAL);
}

template <typename T>
static int matmul_rows(const T* A, int64_t lda, const T* B, int64_t ldb, T* C, int64_t ldc, int64_t M, int64_t K,
                       int64_t N, void* ws, int64_t ws_bytes, rbg_status* st, hipStream_t s) {
  if (!A || !B || !C || !ws || !st || M <= 0 || K <= 0 || N <= 0 || lda < K || ldb < N || ldc < N ||
      K > 0x7fffffff || N > 0x7fffffff || M + K > 0x7fffffff || ((uintptr_t)ws & 255))
    return RBG_E_ARG;
  MmWork<T> w;
  if (ws_bytes < mm_layout<T>(M, K, N, (char*)ws, &w)) return RBG_E_WORKSPACE;
  constexpr int64_t V = 16 / (int64_t)sizeof(T);
  auto aligned = [&](const T* p, int64_t ld) { return ld % V == 0 && ((uintptr_t)p & 15) == 0; };
  hipLaunchKernelGGL((k_mm_scan<T>), dim3((unsigned)((M + K + NT / 64 - 1) / (NT / 64))), dim3(NT), 0, s, A, lda,
                     aligned(A, lda), B, ldb, aligned(B, ldb), M, K, N, w, st);
  RBG_CHECK_LAUNCH();
  const int64_t rows = M > K ? M : K;
  hipLaunchKernelGGL((k_mm_plan<T>), dim3((unsigned)((rows + MM_PLAN_NT / 64 - 1) / (MM_PLAN_NT / 64))),
                     dim3(MM_PLAN_NT), 0, s, M, K, w, st);
  RBG_CHECK_LAUNCH();
  const MmLimits l = mm_limits<T>(M, K, N);
  hipLaunchKernelGGL((k_mm_rows<T>), dim3((unsigned)M), dim3(ROWS_MM_NT), l.lds, s, w, C, ldc, N, l.cells, l.fast,
                     l.general, st);
  RBG_CHECK_LAUNCH();
  return 0;
}

}  // namespace rbg

using namespace rbg;

extern "C" {

int64_t rbg_matmul_rows_workspace_bytes(int64_t M, int64_t K, int64_t N, int32_t elem_bytes) {
  if (M <= 0 || K <= 0 || N <= 0) return 0;
  return elem_bytes == 8 ? mm_layout<int64_t>(M, K, N, nullptr, nullptr)
                         : mm_layout<int32_t>(M, K, N, nullptr, nullptr);
}
int32_t rbg_matmul_rows_fits(int64_t M, int64_t K, int64_t N, int32_t elem_bytes) {
  if (M <= 0 || K <= 0 || N <= 0) return 0;
  return (elem_bytes == 8 ? mm_limits<int64_t>(M, K, N) : mm_limits<int32_t>(M, K, N)).fits;
}
int rbg_matmul_rows_i32(const int32_t* A, int64_t lda, const int32_t* B, int64_t ldb, int32_t* C, int64_t ldc,
                        int64_t M, int64_t K, int64_t N, void* workspace, int64_t workspace_bytes, rbg_status* st,
                        rbg_stream_t stream) {
  return matmul_rows<int32_t>(A, lda, B, ldb, C, ldc, M, K, N, workspace, workspace_bytes, st, (hipStream_t)stream);
}
int rbg_matmul_rows_i64(const int64_t* A, int64_t lda, const int64_t* B, int64_t ldb, int64_t* C, int64_t ldc,
                        int64_t M, int64_t K, int64_t N, void* workspace, int64_t workspace_bytes, rbg_status* st,
                        rbg_stream_t stream) {
  return matmul_rows<int64_t>(A, lda, B, ldb, C, ldc, M, K, N, workspace, workspace_bytes, st, (hipStream_t)stream);
}

}  // extern "C"
