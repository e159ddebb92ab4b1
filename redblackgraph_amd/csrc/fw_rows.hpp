#pragma once
// Dense closure of a triangular matrix from its rows' direct entries.
//
// In a lower triangular matrix of the fast domain (fw_kernels.hpp) a product
// W[i][k] (x) W[k][j] is present only for i > k > j (the pivot cell's products
// change nothing).  So at step k of the naive loop (warshall.c.in:50-107)
//   * row k holds its final values (its last change was at a step below k), and
//   * W[i][k] still holds the input value A[i][k] (a change would need a step
//     above k).
// Row i therefore takes, for its direct entries k ascending,
//     C[i][j] = min(C[i][j], A[i][k] (x) C[k][j]),
// and that is the naive loop's whole sequence of values of the cell: W and the
// largest value ever written (the trajectory maximum) are the naive loop's.
// A pedigree's row has two direct entries at most, so a closure is about
// 1.5 n^2 / 2 products and n^2 cells written, against the n^3 / 6 relaxations
// of the blocked schedules, almost all of which have an absent operand: the
// closure is bound by reading the input and writing the result.
//
// Three launches, no waits between workgroups and nothing read by the host:
//   scan    one wave per row: reads the matrix once, checks the fast domain,
//           keeps each row's off-diagonal entries in ascending column order;
//   levels  one workgroup: each row's level (1 + the largest level among its
//           entries' rows), rows sorted by level;
//   close   one workgroup per slab of columns (128 bytes wide, a cache line a
//           row).  A column depends on itself alone, so a workgroup needs only
//           its own barrier between levels.
//
// Taken when every row has at most rows_slots(n) off-diagonal entries and the
// graph has at most ROWS_MAX_LEVELS levels; a graph with more entries keeps
// the blocked schedules (their cost does not grow with the entries).  Where
// the lines lie: a close pass reads one line per row, slab and entry, so its
// bytes are entries * n^2 / 2 * sizeof(T) from the L2s, level with the
// blocked closure's time at about n / 50 entries a row; and a path of L edges
// has a value of L bits at least, so a graph deeper than 64 levels overflows
// (general mode) unless it is full of shortcuts, which are entries.
#include "fw_kernels.hpp"

namespace rbg {

constexpr int ROWS_MAX_LEVELS = 64;
constexpr int64_t ROWS_MAX_N = 32768;  // one byte of LDS per row in the level pass
constexpr int ROWS_LEVEL_NT = 1024;
constexpr int ROWS_CLOSE_NT = 1024;

__host__ __device__ inline int rows_slots(int64_t n) {
  const int64_t s = n / 64;
  return (int)(s < 8 ? 8 : (s > 128 ? 128 : s));
}

// head word of a row: entries | (diagonal + 1) << 16 | ROW_* flags
enum : uint32_t {
  ROW_BAD = 1u << 20,    // a value outside the fast domain
  ROW_LOWER = 1u << 21,  // an entry below the diagonal
  ROW_UPPER = 1u << 22,  // an entry above it
  ROW_WIDE = 1u << 23,   // more than rows_slots(n) entries
};

// A row in level order: its first two entries inline (a pedigree's father and
// mother), the rest in the row's slots.
template <typename T>
struct alignas(16) RowRec {
  int32_t row;
  int32_t head;  // entries | (diagonal + 1) << 16
  int32_t c0, c1;
  T v0, v1;
};

// ctl words: [0] the side the close pass takes (0: not closed here, 1 lower),
// [1] levels, [CTL_START + l] first position of level l
constexpr int CTL_START = 8;

template <typename T>
struct RowsWork {
  int32_t* ctl;
  uint32_t* head;
  RowRec<T>* rec;
  int32_t* ecol;  // row i's entries at [i * slots]
  T* eval;
  int slots;
};

static inline int64_t rows_align(int64_t x) { return (x + 255) & ~(int64_t)255; }

template <typename T>
static inline int64_t rows_layout(int64_t n, char* base, RowsWork<T>* w) {
  const int slots = rows_slots(n);
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += rows_align(bytes);
    return base + at;
  };
  char* ctl = take(4 * (CTL_START + ROWS_MAX_LEVELS + 1));
  char* head = take(4 * n);
  char* rec = take((int64_t)sizeof(RowRec<T>) * n);
  char* ecol = take(4 * n * slots);
  char* eval = take((int64_t)sizeof(T) * n * slots);
  if (w) *w = RowsWork<T>{(int32_t*)ctl, (uint32_t*)head, (RowRec<T>*)rec, (int32_t*)ecol, (T*)eval, slots};
  return o;
}

// One row, by one wave.  Bound by reading the matrix: 16-byte loads, eight in
// flight per lane; only vectors with an entry go through the ballots that
// place the entries in column order.  A row past its slots is left at once
// (the blocked schedules read the matrix again).
template <typename T>
__device__ inline void rows_scan_row(const T* __restrict__ a, int64_t n, int64_t i, bool vec, RowsWork<T> w) {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int UN = 8;
  const int lane = threadIdx.x & 63;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int32_t* ecol = w.ecol + i * w.slots;
  T* eval = w.eval + i * w.slots;
  int cnt = 0;
  bool bad = false, lo = false, up = false;
  T diag = 0;
  auto emit = [&](int64_t j, const T* v) {
    bool keep[V];
    int before = 0, total = 0;
#pragma unroll
    for (int x = 0; x < V; x++) {
      const bool dg = j + x == i;
      keep[x] = v[x] != 0 && !dg;
      if (dg && v[x] != 0) {
        diag = v[x];
        bad |= v[x] < (T)-1 || v[x] > (T)1;
      }
      if (keep[x]) {
        bad |= v[x] < (T)2;
        lo |= j + x < i;
        up |= j + x > i;
      }
      const uint64_t m = __ballot(keep[x]);
      before += __popcll(m & below);
      total += __popcll(m);
    }
    int p = cnt + before;
#pragma unroll
    for (int x = 0; x < V; x++)
      if (keep[x]) {
        if (p < w.slots) {
          ecol[p] = (int32_t)(j + x);
          eval[p] = v[x];
        }
        p++;
      }
    cnt += total;
  };
  if (vec) {
    const int64_t nv = n / V;
    for (int64_t b = 0; b < nv && cnt <= w.slots; b += 64 * UN) {
      uint4 q[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int64_t k = b + 64 * u + lane;
        q[u] = k < nv ? ((const uint4*)a)[k] : make_uint4(0, 0, 0, 0);
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
    if (nv * V < n) {
      T v[V] = {};
      const int64_t j = nv * V + lane;
      if (j < n) v[0] = a[j];
#pragma unroll
      for (int x = 1; x < V; x++) v[x] = 0;
      // one column per lane here: the zeros beside it stand for columns of
      // other lanes and are never entries
      emit(j, v);
    }
  } else {
    for (int64_t b = 0; b < n && cnt <= w.slots; b += 64 * UN) {
      T s[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        const int64_t j = b + 64 * u + lane;
        s[u] = j < n ? a[j] : (T)0;
      }
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (!__any(s[u] != 0)) continue;
        T v[V] = {};
        v[0] = s[u];
        emit(b + 64 * u + lane, v);
      }
    }
  }
  const uint32_t d = __any(diag == (T)1) ? 2u : (__any(diag == (T)-1) ? 0u : 1u);
  const uint32_t f = (__any(bad) ? (uint32_t)ROW_BAD : 0u) | (__any(lo) ? (uint32_t)ROW_LOWER : 0u) |
                     (__any(up) ? (uint32_t)ROW_UPPER : 0u) | (cnt > w.slots ? (uint32_t)ROW_WIDE : 0u);
  if (lane == 0) w.head[i] = (uint32_t)(cnt < w.slots ? cnt : w.slots) | d << 16 | f;
}

struct LevelShared {
  int hist[ROWS_MAX_LEVELS + 1];
  int next[ROWS_MAX_LEVELS];
  uint32_t flags;
  int deep;
};

// Levels and level order of a lower triangular matrix's rows, by one
// workgroup.  Rows go in chunks of a thread each; a row's entries lie in
// earlier chunks (final) or its own, where the levels only grow, so a chunk
// repeats until no level changed: as many passes as the chunk is deep.
// Returns the flags of all rows.
template <typename T>
__device__ inline uint32_t rows_levels(RowsWork<T> w, int64_t n, LevelShared& L, uint8_t* lev, bool allowed) {
  const int tid = threadIdx.x, nthreads = blockDim.x;
  if (tid == 0) {
    L.flags = 0;
    L.deep = 0;
  }
  if (tid <= ROWS_MAX_LEVELS) L.hist[tid] = 0;
  __syncthreads();
  uint32_t f = 0;
  for (int64_t i = tid; i < n; i += nthreads) f |= w.head[i];
  f &= ROW_BAD | ROW_LOWER | ROW_UPPER | ROW_WIDE;
  if (f) atomicOr(&L.flags, f);
  __syncthreads();
  f = L.flags;
  if (!allowed || (f & (ROW_BAD | ROW_WIDE | ROW_UPPER))) {
    if (tid == 0) w.ctl[0] = 0;
    return f;
  }
  for (int64_t b = 0; b < n; b += nthreads) {
    const int64_t i = b + tid;
    const bool on = i < n;
    const int cnt = on ? (int)(w.head[i] & 0xffff) : 0;
    const int32_t* ec = w.ecol + i * w.slots;
    const int c0 = cnt > 0 ? ec[0] : 0, c1 = cnt > 1 ? ec[1] : 0;
    int lv = 0;
    if (on) lev[i] = 0;
    __syncthreads();
    for (;;) {
      int nl = 0;
      if (cnt > 0) nl = lev[c0] + 1;
      if (cnt > 1) nl = nl > lev[c1] + 1 ? nl : lev[c1] + 1;
      for (int e = 2; e < cnt; e++) {
        const int x = lev[ec[e]] + 1;
        nl = nl > x ? nl : x;
      }
      bool changed = nl > lv;
      if (nl >= ROWS_MAX_LEVELS) {
        L.deep = 1;
        changed = false;
      }
      if (changed) {
        lv = nl;
        lev[i] = (uint8_t)nl;
      }
      if (!__syncthreads_or(changed)) break;
    }
    if (L.deep) {  // written before the barrier above
      if (tid == 0) w.ctl[0] = 0;
      return f;
    }
    if (on) atomicAdd(&L.hist[lv], 1);
  }
  __syncthreads();
  if (tid == 0) {
    int at = 0, levels = 0;
    for (int l = 0; l < ROWS_MAX_LEVELS; l++) {
      L.next[l] = at;
      w.ctl[CTL_START + l] = at;
      if (L.hist[l]) levels = l + 1;
      at += L.hist[l];
    }
    w.ctl[CTL_START + ROWS_MAX_LEVELS] = at;
    w.ctl[1] = levels;
    w.ctl[0] = 1;
  }
  __syncthreads();
  for (int64_t i = tid; i < n; i += nthreads) {
    const uint32_t h = w.head[i];
    const int cnt = (int)(h & 0xffff);
    const int32_t* ec = w.ecol + i * w.slots;
    const T* ev = w.eval + i * w.slots;
    RowRec<T> r{(int32_t)i, (int32_t)(h & 0x3ffff), 0, 0, 0, 0};
    if (cnt > 0) r.c0 = ec[0], r.v0 = ev[0];
    if (cnt > 1) r.c1 = ec[1], r.v1 = ev[1];
    w.rec[atomicAdd(&L.next[lev[i]], 1)] = r;
  }
  return f;
}

// Left operand a of a lane's V cells: a (x) y for the cells y of the entry's
// row.  A cell below 2 is no operand (absent, or the diagonal's identity).
template <typename T, int V>
__device__ inline void rows_relax(typename unsigned_of<T>::type (&cur)[V], T a, const T (&y)[V], int& guard, T& tmax) {
  using U = typename unsigned_of<T>::type;
  const int ma = msb_u((U)a);
#pragma unroll
  for (int x = 0; x < V; x++) {
    const bool present = y[x] > (T)1;
    const int m = present ? msb_u((U)y[x]) : 0;
    const U p = present ? ((U)(a - 1) << m) + (U)y[x] : ~(U)0;
    guard = present && ma + m > guard ? ma + m : guard;
    cur[x] = p < cur[x] ? p : cur[x];
    tmax = (T)cur[x] > tmax ? (T)cur[x] : tmax;
  }
}

template <typename T, int V>
__device__ inline void rows_ld(const T* p, T (&y)[V]) {
  const uint4 q = *(const uint4*)p;
  if constexpr (V == 4) {
    y[0] = (T)q.x, y[1] = (T)q.y, y[2] = (T)q.z, y[3] = (T)q.w;
  } else {
    y[0] = (T)((uint64_t)q.x | (uint64_t)q.y << 32);
    y[1] = (T)((uint64_t)q.z | (uint64_t)q.w << 32);
  }
}

template <typename T, int V>
__device__ inline void rows_st(T* p, const T (&y)[V]) {
  if constexpr (V == 4)
    *(uint4*)p = make_uint4((uint32_t)y[0], (uint32_t)y[1], (uint32_t)y[2], (uint32_t)y[3]);
  else
    *(ulonglong2*)p = make_ulonglong2((unsigned long long)y[0], (unsigned long long)y[1]);
}

constexpr int ROWS_LANES = 8;  // lanes of 16 bytes per row segment: one 128-byte line
template <typename T>
__host__ __device__ inline int64_t rows_slab() {
  return ROWS_LANES * (16 / (int64_t)sizeof(T));
}

struct CloseShared {
  int start[ROWS_MAX_LEVELS + 1];
  long long top;
  int guard;
};

// One slab of columns through every level.  W rows are 16-byte aligned (ld a
// multiple of 128).  Eight lanes hold one row's segment; two rows per lane
// group are in flight so that the four loads of their entries' rows overlap.
template <typename T>
__device__ inline void rows_close_slab(CloseShared& L, RowsWork<T> w, T* W, int64_t ld, int64_t slab, int width,
                                       rbg_status* st) {
  using U = typename unsigned_of<T>::type;
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int UN = 2;
  const int tid = threadIdx.x, G = blockDim.x / ROWS_LANES;
  const int g = tid / ROWS_LANES;
  const int j0 = (int)(slab * rows_slab<T>());
  const int jl = j0 + (tid % ROWS_LANES) * V;
  const int levels = w.ctl[1];
  if (tid <= levels) L.start[tid] = w.ctl[CTL_START + tid];
  if (tid == 0) {
    L.top = 0;
    L.guard = 0;
  }
  __syncthreads();
  int guard = 0;
  T tmax = 0;
  for (int l = 0; l < levels; l++) {
    const int end = L.start[l + 1];
    for (int p = L.start[l] + g; p < end; p += UN * G) {
      RowRec<T> r[UN];
      T y0[UN][V], y1[UN][V];
      int cnt[UN];
#pragma unroll
      for (int u = 0; u < UN; u++) r[u] = w.rec[p + u * G < end ? p + u * G : p];
#pragma unroll
      for (int u = 0; u < UN; u++) {
        cnt[u] = r[u].head & 0xffff;
        if (cnt[u] > 0 && r[u].c0 >= j0) {
          rows_ld<T, V>(W + r[u].c0 * ld + jl, y0[u]);
        } else {
#pragma unroll
          for (int x = 0; x < V; x++) y0[u][x] = 0;
        }
        if (cnt[u] > 1 && r[u].c1 >= j0) {
          rows_ld<T, V>(W + r[u].c1 * ld + jl, y1[u]);
        } else {
#pragma unroll
          for (int x = 0; x < V; x++) y1[u][x] = 0;
        }
      }
#pragma unroll
      for (int u = 0; u < UN; u++) {
        if (p + u * G >= end) break;
        const int row = r[u].row;
        U cur[V];
        const T d = (T)((r[u].head >> 16) & 3) - 1;
#pragma unroll
        for (int x = 0; x < V; x++) {
          cur[x] = ~(U)0;
          if (row == jl + x) cur[x] = (U)e_enc<T>(d);
          if (cnt[u] > 0 && r[u].c0 == jl + x) cur[x] = (U)r[u].v0;
          if (cnt[u] > 1 && r[u].c1 == jl + x) cur[x] = (U)r[u].v1;
        }
        if (cnt[u] > 2) {
          const int32_t* ec = w.ecol + (int64_t)row * w.slots;
          const T* ev = w.eval + (int64_t)row * w.slots;
          for (int e = 2; e < cnt[u]; e++) {
            const int x = ec[e] - jl;
            if (x >= 0 && x < V) {
#pragma unroll
              for (int c = 0; c < V; c++)
                if (x == c) cur[c] = (U)ev[e];
            }
          }
        }
#pragma unroll
        for (int x = 0; x < V; x++) tmax = (T)cur[x] > tmax ? (T)cur[x] : tmax;
        if (cnt[u] > 0) rows_relax<T, V>(cur, r[u].v0, y0[u], guard, tmax);
        if (cnt[u] > 1) rows_relax<T, V>(cur, r[u].v1, y1[u], guard, tmax);
        if (cnt[u] > 2) {
          const int32_t* ec = w.ecol + (int64_t)row * w.slots;
          const T* ev = w.eval + (int64_t)row * w.slots;
          for (int e = 2; e < cnt[u]; e += 4) {
            T y[4][V], a[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const int c = e + q < cnt[u] ? ec[e + q] : -1;
              a[q] = e + q < cnt[u] ? ev[e + q] : (T)2;
              if (c >= j0) {
                rows_ld<T, V>(W + c * ld + jl, y[q]);
              } else {
#pragma unroll
                for (int x = 0; x < V; x++) y[q][x] = 0;
              }
            }
#pragma unroll
            for (int q = 0; q < 4; q++) rows_relax<T, V>(cur, a[q], y[q], guard, tmax);
          }
        }
        T o[V];
#pragma unroll
        for (int x = 0; x < V; x++) o[x] = e_dec<T>((T)cur[x]);
        rows_st<T, V>(W + row * ld + jl, o);
      }
    }
    __syncthreads();  // the level's rows are read by the next ones of this workgroup alone
  }
  const long long t = wave_max_i64(tmax);
  if ((tid & 63) == 0 && t > 0) atomicMax(&L.top, t);
  if (guard > width - 2) atomicMax(&L.guard, guard);
  __syncthreads();
  if (tid == 0) {
    if (L.top > __hip_atomic_load(&st->diameter_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      record_diameter(st, L.top);
    if (L.guard) atomicOr(&st->flags, (uint32_t)RBG_F_NEED_GENERAL);
  }
}

}  // namespace rbg
