#pragma once
// Dense closure of a matrix from its rows' direct entries.
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
// Four launches (three up to ROWS_PLACE_HERE rows), no waits between workgroups and nothing read by the host:
//   scan    one wave per row: reads the matrix once, checks the fast domain,
//           keeps each row's off-diagonal entries in ascending column order;
//   levels  one workgroup: each row's level (1 + the largest level among its
//           entries' rows) and its position in level order;
//   place   the rows' records in level order;
//   close   one workgroup per slab of columns (64 bytes of a row).  A column depends on itself alone, so a workgroup needs only
//           its own barrier between levels.
//
// Taken when every row has at most rows_slots(n) off-diagonal entries and the
// graph has at most ROWS_MAX_LEVELS levels; a graph with more entries keeps
// the blocked schedules, whose cost does not grow with the entries.  Where the
// lines lie: the close pass reads a line per row, slab and entry, and with the
// same number of entries in every row it measured (us, against the blocked
// closure) 151 / 157 at n = 100 with 12, 231 / 246 at 300 with 24, 274 / 563
// at 1000 with 25, 451 / 1489 at 2000 with 50, 1511 / 3747 at 4000 with 100
// and 7603 / 10283 at 8000 with 200, each growing with the entries.  A matrix
// not taken pays for the scan, which the blocked closure's load then repeats, and
// for the level pass: 20 us of 250 at n = 300 with 28, 70 of 10270 at 8000 with
// 204, and up to 110 of 305 where rows of ten entries lie in 28 levels (n = 200,
// unordered); one of another numbering that is tried and has too many cells above
// its largest value (rows_first_value) for two passes more, 10 to 20%.  A path of L edges
// has a value of L bits at least, so a graph deeper than 64 levels overflows
// (general mode) unless it is full of shortcuts, which are entries.
#include "fw_kernels.hpp"

namespace rbg {

constexpr int ROWS_MAX_LEVELS = 64;
constexpr int64_t ROWS_MAX_N = 32640;  // rows in 15 bits; a byte of LDS per row in the level pass
constexpr int64_t ROWS_ANY_MAX_N = 16384;  // other numberings: two bytes of LDS per row (rows_first_value)
constexpr int ROWS_MAX_CELLS = 4096;
constexpr int ROWS_LEVEL_NT = 1024;
constexpr int ROWS_CLOSE_NT = 1024;

__host__ __device__ inline int rows_slots(int64_t n) {
  const int64_t few = n / 12 < 8 ? 8 : (n / 12 > 24 ? 24 : n / 12), s = n / 40;
  return (int)(s < few ? few : (s > 200 ? 200 : s));
}

// A row for the level pass: entry 0's column | entry 1's column << 16
// (ROW_NONE where there is none) | ROW_MORE when it has more entries.  A row
// that keeps the matrix from being closed here is ROW_STOP | why.
enum : uint32_t {
  ROW_NONE = 0x7fff,
  ROW_MORE = 1u << 15,
  ROW_STOP = 1u << 31,
  STOP_BAD = 8,          // a value outside the fast domain
  STOP_WIDE = 16,        // more than rows_slots(n) entries
  ROW_BELOW = 32,        // with ROW_STOP: an entry below the diagonal
  ROW_ABOVE = 64,        // above it
  REC_UPPER = 1u << 26,  // in RowRec::p1_cnt: an entry above the diagonal
};
__host__ __device__ inline int rec_cnt(uint32_t w) { return (int)((w >> 16) & 0xff); }

// A row's first two entries (a pedigree's father and mother) inline, the rest
// in the row's slots.  Eight words; a quad of lanes loads two each.
template <typename T>
struct alignas(16) RowRec {
  uint32_t row_c0;  // row | column of entry 0 << 16
  uint32_t c1_p0;   // column of entry 1 | position of entry 0's row in level order << 16
  uint32_t p1_cnt;  // position of entry 1's row | entries << 16 | (diagonal + 1) << 24
  uint32_t pad;
  T v0, v1;
};
static_assert(sizeof(RowRec<int32_t>) == 32 && sizeof(RowRec<int64_t>) == 32, "a quad's two words per lane");

// ctl words: [0] the side the close pass takes (0: not closed here, 1 lower),
// [1] levels, [CTL_START + l] first position of level l
constexpr int CTL_START = 8;

template <typename T>
struct RowsWork {
  int32_t* ctl;
  uint32_t* entries;  // the level pass's word per row (scan)
  uint16_t* pos;      // each row's position in level order (levels)
  RowRec<T>* rec0;    // in row order (scan)
  RowRec<T>* rec;     // in level order (place)
  int32_t* ecol;  // row i's entries at [i * slots]
  T* eval;
  T* slab_top;      // largest W2 value of each slab
  uint32_t* cells;  // [0] number of cells with W2 > max W, then i | j << 16 of each
  int slots;
};

__host__ __device__ inline int64_t rows_align(int64_t x) { return (x + 255) & ~(int64_t)255; }

template <typename T>
__host__ __device__ inline int64_t rows_layout(int64_t n, char* base, RowsWork<T>* w) {
  const int slots = rows_slots(n);
  int64_t o = 0;
  auto take = [&](int64_t bytes) {
    const int64_t at = o;
    o += rows_align(bytes);
    return base + at;
  };
  char* ctl = take(4 * (CTL_START + ROWS_MAX_LEVELS + 1));
  char* entries = take(4 * (n + 3));  // read four at a time
  char* pos = take(2 * (n + 3));
  char* rec0 = take((int64_t)sizeof(RowRec<T>) * n);
  char* rec = take((int64_t)sizeof(RowRec<T>) * n);
  char* ecol = take(4 * n * slots);
  char* eval = take((int64_t)sizeof(T) * n * slots);
  char* slab_top = take((int64_t)sizeof(T) * (n * (int64_t)sizeof(T) / 64 + 1));
  char* cells = take(4 * (1 + ROWS_MAX_CELLS));
  if (w) *w = RowsWork<T>{(int32_t*)ctl, (uint32_t*)entries, (uint16_t*)pos, (RowRec<T>*)rec0, (RowRec<T>*)rec, (int32_t*)ecol, (T*)eval,
                     (T*)slab_top, (uint32_t*)cells, slots};
  return o;
}

// One row, by one wave.  Bound by reading the matrix: 16-byte loads, eight in
// flight per lane; only vectors with an entry go through the ballots that
// place the entries in column order.  A row past its slots is read to its
// end all the same: the blocked schedules need the sides its entries lie on.
template <typename T>
__device__ inline void rows_scan_row(const T* __restrict__ a, int64_t n, int64_t i, bool vec, RowsWork<T> w) {
  constexpr int V = 16 / (int)sizeof(T);
  constexpr int UN = 8;
  const int lane = threadIdx.x & 63;
  const uint64_t below = ((uint64_t)1 << lane) - 1;
  int32_t* ecol = w.ecol + i * w.slots;
  T* eval = w.eval + i * w.slots;
  RowRec<T>& rec = w.rec0[i];
  uint32_t c0 = ROW_NONE, c1 = ROW_NONE;
  int cnt = 0;
  bool bad = false, up = false;
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
        if (p == 0) c0 = (uint32_t)(j + x), rec.v0 = v[x];
        if (p == 1) c1 = (uint32_t)(j + x), rec.v1 = v[x];
        p++;
      }
    cnt += total;
  };
  if (vec) {
    const int64_t nv = n / V;
    for (int64_t b = 0; b < nv; b += 64 * UN) {
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
    for (int64_t b = 0; b < n; b += 64 * UN) {
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
  // the lanes that met entries 0 and 1 hold their columns
  const uint64_t h0 = __ballot(c0 != ROW_NONE), h1 = __ballot(c1 != ROW_NONE);
  if (h0) c0 = (uint32_t)__builtin_amdgcn_readlane((int)c0, __ffsll((unsigned long long)h0) - 1);
  if (h1) c1 = (uint32_t)__builtin_amdgcn_readlane((int)c1, __ffsll((unsigned long long)h1) - 1);
  const uint32_t d = __any(diag == (T)1) ? 2u : (__any(diag == (T)-1) ? 0u : 1u);
  const uint32_t stop = (__any(bad) ? (uint32_t)STOP_BAD : 0u) | (cnt > w.slots ? (uint32_t)STOP_WIDE : 0u);
  const uint32_t upper = __any(up) ? (uint32_t)REC_UPPER : 0u;
  if (lane == 0) {
    rec.row_c0 = (uint32_t)i | c0 << 16;
    rec.c1_p0 = c1;
    rec.p1_cnt = (uint32_t)(cnt < w.slots ? cnt : w.slots) << 16 | d << 24 | upper;
    w.entries[i] = stop ? ROW_STOP | stop | ((int64_t)c0 < i ? ROW_BELOW : 0u) | (upper ? (uint32_t)ROW_ABOVE : 0u) : c0 | c1 << 16 | (cnt > 2 ? (uint32_t)ROW_MORE : 0u);
  }
}

struct LevelShared {
  int hist[ROWS_MAX_LEVELS];
  int next[ROWS_MAX_LEVELS];
  int marks[4];
  int third;
};

// Level and position of every row, by one workgroup of at least 64 threads
// and n / (4 H) rows; lev: n + 4 bytes of LDS.  Each thread holds 4 H rows'
// words (four neighbours, H times) in registers and sweeps them until no level
// changed, one barrier a sweep: a row's level only grows, and the sweeps are
// at most as many as the graph is deep (few more than one where the rows are
// numbered parents first).  The levels of a cyclic graph grow past
// ROWS_MAX_LEVELS.  One workgroup runs its code once, so its time is
// instruction fetches, barriers and LDS reads: short loops and few of them
// count for more here than loads in flight (N = 8192, 18 levels: 28 us against
// 93 us with one row per thread and pass, chunk by chunk, and 66 us with the
// records moved here, eight unrolled; N = 512: 12 us).  Returns the STOP_*
// reasons (or 2: too deep), 0 when the positions are in w.pos; `sides` has 1
// when entries lie below the diagonal, 2 above; L.third tells whether a row has
// more than two.
template <typename T, int H>
__device__ inline int rows_levels(RowsWork<T> w, int64_t n64, LevelShared& L, uint8_t* lev, int& sides) {
  const int tid = threadIdx.x, lane = tid & 63, nt = blockDim.x, n = (int)n64;
  if (tid < 4) L.marks[tid] = 0;
  if (tid == 0) L.third = 0;
  if (tid < ROWS_MAX_LEVELS) L.hist[tid] = 0;
  uint32_t e[4 * H];
  uint32_t lv[H];  // four levels each
#pragma unroll
  for (int h = 0; h < H; h++) {
    const int row = 4 * (h * nt + tid);
    uint4 q = make_uint4(0, 0, 0, 0);
    if (row < n) {
      q = *(const uint4*)(w.entries + row);
      *(uint32_t*)(lev + row) = 0;
    }
    e[4 * h] = q.x, e[4 * h + 1] = q.y, e[4 * h + 2] = q.z, e[4 * h + 3] = q.w;
    lv[h] = 0;
  }
  int facts = 0;  // STOP_*, ROW_BELOW, ROW_ABOVE
  bool more = false;
#pragma unroll
  for (int x = 0; x < 4 * H; x++) {
    const int row = 4 * ((x / 4) * nt + tid) + x % 4;
    if (row >= n) e[x] = ROW_NONE | ROW_NONE << 16;
    const uint32_t c0 = e[x] & 0x7fff, c1 = (e[x] >> 16) & 0x7fff;
    if (e[x] & ROW_STOP) {
      facts |= (int)(e[x] & 0xff);
      e[x] = (uint32_t)n | (uint32_t)n << 16;
      continue;
    }
    const bool m = (e[x] & ROW_MORE) != 0;
    more |= m;
    if (c0 != ROW_NONE) facts |= (int)c0 < row ? ROW_BELOW : ROW_ABOVE;
    if (c1 != ROW_NONE) facts |= (int)c1 < row ? ROW_BELOW : ROW_ABOVE;
    if (m && (w.rec0[row].p1_cnt & REC_UPPER)) facts |= ROW_ABOVE;
    e[x] = (c0 == ROW_NONE ? (uint32_t)n : c0) | (c1 == ROW_NONE ? (uint32_t)n : c1) << 16 | (m ? 1u << 31 : 0u);
  }
  __syncthreads();
  if (tid == 0) lev[n] = 255;  // an absent entry's level: below 0
  if (more) L.third = 1;
  __syncthreads();
  for (int it = 0;; it++) {
    bool changed = false;
    int worst = 0;
#pragma unroll
    for (int h = 0; h < H; h++) {
      if (4 * h * nt >= n) continue;  // no row of any thread
      const int row = 4 * (h * nt + tid);
      uint32_t nv = 0, third = 0;
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const uint32_t ex = e[4 * h + x];
        const int l0 = (uint8_t)(lev[ex & 0xffff] + 1), l1 = (uint8_t)(lev[(ex >> 16) & 0x7fff] + 1);
        const int nl = l0 > l1 ? l0 : l1;
        third |= (ex >> 31) << x;
        worst = nl > worst ? nl : worst;
        nv |= (uint32_t)nl << (8 * x);
      }
      while (third) {  // rows with further entries, four by a load
        const int x = __builtin_ctz(third);
        third &= third - 1;
        int nl = (int)(nv >> (8 * x) & 0xff);
        const int cnt = rec_cnt(w.rec0[row + x].p1_cnt);
        const int32_t* ec = w.ecol + (int64_t)(row + x) * w.slots;
        int k = 2;
        for (; k + 4 <= cnt; k += 4) {
          int c[4];
#pragma unroll
          for (int q = 0; q < 4; q++) c[q] = ec[k + q];
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int y = lev[c[q]] + 1;
            nl = nl > y ? nl : y;
          }
        }
        for (; k < cnt; k++) {
          const int y = lev[ec[k]] + 1;
          nl = nl > y ? nl : y;
        }
        worst = nl > worst ? nl : worst;
        nv = (nv & ~(0xffu << (8 * x))) | (uint32_t)(nl & 0xff) << (8 * x);
      }
      if (nv != lv[h]) {
        lv[h] = nv;
        changed = true;
        if (row + 3 < n)
          *(uint32_t*)(lev + row) = nv;
        else
          for (int x = 0; row + x < n; x++) lev[row + x] = (uint8_t)(nv >> (8 * x));
      }
    }
    int mark = (__any(changed) ? 1 : 0) | (__any(worst >= ROWS_MAX_LEVELS) ? 2 : 0);
    for (int k = 3; k < 7; k++) mark |= __any(facts & (1 << k)) ? 1 << k : 0;
    if (mark && lane == 0) atomicOr(&L.marks[it & 3], mark);
    if (tid == 0) L.marks[(it + 2) & 3] = 0;  // read two sweeps ago, marked two sweeps on
    __syncthreads();
    const int marks = L.marks[it & 3];  // the same for every thread: the branches below are uniform
    sides = marks >> 5;
    if (marks & (2 | STOP_BAD | STOP_WIDE)) return marks & (2 | STOP_BAD | STOP_WIDE);
    if (!(marks & 1)) break;
  }
#pragma unroll
  for (int x = 0; x < 4 * H; x++)
    if (4 * ((x / 4) * nt + tid) + x % 4 < n) atomicAdd(&L.hist[(lv[x / 4] >> (8 * (x % 4))) & 0xff], 1);
  __syncthreads();
  if (tid < ROWS_MAX_LEVELS) {  // the first wave: an exclusive scan of the level sizes
    const int c = L.hist[tid];
    int incl = c;
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (tid >= d) incl += o;
    }
    L.next[tid] = incl - c;
    w.ctl[CTL_START + tid] = incl - c;
    const uint64_t some = __ballot(c != 0);
    if (tid == 0) {
      w.ctl[CTL_START + ROWS_MAX_LEVELS] = n;
      w.ctl[1] = 64 - __clzll(some);
    }
  }
  __syncthreads();
  for (int i = 4 * tid; i < n; i += 4 * nt) {
    uint16_t at[4];
#pragma unroll
    for (int x = 0; x < 4; x++) at[x] = i + x < n ? (uint16_t)atomicAdd(&L.next[lev[i + x]], 1) : (uint16_t)0;
    *(ushort4*)(w.pos + i) = make_ushort4(at[0], at[1], at[2], at[3]);
  }
  return 0;
}
static_assert(ROWS_MAX_LEVELS == 64, "one wave scans the level sizes");

// Row i's record to its place in level order, with its entries' places.
template <typename T>
__device__ inline void rows_place(RowsWork<T> w, int64_t i) {
  const uint4* p = (const uint4*)(w.rec0 + i);
  uint4 a = p[0];
  const uint4 v = p[1];
  const int cnt = rec_cnt(a.z);
  if (cnt > 0) a.y = (a.y & 0xffff) | (uint32_t)w.pos[a.x >> 16] << 16;
  if (cnt > 1) a.z |= w.pos[a.y & 0xffff];
  uint4* o = (uint4*)(w.rec + w.pos[i]);
  o[0] = a;
  o[1] = v;
}

// Left operand a on a lane's V cells y of the entry's row: cells are kept as
// value - 1 with all ones for an absent one, so that the sum is an unsigned
// min and the stored value cell + 1.  A y below 2 is no operand (absent, or
// the diagonal's identity).  top: largest y met (for the overflow guard);
// tmax: largest cell (all ones counts as -1).
template <typename T, int V>
__device__ inline void rows_relax(typename unsigned_of<T>::type (&cur)[V], T a, const T (&y)[V], T& top, T& tmax) {
  using U = typename unsigned_of<T>::type;
  constexpr int HI = 8 * (int)sizeof(T) - 1;
  const U am = (U)(a - 1);
#pragma unroll
  for (int x = 0; x < V; x++) {
    int z;  // leading zeros; y = 0 gives some number, dropped below
    if constexpr (sizeof(T) == 4)
      z = __builtin_clz((U)y[x]);
    else
      z = __builtin_clzll((U)y[x]);
    const U q = (am << ((HI - z) & HI)) + (U)(y[x] - 1);
    const U p = y[x] > (T)1 ? q : ~(U)0;
    cur[x] = p < cur[x] ? p : cur[x];
    top = y[x] > top ? y[x] : top;
    tmax = (T)cur[x] > tmax ? (T)cur[x] : tmax;
  }
}

// The same product, keeping the largest (natural values, 0 absent).
template <typename T, int V>
__device__ inline void rows_relax_largest(T (&big)[V], T a, const T (&z)[V], T& top) {
  using U = typename unsigned_of<T>::type;
#pragma unroll
  for (int x = 0; x < V; x++) {
    const T p = z[x] > (T)1 ? (T)(((U)(a - 1) << msb_u((U)z[x])) + (U)z[x]) : (T)0;
    big[x] = p > big[x] ? p : big[x];
    top = z[x] > top ? z[x] : top;
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

// 16 bytes of zeros that nothing here reads again
template <typename T>
__device__ inline void rows_st_stream(T* p) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(u32x4{0, 0, 0, 0}, (u32x4*)p);
}

constexpr int ROWS_LANES = 4;  // lanes of 16 bytes per row segment
template <typename T>
__host__ __device__ inline int64_t rows_slab() {
  return ROWS_LANES * (16 / (int64_t)sizeof(T));
}

// 64 KB: two workgroups of 1024 threads per CU; in place, 16 KB for eight of 256
template <bool LARGEST, bool INPLACE>
constexpr int ROWS_RING = INPLACE ? 256 : LARGEST ? 512 : 1024;
template <typename T, bool LARGEST, bool INPLACE>
struct CloseShared {
  static constexpr int ROWS = ROWS_RING<LARGEST, INPLACE>;
  T ring[ROWS][ROWS_LANES][16 / sizeof(T)];
  T ring2[LARGEST ? ROWS : 1][ROWS_LANES][16 / sizeof(T)];
  int start[ROWS_MAX_LEVELS + 1];
  long long top, top2;
  int guard;
};

// Word `lane` of a quad, to all four lanes.
template <int LANE>
__device__ inline uint32_t quad_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, LANE * 0x55, 0xf, 0xf, false);
}
template <typename T>
__device__ inline RowRec<T> rec_of_quad(uint2 q) {
  RowRec<T> r;
  r.row_c0 = quad_bcast<0>(q.x);
  r.c1_p0 = quad_bcast<0>(q.y);
  r.p1_cnt = quad_bcast<1>(q.x);
  if constexpr (sizeof(T) == 4) {
    r.v0 = (T)quad_bcast<2>(q.x);
    r.v1 = (T)quad_bcast<2>(q.y);
  } else {
    r.v0 = (T)((uint64_t)quad_bcast<2>(q.x) | (uint64_t)quad_bcast<2>(q.y) << 32);
    r.v1 = (T)((uint64_t)quad_bcast<3>(q.x) | (uint64_t)quad_bcast<3>(q.y) << 32);
  }
  return r;
}

// One slab of columns through every level.  W rows are 16-byte aligned (ld a
// multiple of 128).  A quad of lanes holds one row's segment.  Entries' rows
// are mostly of the last few levels (parents a few layers up), so the last
// ROWS_RING rows in level order stay in LDS and only older ones are read back
// from memory (N = 8192 int32: 130 us with every row read back, 128-byte
// segments or 64; 93-101 us so, of which about 40 are the writes' own time;
// 2048 rows with one workgroup per CU: 93 us).  The products are not the
// bound: leaving them out changed nothing.  Rows above the slab's first column hold no entry there and
// are never read again: their zeros go out as streaming stores.
//
// LARGEST: any numbering of the vertices.  The closure itself follows from the
// rows' entries as above, level by level, but a cell's first value depends on
// the numbering.  W2 takes the largest path value of every cell (no value a
// cell ever holds is above it), and the slab's largest goes to w.slab_top.
//
// INPLACE: W is the input, lower triangular.  No entry's cell is ever cleared,
// so a segment whose result is all zero was all zero and is not written (128
// components, 0.5 GB of matrices: 481 -> 345 us).
template <typename T, int UN, bool LARGEST, bool INPLACE>
__device__ inline void rows_close_slab(CloseShared<T, LARGEST, INPLACE>& L, RowsWork<T> w, T* W, T* W2, int64_t ld,
                                       int64_t slab, int width, rbg_status* st) {
  using U = typename unsigned_of<T>::type;
  constexpr int V = 16 / (int)sizeof(T);
  const int tid = threadIdx.x, G = blockDim.x / ROWS_LANES, ql = tid % ROWS_LANES;
  const int g = tid / ROWS_LANES;
  const int j0 = (int)(slab * rows_slab<T>());
  const int jl = j0 + ql * V;
  // row offsets in 16-byte units: below 2^32 for ROWS_MAX_N, one 24-bit multiply each
  const uint32_t ld16 = (uint32_t)(ld / V), jl16 = (uint32_t)(jl / V);
  auto off = [&](int row) { return (size_t)(__umul24((uint32_t)row, ld16) + jl16) * V; };
  constexpr int RING = ROWS_RING<LARGEST, INPLACE>;
  const int levels = w.ctl[1];
  if (tid <= levels) L.start[tid] = w.ctl[CTL_START + tid];
  if (tid == 0) {
    L.top = L.top2 = 0;
    L.guard = 0;
  }
  __syncthreads();
  int guard = 0;  // largest MSB(left) + MSB(right) of a product
  T tmax = -1, tmax2 = 0;
  uint2 qr[UN];  // this lane's words of the records
  auto fetch = [&](int p, int end, uint2& q) {
    if (p < end) q = ((const uint2*)(w.rec + p))[ql];
  };
  int base = 0, end = L.start[1];  // this pass: positions base + g + u G of level l
#pragma unroll
  for (int u = 0; u < UN; u++) fetch(base + g + u * G, end, qr[u]);
  for (int l = 0; l < levels;) {
    const int kept = end - RING;  // older positions have left the ring by the end of this level
    RowRec<T> r[UN];
    T y0[UN][V], y1[UN][V], z0[UN][V], z1[UN][V];  // z: of W2
    bool on[UN];
    int cnt[UN], row[UN], c0[UN], c1[UN];
    auto operand = [&](int c, int p, T(&y)[V], T(&z)[V]) {
      if (p >= kept) {
        rows_ld<T, V>(L.ring[p & (RING - 1)][ql], y);
        if (LARGEST) rows_ld<T, V>(L.ring2[p & (RING - 1)][ql], z);
      } else {
        rows_ld<T, V>(W + off(c), y);
        if (LARGEST) rows_ld<T, V>(W2 + off(c), z);
      }
    };
#pragma unroll
    for (int u = 0; u < UN; u++) {
      on[u] = base + g + u * G < end;
      r[u] = rec_of_quad<T>(qr[u]);
      cnt[u] = on[u] ? rec_cnt(r[u].p1_cnt) : 0;
      row[u] = (int)(r[u].row_c0 & 0xffff);
      c0[u] = (int)(r[u].row_c0 >> 16);
      c1[u] = (int)(r[u].c1_p0 & 0xffff);
#pragma unroll
      for (int x = 0; x < V; x++) y0[u][x] = y1[u][x] = z0[u][x] = z1[u][x] = 0;
      if (cnt[u] > 0 && (LARGEST || c0[u] >= j0)) operand(c0[u], (int)(r[u].c1_p0 >> 16), y0[u], z0[u]);
      if (cnt[u] > 1 && (LARGEST || c1[u] >= j0)) operand(c1[u], (int)(r[u].p1_cnt & 0xffff), y1[u], z1[u]);
    }
    // the pass after this one: the same level's, or the next level's first
    int bn = base + UN * G, ln = l, en = end;
    if (bn >= end) {
      ln = l + 1;
      bn = end;
      en = ln < levels ? L.start[ln + 1] : end;
    }
#pragma unroll
    for (int u = 0; u < UN; u++) fetch(bn + g + u * G, en, qr[u]);
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (!on[u]) continue;
      T* out = W + off(row[u]);
      if (!LARGEST && row[u] < j0) {
        if (!INPLACE) rows_st_stream<T>(out);
        continue;
      }
      U cur[V];
      T big[V];
#pragma unroll
      for (int x = 0; x < V; x++) {
        cur[x] = ~(U)0;
        big[x] = 0;
      }
      const int32_t* ec = w.ecol + (int64_t)row[u] * w.slots;
      const T* ev = w.eval + (int64_t)row[u] * w.slots;
      // the input's cells in this lane's columns, and the diagonal's identity
      T one = 0;
      const bool here = (unsigned)(row[u] - jl) < (unsigned)V || (cnt[u] > 0 && (unsigned)(c0[u] - jl) < (unsigned)V) ||
                        (cnt[u] > 1 && (unsigned)(c1[u] - jl) < (unsigned)V) || cnt[u] > 2;
      if (here) {
#pragma unroll
        for (int x = 0; x < V; x++) {
          if (row[u] == jl + x) one = (T)((r[u].p1_cnt >> 24) & 3) - 1;
          if (cnt[u] > 0 && c0[u] == jl + x) cur[x] = (U)r[u].v0 - 1;
          if (cnt[u] > 1 && c1[u] == jl + x) cur[x] = (U)r[u].v1 - 1;
        }
        for (int e = 2; e < cnt[u]; e++) {
          const int c = ec[e] - jl;
#pragma unroll
          for (int x = 0; x < V; x++)
            if (c == x) cur[x] = (U)ev[e] - 1;
        }
#pragma unroll
        for (int x = 0; x < V; x++) {
          if (LARGEST) big[x] = (T)(cur[x] + 1);
          tmax = !LARGEST && (T)cur[x] > tmax ? (T)cur[x] : tmax;
        }
        if (one == (T)1 && tmax < 0) tmax = 0;
      }
      auto relax = [&](T a, const T(&y)[V], const T(&z)[V]) {
        T top = 1;
        if (LARGEST) {
          T none = 0;
          rows_relax<T, V>(cur, a, y, none, none);
          rows_relax_largest<T, V>(big, a, z, top);
        } else {
          rows_relax<T, V>(cur, a, y, top, tmax);
        }
        const int m = top > 1 ? msb_u((U)top) + msb_u((U)a) : 0;
        guard = m > guard ? m : guard;
      };
      if (cnt[u] > 0) relax(r[u].v0, y0[u], z0[u]);
      if (cnt[u] > 1) relax(r[u].v1, y1[u], z1[u]);
      constexpr int EN = LARGEST ? 2 : 4;  // further entries' rows in flight
      for (int e = 2; e < cnt[u]; e += EN) {
        T y[EN][V], z[EN][V], a[EN];
#pragma unroll
        for (int q = 0; q < EN; q++) {
          const int c = e + q < cnt[u] ? ec[e + q] : -1;
          a[q] = e + q < cnt[u] ? ev[e + q] : (T)2;
#pragma unroll
          for (int x = 0; x < V; x++) y[q][x] = z[q][x] = 0;
          if (c >= (LARGEST ? 0 : j0)) {
            rows_ld<T, V>(W + off(c), y[q]);
            if (LARGEST) rows_ld<T, V>(W2 + off(c), z[q]);
          }
        }
#pragma unroll
        for (int q = 0; q < EN; q++) relax(a[q], y[q], z[q]);
      }
      T o[V];
#pragma unroll
      for (int x = 0; x < V; x++) {
        o[x] = (T)(cur[x] + 1);
        if (LARGEST) {
          tmax = (T)cur[x] > tmax ? (T)cur[x] : tmax;
          tmax2 = big[x] > tmax2 ? big[x] : tmax2;
        }
      }
      if (one != 0) {  // the lane of the diagonal; no product reaches that cell
#pragma unroll
        for (int x = 0; x < V; x++)
          if (row[u] == jl + x) o[x] = one;
      }
      T any = 0;
#pragma unroll
      for (int x = 0; x < V; x++) any |= o[x];
      if (!INPLACE || any != 0) rows_st<T, V>(out, o);
      if (LARGEST) rows_st<T, V>(W2 + off(row[u]), big);
      const int p = base + g + u * G;
      if (p >= kept) {
        rows_st<T, V>(L.ring[p & (RING - 1)][ql], o);
        if (LARGEST) rows_st<T, V>(L.ring2[p & (RING - 1)][ql], big);
      }
    }
    if (ln != l) __syncthreads();  // the level's rows are read by the next ones of this workgroup alone
    l = ln;
    base = bn;
    end = en;
  }
  const long long t = wave_max_i64((int64_t)tmax + 1);
  if ((tid & 63) == 0 && t > 0) atomicMax(&L.top, t);
  if (LARGEST) {
    const long long t2 = wave_max_i64((int64_t)tmax2);
    if ((tid & 63) == 0 && t2 > 0) atomicMax(&L.top2, t2);
  }
  if (guard > width - 2) atomicMax(&L.guard, guard);
  __syncthreads();
  if (tid == 0) {
    if (L.top > __hip_atomic_load(&st->diameter_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      record_diameter(st, L.top);
    if (LARGEST) w.slab_top[slab] = (T)L.top2;
    if (L.guard) atomicOr(&st->flags, (uint32_t)RBG_F_NEED_GENERAL);
  }
}

// ---- the trajectory maximum of any numbering --------------------------------
// The largest value any cell ever held is the largest first value of a cell:
// values only fall.  Every first value lies between the cell's final value (W)
// and its largest path value (W2), so with top = max W only the cells with
// W2 > top can hold more than top: none to some hundred (deep pedigrees of a
// thousand vertices and more have 0 to 402).  k_rows_select lists them;
// rows_first_value computes a cell's first value: its path whose largest
// intermediate vertex K is smallest, and among the paths through vertices up
// to K the smallest value -- two small shortest-path sweeps over the vertices
// between i and j.
constexpr int ROWS_MAX_BETWEEN = 1024;

template <typename T>
struct FirstShared {
  int bound[ROWS_MAX_BETWEEN + 1];  // smallest largest-intermediate of a path to j
  typename unsigned_of<T>::type value[ROWS_MAX_BETWEEN + 1];
  uint16_t vid[ROWS_MAX_BETWEEN];
  int m;
};

// By one workgroup; idx: n words of LDS (vertex -> place in vid).  0: the
// vertices between are more than ROWS_MAX_BETWEEN.
template <typename T>
__device__ inline T rows_first_value(FirstShared<T>& F, uint16_t* idx, RowsWork<T> w, const T* W, int64_t ld, int n,
                                     int i, int j) {
  using U = typename unsigned_of<T>::type;
  constexpr uint16_t NONE = 0xffff;
  const int tid = threadIdx.x, nt = blockDim.x;
  if (tid == 0) F.m = 0;
  __syncthreads();
  for (int v = tid; v < n; v += nt) {
    uint16_t at = NONE;
    if (v != i && v != j && W[(int64_t)i * ld + v] > (T)1 && W[(int64_t)v * ld + j] > (T)1) {
      const int p = atomicAdd(&F.m, 1);
      if (p < ROWS_MAX_BETWEEN) {
        F.vid[p] = (uint16_t)v;
        at = (uint16_t)p;
      }
    }
    idx[v] = at;
  }
  __syncthreads();
  const int m = F.m;
  if (m > ROWS_MAX_BETWEEN) {
    __syncthreads();  // the next cell clears F.m
    return 0;
  }
  for (int x = tid; x <= m; x += nt) {
    F.bound[x] = n;
    F.value[x] = ~(U)0;
  }
  __syncthreads();
  // place m is i itself
  bool changed;
  do {
    changed = false;
    for (int x = tid; x <= m; x += nt) {
      const int v = x == m ? i : (int)F.vid[x];
      const int cnt = rec_cnt(w.rec0[v].p1_cnt);
      int b = F.bound[x];
      for (int e = 0; e < cnt; e++) {
        const int c = w.ecol[(int64_t)v * w.slots + e];
        if (c == j) {
          b = -1;
        } else if (idx[c] != NONE) {
          const int through = F.bound[idx[c]];
          const int k = through > c ? through : c;
          b = k < b ? k : b;
        }
      }
      if (b < F.bound[x]) {
        F.bound[x] = b;
        changed = true;
      }
    }
  } while (__syncthreads_or(changed));
  const int K = F.bound[m];
  do {
    changed = false;
    for (int x = tid; x <= m; x += nt) {
      const int v = x == m ? i : (int)F.vid[x];
      const int cnt = rec_cnt(w.rec0[v].p1_cnt);
      U best = F.value[x];
      for (int e = 0; e < cnt; e++) {
        const int c = w.ecol[(int64_t)v * w.slots + e];
        const U a = (U)w.eval[(int64_t)v * w.slots + e];
        U p = ~(U)0;
        if (c == j) {
          p = a;
        } else if (idx[c] != NONE && c <= K) {
          const U y = F.value[idx[c]];
          if (y != ~(U)0) p = ((a - 1) << msb_u(y)) + y;
        }
        best = p < best ? p : best;
      }
      if (best < F.value[x]) {
        F.value[x] = best;
        changed = true;
      }
    }
  } while (__syncthreads_or(changed));
  const T first = (T)F.value[m];
  __syncthreads();  // the next cell's sweeps write what this one read
  return first;
}

}  // namespace rbg
