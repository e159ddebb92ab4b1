// Closure of one matrix from its rows' direct entries: the
// launches of fw_rows.hpp and the C ABI.
#include "fw_rows.hpp"

namespace rbg {

template <typename T>
static __global__ __launch_bounds__(NT) void k_rows_scan(const T* A, int64_t n, int64_t lda, bool vec, RowsWork<T> w) {
  const int64_t i = blockIdx.x * (int64_t)(NT / 64) + threadIdx.x / 64;
  if (i < n) rows_scan_row<T>(A + i * lda, n, i, vec, w);
}

// Up to this many rows the workgroup of the levels also places the records: a
// launch less (n = 512: 54.2 -> 52.7 us a closure, 1100: 93.4 -> 91.5; 4096 int64
// 127.6 -> 131.3, where one CU moves too many records).
constexpr int64_t ROWS_PLACE_HERE = 2048;

// Entries times levels above which a matrix of another numbering with a row of
// more than two entries is not tried:
// the more paths and the longer, the more cells have a largest path value above
// the largest final value (see rows_first_value), and the passes that find out
// that they are too many take up to half of the blocked closure's time again.
// Rows of k entries, unordered int32, us by the rows / blocked (f: tried and not
// closed, the blocked closure's included): n = 200, 6 levels, k = 10 (49 n) 185 /
// 307; 14 levels, k = 6 (76 n) 213 / 306, k = 8 (101 n) 362 / 308; n = 300, 14
// levels, k = 8 (103 n) 413 / 418, k = 10 (128 n) 616 / 415; n = 1000, 14 levels,
// k = 5 (65 n) 345 / 1005, k = 6 (78 n) 1195 f / 1002; n = 6000, 6 levels, k = 10
// (50 n) 849 / 24220, 14 levels, k = 6 (78 n) 24930 f / 24250; n = 8000, 6
// levels, k = 200 (1000 n) 84070 f / 52110.
// (int64, whose blocked closure takes half as long again: n = 200, 14 levels, k =
// 8 (101 n) 367 / 452, k = 10 (128 n) 622 / 453.)
template <typename T>
static int64_t rows_any_work(int64_t n) {
  return (n < 1000 ? (sizeof(T) == 8 ? 110 : 100) : 70) * n;
}

// Also writes the whole status block.  aux[6]: 1 the matrix is lower
// triangular, 2 upper, 3 has entries on both sides (0: not looked at).  ctl[0]
// and aux[5]: the same where it is closed from its rows, else 0.
template <typename T, int H>
static __global__ __launch_bounds__(ROWS_LEVEL_NT) void k_rows_levels(int64_t n, RowsWork<T> w, bool allowed,
                                                                     int64_t any_work, rbg_status* st) {
  extern __shared__ __align__(16) uint8_t lev[];
  __shared__ LevelShared L;
  __shared__ int entries;
  int sides = 0;
  const int stop = allowed ? rows_levels<T, H>(w, n, L, lev, sides) : 1;
  const int side = sides & 2 ? (sides & 1 ? 3 : 2) : 1;
  int code = stop || (side > 1 && n > ROWS_ANY_MAX_N) ? 0 : side;
  if (code > 1 && L.third) {  // uniform, as is what follows
    if (threadIdx.x == 0) entries = 0;
    __syncthreads();
    int mine = 0;
    for (int64_t i = threadIdx.x; i < n; i += ROWS_LEVEL_NT) mine += rec_cnt(w.rec0[i].p1_cnt);
    if (mine) atomicAdd(&entries, mine);
    __syncthreads();
    if ((int64_t)entries * w.ctl[1] > any_work) code = 0;
  }
  if (code && n <= ROWS_PLACE_HERE) {
    __syncthreads();  // every row's position
    for (int64_t i = threadIdx.x; i < n; i += ROWS_LEVEL_NT) rows_place<T>(w, i);
  }
  if (threadIdx.x == 0) {
    status_clear(st);
    if (stop & STOP_BAD) st->flags = RBG_F_PRECOND_FAIL;
    w.ctl[0] = code;
    st->aux[5] = code;
    st->aux[6] = allowed ? side : 0;
    w.cells[0] = 0;
  }
}

template <typename T>
static __global__ __launch_bounds__(NT) void k_rows_place(int64_t n, RowsWork<T> w) {
  const int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x;
  if (w.ctl[0] && i < n) rows_place<T>(w, i);
}

// Workgroup -> slab, `count` of them.  Slabs cost less from left to right
// (their columns' rows start lower); two workgroups share a CU, the first 512
// all start at once and the second 256 of them join the first 256 CU by CU, so
// those take the cheapest slabs.  The XCDs take turns at workgroups: eight
// neighbouring slabs (512 bytes of a row) go to one XCD's L2.
__device__ inline int rows_slab_of(int b, int count) {
  auto grouped = [&](int q) {
    return (q | 63) < count && (q | 63) < 256 ? (q & ~63) + (q & 7) * 8 + ((q & 63) >> 3) : q;
  };
  if (b < 256) return grouped(b);
  if (b < 512) return count - 1 - (b - 256);
  return b - 256;
}

template <typename T, bool LARGEST>
static __global__ __launch_bounds__(ROWS_CLOSE_NT, LARGEST ? 4 : 8) void k_rows_close(RowsWork<T> w, T* W, T* W2,
                                                                                     int64_t ld, int width,
                                                                                     rbg_status* st) {
  __shared__ CloseShared<T, LARGEST, false> L;
  if (LARGEST ? w.ctl[0] < 2 : w.ctl[0] != 1) return;
  rows_close_slab<T, 1, LARGEST, false>(L, w, W, W2, ld, rows_slab_of(blockIdx.x, gridDim.x), width, st);
}

// The slab's cells whose largest path value is above the largest final value;
// a wave's at a time, and no more once they are too many.
template <typename T>
static __global__ __launch_bounds__(NT) void k_rows_select(int64_t n, RowsWork<T> w, const T* W2, int64_t ld,
                                                          const rbg_status* st) {
  constexpr int V = 16 / (int)sizeof(T);
  const T top = (T)st->diameter_max;
  if (w.ctl[0] < 2 || w.slab_top[blockIdx.x] <= top) return;
  const int lane = threadIdx.x & 63;
  const int64_t j = blockIdx.x * rows_slab<T>() + (threadIdx.x % ROWS_LANES) * V;
  for (int64_t i = threadIdx.x / ROWS_LANES; i < n; i += NT / ROWS_LANES) {
    T z[V];
    rows_ld<T, V>(W2 + i * ld + j, z);
    uint64_t above[V];
    int all = 0;
#pragma unroll
    for (int x = 0; x < V; x++) {
      above[x] = __ballot(z[x] > top);
      all += __popcll(above[x]);
    }
    if (all == 0) continue;
    // the lanes at row i < n are the wave's first ones
    uint32_t at = 0;
    if (lane == 0) at = atomicAdd(&w.cells[0], (uint32_t)all);
    at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
    if (at >= ROWS_MAX_CELLS) return;
#pragma unroll
    for (int x = 0; x < V; x++) {
      const uint32_t mine = at + (uint32_t)__popcll(above[x] & (((uint64_t)1 << lane) - 1));
      if (z[x] > top && mine < ROWS_MAX_CELLS) w.cells[1 + mine] = (uint32_t)i | (uint32_t)(j + x) << 16;
      at += (uint32_t)__popcll(above[x]);
    }
  }
}

// First values of the listed cells.  aux[5] = 0: too many cells, or too many
// vertices between one's ends (the trajectory maximum is then not known).
template <typename T>
static __global__ __launch_bounds__(NT) void k_rows_first(int64_t n, RowsWork<T> w, const T* W, int64_t ld,
                                                         rbg_status* st) {
  extern __shared__ uint16_t idx[];
  __shared__ FirstShared<T> F;
  if (w.ctl[0] < 2) return;
  const uint32_t count = w.cells[0];
  if (count > ROWS_MAX_CELLS) {
    if (blockIdx.x == 0 && threadIdx.x == 0) st->aux[5] = 0;
    return;
  }
  for (uint32_t q = blockIdx.x; q < count; q += gridDim.x) {
    const uint32_t c = w.cells[1 + q];
    const T first = rows_first_value<T>(F, idx, w, W, ld, (int)n, (int)(c & 0xffff), (int)(c >> 16));
    if (threadIdx.x == 0) {
      if (first == 0)
        st->aux[5] = 0;
      else
        record_diameter(st, (int64_t)first);
    }
  }
}

template <typename T>
static int rows_args(const void* A, int64_t n, const T* W, int64_t npad, void* wsp, int64_t ws_bytes,
                     const rbg_status* st, RowsWork<T>* w) {
  if (!A || !W || !wsp || !st || n <= 0 || n > ROWS_MAX_N || npad < n || npad % TILE || ((uintptr_t)W & 15) ||
      ((uintptr_t)wsp & 255))
    return RBG_E_ARG;
  // the close pass counts 16-byte units in 32 bits
  if (npad / (16 / (int64_t)sizeof(T)) > 0xffffffffll / n) return RBG_E_ARG;
  return ws_bytes < rows_layout<T>(n, (char*)wsp, w) ? RBG_E_WORKSPACE : 0;
}

template <typename T>
static unsigned rows_slabs(int64_t n) {
  return (unsigned)((n + rows_slab<T>() - 1) / rows_slab<T>());
}

template <typename T>
static int fw_rows(const T* A, int64_t n, int64_t lda, T* W, int64_t npad, void* wsp, int64_t ws_bytes,
                   rbg_status* st, hipStream_t s) {
  RowsWork<T> w;
  const int rc = rows_args<T>(A, n, W, npad, wsp, ws_bytes, st, &w);
  if (rc) return rc;
  if (lda < n) return RBG_E_ARG;
  const bool vec = lda % (16 / (int64_t)sizeof(T)) == 0 && ((uintptr_t)A & 15) == 0;
  hipLaunchKernelGGL((k_rows_scan<T>), dim3((unsigned)((n + NT / 64 - 1) / (NT / 64))), dim3(NT), 0, s, A, n, lda, vec,
                     w);
  RBG_CHECK_LAUNCH();
  // a forced wait limit asks for the persistent closure (rbg_fw_flow_wait_limit)
  const bool allowed = g_flow_limit_override.load() == 0;
  const size_t lds = (size_t)(n + 4);
  if (n <= 8 * ROWS_LEVEL_NT)
    hipLaunchKernelGGL((k_rows_levels<T, 2>), dim3(1), dim3(ROWS_LEVEL_NT), lds, s, n, w, allowed,
                       rows_any_work<T>(n), st);
  else if (n <= 16 * ROWS_LEVEL_NT)
    hipLaunchKernelGGL((k_rows_levels<T, 4>), dim3(1), dim3(ROWS_LEVEL_NT), lds, s, n, w, allowed,
                       rows_any_work<T>(n), st);
  else
    hipLaunchKernelGGL((k_rows_levels<T, 8>), dim3(1), dim3(ROWS_LEVEL_NT), lds, s, n, w, allowed,
                       rows_any_work<T>(n), st);
  RBG_CHECK_LAUNCH();
  if (n > ROWS_PLACE_HERE) {
    hipLaunchKernelGGL((k_rows_place<T>), dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, s, n, w);
    RBG_CHECK_LAUNCH();
  }
  const int p = prof_start(s);
  hipLaunchKernelGGL((k_rows_close<T, false>), dim3(rows_slabs<T>(n)), dim3(ROWS_CLOSE_NT), 0, s, w, W, (T*)nullptr,
                     npad, (int)sizeof(T) * 8, st);
  RBG_CHECK_LAUNCH();
  prof_stop(7, p, s, (double)n * n * sizeof(T));
  return 0;
}

template <typename T>
static int fw_rows_any(int64_t n, T* W, T* W2, int64_t npad, void* wsp, int64_t ws_bytes, rbg_status* st,
                       hipStream_t s) {
  RowsWork<T> w;
  const int rc = rows_args<T>(W2, n, W, npad, wsp, ws_bytes, st, &w);
  if (rc) return rc;
  if (n > ROWS_ANY_MAX_N || ((uintptr_t)W2 & 15)) return RBG_E_ARG;
  const int p = prof_start(s);
  hipLaunchKernelGGL((k_rows_close<T, true>), dim3(rows_slabs<T>(n)), dim3(ROWS_CLOSE_NT), 0, s, w, W, W2, npad,
                     (int)sizeof(T) * 8, st);
  RBG_CHECK_LAUNCH();
  prof_stop(7, p, s, (double)n * n * sizeof(T));
  hipLaunchKernelGGL((k_rows_select<T>), dim3(rows_slabs<T>(n)), dim3(NT), 0, s, n, w, (const T*)W2, npad, st);
  RBG_CHECK_LAUNCH();
  hipLaunchKernelGGL((k_rows_first<T>), dim3(512), dim3(NT), (size_t)(2 * n), s, n, w, (const T*)W, npad, st);
  RBG_CHECK_LAUNCH();
  return 0;
}

}  // namespace rbg

using namespace rbg;

extern "C" {

int64_t rbg_fw_rows_max_n(void) { return ROWS_MAX_N; }

int64_t rbg_fw_rows_workspace_bytes(int64_t n, int32_t elem_bytes) {
  if (n <= 0 || n > ROWS_MAX_N) return 0;
  return elem_bytes == 8 ? rows_layout<int64_t>(n, nullptr, nullptr) : rows_layout<int32_t>(n, nullptr, nullptr);
}
int rbg_fw_rows_i32(const int32_t* A, int64_t n, int64_t lda, int32_t* W, int64_t npad, void* workspace,
                    int64_t workspace_bytes, rbg_status* st, rbg_stream_t stream) {
  return fw_rows<int32_t>(A, n, lda, W, npad, workspace, workspace_bytes, st, (hipStream_t)stream);
}
int rbg_fw_rows_i64(const int64_t* A, int64_t n, int64_t lda, int64_t* W, int64_t npad, void* workspace,
                    int64_t workspace_bytes, rbg_status* st, rbg_stream_t stream) {
  return fw_rows<int64_t>(A, n, lda, W, npad, workspace, workspace_bytes, st, (hipStream_t)stream);
}

int rbg_fw_rows_any_i32(int64_t n, int32_t* W, int32_t* W2, int64_t npad, void* workspace, int64_t workspace_bytes,
                        rbg_status* st, rbg_stream_t stream) {
  return fw_rows_any<int32_t>(n, W, W2, npad, workspace, workspace_bytes, st, (hipStream_t)stream);
}
int rbg_fw_rows_any_i64(int64_t n, int64_t* W, int64_t* W2, int64_t npad, void* workspace, int64_t workspace_bytes,
                        rbg_status* st, rbg_stream_t stream) {
  return fw_rows_any<int64_t>(n, W, W2, npad, workspace, workspace_bytes, st, (hipStream_t)stream);
}

}  // extern "C"
