// Closure of one triangular matrix from its rows' direct entries: the
// launches of fw_rows.hpp and the C ABI.
#include "fw_rows.hpp"

namespace rbg {

template <typename T>
static __global__ __launch_bounds__(NT) void k_rows_scan(const T* A, int64_t n, int64_t lda, bool vec, RowsWork<T> w) {
  const int64_t i = blockIdx.x * (int64_t)(NT / 64) + threadIdx.x / 64;
  if (i < n) rows_scan_row<T>(A + i * lda, n, i, vec, w);
}

// Also writes the whole status block: aux[5] = 1 when the next launches close
// the matrix.
template <typename T>
static __global__ __launch_bounds__(ROWS_LEVEL_NT) void k_rows_levels(int64_t n, RowsWork<T> w, bool allowed,
                                                                     rbg_status* st) {
  extern __shared__ __align__(16) uint8_t lev[];
  __shared__ LevelShared L;
  const int stop = allowed ? rows_levels<T>(w, n, L, lev) : 1;
  if (threadIdx.x == 0) {
    status_clear(st);
    if (stop & STOP_BAD) st->flags = RBG_F_PRECOND_FAIL;
    w.ctl[0] = st->aux[5] = stop == 0;
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

template <typename T>
static __global__ __launch_bounds__(ROWS_CLOSE_NT, 8) void k_rows_close(RowsWork<T> w, T* W, int64_t ld, int width,
                                                                    rbg_status* st) {
  __shared__ CloseShared<T> L;
  if (w.ctl[0] != 1) return;
  rows_close_slab<T, 1>(L, w, W, ld, rows_slab_of(blockIdx.x, gridDim.x), width, st);
}

template <typename T>
static int fw_rows(const T* A, int64_t n, int64_t lda, T* W, int64_t npad, void* wsp, int64_t ws_bytes,
                   rbg_status* st, hipStream_t s) {
  if (!A || !W || !wsp || !st || n <= 0 || n > ROWS_MAX_N || lda < n || npad < n || npad % TILE ||
      ((uintptr_t)W & 15) || ((uintptr_t)wsp & 255))
    return RBG_E_ARG;
  RowsWork<T> w;
  if (ws_bytes < rows_layout<T>(n, (char*)wsp, &w)) return RBG_E_WORKSPACE;
  const bool vec = lda % (16 / (int64_t)sizeof(T)) == 0 && ((uintptr_t)A & 15) == 0;
  hipLaunchKernelGGL((k_rows_scan<T>), dim3((unsigned)((n + NT / 64 - 1) / (NT / 64))), dim3(NT), 0, s, A, n, lda, vec,
                     w);
  RBG_CHECK_LAUNCH();
  // a forced wait limit asks for the persistent closure (rbg_fw_flow_wait_limit)
  const bool allowed = g_flow_limit_override.load() == 0;
  hipLaunchKernelGGL((k_rows_levels<T>), dim3(1), dim3(ROWS_LEVEL_NT), (size_t)(n + 4), s, n, w, allowed, st);
  RBG_CHECK_LAUNCH();
  hipLaunchKernelGGL((k_rows_place<T>), dim3((unsigned)((n + NT - 1) / NT)), dim3(NT), 0, s, n, w);
  RBG_CHECK_LAUNCH();
  const int p = prof_start(s);
  hipLaunchKernelGGL((k_rows_close<T>), dim3((unsigned)((n + rows_slab<T>() - 1) / rows_slab<T>())),
                     dim3(ROWS_CLOSE_NT), 0, s, w, W, npad, (int)sizeof(T) * 8, st);
  RBG_CHECK_LAUNCH();
  prof_stop(7, p, s, (double)n * n * sizeof(T));
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

}  // extern "C"
