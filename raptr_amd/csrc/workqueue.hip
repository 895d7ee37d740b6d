// workqueue.hip -- cylinder-culled (channel, voxel) workqueue on gfx950.
//
// Replaces the serial host scan getWorkqueue (getWorkqueue.hpp:39-243).  One
// workgroup per list entry: per voxel column (ix, iy) the z interval that can
// pass the cull (column_interval), then the reference's float test on the
// voxels of the intervals, columns and z ascending.  A count pass gives each
// entry's candidates, a device-wide scan turns them into output offsets, and an
// emit pass finds the candidates again and writes each at its offset plus its
// rank, so the output keeps the reference's list-major, voxel-ascending order
// exactly.
#include "primitives.hpp"

namespace raptr {
namespace {

constexpr int kWqBlock = 256;
constexpr int kWqTile = 1024;  // voxels per tile of the workspace's layout

struct WqArgs {
  Geom G;
  FastDiv div_y;
  const int* list;
  int list_first;  // cursor list entry
  int vxl_first;   // cursor voxel (applies to list_first only)
};

// Candidates of one list entry.  EMIT: written from out_base on, below limit;
// else counted.  Testing all voxels of the grid took 223 us (count) and 271 us
// (emit) for 3,000 channels of 32^3 voxels (8.4M candidates); the intervals
// hold a ninth of them: 55 and 76 us.  Bound by the FP64 intervals and the tests' VALU.
template <bool EMIT>
__global__ __launch_bounds__(kWqBlock) void k_wq_entry(WqArgs A, int64_t e0, int* counts,
                                                       int64_t* counts64,
                                                       const int64_t* offsets, int64_t limit,
                                                       int* cnl_out, int* vxl_out,
                                                       int* last_pos) {
  constexpr int NW = kWqBlock / kWave, R = 4;  // R: rounds of a wave per segment
  __shared__ int s_scan[NW], s_cnt[2][NW];
  __shared__ int s_lo[kWqBlock], s_pre[kWqBlock];
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int64_t e = e0 + blockIdx.x;
  const int li = A.list_first + int(e);
  const int cnl = A.list[li];
  if (cnl < 0 || cnl >= A.G.nch) {  // an out-of-range channel has no candidates
    if (!EMIT && t == 0) {
      if (counts) counts[e] = 0;
      if (counts64) counts64[e] = 0;
    }
    return;
  }
  const int vstart = e == 0 ? A.vxl_first : 0;
  const int ny = A.G.g.n[1], nz = A.G.g.n[2], ncols = A.G.g.n[0] * ny;
  const LineInterval L(A.G, cnl);
  int64_t done = EMIT ? offsets[e] : 0;
  int mine = 0, buf = 0;
  for (int cb = 0; cb < ncols; cb += kWqBlock) {
    const int cc = cb + t;
    int lo = 0, cnt = 0;
    if (cc < ncols) {
      const int ix = int(fdiv(uint32_t(cc), A.div_y));
      cnt = L.column(A.G.g, ix, cc - ix * ny, lo);
    }
    int tot;
    const int pre = block_exclusive_scan<int, kWqBlock>(cnt, s_scan, &tot);
    if (tot == 0) continue;
    s_lo[t] = lo;
    s_pre[t] = pre;
    __syncthreads();
    for (int s0 = 0; s0 < tot; s0 += kWqBlock * R) {
      uint64_t mask[R];
      int v[R], n = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int k = s0 + (w * R + r) * kWave + lane;
        bool pass = false;
        v[r] = 0;
        if (k < tot) {
          int jl = 0;  // last column with s_pre <= k
#pragma unroll
          for (int j = kWqBlock / 2; j > 0; j >>= 1)
            if (s_pre[jl + j] <= k) jl += j;
          const int col = cb + jl, iz = s_lo[jl] + (k - s_pre[jl]);
          v[r] = col * nz + iz;
          float c[3];
          const int ix = int(fdiv(uint32_t(col), A.div_y));
          voxel_centre(A.G.g, ix, col - ix * ny, iz, c);
          pass = v[r] >= vstart && distance_point_line(L.p0, L.p1, c) < A.G.sumRadii;
        }
        mask[r] = __ballot(pass);
        n += __popcll(mask[r]);
      }
      if (!EMIT) {
        mine += n;
        continue;
      }
      if (lane == 0) s_cnt[buf][w] = n;
      __syncthreads();
      int64_t pos = done;
      for (int ww = 0; ww < NW; ++ww) {
        pos += ww < w ? s_cnt[buf][ww] : 0;
        done += s_cnt[buf][ww];
      }
      buf ^= 1;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int64_t p = pos + __popcll(mask[r] & lanemask_lt());
        if ((mask[r] >> lane & 1) && p < limit) {
          cnl_out[p] = cnl;
          vxl_out[p] = v[r];
          if (p == limit - 1) {
            last_pos[0] = li;
            last_pos[1] = v[r];
          }
        }
        pos += __popcll(mask[r]);
      }
      if (done >= limit) return;
    }
    __syncthreads();  // the columns' words are written again
  }
  if (!EMIT) {
    if (lane == 0) s_cnt[0][w] = mine;
    __syncthreads();
    if (t == 0) {
      int sum = 0;
      for (int ww = 0; ww < NW; ++ww) sum += s_cnt[0][ww];
      if (counts) counts[e] = sum;
      if (counts64) counts64[e] = sum;
    }
  }
}

int make_wq_args(const raptr_setup_t* setup, const raptr_grid_t* grid, const int* d_list,
                 int list_first, int vxl_first, WqArgs* A) {
  RAPTR_TRY(make_geom(setup, grid, &A->G));
  A->div_y = make_fastdiv(uint32_t(grid->n[1]));
  A->list = d_list;
  A->list_first = list_first;
  A->vxl_first = vxl_first;
  return RAPTR_OK;
}

// Launch a per-block kernel over nblk blocks in slices that keep the grid
// below 2^31 work-items.
template <class F>
int launch_sliced(int64_t nblk, F f) {
  const int64_t kMaxBlocks = (int64_t(1) << 31) / kWqBlock;
  for (int64_t b0 = 0; b0 < nblk; b0 += kMaxBlocks) {
    int64_t nb = nblk - b0 < kMaxBlocks ? nblk - b0 : kMaxBlocks;
    f(b0, unsigned(nb));
    RAPTR_LAUNCH_CHECK();
  }
  return RAPTR_OK;
}

}  // namespace
}  // namespace raptr

using namespace raptr;

extern "C" {

size_t raptr_workqueue_workspace_size(const raptr_grid_t* grid, int list_size) {
  if (!grid || list_size < 0) return 0;
  int64_t nvox = int64_t(grid->n[0]) * grid->n[1] * grid->n[2];
  int64_t tiles = (nvox + kWqTile - 1) / kWqTile;
  int64_t nblk = tiles * int64_t(list_size);
  Sizer z;
  z.take<int>(size_t(nblk));
  z.take<int64_t>(size_t(nblk));
  z.take<int64_t>(4);
  return z.bytes() + scan_workspace_bytes(nblk);
}

int raptr_workqueue(const raptr_setup_t* setup, const raptr_grid_t* grid, const int* d_list,
                    int list_size, int* list_id, int* vxl_id, int64_t n, int* d_cnl,
                    int* d_vxl, int64_t capacity, int64_t* n_found, void* d_ws,
                    size_t ws_bytes, raptr_stream_t stream) {
  if (!list_id || !vxl_id || !n_found) return fail(RAPTR_ERR_INVALID_ARG, "null cursor");
  *n_found = 0;
  if (list_size < 0 || (list_size > 0 && !d_list))
    return fail(RAPTR_ERR_INVALID_ARG, "bad list");
  WqArgs A;
  RAPTR_TRY(make_wq_args(setup, grid, d_list, *list_id, *vxl_id, &A));
  if (*list_id < 0 || *list_id > list_size || *vxl_id < 0 || *vxl_id >= A.G.nvox)
    return fail(RAPTR_ERR_INVALID_ARG,
                "invalid cursor (list_id %d, vxl_id %d)", *list_id, *vxl_id);
  if (n == 0 || *list_id == list_size) return RAPTR_OK;
  hipStream_t st = S(stream);
  const int64_t entries = list_size - *list_id;
  const int64_t nblk = entries * ((A.G.nvox + kWqTile - 1) / kWqTile);
  Carver cv(d_ws, ws_bytes);
  int* counts = cv.take<int>(size_t(nblk));
  int64_t* offs = cv.take<int64_t>(size_t(nblk));
  int64_t* small = cv.take<int64_t>(4);
  size_t scan_bytes = scan_workspace_bytes(nblk);
  void* scan_ws = cv.take<char>(scan_bytes);
  if (!cv.ok) return fail(RAPTR_ERR_WORKSPACE, "workqueue workspace too small (%zu < %zu)",
                          ws_bytes, raptr_workqueue_workspace_size(grid, list_size));
  RAPTR_TRY(launch_sliced(entries, [&](int64_t b0, unsigned nb) {
    hipLaunchKernelGGL(k_wq_entry<false>, dim3(nb), dim3(kWqBlock), 0, st, A, b0, counts,
                       (int64_t*)nullptr, (const int64_t*)nullptr, int64_t(0), (int*)nullptr, (int*)nullptr,
                       (int*)nullptr);
  }));
  RAPTR_TRY(scan_exclusive_i32_i64(counts, offs, entries, &small[0], scan_ws, scan_bytes, st));
  int64_t total = 0;
  RAPTR_HIP_TRY(hipMemcpyAsync(&total, &small[0], sizeof(int64_t), hipMemcpyDeviceToHost, st));
  RAPTR_HIP_TRY(hipStreamSynchronize(st));
  bool bounded = n >= 0;
  int64_t found = (bounded && n < total) ? n : total;
  if (found > capacity)
    return fail(RAPTR_ERR_INVALID_ARG, "output capacity %lld < %lld entries",
                (long long)capacity, (long long)found);
  if (found > 0 && (!d_cnl || !d_vxl)) return fail(RAPTR_ERR_INVALID_ARG, "null output");
  int* last = reinterpret_cast<int*>(&small[1]);
  if (found > 0)
    RAPTR_TRY(launch_sliced(entries, [&](int64_t b0, unsigned nb) {
      hipLaunchKernelGGL(k_wq_entry<true>, dim3(nb), dim3(kWqBlock), 0, st, A, b0, (int*)nullptr,
                         (int64_t*)nullptr, (const int64_t*)offs, found, d_cnl, d_vxl, last);
    }));
  int cur[2] = {list_size, 0};
  if (bounded && found == n && found > 0) {
    // Cursor after the n-th entry, as getWorkqueueEntry advances it
    // (getWorkqueue.hpp:101-112).
    int lp[2];
    RAPTR_HIP_TRY(hipMemcpyAsync(lp, last, 2 * sizeof(int), hipMemcpyDeviceToHost, st));
    RAPTR_HIP_TRY(hipStreamSynchronize(st));
    if (lp[1] < A.G.nvox - 1) {
      cur[0] = lp[0];
      cur[1] = lp[1] + 1;
    } else {
      cur[0] = lp[0] + 1;
      cur[1] = 0;
    }
  } else {
    RAPTR_HIP_TRY(hipStreamSynchronize(st));
  }
  *list_id = cur[0];
  *vxl_id = cur[1];
  *n_found = found;
  return RAPTR_OK;
}

int raptr_workqueue_counts(const raptr_setup_t* setup, const raptr_grid_t* grid,
                           const int* d_list, int list_size, int64_t* d_counts,
                           raptr_stream_t stream) {
  if (list_size <= 0) return RAPTR_OK;
  if (!d_list || !d_counts) return fail(RAPTR_ERR_INVALID_ARG, "null argument");
  WqArgs A;
  RAPTR_TRY(make_wq_args(setup, grid, d_list, 0, 0, &A));
  return launch_sliced(list_size, [&](int64_t b0, unsigned nb) {
    hipLaunchKernelGGL(k_wq_entry<false>, dim3(nb), dim3(kWqBlock), 0, S(stream), A, b0,
                       (int*)nullptr, d_counts, (const int64_t*)nullptr, int64_t(0), (int*)nullptr, (int*)nullptr,
                       (int*)nullptr);
  });
}

}  // extern "C"
