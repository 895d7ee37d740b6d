// workqueue.hip -- cylinder-culled (channel, voxel) workqueue on gfx950.
//
// Replaces the serial host scan getWorkqueue (getWorkqueue.hpp:39-243).  One
// workgroup per list entry, or several that share its voxel columns: per column
// (ix, iy) the z interval that can pass the cull (LineInterval), then the
// reference's float test on the voxels of the intervals, columns and z
// ascending; or that test on every voxel, where there are few.  A count pass gives each workgroup's candidates, a device-wide scan
// turns them into output offsets, and an emit pass finds the candidates again
// and writes each at its offset plus its rank, so the output keeps the
// reference's list-major, voxel-ascending order exactly.
#include "primitives.hpp"

namespace raptr {
namespace {

constexpr int kWqBlock = 256;
constexpr int kWqTile = 1024;  // voxels per tile of the workspace's layout

struct WqArgs {
  Geom G;
  FastDiv div_y, div_yz, div_z;
  const int* list;
  int parts;       // workgroups per entry, each with a run of units
  bool every;      // every voxel is tested; units are tiles of kWqTile, else
                   // blocks of kWqBlock columns
  int list_first;  // cursor list entry
  int vxl_first;   // cursor voxel (applies to list_first only)
};

// Candidates of one list entry, or of one of its A.parts parts.  EMIT: written
// from their offset on, below limit; else counted.  Testing all voxels of the
// grid took 223 us (count) and 271 us (emit) for 3,000 channels of 32^3 voxels
// (8.4M candidates); the intervals hold a ninth of them: 55 and 76 us.  Bound by
// the FP64 intervals and the tests' VALU.
template <bool EMIT, bool EVERY>
__global__ __launch_bounds__(kWqBlock) void k_wq_entry(WqArgs A, int64_t e0, int* counts,
                                                       int64_t* counts64,
                                                       const int64_t* offsets, int64_t limit,
                                                       int* cnl_out, int* vxl_out,
                                                       int* last_pos) {
  constexpr int NW = kWqBlock / kWave, R = 4;  // R: rounds of a wave per segment
  __shared__ int s_scan[NW], s_cnt[2][NW];
  __shared__ int s_lo[kWqBlock], s_pre[kWqBlock];
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int64_t e = (e0 + blockIdx.x) / A.parts;
  const int part = int((e0 + blockIdx.x) % A.parts);
  const int li = A.list_first + int(e);
  const int cnl = A.list[li];
  if (cnl < 0 || cnl >= A.G.nch) {  // an out-of-range channel has no candidates
    if (!EMIT && t == 0) {
      if (counts) counts[e * A.parts + part] = 0;
      if (counts64 && A.parts == 1) counts64[e] = 0;
    }
    return;
  }
  const int vstart = e == 0 ? A.vxl_first : 0;
  const int ny = A.G.g.n[1], nz = A.G.g.n[2], ncols = A.G.g.n[0] * ny;
  const LineInterval L(A.G, cnl);
  int64_t done = EMIT ? offsets[e * A.parts + part] : 0;
  if (EMIT && done >= limit) return;
  int mine = 0, buf = 0;
  // this workgroup's columns (EVERY: voxels)
  constexpr int UNIT = EVERY ? kWqTile : kWqBlock;
  const int all = EVERY ? A.G.nvox : ncols;
  const int64_t units = (int64_t(all) + UNIT - 1) / UNIT;
  const int c0 = int(units * part / A.parts) * UNIT;
  const int c1 = part + 1 < A.parts ? int(units * (part + 1) / A.parts) * UNIT : all;
  for (int cb = c0; cb < c1; cb += EVERY ? c1 - c0 : UNIT) {
    int tot = c1 - c0;
    if (!EVERY) {
      const int cc = cb + t;
      int lo = 0, cnt = 0;
      if (cc < c1) {
        const int ix = int(fdiv(uint32_t(cc), A.div_y));
        cnt = L.column(A.G.g, ix, cc - ix * ny, lo);
      }
      const int pre = block_exclusive_scan<int, kWqBlock>(cnt, s_scan, &tot);
      if (tot == 0) continue;
      s_lo[t] = lo;
      s_pre[t] = pre;
      __syncthreads();
    }
    for (int s0 = 0; s0 < tot; s0 += kWqBlock * R) {
      uint64_t mask[R];
      int v[R], n = 0;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int k = s0 + (w * R + r) * kWave + lane;
        bool pass = false;
        v[r] = 0;
        if (k < tot) {
          int ix, iy, iz;
          if (EVERY) {
            v[r] = cb + k;
            ix = int(fdiv(uint32_t(v[r]), A.div_yz));
            const int rem = v[r] - ix * int(A.div_yz.d);
            iy = int(fdiv(uint32_t(rem), A.div_z));
            iz = rem - iy * nz;
          } else {
            int jl = 0;  // last column with s_pre <= k
#pragma unroll
            for (int j = kWqBlock / 2; j > 0; j >>= 1)
              if (s_pre[jl + j] <= k) jl += j;
            const int col = cb + jl;
            ix = int(fdiv(uint32_t(col), A.div_y));
            iy = col - ix * ny;
            iz = s_lo[jl] + (k - s_pre[jl]);
            v[r] = col * nz + iz;
          }
          float c[3];
          voxel_centre(A.G.g, ix, iy, iz, c);
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
      if (counts) counts[e * A.parts + part] = sum;
      if (counts64 && A.parts == 1) counts64[e] = sum;
      if (counts64 && A.parts > 1)
        atomicAdd(reinterpret_cast<unsigned long long*>(&counts64[e]), (unsigned long long)sum);
    }
  }
}

__global__ void k_wq_clear(int64_t* counts64, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += int(gridDim.x) * blockDim.x)
    counts64[i] = 0;
}

// Workgroups that a call should have at least: one per entry left most of the
// device idle on short lists (4 channels of a 96^3 grid 395 us, of 256^3 4,432;
// 64 channels of 96^3 406).  Now 69, 115 and 126; with 1,024, 4,096 and 8,192
// workgroups 64 channels of 96^3 take 135, 105 and 106, 1,024 of them 536, 594
// and 640 (551 with 2,048).
constexpr int64_t kWqGroups = 2048;
// Every voxel is tested on grids of fewer cells along z (3,000 channels of 240 x
// 240 x 2 cells 1,298 us, by intervals 2,176; of 240 x 240 x 4 3,083 and 2,459)
// and on calls of at most that many tiles, which are over before the intervals
// of the first columns stand (one channel of 96^3 51 and 70 us, of 32^3 45 and
// 56, 4 of 96^3 69 and 74); a fourth of them with more than 16 entries (64
// channels of 32^3 59 and 57, 617 of 18^3, with their values, 86 and 84).
constexpr int kWqFlat = 4;
constexpr int64_t kWqFewTiles = 4096;
int make_wq_args(const raptr_setup_t* setup, const raptr_grid_t* grid, const int* d_list,
                 int list_first, int vxl_first, int64_t entries, WqArgs* A) {
  RAPTR_TRY(make_geom(setup, grid, &A->G));
  if (entries < 1) entries = 1;
  const int64_t cols = int64_t(grid->n[0]) * grid->n[1];
  const int64_t tiles = (int64_t(A->G.nvox) + kWqTile - 1) / kWqTile;
  A->every = grid->n[2] < kWqFlat ||
             entries * tiles <= (entries <= 16 ? kWqFewTiles : kWqFewTiles / 4);
  // (an entry has as many counters as tiles)
  const int64_t blocks = (cols + kWqBlock - 1) / kWqBlock;
  int64_t most = A->every || blocks > tiles ? tiles : blocks;
  // a list of one workgroup a CU and more: parts of at least 4 blocks (1,718
  // channels of 24^3 in two parts each took 168 us with their values, 157 in one)
  if (!A->every && entries >= 256) most = blocks >= 8 ? blocks / 4 : 1;
  const int64_t want = ((A->every ? kWqFewTiles : kWqGroups) + entries - 1) / entries;
  A->parts = int(want < most ? want : most);
  A->div_yz = make_fastdiv(uint32_t(grid->n[1] * grid->n[2]));
  A->div_z = make_fastdiv(uint32_t(grid->n[2]));
  A->div_y = make_fastdiv(uint32_t(grid->n[1]));
  A->list = d_list;
  A->list_first = list_first;
  A->vxl_first = vxl_first;
  return RAPTR_OK;
}

// every or by columns
template <bool EMIT, class... T>
void launch_entry(const WqArgs& A, unsigned nb, hipStream_t st, T... args) {
  if (A.every)
    hipLaunchKernelGGL((k_wq_entry<EMIT, true>), dim3(nb), dim3(kWqBlock), 0, st, A, args...);
  else
    hipLaunchKernelGGL((k_wq_entry<EMIT, false>), dim3(nb), dim3(kWqBlock), 0, st, A, args...);
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
  RAPTR_TRY(make_wq_args(setup, grid, d_list, *list_id, *vxl_id, int64_t(list_size) - *list_id, &A));
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
  RAPTR_TRY(launch_sliced(entries * A.parts, [&](int64_t b0, unsigned nb) {
    launch_entry<false>(A, nb, st, b0, counts, (int64_t*)nullptr, (const int64_t*)nullptr, int64_t(0),
                        (int*)nullptr, (int*)nullptr, (int*)nullptr);
  }));
  RAPTR_TRY(scan_exclusive_i32_i64(counts, offs, entries * A.parts, &small[0], scan_ws, scan_bytes, st));
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
    RAPTR_TRY(launch_sliced(entries * A.parts, [&](int64_t b0, unsigned nb) {
      launch_entry<true>(A, nb, st, b0, (int*)nullptr, (int64_t*)nullptr, (const int64_t*)offs, found,
                         d_cnl, d_vxl, last);
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
  RAPTR_TRY(make_wq_args(setup, grid, d_list, 0, 0, list_size, &A));
  if (A.parts > 1) {
    hipLaunchKernelGGL(k_wq_clear, dim3(grid_for(list_size, 256, 1024)), dim3(256), 0, S(stream),
                       d_counts, list_size);
    RAPTR_LAUNCH_CHECK();
  }
  return launch_sliced(int64_t(list_size) * A.parts, [&](int64_t b0, unsigned nb) {
    launch_entry<false>(A, nb, S(stream), b0, (int*)nullptr, d_counts, (const int64_t*)nullptr,
                        int64_t(0), (int*)nullptr, (int*)nullptr, (int*)nullptr);
  });
}

}  // extern "C"
