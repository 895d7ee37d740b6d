// sysmat.hip -- Monte Carlo ray-sampled system matrix on gfx950.
//
// Two entry points follow the reference:
//  * raptr_sm_from_wq: the two-stage path (getSystemMatrixFromWorkqueue.cu:
//    116-281): queues in channel order by runs of a channel, its rays and
//    plane tables made once (k_sm_from_wq_runs); other entries by rays made
//    anew from the counter-based Philox stream.
//  * raptr_sm_build_csr: the production path (what getSystemMatrix +
//    cooSort + coo2csr + csr2ecsr produce, getSystemMatrixDeviceOnly.cu:
//    357-562, wrappers.hpp:185-266), one workgroup per channel.
//    k_sm_rays (see there) marks the voxels that each ray can meet and samples
//    only those; k_sm_build serves what it does not take (per-element rays,
//    zeros kept, masks larger than the LDS), with the steps:
//      1. the channel's rays are generated once into LDS, with per-ray plane
//         tables alpha[dim][k] = (o + k*d - r0)/(r1 - r0) for every grid plane
//         (the voxel-box divisions of the slab method depend only on the
//         plane index, so one division per plane and ray replaces six per
//         voxel and ray, with identical float results);
//      2. the cylinder cull takes the z intervals of 256 voxel columns at a
//         time and compacts the voxels that pass its test into LDS with wave
//         ballots (ascending voxel order preserved);
//      3. candidates are sampled densely (all lanes busy), exact zeros are
//         dropped with a second ballot compaction into an LDS row buffer;
//      4. row buffers are flushed as pieces into a staging area and packed
//         into a CSR with 64-bit row pointers per channel chunk.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>

#include "primitives.hpp"

namespace raptr {

// Scratch of the allocation-free build (raptr_sm_build_csr_noalloc): the
// staging area, counters, piece table and scan space of the fused build in
// device memory that exists from module load to process end, one copy per
// device.  `scratch` is a host-side stand-in in host code: the code below
// takes the array's device address once per device (hipGetSymbolAddress,
// with that device current) and uses only that address.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// the current device's address of `scratch` (looked up on its first use)
int scratch_address(void** out) {
  int dev = 0;
  RAPTR_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxScratchDevices)
    return fail(RAPTR_ERR_NOT_SUPPORTED, "device %d beyond the %d scratch slots", dev,
                kMaxScratchDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(RAPTR_ERR_DEVICE, "hipGetSymbolAddress(scratch) on device %d: %s", dev,
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return RAPTR_OK;
}

constexpr int kSmBlock = 256;
constexpr int kCandCap = 3072;  // >= 2048 + one cull round (256)
constexpr int kCandFlush = 2048;
constexpr int kRowBuf = 3072;   // >= kCandCap: one batch always fits

__device__ inline float min2(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline float max2(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline float min3(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ inline float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// ------------------------------------------------- two-stage kernels
// mean slab length of one pair, its rays made here
__device__ __forceinline__ float pair_value(const Geom& G, int c, int vv, int nrays, uint32_t seed,
                                   int raygen) {
  int ix, iy, iz;
  vxl_split(G.g, vv, ix, iy, iz);
  float box[6] = {plane(G.g, 0, ix),     plane(G.g, 1, iy),     plane(G.g, 2, iz),
                  plane(G.g, 0, ix + 1), plane(G.g, 1, iy + 1), plane(G.g, 2, iz + 1)};
  float a = 0.0f;
  for (int r = 0; r < nrays; ++r) {
    float ray[6];
    make_ray(G, raygen, seed, c, r, ray, vv);
    a += slab_length(box, ray);
  }
  a /= float(nrays);
  return a;
}

__global__ __launch_bounds__(256) void k_sm_from_wq(Geom G, const int* cnl, const int* vxl,
                                                    float* val, int64_t n, int nrays,
                                                    uint32_t seed, int raygen) {
  for (int64_t w = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; w < n;
       w += int64_t(gridDim.x) * blockDim.x) {
    int c = cnl[w], vv = vxl[w];
    if (c < 0 || c >= G.nch || vv < 0 || vv >= G.nvox) {
      val[w] = 0.0f;  // out-of-range pair: no geometry, no value
      continue;
    }
    const float a = pair_value(G, c, vv, nrays, seed, raygen);
    val[w] = a;
  }
}

// k_sm_from_wq for queues in channel order (as raptr_workqueue writes them):
// a workgroup's kWqChunk pairs hold few channels, so it makes a channel's rays
// and plane tables (as k_sm_build's) once in LDS for all of its pairs; a chunk of
// more than max_runs runs takes k_sm_from_wq's way, rays anew for every pair.
// The terms are slab_length's: a ray that misses the voxel adds +0.  8.4M
// pairs of 3,000 channels, 10 rays, 32^3 voxels: 519 -> 97 us,
// bound by the VALU of the ten slab tests.
constexpr int kWqChunk = 1024;

// Runs of a chunk up to which the shared tables pay; 0: not for this call.
// Measured with 2M pairs (us, p planes): pairs alone 15 + 10.5 nrays; shared 8 +
// 1.2 nrays and 8 + 0.0018 nrays p for each run, so 2, 10 and 21 runs with 1, 10
// and 30 rays of 99 planes (12 runs of 10 rays 134 shared, 122 alone; 16 of 30
// 262 and 321), 2, 7 and 12 with 291 (8 runs of 10 rays 120 and 119, 12 of 30 336
// and 318).  On short queues the tables' serial steps outlast the pairs: 65,536
// pairs, 10 rays, 32^3 voxels 9 us alone and 15 shared, 262,144 of 96^3 19 and 19
// to 26, 1M of 256^3 61 and 37 to 49; but many rays of one pair are as serial (64
// pairs, 30 rays, 32^3: 19 and 10).
inline int wq_max_runs(int64_t n, int nrays, int planes) {
  const bool few = n <= 256 && nrays >= 16;
  if (!few && double(n) * nrays < 4e6 + 8e3 * planes) return 0;
  return int((7.5 + 9.3 * nrays) / (8.0 + 0.0018 * double(nrays) * planes));
}

__global__ __launch_bounds__(256) void k_sm_from_wq_runs(Geom G, const int* __restrict__ cnl,
                                                         const int* __restrict__ vxl,
                                                         float* __restrict__ val, int64_t n,
                                                         int nrays, uint32_t seed, int raygen,
                                                         int max_runs, int stride,
                                                         FastDiv div_yz,
                                                         FastDiv div_z) {
  constexpr int PER = kWqChunk / 256;
  extern __shared__ float wq_lds[];
  __shared__ int s_runs[4], s_next;
  float* rays = wq_lds;                // nrays * 8: start, direction
  float* alpha = rays + 8 * nrays;     // nrays * stride: plane table, length
  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int nx = G.g.n[0], ny = G.g.n[1], nz = G.g.n[2];
  const int off1 = nx + 1, off2 = nx + ny + 2, pl = nx + ny + nz + 3;
  const int64_t base = int64_t(blockIdx.x) * kWqChunk;
  int c[PER], v[PER], runs = 0;
  unsigned todo = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int64_t i = base + k * 256 + t;
    c[k] = v[k] = -1;
    if (i < n) {
      c[k] = cnl[i];
      v[k] = vxl[i];
      todo |= 1u << k;
      const int before = i > base ? cnl[i - 1] : c[k] - 1;
      runs += c[k] != before ? 1 : 0;
      // out-of-range pair: no geometry, no value
      if (c[k] < 0 || c[k] >= G.nch || v[k] < 0 || v[k] >= G.nvox) {
        val[i] = 0.0f;
        todo &= ~(1u << k);
      }
    }
  }
  runs = wave_reduce_sum(runs);
  if (lane == 0) s_runs[w] = runs;
  if (t == 0) s_next = kWqChunk;
  __syncthreads();
  if (s_runs[0] + s_runs[1] + s_runs[2] + s_runs[3] > max_runs) {
#pragma unroll 1
    for (int k = 0; k < PER; ++k) {
      const int64_t i = base + k * 256 + t;
      if (todo >> k & 1) val[i] = pair_value(G, cnl[i], vxl[i], nrays, seed, raygen);
    }
    return;
  }
  for (;;) {
    // the first pair left names the channel of this turn
    if (todo) atomicMin(&s_next, (__ffs(int(todo)) - 1) * 256 + t);
    __syncthreads();
    const int next = s_next;
    if (next == kWqChunk) return;
    const int ch = cnl[base + next];
    for (int r = t; r < nrays; r += 256) {
      float ray[6];
      make_ray(G, raygen, seed, ch, r, ray);
      float* ri = rays + 8 * r;
      float d[3];
      bool same = true;
      for (int j = 0; j < 3; ++j) {
        d[j] = ray[3 + j] - ray[j];
        same = same && ray[j] == ray[3 + j];
        ri[j] = ray[j];
        ri[4 + j] = d[j];
      }
      ri[3] = same ? 0.0f : 1.0f;
      alpha[r * stride + pl] = sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    }
    __syncthreads();
    if (t == 0) s_next = kWqChunk;
    for (int p0 = 0; p0 < pl; p0 += kWave) {
      const int p = p0 + lane;
      const int dim = p < off1 ? 0 : (p < off2 ? 1 : 2);
      const int idx = p - (dim == 0 ? 0 : (dim == 1 ? off1 : off2));
      const float pos = plane(G.g, dim, idx);
      if (p < pl)
        for (int r = w; r < nrays; r += 4) {
          const float* ri = rays + 8 * r;
          const float d = ri[4 + dim];
          // a ray without length crosses nothing; an axis that it does not
          // cross is ignored: alternating infinities leave it unbounded there
          float a = ((idx & 1) ? 1.0f : -1.0f) * __builtin_inff();
          if (d != 0.0f) a = (pos - ri[dim]) / d;
          alpha[r * stride + p] = ri[3] == 0.0f ? 0.0f : a;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if ((todo >> k & 1) && c[k] == ch) {
        const int ix = int(fdiv(uint32_t(v[k]), div_yz));
        const int rem = v[k] - ix * int(div_yz.d);
        const int iy = int(fdiv(uint32_t(rem), div_z));
        const float* ax = alpha + ix;
        const float* ay = alpha + off1 + iy;
        const float* az = alpha + off2 + (rem - iy * nz);
        float a = 0.0f;
        for (int r = 0; r < nrays; ++r) {
          const int o = r * stride;
          const float xa = ax[o], xe = ax[o + 1], ya = ay[o], ye = ay[o + 1];
          const float za = az[o], ze = az[o + 1];
          const float lo = max3(min2(xa, xe), min2(ya, ye), min2(za, ze));
          const float hi = min3(max2(xa, xe), max2(ya, ye), max2(za, ze));
          a += max2(hi - lo, 0.0f) * alpha[o + pl];
        }
        val[base + k * 256 + t] = a / float(nrays);
        todo &= ~(1u << k);
      }
    __syncthreads();  // the tables are written again
  }
}

__global__ void k_generate_rays(Geom G, const int* cnl, int n_cnl, int nrays, uint32_t seed,
                                int raygen, float* rays) {
  int64_t total = int64_t(n_cnl) * nrays;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < total;
       k += int64_t(gridDim.x) * blockDim.x) {
    int64_t ci = k / nrays;
    int r = int(k - ci * nrays);
    int c = cnl[ci];
    if (c < 0 || c >= G.nch) {
      for (int q = 0; q < 6; ++q) rays[6 * k + q] = 0.0f;
      continue;
    }
    make_ray(G, raygen, seed, c, r, rays + 6 * k);
  }
}

// ----------------------------------------------------- fused build
struct Piece {
  int row;       // row within chunk
  int within;    // offset of the piece inside its row
  int64_t src;   // staging offset
  int len;
  int pad;
};

// One staging counter for all rows serialises the workgroups (two additions
// to one cache line took 25 ns a row, as long as the row itself), so large
// launches spread their rows over kAreas counters in separate lines.
constexpr int kAreas = kWave;  // (k_rowptr_fill: a lane each)
constexpr int kCountStride = 16;  // counters are 128 bytes apart
static_assert(sizeof(Piece) == 24, "the piece table's entries");

struct BuildArgs {
  Geom G;
  FastDiv div_yz, div_z;
  FastDiv div_c[4];     // channels per angle, id0z, id0y, id1z
  // k_sm_rays: 1 / pitch, farthest plane from 0, half a voxel's diagonal
  float inv_d[3], ext[3];
  float near2;       // squared end offset up to which no voxel can fail the cull
  bool plain_planes; // plane positions are 0 or of moderate size
  int rpb;          // rays per mask bit (k_sm_rays)
  const int* list;  // nullptr: channel = list index (all channels)
  int first;        // first list entry of this launch
  int rows;         // list entries in this launch
  int nrays;
  uint32_t seed;
  int raygen;
  int keep_zeros;   // store zero-valued candidates too (RAPTR_SM_KEEP_ZEROS)
  int by_candidate; // k_sm_build whatever the rays
  int pl;           // planes per ray (nx+1 + ny+1 + nz+1)
  // outputs
  int* row_nnz;     // [rows]
  int* st_col;      // staging
  float* st_val;
  int64_t st_cap;   // entries of one staging area
  int areas;        // staging areas (1 or kAreas), each with its own counter
  unsigned long long* st_count;  // [areas], kCountStride apart
  Piece* pieces;    // [0, rows): each row's first piece; then further ones
  int piece_cap;
  unsigned* piece_count;
  unsigned* flags;  // bit0 staging overflow, bit1 piece overflow
  double* colsum;   // sensitivity / back-projection mode
  // sensitivity: exact fixed-point column sums (value * 2^fx_bits rounded to
  // an integer, added with 64-bit integer atomics, so the result does not
  // depend on the order in which the atomics land); null: FP64 atomics
  unsigned long long* colsum_fx;
  double fx_scale;
  const float* wgt; // back-projection mode: weight per list entry (nullptr: 1)
  const float* xin; // forward-projection mode: image
  double* fwd;      // forward-projection mode: per-row FP64 projection
};

enum { kModeCount = 0, kModeFill = 1, kModeColsum = 2, kModeFwd = 3 };

__device__ inline float sample_voxel(const float* rinfo, const float* alpha, int nrays,
                                     int pl, int ix, int iy, int iz, int off1, int off2) {
  float a = 0.0f;
  for (int r = 0; r < nrays; ++r) {
    const float* ri = rinfo + 8 * r;
    const float* al = alpha + size_t(r) * pl;
    int bits = __float_as_int(ri[7]);
    float amin = 0.0f, amax = 0.0f;
    bool good = false;
    if (bits & 1) {
      float lo = al[ix], hi = al[ix + 1];
      if (hi < lo) {
        float t = lo;
        lo = hi;
        hi = t;
      }
      amin = lo;
      amax = hi;
      good = true;
    }
    if (bits & 2) {
      float lo = al[off1 + iy], hi = al[off1 + iy + 1];
      if (hi < lo) {
        float t = lo;
        lo = hi;
        hi = t;
      }
      amin = good ? (amin < lo ? lo : amin) : lo;
      amax = good ? (hi < amax ? hi : amax) : hi;
      good = true;
    }
    if (bits & 4) {
      float lo = al[off2 + iz], hi = al[off2 + iz + 1];
      if (hi < lo) {
        float t = lo;
        lo = hi;
        hi = t;
      }
      amin = good ? (amin < lo ? lo : amin) : lo;
      amax = good ? (hi < amax ? hi : amax) : hi;
    }
    float len = (amin < amax) ? (amax - amin) * ri[6] : 0.0f;
    a += len;
  }
  return a / float(nrays);
}

// RAPTR_RAYGEN_RAND_ELEMENT: the element's own nrays rays, slab method on
// the voxel box (the arithmetic of k_sm_from_wq, so both paths agree bit
// for bit).
__device__ inline float sample_element(const Geom& G, uint32_t seed, int nrays, int cnl,
                                       int v, int ix, int iy, int iz) {
  float box[6] = {plane(G.g, 0, ix),     plane(G.g, 1, iy),     plane(G.g, 2, iz),
                  plane(G.g, 0, ix + 1), plane(G.g, 1, iy + 1), plane(G.g, 2, iz + 1)};
  float a = 0.0f;
  for (int r = 0; r < nrays; ++r) {
    float ray[6];
    make_ray(G, RAPTR_RAYGEN_RAND_ELEMENT, seed, cnl, r, ray, v);
    a += slab_length(box, ray);
  }
  return a / float(nrays);
}

// staging area of a row (hashed: row lengths repeat with the pixel index)
__device__ inline int staging_area(const BuildArgs& A, int rl) {
  return A.areas == kAreas ? int((uint32_t(rl) * 0x9E3779B1u) >> 26) : 0;
}

// Staging offset of a piece of n entries of row rl (`within`: entries of the
// row before it), entered in the piece table; -1 (and a flag) if full.
__device__ inline long long reserve_piece(const BuildArgs& A, int rl, int within, int n) {
  const int area = staging_area(A, rl);
  const long long off = (long long)atomicAdd(&A.st_count[area * kCountStride],
                                             (unsigned long long)n);
  if (off + n > A.st_cap) {
    atomicOr(A.flags, 1u);
    return -1;
  }
  const unsigned pc = within == 0 ? unsigned(rl) : unsigned(A.rows) + atomicAdd(A.piece_count, 1u);
  if (int64_t(pc) >= A.piece_cap) {
    atomicOr(A.flags, 2u);
    return -1;
  }
  const long long o = area * A.st_cap + off;
  A.pieces[pc] = Piece{rl, within, o, n, 0};
  return o;
}

template <int MODE>
__global__ __launch_bounds__(kSmBlock) void k_sm_build(BuildArgs A) {
  extern __shared__ float smem[];
  __shared__ int wcnt[kSmBlock / kWave];
  __shared__ int s_scan[kSmBlock / kWave];
  __shared__ int s_lo[kSmBlock], s_pre[kSmBlock];
  __shared__ long long s_off;
  const int nr = A.nrays, pl = A.pl;
  float* rinfo = smem;                                   // nr * 8
  float* alpha = rinfo + 8 * nr;                         // nr * pl
  int* cand = reinterpret_cast<int*>(alpha + size_t(nr) * pl);
  float* cval = reinterpret_cast<float*>(cand + kCandCap);
  int* rb_col = reinterpret_cast<int*>(cval + kCandCap);
  float* rb_val = reinterpret_cast<float*>(rb_col + kRowBuf);

  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int nx = A.G.g.n[0], ny = A.G.g.n[1];
  const int off1 = nx + 1, off2 = nx + 1 + ny + 1;

  for (int rl = blockIdx.x; rl < A.rows; rl += gridDim.x) {
    const int li = A.first + rl;
    int cnl = A.list ? A.list[li] : li;
    // an out-of-range channel id yields an empty row (uniform branch)
    const bool bad = cnl < 0 || cnl >= A.G.nch;
    if (bad) cnl = 0;
    // 1. rays and plane tables
    for (int r = t; r < nr; r += kSmBlock) {
      float ray[6];
      make_ray(A.G, A.raygen, A.seed, cnl, r, ray);
      float dx = ray[3] - ray[0], dy = ray[4] - ray[1], dz = ray[5] - ray[2];
      int bits = (ray[0] != ray[3] ? 1 : 0) | (ray[1] != ray[4] ? 2 : 0) |
                 (ray[2] != ray[5] ? 4 : 0);
      float* ri = rinfo + 8 * r;
      ri[0] = ray[0];
      ri[1] = ray[1];
      ri[2] = ray[2];
      ri[3] = dx;
      ri[4] = dy;
      ri[5] = dz;
      ri[6] = sqrtf(dx * dx + dy * dy + dz * dz);
      ri[7] = __int_as_float(bits);
    }
    __syncthreads();
    for (int k = t; k < nr * pl; k += kSmBlock) {
      int r = k / pl, p = k - r * pl;
      int dim = p < off1 ? 0 : (p < off2 ? 1 : 2);
      int idx = p - (dim == 0 ? 0 : (dim == 1 ? off1 : off2));
      const float* ri = rinfo + 8 * r;
      int bits = __float_as_int(ri[7]);
      float v = 0.0f;
      if (bits & (1 << dim)) v = (plane(A.G.g, dim, idx) - ri[dim]) / ri[3 + dim];
      alpha[k] = v;
    }
    __syncthreads();

    int cand_n = 0, rb_n = 0, flushed = 0;
    double proj = 0.0;
    // sample, then keep (or count / accumulate) the candidates in cand[]
    auto process = [&]() {
      // 3. sample candidates densely
      for (int c = t; c < cand_n; c += kSmBlock) {
        int v = cand[c];
        uint32_t qx = fdiv(uint32_t(v), A.div_yz);
        uint32_t rem = uint32_t(v) - qx * A.div_yz.d;
        uint32_t qy = fdiv(rem, A.div_z);
        const int iz = int(rem - qy * A.div_z.d);
        cval[c] = A.raygen == RAPTR_RAYGEN_RAND_ELEMENT
                      ? sample_element(A.G, A.seed, nr, cnl, v, int(qx), int(qy), iz)
                      : sample_voxel(rinfo, alpha, nr, pl, int(qx), int(qy), iz, off1, off2);
      }
      __syncthreads();
      if (MODE == kModeColsum) {
        const double wt = A.wgt ? double(A.wgt[li]) : 1.0;
        for (int c = t; c < cand_n; c += kSmBlock) {
          float a = cval[c];
          if (A.colsum_fx) {
            if (a != 0.0f)
              atomicAdd(&A.colsum_fx[cand[c]],
                        (unsigned long long)llrint(double(a) * A.fx_scale));
          } else if (a != 0.0f && wt != 0.0) {
            atomicAdd(&A.colsum[cand[c]], double(a) * wt);
          }
        }
        __syncthreads();
        cand_n = 0;
        return;
      }
      if (MODE == kModeFwd) {
        for (int c = t; c < cand_n; c += kSmBlock)
          proj += double(cval[c]) * double(A.xin[cand[c]]);
        __syncthreads();
        cand_n = 0;
        return;
      }
      // flush the row buffer first if the candidates could overflow it
      if (MODE == kModeFill && rb_n + cand_n > kRowBuf) {
        if (t == 0) s_off = reserve_piece(A, rl, flushed, rb_n);
        __syncthreads();
        long long o = s_off;
        if (o >= 0)
          for (int k = t; k < rb_n; k += kSmBlock) {
            A.st_col[o + k] = rb_col[k];
            A.st_val[o + k] = rb_val[k];
          }
        flushed += rb_n;
        rb_n = 0;
        __syncthreads();
      }
      // compact non-zeros in candidate order
      for (int c0 = 0; c0 < cand_n; c0 += kSmBlock) {
        int c = c0 + t;
        bool nz = c < cand_n && (A.keep_zeros || cval[c] != 0.0f);
        uint64_t m = __ballot(nz);
        if (lane == 0) wcnt[w] = __popcll(m);
        __syncthreads();
        int pre = 0, tot = 0;
        for (int ww = 0; ww < kSmBlock / kWave; ++ww) {
          int cc = wcnt[ww];
          pre += ww < w ? cc : 0;
          tot += cc;
        }
        if (MODE == kModeFill && nz) {
          int pos = rb_n + pre + __popcll(m & lanemask_lt());
          rb_col[pos] = cand[c];
          rb_val[pos] = cval[c];
        }
        rb_n += tot;
        __syncthreads();
      }
      if (MODE == kModeCount) {
        flushed += rb_n;
        rb_n = 0;
      }
      cand_n = 0;
    };
    // 2. cull: the z intervals of the voxel columns, then the reference's
    // exact float test on every voxel in them.  Columns run in ascending (ix,
    // iy) and z ascends within a column, so the candidates and their order
    // are those of a scan over all voxels.
    const int nz = A.G.g.n[2];
    const int ncols = nx * ny;
    const LineInterval L(A.G, cnl);
    for (int cb = 0; cb < (bad ? 0 : ncols); cb += kSmBlock) {
      const int cc = cb + t;
      int lo = 0, cnt = 0;
      if (cc < ncols) cnt = L.column(A.G.g, cc / ny, cc - (cc / ny) * ny, lo);
      int tot;
      const int pre = block_exclusive_scan<int, kSmBlock>(cnt, s_scan, &tot);
      s_lo[t] = lo;
      s_pre[t] = pre;
      __syncthreads();
      for (int k0 = 0; k0 < tot; k0 += kSmBlock) {
        const int k = k0 + t;
        bool pass = false;
        int v = 0;
        if (k < tot) {
          int jl = 0, jh = kSmBlock - 1;  // last column with s_pre <= k
          while (jl < jh) {
            const int mid = (jl + jh + 1) >> 1;
            if (s_pre[mid] <= k) jl = mid; else jh = mid - 1;
          }
          const int col = cb + jl;
          const int ix = col / ny, iy = col - (col / ny) * ny;
          const int iz = s_lo[jl] + (k - s_pre[jl]);
          v = col * nz + iz;
          float c[3];
          voxel_centre(A.G.g, ix, iy, iz, c);
          pass = distance_point_line(L.p0, L.p1, c) < A.G.sumRadii;
        }
        uint64_t m = __ballot(pass);
        if (lane == 0) wcnt[w] = __popcll(m);
        __syncthreads();
        int wpre = 0, wtot = 0;
        for (int ww = 0; ww < kSmBlock / kWave; ++ww) {
          const int c = wcnt[ww];
          wpre += ww < w ? c : 0;
          wtot += c;
        }
        if (pass) cand[cand_n + wpre + __popcll(m & lanemask_lt())] = v;
        cand_n += wtot;
        __syncthreads();
        if (cand_n >= kCandFlush) process();
      }
      __syncthreads();
    }
    if (cand_n > 0) process();
    if (MODE == kModeFill && rb_n > 0) {
      if (t == 0) s_off = reserve_piece(A, rl, flushed, rb_n);
      __syncthreads();
      long long o = s_off;
      if (o >= 0)
        for (int k = t; k < rb_n; k += kSmBlock) {
          A.st_col[o + k] = rb_col[k];
          A.st_val[o + k] = rb_val[k];
        }
      flushed += rb_n;
      rb_n = 0;
    }
    if (MODE == kModeFwd) {
      // fixed-order block reduction of the per-thread FP64 partials
      proj = wave_reduce_sum(proj);
      __shared__ double wred[kSmBlock / kWave];
      if (lane == 0) wred[w] = proj;
      __syncthreads();
      if (t == 0) {
        double tot = 0.0;
        for (int ww = 0; ww < kSmBlock / kWave; ++ww) tot += wred[ww];
        A.fwd[li] = tot;
      }
    }
    if ((MODE == kModeCount || MODE == kModeFill) && t == 0) A.row_nnz[rl] = flushed;
    if (MODE == kModeFill && t == 0 && flushed == 0) A.pieces[rl] = Piece{rl, 0, 0, 0, 0};
    __syncthreads();
  }
}

// ------------------------------------------- fused build by ray masks
// k_sm_build tests every culled voxel against every ray, and 95 % of its
// candidates turn out to be zero.  Here each ray marks the voxels that it can
// cross, so only those are sampled, by the rays that marked them:
//   1. the channel's rays and their plane tables in LDS, as in k_sm_build;
//   2. the grid is cut into slabs along x or z, whichever the line runs along;
//      per (ray, slab) the cells that the ray can cross there on the two
//      other axes form two ranges, widened by more than their rounding error.
//      The ray's bit goes into the slab's mask words of those cells, kMw words
//      per slab and axis indexed by the cell modulo kMw: cells that share a
//      word, or a range too wide for the words, only add bits.  The ranges
//      also give each x index the (y, z) rectangle that can hold hits;
//   3. the rectangles are walked in ascending voxel order, the two masks of a
//      voxel ANDed; a voxel with bits left is summed over the rays of those
//      bits in ascending order, with k_sm_build's arithmetic.  A ray that
//      is not in the mask does not cross the voxel, its term would be +0, so
//      sums are the same bit for bit.
// On the 52^3 / 30-ray geometry a row walks 446 voxels, 361 keep bits and 358
// are non-zero (k_sm_build: 5,900 candidates).  More than 32 rays share bits
// in runs of `rpb` consecutive rays.
// Bound by VALU issue (80 % busy) and LDS latency: 1,920 VALU instructions a
// wave and row, a quarter each in the plane tables and the masks.  Measured,
// k_sm_build -> masks -> with the voxels in order of their bits, odd table
// strides, one staging request a row and half the barriers: 100,003 rows of
// that geometry 58.0 -> 3.25 -> 1.78 ms, 20,011 rows of 96^3 / 20 rays 17.0 ->
// 0.90 -> 0.66 ms, sensitivity of 147,456 channels (32^3 / 10 rays) 16.9 ->
// 1.19 -> 0.96 ms.
constexpr int kMw = 8;              // mask words per slab and axis
constexpr int kMRow = 768;          // voxels of a segment; entries of the row buffer

// Position of a ray on an axis in cells as base + a * slope, and the bound of
// its rounding error, that of the plane tables included: every term is below
// 2^-23 of (|r0| + ext) * inv, ext the farthest plane; eps is 32 of them.  A
// ray that does not cross the axis is not bounded there: eps infinite.
__device__ inline void axis_line(float r0, float d, float o, float inv, float ext, float* out) {
  out[0] = d != 0.0f ? (r0 - o) * inv : 0.0f;
  out[1] = d * inv;
  out[2] = d != 0.0f ? (fabsf(r0) + ext) * inv * 3.814697265625e-6f : __builtin_inff();
}

// floor to int; out of int range: its nearest end
__device__ inline int floor_int(float a) {
  int r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(a));
  return r;
}

// Cells [c0, c1] that the ray can cross for a in [lo, hi] (finite); empty if
// c0 > c1.
__device__ inline void cell_range(const float* line, int n, float lo, float hi, int& c0, int& c1) {
  const float pa = __builtin_fmaf(lo, line[1], line[0]);
  const float pb = __builtin_fmaf(hi, line[1], line[0]);
  c0 = floor_int(min2(pa, pb) - line[2]);
  c1 = floor_int(max2(pa, pb) + line[2]);
  c0 = c0 > 0 ? c0 : 0;
  c1 = c1 < n - 1 ? c1 : n - 1;
}

// Words that every wave writes alike and reads back: LDS accesses of a wave
// are issued in program order; the compiler must keep that order.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// a is 0 or of magnitude 2^-e .. 2^e
__host__ __device__ inline bool plain_size(float a, int e) {
  const float b = a < 0.0f ? -a : a;
  return b == 0.0f ? e == 60 : b >= 1.0f / float(1ull << e) && b <= float(1ull << e);
}

template <int MODE, bool ONE, int NW>
__global__ __launch_bounds__(NW * kWave) void k_sm_rays(BuildArgs A) {
  constexpr int NT = NW * kWave, CH = kMRow / NW;  // CH: a wave's voxels of a segment
  extern __shared__ float smem[];
  __shared__ int s_wn[NW], s_kept[NW], s_cull[NW];
  __shared__ float s_dev[NW];
  __shared__ int s_pre[kWave], s_wz[kWave];  // of an x index: voxels before it, z cells
  __shared__ int s_bin[32], s_place[32];     // voxels by number of mask bits
  __shared__ unsigned short s_ord[kMRow];    // list positions, most bits first
  __shared__ double s_red[NW];
  __shared__ long long s_off;
  const int nr = A.nrays, pl = A.pl;
  const int nx = A.G.g.n[0], ny = A.G.g.n[1], nz = A.G.g.n[2];
  const int off1 = nx + 1, off2 = nx + 1 + ny + 1;
  const int nsm = nx > nz ? nx : nz;
  // plane table and length of a ray, an odd number of words: the rays of a
  // wave's lanes then lie in different banks
  const int stride = (pl + 1) | 1;
  float* alpha = smem;                                     // nr * stride
  unsigned* my = reinterpret_cast<unsigned*>(alpha + size_t(nr) * stride);  // nsm * kMw
  unsigned* mt = my + nsm * kMw;                           // nsm * kMw
  int* ylo = reinterpret_cast<int*>(mt + nsm * kMw);       // nx each
  int* yhi = ylo + nx;
  int* zlo = yhi + nx;
  int* zhi = zlo + nx;
  // the rays (16 floats each) until the masks stand, then the wave lists
  int* l_vox = zhi + nx;                                   // NW * CH
  unsigned* l_bit = reinterpret_cast<unsigned*>(l_vox + kMRow);  // mask, then value
  float* rays = reinterpret_cast<float*>(l_vox);

  const int t = threadIdx.x, lane = t & (kWave - 1), w = t / kWave;
  const int rl = blockIdx.x;
  const int li = A.first + rl;
  const int cnl = A.list ? A.list[li] : li;
  if (cnl < 0 || cnl >= A.G.nch) {  // out-of-range channel id: an empty row
    if (t == 0) {
      if (MODE == kModeFwd) A.fwd[li] = 0.0;
      if (MODE == kModeCount || MODE == kModeFill) A.row_nnz[rl] = 0;
      if (MODE == kModeFill) A.pieces[rl] = Piece{rl, 0, 0, 0, 0};
    }
    return;
  }
  // cnl_split by multiplications (the channel is uniform: scalar unit)
  uint32_t q = uint32_t(cnl);
  const int ida = int(fdiv(q, A.div_c[0]));
  q -= uint32_t(ida) * A.div_c[0].d;
  const int id0z = int(fdiv(q, A.div_c[1]));
  q -= uint32_t(id0z) * A.div_c[1].d;
  const int id0y = int(fdiv(q, A.div_c[2]));
  q -= uint32_t(id0y) * A.div_c[2].d;
  const int id1z = int(fdiv(q, A.div_c[3]));
  const int id1y = int(q - uint32_t(id1z) * A.div_c[3].d);
  const float sn = A.G.sn[ida], cs = A.G.cs[ida];
  float p0[3], p1[3];
  trafo(A.G.s, 0, sn, cs, id0z, id0y, 0.5f, 0.5f, 0.5f, p0);
  trafo(A.G.s, 1, sn, cs, id1z, id1y, 0.5f, 0.5f, 0.5f, p1);
  // slabs along the axis that the line runs along
  const bool zs = fabsf(p1[2] - p0[2]) > fabsf(p1[0] - p0[0]);
  const int ns = zs ? nz : nx, nt = zs ? nx : nz;
  const int td = zs ? 0 : 2;
  // rays: lane 2k makes the start of ray k, lane 2k + 1 its end (the
  // uniforms of make_ray: three words of the first Philox block, then its
  // fourth and two of the second)
  float far_end = 0.0f;  // largest squared distance of a ray's end from its pixel centre
  bool cullw = false;    // a ray that does not follow the line between the heads
  for (int k = t; k < ((2 * nr + kWave - 1) & ~(kWave - 1)); k += NT) {
    const int r = k >> 1, det = k & 1;
    float b0 = 0.5f, b1 = 0.5f, b2 = 0.5f;
    if (A.raygen != RAPTR_RAYGEN_REGU) {
      uint32_t o[4];
      philox4x32_10(uint32_t(cnl), uint32_t(r), uint32_t(det), 0u, A.seed, 0u, o);
      const uint32_t w3 = __shfl_xor(o[3], 1, kWave);
      b0 = u01(det ? w3 : o[0]);
      b1 = u01(det ? o[0] : o[1]);
      b2 = u01(det ? o[1] : o[2]);
    }
    float e[3], d[3], dev = 0.0f;
    trafo(A.G.s, det, sn, cs, det ? id1z : id0z, det ? id1y : id0y, b0, b1, b2, e);
    bool same = true;
    for (int j = 0; j < 3; ++j) {
      const float far = __shfl_xor(e[j], 1, kWave);  // lane 2k: the ray's end
      same = same && e[j] == far;
      d[j] = far - e[j];
      const float off = e[j] - (det ? p1[j] : p0[j]);
      dev += off * off;
    }
    if (r < nr) far_end = max2(far_end, dev);
    cullw = cullw || (r < nr && (d[0] == 0.0f || d[1] == 0.0f || d[2] == 0.0f));
    if (det == 0 && r < nr) {
      float* ri = rays + 16 * r;
      for (int j = 0; j < 3; ++j) {
        ri[j] = e[j];
        ri[4 + j] = d[j];
      }
      bool plain = A.plain_planes;
      for (int j = 0; j < 3; ++j) plain = plain && plain_size(d[j], 40) && plain_size(e[j], 60);
      ri[3] = same ? 0.0f : plain ? 2.0f : 1.0f;
      axis_line(e[1], d[1], A.G.g.o[1], A.inv_d[1], A.ext[1], ri + 8);
      axis_line(zs ? e[0] : e[2], zs ? d[0] : d[2], A.G.g.o[td], A.inv_d[td], A.ext[td],
                ri + 12);
      ri[7] = 1.0f / d[2];
      ri[11] = 1.0f / d[0];
      ri[15] = 1.0f / d[1];
      alpha[r * stride + pl] = sqrtf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    }
  }
  for (int j = kWave / 2; j > 0; j >>= 1) far_end = max2(far_end, __shfl_xor(far_end, j, kWave));
  if (lane == 0) s_dev[w] = far_end;
  if (t < 32) s_bin[t] = s_place[t] = 0;
  for (int k = t; k < 2 * nsm * kMw; k += NT) my[k] = 0u;
  for (int k = t; k < nx; k += NT) {
    ylo[k] = zlo[k] = 0x7fffffff;
    yhi[k] = zhi[k] = -1;
  }
  __syncthreads();
  // plane tables: a lane keeps its plane, a wave takes every NW-th ray
  for (int p0_ = 0; p0_ < pl; p0_ += kWave) {
    const int p = p0_ + lane;
    const int dim = p < off1 ? 0 : (p < off2 ? 1 : 2);
    const int idx = p - (dim == 0 ? 0 : (dim == 1 ? off1 : off2));
    const int inv = dim == 0 ? 11 : dim == 1 ? 15 : 7;
    const float pos = plane(A.G.g, dim, idx);
    if (p < pl)
      for (int r = w; r < nr; r += NW) {
        const float* ri = rays + 16 * r;
        const float a = pos - ri[dim], d = ri[4 + dim];
        float v;
        if (__builtin_amdgcn_readfirstlane(__float_as_int(ri[3])) == 0x40000000) {
          // a / d from the rounded reciprocal: two residual steps give the
          // correctly rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990)
          // where neither it nor the residuals leave the normal range
          const float y = ri[inv];
          v = a * y;
          v = __builtin_fmaf(__builtin_fmaf(-v, d, a), y, v);
          v = __builtin_fmaf(__builtin_fmaf(-v, d, a), y, v);
        } else {
          // a ray without length crosses nothing; an axis that the ray does
          // not cross is ignored by the slab method: alternating infinities
          // leave every cell unbounded there
          v = ((idx & 1) ? 1.0f : -1.0f) * __builtin_inff();
          if (d != 0.0f) v = a / d;
          if (ri[3] == 0.0f) v = 0.0f;
        }
        alpha[r * stride + p] = v;
      }
  }
  __syncthreads();
  // masks, and the window of cells per slab: a lane keeps its slab
  for (int s0 = 0; s0 < ns; s0 += kWave) {
    const int sl = s0 + lane;
    int wy0 = 0x7fffffff, wy1 = -1, wt0 = 0x7fffffff, wt1 = -1;
    if (sl < ns)
      for (int r = w; r < nr; r += NW) {
        const float* ri = rays + 16 * r;
        const float* al = alpha + r * stride + (zs ? off2 : 0) + sl;
        const float a0 = al[0], a1 = al[1];
        // (an uncrossed slab axis leaves infinities)
        const float lo = max2(min2(a0, a1), -1e30f), hi = min2(max2(a0, a1), 1e30f);
        int y0, y1, t0, t1;
        cell_range(ri + 8, ny, lo, hi, y0, y1);
        cell_range(ri + 12, nt, lo, hi, t0, t1);
        if (y0 > y1 || t0 > t1 || ri[3] == 0.0f || lo >= hi) continue;
        cullw = cullw || lo < 0.0f || hi > 1.0f;
        const unsigned bit = 1u << (ONE ? r : r / A.rpb);
        wy0 = y0 < wy0 ? y0 : wy0;
        wy1 = y1 > wy1 ? y1 : wy1;
        wt0 = t0 < wt0 ? t0 : wt0;
        wt1 = t1 > wt1 ? t1 : wt1;
        unsigned* sy = my + sl * kMw;
        unsigned* st = mt + sl * kMw;
        // mostly one or two cells; kMw of them reach every word
        atomicOr(&sy[y0 & (kMw - 1)], bit);
        atomicOr(&sy[y1 & (kMw - 1)], bit);
        atomicOr(&st[t0 & (kMw - 1)], bit);
        atomicOr(&st[t1 & (kMw - 1)], bit);
        if (y1 - y0 > 1 || t1 - t0 > 1) {
          y1 = y1 - y0 < kMw ? y1 : y0 + kMw;
          t1 = t1 - t0 < kMw ? t1 : t0 + kMw;
          while (++y0 < y1) atomicOr(&sy[y0 & (kMw - 1)], bit);
          while (++t0 < t1) atomicOr(&st[t0 & (kMw - 1)], bit);
        }
      }
    if (wy1 >= 0) {
      const int x0 = zs ? wt0 : sl, x1 = zs ? wt1 : sl;
      for (int x = x0; x <= x1; ++x) {
        atomicMin(&ylo[x], wy0);
        atomicMax(&yhi[x], wy1);
        atomicMin(&zlo[x], zs ? sl : wt0);
        atomicMax(&zhi[x], zs ? sl : wt1);
      }
    }
  }
  // (one store a wave: the compiler keeps no order between the stores of
  // different lanes to one word)
  const int any_cull = __ballot(cullw) != 0u ? 1 : 0;
  if (lane == 0) s_cull[w] = any_cull;
  __syncthreads();

  // Between the heads a ray is no farther from the channel's line than the
  // farther of its ends from its pixel centre, so a voxel that it crosses is
  // within that and half the voxel's diagonal of the line: mostly less than
  // the cull's radius for all rays, by more than the test's rounding error,
  // and no voxel needs the test.  It stays where a ray does not cross an axis
  // (the slab method then takes voxels off the ray) or is crossed outside.
  bool cull = false;
  for (int ww = 0; ww < NW; ++ww) {
    cull = cull || s_cull[ww];
    far_end = max2(far_end, s_dev[ww]);
  }
  cull = cull || !(far_end < A.near2);

  int row_n = 0;  // fill: entries of the row so far
  int count = 0;  // count: this thread's entries
  double proj = 0.0;
  const double wt = (MODE == kModeColsum && A.wgt) ? double(A.wgt[li]) : 1.0;
  // fill: room for a voxel of every rectangle in the staging, one request a
  // row (its answer is waited for when the first entries are written)
  unsigned long long room = 0;
  int vox_all = 0;
  if (MODE == kModeFill) {
    for (int x = lane; x < nx; x += kWave)
      if (yhi[x] >= ylo[x]) vox_all += (yhi[x] - ylo[x] + 1) * (zhi[x] - zlo[x] + 1);
    vox_all = wave_reduce_sum(vox_all);
    if (t == 0) room = atomicAdd(&A.st_count[staging_area(A, rl) * kCountStride],
                                 (unsigned long long)vox_all);
  }
  int* wv = l_vox + w * CH;
  unsigned* wb = l_bit + w * CH;
  // items [k0, k1) of the current rectangles, by one wave: voxels with bits
  // left, listed in order and counted by their number of bits
  auto list_items = [&](int k0, int k1, int xb) -> int {
    int n = 0;
    for (int k = k0 + lane; k - lane < k1; k += kWave) {
      unsigned m = 0u;
      int v = 0;
      if (k < k1) {
        int jl = 0;  // last x index with prefix <= k
#pragma unroll
        for (int j = kWave / 2; j > 0; j >>= 1)
          if (s_pre[jl + j] <= k) jl += j;
        const int ix = xb + jl;
        const int q = k - s_pre[jl], wz = s_wz[jl];
        int qy = int((float(q) + 0.5f) * __builtin_amdgcn_rcpf(float(wz)));
        int qz = q - int(__umul24(unsigned(qy), unsigned(wz)));
        if (qz < 0) qz += wz, --qy;
        if (qz >= wz) qz -= wz, ++qy;
        const int iy = ylo[ix] + qy, iz = zlo[ix] + qz;
        const int sl = zs ? iz : ix, tt = zs ? ix : iz;
        m = my[sl * kMw + (iy & (kMw - 1))] & mt[sl * kMw + (tt & (kMw - 1))];
        v = int(__umul24(unsigned(__umul24(unsigned(ix), unsigned(ny)) + iy), unsigned(nz))) + iz;
      }
      const uint64_t b = __ballot(m != 0u);
      if (m) {
        const int pos = n + __popcll(b & lanemask_lt());
        wv[pos] = v;
        wb[pos] = m;
        atomicAdd(&s_bin[32 - __popc(m)], 1);
      }
      n += __popcll(b);
    }
    return n;
  };
  // value of a voxel: mean over the rays of its bits, 0 outside the cull
  auto sample = [&](int v, unsigned m) -> float {
    float a = 0.0f;
    const int ix = int(fdiv(uint32_t(v), A.div_yz));
    const int rem = v - ix * int(A.div_yz.d);
    const int iy = int(fdiv(uint32_t(rem), A.div_z));
    const int iz = rem - iy * nz;
    // (byte offsets below 2^24: a full-rate multiplication)
    const char* ax = reinterpret_cast<const char*>(alpha + ix);
    const char* ay = reinterpret_cast<const char*>(alpha + off1 + iy);
    const char* az = reinterpret_cast<const char*>(alpha + off2 + iz);
    const char* al = reinterpret_cast<const char*>(alpha + pl);
    while (m) {
      const int b = __ffs(int(m)) - 1;
      m &= m - 1u;
      const int r0 = ONE ? b : b * A.rpb;
      const int r1 = ONE ? b + 1 : (r0 + A.rpb < nr ? r0 + A.rpb : nr);
      for (int r = r0; r < r1; ++r) {
        const unsigned o = __umul24(unsigned(r), 4u * unsigned(stride));
        const float* x = reinterpret_cast<const float*>(ax + o);
        const float* y = reinterpret_cast<const float*>(ay + o);
        const float* z = reinterpret_cast<const float*>(az + o);
        const float xa = x[0], xe = x[1], ya = y[0], ye = y[1], za = z[0], ze = z[1];
        const float lo = max3(min2(xa, xe), min2(ya, ye), min2(za, ze));
        const float hi = min3(max2(xa, xe), max2(ya, ye), max2(za, ze));
        a += max2(hi - lo, 0.0f) * *reinterpret_cast<const float*>(al + o);
      }
    }
    a /= float(nr);
    if (cull && a != 0.0f) {
      float end[3] = {p1[0], p1[1], p1[2]}, ctr[3];
      // (keeps the line's length in here: few channels need it)
      asm volatile("" : "+v"(end[0]), "+v"(end[1]), "+v"(end[2]));
      voxel_centre(A.G.g, ix, iy, iz, ctr);
      if (!(distance_point_line(p0, end, ctr) < A.G.sumRadii)) a = 0.0f;
    }
    return a;
  };
  for (int xb = 0; xb < nx; xb += kWave) {
    // every wave makes the same prefix (and writes the same words)
    int area = 0, wz = 0;
    const int x = xb + lane;
    if (x < nx && yhi[x] >= ylo[x]) {
      wz = zhi[x] - zlo[x] + 1;
      area = (yhi[x] - ylo[x] + 1) * wz;
    }
    const int incl = wave_inclusive_scan(area);
    const int tot = __shfl(incl, kWave - 1, kWave);
    if (tot == 0) continue;
    s_pre[lane] = incl - area;
    s_wz[lane] = wz;
    wave_lds_fence();
    const int nseg = (tot + kMRow - 1) / kMRow;
    const int seg = (tot + nseg - 1) / nseg;
    const int part = (seg + NW - 1) / NW;
    for (int s0 = 0; s0 < tot; s0 += seg) {
      const int s1 = s0 + seg < tot ? s0 + seg : tot;
      const int k0 = s0 + w * part < s1 ? s0 + w * part : s1;
      const int k1 = k0 + part < s1 ? k0 + part : s1;
      const int n = list_items(k0, k1, xb);
      if (lane == 0) s_wn[w] = n;
      __syncthreads();
      int all = 0;
      for (int ww = 0; ww < NW; ++ww) all += s_wn[ww];
      // voxels in order of their number of bits: the lanes of a wave then
      // loop alike (in list order a wave ran 3.9 times its mean)
      const int bin = lane < 32 ? s_bin[lane] : 0;
      const int first = wave_inclusive_scan(bin) - bin;
      for (int c = lane; c - lane < n; c += kWave) {
        const int bb = c < n ? 32 - __popc(wb[c]) : 0;
        const int f = __shfl(first, bb, kWave);
        if (c < n) s_ord[f + atomicAdd(&s_place[bb], 1)] = (unsigned short)(w * CH + c);
      }
      __syncthreads();
      if (t < 32) s_bin[t] = s_place[t] = 0;
      for (int c = t; c < all; c += NT) {
        const int j = s_ord[c];
        const float a = sample(l_vox[j], l_bit[j]);
        if (MODE == kModeCount)
          count += a != 0.0f ? 1 : 0;
        else
          l_bit[j] = __float_as_uint(a);
      }
      if (MODE == kModeFill && t == 0) {
        const int64_t end = int64_t(room) + vox_all;
        s_off = end <= A.st_cap ? int64_t(staging_area(A, rl)) * A.st_cap + int64_t(room) : -1;
      }
      __syncthreads();
      if (MODE == kModeColsum || MODE == kModeFwd) {
        // in list order: neighbouring lanes, neighbouring voxels
        for (int c = lane; c < n; c += kWave) {
          const float a = __uint_as_float(wb[c]);
          const int v = wv[c];
          if (a == 0.0f) continue;
          if (MODE == kModeFwd)
            proj += double(a) * double(A.xin[v]);
          else if (A.colsum_fx)
            atomicAdd(&A.colsum_fx[v], (unsigned long long)llrint(double(a) * A.fx_scale));
          else if (wt != 0.0)
            atomicAdd(&A.colsum[v], double(a) * wt);
        }
      }
      if (MODE == kModeFill) {
        // non-zero entries in list order into the row's staging
        int kept = 0;
        for (int c = lane; c - lane < n; c += kWave)
          kept += __popcll(__ballot(c < n && wb[c] << 1 != 0u));
        if (lane == 0) s_kept[w] = kept;
        __syncthreads();
        int wpre = 0, sum = 0;
        for (int ww = 0; ww < NW; ++ww) {
          wpre += ww < w ? s_kept[ww] : 0;
          sum += s_kept[ww];
        }
        const int64_t off = s_off;
        for (int c = lane; c - lane < n; c += kWave) {
          const unsigned a = c < n ? wb[c] : 0u;
          const uint64_t b = __ballot(a << 1 != 0u);
          if (off >= 0 && a << 1 != 0u) {
            const int64_t pos = off + row_n + wpre + __popcll(b & lanemask_lt());
            A.st_col[pos] = wv[c];
            A.st_val[pos] = __uint_as_float(a);
          }
          wpre += __popcll(b);
        }
        row_n += sum;
      }
      // the lists and counts are written again
      if (s1 < tot || xb + kWave < nx) __syncthreads();
    }
  }
  if (MODE == kModeFill && t == 0) {
    if (vox_all && s_off < 0) atomicOr(A.flags, 1u);
    A.row_nnz[rl] = row_n;
    A.pieces[rl] = Piece{rl, 0, vox_all ? s_off : 0, row_n, 0};
  }
  if (MODE == kModeCount) {
    count = wave_reduce_sum(count);
    if (lane == 0) s_kept[w] = count;
    __syncthreads();
    if (t == 0) {
      int n = 0;
      for (int ww = 0; ww < NW; ++ww) n += s_kept[ww];
      A.row_nnz[rl] = n;
    }
  }
  if (MODE == kModeFwd) {
    // fixed-order block reduction of the per-thread FP64 partials
    proj = wave_reduce_sum(proj);
    if (lane == 0) s_red[w] = proj;
    __syncthreads();
    if (t == 0) {
      double tot = 0.0;
      for (int ww = 0; ww < NW; ++ww) tot += s_red[ww];
      A.fwd[li] = tot;
    }
  }
}

// fixed-point column sums -> FP64, in place
__global__ void k_fx_to_f64(unsigned long long* v, int n, double inv_scale) {
  for (int64_t j = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; j < n;
       j += int64_t(gridDim.x) * blockDim.x) {
    const unsigned long long q = v[j];
    reinterpret_cast<double*>(v)[j] = double(q) * inv_scale;
  }
}

__global__ void k_clear_counts(unsigned long long* a, int na, unsigned long long* b, int nb) {
  for (int i = threadIdx.x; i < na; i += blockDim.x) a[i] = 0;
  for (int i = threadIdx.x; i < nb; i += blockDim.x) b[i] = 0;
}

// row_ptr[i] = base + excl[i], i < rows; row_ptr[rows] = base + *sum; and (st_count
// given) the entries that the fullest of the staging areas was asked for
__global__ void k_rowptr_fill(const int64_t* excl, const int64_t* sum, int rows, int64_t base,
                              int64_t* row_ptr, const unsigned long long* st_count,
                              unsigned long long* most) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (st_count && i < kAreas) {  // the first wave
    unsigned long long v = st_count[i * kCountStride];
    for (int j = kWave / 2; j > 0; j >>= 1) {
      const unsigned long long o = __shfl_xor(v, j, kWave);
      v = o > v ? o : v;
    }
    if (i == 0) *most = v;
  }
  if (i < rows) row_ptr[i] = base + excl[i];
  if (i == 0) row_ptr[rows] = base + *sum;
}

// one block per piece: copy staging -> final CSR position
__global__ __launch_bounds__(256) void k_pieces_copy(const Piece* pieces, int npieces,
                                                     const int64_t* row_ptr_chunk,
                                                     const int* st_col, const float* st_val,
                                                     int* col, float* val) {
  for (int p = blockIdx.x; p < npieces; p += gridDim.x) {
    Piece pc = pieces[p];
    int64_t dst = row_ptr_chunk[pc.row] + pc.within;
    for (int k = threadIdx.x; k < pc.len; k += 256) {
      col[dst + k] = st_col[pc.src + k];
      val[dst + k] = st_val[pc.src + k];
    }
  }
}

size_t build_lds_bytes(int nrays, int pl) {
  return size_t(nrays) * (8 + size_t(pl)) * sizeof(float) +
         size_t(kCandCap) * (sizeof(int) + sizeof(float)) +
         size_t(kRowBuf) * (sizeof(int) + sizeof(float));
}

int make_build_args(const raptr_setup_t* setup, const raptr_grid_t* grid, int nrays,
                    uint32_t seed, int raygen, BuildArgs* A, size_t* lds) {
  std::memset(A, 0, sizeof(BuildArgs));
  RAPTR_TRY(make_geom(setup, grid, &A->G));
  if (nrays <= 0) return fail(RAPTR_ERR_INVALID_ARG, "nrays must be positive");
  if (raygen != RAPTR_RAYGEN_RAND && raygen != RAPTR_RAYGEN_REGU &&
      raygen != RAPTR_RAYGEN_RAND_ELEMENT)
    return fail(RAPTR_ERR_INVALID_ARG, "unknown ray generator %d", raygen);
  A->div_yz = make_fastdiv(uint32_t(grid->n[1] * grid->n[2]));
  A->div_z = make_fastdiv(uint32_t(grid->n[2]));
  A->nrays = nrays;
  A->seed = seed;
  A->raygen = raygen;
  A->pl = grid->n[0] + grid->n[1] + grid->n[2] + 3;
  uint32_t per = uint32_t(setup->n1y);
  A->div_c[3] = make_fastdiv(per);
  A->div_c[2] = make_fastdiv(per *= uint32_t(setup->n1z));
  A->div_c[1] = make_fastdiv(per *= uint32_t(setup->n0y));
  A->div_c[0] = make_fastdiv(per *= uint32_t(setup->n0z));
  A->plain_planes = true;
  for (int d = 0; d < 3; ++d) {
    A->inv_d[d] = 1.0f / grid->d[d];
    A->ext[d] = std::fabs(grid->o[d]) + float(grid->n[d]) * grid->d[d];
    A->plain_planes = A->plain_planes && plain_size(grid->o[d], 60) && plain_size(grid->d[d], 59);
  }
  // the cull's radius less half a voxel's diagonal and the rounding error of
  // its test (the cross product's terms are of the heads' distance squared)
  const float heads = std::fabs(setup->pos1x - setup->pos0x) +
                      float(setup->n0z + setup->n1z) * setup->segz +
                      float(setup->n0y + setup->n1y) * setup->segy;
  const float near = A->G.sumRadii * 0.9999f -
                     0.5f * std::sqrt(grid->d[0] * grid->d[0] + grid->d[1] * grid->d[1] +
                                      grid->d[2] * grid->d[2]) -
                     2e-6f * (heads + A->ext[0] + A->ext[1] + A->ext[2]);
  A->near2 = near > 0.0f ? near * near : 0.0f;
  A->rpb = (nrays + 31) / 32;
  *lds = build_lds_bytes(nrays, A->pl);
  if (*lds > 160 * 1024)
    return fail(RAPTR_ERR_NOT_SUPPORTED,
                "nrays=%d x planes=%d needs %zu B of LDS (> 160 KiB)", nrays, A->pl, *lds);
  return RAPTR_OK;
}

size_t rays_lds_bytes(const BuildArgs& A) {
  const size_t nsm = A.G.g.n[0] > A.G.g.n[2] ? A.G.g.n[0] : A.G.g.n[2];
  const size_t lists = 2 * size_t(kMRow), rays = 16 * size_t(A.nrays);
  return 4 * (size_t(A.nrays) * ((size_t(A.pl) + 1) | 1) + 2 * nsm * kMw + 4 * size_t(A.G.g.n[0]) +
              (lists > rays ? lists : rays));
}

template <void (*KERNEL)(BuildArgs)>
int launch_rows(const BuildArgs& A, size_t lds, hipStream_t st, int threads = kSmBlock) {
  // the kernel's dynamic-LDS limit raised on its first launch per device; not
  // fatal where the default suffices
  static std::atomic<uint64_t> raised{0};
  int dev = 0;
  RAPTR_HIP_TRY(hipGetDevice(&dev));
  const uint64_t bit = uint64_t(1) << (dev & 63);
  if (!(raised.load() & bit)) {
    if (hipFuncSetAttribute((const void*)KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize,
                            160 * 1024) != hipSuccess)
      (void)hipGetLastError();
    raised.fetch_or(bit);
  }
  // with the kernel's own arrays: a launch beyond a CU's LDS aborts the queue
  static std::atomic<int64_t> fixed{-1};
  int64_t own = fixed.load();
  if (own < 0) {
    hipFuncAttributes a;
    RAPTR_HIP_TRY(hipFuncGetAttributes(&a, (const void*)KERNEL));
    fixed.store(own = int64_t(a.sharedSizeBytes));
  }
  if (int64_t(lds) + own > 160 * 1024)
    return fail(RAPTR_ERR_NOT_SUPPORTED,
                "nrays=%d x planes=%d needs %lld B of LDS (> 160 KiB)", A.nrays, A.pl,
                (long long)(int64_t(lds) + own));
  hipLaunchKernelGGL(KERNEL, dim3(unsigned(A.rows)), dim3(threads), lds, st, A);
  RAPTR_LAUNCH_CHECK();
  return RAPTR_OK;
}

// Rays per channel and zeros dropped: k_sm_rays.  Elements with rays of their
// own have no ray to follow and a kept zero is a candidate of the cull alone:
// k_sm_build, also where the masks of a long grid do not fit LDS (its row
// buffers are smaller than they).
template <int MODE>
int launch_build(const BuildArgs& A, size_t lds, hipStream_t st) {
  const size_t lr = rays_lds_bytes(A);
  if (A.by_candidate || A.raygen == RAPTR_RAYGEN_RAND_ELEMENT || A.keep_zeros || lr > 156 * 1024 ||
      int64_t(A.G.g.n[0]) * A.G.g.n[1] >= 1 << 24)
    return launch_rows<k_sm_build<MODE>>(A, lds, st);
  // Two waves a row where the rays' tables are small, four else: a wave's
  // share of each phase must outlast the barriers.  147,456 rows of 10 rays x
  // 99 planes: 0.96 ms with two, 1.02 with four; 40,009 of 17 x 131: 1.04 and
  // 0.98; 100,003 of 30 x 159: 2.23 and 1.78 (8 waves: 2.24).
  if (A.rpb > 1) return launch_rows<k_sm_rays<MODE, false, 4>>(A, lr, st, 256);
  if (A.nrays * A.pl < 1536) return launch_rows<k_sm_rays<MODE, true, 2>>(A, lr, st, 128);
  return launch_rows<k_sm_rays<MODE, true, 4>>(A, lr, st, 256);
}

// Workspace layout of the fused build for a staging area of S entries:
// counters, staging (col, val), per-row nnz and scan, piece table, scan ws.
struct BuildLayout {
  int64_t staging, max_rows, piece_cap;
};

inline BuildLayout build_layout(int64_t S) {
  BuildLayout L;
  L.staging = S;
  L.max_rows = S / 16 + 1;
  if (L.max_rows > (1 << 20)) L.max_rows = 1 << 20;
  L.piece_cap = 2 * L.max_rows + 1024;
  return L;
}

template <class C>
void carve_build(C& c, const BuildLayout& L) {
  c.template take<unsigned long long>(4);
  c.template take<int>(size_t(L.staging));
  c.template take<float>(size_t(L.staging));
  c.template take<int>(size_t(L.max_rows));
  c.template take<int64_t>(size_t(L.max_rows));
  c.template take<char>(size_t(L.piece_cap) * 24);
  c.template take<char>(scan_workspace_bytes(L.max_rows));
}

inline size_t build_bytes(int64_t S) {
  Sizer z;
  carve_build(z, build_layout(S));
  return z.bytes();
}

}  // namespace
}  // namespace raptr

using namespace raptr;

extern "C" {

int raptr_sm_from_wq(const raptr_setup_t* setup, const raptr_grid_t* grid, const int* d_cnl,
                     const int* d_vxl, float* d_val, int64_t wq_length, int nrays,
                     uint32_t seed, int raygen, raptr_stream_t stream) {
  Geom G;
  RAPTR_TRY(make_geom(setup, grid, &G));
  if (nrays <= 0) return fail(RAPTR_ERR_INVALID_ARG, "nrays must be positive");
  if (wq_length < 0) return fail(RAPTR_ERR_INVALID_ARG, "negative length");
  if (raygen != RAPTR_RAYGEN_RAND && raygen != RAPTR_RAYGEN_REGU &&
      raygen != RAPTR_RAYGEN_RAND_ELEMENT)
    return fail(RAPTR_ERR_INVALID_ARG, "unknown ray generator %d", raygen);
  if (wq_length == 0) return RAPTR_OK;
  if (!d_cnl || !d_vxl || !d_val) return fail(RAPTR_ERR_INVALID_ARG, "null buffer");
  const int pl = grid->n[0] + grid->n[1] + grid->n[2] + 3, stride = (pl + 1) | 1;
  const size_t lds = size_t(nrays) * (8 + size_t(stride)) * sizeof(float);
  const int64_t chunks = (wq_length + kWqChunk - 1) / kWqChunk;
  const int max_runs = wq_max_runs(wq_length, nrays, pl);
  // rays per channel whose tables leave a CU two workgroups or more
  if (raygen != RAPTR_RAYGEN_RAND_ELEMENT && lds <= 64 * 1024 && chunks < (1 << 22) &&
      max_runs > 0) {
    hipLaunchKernelGGL(k_sm_from_wq_runs, dim3(unsigned(chunks)), dim3(256), lds, S(stream), G,
                       d_cnl, d_vxl, d_val, wq_length, nrays, seed, raygen, max_runs, stride,
                       make_fastdiv(uint32_t(grid->n[1] * grid->n[2])),
                       make_fastdiv(uint32_t(grid->n[2])));
    RAPTR_LAUNCH_CHECK();
    return RAPTR_OK;
  }
  hipLaunchKernelGGL(k_sm_from_wq, dim3(grid_for(wq_length, 256, 1 << 16)), dim3(256), 0,
                     S(stream), G, d_cnl, d_vxl, d_val, wq_length, nrays, seed, raygen);
  RAPTR_LAUNCH_CHECK();
  return RAPTR_OK;
}

int raptr_generate_rays(const raptr_setup_t* setup, const int* d_cnl, int n_cnl, int nrays,
                        uint32_t seed, int raygen, float* d_rays, raptr_stream_t stream) {
  raptr_grid_t g = {{0, 0, 0}, {1, 1, 1}, {1, 1, 1}};
  Geom G;
  RAPTR_TRY(make_geom(setup, &g, &G));
  if (raygen != RAPTR_RAYGEN_RAND && raygen != RAPTR_RAYGEN_REGU)
    return fail(RAPTR_ERR_INVALID_ARG, "ray listings take RAND or REGU (got %d)", raygen);
  if (n_cnl <= 0 || nrays <= 0) return RAPTR_OK;
  hipLaunchKernelGGL(k_generate_rays, dim3(grid_for(int64_t(n_cnl) * nrays, 256, 1 << 16)),
                     dim3(256), 0, S(stream), G, d_cnl, n_cnl, nrays, seed, raygen, d_rays);
  RAPTR_LAUNCH_CHECK();
  return RAPTR_OK;
}

size_t raptr_sm_build_workspace_size(const raptr_grid_t* grid, int nrays,
                                     int64_t staging_entries) {
  (void)grid;
  (void)nrays;
  if (staging_entries < kRowBuf) staging_entries = kRowBuf;
  return build_bytes(staging_entries);
}

int raptr_sm_build_csr(const raptr_setup_t* setup, const raptr_grid_t* grid,
                       const int* d_list, int list_size, int nrays, uint32_t seed,
                       int raygen, int64_t* d_row_ptr, int* d_col, float* d_val,
                       int64_t capacity, int64_t* nnz, void* d_ws, size_t ws_bytes,
                       raptr_stream_t stream) {
  return raptr_sm_build_csr_ex(setup, grid, d_list, list_size, nrays, seed, raygen, 0,
                               d_row_ptr, d_col, d_val, capacity, nnz, d_ws, ws_bytes,
                               stream);
}

int raptr_sm_build_csr_ex(const raptr_setup_t* setup, const raptr_grid_t* grid,
                          const int* d_list, int list_size, int nrays, uint32_t seed,
                          int raygen, int flags, int64_t* d_row_ptr, int* d_col, float* d_val,
                          int64_t capacity, int64_t* nnz, void* d_ws, size_t ws_bytes,
                          raptr_stream_t stream) {
  if (!nnz || !d_row_ptr) return fail(RAPTR_ERR_INVALID_ARG, "null output");
  *nnz = 0;
  if (list_size < 0 || (list_size > 0 && !d_list))
    return fail(RAPTR_ERR_INVALID_ARG, "bad list");
  if (flags & ~int(RAPTR_SM_KEEP_ZEROS))
    return fail(RAPTR_ERR_INVALID_ARG, "unknown build flags 0x%x", flags);
  BuildArgs A;
  size_t lds = 0;
  RAPTR_TRY(make_build_args(setup, grid, nrays, seed, raygen, &A, &lds));
  A.keep_zeros = (flags & RAPTR_SM_KEEP_ZEROS) ? 1 : 0;
  hipStream_t st = S(stream);
  const bool fill = d_col != nullptr;
  if (fill && !d_val) return fail(RAPTR_ERR_INVALID_ARG, "null values");
  // largest staging area whose layout fits the workspace
  int64_t lo = 0, hi = int64_t(ws_bytes / 8) + 1;
  while (lo + 1 < hi) {
    int64_t mid = lo + (hi - lo) / 2;
    if (build_bytes(mid) <= ws_bytes) lo = mid; else hi = mid;
  }
  if (lo < kRowBuf || !d_ws)
    return fail(RAPTR_ERR_WORKSPACE, "sm_build workspace too small (%zu B)", ws_bytes);
  BuildLayout L = build_layout(lo);
  Carver cv(d_ws, ws_bytes);
  unsigned long long* counters = cv.take<unsigned long long>(4);
  int* st_col = cv.take<int>(size_t(L.staging));
  float* st_val = cv.take<float>(size_t(L.staging));
  int* row_nnz = cv.take<int>(size_t(L.max_rows));
  int64_t* excl = cv.take<int64_t>(size_t(L.max_rows));
  Piece* pieces = reinterpret_cast<Piece*>(cv.take<char>(size_t(L.piece_cap) * 24));
  size_t sb = scan_workspace_bytes(L.max_rows);
  void* scan_ws = cv.take<char>(sb);
  if (!cv.ok) return fail(RAPTR_ERR_WORKSPACE, "sm_build workspace carve failed");
  const int64_t staging = L.staging, max_rows = L.max_rows;
  A.list = d_list;
  A.row_nnz = row_nnz;
  A.st_col = st_col;
  A.st_val = st_val;
  A.piece_count = reinterpret_cast<unsigned*>(&counters[0]);
  A.flags = reinterpret_cast<unsigned*>(&counters[1]);
  A.pieces = pieces;
  // the staging areas' counters: the end of the piece table, from a line on
  const size_t area_at =
      (size_t(L.piece_cap) * 24 - kAreas * kCountStride * sizeof(unsigned long long)) & ~size_t(127);
  unsigned long long* area_counts =
      reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(pieces) + area_at);
  A.piece_cap = int(area_at / sizeof(Piece));

  int64_t total = 0;
  int first = 0;
  // the first chunk measures the density: rows of up to 4,096 entries fit
  int64_t rows0 = staging >> 12;
  if (rows0 < 64) rows0 = 64;
  if (rows0 > max_rows) rows0 = max_rows;
  int rows = int(rows0 < list_size ? rows0 : list_size);
  while (first < list_size) {
    if (rows > list_size - first) rows = list_size - first;
    A.first = first;
    A.rows = rows;
    // few rows may fill the staging unevenly: one area
    A.areas = rows >= kAreas * kCountStride ? kAreas : 1;
    A.st_cap = staging / A.areas;
    A.st_count = A.areas > 1 ? area_counts : &counters[3];
    hipLaunchKernelGGL(k_clear_counts, dim3(1), dim3(256), 0, st, counters, 4, A.st_count,
                       A.areas > 1 ? kAreas * kCountStride : 0);
    RAPTR_LAUNCH_CHECK();
    if (fill)
      RAPTR_TRY(launch_build<kModeFill>(A, lds, st));
    else
      RAPTR_TRY(launch_build<kModeCount>(A, lds, st));
    RAPTR_TRY(scan_exclusive_i32_i64(row_nnz, excl, rows, reinterpret_cast<int64_t*>(&counters[2]),
                                     scan_ws, sb, st));
    hipLaunchKernelGGL(k_rowptr_fill, dim3(grid_for(rows, 256)), dim3(256), 0, st,
                       (const int64_t*)excl, (const int64_t*)&counters[2], rows, total,
                       d_row_ptr + first,
                       A.areas > 1 ? (const unsigned long long*)area_counts : nullptr, &counters[3]);
    RAPTR_LAUNCH_CHECK();
    unsigned long long hc[4];
    RAPTR_HIP_TRY(hipMemcpyAsync(hc, counters, sizeof(hc), hipMemcpyDeviceToHost, st));
    RAPTR_HIP_TRY(hipStreamSynchronize(st));
    if (unsigned(hc[1] & 0xffffffffu)) {
      if (rows == 1) {
        // k_sm_rays asks for room for its rectangles, k_sm_build for entries
        if (A.by_candidate)
          return fail(RAPTR_ERR_WORKSPACE, "row %d does not fit the staging area", first);
        A.by_candidate = 1;
        continue;
      }
      // the rows that would have fitted at what these asked for (of pieces: half)
      const double fit = hc[3] > uint64_t(A.st_cap) ? 0.9 * double(A.st_cap) / double(hc[3]) : 0.5;
      rows = std::max(1, std::min(rows - 1, int(rows * fit)));
      continue;
    }
    A.by_candidate = 0;
    const int64_t chunk_nnz = int64_t(hc[2]);
    if (fill) {
      if (total + chunk_nnz > capacity)
        return fail(RAPTR_ERR_WORKSPACE, "matrix exceeds capacity %lld after row %d",
                    (long long)capacity, first + rows);
      const unsigned np = unsigned(rows) + unsigned(hc[0] & 0xffffffffu);
      hipLaunchKernelGGL(k_pieces_copy, dim3(np < 65536 ? np : 65536), dim3(256), 0, st,
                         (const Piece*)pieces, int(np), (const int64_t*)(d_row_ptr + first),
                         (const int*)st_col, (const float*)st_val, d_col, d_val);
      RAPTR_LAUNCH_CHECK();
    }
    total += chunk_nnz;
    first += rows;
    // next chunk: 0.6 of the staging at these rows' entries, and at most 0.8 of it
    // at what they asked for (k_sm_rays asks for a fourth to twice more than they)
    const double per = std::max(double(chunk_nnz) / 0.6,
                                fill ? double(hc[3]) * A.areas / 0.8 : 0.0);
    int64_t want = per > 0 ? int64_t(double(staging) * rows / per) : max_rows;
    if (want > max_rows) want = max_rows;
    if (want < 1) want = 1;
    rows = int(want);
  }
  if (list_size == 0) {
    const int64_t zero = 0;
    RAPTR_HIP_TRY(hipMemcpyAsync(d_row_ptr, &zero, sizeof(int64_t), hipMemcpyHostToDevice, st));
  }
  RAPTR_HIP_TRY(hipStreamSynchronize(st));
  *nnz = total;
  return RAPTR_OK;
}

int raptr_sm_build_csr_noalloc(const raptr_setup_t* setup, const raptr_grid_t* grid,
                               const int* d_list, int list_size, int nrays, uint32_t seed,
                               int raygen, int flags, int64_t* d_row_ptr, int* d_col,
                               float* d_val, int64_t capacity, int64_t* nnz,
                               raptr_stream_t stream) {
  void* ws = nullptr;
  RAPTR_TRY(scratch_address(&ws));
  const int st = raptr_sm_build_csr_ex(setup, grid, d_list, list_size, nrays, seed, raygen,
                                       flags, d_row_ptr, d_col, d_val, capacity, nnz, ws,
                                       kNoAllocScratchBytes, stream);
  if (st == RAPTR_ERR_WORKSPACE && std::strstr(raptr_last_error(), "staging")) {
    char why[256];
    std::snprintf(why, sizeof(why), "%s", raptr_last_error());  // fail() rewrites it
    return fail(RAPTR_ERR_WORKSPACE,
                "raptr_sm_build_csr_noalloc: a row has more candidates than the %zu-byte "
                "scratch stages (%s)",
                kNoAllocScratchBytes, why);
  }
  return st;
}

int raptr_sensitivity_f64(const raptr_setup_t* setup, const raptr_grid_t* grid, int nrays,
                          uint32_t seed, int raygen, double* d_sens, raptr_stream_t stream) {
  BuildArgs A;
  size_t lds = 0;
  RAPTR_TRY(make_build_args(setup, grid, nrays, seed, raygen, &A, &lds));
  if (!d_sens) return fail(RAPTR_ERR_INVALID_ARG, "null output");
  hipStream_t st = S(stream);
  RAPTR_HIP_TRY(hipMemsetAsync(d_sens, 0, size_t(A.G.nvox) * sizeof(double), st));
  int64_t nch = int64_t(setup->na) * setup->n0z * setup->n0y * setup->n1z * setup->n1y;
  // Fixed point with `bits` fraction bits: no column sum exceeds (channels)
  // x (voxel diagonal, the longest mean chord), so 2^bits times that bound
  // stays below 2^62.  A float value of at least 2^(23 - bits) is a whole
  // multiple of 2^-bits (exact); smaller ones are rounded by at most
  // 2^-(bits + 1).  The integer sums are the same whatever the order of the
  // additions, so the sensitivity is reproducible bit for bit.
  const double diag = std::sqrt(double(grid->d[0]) * grid->d[0] +
                                double(grid->d[1]) * grid->d[1] +
                                double(grid->d[2]) * grid->d[2]);
  const double bound = double(nch > 0 ? nch : 1) * (diag > 0.0 ? diag : 1.0);
  int bits = int(std::floor(62.0 - std::log2(bound)));
  if (bits > 52) bits = 52;
  if (bits < 8)
    return fail(RAPTR_ERR_NOT_SUPPORTED, "sensitivity bound %.3g too large for fixed point",
                bound);
  A.list = nullptr;
  A.wgt = nullptr;
  A.colsum = d_sens;
  A.colsum_fx = reinterpret_cast<unsigned long long*>(d_sens);
  A.fx_scale = std::ldexp(1.0, bits);
  const int64_t kRowsPerLaunch = 1 << 20;
  for (int64_t f = 0; f < nch; f += kRowsPerLaunch) {
    A.first = int(f);
    A.rows = int(nch - f < kRowsPerLaunch ? nch - f : kRowsPerLaunch);
    RAPTR_TRY(launch_build<kModeColsum>(A, lds, st));
  }
  hipLaunchKernelGGL(k_fx_to_f64, dim3(grid_for(A.G.nvox, 256)), dim3(256), 0, st,
                     A.colsum_fx, A.G.nvox, std::ldexp(1.0, -bits));
  RAPTR_LAUNCH_CHECK();
  return RAPTR_OK;
}

int raptr_backproject_f64(const raptr_setup_t* setup, const raptr_grid_t* grid,
                          const int* d_list, const float* d_weights, int list_size, int nrays,
                          uint32_t seed, int raygen, double* d_out, raptr_stream_t stream) {
  BuildArgs A;
  size_t lds = 0;
  RAPTR_TRY(make_build_args(setup, grid, nrays, seed, raygen, &A, &lds));
  if (!d_out || list_size < 0 || (list_size > 0 && (!d_list || !d_weights)))
    return fail(RAPTR_ERR_INVALID_ARG, "bad back-projection arguments");
  hipStream_t st = S(stream);
  RAPTR_HIP_TRY(hipMemsetAsync(d_out, 0, size_t(A.G.nvox) * sizeof(double), st));
  A.list = d_list;
  A.wgt = d_weights;
  A.colsum = d_out;
  const int64_t kRowsPerLaunch = 1 << 20;
  for (int64_t f = 0; f < list_size; f += kRowsPerLaunch) {
    A.first = int(f);
    A.rows = int(list_size - f < kRowsPerLaunch ? list_size - f : kRowsPerLaunch);
    RAPTR_TRY(launch_build<kModeColsum>(A, lds, st));
  }
  return RAPTR_OK;
}

int raptr_forward_project_f64(const raptr_setup_t* setup, const raptr_grid_t* grid,
                              const int* d_list, int list_size, int nrays, uint32_t seed,
                              int raygen, const float* d_x, double* d_out,
                              raptr_stream_t stream) {
  BuildArgs A;
  size_t lds = 0;
  RAPTR_TRY(make_build_args(setup, grid, nrays, seed, raygen, &A, &lds));
  if (!d_x || !d_out) return fail(RAPTR_ERR_INVALID_ARG, "null buffer");
  int64_t nch = int64_t(setup->na) * setup->n0z * setup->n0y * setup->n1z * setup->n1y;
  int64_t rows = d_list ? int64_t(list_size) : nch;
  if (rows < 0) return fail(RAPTR_ERR_INVALID_ARG, "negative list size");
  A.list = d_list;
  A.xin = d_x;
  A.fwd = d_out;
  const int64_t kRowsPerLaunch = 1 << 20;
  for (int64_t f = 0; f < rows; f += kRowsPerLaunch) {
    A.first = int(f);
    A.rows = int(rows - f < kRowsPerLaunch ? rows - f : kRowsPerLaunch);
    RAPTR_TRY(launch_build<kModeFwd>(A, lds, S(stream)));
  }
  return RAPTR_OK;
}

}  // extern "C"
