// Neighbour search on gfx950: counting-sort cell binning, a wavefront-scan
// prefix sum, per-cell id sort, and the exact float32 pair predicate.
//
// Replaces (all XLA-generated in the reference):
//   jax_md/partition.py:294-413   cell_list_fn (hash, argsort, slot scatter, occupancy)
//   jax_md/partition.py:832-909   3^d candidate copies + prune + cumsum compaction
//   jax_md/partition.py:956-976   capacity and NEIGHBOR_LIST_OVERFLOW
//   jax_md/partition.py:1010-1018 rebuild test of update
//   jax_sph/partition.py:208-291  jaxmd_scan chunk budgets
#include <hip/hip_runtime.h>

#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "ens.h"
#include "sph_device.h"
#include "sph_internal.h"
#include "sweep.h"
#include "tile_band.h"

namespace sph {

constexpr int kBlock = 256;

__host__ __device__ inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ------------------------------------------------------------------ helpers
template <typename T>
__global__ void k_fill(T* __restrict__ a, int64_t n, T v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

static hipError_t clear_counts(int32_t* count, int64_t ncell, bool* dirty, hipStream_t st) {
  if (!*dirty) return hipSuccess;
  k_fill<int32_t><<<cdiv(ncell, kBlock), kBlock, 0, st>>>(count, ncell, 0);
  const hipError_t e = hipGetLastError();
  *dirty = e != hipSuccess;
  return e;
}

int clean_histograms(sph_ws* ws, hipStream_t st) {
  hipError_t e = clear_counts(ws->cell_count, ws->ncell, &ws->count_dirty, st);
  if (e == hipSuccess) e = clear_counts(ws->sk.cell_count, ws->sk.ncell, &ws->sk.count_dirty, st);
  return e == hipSuccess ? SPH_OK : hip_fail(e, "clean_histograms");
}

HistogramGuard::~HistogramGuard() {
  (void)clear_counts(ws->cell_count, ws->ncell, &ws->count_dirty, s);
  (void)clear_counts(ws->sk.cell_count, ws->sk.ncell, &ws->sk.count_dirty, s);
}

struct Grid {
  float cs[3];   // cell size (fp32)
  int cps[3];    // cells per side
  int use_cells;
};

void cut_band(const sph_nl_config& c, float* lo, float* hi);

// int32(r / cell_size) per dimension (partition.py:367), clamped into the grid:
// the reference aliases r == side into a wrong cell; clamping keeps it in the last one.
template <int DIM>
__device__ __forceinline__ void cell_coords(const float4 p, const Grid& g, int* c) {
  float x[3] = {p.x, p.y, p.z};
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    // fl32(x / cs), correctly rounded: a float64 quotient rounded to float32 is
    // the correctly rounded float32 quotient (53 >= 2*24 + 2 bits)
    int q = (int)(float)((double)x[d] / (double)g.cs[d]);
    q = q < 0 ? 0 : q;
    q = q >= g.cps[d] ? g.cps[d] - 1 : q;
    c[d] = q;
  }
}

template <int DIM>
__device__ __forceinline__ int cell_hash(const int* c, const Grid& g) {
  int h = c[0] + c[1] * g.cps[0];
  if (DIM == 3) h += c[2] * g.cps[0] * g.cps[1];
  return h;
}

template <int DIM>
__device__ __forceinline__ float4 load_pos(const float* __restrict__ r, int64_t i) {
  float4 p;
  p.x = r[i * DIM + 0];
  p.y = r[i * DIM + 1];
  p.z = DIM == 3 ? r[i * DIM + 2] : 0.0f;
  p.w = 0.0f;
  return p;
}

// ----------------------------------------------------------- binning kernels
// The runs of equal keys in consecutive lanes (particles in id order come in
// runs of one cell): the lanes that start one, and from a starting lane the
// length of its run.  The active lanes must be a prefix of the wavefront.
__device__ __forceinline__ unsigned long long run_starts(int key) {
  const int prev = __shfl_up(key, 1, 64);
  return __ballot((threadIdx.x & 63) == 0 || prev != key);
}
__device__ __forceinline__ int run_length(unsigned long long starts) {
  const int lane = threadIdx.x & 63;
  const unsigned long long active = __ballot(1);
  const unsigned long long later = lane == 63 ? 0ull : (starts >> (lane + 1)) << (lane + 1);
  const int end = later ? __ffsll((long long)later) - 1 : 64 - __clzll((long long)active);
  return end - lane;
}

// atomicAdd(&counter[key], 1) for every active lane, with one atomic per run,
// issued by all runs at once.  Returns nothing: the counts only.
__device__ __forceinline__ void wave_run_inc(int32_t* __restrict__ counter, int key) {
  const unsigned long long starts = run_starts(key);
  const int len = run_length(starts);
  if ((starts >> (threadIdx.x & 63)) & 1ull) atomicAdd(&counter[key], len);
}

// The same, returning the lane's slot.  Bound by the latency of one returning
// atomic: all runs of the wavefront wait for theirs together.  Taking the
// wavefront's distinct keys in turn (one atomic each, in order) waited for some
// 20 of them one after another in 3D: hash of a 45^3 list 22.8 us, now 5.1 us;
// drift and hash of a 24,458-particle 2D step 18.5 us, now 3.4 us.  A key that
// comes in several runs costs one atomic a run, all in flight together.
__device__ __forceinline__ int wave_run_slot(int32_t* __restrict__ counter, int key) {
  const int lane = threadIdx.x & 63;
  const unsigned long long starts = run_starts(key);
  const int len = run_length(starts);
  int base = 0;
  if ((starts >> lane) & 1ull) base = atomicAdd(&counter[key], len);
  const int first = 63 - __clzll((long long)(starts & ((2ull << lane) - 1ull)));
  return __shfl(base, first, 64) + lane - first;
}

// Start of a build: the bits of the list before (sticky), the rest zero.
__device__ __forceinline__ void reset_info(int64_t* __restrict__ info,
                                           const int64_t* __restrict__ prev) {
  info[0] = prev ? prev[0] : 0;
  for (int k = 1; k < 8; ++k) info[k] = 0;
}

template <int DIM>
__device__ __forceinline__ void hash_count_body(const float* __restrict__ r, int n, const Grid& g,
                                                int32_t* __restrict__ cell_count,
                                                int32_t* __restrict__ pcell,
                                                int32_t* __restrict__ pslot,
                                                const int32_t* __restrict__ gate, int blk) {
  if (gate && *gate == 0) return;
  int i = blk * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int h = 0;
  if (g.use_cells) {
    int c[3];
    cell_coords<DIM>(load_pos<DIM>(r, i), g, c);
    h = cell_hash<DIM>(c, g);
  }
  if (!pcell) {
    wave_run_inc(cell_count, h);
    return;
  }
  pcell[i] = h;
  pslot[i] = wave_run_slot(cell_count, h);
}

template <int DIM>
__global__ void k_hash_count(const float* __restrict__ r, int n, Grid g,
                             int32_t* __restrict__ cell_count, int32_t* __restrict__ pcell,
                             int32_t* __restrict__ pslot, const int32_t* __restrict__ gate,
                             int64_t* __restrict__ info = nullptr,
                             const int64_t* __restrict__ prev = nullptr) {
  if (info && blockIdx.x == 0 && threadIdx.x == 0) reset_info(info, prev);
  hash_count_body<DIM>(r, n, g, cell_count, pcell, pslot, gate, blockIdx.x);
}

// si_euler kick + transport velocity + drift + periodic wrap (integrator.py:26-30)
// of block blk's particles; x receives the new position of the thread's own.
// Returns its index, n or more where the thread has none.
template <int DIM>
__device__ __forceinline__ int integrate_block(
    const float* __restrict__ r, const float* __restrict__ u, const float* __restrict__ dudt,
    const float* __restrict__ dvdt, float* __restrict__ r_out, float* __restrict__ u_out,
    float* __restrict__ v_out, int n, float dt, float ctvf, const float* side, int blk, float* x) {
#pragma clang fp contract(off)
  int i;
  if constexpr (DIM == 3) {
    // The block's 3 x kBlock floats of each array pass through LDS, so every
    // wave-wide load and store covers 64 consecutive floats; per-particle
    // stride-3 accesses touch three times as many cache lines per instruction.
    // Every block of a launch starts below n (launches use cdiv(n, kBlock)
    // blocks), and every thread reaches the barriers.
    __shared__ float s[4][3 * kBlock];
    const int i0 = blk * kBlock;
    i = i0 + threadIdx.x;
    const int64_t base = (int64_t)i0 * 3;
    const int lim = 3 * min(kBlock, n - i0);
    for (int k = threadIdx.x; k < lim; k += kBlock) {
      s[0][k] = r[base + k];
      s[1][k] = u[base + k];
      s[2][k] = dudt[base + k];
      s[3][k] = dvdt[base + k];
    }
    __syncthreads();
    float uo[3], vo[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int k = 3 * threadIdx.x + d;
      uo[d] = s[1][k] + dt * s[2][k];
      vo[d] = uo[d] + ctvf * s[3][k];
      float xx = s[0][k] + dt * vo[d];
      if (xx >= side[d] || xx < 0.0f) xx = jmod(xx, side[d]);
      x[d] = xx;
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int k = 3 * threadIdx.x + d;
      s[0][k] = x[d];
      s[1][k] = uo[d];
      s[2][k] = vo[d];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < lim; k += kBlock) {
      r_out[base + k] = s[0][k];
      u_out[base + k] = s[1][k];
      v_out[base + k] = s[2][k];
    }
  } else {
    i = blk * blockDim.x + threadIdx.x;
    if (i >= n) return i;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const int64_t k = (int64_t)i * DIM + d;
      const float uu = u[k] + dt * dudt[k];
      const float vv = uu + ctvf * dvdt[k];
      float xx = r[k] + dt * vv;
      if (xx >= side[d] || xx < 0.0f) xx = jmod(xx, side[d]);
      u_out[k] = uu;
      v_out[k] = vv;
      r_out[k] = xx;
      x[d] = xx;
    }
  }
  return i;
}

// integrate_block fused with the cell hash and histogram of the new position
// (HASH = false: the drift alone, for sets that k_bin_small bins).
template <int DIM, bool HASH>
__global__ __launch_bounds__(kBlock) void k_integrate_hash(
    const float* __restrict__ r, const float* __restrict__ u, const float* __restrict__ dudt,
    const float* __restrict__ dvdt, float* __restrict__ r_out, float* __restrict__ u_out,
    float* __restrict__ v_out, int n, float dt, float ctvf, Grid g, float bx, float by, float bz,
    int32_t* __restrict__ cell_count, int32_t* __restrict__ pcell, int32_t* __restrict__ pslot,
    int64_t* __restrict__ info, const int64_t* __restrict__ prev) {
  if (HASH && blockIdx.x == 0 && threadIdx.x == 0) reset_info(info, prev);
  const float side[3] = {bx, by, bz};
  float x[3] = {0.f, 0.f, 0.f};
  const int i = integrate_block<DIM>(r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, side,
                                     blockIdx.x, x);
  if (!HASH || i >= n) return;
  int h = 0;
  if (g.use_cells) {
    int c[3];
    cell_coords<DIM>(make_float4(x[0], x[1], x[2], 0.0f), g, c);
    h = cell_hash<DIM>(c, g);
  }
  pcell[i] = h;
  pslot[i] = wave_run_slot(cell_count, h);
}

// Skin-list step: integrate_block, the histogram of the new positions on the
// reference grid (for its cell-capacity bit), and the rebuild test: a particle
// that moved more than the trigger distance since the last build (minimum
// image) raises *flag.
template <int DIM>
__device__ __forceinline__ void integrate_skin_body(
    const float* __restrict__ r, const float* __restrict__ u, const float* __restrict__ dudt,
    const float* __restrict__ dvdt, float* __restrict__ r_out, float* __restrict__ u_out,
    float* __restrict__ v_out, int n, float dt, float ctvf, const Grid& g, float bx, float by,
    float bz, int32_t* __restrict__ cell_count, const float4* __restrict__ posb, float trigger_sq,
    int32_t* __restrict__ flag, int blk) {
#pragma clang fp contract(off)
  const float side[3] = {bx, by, bz};
  float x[3] = {0.f, 0.f, 0.f};
  const int i = integrate_block<DIM>(r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, side,
                                     blk, x);
  if (i >= n) return;
  int c[3];
  cell_coords<DIM>(make_float4(x[0], x[1], x[2], 0.0f), g, c);
  wave_run_inc(cell_count, cell_hash<DIM>(c, g));
  const float4 b = posb[i];
  const float pb[3] = {b.x, b.y, b.z};
  float m2 = 0.0f;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const float dd = disp_fast(x[d], pb[d], side[d], 1.0f / side[d]);
    m2 += dd * dd;
  }
  if (m2 > trigger_sq) *flag = 1;  // same value from every writer
}

template <int DIM>
__global__ void k_integrate_skin(const float* __restrict__ r, const float* __restrict__ u,
                                 const float* __restrict__ dudt, const float* __restrict__ dvdt,
                                 float* __restrict__ r_out, float* __restrict__ u_out,
                                 float* __restrict__ v_out, int n, float dt, float ctvf, Grid g,
                                 float bx, float by, float bz, int32_t* __restrict__ cell_count,
                                 const float4* __restrict__ posb, float trigger_sq,
                                 int32_t* __restrict__ flag, int64_t* __restrict__ info,
                                 const int64_t* __restrict__ prev) {
  if (blockIdx.x == 0 && threadIdx.x == 0) reset_info(info, prev);
  integrate_skin_body<DIM>(r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, g, bx, by, bz,
                           cell_count, posb, trigger_sq, flag, blockIdx.x);
}

// Ensembles: largest reference-grid cell occupancy of this step (one workgroup
// a member): sets info[2] and the cell-capacity bit, resets the other info entries (keeping
// the sticky bits of prev[0]) and clears the histogram for the next step.
constexpr int kCellsThreads = 1024;
__device__ __forceinline__ void cells_max_body(int32_t* __restrict__ count, int64_t ncell,
                                               int64_t* __restrict__ info,
                                               const int64_t* __restrict__ prev,
                                               int64_t capacity) {
  __shared__ int wm[kCellsThreads / 64];
  int m = 0;
  for (int64_t i = threadIdx.x; i < ncell; i += kCellsThreads) {
    const int c = count[i];
    m = c > m ? c : m;
    count[i] = 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int y = __shfl_down(m, o, 64);
    m = y > m ? y : m;
  }
  if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    int mm = 0;
    for (int w = 0; w < kCellsThreads / 64; ++w) mm = wm[w] > mm ? wm[w] : mm;
    int64_t bits = prev ? prev[0] : 0;
    if (capacity >= 0 && mm > capacity) bits |= SPH_CELL_LIST_OVERFLOW;
    info[0] = bits;
    for (int k = 1; k < 8; ++k) info[k] = 0;
    info[2] = mm;
  }
}

__global__ void k_max_reduce(const int32_t* __restrict__ a, int64_t n, int64_t* __restrict__ out) {
  int m = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    m = a[i] > m ? a[i] : m;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    int y = __shfl_down(m, o, 64);
    m = y > m ? y : m;
  }
  if ((threadIdx.x & 63) == 0) atomicMax((unsigned long long*)out, (unsigned long long)m);
}

// Exclusive scan: out[k] = sum(in[0:k]) for k in [0, n]; also the largest entry
// (for the cell capacity).  Each workgroup scans `chunk` entries (a multiple of
// kScanTile), four a thread and tile.  What precedes its chunk it adds up
// itself: from the entries (they are in the L2 and no workgroup waits for
// another) or, on long inputs, from the sums of the earlier chunks (SUMS).
constexpr int kScanThreads = 1024;
constexpr int kScanTile = 4 * kScanThreads;
constexpr int kScanSums = 1024;  // chunk sums at most (sph_ws::scan_tmp)

struct ScanPlan {
  int64_t chunk;
  int blocks;
  bool sums;
};
// Adding up the entries costs a workgroup a load a thread for every chunk
// before its own: 7.4 us for 30,300 entries (8 chunks; one workgroup, tile
// after tile, took 37.5 us) and 15.8 us for 129,600 (32 chunks).  With the sums
// both take 5.4 us, after another launch of 2.8 us and its gap: beyond 16
// chunks that is the cheaper one.
static ScanPlan scan_plan(int64_t n, bool have_sums) {
  const int64_t tiles = n > 0 ? cdiv(n, kScanTile) : 1;
  ScanPlan p;
  p.chunk = kScanTile * cdiv(tiles, kScanSums);
  p.blocks = (int)(n > 0 ? cdiv(n, p.chunk) : 1);
  p.sums = have_sums && p.blocks > 16;
  return p;
}

template <typename TIn>
__device__ __forceinline__ void load4(const TIn* __restrict__ in, int64_t i, int64_t n, bool wide,
                                      TIn* v) {
  if (wide && i + 3 < n) {
    const int4 q = *(const int4*)(in + i);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = i + k < n ? in[i + k] : (TIn)0;
  }
}

// Sum over the workgroup, the same in every thread.
template <typename T>
__device__ __forceinline__ T block_sum(T x, T* part) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  __syncthreads();  // part may still be read from an earlier use
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = x;
  __syncthreads();
  T t = 0;
#pragma unroll
  for (int w = 0; w < kScanThreads / 64; ++w) t += part[w];
  return t;
}

template <typename TOut>
__global__ __launch_bounds__(kScanThreads) void k_chunk_sums(const int32_t* __restrict__ in,
                                                             int64_t n, int64_t chunk,
                                                             TOut* __restrict__ sums) {
  __shared__ TOut part[kScanThreads / 64];
  const int64_t lo = blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
  const bool wide = ((uintptr_t)in & 15) == 0;
  TOut s = 0;
  for (int64_t i = lo + 4 * threadIdx.x; i < hi; i += kScanTile) {
    int32_t v[4];
    load4(in, i, n, wide, v);
    s += (TOut)v[0] + v[1] + v[2] + v[3];
  }
  s = block_sum(s, part);
  if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

// blk, nblk: the workgroup's chunk and the chunks of this input.  With a gate,
// runs only when *gate != 0; info (or null) receives the largest entry in
// info[2] (zeroed before) and the cell-capacity bit.
template <typename TOut>
__device__ __forceinline__ void scan_body(const int32_t* __restrict__ in, int64_t n, int64_t chunk,
                                          const TOut* __restrict__ sums, TOut* __restrict__ out,
                                          int64_t* __restrict__ info, int64_t capacity,
                                          const int32_t* __restrict__ gate, int blk, int nblk) {
  __shared__ TOut part[kScanThreads / 64];
  __shared__ int wmax[kScanThreads / 64];
  if (gate && *gate == 0) return;  // uniform
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const bool wide = ((uintptr_t)in & 15) == 0;
  const int64_t lo = blk * chunk, hi = lo + chunk < n ? lo + chunk : n;
  TOut before = 0;
  if (sums) {
    for (int k = t; k < blk; k += kScanThreads) before += sums[k];
  } else {
    for (int64_t i = 4 * t; i < lo; i += kScanTile) {
      int32_t v[4];
      load4(in, i, n, wide, v);
      before += (TOut)v[0] + v[1] + v[2] + v[3];
    }
  }
  TOut carry = blk > 0 ? block_sum(before, part) : (TOut)0;
  int mx = 0;
  for (int64_t base = lo; base < hi; base += kScanTile) {
    const int64_t i0 = base + 4 * t;
    int32_t v[4];
    load4(in, i0, n, wide, v);
    const TOut s = (TOut)v[0] + v[1] + v[2] + v[3];
    mx = max(max(mx, max(v[0], v[1])), max(v[2], v[3]));
    TOut inc = s;  // inclusive scan over the wavefront
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const TOut y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    __syncthreads();  // part of the tile before is no longer read
    if (lane == 63) part[wid] = inc;
    __syncthreads();
    TOut run = carry + inc - s;
    TOut tile = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
      const TOut x = part[w];
      if (w < wid) run += x;
      tile += x;
    }
    carry += tile;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (i0 + k < n) out[i0 + k] = run;
      run += v[k];
    }
  }
  if (t == 0 && blk == nblk - 1) out[n] = carry;
  if (!info) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = max(mx, __shfl_down(mx, o, 64));
  if (lane == 0) wmax[wid] = mx;
  __syncthreads();
  if (t == 0) {
    int m = 0;
    for (int w = 0; w < kScanThreads / 64; ++w) m = max(m, wmax[w]);
    atomicMax((unsigned long long*)&info[2], (unsigned long long)m);
    if (capacity >= 0 && m > capacity)
      atomicOr((unsigned long long*)&info[0], (unsigned long long)SPH_CELL_LIST_OVERFLOW);
  }
}

template <typename TOut>
__global__ __launch_bounds__(kScanThreads) void k_scan(
    const int32_t* __restrict__ in, int64_t n, int64_t chunk, const TOut* __restrict__ sums,
    TOut* __restrict__ out, int64_t* __restrict__ info, int64_t capacity,
    const int32_t* __restrict__ gate) {
  scan_body<TOut>(in, n, chunk, sums, out, info, capacity, gate, blockIdx.x, gridDim.x);
}

// Scans in[0:n] into out[0:n + 1]; scratch (or null) holds kScanSums sums.
template <typename TOut>
static int scan(sph_ws* ws, const char* name, const int32_t* in, int64_t n, TOut* out,
                TOut* scratch, int64_t* info, int64_t capacity, const int32_t* gate,
                hipStream_t st) {
  const ScanPlan p = scan_plan(n, scratch != nullptr);
  if (p.sums)
    SPH_LAUNCH(ws, "scan_sums", st,
               k_chunk_sums<TOut><<<p.blocks, kScanThreads, 0, st>>>(in, n, p.chunk, scratch));
  SPH_LAUNCH(ws, name, st,
             k_scan<TOut><<<p.blocks, kScanThreads, 0, st>>>(
                 in, n, p.chunk, p.sums ? scratch : nullptr, out, info, capacity, gate));
  return SPH_OK;
}

__device__ __forceinline__ void scatter_body(const int32_t* __restrict__ pcell,
                                             const int32_t* __restrict__ pslot,
                                             const int32_t* __restrict__ cell_start,
                                             int32_t* __restrict__ unsorted, int n,
                                             const int32_t* __restrict__ gate, int blk) {
  if (gate && *gate == 0) return;
  int i = blk * blockDim.x + threadIdx.x;
  if (i >= n) return;
  unsorted[cell_start[pcell[i]] + pslot[i]] = i;
}

__global__ void k_scatter(const int32_t* __restrict__ pcell, const int32_t* __restrict__ pslot,
                          const int32_t* __restrict__ cell_start, int32_t* __restrict__ unsorted,
                          int n, const int32_t* __restrict__ gate = nullptr) {
  scatter_body(pcell, pslot, cell_start, unsorted, n, gate, blockIdx.x);
}

// Morton code of the particle's 4^DIM sub-cell inside its cell (2 bits per
// axis, the octant's bits above the quarter's).
template <int DIM>
__device__ __forceinline__ unsigned sub_cell_code(const float4 p, const Grid& g) {
  const float x[3] = {p.x, p.y, p.z};
  unsigned code = 0u;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const float q = (float)((double)x[d] / (double)g.cs[d]);
    int c = (int)q;
    c = c < 0 ? 0 : (c >= g.cps[d] ? g.cps[d] - 1 : c);
    int f = (int)((q - (float)c) * 4.0f);
    f = f < 0 ? 0 : (f > 3 ? 3 : f);
    code |= ((unsigned)(f >> 1) << (DIM + d)) | ((unsigned)(f & 1) << d);
  }
  return code;
}

// Sort key of particle `id` within its cell: the id alone, or (with positions)
// the sub-cell code first and the id second.
template <int DIM>
__device__ __forceinline__ unsigned long long cell_sort_key(int id, const float* __restrict__ r,
                                                            const Grid& g) {
  unsigned long long k = (unsigned)id;
  if (r) k |= (unsigned long long)sub_cell_code<DIM>(load_pos<DIM>(r, id), g) << 32;
  return k;
}

// One wavefront per cell: rank-sort the ids that arrived in the cell.  Without
// positions (r == nullptr) a cell lists its particles in ascending id, like the
// reference's stable argsort; with positions (skin lists, whose order is free)
// the particles of a cell follow a Morton curve over its sub-cells, so that
// consecutive particles, which share wavefronts in the sweeps, are close.
// `clear` (or null): the cell histogram, zeroed here for the next binning.
template <int DIM>
__device__ __forceinline__ void cell_sort_body(const int32_t* __restrict__ cell_start,
                                               const int32_t* __restrict__ unsorted,
                                               int32_t* __restrict__ perm,
                                               int32_t* __restrict__ iperm, int64_t ncell,
                                               const int32_t* __restrict__ gate, int blk,
                                               const float* __restrict__ r, const Grid& g,
                                               int32_t* __restrict__ clear) {
  if (gate && *gate == 0) return;
  const int lane = threadIdx.x & 63;
  const int64_t cell = ((int64_t)blk * blockDim.x + threadIdx.x) >> 6;
  if (cell >= ncell) return;
  if (clear && lane == 0) clear[cell] = 0;
  const int b = cell_start[cell], e = cell_start[cell + 1], n = e - b;
  if (n <= 64) {
    const unsigned long long key = lane < n ? cell_sort_key<DIM>(unsorted[b + lane], r, g)
                                            : ~0ull;
    int rank = 0;
    for (int k = 0; k < n; ++k) {
      const unsigned long long o = __shfl(key, k, 64);
      rank += (o < key) ? 1 : 0;
    }
    if (lane < n) {
      const int id = (int)(unsigned)(key & 0xffffffffull);
      perm[b + rank] = id;
      iperm[id] = b + rank;
    }
  } else {
    // 64 ids against 64 at a time, handed round among the lanes (a load a
    // comparison, each waited for, took 35.3 ms for 5,000 in one cell; so 21.7)
    for (int k0 = 0; k0 < n; k0 += 64) {
      const bool mine = k0 + lane < n;
      const unsigned long long key =
          mine ? cell_sort_key<DIM>(unsorted[b + k0 + lane], r, g) : ~0ull;
      int rank = 0;
      for (int c0 = 0; c0 < n; c0 += 64) {
        const int m = n - c0 < 64 ? n - c0 : 64;
        const unsigned long long other =
            lane < m ? cell_sort_key<DIM>(unsorted[b + c0 + lane], r, g) : ~0ull;
        for (int k = 0; k < m; ++k) rank += __shfl(other, k, 64) < key ? 1 : 0;
      }
      if (mine) {
        const int id = (int)(unsigned)(key & 0xffffffffull);
        perm[b + rank] = id;
        iperm[id] = b + rank;
      }
    }
  }
}

template <int DIM>
__global__ __launch_bounds__(256) void k_cell_sort(const int32_t* __restrict__ cell_start,
                                                   const int32_t* __restrict__ unsorted,
                                                   int32_t* __restrict__ perm,
                                                   int32_t* __restrict__ iperm, int64_t ncell,
                                                   const int32_t* __restrict__ gate,
                                                   const float* __restrict__ r, Grid g,
                                                   int32_t* __restrict__ clear) {
  cell_sort_body<DIM>(cell_start, unsorted, perm, iperm, ncell, gate, blockIdx.x, r, g, clear);
}

// Hash and histogram of the skin grid, gated on the rebuild request; the first
// cell_blocks workgroups instead take kCellsBlock cells each of this step's
// reference-grid histogram: its largest entry into info[2] (reset by the drift)
// with the cell-capacity bit, the histogram cleared for the next step.  They
// ride in this launch because nothing in it depends on them.
constexpr int kCellsBlock = 16 * kBlock;
template <int DIM>
__global__ __launch_bounds__(kBlock) void k_skin_hash(
    const float* __restrict__ r, int n, Grid g, int32_t* __restrict__ cell_count,
    int32_t* __restrict__ pcell, int32_t* __restrict__ pslot, const int32_t* __restrict__ flag,
    int32_t* __restrict__ ref_count, int64_t ref_ncell, int cell_blocks,
    int64_t* __restrict__ info, int64_t capacity) {
  if ((int)blockIdx.x >= cell_blocks) {
    hash_count_body<DIM>(r, n, g, cell_count, pcell, pslot, flag, blockIdx.x - cell_blocks);
    return;
  }
  int m = 0;
#pragma unroll
  for (int q = 0; q < kCellsBlock / kBlock; ++q) {
    const int64_t i = (int64_t)blockIdx.x * kCellsBlock + q * kBlock + threadIdx.x;
    if (i < ref_ncell) {
      m = max(m, ref_count[i]);
      ref_count[i] = 0;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_down(m, o, 64));
  if ((threadIdx.x & 63) == 0 && m > 0) {
    atomicMax((unsigned long long*)&info[2], (unsigned long long)m);
    if (capacity >= 0 && m > capacity)
      atomicOr((unsigned long long*)&info[0], (unsigned long long)SPH_CELL_LIST_OVERFLOW);
  }
}

// Binning of a small particle set by one workgroup, with the histogram, the
// ids and their sort keys in LDS: one launch instead of hash, scan, scatter and
// sort, which a small set spends on launches (4 x 2-6 us).  The same cells and
// the same order inside them.  SKIN: gated on the rebuild request, sub-cell
// order, and before the gate the reference-grid occupancy as in k_skin_hash;
// otherwise the error block is reset and receives the grid's own occupancy.
// A thread takes kBinOwn particles and as many cells: up to kBinMax of each.
// Microseconds a step by separate launches and so: skin step of 2,500 2D
// particles 74.9 and 63.0, of 4,096 74.3 and 63.4, of 4,096 in 3D 90.5 and 88.8
// (a rank among 38 particles a cell instead of 10); exact step 73.2 and 59.8,
// 72.1 and 64.6, 141.6 and 142.1.  Larger sets have more than one workgroup
// can do in the time of the launches saved.
constexpr int kBinThreads = 1024;
constexpr int kBinOwn = 4;
constexpr int kBinMax = kBinOwn * kBinThreads;
static bool bins_small(int n, int64_t ncell) { return n <= kBinMax && ncell <= kBinMax; }

struct BinSmall {
  const float* r;
  int n;
  Grid g;
  int64_t ncell;
  int32_t *cell_start, *perm, *iperm;
  float4* pos;         // not SKIN, or null: the sorted positions
  int32_t* ref_count;  // SKIN
  int64_t ref_ncell;
  int64_t* info;
  const int64_t* prev;  // not SKIN
  int64_t capacity;
  const int32_t* gate;  // SKIN
};

template <int DIM, bool SKIN>
__global__ __launch_bounds__(kBinThreads) void k_bin_small(BinSmall a) {
  __shared__ int32_t start[kBinMax + 1];
  __shared__ uint32_t keys[kBinMax];
  __shared__ int32_t part[kBinThreads / 64];
  __shared__ int32_t occ[kBinThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  int m = 0;
  if (SKIN) {
    for (int64_t i = t; i < a.ref_ncell; i += kBinThreads) {
      m = max(m, a.ref_count[i]);
      a.ref_count[i] = 0;
    }
  }
  const bool run = !SKIN || *a.gate != 0;  // uniform
  int cell[kBinOwn], slot[kBinOwn];
  if (run) {
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) start[t + q * kBinThreads] = 0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) {
      const int i = t + q * kBinThreads;
      cell[q] = slot[q] = 0;
      if (i < a.n) {
        if (a.g.use_cells) {
          int c[3];
          cell_coords<DIM>(load_pos<DIM>(a.r, i), a.g, c);
          cell[q] = cell_hash<DIM>(c, a.g);
        }
        slot[q] = atomicAdd(&start[cell[q]], 1);
      }
    }
    __syncthreads();
    // exclusive scan: thread t takes cells 4t..4t+3
    int v[kBinOwn], s = 0;
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) {
      v[q] = start[kBinOwn * t + q];
      s += v[q];
      if (!SKIN) m = max(m, v[q]);
    }
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(inc, o, 64);
      if (lane >= o) inc += y;
    }
    if (lane == 63) part[wid] = inc;
    __syncthreads();
    int base = inc - s;
#pragma unroll
    for (int w = 0; w < kBinThreads / 64; ++w) base += w < wid ? part[w] : 0;
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) {
      const int c = kBinOwn * t + q;
      start[c] = base;
      if (c <= a.ncell) a.cell_start[c] = base;
      base += v[q];
    }
    if (t == kBinThreads - 1) {
      start[kBinMax] = base;
      if (a.ncell == kBinMax) a.cell_start[kBinMax] = base;
    }
    __syncthreads();
    // sort keys: (sub-cell, id), ids below kBinMax
    uint32_t key[kBinOwn];
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) {
      const int i = t + q * kBinThreads;
      if (i >= a.n) continue;
      key[q] = (uint32_t)i;
      if (SKIN) key[q] |= sub_cell_code<DIM>(load_pos<DIM>(a.r, i), a.g) * (uint32_t)kBinMax;
      keys[start[cell[q]] + slot[q]] = key[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kBinOwn; ++q) {
      const int i = t + q * kBinThreads;
      if (i >= a.n) continue;
      const int b = start[cell[q]], e = start[cell[q] + 1];
      int rank = b;
      for (int k = b; k < e; ++k) rank += keys[k] < key[q] ? 1 : 0;
      a.perm[rank] = i;
      a.iperm[i] = rank;
      if (!SKIN && a.pos) a.pos[rank] = load_pos<DIM>(a.r, i);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_down(m, o, 64));
  if (lane == 0) occ[wid] = m;
  __syncthreads();
  if (t == 0) {
    int mm = 0;
    for (int w = 0; w < kBinThreads / 64; ++w) mm = max(mm, occ[w]);
    if (!SKIN) reset_info(a.info, a.prev);
    a.info[2] = mm;
    if (a.capacity >= 0 && mm > a.capacity) a.info[0] |= SPH_CELL_LIST_OVERFLOW;
  }
}

template <int DIM>
__global__ void k_gather_pos(const float* __restrict__ r, const int32_t* __restrict__ perm,
                             float4* __restrict__ pos, int n) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  pos[s] = load_pos<DIM>(r, perm[s]);
}

// ----------------------------------------------------------- pair build
struct BuildArgs {
  const float4* pos;
  const int32_t* cell_start;
  const int32_t* perm;
  int32_t* ell;
  int32_t* cnt;
  int64_t* info;
  Grid g;
  float box[3], half[3];
  float cutoff_sq;
  // fast filter: squared distances of the cell-adjacent image below `lo` are
  // in, above `hi` out; the band [lo, hi) bounds the difference between that
  // and the exact reference metric, and is decided by the exact predicate.
  // (Skin lists: lo = hi, no band; see test_range.)
  float lo, hi;
  int fast;
  TileBand tile;  // where the filter of k_nl_tile decides, the one above elsewhere
  int range;  // consecutive sorted particles whose pieces a workgroup of k_nl_tile takes
  int n, npad, lane_width, mask_self;
  int64_t* part;          // [2 * gridDim.x]: pairs found and largest list, per workgroup
  int64_t trunc_bits;     // error bits raised when a sub-list overflows
  const int32_t* gate;    // nullable: skip the build when *gate == 0
  int remap;              // XCD-contiguous block order (grid a multiple of 8)
};

// Lane h (of TPP) tests candidates base + h, base + h + TPP, ... of one cell
// range [lo, hi) whose image is shifted by `img`; the TPP lanes of a particle
// step through the range together, 32 candidates each per chunk (so each load
// of the particle's lanes reads TPP consecutive positions), and collect their
// hits in a bit mask.  The particle's hits are numbered in candidate order
// over all its lanes, and hit k goes to sub-list k mod TPP at position k / TPP:
// the sub-lists differ in length by at most one, so the lanes that later sweep
// them finish together, and at each step of a sweep the particles of a
// wavefront read neighbours at similar places of the sorted order.
// The first kStage entries of each sub-list are staged in LDS (in the column
// of the thread that owns the sub-list) and written out row by row at the end,
// so every pair-buffer row is written by whole wavefronts at once; later
// entries go straight to the buffer.  24 staged entries (24 KB per workgroup)
// leave LDS for 6 workgroups per CU, which matches the 6 waves per SIMD the
// build's registers allow.
constexpr int kStage = 24;

// BAND = false (skin lists): pairs are kept by the fast squared distance
// alone.  A skin list must hold every pair within cutoff + 0.98 skin (the
// most two particles can close before the next rebuild), so rounding at its
// outer edge, cutoff + skin, cannot drop a pair that matters.  Skin lists of
// 160,000 and 409,600 2D particles 30.6 and 52.6 us, with the band's
// comparisons and each candidate's index clamped 37.3 and 62.1; of an ensemble
// of 64 members (565,000 2D particles) 129 and 157.
template <int DIM, int TPP, bool ORDERED, bool BAND>
__device__ __forceinline__ void test_range(const BuildArgs& a, int s, int h, const float4 ps,
                                           int sid, int lo, int hi, const float* img,
                                           int32_t* __restrict__ out0, int32_t* stage0,
                                           int& count) {
  // out0: entry 0 of the particle's sub-list 0; stage0: the stage column of
  // the particle's lane 0 (sub-list q is column stage0 + q)
  const float sx = ps.x - img[0], sy = ps.y - img[1], sz = ps.z - img[2];
  constexpr int G = 8;  // candidates whose loads are issued together
  for (int base = lo; base < hi; base += 32 * TPP) {  // same trip count on all TPP lanes
    const int c0 = base + h;
    int nb = c0 < hi ? (hi - c0 + TPP - 1) / TPP : 0;
    nb = nb < 32 ? nb : 32;
    unsigned mask = 0u;
    for (int t0 = 0; t0 < nb; t0 += G) {
      float4 pg[G];
      if (BAND) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int b = c0 + (t0 + u) * TPP;
          const int bc = b < hi ? b : hi - 1;
          __builtin_assume(bc >= 0);  // sorted slots: no sign extension in the address
          pg[u] = a.pos[bc];
        }
      } else {
        // skin builds read past the range into the padded tail (kSkinPosPad),
        // from one address with constant offsets; those candidates are masked
        // off below
        __builtin_assume(c0 >= 0);
        const float4* __restrict__ pb = a.pos + (c0 + t0 * TPP);
#pragma unroll
        for (int u = 0; u < G; ++u) pg[u] = pb[u * TPP];
      }
      unsigned got = 0u;  // bit u: candidate t0 + u is a pair
      if (!BAND) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const float4 pb = pg[u];
          got |= dist2<DIM>(sx - pb.x, sy - pb.y, sz - pb.z) < a.lo ? 1u << u : 0u;
        }
      } else if (a.fast) {
        bool near = false;  // some candidate lies in the band around the cutoff
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const float4 pb = pg[u];
          const float d2 = dist2<DIM>(sx - pb.x, sy - pb.y, sz - pb.z);
          got |= d2 < a.lo ? 1u << u : 0u;
          near = near || (d2 >= a.lo && d2 < a.hi);
        }
        if (near) {  // rare: the exact reference metric decides the band
#pragma unroll
          for (int u = 0; u < G; ++u) {
            const float4 pb = pg[u];
            const float d2 = dist2<DIM>(sx - pb.x, sy - pb.y, sz - pb.z);
            if (d2 >= a.lo && d2 < a.hi &&
                metric_sq_exact<DIM>(ps, pb, a.box, a.half) < a.cutoff_sq)
              got |= 1u << u;
          }
        }
      } else {
#pragma unroll
        for (int u = 0; u < G; ++u)
          if (metric_sq_exact<DIM>(ps, pg[u], a.box, a.half) < a.cutoff_sq) got |= 1u << u;
      }
      if (ORDERED) {  // candidates past the range are dropped before perm is read
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int b = c0 + (t0 + u) * TPP;
          if ((got >> u) & 1u && (t0 + u >= nb || !(a.perm[b] < sid))) got &= ~(1u << u);
        }
      }
      mask |= got << t0;
    }
    // drop the candidates past the range, and the particle itself
    if (nb < 32) mask &= (1u << nb) - 1u;
    if (a.mask_self) {
      const int ds = s - c0;
      if (ds >= 0 && ds % TPP == 0 && ds / TPP < 32) mask &= ~(1u << (ds / TPP));
    }
    // candidate base + t TPP + h follows the particle's hits at smaller t on
    // every lane and at the same t on the lanes below h
    unsigned m[TPP];
    int total = 0;
#pragma unroll
    for (int q = 0; q < TPP; ++q) {
      m[q] = __shfl(mask, q, TPP);
      total += __popc(m[q]);
    }
    while (mask) {
      const int t = __ffs(mask) - 1;
      mask &= mask - 1u;
      const unsigned upto = (2u << t) - 1u;  // bits 0..t (all 32 for t = 31)
      const unsigned below = upto >> 1;      // bits 0..t-1
      unsigned k = (unsigned)count;
#pragma unroll
      for (int q = 0; q < TPP; ++q) k += __popc(m[q] & (q < h ? upto : below));
      const int32_t b = c0 + t * TPP;
      const unsigned q = k % TPP, pos = k / TPP;
      if (pos < (unsigned)kStage) stage0[pos * kBlock + q] = b;
      else if (pos < (unsigned)a.lane_width)
        out0[(int64_t)(q * (unsigned)a.lane_width + pos) * a.npad] = b;
    }
    count += total;
  }
}

// Per-workgroup partials of a build: total pairs (sum of the threads' shares)
// and the largest list.  Every thread of the workgroup calls it.
__device__ __forceinline__ void build_partials(int64_t* __restrict__ part, int blk, int share,
                                               int count) {
  __shared__ unsigned long long tot[kBlock / 64];
  __shared__ int mx[kBlock / 64];
  unsigned long long v = (unsigned long long)share;
  int m = count;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    v += __shfl_down(v, o, 64);
    int y = __shfl_down(m, o, 64);
    m = y > m ? y : m;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) { tot[wid] = v; mx[wid] = m; }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    int mm = 0;
    for (int w = 0; w < kBlock / 64; ++w) { t += tot[w]; mm = mx[w] > mm ? mx[w] : mm; }
    part[2 * blk] = (int64_t)t;
    part[2 * blk + 1] = mm;
  }
}

// The counts of a particle's sub-list h of `share` hits (of `count`), and the
// overflow report of a particle whose sub-lists were truncated.
template <int TPP, typename Args>
__device__ __forceinline__ void store_count(const Args& a, int s, int h, int share, int count) {
  a.cnt[h * a.npad + s] = share < a.lane_width ? share : a.lane_width;
  if (h == 0 && count > TPP * a.lane_width) {  // some sub-list of s was truncated
    atomicAdd((unsigned long long*)&a.info[5], 1ull);
    if (a.trunc_bits) atomicOr((unsigned long long*)&a.info[0], (unsigned long long)a.trunc_bits);
  }
}

// TPP lanes per sorted particle (the sender): each visits the 3^d cells around
// the particle's own cell as 3^(d-1) contiguous x-strips, keeps its share of
// the receivers with d^2 < cutoff^2 and stores them in its own sub-list.
// blk: the workgroup's block within this list's grid; it also indexes the
// workgroup's partials.
template <int DIM, int TPP, bool ORDERED, bool BAND>
__device__ __forceinline__ void nl_build_body(const BuildArgs& a, const int blk) {
  __shared__ int32_t stage_buf[kStage][kBlock];
  if (a.gate && *a.gate == 0) return;  // uniform over the list's grid
  const int tid = blk * blockDim.x + threadIdx.x;
  const int s = tid / TPP, h = tid % TPP;
  int count = 0;  // hits of the particle (the same in its TPP lanes)
  if (s < a.n) {
    const float4 ps = a.pos[s];
    const int sid = ORDERED ? a.perm[s] : 0;
    int32_t* out = a.ell + s;                           // sub-list 0 of s
    int32_t* stage = &stage_buf[0][threadIdx.x - h];    // stage column of lane 0 of s
    float img[3] = {0.0f, 0.0f, 0.0f};
    if (!a.g.use_cells) {
      test_range<DIM, TPP, ORDERED, BAND>(a, s, h, ps, sid, 0, a.n, img, out, stage, count);
    } else {
      int c[3];
      cell_coords<DIM>(ps, a.g, c);
      const int nx = a.g.cps[0], ny = a.g.cps[1];
      const int nz = DIM == 3 ? a.g.cps[2] : 1;
      const int z0 = DIM == 3 ? -1 : 0, z1 = DIM == 3 ? 1 : 0;
      for (int dz = z0; dz <= z1; ++dz) {
        int cz = DIM == 3 ? c[2] + dz : 0;
        img[2] = 0.0f;
        if (cz < 0) { cz += nz; img[2] = -a.box[2]; }
        else if (cz >= nz) { cz -= nz; img[2] = a.box[2]; }
        for (int dy = -1; dy <= 1; ++dy) {
          int cy = c[1] + dy;
          img[1] = 0.0f;
          if (cy < 0) { cy += ny; img[1] = -a.box[1]; }
          else if (cy >= ny) { cy -= ny; img[1] = a.box[1]; }
          const int row = (cz * ny + cy) * nx;
          if (c[0] >= 1 && c[0] + 1 < nx) {
            img[0] = 0.0f;
            test_range<DIM, TPP, ORDERED, BAND>(a, s, h, ps, sid, a.cell_start[row + c[0] - 1],
                                    a.cell_start[row + c[0] + 2], img, out, stage, count);
          } else {
            for (int dx = -1; dx <= 1; ++dx) {
              int cx = c[0] + dx;
              img[0] = 0.0f;
              if (cx < 0) { cx += nx; img[0] = -a.box[0]; }
              else if (cx >= nx) { cx -= nx; img[0] = a.box[0]; }
              test_range<DIM, TPP, ORDERED, BAND>(a, s, h, ps, sid, a.cell_start[row + cx],
                                      a.cell_start[row + cx + 1], img, out, stage, count);
            }
          }
        }
      }
    }
  }
  // the particle's other lanes wrote into this thread's stage column
  __syncthreads();
  // this lane's sub-list: hits h, h + TPP, ... of the particle
  const int share = s < a.n ? (count + TPP - 1 - h) / TPP : 0;
  if (s < a.n) {
    int32_t* out = a.ell + ((int64_t)h * a.lane_width) * a.npad + s;
    const int32_t* stage = &stage_buf[0][threadIdx.x];
    int staged = share < kStage ? share : kStage;
    staged = staged < a.lane_width ? staged : a.lane_width;  // never past the sub-list
    for (int k = 0; k < staged; ++k) out[(int64_t)k * a.npad] = stage[k * kBlock];
    store_count<TPP>(a, s, h, share, count);
  }
  build_partials(a.part, blk, share, count);
}

template <int DIM, int TPP, bool ORDERED, bool BAND>
__global__ __launch_bounds__(kBlock, ORDERED ? 1 : 6) void k_nl_build(BuildArgs a) {
  nl_build_body<DIM, TPP, ORDERED, BAND>(a, logical_block(a.remap));
}

// ------------------------------------------------- pair build, matrix cores
// The same lists as nl_build_body (hits in candidate order, dealt round-robin),
// for the unordered builds of a grid whose cell-adjacent image decides.  A
// wavefront takes up to tile_rows particles of one cell (a "piece").  Their
// candidates, the 3^(d-1) strips of cells (3^d cells at a face), are numbered
// one after another and taken 64 at a time, one a lane; v_mfma_f32_4x4x1 with
// the particles' block broadcast then gives 4 particles x 64 candidates of
//   |a|^2 + |b|^2 - 2 a.b,   a, b relative to the cell's centre,
// one particle a register, one candidate a lane, so a comparison's lane mask is
// that particle's hits in candidate order: a hit's number is a count of the
// mask's lower bits, and only the store to the stage runs for hits alone.
// Squares within a band of the cutoff are decided by the filter of
// nl_build_body.
// Bound by the issue of instructions (vector 83%, scalar 35% of the cycles, the
// matrix cores busy in 12%), 10 for a particle and 64 candidates; a lane that
// tests candidates of its own takes 9 per candidate and 25 per hit, in a loop as
// long as the wavefront's longest.  Exact list of 1,000,000 3D particles
// 647 -> 398 us; tile_pays() has the other sizes.
// A stage entry is 16 bits (segment and offset in it, from which the sorted
// index follows), so that 7 workgroups' stages fit a CU's LDS; entries past
// the stage, and those of segments over 2,047 long, go straight to the buffer.
constexpr int kTileSegBits = 11;
constexpr int kCandBits = 27;  // the same in a register: 5 bits of segment, 27 of offset
static_assert(kCandBits - kTileSegBits == 16, "an entry is the halves of a code, or'ed");
constexpr int tile_stage(int dim) { return dim == 3 ? 176 : 48; }
// Particles of a piece: a 3D cell's 28 to 38 in two or three, a 2D cell's 9 to
// 11 in one (with 16 rows, seven of them idle, 150 us at 810,000 particles).
constexpr int tile_rows(int dim) { return dim == 3 ? 16 : 12; }

__device__ __forceinline__ int lane_i(int x, int l) { return __builtin_amdgcn_readlane(x, l); }
__device__ __forceinline__ float lane_f(float x, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

template <int Q, int NQ, typename F>
__device__ __forceinline__ void for_blocks(F&& f) {
  f(std::integral_constant<int, Q>{});
  if constexpr (Q + 1 < NQ) for_blocks<Q + 1, NQ>(f);
}

// The arguments stay in memory (read by scalar loads, again for each piece and
// in the rare paths): all of them beside a count for each particle are more
// than the scalar registers hold, and a spilled one costs vector instructions.
using ColdArgs = const __attribute__((address_space(4))) BuildArgs;
__device__ __forceinline__ ColdArgs* again(ColdArgs* a) {
  asm volatile("" : "+s"(a));
  return a;
}

// R: consecutive sorted particles of a workgroup, which takes the pieces that
// start there (tile_pays, or what the caller's grid makes of it).
template <int DIM, int TPP>
__device__ __forceinline__ void nl_tile_body(ColdArgs* args, const int blk, const int R) {
  constexpr int W = kBlock / 64, S = tile_stage(DIM), P = tile_rows(DIM);
  constexpr int kRowLanes = 16;        // lane l: particle l mod 16 of the piece
  constexpr int L = 64 / kRowLanes;    // and one of so many for it in the write-out
  static_assert(P <= kRowLanes, "a lane a particle");
  typedef float v4f __attribute__((ext_vector_type(4)));
  typedef unsigned long long mask_t;
  using Entry = __attribute__((address_space(3))) uint16_t;
  // rows of an odd number of words: the lanes that read one entry of each
  // particle fall on different banks
  constexpr int kRow = S + 2;
  static_assert(kRow / 2 % 2 == 1, "odd row length");
  __shared__ uint16_t stage_buf[W][P * kRow];
  const int32_t* gate = args->gate;
  if (gate && *gate == 0) return;  // uniform over the list's grid
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = args->n;
  const float4* __restrict__ pos = args->pos;
  const uint16_t* stage = stage_buf[wv];
  // entry 0 of row 0, counted in entries from the start of the LDS
  const unsigned row0 = (unsigned)(uintptr_t)(Entry*)stage / 2;
  const int p = lane % kRowLanes, part = lane / kRowLanes;
  int found = 0, most_found = 0;  // pairs and largest list of this wavefront's pieces
  const int end = min(n, (blk + 1) * R);
  for (int g0 = blk * R; g0 < end; g0 += 64) {
    // ---- the cells of 64 particles, one a lane, the same in every wavefront
    const int s = g0 + lane < end ? g0 + lane : end - 1;
    int cc[3] = {0, 0, 0}, cell_lo, cell_hi;
    {
      const Grid g = {{args->g.cs[0], args->g.cs[1], args->g.cs[2]},
                      {args->g.cps[0], args->g.cps[1], args->g.cps[2]}, 1};
      cell_coords<DIM>(pos[s], g, cc);
      const int32_t* start = args->cell_start + cell_hash<DIM>(cc, g);
      cell_lo = start[0];
      cell_hi = start[1];
    }
    // the particles that start a piece; the wavefronts take them in turn
    mask_t pieces = __ballot(g0 + lane < end && (unsigned)(s - cell_lo) % P == 0u);
    for (int turn = 0; pieces; ++turn) {
      const int l = __ffsll((long long)pieces) - 1;
      pieces &= pieces - 1ull;
      if (turn % W != wv) continue;
      ColdArgs* const a = again(args);
      const int s0 = g0 + l;
      const int np = min(P, lane_i(cell_hi, l) - s0);
      const int nx = a->g.cps[0], ny = a->g.cps[1], nz = DIM == 3 ? a->g.cps[2] : 1;
      const int cx = lane_i(cc[0], l), cy = lane_i(cc[1], l);
      const int cz = DIM == 3 ? lane_i(cc[2], l) : 0;
      const float4 ps = pos[s0 + (p < np ? p : np - 1)];
      // ---- its segments of candidates, one a lane, in the order of the cells
      const bool face = cx < 1 || cx + 1 >= nx;
      const int nseg = (DIM == 3 ? 9 : 3) * (face ? 3 : 1);
      int lo = 0, len = 0;
      float ix = 0.0f, iy = 0.0f, iz = 0.0f;  // image of the segment's cells
      if (lane < nseg) {
        const int strip = face ? lane / 3 : lane;
        int x = face ? cx + lane % 3 - 1 : cx - 1;
        int y = cy + strip % 3 - 1, z = DIM == 3 ? cz + strip / 3 - 1 : 0;
        if (x < 0) { x += nx; ix = -a->box[0]; }
        else if (x >= nx) { x -= nx; ix = a->box[0]; }
        if (y < 0) { y += ny; iy = -a->box[1]; }
        else if (y >= ny) { y -= ny; iy = a->box[1]; }
        if (z < 0) { z += nz; iz = -a->box[2]; }
        else if (z >= nz) { z -= nz; iz = a->box[2]; }
        const int32_t* start = a->cell_start + (z * ny + y) * nx + x;
        lo = start[0];
        len = start[face ? 1 : 3] - lo;
      }
      const bool image = __ballot(ix != 0.0f || iy != 0.0f || iz != 0.0f) != 0ull;
      // entries a particle can stage
      const int room = __ballot(len >= 1 << kTileSegBits) != 0ull ? 0 : S;
      // inclusive scan over 32 lanes, a row of 16 at a time
      int pre = len;
      pre += __builtin_amdgcn_update_dpp(0, pre, 0x111, 0xf, 0xf, true);  // row_shr:1
      pre += __builtin_amdgcn_update_dpp(0, pre, 0x112, 0xf, 0xf, true);
      pre += __builtin_amdgcn_update_dpp(0, pre, 0x114, 0xf, 0xf, true);
      pre += __builtin_amdgcn_update_dpp(0, pre, 0x118, 0xf, 0xf, true);
      int total = lane_i(pre, 15);
      pre += lane >= 16 ? total : 0;
      total = lane_i(pre, 31);
      pre -= len;
      const int shift = lo - pre;                     // sorted index of a candidate
      const unsigned code = ((unsigned)lane << kCandBits) - (unsigned)pre;  // and its code
      // particle s0's number as a candidate (in the middle segment), for mask_self
      const int self0 = a->mask_self ? s0 - lane_i(shift, nseg / 2) : -(1 << 30);
      // ---- the particles, relative to the cell's centre
      const float csx = a->g.cs[0], csy = a->g.cs[1], csz = a->g.cs[2];
      const float ox = ((float)cx + 0.5f) * csx, oy = ((float)cy + 0.5f) * csy;
      const float oz = DIM == 3 ? ((float)cz + 0.5f) * csz : 0.0f;
      float ax = ps.x - ox, ay = ps.y - oy, az = DIM == 3 ? ps.z - oz : 0.0f;
      float aa = dist2<DIM>(ax, ay, az);
      // d below is the square less `mid`; hits are under -width, and the
      // exact filter decides within width
      const float mid = 0.5f * (a->tile.lo + a->tile.hi);
      float width = 0.5f * (a->tile.hi - a->tile.lo);
      const bool inside = fabsf(ax) <= a->tile.inside[0] && fabsf(ay) <= a->tile.inside[1] &&
                          (DIM == 2 || fabsf(az) <= a->tile.inside[2]);
      ax *= -2.0f;
      ay *= -2.0f;
      az *= -2.0f;
      if (__ballot(!inside)) {
        // a particle outside its cell (unwrapped positions are clamped into
        // the grid) or not finite: the filter's bounds do not hold, and every
        // candidate of the piece is left to the exact one
        aa = ax = ay = az = 0.0f;
        width = 3.4e38f;
      }
      if (p >= np) aa = INFINITY;  // no particle: no hits
      int seg = 0;  // the last segment that starts before the candidates seen end
      const int full = (int)row0 + room;
      int tops = (int)row0;  // lane q: the next entry of row q, less q kRow
      // A chunk of candidates is requested before the tests of the one before
      // (past the end: s0 again); more ahead gained nothing.
      // c, at: candidate c0 + lane, its segment and offset in it, and its
      // position, three words of it: a fourth that nothing reads would be some
      // other value's register next, which then waits for the load
      struct Xyz { float x, y, z; };
      unsigned c_next = 0;
      Xyz at_next{0.f, 0.f, 0.f};
      for (int c0 = -64; c0 < total; c0 += 64) {
        const unsigned c = c_next;
        const Xyz at = at_next;
        const int o = c0 + 64 + lane;
        int to_j = lane_i(shift, seg);
        unsigned to_c = (unsigned)lane_i((int)code, seg);
        while (seg + 1 < nseg) {
          const int first = lane_i(pre, seg + 1);
          if (first >= c0 + 128) break;
          ++seg;
          const bool on = o >= first;
          const int tj = lane_i(shift, seg), tc = lane_i((int)code, seg);
          to_j = on ? tj : to_j;
          to_c = on ? (unsigned)tc : to_c;
        }
        at_next = *(const Xyz*)(pos + (unsigned)(o < total ? o + to_j : s0));
        c_next = (unsigned)o + to_c;
        const float4 pb = make_float4(at.x, at.y, at.z, 0.0f);
        if (c0 >= 0) {
          const bool valid = c0 + lane < total;
          float cix = 0.0f, ciy = 0.0f, ciz = 0.0f;  // its image
          if (image) {
            cix = __shfl(ix, (int)(c >> kCandBits), 64);
            ciy = __shfl(iy, (int)(c >> kCandBits), 64);
            if (DIM == 3) ciz = __shfl(iz, (int)(c >> kCandBits), 64);
          }
          const float bx = pb.x - (ox - cix), by = pb.y - (oy - ciy);
          const float bz = DIM == 3 ? pb.z - (oz - ciz) : 0.0f;
          const uint16_t entry = (uint16_t)((c >> (kCandBits - kTileSegBits)) | c);
          const float bb = valid ? dist2<DIM>(bx, by, bz) - mid : INFINITY;
          const v4f b4 = {bb, bb, bb, bb};
          v4f d[P / 4];  // one chain a block, side by side
          for_blocks<0, P / 4>([&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            d[Q] = __builtin_amdgcn_mfma_f32_4x4x1f32(aa, 1.0f, b4, 4, Q, 0);
          });
          for_blocks<0, P / 4>([&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            d[Q] = __builtin_amdgcn_mfma_f32_4x4x1f32(ax, bx, d[Q], 4, Q, 0);
          });
          for_blocks<0, P / 4>([&](auto qc) {
            constexpr int Q = decltype(qc)::value;
            d[Q] = __builtin_amdgcn_mfma_f32_4x4x1f32(ay, by, d[Q], 4, Q, 0);
          });
          if (DIM == 3)
            for_blocks<0, P / 4>([&](auto qc) {
              constexpr int Q = decltype(qc)::value;
              d[Q] = __builtin_amdgcn_mfma_f32_4x4x1f32(az, bz, d[Q], 4, Q, 0);
            });
          const int self = c0 + lane - self0;  // the particle this candidate is, if any
          if (__ballot(self >= 0 && self < np)) {
#pragma unroll
            for (int q = 0; q < P; ++q) d[q / 4][q % 4] = self == q ? INFINITY : d[q / 4][q % 4];
          }
          float nearest = INFINITY;
#pragma unroll
          for (int q = 0; q < P; ++q) nearest = fminf(nearest, fabsf(d[q / 4][q % 4]));
          mask_t m[P];
          int hits = 0;  // lane q: those of particle q
#pragma unroll
          for (int q = 0; q < P; ++q) {
            m[q] = __ballot(d[q / 4][q % 4] < -width);
            // one lane of hits (the compiler has no builtin for it)
            asm("v_writelane_b32 %0, %1, %2" : "+v"(hits) : "s"((int)__popcll(m[q])), "n"(q));
          }
          // the hits of each particle that `hit_of` gives as a lane mask, to the stage
          const auto stage_hits = [&](auto&& hit_of) __attribute__((always_inline)) {
            for_blocks<0, P / 4>([&](auto qc) {
              constexpr int q0 = 4 * decltype(qc)::value;
              if (q0 >= np) return;  // uniform
#pragma unroll
              for (int q = q0; q < q0 + 4; ++q) {
                const mask_t mq = hit_of(q);
                const unsigned k =
                    __builtin_amdgcn_mbcnt_hi((unsigned)(mq >> 32),
                                              __builtin_amdgcn_mbcnt_lo((unsigned)mq, 0u));
                const unsigned row = (unsigned)lane_i(tops, q);
                Entry* const to = (Entry*)(uintptr_t)((k + row) << 1) + q * kRow;
                if (__builtin_expect(__builtin_amdgcn_inverse_ballot_w64(mq), 1)) *to = entry;
              }
            });
            tops += hits;
          };
          if (__builtin_expect(__ballot(nearest < width || tops + hits > full) == 0ull, 1)) {
            stage_hits([&](int q) { return m[q]; });
          } else {
            // A lane's hits and its pairs within the band, a bit a particle; the
            // exact filter decides the latter, one of each lane at a time.  On a
            // lattice a chunk has some 40 such pairs, nearly every particle one:
            // 1,000,000 on one took 1,503 us particle by particle (the lanes' build
            // 902), so 825.
            unsigned in = 0u, near = 0u;
#pragma unroll
            for (int q = 0; q < P; ++q) {
              in |= d[q / 4][q % 4] < -width ? 1u << q : 0u;
              near |= fabsf(d[q / 4][q % 4]) < width ? 1u << q : 0u;
            }
            ColdArgs* const e = again(args);
            const float box[3] = {e->box[0], e->box[1], e->box[2]};
            const float half[3] = {e->half[0], e->half[1], e->half[2]};
            const float flo = e->lo, fhi = e->hi, csq = e->cutoff_sq;
            while (__ballot(near != 0u)) {
              const int q = near != 0u ? __ffs((int)near) - 1 : 0;
              const float4 pq = make_float4(__shfl(ps.x, q, 64), __shfl(ps.y, q, 64),
                                            DIM == 3 ? __shfl(ps.z, q, 64) : 0.0f, 0.0f);
              const float d2 = dist2<DIM>(pq.x - cix - pb.x, pq.y - ciy - pb.y,
                                          DIM == 3 ? pq.z - ciz - pb.z : 0.0f);
              const bool hit =
                  d2 < flo || (d2 < fhi && metric_sq_exact<DIM>(pq, pb, box, half) < csq);
              in |= hit && near != 0u ? 1u << q : 0u;
              near &= near - 1u;
            }
#pragma unroll
            for (int q = 0; q < P; ++q)
              asm("v_writelane_b32 %0, %1, %2"
                  : "+v"(hits) : "s"((int)__popcll(__ballot(in >> q & 1u))), "n"(q));
            if (__ballot(tops + hits > full) == 0ull) {
              stage_hits([&](int q) { return (mask_t)__ballot(in >> q & 1u); });
            } else {
              // hits past the stage go straight to the buffer
              ColdArgs* const f = again(args);
              const int lane_width = f->lane_width;
              const int cj =
                  __shfl(lo, (int)(c >> kCandBits), 64) + (int)(c & ((1u << kCandBits) - 1u));
#pragma unroll 1
              for (int q = 0; q < np; ++q) {
                const bool hit = in >> q & 1u;
                const mask_t mq = __ballot(hit);
                const int t = lane_i(tops, q);
                const int k = t - (int)row0 +  // its number among the particle's hits
                              (int)__builtin_amdgcn_mbcnt_hi(
                                  (unsigned)(mq >> 32),
                                  __builtin_amdgcn_mbcnt_lo((unsigned)mq, 0u));
                if (hit && k < room)
                  *(Entry*)(uintptr_t)((k + row0 + q * kRow) << 1) = entry;
                else if (hit && k / TPP < lane_width)
                  f->ell[((int64_t)(k % TPP) * lane_width + k / TPP) * f->npad + s0 + q] = cj;
                tops = lane == q ? t + (int)__popcll(mq) : tops;
              }
            }
          }
        }
      }
      // ---- counts, and the staged entries in the order of the buffer's rows
      const int own = __shfl(tops, p, 64) - (int)row0;  // 0 where there is no particle
      int most = own;
#pragma unroll
      for (int o = kRowLanes / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
      most = __builtin_amdgcn_readfirstlane(most);
      __builtin_amdgcn_wave_barrier();
      ColdArgs* const b = again(args);
      const int lane_width = b->lane_width, npad = b->npad;
      found += part == 0 ? own : 0;
      most_found = most > most_found ? most : most_found;
      if (p < np && part < TPP)
        store_count<TPP>(*b, s0 + p, part, (own + TPP - 1 - part) / TPP, own);
      // hit k goes to sub-list k mod TPP at k / TPP
      const int staged = min(p < np ? min(own, room) : 0, TPP * lane_width);
      most = min(most, room);
      int32_t* out = b->ell + ((int64_t)(part % TPP) * lane_width + part / TPP) * npad + s0 + p;
      const int64_t row = (L / TPP) * (int64_t)npad;
      constexpr int kAhead = 4;  // rows whose LDS reads are in flight together
      for (int k0 = 0; k0 < most; k0 += L * kAhead) {
        int e[kAhead], j[kAhead];
#pragma unroll
        for (int t = 0; t < kAhead; ++t)  // in the stage also past its last entry
          e[t] = stage[min(min(p, P - 1) * kRow + k0 + L * t + part, P * kRow - 1)];
#pragma unroll
        for (int t = 0; t < kAhead; ++t)
          j[t] = __shfl(lo, e[t] >> kTileSegBits, 64) + (e[t] & ((1 << kTileSegBits) - 1));
#pragma unroll
        for (int t = 0; t < kAhead; ++t) {
          if (k0 + L * t + part < staged) *out = j[t];
          out += row;
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  build_partials(again(args)->part, blk, found, most_found);
}

template <int DIM, int TPP>
__global__ __launch_bounds__(kBlock, 6) void k_nl_tile(BuildArgs) {
  // the kernel's one argument, where it lies
  ColdArgs* const args = (ColdArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  nl_tile_body<DIM, TPP>(args, logical_block(args->remap), args->range);
}

__global__ void k_finalize(int64_t* __restrict__ info, int64_t max_occ) {
  if (threadIdx.x == 0 && info[1] > max_occ) info[0] |= SPH_NEIGHBOR_LIST_OVERFLOW;
}

constexpr int kReduceThreads = 1024;
__global__ __launch_bounds__(kReduceThreads) void k_reduce_parts(Reduce a) {
  reduce_parts_body<kReduceThreads>(a);
}

template <int DIM>
__global__ void k_needs_rebuild(const float* __restrict__ r, const float* __restrict__ ref, int n,
                                Grid g, float bx, float by, float bz, float thr_sq,
                                int64_t* __restrict__ info) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float box[3] = {bx, by, bz};
  float half[3] = {bx * 0.5f, by * 0.5f, bz * 0.5f};
  float d2 = metric_sq_exact<DIM>(load_pos<DIM>(r, i), load_pos<DIM>(ref, i), box, half);
  if (d2 > thr_sq) atomicOr((unsigned long long*)&info[4], 1ull);
}

// ----------------------------------------------------------- idx writer
__global__ void k_counts_orig(const int32_t* __restrict__ perm, const int32_t* __restrict__ cnt,
                              int32_t* __restrict__ cnt_id, int n, int npad, int tpp) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int c = 0;
  for (int h = 0; h < tpp; ++h) c += cnt[h * npad + s];
  cnt_id[perm[s]] = c;
}

// Receivers of each sender in sub-list order (sub-list 0, then 1, ...), written
// to its segment off[sender] of idx.  A workgroup takes kIdxTile consecutive
// sorted senders: it reads kIdxRows rows of every sub-list at a time (a row is
// contiguous over the senders), looks the ids up, and turns the tile around
// through LDS, so that a wavefront writes one sender's receivers side by side.
// Ten rows are in flight a thread: waiting for each (ids and all) took 531 us
// where this takes 488 us (1,000,000 particles, 113 pairs each: 1.35 GB at
// 2.8 TB/s, bound by stores that start and end inside cache lines); a thread
// per sender, which wrote 4 B here and there, took 4,824 us.
constexpr int kIdxTile = 32, kIdxRows = 40;

template <int TPP>
__global__ __launch_bounds__(kBlock) void k_write_idx(
    const int32_t* __restrict__ perm, const int32_t* __restrict__ cnt,
    const int32_t* __restrict__ ell, const int64_t* __restrict__ off, int32_t* __restrict__ idx,
    int64_t max_occ, int n, int npad, int lane_width) {
  __shared__ int32_t tile[TPP][kIdxRows][kIdxTile + 1];
  __shared__ int32_t own[kIdxTile];  // the sender
  __shared__ int64_t seg[kIdxTile];  // its segment
  __shared__ int32_t count[TPP][kIdxTile];
  __shared__ int rows;  // the longest sub-list of the tile
  const int s0 = blockIdx.x * kIdxTile;
  const int ns = min(kIdxTile, n - s0);
  if (threadIdx.x == 0) rows = 0;
  __syncthreads();
  if (threadIdx.x < kIdxTile) {
    const int c = threadIdx.x;
    own[c] = c < ns ? perm[s0 + c] : 0;
    seg[c] = c < ns ? off[own[c]] : 0;
    for (int h = 0; h < TPP; ++h) count[h][c] = c < ns ? cnt[h * npad + s0 + c] : 0;
    atomicMax(&rows, count[0][c]);  // sub-list 0 is never shorter than the others
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int kLoads = 10;  // rows a thread has in flight
  static_assert(TPP * kIdxRows * kIdxTile % (kLoads * kBlock) == 0, "whole batches of loads");
  for (int k0 = 0; k0 < rows; k0 += kIdxRows) {
    for (int t0 = threadIdx.x; t0 < TPP * kIdxRows * kIdxTile; t0 += kLoads * kBlock) {
      int32_t j[kLoads];
#pragma unroll
      for (int q = 0; q < kLoads; ++q) {
        const int t = t0 + q * kBlock;
        const int c = t % kIdxTile, k = k0 + t / kIdxTile % kIdxRows, h = t / (kIdxTile * kIdxRows);
        j[q] = -1;
        if (k < count[h][c]) j[q] = ell[((int64_t)h * lane_width + k) * npad + s0 + c];
      }
#pragma unroll
      for (int q = 0; q < kLoads; ++q)
        if (j[q] >= 0) j[q] = perm[j[q]];
#pragma unroll
      for (int q = 0; q < kLoads; ++q) {
        const int t = t0 + q * kBlock;
        tile[t / (kIdxTile * kIdxRows)][t / kIdxTile % kIdxRows][t % kIdxTile] = j[q];
      }
    }
    __syncthreads();
    for (int c = wave; c < ns; c += kBlock / 64) {
      const int a = own[c];
      int64_t p0 = seg[c] + k0;
#pragma unroll
      for (int h = 0; h < TPP; ++h) {
        const int m = count[h][c];
        const int64_t p = p0 + lane;
        if (lane < kIdxRows && k0 + lane < m && p < max_occ) {
          idx[p] = tile[h][lane][c];
          idx[max_occ + p] = a;
        }
        p0 += m;
      }
    }
    __syncthreads();
  }
}

// Entries *total .. max_occ of both rows hold n.
constexpr int kPadBlocks = 2048;
__global__ __launch_bounds__(kBlock) void k_pad_idx(int32_t* __restrict__ idx, int64_t max_occ,
                                                    const int64_t* __restrict__ total, int n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t p = *total + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < max_occ;
       p += stride) {
    idx[p] = n;
    idx[max_occ + p] = n;
  }
}

static unsigned pad_blocks(int64_t max_occ) {
  const int64_t b = cdiv(max_occ, kBlock);
  return (unsigned)(b < kPadBlocks ? b : kPadBlocks);
}

// idx of a skin list: the pairs of each sender (sub-list order) that pass the
// exact reference predicate at positions r.  WRITE = false counts them per
// original id; WRITE = true stores them from the scanned offsets.
struct SkinIdxArgs {
  const float* r;
  const int32_t *perm, *cnt, *ell;
  int32_t* cnt_id;
  const int64_t* off;
  int32_t* idx;
  int64_t max_occ;
  float box[3], half[3];
  float cutoff_sq;
  int n, npad, tpp, lane_width;
  // reference cells no wider than the cutoff: the pair's reference cells must
  // be adjacent (the grid of the reference's candidate search)
};

template <int DIM, bool WRITE>
__global__ void k_skin_pairs(SkinIdxArgs a) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.n) return;
  const int i = a.perm[s];
  const float4 ri = load_pos<DIM>(a.r, i);
  int64_t p = WRITE ? a.off[i] : 0;
  for (int h = 0; h < a.tpp; ++h) {
    const int c = a.cnt[h * a.npad + s];
    const int32_t* lst = a.ell + ((int64_t)h * a.lane_width) * a.npad + s;
    for (int k = 0; k < c; ++k) {
      const int j = a.perm[lst[(int64_t)k * a.npad]];
      if (!(metric_sq_exact<DIM>(ri, load_pos<DIM>(a.r, j), a.box, a.half) < a.cutoff_sq))
        continue;
      if (WRITE && p < a.max_occ) {
        a.idx[p] = j;
        a.idx[a.max_occ + p] = i;
      }
      ++p;
    }
  }
  if (!WRITE) a.cnt_id[i] = (int32_t)p;
}

__global__ void k_chunk_budget(const int64_t* __restrict__ off, int n, int64_t n_sub,
                               int64_t budget, int64_t* __restrict__ info) {
  int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t lo = k * n_sub;
  if (lo >= n) return;
  int64_t hi = lo + n_sub < n ? lo + n_sub : n;
  if (off[hi] - off[lo] > budget) {
    atomicOr((unsigned long long*)&info[0], (unsigned long long)SPH_CELL_LIST_OVERFLOW);
    atomicAdd((unsigned long long*)&info[6], 1ull);
  }
}

Grid make_grid(const sph_nl_config& c) {
  Grid g;
  for (int d = 0; d < 3; ++d) {
    g.cs[d] = c.cell_size[d];
    g.cps[d] = c.cps[d] > 0 ? c.cps[d] : 1;
  }
  g.use_cells = c.use_cells;
  return g;
}

// Kick/drift/wrap of the state fused with the histogram of the new positions;
// resets the error block.
int integrate_and_hash(sph_ws* ws, const float* r, const float* u, const float* dudt,
                       const float* dvdt, float* r_out, float* u_out, float* v_out, float dt,
                       float ctvf, const float* box, const int64_t* prev_info, int64_t* info,
                       hipStream_t st) {
  const auto& c = ws->cfg;
  const int n = c.n;
  Grid g = make_grid(c);
  const bool small = bins_small(n, ws->ncell);
  ws->count_dirty = !small;
  const auto kernel = small
                          ? (c.dim == 2 ? k_integrate_hash<2, false> : k_integrate_hash<3, false>)
                          : (c.dim == 2 ? k_integrate_hash<2, true> : k_integrate_hash<3, true>);
  SPH_LAUNCH(ws, "integrate_hash", st,
             kernel<<<cdiv(n, kBlock), kBlock, 0, st>>>(
                 r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, g, box[0], box[1],
                 c.dim == 3 ? box[2] : 0.0f, ws->cell_count, ws->pcell, ws->pslot, info,
                 prev_info));
  return SPH_OK;
}

// Order of the particles at r by cells and ids: scan of the histogram, scatter,
// per-cell id sort (a small set in one launch, hash included); then (want_pos)
// the sorted positions the pair build reads.
int bin_finish(sph_ws* ws, int bank, const float* r, bool want_pos, const int64_t* prev_info,
               int64_t* info, hipStream_t st) {
  const auto& c = ws->cfg;
  const int n = c.n;
  Bank& B = ws->bank[bank];
  if (bins_small(n, ws->ncell)) {
    const BinSmall b{r, n, make_grid(c), ws->ncell, B.cell_start, B.perm, B.iperm,
                     want_pos ? B.pos : nullptr, nullptr, 0, info, prev_info,
                     c.use_cells ? (int64_t)c.cell_capacity : (int64_t)-1, nullptr};
    if (c.dim == 2)
      SPH_LAUNCH(ws, "bin", st, (k_bin_small<2, false><<<1, kBinThreads, 0, st>>>(b)));
    else
      SPH_LAUNCH(ws, "bin", st, (k_bin_small<3, false><<<1, kBinThreads, 0, st>>>(b)));
    return SPH_OK;
  }
  const int rc = scan<int32_t>(ws, "scan_cells", ws->cell_count, ws->ncell, B.cell_start,
                               (int32_t*)ws->scan_tmp, info,
                               c.use_cells ? (int64_t)c.cell_capacity : (int64_t)-1, nullptr, st);
  if (rc) return rc;
  SPH_LAUNCH(ws, "scatter", st,
             k_scatter<<<cdiv(n, kBlock), kBlock, 0, st>>>(ws->pcell, ws->pslot, B.cell_start,
                                                         ws->unsorted, n));
  SPH_LAUNCH(ws, "cell_sort", st,
             k_cell_sort<3><<<cdiv(ws->ncell * 64, 256), 256, 0, st>>>(
                 B.cell_start, ws->unsorted, B.perm, B.iperm, ws->ncell, nullptr, nullptr,
                 Grid{}, ws->cell_count));
  ws->count_dirty = false;
  if (!want_pos) return SPH_OK;
  if (c.dim == 2)
    SPH_LAUNCH(ws, "gather_pos", st,
               k_gather_pos<2><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, B.perm, B.pos, n));
  else
    SPH_LAUNCH(ws, "gather_pos", st,
               k_gather_pos<3><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, B.perm, B.pos, n));
  return SPH_OK;
}

int bin_particles(sph_ws* ws, int bank, const float* r, const int64_t* prev_info, int64_t* info,
                  hipStream_t st) {
  const auto& c = ws->cfg;
  const int n = c.n;
  Grid g = make_grid(c);
  if (!bins_small(n, ws->ncell)) {
    const auto kernel = c.dim == 2 ? k_hash_count<2> : k_hash_count<3>;
    ws->count_dirty = true;
    SPH_LAUNCH(ws, "hash_count", st,
               kernel<<<cdiv(n, kBlock), kBlock, 0, st>>>(
                   r, n, g, ws->cell_count, ws->pcell, ws->pslot, nullptr, info, prev_info));
  }
  return bin_finish(ws, bank, r, true, prev_info, info, st);
}

// The cell-adjacent image is the minimum image of every pair within the cutoff
// when each side has >= 5 cells (2 cells < box/2).  Both the fast and the exact
// squared distance are then within a few ulp(box) per component of the true
// one (see cut_band).
static bool fast_filter(const sph_nl_config& c) {
  if (!c.use_cells) return false;
  for (int d = 0; d < c.dim; ++d)
    if (c.cps[d] < 5) return false;
  return true;
}

// Where k_nl_tile is the faster build, by the pairs a particle has within reach
// and the particles that a cell then holds (means over the particles).  A
// wavefront spends a piece's time on however few particles the piece has, so
// cells must hold some; and hits past a particle's stage cost its slow path, so
// most lists must fit.  Small sets leave SIMDs idle, where both matter less.  In
// 2D a piece's 64 candidates at a time are two chunks half full for each 9
// particles, which pays until there are pieces for every SIMD: `most` cells.
// Microseconds by the lanes' build and so, noisy lattices, exact lists:
//   3D 9,000 particles, 0.5 a cell 41, 34; 30,000, 1 a cell 37, 40; 1.5 38, 35;
//   59 (252 pairs) 137, 90
//   60,000, 1 a cell 44, 63; 3 46, 39; 27 91, 51; 45 (194 pairs) 141, 135;
//   60 (255 pairs) 122, 163
//   300,000, 2.6 a cell 144, 150; 3.1 142, 128; 28 253, 136; 51 (215 pairs) 432,
//   395; 1,000,000, 2.5 a cell 339, 417; 3 347, 367; 4 344, 305
//   2D 20,000, 2 a cell 19, 20; 3 21, 16; 32 (99 pairs) 58, 25
//   60,000, 3 a cell 21, 25; 4 (14,900 cells) 22, 21; 9 27, 20; 16 (49 pairs) 40, 35
//   100,000, 5 a cell (19,900 cells) 26, 27; 7 30, 24; 16 (49 pairs, 6,200 cells)
//   41, 46; 20 (62 pairs, 5,000 cells) 50, 42
//   145,000, 4 a cell 25, 37; 9 (16,100 cells) 34, 30; 180,000, 9 (19,900) 36, 37
// 5,000 particles, half of them in one 3D cell (650 pairs) 175, 218.
// Returns 0, or the consecutive particles a workgroup takes.  Its four wavefronts
// take in turn the pieces that start there, and it lasts as long as the one with
// the most: 32 leaves most with one; 48, fewer workgroups, is the faster where
// about a piece each still covers them and every SIMD has work (27 a cell 21,952
// particles 32 and 42 us, 97,336 69 and 66, 262,144 147 and 127, 2,097,152 1,024
// and 834, skin lists at 35 a cell 1,199 and 996; 8 a cell 262,144 74 and 79,
// 2,097,152 503 and 521, skin lists at 10 a cell 81 and 83, 535 and 514).
static constexpr double kBall[] = {0.0, 2.0, 3.14, 4.19};
static int tile_pays(int dim, int64_t n, double pairs, const float* cell, float reach,
                     double most) {
  double held = pairs / kBall[dim];
  for (int d = 0; d < dim; ++d) held *= (double)cell[d] / (double)reach;
  if (dim == 3) {
    if (held < (n < 15000 ? 0.2 : n < 40000 ? 0.8 : 2.8) || pairs > (n < 40000 ? 400.0 : 220.0))
      return 0;
    constexpr int kMore = 48;
    const double cell_holds = held * (pairs + 1.0) / pairs;  // the particle itself too
    const double pieces = kMore * std::ceil(cell_holds / tile_rows(3)) / cell_holds;
    return n >= 80000 && pieces <= 5.5 ? kMore : kTileRange;
  }
  const double cells = (double)n / held;
  return held >= 2.3 && cells <= most && (pairs <= 40.0 || cells <= 5200.0) ? kTileRange : 0;
}

// Pairs of a particle within the cutoff, itself apart: as told (sph_ws_tune),
// else as if the particles filled the box.
static double mean_pairs(const sph_ws* ws) {
  const auto& c = ws->cfg;
  if (ws->pairs > 0) return (double)ws->pairs / c.n - (c.mask_self ? 0.0 : 1.0);
  double pairs = kBall[c.dim] * c.n;
  for (int d = 0; d < c.dim; ++d) pairs *= (double)c.cutoff / (double)c.box[d];
  return pairs;
}

// Exact lists: k_nl_tile's filter is the fast one's, and ordered (half) lists
// compare ids candidate by candidate.
static int tile_range(const sph_ws* ws) {
  const auto& c = ws->cfg;
  if (!fast_filter(c) || c.ordered) return 0;
  return tile_pays(c.dim, c.n, mean_pairs(ws), c.cell_size, c.cutoff, 18000.0);
}
// Skin lists, which the lanes build without a band: 2D 48,400 particles 22.8 and
// 17.0 us, 96,100 (9,100 cells) 26.0 and 24.4, 136,900 31.2 and 30.3; Wendland C2
// 14,400 16.6 and 11.7, 57,600 (12,200 cells) 17.3 and 18.9.
static int skin_tile_range(const sph_ws* ws) {
  const auto& c = ws->cfg;
  const float reach = c.cutoff + ws->sk.skin;
  double pairs = mean_pairs(ws);
  for (int d = 0; d < c.dim; ++d) pairs *= (double)reach / (double)c.cutoff;
  return tile_pays(c.dim, c.n, pairs, ws->sk.cell_size, reach, 10000.0);
}

static unsigned build_grid(const sph_ws* ws, int range) {
  const auto& c = ws->cfg;
  const int64_t blocks = range ? cdiv(c.n, range) : cdiv((int64_t)c.n * ws->tpp, kBlock);
  return xcd_grid(blocks, ws->xcd_remap);
}

int build_pairs(sph_ws* ws, int bank, int64_t* info, hipStream_t st) {
  const auto& c = ws->cfg;
  Bank& B = ws->bank[bank];
  BuildArgs a;
  a.pos = B.pos;
  a.cell_start = B.cell_start;
  a.perm = B.perm;
  a.ell = B.ell;
  a.cnt = B.cnt;
  a.info = info;
  a.g = make_grid(c);
  for (int d = 0; d < 3; ++d) {
    a.box[d] = c.box[d];
    a.half[d] = c.box[d] * 0.5f;
  }
  a.cutoff_sq = c.cutoff_sq;
  a.n = c.n;
  a.npad = ws->npad;
  a.lane_width = ws->lane_width;
  a.mask_self = c.mask_self;
  a.part = ws->part_build;
  // 3^d x cell capacity entries per particle never truncate; a narrower
  // buffer reports a truncated sub-list as an overflow
  a.trunc_bits = ws->ell_overflow ? SPH_NEIGHBOR_LIST_OVERFLOW : 0;
  a.gate = nullptr;
  a.remap = ws->xcd_remap;
  a.fast = fast_filter(c);
  a.range = tile_range(ws);
  cut_band(c, &a.lo, &a.hi);
  a.tile = tile_band(a.box, a.g.cs, c.dim, c.cutoff, a.cutoff_sq);
  constexpr int T2 = tpp_of(2), T3 = tpp_of(3);
  const bool d2 = c.dim == 2;
  const auto kernel =
      a.range     ? (d2 ? k_nl_tile<2, T2> : k_nl_tile<3, T3>)
      : c.ordered ? (d2 ? k_nl_build<2, T2, true, true> : k_nl_build<3, T3, true, true>)
                  : (d2 ? k_nl_build<2, T2, false, true> : k_nl_build<3, T3, false, true>);
  SPH_LAUNCH(ws, "nl_build", st, (kernel<<<build_grid(ws, a.range), kBlock, 0, st>>>(a)));
  return SPH_OK;
}

// What an exact build leaves to reduce: occupancy info[1], largest list
// info[3], and the overflow bit when max_occupancy >= 0.
Reduce build_tail(sph_ws* ws, int64_t max_occupancy, int64_t* info) {
  const int blocks = (int)build_grid(ws, tile_range(ws));
  return Reduce{ws->part_build, blocks, &info[1], &info[3], info, max_occupancy, nullptr, nullptr};
}

// The exact-predicate band of the pair build: squared distances (fp32, minimum
// image, explicit FMA) below lo are inside the cutoff, at or above hi outside;
// in between the reference metric decides.  The two differ by a few ulp(box)
// per component, which `band` bounds with a wide margin.
void cut_band(const sph_nl_config& c, float* lo, float* hi) {
  float maxbox = 0.0f;
  for (int d = 0; d < c.dim; ++d) maxbox = c.box[d] > maxbox ? c.box[d] : maxbox;
  const float ulp_box = std::nextafter(maxbox, INFINITY) - maxbox;
  const float ulp_c2 = std::nextafter(c.cutoff_sq, INFINITY) - c.cutoff_sq;
  const float band = 64.0f * c.cutoff * ulp_box + 16.0f * ulp_c2;
  *lo = c.cutoff_sq - band;
  *hi = c.cutoff_sq + band;
}

static Grid skin_grid(const sph_ws* ws) {
  Grid g;
  for (int d = 0; d < 3; ++d) {
    g.cs[d] = ws->sk.cell_size[d];
    g.cps[d] = ws->sk.cps[d];
  }
  g.use_cells = 1;
  return g;
}

// First half of a skin-list step: kick/drift with the rebuild test and the
// reference-grid occupancy; then, only if a rebuild was requested, the
// skin-grid binning (hash, scan, scatter, per-cell sort).
int skin_begin(sph_ws* ws, const float* r, const float* u, const float* dudt, const float* dvdt,
               float* r_out, float* u_out, float* v_out, float dt, float ctvf, const float* box,
               const int64_t* prev_info, int64_t* info, hipStream_t st) {
  const auto& c = ws->cfg;
  auto& S = ws->sk;
  const int n = c.n;
  const Grid g = make_grid(c);
  const Grid gs = skin_grid(ws);
  const unsigned nb = (unsigned)cdiv(n, kBlock);
  ws->count_dirty = true;
  if (c.dim == 2)
    SPH_LAUNCH(ws, "integrate_skin", st,
               k_integrate_skin<2><<<nb, kBlock, 0, st>>>(
                   r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, g, box[0], box[1], 0.0f,
                   ws->cell_count, S.posb, S.trigger_sq, S.flag, info, prev_info));
  else
    SPH_LAUNCH(ws, "integrate_skin", st,
               k_integrate_skin<3><<<nb, kBlock, 0, st>>>(
                   r, u, dudt, dvdt, r_out, u_out, v_out, n, dt, ctvf, g, box[0], box[1], box[2],
                   ws->cell_count, S.posb, S.trigger_sq, S.flag, info, prev_info));
  if (bins_small(n, S.ncell)) {
    const BinSmall b{r_out, n, gs, S.ncell, S.b.cell_start, S.b.perm, S.b.iperm, nullptr,
                     ws->cell_count, ws->ncell, info, nullptr, (int64_t)c.cell_capacity, S.flag};
    if (c.dim == 2)
      SPH_LAUNCH(ws, "skin_bin", st, (k_bin_small<2, true><<<1, kBinThreads, 0, st>>>(b)));
    else
      SPH_LAUNCH(ws, "skin_bin", st, (k_bin_small<3, true><<<1, kBinThreads, 0, st>>>(b)));
    ws->count_dirty = false;
    return SPH_OK;
  }
  const int cb = (int)cdiv(ws->ncell, kCellsBlock);
  S.count_dirty = true;
  if (c.dim == 2)
    SPH_LAUNCH(ws, "skin_hash", st,
               k_skin_hash<2><<<nb + cb, kBlock, 0, st>>>(r_out, n, gs, S.cell_count, ws->pcell,
                                                         ws->pslot, S.flag, ws->cell_count,
                                                         ws->ncell, cb, info,
                                                         (int64_t)c.cell_capacity));
  else
    SPH_LAUNCH(ws, "skin_hash", st,
               k_skin_hash<3><<<nb + cb, kBlock, 0, st>>>(r_out, n, gs, S.cell_count, ws->pcell,
                                                         ws->pslot, S.flag, ws->cell_count,
                                                         ws->ncell, cb, info,
                                                         (int64_t)c.cell_capacity));
  ws->count_dirty = false;
  const int rc = scan<int32_t>(ws, "skin_scan", S.cell_count, S.ncell, S.b.cell_start,
                               (int32_t*)ws->scan_tmp, nullptr, -1, S.flag, st);
  if (rc) return rc;
  SPH_LAUNCH(ws, "skin_scatter", st,
             k_scatter<<<nb, kBlock, 0, st>>>(ws->pcell, ws->pslot, S.b.cell_start, ws->unsorted,
                                              n, S.flag));
  if (c.dim == 2)
    SPH_LAUNCH(ws, "skin_sort", st,
               k_cell_sort<2><<<cdiv(S.ncell * 64, 256), 256, 0, st>>>(
                   S.b.cell_start, ws->unsorted, S.b.perm, S.b.iperm, S.ncell, S.flag, r_out, gs,
                   S.cell_count));
  else
    SPH_LAUNCH(ws, "skin_sort", st,
               k_cell_sort<3><<<cdiv(S.ncell * 64, 256), 256, 0, st>>>(
                   S.b.cell_start, ws->unsorted, S.b.perm, S.b.iperm, S.ncell, S.flag, r_out, gs,
                   S.cell_count));
  S.count_dirty = false;
  return SPH_OK;
}

// Second half: the skin pair lists (cutoff + skin) from the sorted build
// positions, only if a rebuild was requested.  Pair totals are not counted
// here (the sweeps count the pairs inside the cutoff); info[7] receives the
// largest list of one particle, and an overflowing sub-list raises
// SPH_NEIGHBOR_LIST_OVERFLOW so the caller re-allocates.
static BuildArgs skin_build_args(sph_ws* ws, int64_t* info) {
  const auto& c = ws->cfg;
  auto& S = ws->sk;
  BuildArgs a;
  a.pos = S.b.pos;
  a.cell_start = S.b.cell_start;
  a.perm = S.b.perm;
  a.ell = S.b.ell;
  a.cnt = S.b.cnt;
  a.info = info;
  a.g = skin_grid(ws);
  for (int d = 0; d < 3; ++d) {
    a.box[d] = c.box[d];
    a.half[d] = c.box[d] * 0.5f;
  }
  a.cutoff_sq = S.reach_sq;
  a.fast = 1;
  a.range = skin_tile_range(ws);
  a.lo = a.hi = S.reach_sq;
  a.tile = tile_band(a.box, a.g.cs, c.dim, c.cutoff + S.skin, a.cutoff_sq);
  a.n = c.n;
  a.npad = ws->npad;
  a.lane_width = S.lane_width;
  a.mask_self = c.mask_self;
  a.part = ws->part_build;
  a.trunc_bits = SPH_NEIGHBOR_LIST_OVERFLOW;
  a.gate = S.flag;
  a.remap = ws->xcd_remap;
  return a;
}

int skin_build(sph_ws* ws, int64_t* info, hipStream_t st) {
  const auto& c = ws->cfg;
  auto& S = ws->sk;
  const BuildArgs a = skin_build_args(ws, info);
  constexpr int T2 = tpp_of(2), T3 = tpp_of(3);
  const bool d2 = c.dim == 2;
  const auto kernel =
      a.range ? (d2 ? k_nl_tile<2, T2> : k_nl_tile<3, T3>)
              : (d2 ? k_nl_build<2, T2, false, false> : k_nl_build<3, T3, false, false>);
  SPH_LAUNCH(ws, "skin_build", st, (kernel<<<build_grid(ws, a.range), kBlock, 0, st>>>(a)));
  return SPH_OK;
}

// What a skin build leaves to reduce: the largest list of one particle ->
// info[7] (only on a rebuild).
Reduce skin_build_tail(sph_ws* ws, int64_t* info) {
  const int blocks = (int)build_grid(ws, skin_tile_range(ws));
  return Reduce{ws->part_build, blocks, nullptr, &info[7], info, -1, ws->sk.flag, nullptr};
}

// End of a skin-list step: occupancy and largest list from the counting
// density sweep's partials, the overflow bit, and the rebuild request is consumed.
Reduce skin_step_tail(sph_ws* ws, int64_t max_occupancy, int64_t* info) {
  const int blocks = (int)xcd_grid(cdiv((int64_t)ws->cfg.n * ws->tpp, kBlock), ws->xcd_remap);
  return Reduce{ws->part_sweep, blocks, &info[1], &info[3], info, max_occupancy, nullptr,
                ws->sk.flag};
}

// pair counts per original id and their exclusive scan (off64[0..N])
int pair_offsets(sph_ws* ws, int bank, hipStream_t st) {
  const int n = ws->cfg.n;
  Bank& B = ws->bank[bank];
  SPH_LAUNCH(ws, "counts_orig", st,
             k_counts_orig<<<cdiv(n, kBlock), kBlock, 0, st>>>(B.perm, B.cnt, ws->cnt_id, n,
                                                             ws->npad, ws->tpp));
  return scan<int64_t>(ws, "scan_pairs", ws->cnt_id, n, ws->off64, ws->scan_tmp, nullptr, -1,
                       nullptr, st);
}

// ------------------------------------------------------------ ensembles
// Batched forms of the skin-step phases above (skin_begin, skin_build): one
// launch serves every member.  Per-member arguments are those the
// single-simulation launches pass; the bodies are shared.  The reductions that
// ride in a single simulation's sweeps (skin_build_tail, skin_step_tail) are
// launches of their own here, as is the reference-grid occupancy.
struct EnsInteg {
  const float *r, *u, *dudt, *dvdt;
  float *r_out, *u_out, *v_out;
  int n;
  float dt, ctvf;
  Grid g;
  float box[3];
  int32_t* cell_count;
  const float4* posb;
  float trigger_sq;
  int32_t* flag;
};

struct EnsCells {
  int32_t* count;
  int64_t ncell;
  int64_t* info;
  const int64_t* prev;
  int64_t capacity;
};

struct EnsBin {  // skin-grid binning, all gated on the member's rebuild flag
  const float* r;
  int n;
  Grid g;
  int32_t *cell_count, *pcell, *pslot, *flag, *cell_start;
  int64_t ncell;
  int32_t *unsorted, *perm, *iperm;
};

struct EnsNL {
  int n = 0;
  std::vector<sph_ws*> ws;
  EnsInteg* integ = nullptr;
  EnsCells* cells = nullptr;
  EnsBin* bin = nullptr;
  BuildArgs* build = nullptr;
  Reduce* red_build = nullptr;
  Reduce* red_sweep = nullptr;
};

template <int DIM>
__global__ void k_integrate_skin_ens(const EnsInteg* __restrict__ t,
                                     const EnsBlock* __restrict__ map) {
  const EnsBlock m = map[blockIdx.x];
  if (m.sim < 0) return;
  const EnsInteg& a = t[m.sim];
  integrate_skin_body<DIM>(a.r, a.u, a.dudt, a.dvdt, a.r_out, a.u_out, a.v_out, a.n, a.dt,
                           a.ctvf, a.g, a.box[0], a.box[1], a.box[2], a.cell_count, a.posb,
                           a.trigger_sq, a.flag, m.blk);
}

// one workgroup per member
__global__ __launch_bounds__(kCellsThreads) void k_cells_max_ens(const EnsCells* __restrict__ t) {
  const EnsCells& a = t[blockIdx.x];
  cells_max_body(a.count, a.ncell, a.info, a.prev, a.capacity);
}

template <int DIM>
__global__ void k_hash_count_ens(const EnsBin* __restrict__ t, const EnsBlock* __restrict__ map) {
  const EnsBlock m = map[blockIdx.x];
  if (m.sim < 0) return;
  const EnsBin& a = t[m.sim];
  hash_count_body<DIM>(a.r, a.n, a.g, a.cell_count, a.pcell, a.pslot, a.flag, m.blk);
}

// one workgroup per member
__global__ __launch_bounds__(kScanThreads) void k_scan_ens(const EnsBin* __restrict__ t) {
  const EnsBin& a = t[blockIdx.x];
  scan_body<int32_t>(a.cell_count, a.ncell, cdiv(a.ncell, kScanTile) * kScanTile, nullptr,
                     a.cell_start, nullptr, -1, a.flag, 0, 1);
}

__global__ void k_scatter_ens(const EnsBin* __restrict__ t, const EnsBlock* __restrict__ map) {
  const EnsBlock m = map[blockIdx.x];
  if (m.sim < 0) return;
  const EnsBin& a = t[m.sim];
  scatter_body(a.pcell, a.pslot, a.cell_start, a.unsorted, a.n, a.flag, m.blk);
}

template <int DIM>
__global__ __launch_bounds__(256) void k_cell_sort_ens(const EnsBin* __restrict__ t,
                                                       const EnsBlock* __restrict__ map) {
  const EnsBlock m = map[blockIdx.x];
  if (m.sim < 0) return;
  const EnsBin& a = t[m.sim];
  cell_sort_body<DIM>(a.cell_start, a.unsorted, a.perm, a.iperm, a.ncell, a.flag, m.blk, a.r,
                      a.g, a.cell_count);
}

// The members of a 2D ensemble are many particles together, where the lanes'
// build is the faster one (see skin_tile_range()).
template <int DIM, int TPP>
__global__ __launch_bounds__(kBlock, 6) void k_nl_build_ens(const BuildArgs* __restrict__ t,
                                                            const EnsBlock* __restrict__ map) {
  const EnsBlock m = map[blockIdx.x];
  if (m.sim < 0) return;
  // a block of the map is kBlock / TPP particles
  if constexpr (DIM == 3)
    nl_tile_body<DIM, TPP>((ColdArgs*)(t + m.sim), m.blk, kBlock / TPP);
  else
    nl_build_body<DIM, TPP, false, false>(t[m.sim], m.blk);
}

// one workgroup per member
__global__ __launch_bounds__(kReduceThreads) void k_reduce_parts_ens(
    const Reduce* __restrict__ t) {
  reduce_parts_body<kReduceThreads>(t[blockIdx.x]);
}

template <typename T>
static int upload(const std::vector<T>& h, T** d) {
  hipError_t e = hipMalloc((void**)d, sizeof(T) * h.size());
  if (e != hipSuccess) return hip_fail(e, "ensemble tables");
  e = hipMemcpy(*d, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice);
  if (e != hipSuccess) return hip_fail(e, "ensemble tables");
  return SPH_OK;
}

int ens_nl_create(const std::vector<EnsMember>& members, EnsNL** out) {
  const int n = (int)members.size();
  std::vector<EnsInteg> integ(n);
  std::vector<EnsCells> cells(n);
  std::vector<EnsBin> bin(n);
  std::vector<BuildArgs> build(n);
  std::vector<Reduce> rb(n), rs(n);
  for (int k = 0; k < n; ++k) {
    const EnsMember& m = members[k];
    sph_ws* ws = m.ws;
    const auto& c = ws->cfg;
    auto& S = ws->sk;
    const int64_t lane_blocks = cdiv((int64_t)c.n * ws->tpp, kBlock);
    integ[k] = EnsInteg{m.in.r, m.in.u, m.in.dudt, m.in.dvdt, m.r_out, m.out.u, m.out.v, c.n,
                        m.dt, m.ctvf, make_grid(c), {m.prm.box[0], m.prm.box[1], m.prm.box[2]},
                        ws->cell_count, S.posb, S.trigger_sq, S.flag};
    cells[k] = EnsCells{ws->cell_count, ws->ncell, m.info, m.prev_info,
                        (int64_t)c.cell_capacity};
    bin[k] = EnsBin{m.r_out, c.n, skin_grid(ws), S.cell_count, ws->pcell, ws->pslot, S.flag,
                    S.b.cell_start, S.ncell, ws->unsorted, S.b.perm, S.b.iperm};
    build[k] = skin_build_args(ws, m.info);
    rb[k] = Reduce{ws->part_build, (int)lane_blocks, nullptr, &m.info[7], m.info, -1, S.flag,
                      nullptr};
    rs[k] = Reduce{ws->part_sweep, (int)lane_blocks, &m.info[1], &m.info[3], m.info,
                      m.max_occupancy, nullptr, S.flag};
  }
  EnsNL* t = new EnsNL;
  t->n = n;
  for (const EnsMember& m : members) t->ws.push_back(m.ws);
  int rc = upload(integ, &t->integ);
  if (!rc) rc = upload(cells, &t->cells);
  if (!rc) rc = upload(bin, &t->bin);
  if (!rc) rc = upload(build, &t->build);
  if (!rc) rc = upload(rb, &t->red_build);
  if (!rc) rc = upload(rs, &t->red_sweep);
  if (rc) {
    ens_nl_destroy(t);
    return rc;
  }
  *out = t;
  return SPH_OK;
}

void ens_nl_destroy(EnsNL* t) {
  if (!t) return;
  (void)hipFree(t->integ);
  (void)hipFree(t->cells);
  (void)hipFree(t->bin);
  (void)hipFree(t->build);
  (void)hipFree(t->red_build);
  (void)hipFree(t->red_sweep);
  delete t;
}

int ens_skin_begin(EnsNL* t, int dim, const EnsMap& part, const EnsMap& cells, sph_ws* prof,
                   hipStream_t st) {
  for (sph_ws* ws : t->ws) ws->count_dirty = true;
  if (dim == 2)
    SPH_LAUNCH(prof, "ens_integrate_skin", st,
               k_integrate_skin_ens<2><<<part.blocks, kBlock, 0, st>>>(t->integ, part.d));
  else
    SPH_LAUNCH(prof, "ens_integrate_skin", st,
               k_integrate_skin_ens<3><<<part.blocks, kBlock, 0, st>>>(t->integ, part.d));
  SPH_LAUNCH(prof, "ens_cells_max", st,
             k_cells_max_ens<<<t->n, kCellsThreads, 0, st>>>(t->cells));
  for (sph_ws* ws : t->ws) {
    ws->count_dirty = false;
    ws->sk.count_dirty = true;
  }
  if (dim == 2)
    SPH_LAUNCH(prof, "ens_skin_hash", st,
               k_hash_count_ens<2><<<part.blocks, kBlock, 0, st>>>(t->bin, part.d));
  else
    SPH_LAUNCH(prof, "ens_skin_hash", st,
               k_hash_count_ens<3><<<part.blocks, kBlock, 0, st>>>(t->bin, part.d));
  SPH_LAUNCH(prof, "ens_skin_scan", st, k_scan_ens<<<t->n, kScanThreads, 0, st>>>(t->bin));
  SPH_LAUNCH(prof, "ens_skin_scatter", st,
             k_scatter_ens<<<part.blocks, kBlock, 0, st>>>(t->bin, part.d));
  if (dim == 2)
    SPH_LAUNCH(prof, "ens_skin_sort", st,
               k_cell_sort_ens<2><<<cells.blocks, 256, 0, st>>>(t->bin, cells.d));
  else
    SPH_LAUNCH(prof, "ens_skin_sort", st,
               k_cell_sort_ens<3><<<cells.blocks, 256, 0, st>>>(t->bin, cells.d));
  for (sph_ws* ws : t->ws) ws->sk.count_dirty = false;
  return SPH_OK;
}

int ens_skin_build(EnsNL* t, int dim, const EnsMap& lanes, sph_ws* prof, hipStream_t st) {
  constexpr int T2 = tpp_of(2), T3 = tpp_of(3);
  if (dim == 2)
    SPH_LAUNCH(prof, "ens_skin_build", st,
               (k_nl_build_ens<2, T2><<<lanes.blocks, kBlock, 0, st>>>(t->build, lanes.d)));
  else
    SPH_LAUNCH(prof, "ens_skin_build", st,
               (k_nl_build_ens<3, T3><<<lanes.blocks, kBlock, 0, st>>>(t->build, lanes.d)));
  SPH_LAUNCH(prof, "ens_reduce_skin", st,
             k_reduce_parts_ens<<<t->n, kReduceThreads, 0, st>>>(t->red_build));
  return SPH_OK;
}

int ens_skin_finish(EnsNL* t, sph_ws* prof, hipStream_t st) {
  SPH_LAUNCH(prof, "ens_reduce_pairs", st,
             k_reduce_parts_ens<<<t->n, kReduceThreads, 0, st>>>(t->red_sweep));
  return SPH_OK;
}

}  // namespace sph

using namespace sph;

static int check_ws(sph_ws* ws, int bank) {
  if (!ws) { set_error("null workspace"); return SPH_ERR_ARG; }
  if (bank < 0 || bank > 1) { set_error("bank must be 0 or 1"); return SPH_ERR_ARG; }
  return SPH_OK;
}

namespace sph {
// Grid of a cell-occupancy count; false (with the error set) on a bad argument.
static bool fill_grid(const char* who, int32_t dim, int32_t n, const float* r,
                      const float* cell_size, const int32_t* cps, const int64_t* info, Grid* g,
                      int64_t* nc) {
  if (!r || !cell_size || !cps || !info || n < 0 || (dim != 2 && dim != 3)) {
    set_error(std::string(who) + ": bad argument");
    return false;
  }
  *nc = 1;
  for (int d = 0; d < 3; ++d) {
    g->cs[d] = d < dim ? cell_size[d] : 1.0f;
    g->cps[d] = d < dim ? cps[d] : 1;
    if (g->cps[d] < 1) { set_error("cps must be >= 1"); return false; }
    *nc *= g->cps[d];
  }
  g->use_cells = 1;
  return true;
}

// Clears `counts` (nc cells), histograms r into it and writes the largest
// count to info[2]; every buffer is cleared by a kernel, none by a memset.
static int fill_max_run(int32_t dim, int32_t n, const float* r, const Grid& g, int64_t nc,
                        int32_t* counts, int64_t* info, hipStream_t st) {
  sph_ws* ws = nullptr;  // no profiling without a workspace
  SPH_LAUNCH(ws, "fill", st, k_fill<int32_t><<<cdiv(nc, kBlock), kBlock, 0, st>>>(counts, nc, 0));
  SPH_LAUNCH(ws, "fill", st, k_fill<int64_t><<<1, 64, 0, st>>>(info + 2, 1, 0));
  if (n > 0) {
    if (dim == 2)
      SPH_LAUNCH(ws, "hash_count", st,
                 k_hash_count<2><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, n, g, counts, nullptr,
                                                                   nullptr, nullptr));
    else
      SPH_LAUNCH(ws, "hash_count", st,
                 k_hash_count<3><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, n, g, counts, nullptr,
                                                                   nullptr, nullptr));
  }
  int64_t blocks = cdiv(nc, kBlock);
  blocks = blocks > 1024 ? 1024 : blocks;
  SPH_LAUNCH(ws, "max_reduce", st, k_max_reduce<<<blocks, kBlock, 0, st>>>(counts, nc, info + 2));
  return SPH_OK;
}

// Cell counts of sph_nl_fill_max_static: one copy per GPU, held until the
// process ends.  Host code never passes this name to a kernel (on the host it
// is a stand-in, not a device address); it uses the per-device address that
// hipGetSymbolAddress returns.
static __device__ __align__(256) int32_t scratch[SPH_FILL_MAX_STATIC_CELLS];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static int32_t* g_scratch_ptr[kMaxDevices];  // nullptr until looked up on that device

// Device address of `scratch` on the current device, looked up once per device.
static int scratch_of_current_device(int32_t** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("sph_nl_fill_max_static: no current HIP device");
    return SPH_ERR_HIP;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      set_error(std::string("sph_nl_fill_max_static: hipGetSymbolAddress: ") +
                hipGetErrorString(e));
      return SPH_ERR_HIP;
    }
    g_scratch_ptr[dev] = static_cast<int32_t*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return SPH_OK;
}

// ----------------------------------------------------------- dense cell list
// Slot of the particle at sorted position s (cell-major, ascending id inside a
// cell): cell * capacity + s mod capacity, the scatter index of
// partition.py:368-385.  A cell's particles take consecutive slots from its
// first sorted position mod capacity, wrapping inside the cell, so up to
// `capacity` of them never collide.  In an overflowing cell the particle
// capacity places later in the cell takes the slot (the later scatter update
// wins), so every slot has exactly one writer.
__device__ __forceinline__ int64_t cell_list_slot(const int32_t* __restrict__ perm,
                                                  const int32_t* __restrict__ pcell,
                                                  const int32_t* __restrict__ cell_start, int s,
                                                  int64_t cap, int* id) {
  *id = perm[s];
  const int h = pcell[*id];
  if ((int64_t)s + cap < (int64_t)cell_start[h + 1]) return -1;  // overwritten later
  return (int64_t)h * cap + s % cap;
}

template <int DIM>
__global__ void k_cell_list_fill(const float* __restrict__ r, const int32_t* __restrict__ perm,
                                 const int32_t* __restrict__ pcell,
                                 const int32_t* __restrict__ cell_start, int n, int64_t cap,
                                 float* __restrict__ pos_buf, int32_t* __restrict__ id_buf) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  int id;
  const int64_t slot = cell_list_slot(perm, pcell, cell_start, s, cap, &id);
  if (slot < 0) return;
  id_buf[slot] = id;
#pragma unroll
  for (int d = 0; d < DIM; ++d) pos_buf[slot * DIM + d] = r[(int64_t)id * DIM + d];
}

// One 32-bit word of a per-particle side array (`width` words per particle).
__global__ void k_cell_list_named(const uint32_t* __restrict__ src, int width,
                                  const int32_t* __restrict__ perm,
                                  const int32_t* __restrict__ pcell,
                                  const int32_t* __restrict__ cell_start, int n, int64_t cap,
                                  uint32_t* __restrict__ dst) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)n * width) return;
  const int s = (int)(t / width), w = (int)(t - (int64_t)s * width);
  int id;
  const int64_t slot = cell_list_slot(perm, pcell, cell_start, s, cap, &id);
  if (slot < 0) return;
  dst[slot * width + w] = src[(int64_t)id * width + w];
}
}  // namespace sph

extern "C" int sph_nl_fill_max(int32_t dim, int32_t n, const float* r, const float* cell_size,
                               const int32_t* cps, int32_t* counts, int64_t* info,
                               hipStream_t st) {
  Grid g;
  int64_t nc = 0;
  if (!counts) { set_error("sph_nl_fill_max: bad argument"); return SPH_ERR_ARG; }
  if (!fill_grid("sph_nl_fill_max", dim, n, r, cell_size, cps, info, &g, &nc)) return SPH_ERR_ARG;
  return fill_max_run(dim, n, r, g, nc, counts, info, st);
}

extern "C" int sph_nl_fill_max_static(int32_t dim, int32_t n, const float* r,
                                      const float* cell_size, const int32_t* cps, int64_t* info,
                                      hipStream_t st) {
  Grid g;
  int64_t nc = 0;
  if (!fill_grid("sph_nl_fill_max_static", dim, n, r, cell_size, cps, info, &g, &nc))
    return SPH_ERR_ARG;
  if (nc > SPH_FILL_MAX_STATIC_CELLS) {
    set_error("sph_nl_fill_max_static: the grid has " + std::to_string(nc) +
              " cells, more than the " + std::to_string(SPH_FILL_MAX_STATIC_CELLS) +
              " its static scratch holds (use sph_nl_fill_max with caller scratch)");
    return SPH_ERR_SIZE;
  }
  int32_t* counts = nullptr;
  const int rc = scratch_of_current_device(&counts);
  if (rc != SPH_OK) return rc;
  return fill_max_run(dim, n, r, g, nc, counts, info, st);
}

extern "C" size_t sph_cell_list_work_bytes(int64_t n, int64_t cell_count) {
  if (n < 0 || cell_count < 1) return 0;
  // counts, cell starts, cell and arrival slot per particle, arrivals, sorted ids, inverse
  return (size_t)(2 * cell_count + 1 + 5 * n) * sizeof(int32_t);
}

extern "C" int sph_cell_list(int32_t dim, int32_t n, const float* r, const float* cell_size,
                             const int32_t* cps, int64_t capacity, float* position_buffer,
                             int32_t* id_buffer, int32_t n_named, const uint32_t* const* named,
                             const int32_t* named_width, const uint32_t* named_fill,
                             uint32_t* const* named_buffer, void* work, size_t work_bytes,
                             int64_t* info, hipStream_t st) {
  Grid g;
  int64_t nc = 0;
  if (!fill_grid("sph_cell_list", dim, n, r, cell_size, cps, info, &g, &nc)) return SPH_ERR_ARG;
  if (!position_buffer || !id_buffer || !work || n_named < 0 ||
      (n_named > 0 && (!named || !named_width || !named_fill || !named_buffer))) {
    set_error("sph_cell_list: bad argument");
    return SPH_ERR_ARG;
  }
  if (nc > INT32_MAX) { set_error("sph_cell_list: more than 2^31 - 1 cells"); return SPH_ERR_SIZE; }
  if (capacity < 1 || nc * capacity > INT64_MAX / 4 / dim) {
    set_error("sph_cell_list: capacity must be >= 1 and the buffers addressable");
    return SPH_ERR_ARG;
  }
  if (work_bytes < sph_cell_list_work_bytes(n, nc)) {
    set_error("sph_cell_list: work buffer smaller than sph_cell_list_work_bytes");
    return SPH_ERR_SIZE;
  }
  for (int b = 0; b < n_named; ++b)
    if (!named[b] || !named_buffer[b] || named_width[b] < 1) {
      set_error("sph_cell_list: bad side array " + std::to_string(b));
      return SPH_ERR_ARG;
    }
  int32_t* counts = static_cast<int32_t*>(work);
  int32_t* start = counts + nc;
  int32_t* pcell = start + nc + 1;
  int32_t* pslot = pcell + n;
  int32_t* unsorted = pslot + n;
  int32_t* perm = unsorted + n;
  int32_t* iperm = perm + n;
  const int64_t slots = nc * capacity;
  sph_ws* ws = nullptr;  // no profiling without a workspace
  // empty slots: position 0, id N, side arrays their fill word (partition.py:334-358)
  SPH_LAUNCH(ws, "fill", st,
             k_fill<float><<<cdiv(slots * dim, kBlock), kBlock, 0, st>>>(position_buffer,
                                                                        slots * dim, 0.0f));
  SPH_LAUNCH(ws, "fill", st,
             k_fill<int32_t><<<cdiv(slots, kBlock), kBlock, 0, st>>>(id_buffer, slots, n));
  for (int b = 0; b < n_named; ++b) {
    const int64_t words = slots * named_width[b];
    SPH_LAUNCH(ws, "fill", st,
               k_fill<uint32_t><<<cdiv(words, kBlock), kBlock, 0, st>>>(named_buffer[b], words,
                                                                       named_fill[b]));
  }
  SPH_LAUNCH(ws, "fill", st, k_fill<int32_t><<<cdiv(nc, kBlock), kBlock, 0, st>>>(counts, nc, 0));
  if (n > 0) {
    if (dim == 2)
      SPH_LAUNCH(ws, "hash_count", st,
                 k_hash_count<2><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, n, g, counts, pcell,
                                                                   pslot, nullptr));
    else
      SPH_LAUNCH(ws, "hash_count", st,
                 k_hash_count<3><<<cdiv(n, kBlock), kBlock, 0, st>>>(r, n, g, counts, pcell,
                                                                   pslot, nullptr));
  }
  // cell starts, the largest occupancy into info[2], CELL_LIST_OVERFLOW into info[0]
  SPH_LAUNCH(ws, "fill", st, k_fill<int64_t><<<1, 64, 0, st>>>(info + 2, 1, 0));
  // (chunk sums in the sorted ids' place, which nothing has written yet)
  int32_t* const sums = 3 * (int64_t)n >= kScanSums ? unsorted : nullptr;
  const int rc = scan<int32_t>(ws, "scan_cells", counts, nc, start, sums, info, capacity, nullptr,
                               st);
  if (rc) return rc;
  if (n == 0) return SPH_OK;
  SPH_LAUNCH(ws, "scatter", st,
             k_scatter<<<cdiv(n, kBlock), kBlock, 0, st>>>(pcell, pslot, start, unsorted, n));
  // ascending id inside each cell: the order of the reference's stable argsort
  SPH_LAUNCH(ws, "cell_sort", st,
             k_cell_sort<3><<<cdiv(nc * 64, 256), 256, 0, st>>>(start, unsorted, perm, iperm, nc,
                                                               nullptr, nullptr, Grid{}, nullptr));
  if (dim == 2)
    SPH_LAUNCH(ws, "cell_list_fill", st,
               k_cell_list_fill<2><<<cdiv(n, kBlock), kBlock, 0, st>>>(
                   r, perm, pcell, start, n, capacity, position_buffer, id_buffer));
  else
    SPH_LAUNCH(ws, "cell_list_fill", st,
               k_cell_list_fill<3><<<cdiv(n, kBlock), kBlock, 0, st>>>(
                   r, perm, pcell, start, n, capacity, position_buffer, id_buffer));
  for (int b = 0; b < n_named; ++b)
    SPH_LAUNCH(ws, "cell_list_named", st,
               k_cell_list_named<<<cdiv((int64_t)n * named_width[b], kBlock), kBlock, 0, st>>>(
                   named[b], named_width[b], perm, pcell, start, n, capacity, named_buffer[b]));
  return SPH_OK;
}

extern "C" int sph_nl_needs_rebuild(sph_ws* ws, const float* r, const float* r_ref,
                                    float threshold_sq, int64_t* info, hipStream_t st) {
  if (!ws || !r || !r_ref || !info) { set_error("sph_nl_needs_rebuild: null"); return SPH_ERR_ARG; }
  const auto& c = ws->cfg;
  Grid g = make_grid(c);
  SPH_LAUNCH(ws, "fill", st, k_fill<int64_t><<<1, 64, 0, st>>>(info + 4, 1, 0));
  if (c.dim == 2)
    SPH_LAUNCH(ws, "needs_rebuild", st,
               k_needs_rebuild<2><<<cdiv(c.n, kBlock), kBlock, 0, st>>>(
                   r, r_ref, c.n, g, c.box[0], c.box[1], c.box[2], threshold_sq, info));
  else
    SPH_LAUNCH(ws, "needs_rebuild", st,
               k_needs_rebuild<3><<<cdiv(c.n, kBlock), kBlock, 0, st>>>(
                   r, r_ref, c.n, g, c.box[0], c.box[1], c.box[2], threshold_sq, info));
  return SPH_OK;
}

extern "C" int sph_nl_build(sph_ws* ws, int bank, const float* r, const int64_t* prev_info,
                            int64_t max_occupancy, int64_t* info, hipStream_t st) {
  int rc = check_ws(ws, bank);
  if (rc) return rc;
  if (!r || !info) { set_error("sph_nl_build: null"); return SPH_ERR_ARG; }
  const HistogramGuard guard{ws, st};
  rc = clean_histograms(ws, st);
  if (rc) return rc;
  rc = bin_particles(ws, bank, r, prev_info, info, st);
  if (rc) return rc;
  rc = build_pairs(ws, bank, info, st);
  if (rc) return rc;
  SPH_LAUNCH(ws, "reduce_pairs", st,
             k_reduce_parts<<<1, kReduceThreads, 0, st>>>(build_tail(ws, max_occupancy, info)));
  return SPH_OK;
}

extern "C" int sph_nl_finalize(sph_ws* ws, int64_t max_occupancy, int64_t* info, hipStream_t st) {
  if (!ws || !info) { set_error("sph_nl_finalize: null"); return SPH_ERR_ARG; }
  SPH_LAUNCH(ws, "finalize", st, k_finalize<<<1, 64, 0, st>>>(info, max_occupancy));
  return SPH_OK;
}

extern "C" int sph_nl_scan_budget(sph_ws* ws, int bank, int64_t n_sub, int64_t budget,
                                  int64_t* info, hipStream_t st) {
  int rc = check_ws(ws, bank);
  if (rc) return rc;
  if (n_sub <= 0 || !info) { set_error("sph_nl_scan_budget: bad argument"); return SPH_ERR_ARG; }
  rc = pair_offsets(ws, bank, st);
  if (rc) return rc;
  int64_t chunks = cdiv(ws->cfg.n, n_sub);
  SPH_LAUNCH(ws, "chunk_budget", st,
             k_chunk_budget<<<cdiv(chunks, kBlock), kBlock, 0, st>>>(ws->off64, ws->cfg.n, n_sub,
                                                                     budget, info));
  return SPH_OK;
}

extern "C" int sph_nl_write_idx(sph_ws* ws, int bank, int32_t* idx, int64_t max_occupancy,
                                const int64_t* info, hipStream_t st) {
  int rc = check_ws(ws, bank);
  if (rc) return rc;
  if (!idx || max_occupancy < 0) { set_error("sph_nl_write_idx: bad argument"); return SPH_ERR_ARG; }
  if (max_occupancy == 0) return SPH_OK;
  rc = pair_offsets(ws, bank, st);
  if (rc) return rc;
  const int n = ws->cfg.n;
  Bank& B = ws->bank[bank];
  constexpr int T2 = tpp_of(2), T3 = tpp_of(3);
  const dim3 grid((unsigned)cdiv(n, kIdxTile));
  if (ws->cfg.dim == 2)
    SPH_LAUNCH(ws, "write_idx", st,
               (k_write_idx<T2><<<grid, kBlock, 0, st>>>(B.perm, B.cnt, B.ell, ws->off64, idx,
                                                     max_occupancy, n, ws->npad, ws->lane_width)));
  else
    SPH_LAUNCH(ws, "write_idx", st,
               (k_write_idx<T3><<<grid, kBlock, 0, st>>>(B.perm, B.cnt, B.ell, ws->off64, idx,
                                                     max_occupancy, n, ws->npad, ws->lane_width)));
  SPH_LAUNCH(ws, "pad_idx", st,
             k_pad_idx<<<pad_blocks(max_occupancy), kBlock, 0, st>>>(idx, max_occupancy,
                                                                    ws->off64 + n, n));
  (void)info;
  return SPH_OK;
}

extern "C" int sph_nl_write_idx_skin(sph_ws* ws, const float* r, int32_t* idx,
                                     int64_t max_occupancy, hipStream_t st) {
  if (!ws || !r || !idx || max_occupancy < 0) {
    set_error("sph_nl_write_idx_skin: bad argument");
    return SPH_ERR_ARG;
  }
  if (!ws->sk.on || !ws->sk.stepped) {
    set_error("sph_nl_write_idx_skin: no skin lists built by sph_step on this workspace");
    return SPH_ERR_ARG;
  }
  if (max_occupancy == 0) return SPH_OK;
  const auto& c = ws->cfg;
  const int n = c.n;
  SkinIdxArgs a;
  a.r = r;
  a.perm = ws->sk.b.perm;
  a.cnt = ws->sk.b.cnt;
  a.ell = ws->sk.b.ell;
  a.cnt_id = ws->cnt_id;
  a.off = ws->off64;
  a.idx = idx;
  a.max_occ = max_occupancy;
  for (int d = 0; d < 3; ++d) {
    a.box[d] = c.box[d];
    a.half[d] = c.box[d] * 0.5f;
  }
  a.cutoff_sq = c.cutoff_sq;
  a.n = n;
  a.npad = ws->npad;
  a.tpp = ws->tpp;
  a.lane_width = ws->sk.lane_width;
  const unsigned nb = (unsigned)cdiv(n, kBlock);
  if (c.dim == 2)
    SPH_LAUNCH(ws, "skin_idx_count", st, (k_skin_pairs<2, false><<<nb, kBlock, 0, st>>>(a)));
  else
    SPH_LAUNCH(ws, "skin_idx_count", st, (k_skin_pairs<3, false><<<nb, kBlock, 0, st>>>(a)));
  const int rc = scan<int64_t>(ws, "scan_pairs", ws->cnt_id, n, ws->off64, ws->scan_tmp, nullptr,
                               -1, nullptr, st);
  if (rc) return rc;
  if (c.dim == 2)
    SPH_LAUNCH(ws, "skin_idx_write", st, (k_skin_pairs<2, true><<<nb, kBlock, 0, st>>>(a)));
  else
    SPH_LAUNCH(ws, "skin_idx_write", st, (k_skin_pairs<3, true><<<nb, kBlock, 0, st>>>(a)));
  SPH_LAUNCH(ws, "pad_idx", st,
             k_pad_idx<<<pad_blocks(max_occupancy), kBlock, 0, st>>>(idx, max_occupancy,
                                                                    ws->off64 + n, n));
  return SPH_OK;
}
