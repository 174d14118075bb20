// knn.hip — k nearest neighbours per query within its cloud, on gfx950.
//
// Replaces knn_kernel<MAX_K> + build_batch_map_kernel (geoembodied/csrc/knn_kernel.cu:113-193)
// with the semantics of _knn_bruteforce (geoembodied/csrc/__init__.py:435-492) made total: the
// k smallest keys (d, j), ascending, padded with -1 / 1e30f.
//
// One 256-thread workgroup serves up to 256 queries of a single cloud (a prepare kernel maps
// workgroups to (cloud, query tile) without a host round trip).  The cloud's sources stream
// through LDS in 1024-point tiles; every thread reads the same LDS entry at a time (broadcast,
// no bank conflicts) and keeps its candidates as a sorted register array.  Sources arrive in
// ascending index order, so a new candidate enters the list only on a strictly smaller
// distance and lands after every equal one — exactly the (d, j) order.
// Non-finite distances never enter the list (they report as padding).
#include "scan.hpp"

namespace geo {
namespace {

constexpr int kKnnThreads = 256;
constexpr int kKnnTile = 1024;

// tiles[b] = first workgroup of cloud b; tiles[B] = total workgroups.  Offsets are clamped to
// [0, N] so inconsistent ptr arrays stay memory-safe.
__global__ __launch_bounds__(kScanThreads) void knn_prepare_kernel(const int64_t* __restrict__ ptr_q,
                                                                   int64_t B, int64_t Nq,
                                                                   int64_t* __restrict__ tiles) {
  __shared__ int64_t lds[kScanThreads / kWave];
  int64_t carry = 0;
  for (int64_t base = 0; base < B; base += kScanThreads) {
    const int64_t b = base + threadIdx.x;
    int64_t nt = 0;
    if (b < B) {
      int64_t a = ptr_q[b], c = ptr_q[b + 1];
      a = a < 0 ? 0 : (a > Nq ? Nq : a);
      c = c < a ? a : (c > Nq ? Nq : c);
      nt = (c - a + kKnnThreads - 1) / kKnnThreads;
    }
    int64_t total;
    const int64_t off = block_exclusive_scan<int64_t>(nt, lds, total);
    if (b < B) tiles[b] = carry + off;
    carry += total;
  }
  if (threadIdx.x == 0) tiles[B] = carry;
}

// k above the largest list (kKnnMaxList) is served in passes of at most kKnnMaxList columns:
// pass p writes columns [col0, col0 + width) of each row (LB = true for p > 0) and admits only
// sources whose key (d, j) is above the key in column col0 - 1, which the previous pass wrote,
// so the passes together list the k smallest keys in order.  A row whose column col0 - 1 is
// padding has no further neighbours: the pass leaves its padding.
constexpr int kKnnMaxList = 128;

template <int KMAX, bool LB = false>
__global__ __launch_bounds__(kKnnThreads) void knn_kernel(
    const float* __restrict__ query, int64_t Nq, const float* __restrict__ source, int64_t Ns,
    const int64_t* __restrict__ ptr_q, const int64_t* __restrict__ ptr_s,
    const int64_t* __restrict__ tiles, int64_t B, int k, int64_t* __restrict__ out_idx,
    float* __restrict__ out_dist, int col0, int width) {
  __shared__ float4 tile[kKnnTile];
  const int64_t blk = blockIdx.x;
  if (blk >= tiles[B]) return;
  // cloud of this workgroup: last b with tiles[b] <= blk
  int64_t lo = 0, hi = B - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) >> 1;
    if (tiles[mid] <= blk) lo = mid; else hi = mid - 1;
  }
  const int64_t b = lo;
  int64_t qa = ptr_q[b], qc = ptr_q[b + 1];
  qa = qa < 0 ? 0 : (qa > Nq ? Nq : qa);
  qc = qc < qa ? qa : (qc > Nq ? Nq : qc);
  int64_t sa = ptr_s[b], sc = ptr_s[b + 1];
  sa = sa < 0 ? 0 : (sa > Ns ? Ns : sa);
  sc = sc < sa ? sa : (sc > Ns ? Ns : sc);
  const int64_t q = qa + (blk - tiles[b]) * kKnnThreads + threadIdx.x;
  bool qok = q < qc;
  float lbd = -__builtin_inff();  // key of column col0 - 1 (passes after the first)
  int64_t lbj = -1;
  if constexpr (LB) {
    if (qok) {
      lbj = out_idx[q * k + col0 - 1];
      lbd = out_dist[q * k + col0 - 1];
      qok = lbj >= 0;  // padding there: nothing further to list
    }
  }

  float qx = 0.f, qy = 0.f, qz = 0.f;
  if (qok) {
    qx = query[3 * q];
    qy = query[3 * q + 1];
    qz = query[3 * q + 2];
  }
  float D[KMAX];
  int J[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; ++i) {
    D[i] = __builtin_inff();
    J[i] = -1;
  }
  for (int64_t s0 = sa; s0 < sc; s0 += kKnnTile) {
    const int n = static_cast<int>(min(static_cast<int64_t>(kKnnTile), sc - s0));
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kKnnThreads) {
      const float* p = source + 3 * (s0 + i);
      tile[i] = make_float4(p[0], p[1], p[2], 0.f);
    }
    __syncthreads();
    for (int i = 0; i < n; ++i) {
      const float4 p = tile[i];
      const float d = sqdist(qx, qy, qz, p.x, p.y, p.z);
      bool above = true;
      if constexpr (LB) above = d > lbd || (d == lbd && s0 + i > lbj);
      if (above && d < D[KMAX - 1]) {
        const int j = static_cast<int>(s0 + i);
#pragma unroll
        for (int m = KMAX - 1; m > 0; --m) {
          const bool shift = d < D[m - 1];
          const bool here = !shift && d < D[m];
          D[m] = shift ? D[m - 1] : (here ? d : D[m]);
          J[m] = shift ? J[m - 1] : (here ? j : J[m]);
        }
        if (d < D[0]) {
          D[0] = d;
          J[0] = j;
        }
      }
    }
  }
  if (qok) {
    int64_t* oi = out_idx + q * k + col0;
    float* od = out_dist + q * k + col0;
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
      if (i < width) {
        oi[i] = J[i] >= 0 ? static_cast<int64_t>(J[i]) : -1;
        od[i] = J[i] >= 0 ? D[i] : 1e30f;
      }
    }
  }
}

template <int KMAX>
int launch_knn(const float* query, int64_t Nq, const float* source, int64_t Ns,
               const int64_t* ptr_q, const int64_t* ptr_s, const int64_t* tiles, int64_t B, int k,
               int64_t* out_idx, float* out_dist, hipStream_t st, int col0 = 0, int width = -1) {
  const int64_t grid = ceil_div(Nq, kKnnThreads) + B;
  if (width < 0) width = k;
  if (col0 == 0)
    hipLaunchKernelGGL((knn_kernel<KMAX, false>), dim3(grid), dim3(kKnnThreads), 0, st, query, Nq,
                       source, Ns, ptr_q, ptr_s, tiles, B, k, out_idx, out_dist, col0, width);
  else
    hipLaunchKernelGGL((knn_kernel<KMAX, true>), dim3(grid), dim3(kKnnThreads), 0, st, query, Nq,
                       source, Ns, ptr_q, ptr_s, tiles, B, k, out_idx, out_dist, col0, width);
  GEO_LAUNCH_CHECK("knn_kernel");
  return GEO_OK;
}

// --------------------------------------------------------------------------- grid search ---
// Clouds of many sources and k <= 32: each source cloud is binned into a uniform grid (cell
// edge chosen so a cell holds about k/4 points at the cloud's mean density, at most 1024 cells
// per axis and 2n + 64 cells), sources are counting-sorted by cell, and each query visits the
// cells in shells of growing Chebyshev radius around its own cell.  After a shell it stops when
// its k-th distance is below a bound that every unvisited source provably exceeds: the query's
// distance to the faces of the visited block, measured in cell units minus 1e-3 of a cell (the
// cell coordinates are rounded fp32 values below 1024, accurate to ~1e-4 cells), scaled by the
// cell edge and shrunk by 1e-5 relative (the fp32 distance of a farther point can round down
// by less than that).  The stop test is strict, so a source at exactly the k-th distance with a
// smaller index cannot be missed.  Candidates arrive in cell order, so the register list keeps
// the total order (d, j) explicitly, as one 64-bit key per entry (distance bits, index).
constexpr int kKnnGridThreads = 256;
constexpr int kKnnSetupThreads = 1024;
constexpr int kKnnGridMaxAxis = 1024;
constexpr int kKnnGridMaxK = 32;
constexpr double kKnnCellTarget = 0.25;  // points per cell per neighbour (measured best)
constexpr int kKnnCellCap = 2;            // cells per point
constexpr int64_t kKnnWideSources = 65536; // one cloud this large: a wave per query for k <= 8
constexpr int kKnnBoxParts = 64;           // most workgroups per cloud for the bounding box
constexpr int64_t kKnnBoxChunk = 16384;    // points per bounding-box workgroup
constexpr int64_t kKnnCloudCells = 65;     // cells of a cloud beyond kKnnCellCap per point, with the end entry
constexpr int kKnnBuildCells = 16384;      // most cells of a cloud whose grid one workgroup builds (LDS)
constexpr int64_t kKnnBuildSources = 81920; // most sources of a call that takes that way
constexpr int kKnnBuildPts = 8;            // points per thread held in registers there

struct KnnGrid {
  float ox, oy, oz, inv_h, h;
  int dx, dy, dz, base, ncells;
};

struct KnnGridWs {
  KnnGrid* grid;
  int32_t* cell_cnt;
  int32_t* cell_start;
  uint64_t* cell_scan;  // look-back status of the cell scan; zeroed with cell_cnt (carved next)
  int32_t* pt_cell;
  int32_t* pt_rank;
  float4* spos;
  uint32_t* box_part;  // [B][kKnnBoxParts][6] partial bounding boxes (order keys)
  int64_t cells_max;
};

KnnGridWs carve_knn_grid(void* base, int64_t Ns, int64_t B, size_t* bytes) {
  Carver c(base);
  KnnGridWs w;
  const int64_t nn = Ns > 0 ? Ns : 1, bb = B > 0 ? B : 1;
  w.cells_max = kKnnCellCap * Ns + kKnnCloudCells * bb;
  w.grid = c.take<KnnGrid>(bb);
  w.cell_cnt = c.take<int32_t>(w.cells_max + 1);
  w.cell_scan = c.take<uint64_t>(scan_lookback_elems(w.cells_max + 1));
  w.cell_start = c.take<int32_t>(w.cells_max + 1);
  w.pt_cell = c.take<int32_t>(nn);
  w.pt_rank = c.take<int32_t>(nn);
  w.spos = c.take<float4>(nn);
  w.box_part = c.take<uint32_t>(bb * kKnnBoxParts * 6);
  *bytes = c.used;
  return w;
}

__device__ __forceinline__ int64_t clamp_range(int64_t v, int64_t n) { return v < 0 ? 0 : (v > n ? n : v); }

// Partial bounding boxes of large clouds: block (p, b) reduces the p-th of `parts` equal slices
// of cloud b into box_part[b][p] (order keys, so the minimum and maximum are integer ones).
__global__ __launch_bounds__(kKnnSetupThreads) void knn_grid_box_part(
    const float* __restrict__ source, int64_t Ns, const int64_t* __restrict__ ptr_s, int parts,
    uint32_t* __restrict__ box_part) {
  constexpr int W = kKnnSetupThreads / kWave;
  __shared__ uint32_t red[6][W];
  const int p = blockIdx.x, b = blockIdx.y;
  const int64_t sa = clamp_range(ptr_s[b], Ns);
  const int64_t sc = sa > clamp_range(ptr_s[b + 1], Ns) ? sa : clamp_range(ptr_s[b + 1], Ns);
  const int64_t chunk = (sc - sa + parts - 1) / parts;
  const int64_t pa = sa + p * chunk, pc = min(sc, pa + chunk);
  const int t = threadIdx.x, w = t / kWave;
  uint32_t mn[3] = {~0u, ~0u, ~0u}, mx[3] = {0u, 0u, 0u};
  for (int64_t i = pa + t; i < pc; i += kKnnSetupThreads) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t kk = float_order_key(source[3 * i + a]);
      mn[a] = min(mn[a], kk);
      mx[a] = max(mx[a], kk);
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    mn[a] = wave_min_u32(mn[a]);
    mx[a] = wave_max_u32(mx[a]);
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) { red[a][w] = mn[a]; red[3 + a][w] = mx[a]; }
  }
  __syncthreads();
  if (t < 6) {
    uint32_t v = red[t][0];
    for (int ww = 1; ww < W; ++ww) v = t < 3 ? min(v, red[t][ww]) : max(v, red[t][ww]);
    box_part[(static_cast<int64_t>(b) * kKnnBoxParts + p) * 6 + t] = v;
  }
}

// The grid of a cloud of n points with the bounding box lo..hi and at most `cap` cells.
__device__ KnnGrid knn_make_grid(const float (&lo)[3], const float (&hi)[3], int64_t n, int k, double cap) {
  KnnGrid g{0.f, 0.f, 0.f, 0.f, 0.f, 1, 1, 1, 0, 1};
  double ext[3];
  bool finite = n > 0;
  for (int a = 0; a < 3; ++a) {
    ext[a] = static_cast<double>(hi[a]) - static_cast<double>(lo[a]);
    finite = finite && ext[a] >= 0.0 && ext[a] < 1e30;
  }
  if (finite) {
    const double emax = fmax(fmax(ext[0], ext[1]), ext[2]);
    const double target = fmax(kKnnCellTarget * k, 1.0);
    double h = emax;  // fixed point of h = cbrt(prod max(ext, h) * target / n)
    for (int it = 0; it < 12 && h > 0.0; ++it) {
      const double next = cbrt(fmax(ext[0], h) * fmax(ext[1], h) * fmax(ext[2], h) * target / static_cast<double>(n));
      if (next == h) break;  // settled: the further steps would repeat it
      h = next;
    }
    if (h > 0.0) {
      int64_t d[3] = {1, 1, 1};
      bool ok = false;
      for (int it = 0; it < 64 && !ok; ++it) {
        double prod = 1.0, worst = 0.0;
        for (int a = 0; a < 3; ++a) {
          const double q = floor(ext[a] / h) + 1.0;
          d[a] = q < 4.0 * kKnnGridMaxAxis ? static_cast<int64_t>(q) : 4 * kKnnGridMaxAxis;
          prod *= static_cast<double>(d[a]);
          worst = fmax(worst, static_cast<double>(d[a]) / kKnnGridMaxAxis);
        }
        ok = prod <= cap && worst <= 1.0;
        if (!ok) h *= fmax(fmax(cbrt(prod / cap), worst), 1.0) * 1.01;
      }
      if (ok) {
        g.ox = lo[0]; g.oy = lo[1]; g.oz = lo[2];
        g.inv_h = static_cast<float>(1.0 / h);
        g.h = static_cast<float>(h * (1.0 - 1e-6));
        g.dx = static_cast<int>(d[0]); g.dy = static_cast<int>(d[1]); g.dz = static_cast<int>(d[2]);
      }
    }
  }
  g.ncells = n > 0 ? g.dx * g.dy * g.dz : 0;
  return g;
}

// One block per source cloud: bounding box (from `parts` partial boxes when parts > 0), then
// (thread 0) the grid of that cloud.
__global__ __launch_bounds__(kKnnSetupThreads) void knn_grid_setup(
    const float* __restrict__ source, int64_t Ns, const int64_t* __restrict__ ptr_s, int k,
    KnnGrid* __restrict__ grid, const uint32_t* __restrict__ box_part, int parts) {
  constexpr int W = kKnnSetupThreads / kWave;
  __shared__ uint32_t red[6][W];
  const int b = blockIdx.x;
  const int64_t sa = clamp_range(ptr_s[b], Ns);
  const int64_t sc = sa > clamp_range(ptr_s[b + 1], Ns) ? sa : clamp_range(ptr_s[b + 1], Ns);
  const int t = threadIdx.x, w = t / kWave;
  uint32_t mn[3] = {~0u, ~0u, ~0u}, mx[3] = {0u, 0u, 0u};
  if (parts > 0) {
    if (t < parts) {
      const uint32_t* bp = box_part + (static_cast<int64_t>(b) * kKnnBoxParts + t) * 6;
#pragma unroll
      for (int a = 0; a < 3; ++a) { mn[a] = bp[a]; mx[a] = bp[3 + a]; }
    }
  } else {
#pragma unroll 4
    for (int64_t i = sa + t; i < sc; i += kKnnSetupThreads) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const uint32_t kk = float_order_key(source[3 * i + a]);
        mn[a] = min(mn[a], kk);
        mx[a] = max(mx[a], kk);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    mn[a] = wave_min_u32(mn[a]);
    mx[a] = wave_max_u32(mx[a]);
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) { red[a][w] = mn[a]; red[3 + a][w] = mx[a]; }
  }
  __syncthreads();
  if (t != 0) return;
  float lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    uint32_t m0 = red[a][0], m1 = red[3 + a][0];
    for (int ww = 1; ww < W; ++ww) { m0 = min(m0, red[a][ww]); m1 = max(m1, red[3 + a][ww]); }
    lo[a] = float_from_order_key(m0);
    hi[a] = float_from_order_key(m1);
  }
  const int64_t n = sc - sa;
  grid[b] = knn_make_grid(lo, hi, n, k, kKnnCellCap * static_cast<double>(n) + 64.0);
}

// Single block: cell bases (exclusive scan of the cells per cloud).
__global__ __launch_bounds__(kScanThreads) void knn_grid_base(KnnGrid* __restrict__ grid, int64_t B) {
  __shared__ int64_t lds[kScanThreads / kWave];
  int64_t carry = 0;
  for (int64_t base = 0; base < B; base += kScanThreads) {
    const int64_t b = base + threadIdx.x;
    const int64_t cells = b < B ? grid[b].ncells : 0;
    int64_t total;
    const int64_t off = block_exclusive_scan<int64_t>(cells, lds, total);
    if (b < B) grid[b].base = static_cast<int>(carry + off);
    carry += total;
  }
}

__device__ __forceinline__ int knn_cell_coord(float p, float o, float inv_h, int dim, float* u_out) {
#pragma clang fp contract(off)
  const float u = (p - o) * inv_h;
  *u_out = u;
  const int c = static_cast<int>(floorf(u));
  return c < 0 ? 0 : (c >= dim ? dim - 1 : c);
}

// Last b in [0, B) with ptr[b] <= i (the cloud holding index i, if any).
__device__ __forceinline__ int64_t cloud_of_index(const int64_t* __restrict__ ptr, int64_t B, int64_t i) {
  int64_t lo = 0, hi = B;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (ptr[mid + 1] <= i) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__global__ __launch_bounds__(kKnnGridThreads) void knn_grid_cell(
    const float* __restrict__ source, int64_t Ns, const int64_t* __restrict__ ptr_s, int64_t B,
    KnnGridWs w) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= Ns) return;
  const int64_t b = cloud_of_index(ptr_s, B, i);
  if (b >= B || i < ptr_s[b] || i >= ptr_s[b + 1]) {
    w.pt_cell[i] = -1;
    return;
  }
  const KnnGrid g = w.grid[b];
  float u;
  const int cx = knn_cell_coord(source[3 * i], g.ox, g.inv_h, g.dx, &u);
  const int cy = knn_cell_coord(source[3 * i + 1], g.oy, g.inv_h, g.dy, &u);
  const int cz = knn_cell_coord(source[3 * i + 2], g.oz, g.inv_h, g.dz, &u);
  const int c = g.base + (cx * g.dy + cy) * g.dz + cz;
  w.pt_cell[i] = c;
  w.pt_rank[i] = cell_rank(&w.cell_cnt[c], c);
}

__global__ __launch_bounds__(kKnnGridThreads) void knn_grid_scatter(const float* __restrict__ source,
                                                                    int64_t Ns, KnnGridWs w) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= Ns) return;
  const int c = w.pt_cell[i];
  if (c < 0) return;
  w.spos[w.cell_start[c] + w.pt_rank[i]] =
      make_float4(source[3 * i], source[3 * i + 1], source[3 * i + 2], __int_as_float(static_cast<int>(i)));
}

// The whole grid of one cloud by one workgroup: bounding box, cells counted in LDS, exclusive
// scan, scatter.  Cloud b's cells start at kKnnCellCap * ptr[b] + kKnnCloudCells * b, so no scan
// over clouds is needed, and its end entry is its own.  The first kKnnBuildPts * 1024 points stay
// in registers through all passes, points beyond are read again (their ranks go through global
// memory).
// What bounds it: the latency of one load, three barriers' worth of reductions and the serial
// grid parameters; 16 clouds of about 4096 points 10 us, against 27 us and six launches for box, cell
// bases, zero fill, count, scan and scatter over all clouds (each 2.5 to 6 us, latency as well).
__global__ __launch_bounds__(kKnnSetupThreads) void knn_grid_build(
    const float* __restrict__ source, int64_t Ns, const int64_t* __restrict__ ptr_s, int k, KnnGridWs w) {
  constexpr int T = kKnnSetupThreads, W = T / kWave;
  __shared__ int cnt[kKnnBuildCells];
  __shared__ uint32_t red[6][W];
  __shared__ KnnGrid sg;
  const int b = blockIdx.x;
  const int64_t sa = clamp_range(ptr_s[b], Ns);
  const int64_t sc = max(sa, clamp_range(ptr_s[b + 1], Ns));
  const int n = static_cast<int>(sc - sa);
  const float* pts = source + 3 * sa;
  const int t = threadIdx.x, wv = t / kWave;
  float px[kKnnBuildPts], py[kKnnBuildPts], pz[kKnnBuildPts];
  uint32_t mn[3] = {~0u, ~0u, ~0u}, mx[3] = {0u, 0u, 0u};
  auto grow = [&](float x, float y, float z) {
    const uint32_t kk[3] = {float_order_key(x), float_order_key(y), float_order_key(z)};
#pragma unroll
    for (int a = 0; a < 3; ++a) { mn[a] = min(mn[a], kk[a]); mx[a] = max(mx[a], kk[a]); }
  };
  // the points beyond the registers, a batch of independent loads at a time
  auto rest = [&](auto f) {
    for (int i0 = kKnnBuildPts * T + t; i0 < n; i0 += kKnnBuildPts * T) {
      float x[kKnnBuildPts], y[kKnnBuildPts], z[kKnnBuildPts];
#pragma unroll
      for (int s = 0; s < kKnnBuildPts; ++s) {
        const int i = min(i0 + s * T, n - 1);
        x[s] = pts[3 * i]; y[s] = pts[3 * i + 1]; z[s] = pts[3 * i + 2];
      }
#pragma unroll
      for (int s = 0; s < kKnnBuildPts; ++s)
        if (i0 + s * T < n) f(i0 + s * T, x[s], y[s], z[s]);
    }
  };
#pragma unroll
  for (int s = 0; s < kKnnBuildPts; ++s) {
    const int i = s * T + t;
    px[s] = py[s] = pz[s] = 0.f;
    if (i < n) { px[s] = pts[3 * i]; py[s] = pts[3 * i + 1]; pz[s] = pts[3 * i + 2]; }
  }
  for (int c = t; c < kKnnBuildCells / 4; c += T) reinterpret_cast<int4*>(cnt)[c] = make_int4(0, 0, 0, 0);
#pragma unroll
  for (int s = 0; s < kKnnBuildPts; ++s)
    if (s * T + t < n) grow(px[s], py[s], pz[s]);
  rest([&](int, float x, float y, float z) { grow(x, y, z); });
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    mn[a] = wave_min_u32(mn[a]);
    mx[a] = wave_max_u32(mx[a]);
  }
  if (lane_id() == 0) {
#pragma unroll
    for (int a = 0; a < 3; ++a) { red[a][wv] = mn[a]; red[3 + a][wv] = mx[a]; }
  }
  __syncthreads();
  if (t == 0) {
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
      uint32_t m0 = red[a][0], m1 = red[3 + a][0];
#pragma unroll
      for (int ww = 1; ww < W; ++ww) { m0 = min(m0, red[a][ww]); m1 = max(m1, red[3 + a][ww]); }
      lo[a] = float_from_order_key(m0);
      hi[a] = float_from_order_key(m1);
    }
    const double cells = kKnnCellCap * static_cast<double>(n) + 64.0;
    KnnGrid g = knn_make_grid(lo, hi, n, k, fmin(cells, static_cast<double>(kKnnBuildCells)));
    g.base = static_cast<int>(kKnnCellCap * sa + kKnnCloudCells * b);
    sg = g;
    w.grid[b] = g;
  }
  __syncthreads();
  const KnnGrid g = sg;
  auto cell_of = [&](float x, float y, float z) {
    float u;
    const int cx = knn_cell_coord(x, g.ox, g.inv_h, g.dx, &u);
    const int cy = knn_cell_coord(y, g.oy, g.inv_h, g.dy, &u);
    const int cz = knn_cell_coord(z, g.oz, g.inv_h, g.dz, &u);
    return (cx * g.dy + cy) * g.dz + cz;
  };
  int cell[kKnnBuildPts], rank[kKnnBuildPts];
#pragma unroll
  for (int s = 0; s < kKnnBuildPts; ++s) {
    cell[s] = rank[s] = 0;
    if (s * T + t < n) {
      cell[s] = cell_of(px[s], py[s], pz[s]);
      rank[s] = atomicAdd(&cnt[cell[s]], 1);
    }
  }
  rest([&](int i, float x, float y, float z) { w.pt_rank[sa + i] = atomicAdd(&cnt[cell_of(x, y, z)], 1); });
  __syncthreads();
  // exclusive scan: `per` consecutive cells a thread, the sums over the waves in LDS
  const int per = (g.ncells + T - 1) / T;
  const int c0 = min(t * per, g.ncells), c1 = min(c0 + per, g.ncells);
  int sum = 0;
  for (int c = c0; c < c1; ++c) sum += cnt[c];
  const int inc = static_cast<int>(wave_inclusive_sum_dpp(static_cast<uint32_t>(sum)));
  if (lane_id() == kWave - 1) red[0][wv] = static_cast<uint32_t>(inc);
  __syncthreads();
  int off = static_cast<int>(sa) + inc - sum;
  for (int ww = 0; ww < wv; ++ww) off += static_cast<int>(red[0][ww]);
  for (int c = c0; c < c1; ++c) {
    const int v = cnt[c];
    cnt[c] = off;
    off += v;
  }
  __syncthreads();
  for (int c = t; c < g.ncells; c += T) w.cell_start[g.base + c] = cnt[c];
  if (t == 0) w.cell_start[g.base + g.ncells] = static_cast<int>(sc);
#pragma unroll
  for (int s = 0; s < kKnnBuildPts; ++s) {
    const int i = s * T + t;
    if (i < n)
      w.spos[cnt[cell[s]] + rank[s]] = make_float4(px[s], py[s], pz[s], __int_as_float(static_cast<int>(sa) + i));
  }
  rest([&](int i, float x, float y, float z) {
    w.spos[cnt[cell_of(x, y, z)] + w.pt_rank[sa + i]] =
        make_float4(x, y, z, __int_as_float(static_cast<int>(sa) + i));
  });
}

// Candidate key: the distance's bits above the source index, read as a double.  Squared distances
// are non-negative floats, whose bits order like the values, and positive doubles order like their
// bits, so one compare gives the total order used throughout (distance, then source index), and
// min and max are one instruction each.  No key has the exponent of an infinity or a NaN: the high
// word is at most 0x7f800000.  An empty slot holds kKnnNone, above every finite distance.
__device__ __forceinline__ double knn_key(float d, int j) {
  return __hiloint2double(__float_as_int(d), j);
}
__device__ __forceinline__ double knn_none() { return __hiloint2double(0x7f800000, 0); }
__device__ __forceinline__ double knn_min(double a, double b) {
  double r;  // the instruction itself: fmin() would first quieten operands that are never NaN
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double knn_max(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// Sorted list of one lane, of which at most the first `used` slots are taken; inserts (d, j) if it
// is below the last slot and below lim (infinite and NaN distances never enter).
template <int KMAX>
__device__ __forceinline__ void knn_insert(double (&L)[KMAX], int used, double lim, float d, int j) {
  const double key = knn_key(d, j);
  if (__float_as_uint(d) < 0x7f800000u && key < lim && key < L[KMAX - 1]) {
#pragma unroll
    for (int m = KMAX - 1; m > 0; --m)
      if (m <= used) L[m] = knn_max(L[m - 1], knn_min(key, L[m]));
    L[0] = knn_min(key, L[0]);
  }
}

// Merge with the list of another lane (at lane ^ MASK, or mirrored where every lane of the halves
// holds the same list): keep the KMAX smallest of both, sorted.  The element-wise minimum of one
// list and the other reversed is bitonic and holds exactly the KMAX smallest; half-cleaners sort
// it.  Both lanes end with the same list.
template <int KMAX, int MASK>
__device__ __forceinline__ void knn_merge(double (&L)[KMAX]) {
  auto other = [](int v) -> int {
    if constexpr (MASK == 1) return static_cast<int>(dpp_u32<kDppXor1>(static_cast<uint32_t>(v)));
    else if constexpr (MASK == 2) return static_cast<int>(dpp_u32<kDppXor2>(static_cast<uint32_t>(v)));
    else if constexpr (MASK == 4) return static_cast<int>(dpp_u32<kDppHalfMirror>(static_cast<uint32_t>(v)));
    else if constexpr (MASK == 8) return static_cast<int>(dpp_u32<kDppMirror>(static_cast<uint32_t>(v)));
    else return __shfl_xor(v, MASK, kWave);
  };
  double P[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; ++i) P[i] = __hiloint2double(other(__double2hiint(L[i])), other(__double2loint(L[i])));
#pragma unroll
  for (int i = 0; i < KMAX; ++i) L[i] = knn_min(L[i], P[KMAX - 1 - i]);
#pragma unroll
  for (int sd = KMAX / 2; sd > 0; sd >>= 1) {
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
      if ((i & sd) == 0) {
        const double a = L[i], c = L[i + sd];
        L[i] = knn_min(a, c);
        L[i + sd] = knn_max(a, c);
      }
    }
  }
}
template <int KMAX, int G>
__device__ __forceinline__ void knn_merge_group(double (&L)[KMAX]) {
  knn_merge<KMAX, 1>(L);
  knn_merge<KMAX, 2>(L);
  knn_merge<KMAX, 4>(L);
  if constexpr (G >= 16) knn_merge<KMAX, 8>(L);
  if constexpr (G >= 32) knn_merge<KMAX, 16>(L);
  if constexpr (G >= 64) knn_merge<KMAX, 32>(L);
}

// G lanes per query: the lanes of a group split every visited cell range (consecutive sources,
// so the group's loads are contiguous), and each keeps its own sorted list of its KMAX nearest.
// After every step the lists are merged, the stop test reads the k-th key, and where the search
// goes on lane 0 keeps the merged list and the others start empty.
//
// What bounded the earlier form of this search was the chain of dependent loads: it read the
// bounds of one row of cells and then that row's points, nine times for the 27 cells around the
// query and 34 times for the next shell, and the 64-bit integer list steps beside it.  Here
//  - the first step takes the 27 cells at once: the nine rows' bounds come with one load per lane
//    and the first G points of every row with nine independent loads (G = 64, a query in a dense
//    part of one large cloud, starts with the query's own cell instead);
//  - in a later shell every lane forms one row (or one of the two cells) of the shell, drops it or
//    cuts its z range if the k-th distance rules it out, and reads its bounds; the group then
//    goes through the ranges that are left, two at a time;
//  - the list steps are one minimum and one maximum of doubles per slot (knn_key), and the i-th
//    point of the first step can only have i slots in front of it.
// A dropped row or cell is at least its distance in cell units minus 1e-3 of a cell per axis away,
// scaled and shrunk as the stop test's bound is.
// Whole calls with the one-workgroup grid, before -> now: 16 clouds of 4096 points on a sphere, a
// quarter of them as queries, k = 16 60 -> 27 us, k = 3 43 -> 21 us; cubes of 4096 points, k = 16 87
// -> 29 us.  With the grid by six launches as before: 32 cubes x 4096 queries, k = 32 821 -> 253 us;
// a lidar frame of 131,072 points against itself, k = 8 500 -> 325 us, a quarter of it k = 16 407 ->
// 318 us; 512 cubes of 1024 points, k = 3 133 -> 96 us.
template <int KMAX, int G>
__global__ __launch_bounds__(kKnnGridThreads) void knn_grid_query(
    const float* __restrict__ query, int64_t Nq, const int64_t* __restrict__ ptr_q, int64_t B,
    KnnGridWs w, int k, int64_t* __restrict__ out_idx, float* __restrict__ out_dist) {
  constexpr bool kBlock = G < kWave;  // first step: 27 cells
  const int64_t gt = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t q = gt / G;
  const int lane = lane_id(), gl = lane % G, gb = lane - gl;
  int64_t b = 0;
  if (B <= kWave) {
    // the wave's 64 / G queries against all cloud ends at once
    const int64_t end = lane < B ? ptr_q[lane + 1] : INT64_MAX;
    const int64_t q0 = (gt - lane) / G;
#pragma unroll
    for (int i = 0; i < kWave / G; ++i) {
      const int c = __popcll(__ballot(end <= q0 + i));
      if (gb == i * G) b = c;
    }
  }
  if (q >= Nq) return;  // whole groups leave together (G divides the block)
  if (B > kWave) b = cloud_of_index(ptr_q, B, q);
  const bool covered = b < B && q >= ptr_q[b] && q < ptr_q[b + 1];
  if (!covered || w.grid[b].ncells == 0) {  // no cloud, or an empty source cloud: padding
    for (int i = gl; i < k; i += G) {
      out_idx[q * k + i] = -1;
      out_dist[q * k + i] = 1e30f;
    }
    return;
  }
  const KnnGrid g = w.grid[b];
  const int32_t* __restrict__ cell_start = w.cell_start + g.base;
  const float qx = query[3 * q], qy = query[3 * q + 1], qz = query[3 * q + 2];
  float ux, uy, uz;
  const int cx = knn_cell_coord(qx, g.ox, g.inv_h, g.dx, &ux);
  const int cy = knn_cell_coord(qy, g.oy, g.inv_h, g.dy, &uy);
  const int cz = knn_cell_coord(qz, g.oz, g.inv_h, g.dz, &uz);
  const double none = knn_none();
  double L[KMAX];
#pragma unroll
  for (int i = 0; i < KMAX; ++i) L[i] = none;
  double lim = none;  // the k-th key so far

  auto insert = [&](const float4& s, int used) {
    knn_insert<KMAX>(L, used, lim, sqdist(qx, qy, qz, s.x, s.y, s.z), __float_as_int(s.w));
  };
  int r = kBlock ? 1 : 0;
  if constexpr (kBlock) {
    auto bounds = [&](int i) {  // of the i-th of the nine rows
      const int ix = cx - 1 + i / 3, iy = cy - 1 + i % 3;
      int2 v = make_int2(0, 0);
      if (i < 9 && ix >= 0 && ix < g.dx && iy >= 0 && iy < g.dy) {
        const int c = (ix * g.dy + iy) * g.dz;
        v = make_int2(cell_start[c + max(cz - 1, 0)], cell_start[c + min(cz + 1, g.dz - 1) + 1]);
      }
      return v;
    };
    const int2 own = bounds(gl);
    int2 row[9];
    float4 s[9];
    if constexpr (G < 9) row[8] = bounds(8);
    bool more = false;
#pragma unroll
    for (int i = 0; i < 9; ++i) {
      if (i < G) row[i] = make_int2(__shfl(own.x, gb + i, kWave), __shfl(own.y, gb + i, kWave));
      const int p = row[i].x + gl;
      s[i] = w.spos[p < row[i].y ? p : 0];
      more = more || row[i].x + G < row[i].y;
    }
#pragma unroll
    for (int i = 0; i < 9; ++i)
      if (row[i].x + gl < row[i].y) insert(s[i], i);
    if (more) {
#pragma unroll
      for (int i = 0; i < 9; ++i)
        for (int p = row[i].x + G + gl; p < row[i].y; p += G) insert(w.spos[p], KMAX);
    }
  } else {
    const int c = (cx * g.dy + cy) * g.dz + cz;
    for (int p = cell_start[c] + gl, e = cell_start[c + 1]; p < e; p += G) insert(w.spos[p], KMAX);
  }
  const int maxr = max(max(g.dx, g.dy), g.dz);
  const float ih2 = 1.00003f / (g.h * g.h);
  for (;;) {
    knn_merge_group<KMAX, G>(L);
    // distance (cell units) from the query to the faces of the visited block that still have
    // cells beyond them
    float gap = __builtin_inff();
    if (cx - r > 0) gap = fminf(gap, ux - static_cast<float>(cx - r));
    if (cx + r < g.dx - 1) gap = fminf(gap, static_cast<float>(cx + r + 1) - ux);
    if (cy - r > 0) gap = fminf(gap, uy - static_cast<float>(cy - r));
    if (cy + r < g.dy - 1) gap = fminf(gap, static_cast<float>(cy + r + 1) - uy);
    if (cz - r > 0) gap = fminf(gap, uz - static_cast<float>(cz - r));
    if (cz + r < g.dz - 1) gap = fminf(gap, static_cast<float>(cz + r + 1) - uz);
    if (gap == __builtin_inff()) break;  // every cell of the cloud visited
    const float gr = (gap - 1e-3f) * g.h;
    const float bound = gap > 1e-3f ? gr * gr * (1.0f - 1e-5f) : 0.0f;
#pragma unroll
    for (int i = 0; i < KMAX; ++i)
      if (i == k - 1) lim = L[i];
    if (lim < knn_key(bound, 0) || ++r > maxr) break;
    if (gl != 0) {
#pragma unroll
      for (int i = 0; i < KMAX; ++i) L[i] = none;
    }
    // shell r: rows on its x and y faces whole, the others by their two end cells
    const float kd = __int_as_float(__double2hiint(lim));  // inf while fewer than k are known
    const float cut = kd * ih2;                            // in squared cell units
    const int x0 = max(cx - r, 0), y0 = max(cy - r, 0);
    const int ny = min(cy + r, g.dy - 1) - y0 + 1;
    const int items = 2 * (min(cx + r, g.dx - 1) - x0 + 1) * ny;
    for (int t0 = 0; t0 < items; t0 += G) {
      const int t = t0 + gl;
      int2 own = make_int2(0, 0);
      if (t < items) {
        const unsigned rw = static_cast<unsigned>(t) >> 1;
        const int ix = x0 + static_cast<int>(rw / static_cast<unsigned>(ny));
        const int iy = y0 + static_cast<int>(rw % static_cast<unsigned>(ny));
        const float fx = static_cast<float>(ix), fy = static_cast<float>(iy);
        const float dx = fmaxf(fmaxf(fx - ux, ux - fx - 1.0f) - 1e-3f, 0.0f);
        const float dy = fmaxf(fmaxf(fy - uy, uy - fy - 1.0f) - 1e-3f, 0.0f);
        const float rem = cut - (dx * dx + dy * dy);
        int za = 0, zb = -1;
        if (!(rem < 0.0f)) {
          const float rz = sqrtf(rem) + 2e-3f;
          const bool face = ix == cx - r || ix == cx + r || iy == cy - r || iy == cy + r;
          if (!face) {
            za = zb = (t & 1) ? cz + r : cz - r;
            const float fz = static_cast<float>(za);
            if (za < 0 || za >= g.dz || fz - uz > rz || uz - fz - 1.0f > rz) zb = za - 1;
          } else if ((t & 1) == 0) {
            // a cell that ends below uz - rz or begins above uz + rz is too far
            const float z0 = static_cast<float>(max(cz - r, 0)), z1 = static_cast<float>(min(cz + r, g.dz - 1));
            za = static_cast<int>(fminf(fmaxf(floorf(uz - rz), z0), z1 + 1.0f));
            zb = static_cast<int>(fmaxf(fminf(floorf(uz + rz), z1), z0 - 1.0f));
          }
        }
        if (za <= zb) {
          const int c = (ix * g.dy + iy) * g.dz;
          own = make_int2(cell_start[c + za], cell_start[c + zb + 1]);
        }
      }
      uint64_t left = __ballot(own.x < own.y) >> gb;
      if constexpr (G < kWave) left &= (1ull << G) - 1;
      while (left != 0) {
        const int i0 = __builtin_ctzll(left);
        left &= left - 1;
        const int i1 = left != 0 ? __builtin_ctzll(left) : i0;
        const bool two = left != 0;
        left &= left - 1;
        const int a0 = __shfl(own.x, gb + i0, kWave), e0 = __shfl(own.y, gb + i0, kWave);
        const int a1 = __shfl(own.x, gb + i1, kWave), e1 = two ? __shfl(own.y, gb + i1, kWave) : a1;
        const float4 s0 = w.spos[a0 + gl < e0 ? a0 + gl : 0], s1 = w.spos[a1 + gl < e1 ? a1 + gl : 0];
        if (a0 + gl < e0) insert(s0, KMAX);
        if (a1 + gl < e1) insert(s1, KMAX);
        for (int p = a0 + G + gl; p < e0; p += G) insert(w.spos[p], KMAX);
        for (int p = a1 + G + gl; p < e1; p += G) insert(w.spos[p], KMAX);
      }
    }
  }
  int64_t* oi = out_idx + q * k;
  float* od = out_dist + q * k;
#pragma unroll
  for (int i = 0; i < KMAX; ++i) {
    if (i < k && i % G == gl) {
      const bool any = L[i] < none;
      oi[i] = any ? static_cast<int64_t>(__double2loint(L[i])) : -1;
      od[i] = any ? __int_as_float(__double2hiint(L[i])) : 1e30f;
    }
  }
}

bool knn_use_grid(int64_t Ns, int64_t B, int64_t k) {
  return k >= 1 && k <= kKnnGridMaxK && B >= 1 && Ns >= 1024 * B;
}

int launch_knn_grid(const float* query, int64_t Nq, const float* source, int64_t Ns,
                    const int64_t* ptr_q, const int64_t* ptr_s, int64_t B, int k, int64_t* out_idx,
                    float* out_dist, void* workspace, hipStream_t st) {
  size_t bytes = 0;
  const KnnGridWs w = carve_knn_grid(workspace, Ns, B, &bytes);
  // Clouds of up to kKnnBuildCells / kKnnCellCap points on average: each cloud's grid by one
  // workgroup, 10 us and one launch against 27 us and six (16 clouds of about 4096 points).  The sizes are not known here, and
  // one cloud may hold nearly all points: one workgroup needs as long as the six launches for about
  // 25,000 points and 70 us more for 65,000 (four clouds of 16,384 and four of 1 point, k = 16, 70
  // -> 46 us in all; 15 clouds of 64 points and one of 64,576 92 -> 133 us), so the sum is bounded.
  if (Ns <= B * (kKnnBuildCells / kKnnCellCap) && Ns <= kKnnBuildSources) {
    hipLaunchKernelGGL(knn_grid_build, dim3(static_cast<unsigned>(B)), dim3(kKnnSetupThreads), 0, st, source, Ns,
                       ptr_s, k, w);
    GEO_LAUNCH_CHECK("knn_grid_build");
  } else {
    // Clouds of more than 2 * kKnnBoxChunk points on average: the bounding box is reduced by up to
    // kKnnBoxParts workgroups per cloud first (one workgroup reading a 131,072-point cloud took
    // 23 us), the setup then combines their partial boxes.
    const int64_t avg = ceil_div(Ns, B);
    const int64_t want = ceil_div(avg, kKnnBoxChunk);
    const int parts = avg > 2 * kKnnBoxChunk ? static_cast<int>(want < kKnnBoxParts ? want : kKnnBoxParts) : 0;
    if (parts > 0) {
      hipLaunchKernelGGL(knn_grid_box_part, dim3(parts, static_cast<unsigned>(B)),
                         dim3(kKnnSetupThreads), 0, st, source, Ns, ptr_s, parts, w.box_part);
      GEO_LAUNCH_CHECK("knn_grid_box_part");
    }
    hipLaunchKernelGGL(knn_grid_setup, dim3(B), dim3(kKnnSetupThreads), 0, st, source, Ns, ptr_s, k,
                       w.grid, w.box_part, parts);
    GEO_LAUNCH_CHECK("knn_grid_setup");
    hipLaunchKernelGGL(knn_grid_base, dim3(1), dim3(kScanThreads), 0, st, w.grid, B);
    GEO_LAUNCH_CHECK("knn_grid_base");
    // cell counts and the scan's look-back status are carved next to each other: one zero fill
    const int64_t zero_words =
        (reinterpret_cast<char*>(w.cell_scan + scan_lookback_elems(w.cells_max + 1)) -
         reinterpret_cast<char*>(w.cell_cnt)) / static_cast<int64_t>(sizeof(int32_t));
    int rc = device_fill<int32_t>(w.cell_cnt, zero_words, 0, st);
    if (rc) return rc;
    const unsigned gs = static_cast<unsigned>(ceil_div(Ns, kKnnGridThreads));
    hipLaunchKernelGGL(knn_grid_cell, dim3(gs), dim3(kKnnGridThreads), 0, st, source, Ns, ptr_s, B, w);
    GEO_LAUNCH_CHECK("knn_grid_cell");
    rc = device_exclusive_scan_lookback<int32_t, int32_t>(w.cell_cnt, w.cells_max + 1, w.cell_start,
                                                          nullptr, false, w.cell_scan, st);
    if (rc) return rc;
    hipLaunchKernelGGL(knn_grid_scatter, dim3(gs), dim3(kKnnGridThreads), 0, st, source, Ns, w);
    GEO_LAUNCH_CHECK("knn_grid_scatter");
  }
  // Lanes per query: a wave runs as long as its slowest query.  In one scene-scale cloud (a
  // lidar frame) density varies by orders of magnitude, so the few queries in dense regions
  // scan hundreds of candidates: a whole wave per query for k <= 8 there (C5 with 8 lanes
  // 0.42 ms, 16 lanes 0.196, 32 lanes 0.152, 64 lanes 0.147 ms); batched object-scale clouds
  // are near uniform and do best with 8 (32 costs them ~10%).
  const bool wide = B == 1 && Ns >= kKnnWideSources;
#define GEO_KNN_GRID_LAUNCH(KV, GV)                                                             \
  {                                                                                             \
    const unsigned gq = static_cast<unsigned>(ceil_div(Nq * GV, kKnnGridThreads));             \
    hipLaunchKernelGGL((knn_grid_query<KV, GV>), dim3(gq), dim3(kKnnGridThreads), 0, st, query, \
                       Nq, ptr_q, B, w, k, out_idx, out_dist);                                  \
    GEO_LAUNCH_CHECK("knn_grid_query");                                                         \
    return GEO_OK;                                                                              \
  }
#define GEO_KNN_GRID_CASE(KV, GV)                                                               \
  if (k <= KV) {                                                                                \
    if (GV == 8 && wide) GEO_KNN_GRID_LAUNCH(KV, 64)                                             \
    GEO_KNN_GRID_LAUNCH(KV, GV)                                                                 \
  }
  GEO_KNN_GRID_CASE(1, 8) GEO_KNN_GRID_CASE(2, 8) GEO_KNN_GRID_CASE(4, 8)
  GEO_KNN_GRID_CASE(8, 8) GEO_KNN_GRID_CASE(16, 16) GEO_KNN_GRID_CASE(32, 16)
#undef GEO_KNN_GRID_CASE
#undef GEO_KNN_GRID_LAUNCH
  return set_error(GEO_ERR_UNSUPPORTED, "knn: k=%d unsupported by the grid search", k);
}

}  // namespace
}  // namespace geo

using namespace geo;

extern "C" size_t geo_knn_workspace_bytes(int64_t Nq, int64_t Ns, int64_t B, int64_t k) {
  (void)Nq;
  if (Ns < 0 || B < 0) return 0;
  if (knn_use_grid(Ns, B, k)) {
    size_t bytes = 0;
    carve_knn_grid(nullptr, Ns, B, &bytes);
    return bytes;
  }
  return static_cast<size_t>(B + 1) * sizeof(int64_t);
}

extern "C" int geo_knn(const float* query, int64_t Nq, const float* source, int64_t Ns,
                       const int64_t* ptr_q, const int64_t* ptr_s, int64_t B, int64_t k,
                       int64_t* out_idx, float* out_dist, void* workspace, size_t workspace_bytes,
                       void* stream) {
  GEO_REQUIRE(Nq >= 0 && Ns >= 0 && B >= 0, "knn: negative size");
  GEO_REQUIRE(k >= 0, "knn: k must be non-negative (got %lld)", (long long)k);
  GEO_REQUIRE(k < 0x7fffffffLL, "knn: k=%lld exceeds int32", (long long)k);
  GEO_REQUIRE(Nq < 0x7fffffffLL && Ns < 0x7fffffffLL, "knn: sizes exceed int32 indexing");
  if (Nq == 0 || k == 0) return GEO_OK;
  GEO_REQUIRE(query && out_idx && out_dist && ptr_q && ptr_s, "knn: null pointer");
  const size_t need = geo_knn_workspace_bytes(Nq, Ns, B, k);
  if (workspace == nullptr || workspace_bytes < need)
    return set_error(GEO_ERR_WORKSPACE, "knn: workspace %zu bytes, need %zu", workspace_bytes,
                     need);
  hipStream_t st = as_stream(stream);
  int64_t* tiles = static_cast<int64_t*>(workspace);
  if (B == 0) {
    // no clouds: every query row is padding
    int rc = device_fill<int64_t>(out_idx, Nq * k, -1, st);
    if (rc) return rc;
    return device_fill<float>(out_dist, Nq * k, 1e30f, st);
  }
  GEO_REQUIRE(Ns == 0 || source != nullptr, "knn: null source");
  const int kk = static_cast<int>(k);
  // the grid search writes every output row itself (padding for queries outside every cloud)
  if (knn_use_grid(Ns, B, k))
    return launch_knn_grid(query, Nq, source, Ns, ptr_q, ptr_s, B, kk, out_idx, out_dist,
                           workspace, st);
  // Queries outside every cloud keep padding.
  int rc = device_fill<int64_t>(out_idx, Nq * k, -1, st);
  if (rc) return rc;
  rc = device_fill<float>(out_dist, Nq * k, 1e30f, st);
  if (rc) return rc;
  hipLaunchKernelGGL(knn_prepare_kernel, dim3(1), dim3(kScanThreads), 0, st, ptr_q, B, Nq, tiles);
  GEO_LAUNCH_CHECK("knn_prepare_kernel");
  if (kk > kKnnMaxList) {  // passes of kKnnMaxList columns, the last one narrower
    for (int col0 = 0; col0 < kk; col0 += kKnnMaxList) {
      const int width = kk - col0 < kKnnMaxList ? kk - col0 : kKnnMaxList;
      rc = width <= 32 ? launch_knn<32>(query, Nq, source, Ns, ptr_q, ptr_s, tiles, B, kk, out_idx,
                                        out_dist, st, col0, width)
         : width <= 64 ? launch_knn<64>(query, Nq, source, Ns, ptr_q, ptr_s, tiles, B, kk, out_idx,
                                        out_dist, st, col0, width)
         : width <= 96 ? launch_knn<96>(query, Nq, source, Ns, ptr_q, ptr_s, tiles, B, kk, out_idx,
                                        out_dist, st, col0, width)
                       : launch_knn<128>(query, Nq, source, Ns, ptr_q, ptr_s, tiles, B, kk, out_idx,
                                         out_dist, st, col0, width);
      if (rc) return rc;
    }
    return GEO_OK;
  }
#define GEO_KNN_CASE(KV) \
  if (kk <= KV) return launch_knn<KV>(query, Nq, source, Ns, ptr_q, ptr_s, tiles, B, kk, out_idx, out_dist, st);
  GEO_KNN_CASE(1) GEO_KNN_CASE(2) GEO_KNN_CASE(3) GEO_KNN_CASE(4) GEO_KNN_CASE(5)
  GEO_KNN_CASE(6) GEO_KNN_CASE(7) GEO_KNN_CASE(8) GEO_KNN_CASE(10) GEO_KNN_CASE(12)
  GEO_KNN_CASE(16) GEO_KNN_CASE(24) GEO_KNN_CASE(32) GEO_KNN_CASE(48) GEO_KNN_CASE(64)
  GEO_KNN_CASE(96) GEO_KNN_CASE(128)
#undef GEO_KNN_CASE
  return set_error(GEO_ERR_UNSUPPORTED, "knn: k=%d unsupported", kk);
}
