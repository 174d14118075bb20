// fps.hip — farthest-point sampling for packed point clouds on gfx950.
//
// Replaces fps_kernel<512> (geoembodied/csrc/fps_kernel.cu:40-153) with the semantics of the
// CPU path _fps_iterative_fallback (geoembodied/csrc/__init__.py:600-654): start at the first
// point of the cloud, each step take the LOWEST index attaining max(min squared distance).
//
// Four kernels, chosen by the largest cloud of the batch:
//   bucketed (clouds of up to 8192 points, the common case): one 1024-thread workgroup per
//     cloud, points ordered along a Hilbert cell grid so that each register slot of a wave holds
//     a compact bucket of 64 points; a bucket is only updated when a new centroid can lower
//     one of its distances (an exact test, see below), and several centroids are taken from the
//     cached per-bucket maxima per round, where they provably follow each other.  A cloud of up
//     to 384 points is sampled by one wave of that workgroup.
//   register (8193 to 16384 points, few samples): thread t owns local points t, t+256, ... with x,
//     y, z and the running min distance in VGPRs; every point is updated every iteration.
//   large (8193 to 196,608 points): the bucket scheme with points sorted along the Hilbert curve
//     in the workspace and bucket records in LDS (see its section below).
//   streaming (larger clouds): positions read from HBM/L2 each iteration, running min
//     distance in the workspace.
// The register and streaming kernels reduce (distance bits, index) per iteration to one winner
// with one barrier: a wave max of the bits (DPP), the lowest index among the lanes holding it, then
// one LDS record per wave double-buffered by iteration parity.  Squared distances are non-negative
// floats, whose bit patterns order like the values.
#include "radix.hpp"

namespace geo {
namespace {

constexpr int kFpsThreads = 256;
constexpr int kFpsWaves = kFpsThreads / kWave;
constexpr int kFpsLdsPoints = 8192;         // largest cloud of the bucketed kernel
constexpr int kFpsRegisterPoints = 16384;   // largest cloud of the register kernel
constexpr int kFpsRegisterSamples = 80;     // most samples of a cloud it is chosen for
constexpr int kFpsBucketThreads = 1024;
constexpr int kFpsRound = 16;  // most centroids that one round of the bucketed kernel takes
constexpr int kFpsFew = 96;    // samples up to which it takes one centroid per step, see fps_is_few
constexpr int kFpsLead = 48;   // first centroids taken so by its largest variant; below kFpsFew
constexpr int kFpsStreamThreads = 1024;
constexpr int kFpsStreamWaves = kFpsStreamThreads / kWave;

struct alignas(8) FpsSlot {
  uint32_t dist_bits;
  uint32_t idx;
};

// prepare: clamp k to [0, n], exclusive offsets, total, max cloud, ptr validation.
__global__ __launch_bounds__(kScanThreads) void fps_prepare_kernel(
    const int64_t* __restrict__ ptr, const int64_t* __restrict__ kpb, int64_t k_all, int64_t B,
    int64_t N_total, int64_t* __restrict__ out_ptr, int64_t* __restrict__ info,
    int64_t* __restrict__ info_host, int64_t* __restrict__ most) {
  __shared__ int64_t lds[kScanThreads / kWave];
  __shared__ unsigned long long s_max, s_bad, s_most;
  constexpr unsigned long long kNone = ~0ull;
  if (threadIdx.x == 0) {
    s_max = s_most = 0;
    s_bad = (ptr[0] >= 0 && ptr[0] <= N_total) ? kNone : 1ull;  // 1-based entry index
  }
  __syncthreads();
  int64_t carry = 0;
  for (int64_t base = 0; base < B; base += kScanThreads) {
    const int64_t b = base + threadIdx.x;
    int64_t k = 0;
    if (b < B) {
      const int64_t p0 = ptr[b], p1 = ptr[b + 1];
      const int64_t n = p1 - p0;
      if (n < 0 || p1 > N_total) atomicMin(&s_bad, static_cast<unsigned long long>(b + 2));
      const int64_t nn = n > 0 ? n : 0;
      k = kpb ? kpb[b] : k_all;  // one k for every cloud when no per-cloud array is given
      k = k < 0 ? 0 : (k > nn ? nn : k);
      atomicMax(&s_max, static_cast<unsigned long long>(nn));
      if (most) atomicMax(&s_most, static_cast<unsigned long long>(k));
    }
    int64_t total;
    const int64_t off = block_exclusive_scan<int64_t>(k, lds, total);
    if (b < B) out_ptr[b] = carry + off;
    carry += total;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int64_t bad = s_bad == kNone ? 0 : static_cast<int64_t>(s_bad);
    out_ptr[B] = carry;
    info[0] = carry;
    info[1] = static_cast<int64_t>(s_max);
    info[2] = bad;
    if (most) *most = static_cast<int64_t>(s_most);
    if (info_host) {  // mapped pinned host copy, read by the host once this kernel has finished
      info_host[0] = carry;
      info_host[1] = static_cast<int64_t>(s_max);
      info_host[2] = bad;
      __threadfence_system();
    }
  }
}

// Wave-level argmax of (dist_bits, idx): max dist, lowest idx on ties.  Uniform result.
__device__ __forceinline__ void wave_argmax(uint32_t bits, uint32_t idx, uint32_t& wbits,
                                            uint32_t& widx) {
  wbits = wave_max_u32(bits);
  widx = wave_min_u32(bits == wbits ? idx : 0xffffffffu);
}

template <int PTS>
__global__ __launch_bounds__(kFpsThreads) void fps_register_kernel(
    const float* __restrict__ pos, const int64_t* __restrict__ ptr,
    const int64_t* __restrict__ out_ptr, int64_t* __restrict__ out_idx) {
  __shared__ FpsSlot slots[2][kFpsWaves];

  const int b = blockIdx.x;
  const int64_t start = ptr[b];
  const int n = static_cast<int>(ptr[b + 1] - start);
  const int64_t o0 = out_ptr[b];
  const int k = static_cast<int>(out_ptr[b + 1] - o0);
  const int t = threadIdx.x;
  const int w = t / kWave;
  if (k <= 0 || n <= 0) return;
  if (k >= n) {  // every point, in index order
    for (int i = t; i < n; i += kFpsThreads) out_idx[o0 + i] = start + i;
    return;
  }
  const float* P = pos + start * 3;

  float px[PTS], py[PTS], pz[PTS], md[PTS];
#pragma unroll
  for (int s = 0; s < PTS; ++s) {
    const int l = t + s * kFpsThreads;
    if (l < n) {
      px[s] = P[3 * l];
      py[s] = P[3 * l + 1];
      pz[s] = P[3 * l + 2];
      md[s] = __builtin_inff();
    } else {
      px[s] = py[s] = pz[s] = 0.f;
      md[s] = 0.f;  // never wins: its index is above every valid one
    }
  }
  float cx = P[0], cy = P[1], cz = P[2];
  if (t == 0) out_idx[o0] = start;

  for (int it = 1; it < k; ++it) {
    uint32_t bbits = 0, bidx = 0xffffffffu;
#pragma unroll
    for (int s = 0; s < PTS; ++s) {
      const int l = t + s * kFpsThreads;
      if (l < n) {
        const float d = sqdist(px[s], py[s], pz[s], cx, cy, cz);
        md[s] = fminf(md[s], d);
      }
      const uint32_t mb = __float_as_uint(md[s]);
      if (mb > bbits || bidx == 0xffffffffu) {
        bbits = mb;
        bidx = static_cast<uint32_t>(l);
      }
    }
    uint32_t wbits, widx;
    wave_argmax(bbits, bidx, wbits, widx);
    FpsSlot* sl = slots[it & 1];
    if (lane_id() == 0) sl[w] = FpsSlot{wbits, widx};
    lds_barrier();  // waves share only LDS in this loop
    uint32_t gbits = sl[0].dist_bits, gidx = sl[0].idx;
#pragma unroll
    for (int ww = 1; ww < kFpsWaves; ++ww) {
      const FpsSlot o = sl[ww];
      if (o.dist_bits > gbits || (o.dist_bits == gbits && o.idx < gidx)) {
        gbits = o.dist_bits;
        gidx = o.idx;
      }
    }
    gidx = __builtin_amdgcn_readfirstlane(gidx);
    cx = P[3 * gidx]; cy = P[3 * gidx + 1]; cz = P[3 * gidx + 2];
    if (t == 0) out_idx[o0 + it] = start + gidx;
  }
}

// ------------------------------------------------------------------ bucketed kernel ---
//
// Clouds of up to 8192 points.  The cloud is first ordered along a 16^3 Hilbert cell grid
// (LDS counting sort), so the 64 points a wave holds in one register slot -- a bucket -- lie
// close together.  Each bucket has its bounding box and a record of its farthest point: max min
// distance, lowest index attaining it, position, and the rest bound: the most that any other point
// of the bucket has left once that point is a centroid, max over p of min(md(p), d(p, farthest)),
// with the lowest index attaining that.
//
// The loop takes several centroids per round.  Order all records, and the rest bounds with them, by
// (distance, lower index), and let i be ahead of j.  Record j is the greedy choice right after the
// records ahead of it if
//   d(point i, point j) >= md(point j) for every i ahead (none of them lowers its point), and
//   rest bound of i comes after record j for every i ahead (no other point of their buckets, at the
//   value it can still have, comes first):
// every other point comes after its own bucket's record and values only fall, so nothing can come
// between.  The round takes the records from the front up to the first that fails (the first one
// never does).  Rounds therefore give exactly the one-at-a-time sequence; on 16 surface clouds of
// 4096 points a round takes 7.6 centroids (at most 16), 135 rounds for 1024 samples, 1.6 us each,
// where one centroid took 0.46 us: 470 -> 239 us.
// Equal distances (points on a lattice or in voxels): the rest bound's index is what keeps rounds
// long there.  With its distance alone, another point of a bucket at the record's distance ended
// the round, and rounds of one or two centroids cost more than one centroid at a time did.  16^3
// lattice to 1024 samples, one at a time -> distance alone -> now: in order 524 -> 820 -> 459 us,
// shuffled 525 -> 853 -> 268 us.  The index is looked for only where several points hold a
// bucket's max (elsewhere 0, before all others, which ends a round at an equal distance in another
// bucket: 3% more rounds on lattices).  It costs clouds of 1000 to 2000 points 1 to 3%.
// Where the first record's distance is 0 every point lies on a sample, and the lowest index is the
// choice for all that is left: no further rounds (one point 4096 times: 855 -> 28 us a call).
// A round costs two LDS barriers:
//   check   every wave tests the listed records pairwise, lane = 16 * (j mod 4) + i
//   update  the wave's buckets against the round's centroids (bound test below), records of the
//           buckets whose farthest point fell; the wave with the most of them sets the pace
//   rank    every wave places its own records among all (one ballot each) and lists the first 16
// Half the threads with twice the buckets each measured 310 us, a quarter 504 us; the check made by
// each record's own wave before the second barrier (no list of bounds) 240 us.
//
// Bound test, one lane per (bucket, centroid): with
//   g_a = max(lo_a - c_a, c_a - hi_a, 0),  lb = (g_x*g_x + g_y*g_y) + g_z*g_z
// evaluated with the same fp32 operations as the distance, every rounded operation is monotone,
// so lb <= d(p, c) holds exactly for every point p of the bucket; when lb >= the bucket's max
// min-distance no point of the bucket can change and the pair is skipped.  Skipping is therefore
// exact; a bucket's record is re-reduced only when its farthest point fell.
constexpr int kCellBits = 4;                  // 16 cells per axis
constexpr int kCells = 1 << (3 * kCellBits);  // 4096

__device__ __forceinline__ uint32_t spread10(uint32_t v) {  // 10 bits -> every third bit
  v &= 0x3ffu;
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

// Position of cell (x, y, z) (b <= 10 bits per axis) along the 3-D Hilbert curve: the
// coordinates are brought to the curve's transposed form (J. Skilling, "Programming the Hilbert
// curve", AIP Conf. Proc. 707, 381 (2004): undo the excess work of each level from the top bit
// down, then Gray-decode), and the transposed bits interleaved x, y, z from the most significant.
// Consecutive positions are adjacent cells, so runs of points in this order have smaller boxes
// than runs in Morton order, whose curve jumps between distant cells (C5, 64-point buckets: mean
// box volume 61 against 148, buckets passing the bound test per FPS iteration 11.7 against 21.5).
__device__ __forceinline__ uint32_t hilbert3(uint32_t x, uint32_t y, uint32_t z, int b) {
  uint32_t X[3] = {x, y, z};
  const uint32_t top = 1u << (b - 1);
  for (uint32_t q = top; q > 1; q >>= 1) {
    const uint32_t p = q - 1;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (X[i] & q) {
        X[0] ^= p;
      } else {
        const uint32_t t = (X[0] ^ X[i]) & p;
        X[0] ^= t;
        X[i] ^= t;
      }
    }
  }
  X[1] ^= X[0];
  X[2] ^= X[1];
  uint32_t t = 0;
  for (uint32_t q = top; q > 1; q >>= 1)
    if (X[2] & q) t ^= q - 1;
  return (spread10(X[0] ^ t) << 2) | (spread10(X[1] ^ t) << 1) | spread10(X[2] ^ t);
}

__device__ __forceinline__ int cell16(float p, float lo, float scale) {
  int c = static_cast<int>((p - lo) * scale);
  return c < 0 ? 0 : (c > 15 ? 15 : c);
}


// order[q] = local index of the cloud's q-th point along the Hilbert curve of a 16^3 cell grid
// over the cloud's bounding box (LDS counting sort by cell; the order within a cell follows the
// atomics, which only changes which bucket a point joins, never a result).  hist holds kCells
// ints, red 6 x (THREADS / 64) words, code_rank 8 n and order 4 n bytes; ends behind a barrier.
template <int THREADS>
__device__ void fps_hilbert_order(const float* __restrict__ P, int n, int* hist,
                                  uint32_t (*red)[THREADS / kWave], int2* code_rank, int* order) {
  constexpr int WAVES = THREADS / kWave;
  const int t = threadIdx.x;
  const int w = t / kWave;
  const int lane = lane_id();
  // 1. bounding box of the cloud
  {
    uint32_t mn[3] = {~0u, ~0u, ~0u}, mx[3] = {0u, 0u, 0u};
    for (int i = t; i < n; i += THREADS) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const uint32_t kk = float_order_key(P[3 * i + a]);
        mn[a] = min(mn[a], kk);
        mx[a] = max(mx[a], kk);
      }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      mn[a] = wave_min_u32(mn[a]);
      mx[a] = wave_max_u32(mx[a]);
    }
    if (lane == 0) {
#pragma unroll
      for (int a = 0; a < 3; ++a) { red[a][w] = mn[a]; red[3 + a][w] = mx[a]; }
    }
    for (int i = t; i < kCells; i += THREADS) hist[i] = 0;
    __syncthreads();
  }
  float lo[3], scale[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    uint32_t m0 = red[a][0], m1 = red[3 + a][0];
    for (int ww = 1; ww < WAVES; ++ww) { m0 = min(m0, red[a][ww]); m1 = max(m1, red[3 + a][ww]); }
    lo[a] = float_from_order_key(m0);
    const float ext = float_from_order_key(m1) - lo[a];
    scale[a] = ext > 0.f ? 16.f / ext : 0.f;
  }

  // 2. counting sort by Hilbert cell: int2 (code, rank) per point, then the order
  for (int i = t; i < n; i += THREADS) {
    const int cx = cell16(P[3 * i], lo[0], scale[0]);
    const int cy = cell16(P[3 * i + 1], lo[1], scale[1]);
    const int cz = cell16(P[3 * i + 2], lo[2], scale[2]);
    const int code = static_cast<int>(hilbert3(cx, cy, cz, kCellBits));
    code_rank[i] = make_int2(code, atomicAdd(&hist[code], 1));
  }
  __syncthreads();
  {  // exclusive scan of hist in place: thread t owns kCells / THREADS consecutive cells
    constexpr int PER = kCells / THREADS;
    int v[PER], s = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) { v[j] = hist[t * PER + j]; s += v[j]; }
    const int incl = wave_inclusive_sum_int(s);
    __syncthreads();
    if (lane == kWave - 1) red[0][w] = static_cast<uint32_t>(incl);
    __syncthreads();
    int off = incl - s;
    for (int ww = 0; ww < w; ++ww) off += static_cast<int>(red[0][ww]);
#pragma unroll
    for (int j = 0; j < PER; ++j) { hist[t * PER + j] = off; off += v[j]; }
  }
  __syncthreads();
  for (int i = t; i < n; i += THREADS) {
    const int2 cr = code_rank[i];
    order[hist[cr.x] + cr.y] = i;
  }
  __syncthreads();
}

// Order of the greedy choice as one double: distance bits (a non-negative float) above the index
// complement, so the larger distance comes first and, among equal ones, the lower index.  A
// positive double orders like its bit pattern, and 0x7f800000 (+inf as a float) in the high word
// is still a finite double.
__device__ __forceinline__ double fps_key(uint32_t bits, uint32_t idx) {
  return __hiloint2double(static_cast<int>(bits), static_cast<int>(~idx));
}
__device__ __forceinline__ uint32_t fps_key_index(double key) {
  return ~static_cast<uint32_t>(__double2loint(key));
}

// The lanes of a round's check that hold a pair (i, j): i = lane % 16 ahead of j = `j` + lane / 16.
// As constants: formed by a compare in every round they cost a few of the 1000 to 1600 ns it takes
// (16 clouds of 4096 points to 1024 samples 237.6 -> 234.3 us, one of 2048 to 512 145.4 -> 143.2; a
// branch around the compare of keys, taken where distances are equal, 152).
constexpr uint64_t fps_ahead(int j) {
  uint64_t m = 0;
  for (int r = 0; r < 4; ++r) m |= static_cast<uint64_t>((1u << (j + r)) - 1u) << (16 * r);
  return m;
}

// Clouds of up to kFpsWavePoints points: one wave, point s * 64 + lane in slot s of the lane, one
// centroid per step and no barrier.  They have too few buckets for rounds (up to 64 points are one,
// which gives one centroid per round).  What bounds a step is its chain of instructions, which grows
// with the slots; a round's is its two barriers.  Batches of 64 clouds, kernel times one at a time
// with a barrier -> rounds -> one wave: 64 points to 32 samples 18.2 -> 29.1 -> 6.2 us, 128 to 64 29.3
// -> 37.4 -> 12.5, 256 to 128 51.0 -> 47.6 -> 32.7, 384 to 192 74 -> 66 -> 60, to 380 139 -> 116 -> 118.
// With eight slots 512 points to 256 take 96 us against 75 of the rounds, 1024 with sixteen 165 / 77.
constexpr int kFpsWavePoints = 384;
template <int S>
__device__ __forceinline__ void fps_one_wave(const float* __restrict__ P, int n, int k, int64_t start,
                                             int64_t* __restrict__ out) {
  const int lane = lane_id();
  float px[S], py[S], pz[S];
  uint32_t md[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int i = s * kWave + lane, at = i < n ? i : 0;
    px[s] = P[3 * at]; py[s] = P[3 * at + 1]; pz[s] = P[3 * at + 2];
    md[s] = i < n ? 0x7f800000u : 0u;  // padding never comes before point 0
  }
  int l = 0, idx = 0;
  float cx = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(px[0])));
  float cy = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(py[0])));
  float cz = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(pz[0])));
  for (int it = 0;; ++it) {
    if (lane == 0) out[it] = start + idx;
    if (it + 1 >= k) break;
    uint32_t m = 0u;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      md[s] = min(md[s], __float_as_uint(sqdist(px[s], py[s], pz[s], cx, cy, cz)));
      m = max(m, md[s]);
    }
    m = wave_max_u32(m);
    // the first slot that holds the maximum, its first lane: the lowest index
#pragma unroll
    for (int s = S - 1; s >= 0; --s) {
      const uint64_t hit = __ballot(md[s] == m);
      if (hit) {  // wave-uniform
        l = __builtin_ctzll(hit);
        idx = s * kWave + l;
        cx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px[s]), l));
        cy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py[s]), l));
        cz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pz[s]), l));
      }
    }
  }
}

// The greedy choice over a workgroup from each wave's maximum m (bits) and lowest index j attaining
// it.  best: three zeroed slots used in turn, `at` the next one.
__device__ __forceinline__ int fps_best(unsigned long long* best, int& at, uint32_t m, uint32_t j) {
  if (lane_id() == 0) atomicMax(&best[at], (static_cast<unsigned long long>(m) << 32) | static_cast<uint32_t>(~j));
  lds_barrier();
  const int idx = __builtin_amdgcn_readfirstlane(static_cast<int>(~static_cast<uint32_t>(best[at])));
  // every wave has read the slot before this one, which is next used two barriers on
  at = at == 2 ? 0 : at + 1;
  if (threadIdx.x == 0) best[at == 2 ? 0 : at + 1] = 0;
  return idx;
}

// Few samples of a cloud of more than kFpsWavePoints points: one centroid per step by the whole
// workgroup, the points in registers as they come and in LDS (xyz, 12 B per point).  Ordering the
// cloud does not pay for so few, and the first centroids lower nearly every point, so that rounds
// take one or two of them.  What bounds a step is its vector instructions (eight points a lane: 0.79
// us) and below that its barrier, the atomic and the chain behind it (one point: 0.34 us).
// Call times with rounds -> now, 16 surface clouds: 4096 points to 16 samples 41 -> 25 us, to 64 67 ->
// 45, to 128 88 -> 81, to 192 100 / 116; 8192 points to 32 82 -> 38, to 96 125 -> 89; 1024 points to 64
// 42 -> 32, to 128 57 / 56, to 192 70 / 79.  One cloud, where rounds pay earliest: 2048 points to 96 52 ->
// 50, to 128 60 / 64; 4096 to 128 84 -> 79.  Above 4096 points the rounds begin with such steps too
// (kFpsLead) and pay from about 110 samples on (4200 points to 128 104 / 121).
template <int PTS>
__device__ __forceinline__ bool fps_is_few(int k, int n) {
  if (n <= 512) return k <= 128;  // at most eight buckets: 256 clouds of 400 to 128 61 -> 54 us
  return k <= (PTS == 8 ? kFpsFew : max(kFpsFew, 64 + n / 64));
}
template <int PTS, int THREADS>
__device__ __forceinline__ void fps_few(const float* __restrict__ P, int n, int k, int64_t start,
                                        int64_t* __restrict__ out, float* xyz,
                                        unsigned long long* best) {
  const int t = threadIdx.x, lane = lane_id();
  float px[PTS], py[PTS], pz[PTS];
  uint32_t md[PTS];
  for (int i = t; i < 3 * n; i += THREADS) xyz[i] = P[i];
  if (t < 3) best[t] = 0;
  lds_barrier();
#pragma unroll
  for (int s = 0; s < PTS; ++s) {
    const int i = s * THREADS + t, at = i < n ? i : 0;
    px[s] = xyz[3 * at]; py[s] = xyz[3 * at + 1]; pz[s] = xyz[3 * at + 2];
    md[s] = i < n ? 0x7f800000u : 0u;  // padding never comes before point 0
  }
  int idx = 0, at = 0;  // at: the slot of best in use
  for (int it = 0;; ++it) {
    if (t == 0) out[it] = start + idx;
    if (it + 1 >= k) break;
    const float cx = xyz[3 * idx], cy = xyz[3 * idx + 1], cz = xyz[3 * idx + 2];
    uint32_t m = 0u;
#pragma unroll
    for (int s = 0; s < PTS; ++s) {
      md[s] = min(md[s], __float_as_uint(sqdist(px[s], py[s], pz[s], cx, cy, cz)));
      m = max(m, md[s]);
    }
    m = wave_max_u32(m);
    // the wave's first slot that holds the maximum, its first lane: the lowest index
    uint32_t j = 0;
#pragma unroll
    for (int s = PTS - 1; s >= 0; --s) {
      const uint64_t hit = __ballot(md[s] == m);
      if (hit) j = static_cast<uint32_t>(s * THREADS + (t - lane) + __builtin_ctzll(hit));
    }
    idx = fps_best(best, at, m, j);
  }
}

template <int PTS, int THREADS>
__global__ __launch_bounds__(THREADS) void fps_bucket_kernel(
    const float* __restrict__ pos, const int64_t* __restrict__ ptr,
    const int64_t* __restrict__ out_ptr, int64_t* __restrict__ out_idx,
    const int64_t* __restrict__ guard) {
  constexpr int WAVES = THREADS / kWave;
  constexpr int NB = PTS * WAVES;              // buckets
  constexpr int SETS = (NB + kWave - 1) / kWave;  // records per lane in the selection
  constexpr int TESTS = (PTS + 3) / 4;         // bound tests per round: 4 slots x 16 centroids each
  // Launched before the host has seen the prepare kernel's summary: do nothing unless ptr was
  // valid and every cloud fits this variant (the host then launches the right one).
  if (guard != nullptr && (guard[2] != 0 || guard[1] > PTS * THREADS)) return;
  __shared__ double rkey[NB < kWave ? kWave : NB];  // key of each bucket's farthest point, see fps_key
  __shared__ float4 list[kFpsRound];   // the first records: position, (bits) min distance
  __shared__ double2 lkey[kFpsRound];  // their keys and rest bounds
  __shared__ int hist[kCells];
  __shared__ uint32_t red[6][WAVES];
  extern __shared__ int2 scratch[];  // sort scratch, 12 B per point

  const int b = blockIdx.x;
  const int64_t start = ptr[b];
  const int n = static_cast<int>(ptr[b + 1] - start);
  const int64_t o0 = out_ptr[b];
  const int k = static_cast<int>(out_ptr[b + 1] - o0);
  const int t = threadIdx.x;
  const int w = t / kWave;
  const int lane = lane_id();
  if (k <= 0 || n <= 0) return;
  if (k >= n) {
    for (int i = t; i < n; i += THREADS) out_idx[o0 + i] = start + i;
    return;
  }
  const float* P = pos + start * 3;
  if (n <= kFpsWavePoints) {
    if (w != 0) return;
    if (n <= kWave) fps_one_wave<1>(P, n, k, start, out_idx + o0);
    else if (n <= 2 * kWave) fps_one_wave<2>(P, n, k, start, out_idx + o0);
    else if (n <= 4 * kWave) fps_one_wave<4>(P, n, k, start, out_idx + o0);
    else fps_one_wave<6>(P, n, k, start, out_idx + o0);
    return;
  }

  if (fps_is_few<PTS>(k, n)) {
    fps_few<PTS, THREADS>(P, n, k, start, out_idx + o0, reinterpret_cast<float*>(scratch),
                          reinterpret_cast<unsigned long long*>(rkey));
    return;
  }

  // 1-2. the cloud ordered along the Hilbert curve of its cell grid
  int2* code_rank = scratch;
  int* order = reinterpret_cast<int*>(scratch + n);
  fps_hilbert_order<THREADS>(P, n, hist, red, code_rank, order);

  // 3. registers.  Bucket j = 64 consecutive sorted points; wave w owns buckets w, w+WAVES, ...
  //    (neighbouring buckets on different waves, so the buckets near a centroid spread over
  //    the SIMDs); slot s of wave w holds bucket s*WAVES + w.
  float px[PTS], py[PTS], pz[PTS];
  uint32_t md[PTS], oi[PTS];  // running min distance (bits), index
  // loads at clamped slots, values selected after (a load under `q < n` became a branch and a
  // wait before the next slot's)
#pragma unroll
  for (int s = 0; s < PTS; ++s) {
    const int q = (s * WAVES + w) * kWave + lane;
    const bool in = q < n;
    const int i = order[in ? q : 0];
    const float x = P[3 * i], y = P[3 * i + 1], z = P[3 * i + 2];
    oi[s] = in ? static_cast<uint32_t>(i) : 0xffffffffu;
    px[s] = in ? x : 0.f;
    py[s] = in ? y : 0.f;
    pz[s] = in ? z : 0.f;
    md[s] = in ? 0x7f800000u : 0u;  // padding: never changes, never wins
  }

  // The first centroids lower nearly every point, and a round of one or two of them that forms all
  // records again (eight a wave) takes longer than a step that only lowers and compares: without
  // them 16 clouds of 8192 points to 192 samples took 180 us (143 with), to 512 269 (237), 6000
  // points to 192 161 (140); a cloud of 8192 to 4096 972 (937).
  constexpr int lead = PTS == 8 ? kFpsLead : 0;
  if constexpr (lead > 0) {
    float* xyz = reinterpret_cast<float*>(scratch);
    unsigned long long* best = reinterpret_cast<unsigned long long*>(rkey);
    lds_barrier();  // the order is read
#pragma unroll
    for (int s = 0; s < PTS; ++s) {
      if (oi[s] == 0xffffffffu) continue;
      xyz[3 * oi[s]] = px[s];
      xyz[3 * oi[s] + 1] = py[s];
      xyz[3 * oi[s] + 2] = pz[s];
    }
    if (t < 3) best[t] = 0;
    lds_barrier();
    int idx = 0, at = 0;
    for (int it = 0;; ++it) {
      if (t == 0) out_idx[o0 + it] = start + idx;
      const float cx = xyz[3 * idx], cy = xyz[3 * idx + 1], cz = xyz[3 * idx + 2];
      uint32_t m = 0u;
#pragma unroll
      for (int s = 0; s < PTS; ++s) {
        md[s] = min(md[s], __float_as_uint(sqdist(px[s], py[s], pz[s], cx, cy, cz)));
        m = max(m, md[s]);
      }
      if (it + 1 == lead) break;
      m = wave_max_u32(m);
      uint32_t j = 0xffffffffu;
#pragma unroll
      for (int s = 0; s < PTS; ++s) j = min(j, md[s] == m ? oi[s] : 0xffffffffu);
      idx = fps_best(best, at, m, wave_min_u32(j));
    }
    lds_barrier();  // rkey holds the records from here on
  }

  // 4. bucket records: box and max (bits) of slot 4 h + lane / 16 in the lane; the farthest point
  //    (bits, index, lane, position) and the rest bound of slot s as scalars.
  float blx[TESTS], bly[TESTS], blz[TESTS], bhx[TESTS], bhy[TESTS], bhz[TESTS];
  uint32_t bmax[TESTS];
  uint32_t bm[PTS], bi[PTS], al[PTS], rs[PTS];
  uint32_t ri[PTS];  // lowest index at the rest bound, 0 = not known
  float sx[PTS], sy[PTS], sz[PTS];
  // the record and rest bound of slot s, whose points have the min distances mb (bits)
  auto record = [&](int s, uint32_t mb) {
    const uint32_t mx = wave_max_u32(mb);
    const uint64_t hit = __ballot(mb == mx);
    ri[s] = 0u;
    if ((hit & (hit - 1)) == 0) {  // one lane holds the maximum (distance ties are rare)
      al[s] = static_cast<uint32_t>(__builtin_ctzll(hit));
      bi[s] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(oi[s]), al[s]));
    } else {
      bi[s] = wave_min_u32(mb == mx ? oi[s] : 0xffffffffu);
      al[s] = static_cast<uint32_t>(__builtin_ctzll(__ballot(mb == mx && oi[s] == bi[s]) | (1ull << 63)));
      // the others at the maximum that stay there
      const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px[s]), al[s]));
      const float y = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py[s]), al[s]));
      const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pz[s]), al[s]));
      const bool stay = mb == mx && __float_as_uint(sqdist(px[s], py[s], pz[s], x, y, z)) >= mx;
      if (__ballot(stay)) ri[s] = wave_min_u32(stay ? oi[s] : 0xffffffffu);
    }
    bm[s] = mx;
    if (lane / 16 == s % 4) bmax[s / 4] = mx;
    if (lane == 0) rkey[s * WAVES + w] = fps_key(mx, bi[s]);
    sx[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px[s]), al[s]));
    sy[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py[s]), al[s]));
    sz[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pz[s]), al[s]));
    // what the bucket's other points can reach once that point is a centroid (its own lane
    // gives 0)
    rs[s] = wave_max_u32(
        min(mb, __float_as_uint(sqdist(px[s], py[s], pz[s], sx[s], sy[s], sz[s]))));
  };
#pragma unroll
  for (int h = 0; h < TESTS; ++h) {
    blx[h] = bly[h] = blz[h] = __builtin_inff();
    bhx[h] = bhy[h] = bhz[h] = -__builtin_inff();
    bmax[h] = 0u;
  }
#pragma unroll
  for (int s = 0; s < PTS; ++s) {
    const bool valid = oi[s] != 0xffffffffu;
    const uint32_t l0 = wave_min_u32(valid ? float_order_key(px[s]) : ~0u);
    const uint32_t l1 = wave_min_u32(valid ? float_order_key(py[s]) : ~0u);
    const uint32_t l2 = wave_min_u32(valid ? float_order_key(pz[s]) : ~0u);
    const uint32_t h0 = wave_max_u32(valid ? float_order_key(px[s]) : 0u);
    const uint32_t h1 = wave_max_u32(valid ? float_order_key(py[s]) : 0u);
    const uint32_t h2 = wave_max_u32(valid ? float_order_key(pz[s]) : 0u);
    const bool any = (s * WAVES + w) * kWave < n;
    if constexpr (lead > 0) {
      if (lane / 16 == s % 4 && any) {
        blx[s / 4] = float_from_order_key(l0); bly[s / 4] = float_from_order_key(l1);
        blz[s / 4] = float_from_order_key(l2); bhx[s / 4] = float_from_order_key(h0);
        bhy[s / 4] = float_from_order_key(h1); bhz[s / 4] = float_from_order_key(h2);
      }
      record(s, md[s]);
      continue;
    }
    // no centroid yet: every distance is +inf, so the record is the lowest index; it stands until that point falls,
    // which it never does where squared distances overflow (no update then touches the bucket)
    bm[s] = any ? 0x7f800000u : 0u;
    bi[s] = wave_min_u32(oi[s]);
    al[s] = static_cast<uint32_t>(__builtin_ctzll(__ballot(oi[s] == bi[s]) | (1ull << 63)));
    rs[s] = 0x7f800000u;
    ri[s] = 0u;
    sx[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(px[s]), al[s]));
    sy[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(py[s]), al[s]));
    sz[s] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pz[s]), al[s]));
    if (lane / 16 == s % 4 && any) {
      blx[s / 4] = float_from_order_key(l0); bly[s / 4] = float_from_order_key(l1);
      blz[s / 4] = float_from_order_key(l2); bhx[s / 4] = float_from_order_key(h0);
      bhy[s / 4] = float_from_order_key(h1); bhz[s / 4] = float_from_order_key(h2);
      bmax[s / 4] = 0x7f800000u;
    }
    if (lane == 0) rkey[s * WAVES + w] = fps_key(bm[s], bi[s]);
  }
  if (NB < kWave && t >= NB && t < kWave) rkey[t] = 0.0;  // no key is below 0
  if (t == 0) {
    list[0] = make_float4(P[0], P[1], P[2], __builtin_inff());
    lkey[0] = make_double2(fps_key(0u, 0u), 0.0);
  }
  // rank: every wave places its own records among all of them and lists the first kFpsRound
  auto rank_records = [&]() {
    double kk[SETS];
#pragma unroll
    for (int e = 0; e < SETS; ++e) {
      kk[e] = rkey[e * kWave + lane];
    }
#pragma unroll
    for (int s = 0; s < PTS; ++s) {
      const double kj = fps_key(bm[s], bi[s]);
      int rank = 0;
#pragma unroll
      for (int e = 0; e < SETS; ++e) rank += __builtin_popcountll(__ballot(kk[e] > kj));
      if (rank < kFpsRound && (s * WAVES + w) * kWave < n && lane == 0) {
        list[rank] = make_float4(sx[s], sy[s], sz[s], __uint_as_float(bm[s]));
        lkey[rank] = make_double2(kj, fps_key(rs[s], ri[s]));
      }
    }
  };
  lds_barrier();
  if constexpr (lead > 0) {
    rank_records();
    lds_barrier();
  }

  // records that exist: no more can be taken in one round
  const int cap = min(kFpsRound, (n + kWave - 1) / kWave);
  const int li = lane & (kFpsRound - 1);
  int done = lead, kend = k;
  for (;;) {
    // which of the listed records are the next centroids: record j is one if no record i ahead of
    // it can lower its point, and no other point of a bucket ahead can come before it
    const float4 c = list[li];
    const double rb = lkey[li].y;
    int A = 1;
    if (done != 0) {
      A = kFpsRound;
#pragma unroll
      for (int g = 0; g < kFpsRound; g += 8) {  // four records per step, lane = 16 * record + i
        const int j0 = g + lane / 16, j1 = j0 + 4;
        const float4 p0 = list[j0], p1 = list[j1];
        const uint32_t d0 = __float_as_uint(sqdist(c.x, c.y, c.z, p0.x, p0.y, p0.z));
        const uint32_t d1 = __float_as_uint(sqdist(c.x, c.y, c.z, p1.x, p1.y, p1.z));
        const uint64_t b0 = (__ballot(d0 < __float_as_uint(p0.w)) | __ballot(rb > lkey[j0].x)) & fps_ahead(g);
        const uint64_t b1 = (__ballot(d1 < __float_as_uint(p1.w)) | __ballot(rb > lkey[j1].x)) & fps_ahead(g + 4);
        if (b0 | b1) {
          A = g + (b0 ? __builtin_ctzll(b0) : 64 + __builtin_ctzll(b1)) / 16;
          break;
        }
      }
      A = min(min(A, cap), kend - done);
      // every point lies on a sample (through kend: another exit from the loop costs 2%)
      if (A == 1 && __builtin_amdgcn_readfirstlane(__float_as_int(c.w)) == 0) kend = A = 0;
    }
    if (w == 0 && lane < A) out_idx[o0 + done + lane] = start + fps_key_index(lkey[li].x);
    done += A;
    if (done >= kend) break;

    // update: the wave's buckets against the round's centroids
#pragma unroll
    for (int h = 0; h < TESTS; ++h) {
      float gx, gy, gz;
      {
#pragma clang fp contract(off)
        gx = fmaxf(fmaxf(blx[h] - c.x, c.x - bhx[h]), 0.f);
        gy = fmaxf(fmaxf(bly[h] - c.y, c.y - bhy[h]), 0.f);
        gz = fmaxf(fmaxf(blz[h] - c.z, c.z - bhz[h]), 0.f);
      }
      const float lb = sqdist(gx, gy, gz, 0.f, 0.f, 0.f);
      const uint64_t act = __ballot(__float_as_uint(lb) < bmax[h]) & __ballot(li < A);
      if (!act) continue;
#pragma unroll
      for (int s = 4 * h; s < PTS && s < 4 * h + 4; ++s) {
        uint32_t m = static_cast<uint32_t>(act >> (16 * (s % 4))) & 0xffffu;
        if (!m) continue;
        const uint32_t old = md[s];
        uint32_t mb = old;
        do {
          const int l = __builtin_ctz(m);
          m &= m - 1;
          const float cx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.x), l));
          const float cy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.y), l));
          const float cz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.z), l));
          // distances are non-negative floats, ordered like their bit patterns: the running
          // minimum is an integer min (no NaN canonicalisation step)
          mb = min(mb, __float_as_uint(sqdist(px[s], py[s], pz[s], cx, cy, cz)));
        } while (m);
        md[s] = mb;
        // Values only fall: while the point holding the bucket's max keeps its value, the record
        // (max, lowest index attaining it) stands, and its rest bound still holds.
        if (!((__ballot(mb < old) >> al[s]) & 1ull)) continue;
        record(s, mb);
      }
    }
    lds_barrier();  // waves share only LDS in this loop

    rank_records();
    lds_barrier();
  }
  for (int i = done + t; i < k; i += THREADS) out_idx[o0 + i] = start;  // distances all 0
}

template <int PTS, int THREADS>
int launch_bucket(const float* pos, const int64_t* ptr, const int64_t* out_ptr, int64_t B,
                  int64_t max_cloud, int64_t* out, hipStream_t st,
                  const int64_t* guard = nullptr) {
  const size_t lds = static_cast<size_t>(max_cloud > 0 ? max_cloud : 1) * 12;
  GEO_HIP_CHECK(hipFuncSetAttribute(
      reinterpret_cast<const void*>(&fps_bucket_kernel<PTS, THREADS>),
      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kFpsLdsPoints * 12)));
  hipLaunchKernelGGL((fps_bucket_kernel<PTS, THREADS>), dim3(B), dim3(THREADS), lds, st, pos, ptr,
                     out_ptr, out, guard);
  GEO_LAUNCH_CHECK("fps_bucket_kernel");
  return GEO_OK;
}

// Streaming kernel for clouds larger than the register kernel holds.
__global__ __launch_bounds__(kFpsStreamThreads) void fps_stream_kernel(
    const float* __restrict__ pos, const int64_t* __restrict__ ptr,
    const int64_t* __restrict__ out_ptr, int64_t* __restrict__ out_idx, float* __restrict__ mind) {
  __shared__ FpsSlot slots[2][kFpsStreamWaves];
  const int b = blockIdx.x;
  const int64_t start = ptr[b];
  const int n = static_cast<int>(ptr[b + 1] - start);
  const int64_t o0 = out_ptr[b];
  const int k = static_cast<int>(out_ptr[b + 1] - o0);
  const int t = threadIdx.x;
  const int w = t / kWave;
  if (k <= 0 || n <= 0) return;
  if (k >= n) {
    for (int i = t; i < n; i += kFpsStreamThreads) out_idx[o0 + i] = start + i;
    return;
  }
  const float* P = pos + start * 3;
  float* M = mind + start;
  for (int i = t; i < n; i += kFpsStreamThreads) M[i] = __builtin_inff();
  float cx = P[0], cy = P[1], cz = P[2];
  if (t == 0) out_idx[o0] = start;
  __syncthreads();
  for (int it = 1; it < k; ++it) {
    uint32_t bbits = 0, bidx = 0xffffffffu;
    for (int i = t; i < n; i += kFpsStreamThreads) {
      const float d = sqdist(P[3 * i], P[3 * i + 1], P[3 * i + 2], cx, cy, cz);
      const float m = fminf(M[i], d);
      M[i] = m;
      const uint32_t mb = __float_as_uint(m);
      if (mb > bbits || bidx == 0xffffffffu) {
        bbits = mb;
        bidx = static_cast<uint32_t>(i);
      }
    }
    uint32_t wbits, widx;
    wave_argmax(bbits, bidx, wbits, widx);
    FpsSlot* sl = slots[it & 1];
    if (lane_id() == 0) sl[w] = FpsSlot{wbits, widx};
    lds_barrier();  // each thread reads back only its own M entries: waves share only LDS
    uint32_t gbits = sl[0].dist_bits, gidx = sl[0].idx;
    for (int ww = 1; ww < kFpsStreamWaves; ++ww) {
      const FpsSlot o = sl[ww];
      if (o.dist_bits > gbits || (o.dist_bits == gbits && o.idx < gidx)) {
        gbits = o.dist_bits;
        gidx = o.idx;
      }
    }
    gidx = __builtin_amdgcn_readfirstlane(gidx);
    cx = P[3 * gidx]; cy = P[3 * gidx + 1]; cz = P[3 * gidx + 2];
    if (t == 0) out_idx[o0 + it] = start + gidx;
  }
}

// ---------------------------------------------------------------------------- large clouds ---
// Clouds larger than the bucketed kernel holds (up to kFpsLargeMaxPoints).  The batch is
// reordered by a device radix sort on (cloud + 1, Hilbert position of the point in its cloud's
// box), which keeps every cloud on its own index range, and each cloud is cut into buckets of 64
// consecutive sorted points.  Positions (with the original index) and running min distances
// stay in the workspace, 20 bytes per point, which for one cloud fits the L2 of the XCD that
// runs it.  One 1024-thread workgroup per cloud takes several centroids per round, by the rule of
// the bucketed kernel over the records in LDS:
//   check   the listed records pairwise (every wave)
//   test    boxes of 64 buckets against all centroids, then the buckets of the boxes that one may
//           reach; touched buckets join a queue with the set of their centroids
//   update  the queue shared by all waves, three buckets of a wave loaded together; records whose
//           farthest point fell are re-reduced and their groups marked
//   groups  buckets g, g + 128, ... form group g, so neighbouring buckets lie in different groups;
//           best and second record of the marked groups, one 16-lane row each
//   rank    no record other than a group's best comes before the first second record t0, so the bests
//           before t0, in order, are the next records of the whole cloud: the list
// A 32^3 lattice to 4096 samples, one at a time -> rounds by distance alone -> now: in order 5.55 ->
// 7.79 -> 3.15 ms, shuffled 5.51 -> 7.76 -> 1.91 ms.
// A 131,072-point lidar frame to 16,384 samples: 1,634 rounds of 10.0 centroids and 5.5 us,
// 22.4 -> 9.1 ms (one centroid per iteration took 1.36 us).  A round of 13,300 cycles issues 461
// vector instructions per wave, 55% of what the CU's four SIMDs can issue in that time.  Tried
// without gain: the queue's buckets handed to whichever wave is free (9.3 ms), tests per 16 buckets
// with a centroid list per row (9.3), one bucket prefetched ahead (9.6), four or eight loaded
// together (9.2, 9.6), min distances stored only where they fell (9.5: the conditional store makes
// every later load wait for it).
constexpr int kFpsLargeThreads = 1024;
constexpr int kFpsLargeWaves = kFpsLargeThreads / kWave;
constexpr int kFpsLargeSlots = 3;
constexpr int kFpsLargeBatch = 3;  // a wave's queued buckets loaded together
constexpr int64_t kFpsLargeMaxPoints =
    static_cast<int64_t>(kFpsLargeSlots) * kFpsLargeThreads * kWave;  // 196,608
constexpr int64_t kFpsLargeMaxClouds = (1 << 11) - 2;                  // cloud id + 1 in 11 bits

// bbox[6 b .. 6 b + 5] = (lo x, lo y, lo z, hi x, hi y, hi z) of cloud b; one block per cloud.
__global__ __launch_bounds__(kFpsLargeThreads) void fps_large_bbox_kernel(
    const float* __restrict__ pos, const int64_t* __restrict__ ptr, float* __restrict__ bbox) {
  __shared__ uint32_t red[6][kFpsLargeWaves];
  const int b = blockIdx.x;
  const int64_t s = ptr[b], e = ptr[b + 1];
  const int t = threadIdx.x, w = t / kWave;
  uint32_t mn[3] = {~0u, ~0u, ~0u}, mx[3] = {0u, 0u, 0u};
  for (int64_t i = s + t; i < e; i += kFpsLargeThreads) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t kk = float_order_key(pos[3 * i + a]);
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
    for (int ww = 1; ww < kFpsLargeWaves; ++ww) v = t < 3 ? min(v, red[t][ww]) : max(v, red[t][ww]);
    bbox[6 * b + t] = (e > s) ? float_from_order_key(v) : 0.f;
  }
}

// keys[i] = (cloud + 1) << 3 mbits | Hilbert position (mbits per axis) of point i in its cloud's
// box; points before the first cloud get cloud field 0, points after the last B + 1.
__global__ void fps_large_keys_kernel(const float* __restrict__ pos, const int64_t* __restrict__ ptr,
                                      int64_t B, int64_t N, const float* __restrict__ bbox,
                                      int mbits, uint32_t* __restrict__ keys) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= N) return;
  int64_t lo = 0, hi = B + 1;  // number of ptr entries <= i
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (ptr[mid] <= i) lo = mid + 1; else hi = mid;
  }
  uint32_t code = 0;
  if (lo >= 1 && lo <= B) {
    const float* bb = bbox + 6 * (lo - 1);
    const float cells = static_cast<float>(1 << mbits);
    uint32_t c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float ext = bb[3 + a] - bb[a];
      const float q = ext > 0.f ? (pos[3 * i + a] - bb[a]) * (cells / ext) : 0.f;
      const int ci = static_cast<int>(q);
      c[a] = static_cast<uint32_t>(ci < 0 ? 0 : (ci >= (1 << mbits) ? (1 << mbits) - 1 : ci));
    }
    code = hilbert3(c[0], c[1], c[2], mbits);
  }
  keys[i] = (static_cast<uint32_t>(lo) << (3 * mbits)) | code;
}

// Bucket j of cloud b (64 sorted points, one wave): positions and original index bits, min distances
// +inf, and the bucket's box at boxes[a][fps_large_box0 + j] (lo x, y, z, hi x, y, z by a).  The
// points lie in sorted order, except that the one with the lowest index changes places with the
// first: it is the bucket's record while all distances are +inf.
__device__ __forceinline__ int64_t fps_large_box0(int64_t start, int b) { return (start >> 6) + b; }

__global__ __launch_bounds__(256) void fps_large_gather_kernel(
    const float* __restrict__ pos, const uint32_t* __restrict__ order, const int64_t* __restrict__ ptr,
    int64_t box_stride, float4* __restrict__ q, uint32_t* __restrict__ md, float* __restrict__ boxes) {
  const int b = blockIdx.y;
  const int64_t start = ptr[b], n = ptr[b + 1] - start;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * 4 + threadIdx.x / kWave;
  if (j * kWave >= n) return;
  const int lane = lane_id();
  const int64_t l = j * kWave + lane;
  const int64_t at = start + (l < n ? l : n - 1);  // past the end: the last point again
  const uint32_t i = order[at];
  const float x = pos[3 * static_cast<int64_t>(i)], y = pos[3 * static_cast<int64_t>(i) + 1],
              z = pos[3 * static_cast<int64_t>(i) + 2];
  const int low = __builtin_ctzll(__ballot(i == wave_min_u32(i)) | (1ull << 63));
  if (l < n) {
    q[lane == low ? at - lane : (lane == 0 ? at + low : at)] = make_float4(x, y, z, __uint_as_float(i));
    md[at] = 0x7f800000u;
  }
  const uint32_t kx = float_order_key(x), ky = float_order_key(y), kz = float_order_key(z);
  const float bx[6] = {float_from_order_key(wave_min_u32(kx)), float_from_order_key(wave_min_u32(ky)),
                       float_from_order_key(wave_min_u32(kz)), float_from_order_key(wave_max_u32(kx)),
                       float_from_order_key(wave_max_u32(ky)), float_from_order_key(wave_max_u32(kz))};
  if (lane == 0) {
#pragma unroll
    for (int a = 0; a < 6; ++a) boxes[a * box_stride + fps_large_box0(start, b) + j] = bx[a];
  }
}

// Bytes of dynamic LDS for clouds of up to nb buckets.
constexpr int kFpsLargeGroups = 128;
__host__ __device__ inline size_t fps_large_lds(int nb) {
  return static_cast<size_t>(nb) * (sizeof(float4) + sizeof(double) + 2 * sizeof(uint32_t) + sizeof(uint16_t)) +
         kFpsLargeGroups * sizeof(uint16_t) + 16;
}

template <int S>
__global__ __launch_bounds__(kFpsLargeThreads) void fps_large_kernel(
    const float* __restrict__ pos, const float4* __restrict__ Qall, uint32_t* __restrict__ Mall,
    const float* __restrict__ boxes, int64_t box_stride, int nb_max,
    const int64_t* __restrict__ ptr, const int64_t* __restrict__ out_ptr,
    int64_t* __restrict__ out_idx) {
  constexpr int G = kFpsLargeGroups;
  constexpr int W = kFpsLargeWaves;
  extern __shared__ float4 large_lds[];
  float4* rec = large_lds;                                       // farthest point, (bits) rest bound
  double* rkey = reinterpret_cast<double*>(rec + nb_max);        // its key, see fps_key
  uint32_t* rlow = reinterpret_cast<uint32_t*>(rkey + nb_max);   // lowest index at the rest bound, 0 = not known
  uint32_t* queue = rlow + nb_max;                               // bucket << 16 | centroids
  uint16_t* dirty = reinterpret_cast<uint16_t*>(queue + nb_max); // groups whose records changed
  __shared__ double gkey[G];         // best record of each group (buckets g, g + G, ...)
  __shared__ uint32_t gbkt[G];       // its bucket
  __shared__ uint32_t gsec[G], glow[G];  // the group's second record: distance bits, complement of the index
  __shared__ float4 list[kFpsRound];   // as in the bucketed kernel
  __shared__ double2 lkey[kFpsRound];
  __shared__ int n_queue, n_dirty;

  const int b = blockIdx.x;
  const int64_t start = ptr[b];
  const int n = static_cast<int>(ptr[b + 1] - start);
  const int64_t o0 = out_ptr[b];
  const int k = static_cast<int>(out_ptr[b + 1] - o0);
  const int t = threadIdx.x;
  const int w = t / kWave;
  const int lane = lane_id();
  if (k <= 0 || n <= 0) return;
  if (k >= n) {
    for (int i = t; i < n; i += kFpsLargeThreads) out_idx[o0 + i] = start + i;
    return;
  }
  const float4* Q = Qall + start;
  uint32_t* M = Mall + start;
  const int nb = (n + kWave - 1) / kWave;
  const uint32_t ustart = static_cast<uint32_t>(start);
  const int li = lane & (kFpsRound - 1);
  const int row = lane / 16;

  // Slot r of wave w holds the boxes of buckets 64 (w + 16 r) + lane; lane 16 r + c (any c) the
  // box of the whole slot and a bound of its records' distances.
  float blx[S], bly[S], blz[S], bhx[S], bhy[S], bhz[S];
  float slx = __builtin_inff(), sly = slx, slz = slx, shx = -slx, shy = -slx, shz = -slx;
  uint32_t smax = 0u;
#pragma unroll
  for (int r = 0; r < S; ++r) {
    const int bk = kWave * (w + W * r) + lane;
    const bool in = bk < nb;
    const float* bx = boxes + fps_large_box0(start, b) + (in ? bk : 0);
    const float v[6] = {bx[0], bx[box_stride], bx[2 * box_stride], bx[3 * box_stride],
                        bx[4 * box_stride], bx[5 * box_stride]};
    blx[r] = in ? v[0] : __builtin_inff();
    bly[r] = in ? v[1] : __builtin_inff();
    blz[r] = in ? v[2] : __builtin_inff();
    bhx[r] = in ? v[3] : -__builtin_inff();
    bhy[r] = in ? v[4] : -__builtin_inff();
    bhz[r] = in ? v[5] : -__builtin_inff();
    const float l0 = float_from_order_key(wave_min_u32(float_order_key(blx[r])));
    const float l1 = float_from_order_key(wave_min_u32(float_order_key(bly[r])));
    const float l2 = float_from_order_key(wave_min_u32(float_order_key(blz[r])));
    const float h0 = float_from_order_key(wave_max_u32(float_order_key(bhx[r])));
    const float h1 = float_from_order_key(wave_max_u32(float_order_key(bhy[r])));
    const float h2 = float_from_order_key(wave_max_u32(float_order_key(bhz[r])));
    if (row == r && kWave * (w + W * r) < nb) {
      slx = l0; sly = l1; slz = l2; shx = h0; shy = h1; shz = h2;
      smax = 0x7f800000u;
    }
    if (in) {  // all distances +inf: the bucket's lowest index (its first point), nothing known
      const float4 p = Q[bk * kWave];
      rec[bk] = make_float4(p.x, p.y, p.z, __builtin_inff());
      rlow[bk] = 0u;
      rkey[bk] = fps_key(0x7f800000u, __float_as_uint(p.w) - ustart);
    }
  }
  if (t < G) dirty[t] = static_cast<uint16_t>(t);  // every group is formed in the first round
  if (t == 0) {
    list[0] = make_float4(pos[3 * start], pos[3 * start + 1], pos[3 * start + 2], __builtin_inff());
    lkey[0] = make_double2(fps_key(0u, 0u), 0.0);
    n_queue = 0;
    n_dirty = G;
  }
  __syncthreads();

  int done = 0, cap = 1, kend = k;
  for (;;) {
    // check: as in the bucketed kernel, over the listed records
    const float4 c = list[li];
    const double rb = lkey[li].y;
    int A = cap;
    if (cap > 1) {
#pragma unroll
      for (int g = 0; g < kFpsRound; g += 8) {  // four records per step, lane = 16 * record + i
        const int j0 = g + row, j1 = j0 + 4;
        const float4 p0 = list[j0], p1 = list[j1];
        const uint32_t d0 = __float_as_uint(sqdist(c.x, c.y, c.z, p0.x, p0.y, p0.z));
        const uint32_t d1 = __float_as_uint(sqdist(c.x, c.y, c.z, p1.x, p1.y, p1.z));
        const uint64_t b0 = (__ballot(d0 < __float_as_uint(p0.w)) | __ballot(rb > lkey[j0].x)) & fps_ahead(g);
        const uint64_t b1 = (__ballot(d1 < __float_as_uint(p1.w)) | __ballot(rb > lkey[j1].x)) & fps_ahead(g + 4);
        if (b0 | b1) {
          A = min(A, g + static_cast<int>(b0 ? __builtin_ctzll(b0) : 64 + __builtin_ctzll(b1)) / 16);
          break;
        }
      }
    }
    A = min(A, kend - done);
    if (A == 1 && __builtin_amdgcn_readfirstlane(__float_as_int(c.w)) == 0) kend = A = 0;
    if (w == 0 && lane < A) out_idx[o0 + done + lane] = start + fps_key_index(lkey[li].x);
    done += A;
    if (done >= kend) break;

    // test: slots against centroids, lane = 16 * slot + centroid, then the buckets of the slots that
    // a centroid may reach
    {
      float gx, gy, gz;
      {
#pragma clang fp contract(off)
        gx = fmaxf(fmaxf(slx - c.x, c.x - shx), 0.f);
        gy = fmaxf(fmaxf(sly - c.y, c.y - shy), 0.f);
        gz = fmaxf(fmaxf(slz - c.z, c.z - shz), 0.f);
      }
      const float slb = sqdist(gx, gy, gz, 0.f, 0.f, 0.f);
      const uint64_t act = __ballot(__float_as_uint(slb) < smax) & __ballot(li < A);
      if (act) {
        uint32_t touched[S];
        int total = 0;
#pragma unroll
        for (int r = 0; r < S; ++r) {
          touched[r] = 0u;
          uint32_t m = static_cast<uint32_t>(act >> (16 * r)) & 0xffffu;
          if (!m) continue;
          const int bk = kWave * (w + W * r) + lane;
          const uint32_t mx = bk < nb ? static_cast<uint32_t>(__double2hiint(rkey[bk])) : 0u;
          const uint32_t top = wave_max_u32(mx);
          if (row == r) smax = top;
          do {
            const int l = __builtin_ctz(m);
            m &= m - 1;
            const float cx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.x), l));
            const float cy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.y), l));
            const float cz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.z), l));
            float hx, hy, hz;
            {
#pragma clang fp contract(off)
              hx = fmaxf(fmaxf(blx[r] - cx, cx - bhx[r]), 0.f);
              hy = fmaxf(fmaxf(bly[r] - cy, cy - bhy[r]), 0.f);
              hz = fmaxf(fmaxf(blz[r] - cz, cz - bhz[r]), 0.f);
            }
            const float lb = sqdist(hx, hy, hz, 0.f, 0.f, 0.f);
            touched[r] |= __float_as_uint(lb) < mx ? 1u << l : 0u;
          } while (m);
          total += __builtin_popcountll(__ballot(touched[r] != 0u));
        }
        if (total) {
          int base = 0;
          if (lane == 0) base = atomicAdd(&n_queue, total);
          base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
          for (int r = 0; r < S; ++r) {
            const uint64_t on = __ballot(touched[r] != 0u);
            if (touched[r])
              queue[base + __builtin_popcountll(on & lanemask_lt())] =
                  static_cast<uint32_t>(kWave * (w + W * r) + lane) << 16 | touched[r];
            base += __builtin_popcountll(on);
          }
        }
      }
    }
    lds_barrier();

    // update: the queued buckets in turn by all waves, kFpsLargeBatch of a wave's loaded at a time
    const int total = __builtin_amdgcn_readfirstlane(n_queue);
    for (int first = w; first < total; first += W * kFpsLargeBatch) {
      uint32_t item[kFpsLargeBatch], mo[kFpsLargeBatch];
      float4 p[kFpsLargeBatch];
      // this wave's share of the queue, one item per lane (past the end: the last one again)
      const uint32_t mine = queue[min(first + W * lane, total - 1)];
#pragma unroll
      for (int u = 0; u < kFpsLargeBatch; ++u) {
        item[u] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(mine), u));
        const int q = min(static_cast<int>(item[u] >> 16) * kWave + lane, n - 1);
        p[u] = Q[q];
        mo[u] = M[q];
      }
#pragma unroll
      for (int u = 0; u < kFpsLargeBatch; ++u) {
        if (first + W * u >= total) break;
        const float4 pt = p[u];
        const int bk = static_cast<int>(item[u] >> 16);
        const int q = bk * kWave + lane;
        const uint32_t old = q < n ? mo[u] : 0u;  // past the end: never changes, never wins
        const uint32_t holder = static_cast<uint32_t>(__double2loint(rkey[bk]));
        uint32_t m = item[u] & 0xffffu;
        uint32_t mb = old;
        do {
          const int l = __builtin_ctz(m);
          m &= m - 1;
          const float cx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.x), l));
          const float cy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.y), l));
          const float cz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.z), l));
          mb = min(mb, __float_as_uint(sqdist(pt.x, pt.y, pt.z, cx, cy, cz)));
        } while (m);
        if (q < n) M[q] = mb;
        // Values only fall: while the point holding the bucket's max keeps its value, the record
        // (max, lowest index attaining it) stands, and its rest bound still holds.
        const uint32_t nidx = ~(__float_as_uint(pt.w) - ustart);
        if ((__ballot(mb < old) & __ballot(nidx == holder)) == 0ull) continue;
        const uint32_t mx = wave_max_u32(mb);
        const uint64_t hit = __ballot(mb == mx && q < n);
        int sl;
        uint32_t ni, nlow = 0u;
        if ((hit & (hit - 1)) == 0) {  // one lane holds the maximum (distance ties are rare)
          sl = __builtin_ctzll(hit | (1ull << 63));
          ni = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(nidx), sl));
        } else {
          ni = wave_max_u32(mb == mx && q < n ? nidx : 0u);
          sl = __builtin_ctzll(__ballot(mb == mx && q < n && nidx == ni) | (1ull << 63));
          // the others at the maximum that stay there
          const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.x), sl));
          const float y = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.y), sl));
          const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.z), sl));
          const bool stay = mb == mx && q < n && __float_as_uint(sqdist(pt.x, pt.y, pt.z, x, y, z)) >= mx;
          if (__ballot(stay)) nlow = ~wave_max_u32(stay ? nidx : 0u);
        }
        const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.x), sl));
        const float y = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.y), sl));
        const float z = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pt.z), sl));
        const uint32_t rest =
            wave_max_u32(min(mb, __float_as_uint(sqdist(pt.x, pt.y, pt.z, x, y, z))));
        if (lane == 0) {
          rec[bk] = make_float4(x, y, z, __uint_as_float(rest));
          rlow[bk] = nlow;
          rkey[bk] = fps_key(mx, ~ni);
          dirty[atomicAdd(&n_dirty, 1)] = static_cast<uint16_t>(bk % G);
        }
      }
    }
    __syncthreads();  // min distances too: the next round's waves take other buckets

    // groups: best and second record of every group with a changed record, one 16-lane row each
    {
      const int changed = __builtin_amdgcn_readfirstlane(n_dirty);
      if (t == 0) n_queue = 0;
      for (int at = 4 * w; at < changed; at += 4 * W) {
        const int g = dirty[min(at + row, changed - 1)];
        const int m0 = g + G * li, m1 = m0 + 16 * G;
        double best = m0 < nb ? rkey[m0] : 0.0, other = 0.0;
        int bk = m0;
        if (S > 2) {  // more than 16 buckets per group
          other = m1 < nb ? rkey[m1] : 0.0;
          if (other > best) {
            const double x = best;
            best = other;
            other = x;
            bk = m1;
          }
        }
        const uint32_t hi = static_cast<uint32_t>(__double2hiint(best));
        const uint32_t top = row_max_u32(hi);
        const uint32_t lo = hi == top ? static_cast<uint32_t>(__double2loint(best)) : 0u;
        const uint32_t low = row_max_u32(lo);
        const bool winner = hi == top && lo == low;  // one lane, or lanes without a record
        const double left = winner ? other : best;
        const uint32_t lhi = static_cast<uint32_t>(__double2hiint(left));
        const uint32_t sec = row_max_u32(lhi);
        const uint32_t slo = row_max_u32(lhi == sec ? static_cast<uint32_t>(__double2loint(left)) : 0u);
        if (winner) {
          gkey[g] = best;
          gbkt[g] = bk;
          gsec[g] = sec;
          glow[g] = slo;
        }
      }
    }
    lds_barrier();

    // rank: no record that is not a group's best exceeds t0; the bests above it, each placed among
    // all of them, are the list
    {
      const double ka = gkey[lane], kb = gkey[kWave + lane];
      const uint32_t t0 = wave_max_u32(max(gsec[lane], gsec[kWave + lane]));
      if (t == 0) n_dirty = 0;
      uint64_t ca = __ballot(static_cast<uint32_t>(__double2hiint(ka)) > t0);
      uint64_t cb = __ballot(static_cast<uint32_t>(__double2hiint(kb)) > t0);
      if (!(ca | cb)) {  // equal distances across groups: by the indices too
        const uint32_t lo = wave_max_u32(max(gsec[lane] == t0 ? glow[lane] : 0u,
                                             gsec[kWave + lane] == t0 ? glow[kWave + lane] : 0u));
        const double t1 = __hiloint2double(static_cast<int>(t0), static_cast<int>(lo));
        ca = __ballot(ka > t1);
        cb = __ballot(kb > t1);
      }
      const int na = __builtin_popcountll(ca), nc = na + __builtin_popcountll(cb);
      const uint64_t lt = lanemask_lt();
      const int pa = __builtin_popcountll(ca & lt), pb = na + __builtin_popcountll(cb & lt);
      for (int at = w; at < nc; at += W) {
        const uint64_t mine = at < na ? ca & __ballot(pa == at) : cb & __ballot(pb == at);
        const int l = __builtin_ctzll(mine | (1ull << 63));
        const uint64_t kj = readlane_u64(__double_as_longlong(at < na ? ka : kb), l);
        const double dj = __longlong_as_double(static_cast<long long>(kj));
        const int rank = __builtin_popcountll(__ballot(ka > dj)) + __builtin_popcountll(__ballot(kb > dj));
        if (rank < kFpsRound && lane == 0) {
          const uint32_t bk = gbkt[l + (at < na ? 0 : kWave)];
          const float4 r = rec[bk];
          list[rank] = make_float4(r.x, r.y, r.z, __uint_as_float(static_cast<uint32_t>(kj >> 32)));
          lkey[rank] = make_double2(dj, fps_key(__float_as_uint(r.w), rlow[bk]));
        }
      }
      cap = min(max(nc, 1), kFpsRound);
    }
    lds_barrier();
  }
  for (int i = done + t; i < k; i += kFpsLargeThreads) out_idx[o0 + i] = start;  // distances all 0
}

struct FpsLargeWs {
  float4* q;
  uint32_t* md;
  float *bbox, *boxes;
  uint32_t *keys, *skeys, *order;
  RadixBuffers rx;
};

// Width of the sort keys (cloud + 1, Hilbert position): the cloud field holds 0 .. B + 1 and each
// axis of the Hilbert grid gets the same share of the rest, at most 10 bits.
int fps_large_key_bits(int64_t B, int* axis_bits) {
  int cbits = 0;
  while ((static_cast<uint64_t>(B + 1) >> cbits) != 0) ++cbits;
  int mbits = (32 - cbits) / 3;
  if (mbits > 10) mbits = 10;
  if (axis_bits) *axis_bits = mbits;
  return cbits + 3 * mbits;
}

int64_t fps_large_box_stride(int64_t B, int64_t N) { return N / kWave + B + 1; }

FpsLargeWs carve_fps_large(void* base, int64_t B, int64_t N, size_t* bytes) {
  Carver c(base);
  FpsLargeWs w;
  w.q = c.take<float4>(N);
  w.md = c.take<uint32_t>(N);
  w.bbox = c.take<float>(6 * (B > 0 ? B : 1));
  w.boxes = c.take<float>(6 * fps_large_box_stride(B, N));
  w.keys = c.take<uint32_t>(N);
  w.skeys = c.take<uint32_t>(N);
  w.order = c.take<uint32_t>(N);
  w.rx = carve_radix(c, N, fps_large_key_bits(B, nullptr));
  *bytes = c.used;
  return w;
}

bool fps_use_large(int64_t B, int64_t max_cloud) {
  return max_cloud > kFpsLdsPoints && max_cloud <= kFpsLargeMaxPoints && B <= kFpsLargeMaxClouds;
}

template <int S>
int launch_large_rounds(const float* pos, const FpsLargeWs& w, int64_t stride, int nb,
                        const int64_t* ptr, const int64_t* out_ptr, int64_t B, int64_t* out,
                        hipStream_t st) {
  GEO_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&fps_large_kernel<S>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(fps_large_lds(S * kFpsLargeThreads))));
  hipLaunchKernelGGL((fps_large_kernel<S>), dim3(B), dim3(kFpsLargeThreads), fps_large_lds(nb), st,
                     pos, w.q, w.md, w.boxes, stride, nb, ptr, out_ptr, out);
  GEO_LAUNCH_CHECK("fps_large_kernel");
  return GEO_OK;
}

int launch_large(const float* pos, int64_t N, const int64_t* ptr, const int64_t* out_ptr,
                 int64_t B, int64_t max_cloud, int64_t* out, void* workspace, hipStream_t st) {
  size_t bytes = 0;
  const FpsLargeWs w = carve_fps_large(workspace, B, N, &bytes);
  hipLaunchKernelGGL(fps_large_bbox_kernel, dim3(B), dim3(kFpsLargeThreads), 0, st, pos, ptr, w.bbox);
  GEO_LAUNCH_CHECK("fps_large_bbox_kernel");
  int mbits = 0;
  fps_large_key_bits(B, &mbits);
  const unsigned grid = static_cast<unsigned>(ceil_div(N, 256));
  hipLaunchKernelGGL(fps_large_keys_kernel, dim3(grid), dim3(256), 0, st, pos, ptr, B, N, w.bbox,
                     mbits, w.keys);
  GEO_LAUNCH_CHECK("fps_large_keys_kernel");
  int rc = radix_sort<kRxKeysIota>(w.keys, nullptr, N, 0, w.skeys, w.order, w.rx, st);
  if (rc) return rc;
  const int64_t nb = ceil_div(max_cloud, kWave);
  const int64_t stride = fps_large_box_stride(B, N);
  hipLaunchKernelGGL(fps_large_gather_kernel, dim3(static_cast<unsigned>(ceil_div(nb, 4)), B), dim3(256),
                     0, st, pos, w.order, ptr, stride, w.q, w.md, w.boxes);
  GEO_LAUNCH_CHECK("fps_large_gather_kernel");
  if (nb <= kFpsLargeThreads)
    return launch_large_rounds<1>(pos, w, stride, static_cast<int>(nb), ptr, out_ptr, B, out, st);
  if (nb <= 2 * kFpsLargeThreads)
    return launch_large_rounds<2>(pos, w, stride, static_cast<int>(nb), ptr, out_ptr, B, out, st);
  return launch_large_rounds<3>(pos, w, stride, static_cast<int>(nb), ptr, out_ptr, B, out, st);
}

}  // namespace
}  // namespace geo

using namespace geo;

static int fps_prepare(const int64_t* ptr, const int64_t* k_per_batch, int64_t B, int64_t N_total,
                       int64_t* out_ptr, int64_t* info, int64_t* most, void* stream) {
  GEO_REQUIRE(B >= 0 && N_total >= 0, "fps_prepare: negative size");
  GEO_REQUIRE(ptr && out_ptr && info && (B == 0 || k_per_batch), "fps_prepare: null pointer");
  hipLaunchKernelGGL(fps_prepare_kernel, dim3(1), dim3(kScanThreads), 0, as_stream(stream), ptr,
                     k_per_batch, int64_t{0}, B, N_total, out_ptr, info,
                     static_cast<int64_t*>(nullptr), most);
  GEO_LAUNCH_CHECK("fps_prepare_kernel");
  return GEO_OK;
}

extern "C" int geo_fps_prepare(const int64_t* ptr, const int64_t* k_per_batch, int64_t B,
                               int64_t N_total, int64_t* out_ptr, int64_t* info, void* stream) {
  return fps_prepare(ptr, k_per_batch, B, N_total, out_ptr, info, nullptr, stream);
}

extern "C" int geo_fps_prepare_most(const int64_t* ptr, const int64_t* k_per_batch, int64_t B,
                                    int64_t N_total, int64_t* out_ptr, int64_t* info, void* stream) {
  return fps_prepare(ptr, k_per_batch, B, N_total, out_ptr, info, info ? info + 3 : nullptr, stream);
}

extern "C" int geo_fps_prepare_uniform(const int64_t* ptr, int64_t k, int64_t B, int64_t N_total,
                                       int64_t* out_ptr, int64_t* info, int64_t* info_host,
                                       void* stream) {
  GEO_REQUIRE(B >= 0 && N_total >= 0, "fps_prepare: negative size");
  GEO_REQUIRE(ptr && out_ptr && info, "fps_prepare: null pointer");
  int64_t* host_dev = nullptr;
  if (info_host) {
    GEO_HIP_CHECK(hipHostGetDevicePointer(reinterpret_cast<void**>(&host_dev), info_host, 0));
    GEO_REQUIRE(host_dev != nullptr, "fps_prepare: info_host is not mapped pinned memory");
  }
  hipLaunchKernelGGL(fps_prepare_kernel, dim3(1), dim3(kScanThreads), 0, as_stream(stream), ptr,
                     static_cast<const int64_t*>(nullptr), k, B, N_total, out_ptr, info, host_dev,
                     static_cast<int64_t*>(nullptr));
  GEO_LAUNCH_CHECK("fps_prepare_kernel");
  return GEO_OK;
}

extern "C" int geo_fps_guarded(const float* pos, int64_t N_total, const int64_t* ptr,
                               const int64_t* out_ptr, int64_t B, int64_t max_cloud_guess,
                               int64_t* out_idx, const int64_t* info, int64_t* capacity,
                               void* stream) {
  GEO_REQUIRE(capacity != nullptr, "fps_guarded: null capacity");
  *capacity = 0;
  GEO_REQUIRE(B >= 0 && N_total >= 0 && max_cloud_guess >= 0, "fps_guarded: negative size");
  GEO_REQUIRE(N_total < 0x7fffffffLL, "fps: N_total exceeds int32 indexing");
  if (B == 0 || max_cloud_guess == 0 || max_cloud_guess > kFpsLdsPoints) return GEO_OK;
  GEO_REQUIRE(pos && ptr && out_ptr && out_idx && info, "fps_guarded: null pointer");
  hipStream_t st = as_stream(stream);
  const int64_t p2 = ceil_div(max_cloud_guess, kFpsBucketThreads);
  const int pts = p2 <= 1 ? 1 : (p2 <= 2 ? 2 : (p2 <= 4 ? 4 : 8));
  const int64_t cap = static_cast<int64_t>(pts) * kFpsBucketThreads;
  int rc;
  switch (pts) {
    case 1: rc = launch_bucket<1, kFpsBucketThreads>(pos, ptr, out_ptr, B, cap, out_idx, st, info); break;
    case 2: rc = launch_bucket<2, kFpsBucketThreads>(pos, ptr, out_ptr, B, cap, out_idx, st, info); break;
    case 4: rc = launch_bucket<4, kFpsBucketThreads>(pos, ptr, out_ptr, B, cap, out_idx, st, info); break;
    default: rc = launch_bucket<8, kFpsBucketThreads>(pos, ptr, out_ptr, B, cap, out_idx, st, info); break;
  }
  if (rc == GEO_OK) *capacity = cap;
  return rc;
}

extern "C" size_t geo_fps_workspace_bytes(int64_t B, int64_t N_total, int64_t max_cloud) {
  if (B < 0 || N_total < 0 || max_cloud < 0) return 0;
  if (fps_use_large(B, max_cloud)) {
    size_t bytes = 0;
    carve_fps_large(nullptr, B, N_total, &bytes);
    return bytes;
  }
  if (max_cloud > kFpsRegisterPoints) return static_cast<size_t>(N_total > 0 ? N_total : 1) * 4;
  return 0;
}

extern "C" int geo_fps(const float* pos, int64_t N_total, const int64_t* ptr,
                       const int64_t* out_ptr, int64_t B, int64_t max_cloud, int64_t* out_idx,
                       void* workspace, size_t workspace_bytes, void* stream) {
  return geo_fps_most(pos, N_total, ptr, out_ptr, B, max_cloud, max_cloud, out_idx, workspace,
                      workspace_bytes, stream);
}

extern "C" int geo_fps_total(const float* pos, int64_t N_total, const int64_t* ptr,
                             const int64_t* out_ptr, int64_t B, int64_t max_cloud, int64_t total,
                             int64_t* out_idx, void* workspace, size_t workspace_bytes,
                             void* stream) {
  return geo_fps_most(pos, N_total, ptr, out_ptr, B, max_cloud, B > 0 ? ceil_div(total, B) : 0, out_idx,
                      workspace, workspace_bytes, stream);
}

extern "C" int geo_fps_most(const float* pos, int64_t N_total, const int64_t* ptr,
                            const int64_t* out_ptr, int64_t B, int64_t max_cloud, int64_t most,
                            int64_t* out_idx, void* workspace, size_t workspace_bytes,
                            void* stream) {
  GEO_REQUIRE(B >= 0 && N_total >= 0 && max_cloud >= 0, "fps: negative size");
  GEO_REQUIRE(max_cloud <= N_total, "fps: max_cloud %lld > N_total %lld", (long long)max_cloud,
              (long long)N_total);
  GEO_REQUIRE(N_total < 0x7fffffffLL, "fps: N_total exceeds int32 indexing");
  if (B == 0 || max_cloud == 0) return GEO_OK;
  GEO_REQUIRE(pos && ptr && out_ptr && out_idx, "fps: null pointer");
  hipStream_t st = as_stream(stream);
  const int64_t need = static_cast<int64_t>(geo_fps_workspace_bytes(B, N_total, max_cloud));
  const bool room = workspace != nullptr && workspace_bytes >= static_cast<size_t>(need);
  if (need > 0 && !room && max_cloud > kFpsRegisterPoints)
    return set_error(GEO_ERR_WORKSPACE, "fps: workspace %zu bytes, need %lld", workspace_bytes,
                     (long long)need);
  if (max_cloud <= kFpsLdsPoints) {
    // 1024 threads: four waves per SIMD hide much of the per-iteration dependency chain.
    const int64_t p2 = ceil_div(max_cloud, kFpsBucketThreads);
    if (p2 <= 1) return launch_bucket<1, kFpsBucketThreads>(pos, ptr, out_ptr, B, max_cloud, out_idx, st);
    if (p2 <= 2) return launch_bucket<2, kFpsBucketThreads>(pos, ptr, out_ptr, B, max_cloud, out_idx, st);
    if (p2 <= 4) return launch_bucket<4, kFpsBucketThreads>(pos, ptr, out_ptr, B, max_cloud, out_idx, st);
    return launch_bucket<8, kFpsBucketThreads>(pos, ptr, out_ptr, B, max_cloud, out_idx, st);
  }
  // Up to 16,384 points and few samples in every cloud (the register kernel's steps take as long
  // for a small cloud, and the one with the most samples ends last): no set-up.  The
  // large kernel's sort and first rounds cost about 90 us more, its later rounds a tenth as much
  // per sample (12,000 points: 64 samples 197 against 225 us, 375 samples 1069 against 399 us,
  // 6000 samples 16.9 against 2.2 ms); they cross at 73 to 87 samples between 8,200 and 16,384.
  // Callers that bring no workspace for such clouds get it as well.
  if (max_cloud <= kFpsRegisterPoints &&
      (most <= kFpsRegisterSamples || !room || !fps_use_large(B, max_cloud))) {
    hipLaunchKernelGGL((fps_register_kernel<kFpsRegisterPoints / kFpsThreads>), dim3(B),
                       dim3(kFpsThreads), 0, st, pos, ptr, out_ptr, out_idx);
    GEO_LAUNCH_CHECK("fps_register_kernel");
    return GEO_OK;
  }
  if (fps_use_large(B, max_cloud))
    return launch_large(pos, N_total, ptr, out_ptr, B, max_cloud, out_idx, workspace, st);
  hipLaunchKernelGGL(fps_stream_kernel, dim3(B), dim3(kFpsStreamThreads), 0, st, pos, ptr,
                     out_ptr, out_idx, static_cast<float*>(workspace));
  GEO_LAUNCH_CHECK("fps_stream_kernel");
  return GEO_OK;
}
