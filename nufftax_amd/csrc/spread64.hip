// 3D FP64 spreading by output regions on the matrix cores.
//
// The fine grid is cut into regions of 16 x 16 x 8 cells (x, y, z).  A block owns one region and
// sums the contributions of every point whose support meets it,
//   fw[z][y][x] += sum_j (c_j wz_j(z) wy_j(y)) wx_j(x)         (nufftax/core/spread.py:543-593)
// so 4 points are, per z slice and part (re, im), one v_mfma_f64_16x16x4f64 with
// A[y][j] = c_j wy_j(y) wz_j(z) and B[j][x] = wx_j(x); a cell outside a point's support has weight
// zero.  The sums stay in registers until the region is done and are stored once: no atomics per
// point and cell, no tile in LDS and no cleared grid.
//
// Why regions of the output: the atomic kernels (k_spread_tiled: 2 ns^3 ds_add_f64 per point,
// 2.4 lane-operations per clock and CU; k_spread_global_wave: global FP64 atomics, 144 G/s) are
// bound by their atomics.  A point meets (16 + ns - 1)^2 / 16^2 regions in (x, y) on average (3.3 at
// ns = 14, 2.4 at ns = 10) and there costs 2 MFMAs of 64 clocks per 4 points and slice in
// its support, which is the matrix cores' FP64 rate with that factor of products with zero.
// (Sub-bin windows, as in the FP32 kernels, would avoid the factor, but a 16-cell window leaves
// 2 support starts per side at ns = 14: a few points for each 4096 cells to be added up.)
// 8 slices take 128 accumulator registers per lane, 168 in all, so three waves share a SIMD.  Counters of 500k clustered
// points at ns = 14 on 128^3 cells (784 us): matrix cores 44% busy, vector units 28%, 1.7 GB fetched (weights, once per
// region that a point meets).
//
// Passes of one spread (M points, sorted):
//   k_tab64      per point, in sorted order: its 3 ns kernel weights, its support starts and
//                its strengths; a (point, strength) that is not finite is left out (all zero) and listed
//   k_tasks64    per region: number of candidate points (the bins that its halo meets), cut into
//                tasks of at most 2048 candidates; regions of several tasks are listed
//   k_zero64     clears the listed regions (their tasks add with atomics)
//   k_spread64   one task at a time per block, taken from a counter
//   k_fix64      the listed non-finite (point, strength) pairs, one wave each, with atomics: zero
//                weights of a matrix product would spread their NaN over the whole region
#include <algorithm>

#include "si_kernels.hpp"

namespace nufftx {

namespace {

constexpr int kRX = 16, kRY = 16, kRZ = 8;   // region cells
constexpr int kCells = kRX * kRY * kRZ;
constexpr int kThreads64 = 256;              // 4 waves share a region's candidates
constexpr int kWaves64 = kThreads64 / 64;
constexpr int kCandMin = 256, kCandMax = 2048;  // candidates per task (Sizes64)
constexpr int kRunsMax = 256;                // runs of consecutive bins around a region
constexpr int kListMax = 128;                // points waiting for the matrix products, per wave
// bytes of weights and of all buffers that a spread keeps at most; more points or transforms take the atomic kernels
// (24 bytes per point and transform: the bound also keeps the counter of pairs in 31 bits)
constexpr int64_t kTabMaxBytes = (int64_t)2 << 30, kMaxBytes64 = (int64_t)4 << 30;

typedef double d4 __attribute__((ext_vector_type(4)));

struct Reg64Args {
  int64_t M, n_trans, grid_cells;
  int nf[3], bs[3], nb[3], nr[3];  // nr: regions per dimension
  int regions, max_tasks, zero_out, cand;  // cand: candidates per task
  const int32_t* bin_start;
  const int32_t* perm;
  const void* coord[3];
  double beta, c;
  double* tab;   // [M][3 NS] weights x, y, z
  int4* start;   // [M] support starts
  double2* cs;   // [n_trans][M] strengths
  int4* task;    // {region, first candidate, last + 1, tasks of the region}
  int32_t* heavy;  // regions of several tasks
  int2* bad;     // {sorted slot, transform}
  int32_t* cnt;  // {tasks, next task, heavy regions, bad pairs}
};

__device__ __forceinline__ int mod_nf(int v, int nf) {
  v %= nf;
  return v < 0 ? v + nf : v;
}

// Bins of dimension d that hold points whose support may meet cells [x0, x0 + len): their cells lie
// in [x0 - NS/2, x0 + len - 1 + NS/2].  At most two intervals [lo, hi] (the range may wrap).
struct BinRange {
  int lo0, hi0, lo1, hi1, n;
};
template <int NS>
__device__ __forceinline__ BinRange bin_range(int x0, int len, int nf, int bs, int nb) {
  BinRange r;
  r.n = 1;
  r.lo0 = r.lo1 = 0;
  r.hi0 = nb - 1;
  r.hi1 = -1;
  if (len + NS >= nf) return r;
  const int lo = mod_nf(x0 - NS / 2, nf) / bs, hi = mod_nf(x0 + len - 1 + NS / 2, nf) / bs;
  if (mod_nf(x0 - NS / 2, nf) <= mod_nf(x0 + len - 1 + NS / 2, nf)) {
    r.lo0 = lo;
    r.hi0 = hi;
  } else if (lo > hi) {  // wraps; lo <= hi: the two ends share a bin, every bin is in range
    r.n = 2;
    r.hi0 = hi;
    r.lo1 = lo;
    r.hi1 = nb - 1;
  }
  return r;
}
__device__ __forceinline__ int range_count(const BinRange& r) {
  return r.hi0 - r.lo0 + 1 + (r.hi1 - r.lo1 + 1 > 0 ? r.hi1 - r.lo1 + 1 : 0);
}
__device__ __forceinline__ int range_bin(const BinRange& r, int q) {
  const int n0 = r.hi0 - r.lo0 + 1;
  return q < n0 ? r.lo0 + q : r.lo1 + q - n0;
}

struct RegionRuns {
  BinRange x, y, z;
  int ny, n;  // runs: (x interval, y bin, z bin)
};
template <int NS>
__device__ __forceinline__ RegionRuns region_runs(const Reg64Args& a, const int (&org)[3]) {
  RegionRuns r;
  r.x = bin_range<NS>(org[0], kRX, a.nf[0], a.bs[0], a.nb[0]);
  r.y = bin_range<NS>(org[1], kRY, a.nf[1], a.bs[1], a.nb[1]);
  r.z = bin_range<NS>(org[2], kRZ, a.nf[2], a.bs[2], a.nb[2]);
  r.ny = range_count(r.y);
  r.n = min(r.x.n * r.ny * range_count(r.z), kRunsMax);  // (the host admits only grids that fit)
  return r;
}
// sorted slots [lo, hi) of run q
__device__ __forceinline__ int2 run_slots(const Reg64Args& a, const RegionRuns& r, int q) {
  const int ix = q % r.x.n;
  q /= r.x.n;
  const int by = range_bin(r.y, q % r.ny), bz = range_bin(r.z, q / r.ny);
  const int row = (bz * a.nb[1] + by) * a.nb[0];
  return make_int2(a.bin_start[row + (ix ? r.x.lo1 : r.x.lo0)], a.bin_start[row + (ix ? r.x.hi1 : r.x.hi0) + 1]);
}

__device__ __forceinline__ void region_origin(const Reg64Args& a, int region, int (&org)[3]) {
  org[0] = region % a.nr[0] * kRX;
  region /= a.nr[0];
  org[1] = region % a.nr[1] * kRY;
  org[2] = region / a.nr[1] * kRZ;
}

// A block takes kTabPts sorted points: thread (d, point) folds one coordinate and evaluates its NS weights,
// which leave through LDS as one run of adjacent doubles (500k points, ns = 14: 68 us; one thread per weight,
// which gathered and folded each coordinate NS times, took 126).
constexpr int kTabPts = 64;
template <int NS>
__global__ void __launch_bounds__(3 * kTabPts) k_tab64(Reg64Args a, const cplx<double>* __restrict__ c) {
  constexpr int L = 3 * NS;
  __shared__ double sw[kTabPts][L + 1];
  __shared__ int sfin[kTabPts];
  const int64_t j0 = (int64_t)blockIdx.x * kTabPts;
  const int pt = (int)threadIdx.x % kTabPts, d = (int)threadIdx.x / kTabPts;
  const int64_t j = j0 + pt;
  const int n = (int)min((int64_t)kTabPts, a.M - j0);
  if (d == 0) sfin[pt] = 1;
  __syncthreads();
  const int p = pt < n ? a.perm[j] : -1;
  const bool valid = (unsigned)p < (unsigned)a.M;
  if (valid) {
    const double x = static_cast<const double*>(d == 0 ? a.coord[0] : d == 1 ? a.coord[1] : a.coord[2])[p];
    const Folded f = fold_coord(x, d == 0 ? a.nf[0] : d == 1 ? a.nf[1] : a.nf[2]);
    const int i0 = support_start(f, NS / 2);
    const double t = (double)i0 - f.xs;
    const bool fin = isfinite(x);
    if (!fin) sfin[pt] = 0;
    reinterpret_cast<int*>(a.start + j)[d] = i0;
#pragma unroll
    for (int k = 0; k < NS; ++k) sw[pt][d * NS + k] = fin ? es_phi(t + (double)k, a.beta, a.c) : 0.0;
  }
  __syncthreads();
  if (valid)
    for (int64_t t = d; t < a.n_trans; t += 3) {
      const cplx<double> v = c[t * a.M + p];
      const bool ok = sfin[pt] && isfinite(v.re) && isfinite(v.im);
      a.cs[t * a.M + j] = ok ? make_double2(v.re, v.im) : make_double2(0.0, 0.0);
      if (!ok) a.bad[atomicAdd(&a.cnt[3], 1)] = make_int2((int)j, (int)t);  // once per pair: capacity n_trans M
    }
  for (int e = (int)threadIdx.x; e < n * L; e += 3 * kTabPts) a.tab[j0 * L + e] = sw[e / L][e % L];
}

// A block counts kTaskRegions regions, one wave at a time each, and takes their tasks' places with one atomic
// (one per region: 116 us for the 9826 regions of a 270^3 grid, all on one counter).
constexpr int kTaskRegions = 32;
template <int NS>
__global__ void __launch_bounds__(256) k_tasks64(Reg64Args a) {
  __shared__ int cand[kTaskRegions], base[kTaskRegions];
  const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
  const int r0 = (int)blockIdx.x * kTaskRegions;
#pragma unroll 2
  for (int u = wave; u < kTaskRegions; u += 4) {
    int n = 0;
    if (r0 + u < a.regions) {
      int org[3];
      region_origin(a, r0 + u, org);
      const RegionRuns r = region_runs<NS>(a, org);
      for (int q = lane; q < r.n; q += 64) {
        const int2 s = run_slots(a, r, q);
        n += s.y - s.x;
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (lane == 0) cand[u] = n;
  }
  __syncthreads();
  auto parts = [&](int u) { return r0 + u < a.regions ? max(1, (cand[u] + a.cand - 1) / a.cand) : 0; };
  if (wave == 0) {
    const int v = lane < kTaskRegions ? parts(lane) : 0;
    int incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(incl, off, 64);
      if (lane >= off) incl += t;
    }
    int first = 0;
    if (lane == 63) first = atomicAdd(&a.cnt[0], incl);
    first = __shfl(first, 63, 64);
    if (lane < kTaskRegions) base[lane] = first + incl - v;
    if (v > 1) a.heavy[atomicAdd(&a.cnt[2], 1)] = r0 + lane;
  }
  __syncthreads();
  for (int u = wave; u < kTaskRegions; u += 4) {
    const int np = parts(u), n = cand[u];
    for (int q = lane; q < np; q += 64)
      if (base[u] + q < a.max_tasks)
        a.task[base[u] + q] =
            make_int4(r0 + u, (int)((int64_t)n * q / np), (int)((int64_t)n * (q + 1) / np), np);
  }
}

// Clears the regions whose tasks add with atomics.
__global__ void __launch_bounds__(256) k_zero64(Reg64Args a, double2* __restrict__ fw) {
  const int n = a.cnt[2];
  for (int h = blockIdx.x; h < n; h += gridDim.x) {
    int org[3];
    region_origin(a, a.heavy[h], org);
    for (int e = threadIdx.x; e < kCells; e += blockDim.x) {
      const int x = org[0] + e % kRX, y = org[1] + e / kRX % kRY, z = org[2] + e / (kRX * kRY);
      if (x >= a.nf[0] || y >= a.nf[1] || z >= a.nf[2]) continue;
      for (int64_t t = 0; t < a.n_trans; ++t)
        fw[t * a.grid_cells + ((int64_t)z * a.nf[1] + y) * a.nf[0] + x] = make_double2(0.0, 0.0);
    }
  }
}

// position of region cell 0 in the support that starts at s, as an offset in [-15, NS - 1]; false if the
// support does not meet the region's len cells
template <int NS>
__device__ __forceinline__ bool region_offset(int org, int len, int s, int nf, int& o) {
  const int ox = mod_nf(org - s, nf);
  o = ox < NS ? ox : ox - nf;
  return ox < NS || ox > nf - len;
}

// weight index of region cell i for offset o: in [0, NS) inside the support
__device__ __forceinline__ int weight_index(int o, int i, int nf) {
  int k = o + i;
  k = k < 0 ? k + nf : k;
  return k >= nf ? k - nf : k;
}

// lane Z of each row of 16 lanes, to the whole row
template <int Z>
__device__ __forceinline__ double row_bcast(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xFFFFFFFFll), 0x150 + Z, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + Z, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// slices Z .. kRZ - 1 of one group of 4 points: both parts' products into the accumulators
template <int Z>
__device__ __forceinline__ void slices(unsigned mask, double are, double aim, double b, double wz, d4 (&re)[kRZ],
                                       d4 (&im)[kRZ]) {
  if constexpr (Z < kRZ) {
    if (mask >> Z & 1u) {  // uniform: some point's support holds the slice
      const double w = row_bcast<Z>(wz);
      re[Z] = __builtin_amdgcn_mfma_f64_16x16x4f64(are * w, b, re[Z], 0, 0, 0);
      im[Z] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim * w, b, im[Z], 0, 0, 0);
    }
    slices<Z + 1>(mask, are, aim, b, wz, re, im);
  }
}

// Orders a wave's LDS writes before its later reads of other lanes' data, and the reverse.
__device__ __forceinline__ void wave_sync64() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// MFMA operand layout (v_mfma_f64_16x16x4f64): A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k,
// D[i][j] in lane j + 16 (i % 4), element i / 4.
template <int NS>
__global__ void __launch_bounds__(kThreads64, 3) k_spread64(Reg64Args a, double2* __restrict__ fw) {
  __shared__ int run_first[kRunsMax], run_base[kRunsMax];  // first slot; candidates before the run
  __shared__ int2 list[kWaves64][kListMax];                // {slot, offsets in the region}
  __shared__ double2 part[2][kWaves64][kRX * kRY];
  __shared__ int wsum[kWaves64], s_task;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, k = lane >> 4;
  const int ntasks = min(a.cnt[0], a.max_tasks);
  const int64_t total = (int64_t)ntasks * a.n_trans;
  for (;;) {
    __syncthreads();  // s_task, the runs and `part` are free again
    if (tid == 0) s_task = atomicAdd(&a.cnt[1], 1);
    __syncthreads();
    const int tk = s_task;
    if (tk >= total) return;  // the counter only grows: every block gets here
    const int tr = tk / ntasks;
    const int4 task = a.task[tk - tr * ntasks];
    int org[3];
    region_origin(a, task.x, org);
    const RegionRuns rr = region_runs<NS>(a, org);
    // candidates before each run (kRunsMax == blockDim.x: one run per thread)
    {
      static_assert(kRunsMax == kThreads64, "one run per thread");
      int2 s = make_int2(0, 0);
      if (tid < rr.n) s = run_slots(a, rr, tid);
      const int v = s.y - s.x;
      int incl = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(incl, off, 64);
        if (lane >= off) incl += t;
      }
      if (lane == 63) wsum[wave] = incl;
      __syncthreads();
      int before = 0;
      for (int w = 0; w < wave; ++w) before += wsum[w];
      run_first[tid] = s.x;
      run_base[tid] = before + incl - v;
      __syncthreads();
    }
    d4 re[kRZ], im[kRZ];
#pragma unroll
    for (int z = 0; z < kRZ; ++z) re[z] = im[z] = d4{0.0, 0.0, 0.0, 0.0};
    const double2* cs = a.cs + (int64_t)tr * a.M;
    int2* const my = list[wave];
    int nlist = 0;

    // one group of 4 listed points from entry g on: this lane's weights and strength
    struct Operands {
      double wx, wy, wz, cre, cim;
      unsigned mask;
    };
    auto load = [&](int g, int n) {
      Operands o;
      const int2 en = my[min(g + k, n - 1)];
      const bool on = g + k < n;
      const int ox = (int)(signed char)(en.y & 0xFF), oy = (int)(signed char)(en.y >> 8 & 0xFF),
                oz = (int)(signed char)(en.y >> 16 & 0xFF);
      const int kx = weight_index(ox, i, a.nf[0]), ky = weight_index(oy, i, a.nf[1]), kz = weight_index(oz, i, a.nf[2]);
      const double* w = a.tab + (int64_t)en.x * (3 * NS);
      const bool vx = kx < NS, vy = ky < NS, vz = on && i < kRZ && kz < NS;
      const double2 cv = cs[en.x];
      o.wx = w[vx ? kx : 0];
      o.wy = w[NS + (vy ? ky : 0)];
      o.wz = w[2 * NS + (vz ? kz : 0)];
      o.wx = vx ? o.wx : 0.0;
      o.wy = vy ? o.wy : 0.0;
      o.wz = vz ? o.wz : 0.0;
      o.cre = on ? cv.x : 0.0;
      o.cim = on ? cv.y : 0.0;
      const uint64_t b = __ballot(vz);
      o.mask = (unsigned)((b | b >> 16 | b >> 32 | b >> 48) & 0xFFu);
      return o;
    };
    auto process = [&](int n) {  // the next group's operands load while a group multiplies
      Operands o = load(0, n);
      for (int g = 0; g < n; g += 4) {
        const Operands cur = o;
        if (g + 4 < n) o = load(g + 4, n);
        slices<0>(cur.mask, cur.cre * cur.wy, cur.cim * cur.wy, cur.wx, cur.wz, re, im);
      }
    };

    // candidates in steps of 64 per wave; those that meet the region go into the wave's list.  The next step's
    // slot and support start load while the listed points multiply.
    auto candidate = [&](int cand, int& slot) {
      slot = -1;
      if (cand >= task.z) return make_int4(0, 0, 0, 0);
      int lo = 0, hi = rr.n;  // the last run that starts at or before the candidate
      while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (run_base[mid] <= cand)
          lo = mid;
        else
          hi = mid;
      }
      slot = run_first[lo] + cand - run_base[lo];
      return a.start[slot];
    };
    int slot;
    int4 st = candidate(task.y + 64 * wave + lane, slot);
    for (int c0 = task.y + 64 * wave; c0 < task.z; c0 += kThreads64) {
      int ox, oy, oz;
      bool hit = slot >= 0;
      hit = region_offset<NS>(org[0], kRX, st.x, a.nf[0], ox) && hit;
      hit = region_offset<NS>(org[1], kRY, st.y, a.nf[1], oy) && hit;
      hit = region_offset<NS>(org[2], kRZ, st.z, a.nf[2], oz) && hit;
      const uint64_t m = __ballot(hit);
      if (hit) my[nlist + popc_below(m)] = make_int2(slot, (ox & 0xFF) | (oy & 0xFF) << 8 | (oz & 0xFF) << 16);
      nlist += (int)__popcll(m);
      wave_sync64();
      st = candidate(c0 + kThreads64 + lane, slot);
      if (nlist > kListMax - 64) {  // whole groups now, the rest stays
        const int n = nlist & ~3;
        process(n);
        const int left = nlist - n;
        int2 keep = make_int2(0, 0);
        if (lane < left) keep = my[n + lane];
        wave_sync64();
        if (lane < left) my[lane] = keep;
        wave_sync64();
        nlist = left;
      }
    }
    if (nlist > 0) process(nlist);

    // the four waves' sums, slice by slice (two buffers: one barrier per slice)
    double2* fT = fw + (int64_t)tr * a.grid_cells;
    const int x = org[0] + (tid & 15), y = org[1] + (tid >> 4);
#pragma unroll
    for (int z = 0; z < kRZ; ++z) {
#pragma unroll
      for (int e = 0; e < 4; ++e) part[z & 1][wave][(4 * e + k) * kRX + i] = make_double2(re[z][e], im[z][e]);
      __syncthreads();
      double2 v = part[z & 1][0][tid];
#pragma unroll
      for (int w = 1; w < kWaves64; ++w) {
        const double2 u = part[z & 1][w][tid];
        v.x += u.x;
        v.y += u.y;
      }
      if (x < a.nf[0] && y < a.nf[1] && org[2] + z < a.nf[2]) {
        double2* cell = fT + ((int64_t)(org[2] + z) * a.nf[1] + y) * a.nf[0] + x;
        if (task.w > 1) {
          if (v.x != 0.0) atomic_add_global(&cell->x, v.x);
          if (v.y != 0.0) atomic_add_global(&cell->y, v.y);
        } else if (a.zero_out) {
          *cell = v;
        } else if (v.x != 0.0 || v.y != 0.0) {
          const double2 old = *cell;
          *cell = make_double2(old.x + v.x, old.y + v.y);
        }
      }
    }
  }
}

// The (point, strength) pairs left out as not finite: one wave each, lane q takes support cell q, q + 64, ...
template <int NS>
__global__ void __launch_bounds__(256) k_fix64(Reg64Args a, const cplx<double>* __restrict__ c,
                                               cplx<double>* __restrict__ fw) {
  const int n = a.cnt[3], lane = (int)threadIdx.x & 63;
  for (int b = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6); b < n; b += (int)gridDim.x * 4) {
    const int2 en = a.bad[b];
    const int p = a.perm[en.x];
    if ((unsigned)p >= (unsigned)a.M) continue;
    const cplx<double> v = c[(int64_t)en.y * a.M + p];
    cplx<double>* fT = fw + (int64_t)en.y * a.grid_cells;
    Folded f[3];
    int i0[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      f[d] = fold_coord(static_cast<const double*>(a.coord[d])[p], a.nf[d]);
      i0[d] = support_start(f[d], NS / 2);
    }
    for (int q = lane; q < NS * NS * NS; q += 64) {
      const int kk[3] = {q % NS, q / NS % NS, q / (NS * NS)};
      double w = 1.0;
      int64_t cell = 0;
#pragma unroll
      for (int d = 2; d >= 0; --d) {
        w *= es_phi(((double)i0[d] - f[d].xs) + (double)kk[d], a.beta, a.c);
        cell = cell * a.nf[d] + wrap_idx(i0[d] + kk[d], a.nf[d]);
      }
      atomic_add_global(&fT[cell].re, v.re * w);
      atomic_add_global(&fT[cell].im, v.im * w);
    }
  }
}

__global__ void k_zero_cnt64(int32_t* cnt) {
  if (threadIdx.x < 4) cnt[threadIdx.x] = 0;
}

// Candidates per task: 2048, less where the expected candidates would not give every resident block two
// tasks (30k points, 32^3 grid, 16 regions: 203 us per call with 2048, 140 with 256), down to 256 (each wave
// then has one step, and a task adds 4096 values for it).
struct Sizes64 {
  int nr[3], cand;
  int64_t regions, tasks;
};
constexpr int kBlocks64 = 768;  // three blocks per CU (registers), 256 CUs

// regions per dimension, and a bound of the tasks: the regions' candidate ranges hold a bin of dimension d
// at most (16 + ns + 2 bs - 2) / 16 + 2 times (8 in z)
Sizes64 sizes64(const Geometry& g, int64_t M) {
  Sizes64 z;
  const int len[3] = {kRX, kRY, kRZ};
  int64_t visits = 1;
  double expect = (double)M;
  z.regions = 1;
  for (int d = 0; d < 3; ++d) {
    z.nr[d] = (g.nf[d] + len[d] - 1) / len[d];
    z.regions *= z.nr[d];
    visits *= std::min<int64_t>(z.nr[d], (len[d] + g.ns + 2 * g.bs[d] - 2) / len[d] + 2);
    expect *= std::min((double)z.nr[d], (double)(len[d] + g.ns + g.bs[d]) / len[d]);
  }
  z.cand = (int)std::min<double>(kCandMax, std::max<double>(kCandMin, expect / (2 * kBlocks64)));
  z.tasks = z.regions + M * visits / z.cand + 1;
  return z;
}

int64_t runs64(const Geometry& g) {  // most runs around a region
  auto bins = [&](int d, int len) { return std::min<int64_t>(g.nb[d], (len + g.ns - 1) / g.bs[d] + 3); };
  return 2 * bins(1, kRY) * bins(2, kRZ);
}

}  // namespace

// Whether M points on a geometry are spread by regions: 3D FP64, supports that fit the grid, runs and weights
// that fit their bounds, and where it is the faster one (whole type-1 calls, against the atomic kernels): the atomic
// kernels' work grows with ns^3, the regions' little with ns, so from ns = 12 on at every size measured (2048 points on
// 32^3: 126 -> 86 us; 500k clustered points on 128^3, ns = 14: 4635 -> 1040 us); at ns = 10 from 100 regions on (20k uniform
// points: 32^3 grid, 16 regions, 96 -> 124 us, 64^3, 128 regions, 283 -> 149 us).  At ns = 8 the atomic kernels are slow where
// points crowd the tiles' cells, so it depends on the points: 400 regions and more 1.0 .. 3.5x (but 0.85x for 2100
// clustered points on 96^3); 100 .. 400 regions clustered points from 20k on 1.2 .. 2.0x, uniform ones 0.76 .. 1.1x (64^3:
// 20k points 107 -> 135 us uniform, 221 -> 132 clustered), fewer points 0.74 .. 1.17x, so from 16384 points on.  Not below
// (50k points on 128^3: ns = 6 299 -> 249 us uniform but 194 -> 228 us clustered, and 1M points 457 -> 826 us).
bool spread64_applicable(const Geometry& g, int prec, int64_t M, int64_t n_trans) {
  if (g.dim != 3 || prec != kF64 || g.ns < 8 || M < kSpread64MinPoints) return false;
  for (int d = 0; d < 3; ++d)
    if (g.nf[d] < g.ns) return false;
  const Sizes64 z = sizes64(g, M);
  if (g.ns < 12 && z.regions < 100) return false;
  if (g.ns == 8 && z.regions < 400 && M < 16384) return false;
  return z.regions < INT32_MAX && runs64(g) <= kRunsMax &&
         M * 3 * g.ns * (int64_t)sizeof(double) <= kTabMaxBytes && spread64_bytes(g, M, n_trans) <= kMaxBytes64 &&
         z.tasks <= (INT32_MAX - kBlocks64) / n_trans;  // a task number per transform, and one past the last per block
}

int64_t spread64_bytes(const Geometry& g, int64_t M, int64_t n_trans) {
  const Sizes64 z = sizes64(g, M);
  return M * (3 * g.ns * (int64_t)sizeof(double) + (int64_t)sizeof(int4)) + n_trans * M * (int64_t)(sizeof(double2) + sizeof(int2)) +
         z.tasks * (int64_t)sizeof(int4) + (z.regions + 4) * (int64_t)sizeof(int32_t);
}

// Buffers of a spread, the largest last: a set that cannot be had leaves the small ones only.
hipError_t spread64_reserve(PointSet& ps, const Geometry& g, int64_t n_trans) {
  const Sizes64 z = sizes64(g, ps.M);
  hipError_t e;
  if ((e = grow_buffer(ps.heavy64, ps.cap_heavy64, z.regions + 4, ps.retired)) != hipSuccess) return e;
  if ((e = grow_buffer(ps.task64, ps.cap_task64, z.tasks, ps.retired)) != hipSuccess) return e;
  if ((e = grow_buffer(ps.start64, ps.cap_start64, ps.M, ps.retired)) != hipSuccess) return e;
  if ((e = grow_buffer(ps.bad64, ps.cap_bad64, ps.M * n_trans, ps.retired)) != hipSuccess) return e;
  if ((e = grow_buffer(ps.cs64, ps.cap_cs64, ps.M * n_trans, ps.retired)) != hipSuccess) return e;
  return grow_buffer(ps.tab64, ps.cap_tab64, ps.M * 3 * g.ns, ps.retired);
}

bool spread64_reserved(const PointSet& ps, const Geometry& g, int64_t n_trans) {
  const Sizes64 z = sizes64(g, ps.M);
  return ps.cap_heavy64 >= z.regions + 4 && ps.cap_task64 >= z.tasks && ps.cap_start64 >= ps.M &&
         ps.cap_bad64 >= ps.M * n_trans && ps.cap_cs64 >= ps.M * n_trans && ps.cap_tab64 >= ps.M * 3 * g.ns;
}

hipError_t launch_spread64(const GridOpArgs& ga, const void* c, void* fw, hipStream_t s) {
  const PointSet& ps = *ga.ps;
  const Geometry& g = *ga.g;
  const Sizes64 z = sizes64(g, ps.M);
  Reg64Args a;
  a.M = ps.M;
  a.n_trans = ga.n_trans;
  a.grid_cells = g.grid_cells();
  for (int d = 0; d < 3; ++d) {
    a.nf[d] = g.nf[d];
    a.bs[d] = g.bs[d];
    a.nb[d] = g.nb[d];
    a.nr[d] = z.nr[d];
    a.coord[d] = ps.coord[d];
  }
  a.regions = (int)z.regions;
  a.max_tasks = (int)z.tasks;
  a.cand = z.cand;
  a.zero_out = ga.zero_out ? 1 : 0;
  a.bin_start = ps.bin_start;
  a.perm = ps.perm;
  a.beta = ga.beta;
  a.c = ga.c;
  a.tab = ps.tab64;
  a.start = ps.start64;
  a.cs = ps.cs64;
  a.task = ps.task64;
  a.cnt = ps.heavy64;
  a.heavy = ps.heavy64 + 4;
  a.bad = ps.bad64;
  const cplx<double>* cd = static_cast<const cplx<double>*>(c);
  auto launch = [&](auto nsc) -> hipError_t {
    constexpr int NS = decltype(nsc)::value;
    hipLaunchKernelGGL(k_zero_cnt64, dim3(1), dim3(64), 0, s, a.cnt);
    hipLaunchKernelGGL(k_tab64<NS>, dim3((unsigned)((ps.M + kTabPts - 1) / kTabPts)), dim3(3 * kTabPts), 0, s, a, cd);
    hipLaunchKernelGGL(k_tasks64<NS>, dim3((unsigned)((z.regions + kTaskRegions - 1) / kTaskRegions)), dim3(256), 0, s, a);
    if (ga.zero_out) hipLaunchKernelGGL(k_zero64, dim3(512), dim3(256), 0, s, a, static_cast<double2*>(fw));
    hipLaunchKernelGGL(k_spread64<NS>, dim3(kBlocks64), dim3(kThreads64), 0, s, a, static_cast<double2*>(fw));
    hipLaunchKernelGGL(k_fix64<NS>, dim3(64), dim3(256), 0, s, a, cd, static_cast<cplx<double>*>(fw));
    return hipGetLastError();
  };
  switch (g.ns) {
    case 8: return launch(std::integral_constant<int, 8>{});
    case 10: return launch(std::integral_constant<int, 10>{});
    case 12: return launch(std::integral_constant<int, 12>{});
    case 14: return launch(std::integral_constant<int, 14>{});
    case 16: return launch(std::integral_constant<int, 16>{});
  }
  return hipErrorInvalidValue;  // spread64_applicable admits no other
}

}  // namespace nufftx
