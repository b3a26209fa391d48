// 3D FP32 interpolation on the matrix cores: the transpose of the window spread of si_win3.hpp.
//
// The points of one sub-bin of 8 x 8 x 4 support starts read one window F of 16 x 16 x (4 + ns) cells:
//   v_j = sum_z wz_j(z) sum_y wy_j(y) sum_x F[z][y][x] wx_j(x)        (nufftax/core/spread.py:661-715)
// so for 16 points the x sums of one z slice and part are one matrix product G = F Bx.  F and wx are split into
// two fp16 parts (hi + lo: 22 bits and more, scaled to the top of fp16's range, as in the spread), and the K = 32 of
// v_mfma_f32_16x16x32_f16 holds the 16 x twice, [F_lo | F_hi] against [B_lo ; B_lo] and then [B_hi ; B_hi]: all four
// products in two instructions, nothing left out but the roundings of lo, the small ones summed first.  The tile is staged in LDS
// already split, as four fp16 planes (re and im, hi and lo: 8 bytes a cell, as FP32), so that a lane reads 8 cells of one plane
// with one 16-byte read, its operand; a window is read once per sub-bin that a wave visits, into (4 + ns) * 8
// registers.  A group then costs two MFMAs and 5 FMAs per slice and part.  (Windows read from the grid by each wave,
// 64 rows a load: 1937 us where the thread-per-point gather takes 1170; 8M points.)
//
// What bounds the thread-per-point gather (k_gather_wide) is its LDS: 8 ns^3 bytes and a quarter per point, at scattered
// rows (8M clustered points, ns = 8, 128^3 modes: 41 GB, 520 us at the LDS's rate, 1170 measured).  Here a point's cells
// are shared by its group.  1031 us measured for those points, two blocks per CU (78 KB of LDS, 191 registers); counters:
// vector units 49% busy, matrix cores 17%, LDS 6%, and 3.9 GB fetched, most of it lines of 128 bytes for coordinates
// read through the sort's permutation (96 MB of them): memory and arithmetic take about 0.8 and 0.7 of the time, in part
// one after the other.
//
// Block = one subproblem (points of one bin, 1024 at a time), 4 waves:
//   1. order: every point's words (support start in the tile, fraction) into LDS, and its place in sub-bin order
//      (sub-bins padded to multiples of 16); the tile's cells load meanwhile and are split into the planes;
//   2. contiguous ranges of groups per wave; per group the lanes evaluate the 3 ns weights of the 16 points into LDS
//      rows with zeros around them (read at the point's offset in the window), then multiply.
// A tile that holds a non-finite value would spread it through the zero weights: its points take their own cells
// one by one.  So do points whose result is small beside the tile's largest value (2^-13), whose cells the common
// scale of the tile leaves too few bits.
//
// MFMA operand layout: A[i][k] in lane i + 16 (k / 8), element k % 8; B[k][j] in lane j + 16 (k / 8), element k % 8;
// D[i][j] in lane j + 16 (i / 4), element i % 4.
#pragma once

#include "si_win3.hpp"

namespace nufftx {

constexpr int kG3Threads = 256;
constexpr int kG3Waves = kG3Threads / 64;
constexpr int kG3Ppt = 4;                             // points per thread while ordering
constexpr int kG3MaxSub = kG3Threads * kG3Ppt;        // points ordered at once
constexpr int kG3K = 16;                              // points per group
constexpr int kG3RowF = kG3K * kWinRow + 16;          // x or y weight rows of a wave (17 floats a row, trailing zeros)
constexpr int kG3WaveF = 2 * kG3RowF + kG3K * kW3RowZ + 16 + 4 * kG3K;  // floats per wave: x, y, z rows, meta
constexpr int kG3Order = kG3MaxSub + 16 * (kG3K - 1);

// staged cells per dimension: whole windows (nsx sub-bins reach 8 nsx + 8 cells whatever ns)
struct Gather3Tile {
  int nsx, nsy, nsz, tx, ty, tz, cells;
};
__host__ __device__ inline Gather3Tile gather3_tile(const int (&bs)[3], int ns) {
  Gather3Tile t;
  t.nsx = bs[0] / kW3SB;
  t.nsy = bs[1] / kW3SB;
  t.nsz = bs[2] / kW3SBZ;
  t.tx = kW3SB * t.nsx + 8;
  t.ty = kW3SB * t.nsy + 8;
  t.tz = kW3SBZ * t.nsz + ns;
  t.cells = t.tx * t.ty * t.tz;
  return t;
}
constexpr int kG3Quads = 6;  // four-cell pieces of the tile per thread: 24 x 16 x 16 cells

struct Gather3Lds {
  uint3 word[kG3MaxSub];       // tile-relative words of the points (g3_word)
  uint16_t order[kG3Order];
  alignas(16) float wave[kG3Waves][kG3WaveF];
  unsigned short wcnt[kG3Ppt * kG3Waves * 16];
  int cnt[16], start[17];
  unsigned smax;
};

// tile-relative word of one coordinate: support start - org << 25 | round((t + ns/2) 2^25), t = start - xs.  (The compact
// records' 2^-24 cells would be the next largest error of the gather after the FP32 sums.)
template <int NS>
__device__ __forceinline__ unsigned g3_word(double x, int nf, int org) {
  const Folded f = fold_coord(x, nf);
  const int i0 = support_start(f, NS / 2);
  const double u = ((double)i0 - f.xs + (double)(NS / 2)) * 33554432.0;  // 2^25
  return ((unsigned)(i0 - org) << 25) | (unsigned)fmin(fmax(rint(u), 0.0), 33554431.0);
}

// Results below this (in the products' units, where the tile's largest value is about 2^29) are taken from the cells instead:
// an fp16 lo part resolves 2^-24 at least (the matrix cores take subnormal fp16 operands as they are), so the products of a
// cell are off by up to 2^-11 of these units, which a sum of 2^16 carries in its last FP32 bits.
constexpr float kG3Small = 65536.0f;

// sum over the four lanes i, i + 16, i + 32, i + 48 of a point
template <typename T>
__device__ __forceinline__ T quad_sum(T v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

template <typename CT, int NS, bool POLY>
__global__ void __launch_bounds__(kG3Threads, 2) k_gather_win3(SIArgs<float> a, const cplx<float>* __restrict__ fw,
                                                               cplx<float>* __restrict__ out) {
  constexpr int WZ = kW3SBZ + NS;
  constexpr uint16_t kPad = 0xFFFF, kBad = 0x8000;  // entries of the order: slot, and a mark
  static_assert(kG3MaxSub < kBad, "slots leave the mark free");
  __shared__ __align__(16) Gather3Lds L;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  _Float16* const planes = reinterpret_cast<_Float16*>(smem_raw);  // [re hi, re lo, im hi, im lo][z][y][x]
  const int sub = blockIdx.x, tr = blockIdx.y;
  if (sub >= *a.nsub) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int4 sd = a.subprob[sub];
  const Gather3Tile T = gather3_tile(a.bs, NS);
  const int nsx = T.nsx, nsy = T.nsy, nsz = T.nsz;
  int org[3];
  tile_origin<3>(sd, a.bs, a.nb, NS / 2, org);
  const cplx<float>* fT = fw + (int64_t)tr * a.grid_cells;
  float* const rowx = L.wave[wave];
  float* const rowy = rowx + kG3RowF;
  float* const rowz = rowy + kG3RowF;
  int4* const meta = reinterpret_cast<int4*>(rowz + kG3K * kW3RowZ + 16);  // {x, y, z read index, point index}
  static_assert((2 * kG3RowF + kG3K * kW3RowZ + 16) % 4 == 0 && kG3WaveF % 4 == 0, "meta is 16-byte aligned");
  for (int e = lane; e < 2 * kG3RowF + kG3K * kW3RowZ + 16; e += 64) rowx[e] = 0.0f;  // the rows' zeros stay zero
  if (tid == 0) L.smax = 0u;

  // ---- the tile's cells, four neighbours in x at a time (they load while the points are ordered)
  cplx<float> cell[kG3Quads][4];
#pragma unroll
  for (int u = 0; u < kG3Quads; ++u) {
    const int q = tid + u * kG3Threads;  // quad: x fastest
    const int x = q % (T.tx >> 2) * 4, yz = q / (T.tx >> 2);
    const int y = yz % T.ty, z = yz / T.ty;
#pragma unroll
    for (int e = 0; e < 4; ++e) cell[u][e] = cplx<float>{0.0f, 0.0f};
    if (4 * q < T.cells) {
      const cplx<float>* src =
          fT + ((int64_t)wrap_near(org[2] + z, a.nf[2]) * a.nf[1] + wrap_near(org[1] + y, a.nf[1])) * a.nf[0];
#pragma unroll
      for (int e = 0; e < 4; ++e) cell[u][e] = src[wrap_near(org[0] + x + e, a.nf[0])];
    }
  }

  // ---- 1. words and order of points base .. base + 1023
  const auto order_points = [&](int base) {
    if (tid < kG3Ppt * kG3Waves * 16 / 2) reinterpret_cast<unsigned*>(L.wcnt)[tid] = 0u;
    __syncthreads();
    int sb[kG3Ppt], rank[kG3Ppt];
    bool bad[kG3Ppt];  // a coordinate is not finite: NaN weights, a NaN result
#pragma unroll
    for (int r = 0; r < kG3Ppt; ++r) {
      const int j = tid + r * kG3Threads;
      sb[r] = -1;
      bad[r] = false;
      if (base + j < sd.z) {
        const int p = a.perm[sd.y + base + j];
        uint3 w = make_uint3(0u, 0u, 0u);
        double xyz[3] = {0.0, 0.0, 0.0};
        if ((unsigned)p < (unsigned)a.M) {
#pragma unroll
          for (int d = 0; d < 3; ++d) xyz[d] = (double)static_cast<const CT*>(a.coord[d])[p];
          w = make_uint3(g3_word<NS>(xyz[0], a.nf[0], org[0]), g3_word<NS>(xyz[1], a.nf[1], org[1]),
                         g3_word<NS>(xyz[2], a.nf[2], org[2]));
        }
        L.word[j] = w;
        bad[r] = !(isfinite(xyz[0]) && isfinite(xyz[1]) && isfinite(xyz[2]));
        const int sx = min((int)(w.x >> 25) / kW3SB, nsx - 1), sy = min((int)(w.y >> 25) / kW3SB, nsy - 1);
        const int sz = min((int)(w.z >> 25) / kW3SBZ, nsz - 1);
        sb[r] = (sz * nsy + sy) * nsx + sx;
      }
    }
#pragma unroll
    for (int r = 0; r < kG3Ppt; ++r) {
      const bool valid = sb[r] >= 0;
      uint64_t m = __ballot(valid);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const uint64_t bal = __ballot(valid && ((sb[r] >> b) & 1));
        m &= ((sb[r] >> b) & 1) ? bal : ~bal;
      }
      rank[r] = popc_below(m);
      if (valid && rank[r] == 0) L.wcnt[(r * kG3Waves + wave) * 16 + sb[r]] = (unsigned short)__popcll(m);
    }
    __syncthreads();
    if (tid < 16) {  // counts per sub-bin, padded starts (16 lanes of one wave), first slot of every (pass, wave) run
      int c = 0;
#pragma unroll
      for (int e = 0; e < kG3Ppt * kG3Waves; ++e) c += L.wcnt[e * 16 + tid];
      const int padded = (c + kG3K - 1) & ~(kG3K - 1);
      int incl = padded;
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) {
        const int t = __shfl_up(incl, off, 16);
        if (tid >= off) incl += t;
      }
      L.cnt[tid] = c;
      L.start[tid] = incl - padded;
      if (tid == 15) L.start[16] = incl;
      int run = incl - padded;
#pragma unroll
      for (int e = 0; e < kG3Ppt * kG3Waves; ++e) {
        const int v = L.wcnt[e * 16 + tid];
        L.wcnt[e * 16 + tid] = (unsigned short)run;
        run += v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kG3Ppt; ++r)
      if (sb[r] >= 0)
        L.order[L.wcnt[(r * kG3Waves + wave) * 16 + sb[r]] + rank[r]] =
            (uint16_t)((tid + r * kG3Threads) | (bad[r] ? kBad : 0));
    if (tid < 16 * (kG3K - 1)) {
      const int s = tid / (kG3K - 1), slot = L.start[s] + L.cnt[s] + tid % (kG3K - 1);
      if (slot < L.start[s + 1]) L.order[slot] = kPad;
    }
  };
  order_points(0);
  // the tile's scale (its largest |re|, |im|: bit patterns order as the values, NaN above all), then the planes
  {
    unsigned mx = 0;
#pragma unroll
    for (int u = 0; u < kG3Quads; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        mx = max(mx, max(__float_as_uint(fabsf(cell[u][e].re)), __float_as_uint(fabsf(cell[u][e].im))));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, off, 64));
    if (lane == 0) atomicMax(&L.smax, mx);
  }
  __syncthreads();
  const float fm = __uint_as_float(L.smax);
  const bool fine = isfinite(fm);
  int ke = 0;  // A = F 2^ke, |A| < 2^15
  if (fine && fm > 0.0f) {
    (void)frexpf(fm, &ke);
    ke = 15 - ke;
  }
  const int kout = -ke - 14;  // B carries 2^14
#pragma unroll
  for (int u = 0; u < kG3Quads; ++u) {
    const int q = tid + u * kG3Threads;
    float v[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = ldexpf(cell[u][e].re, ke);
      v[4 + e] = ldexpf(cell[u][e].im, ke);
    }
    wh_h8 hi, lo;
    split_f16(v, hi, lo);
    if (4 * q < T.cells) {
      typedef _Float16 h4 __attribute__((ext_vector_type(4)));
      *reinterpret_cast<h4*>(planes + 4 * q) = h4{hi[0], hi[1], hi[2], hi[3]};
      *reinterpret_cast<h4*>(planes + T.cells + 4 * q) = h4{lo[0], lo[1], lo[2], lo[3]};
      *reinterpret_cast<h4*>(planes + 2 * T.cells + 4 * q) = h4{hi[4], hi[5], hi[6], hi[7]};
      *reinterpret_cast<h4*>(planes + 3 * T.cells + 4 * q) = h4{lo[4], lo[5], lo[6], lo[7]};
    }
  }
  __syncthreads();

  // ---- 2. groups of 16 points of one sub-bin
  const int i = lane & 15, kq = lane >> 4;
  // weight staging: this lane's row, its entry of the window's first cell, its dimension's sub-bins
  const unsigned* const word = reinterpret_cast<const unsigned*>(L.word);
  const int mybase = kq < 2 ? kWinRow * i + (16 - NS) : kW3RowZ * i + kW3SBZ;
  float* const myrow = (kq == 0 ? rowx : kq == 1 ? rowy : rowz) + mybase;
  const int mysh = kq < 2 ? 3 : 2, myn = (kq == 0 ? nsx : kq == 1 ? nsy : nsz) - 1;
  static_assert(kW3SB == 8 && kW3SBZ == 4, "sub-bin sides are shifts");
  wh_h8 fre[WZ], fim[WZ];
  for (int base = 0;;) {
    const int NG = L.start[16] / kG3K;
    const int g0 = NG * wave / kG3Waves, g1 = NG * (wave + 1) / kG3Waves;
    int next = 0, s = -1;
    for (int g = g0; g < g1; ++g) {
      if (kG3K * g >= next) {
        do {
          ++s;
        } while (s < 15 && L.start[s + 1] <= kG3K * g);
        next = L.start[s + 1];
        // the window: lane (y = i, kq) takes x = 8 (kq & 1) .. + 7 of row i of every slice, of the lo (kq < 2) or hi plane
        const int at = ((s / (nsx * nsy) * kW3SBZ) * T.ty + (s / nsx % nsy) * kW3SB + i) * T.tx + (s % nsx) * kW3SB + 8 * (kq & 1) +
                       (kq < 2 ? T.cells : 0);
#pragma unroll
        for (int z = 0; z < WZ; ++z) {
          fre[z] = *reinterpret_cast<const wh_h8*>(planes + at + z * T.ty * T.tx);
          fim[z] = *reinterpret_cast<const wh_h8*>(planes + at + z * T.ty * T.tx + 2 * T.cells);
        }
      }
      // -- weights and read indices: lanes 0-15 x, 16-31 y, 32-47 z of point i, 48-63 its index
      {
        const int entry = L.order[kG3K * g + i], slot = entry & (kBad - 1);
        const bool real = entry != kPad;
        if (kq < 3) {
          const unsigned wd = real ? word[3 * slot + kq] : 0u;
          float wt[NS];
          if constexpr (POLY) {
            // v = 2 (t + NS/2) - 1, exactly (|u - 2^24| <= 2^24)
            es_poly_weights<NS>((float)((int)(wd & 0x1FFFFFFu) - 16777216) * (1.0f / 16777216.0f), a.poly, wt);
          } else {
            const float t = (float)((double)(wd & 0x1FFFFFFu) * (1.0 / 33554432.0) - (double)(NS / 2));
#pragma unroll
            for (int m = 0; m < NS; ++m) wt[m] = es_phi_in(t + (float)m, a.es.beta_log2e, a.es.c);
          }
          const float sc = real && (entry & kBad) ? NAN : kq == 0 ? 16384.0f : 1.0f;
#pragma unroll
          for (int m = 0; m < NS; ++m) myrow[m] = wt[m] * sc;
          const int l = (int)(wd >> 25);
          reinterpret_cast<int*>(meta + i)[kq] = mybase - (l - (min(l >> mysh, myn) << mysh));
        } else {
          reinterpret_cast<int*>(meta + i)[3] = real ? a.perm[sd.y + base + slot] : -1;
        }
      }
      wave_sync_win();
      const int4 mt = meta[i];
      float sr = 0.0f, si = 0.0f;
      bool cells = !fine;
      if (fine) {
        float bx[8], wy[4];
#pragma unroll
        for (int e = 0; e < 8; ++e) bx[e] = rowx[mt.x + 8 * (kq & 1) + e];
#pragma unroll
        for (int e = 0; e < 4; ++e) wy[e] = rowy[mt.y + 4 * kq + e];
        wh_h8 bh, bl;
        split_f16(bx, bh, bl);
        const win_f4 zero4 = {0.f, 0.f, 0.f, 0.f};
        // The sums over slices and lanes in FP64 make up for the split's roundings: relative l2 1.12e-7 on random grids, the
        // gather of one thread per point 1.16e-7 (two or six slices summed in FP32 first: 1.17 and 1.20e-7; 8M clustered
        // points, 128^3 modes, whole type 2 1365 us, with those 1342 and 1322).
        double zr = 0.0, zi = 0.0;
#pragma unroll
        for (int z = 0; z < WZ; ++z) {
          win_f4 gr = __builtin_amdgcn_mfma_f32_16x16x32_f16(fre[z], bl, zero4, 0, 0, 0);
          win_f4 gi = __builtin_amdgcn_mfma_f32_16x16x32_f16(fim[z], bl, zero4, 0, 0, 0);
          gr = __builtin_amdgcn_mfma_f32_16x16x32_f16(fre[z], bh, gr, 0, 0, 0);
          gi = __builtin_amdgcn_mfma_f32_16x16x32_f16(fim[z], bh, gi, 0, 0, 0);
          const float wz = rowz[mt.z + z];
          float pr = gr[0] * wy[0], pi = gi[0] * wy[0];
#pragma unroll
          for (int e = 1; e < 4; ++e) {
            pr = fmaf(gr[e], wy[e], pr);
            pi = fmaf(gi[e], wy[e], pi);
          }
          zr = fma((double)pr, (double)wz, zr);
          zi = fma((double)pi, (double)wz, zi);
        }
        sr = (float)quad_sum(zr + (double)sr);
        si = (float)quad_sum(zi + (double)si);
        cells = fm > 0.0f && fmaxf(fabsf(sr), fabsf(si)) < kG3Small;
        sr = ldexpf(sr, kout);
        si = ldexpf(si, kout);
      }
      cells = cells && mt.w >= 0;
      if (__any(cells)) {  // (rare, or a tile that is not finite)
        // support rows of the point, lane kq the slices kq, kq + 4, ..: its own cells only, in FP32
        float cr = 0.0f, ci = 0.0f;
        if (cells) {
          const uint3 w = L.word[L.order[kG3K * g + i] & (kBad - 1)];
          const int x0 = org[0] + (int)(w.x >> 25), y0 = org[1] + (int)(w.y >> 25), z0 = org[2] + (int)(w.z >> 25);
          for (int z = kq; z < NS; z += 4) {
            float pr = 0.0f, pi = 0.0f;
            for (int y = 0; y < NS; ++y) {
              const cplx<float>* src = fT + ((int64_t)wrap_idx(z0 + z, a.nf[2]) * a.nf[1] + wrap_idx(y0 + y, a.nf[1])) * a.nf[0];
              float rr = 0.0f, ri = 0.0f;
              for (int x = 0; x < NS; ++x) {
                const cplx<float> v = src[wrap_idx(x0 + x, a.nf[0])];
                const float wx = rowx[kWinRow * i + (16 - NS) + x] * (1.0f / 16384.0f);
                rr = fmaf(v.re, wx, rr);
                ri = fmaf(v.im, wx, ri);
              }
              const float wy = rowy[kWinRow * i + (16 - NS) + y];
              pr = fmaf(rr, wy, pr);
              pi = fmaf(ri, wy, pi);
            }
            const float wz = rowz[kW3RowZ * i + kW3SBZ + z];
            cr = fmaf(pr, wz, cr);
            ci = fmaf(pi, wz, ci);
          }
        }
        cr = quad_sum(cr);
        ci = quad_sum(ci);
        if (cells) {
          sr = cr;
          si = ci;
        }
      }
      if (kq == 0 && (unsigned)mt.w < (unsigned)a.M) out[(int64_t)tr * a.M + mt.w] = cplx<float>{sr, si};
      wave_sync_win();  // the next group overwrites the rows
    }
    base += kG3MaxSub;
    if (base >= sd.z) break;
    __syncthreads();  // all waves are done with the words and the order
    order_points(base);
    __syncthreads();
  }
}

}  // namespace nufftx
