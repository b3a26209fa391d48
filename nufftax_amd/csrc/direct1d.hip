// 1D spreading and interpolation without a sort.
//
// A 1D support is ns adjacent cells, so what the bin-sort buys in 2D and 3D (tiles of the grid in LDS, shared by
// the points of a bin) costs more here than it gives: three to five launches, and then gathers and scatters of 4
// to 16 bytes through the permutation.  Points are taken in the caller's order instead, read and written whole:
//   k_spread1d   grids of up to kSpread1dCells cells: every block spreads its share of the points into an LDS copy
//                of the whole grid (the accumulators of k_spread_tiled: exact 64-bit fixed point in FP32,
//                ds_add_f64 in FP64) and adds it to the grid; a single block stores it.  100k points, 2048 cells:
//                11 us and a clear, against sort 24, strength bound 5 and spread 12 us in 7 launches.
//   k_interp1d   any grid: one thread per point reads its ns cells from LDS (grids of up to kInterp1dCells, staged
//                by every block) or from memory.  3M points, 2M cells (16 MB): 65 us against sort 75 and gather 78.
// Larger grids are spread from sorted points, as before: an LDS tile per bin is what saves them the global atomics.
#include <algorithm>

#include "si_kernels.hpp"

namespace nufftx {

namespace {

constexpr int kSpread1dCells = 4096;   // 64 KB of accumulators
constexpr int kInterp1dCells = 4096;   // 32 KB (FP32) or 64 KB (FP64) of grid
constexpr int kThreads1d = 512;
constexpr int kPpt1d = 4;              // points per thread and step
constexpr int kBlocks1d = 512;         // blocks of a launch aimed at where there are more points than a step of each

template <typename T>
struct Args1d {
  const void* x;
  int64_t M;
  int nf, per_block;  // points per block
  EsArgs<T> es;
};

// The ns support cells of a point fold onto the grid by at most one subtraction (nf >= ns), or a remainder.
__device__ __forceinline__ int wrap1d(int g, int nf) {
  if (g < 0) g += nf;
  if (g >= nf) g -= nf;
  return (unsigned)g < (unsigned)nf ? g : wrap_idx(g, nf);
}

template <typename T, typename CT, int NS>
__global__ void __launch_bounds__(kThreads1d) k_spread1d(Args1d<T> a, const cplx<T>* __restrict__ c,
                                                         cplx<T>* __restrict__ fw, int store) {
  constexpr bool kFixed = std::is_same<T, float>::value;
  using Acc = typename std::conditional<kFixed, unsigned long long, double>::type;
  extern __shared__ __align__(16) unsigned char smem1d[];
  Acc* sre = reinterpret_cast<Acc*>(smem1d);
  Acc* sim = sre + a.nf;
  __shared__ unsigned smax;
  const int tid = (int)threadIdx.x;
  const cplx<T>* cT = c + (int64_t)blockIdx.y * a.M;
  cplx<T>* fT = fw + (int64_t)blockIdx.y * a.nf;
  const int64_t lo = (int64_t)blockIdx.x * a.per_block, hi = min(a.M, lo + (int64_t)a.per_block);
  for (int i = tid; i < a.nf; i += kThreads1d) {
    sre[i] = (Acc)0;
    sim[i] = (Acc)0;
  }
  if (tid == 0) smax = 0u;
  __syncthreads();
  // fixed-point scale: every partial sum of a cell is below B = 2 n max(|re c|, |im c|) over the block's points
  double scale = 1.0, inv_scale = 1.0;
  bool finite = true;
  if constexpr (kFixed) {
    unsigned m = 0;
    for (int64_t i = lo + tid; i < hi; i += kThreads1d) {
      const cplx<T> v = cT[i];
      m = max(m, max(__float_as_uint(fabsf(v.re)), __float_as_uint(fabsf(v.im))));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off, 64));
    if ((tid & 63) == 0) atomicMax(&smax, m);
    __syncthreads();
    const double B = 2.0 * (double)(hi - lo) * (double)__uint_as_float(smax);
    finite = isfinite(B);
    if (finite && B > 0.0) {
      int e;
      (void)frexp(B, &e);  // B < 2^e
      scale = ldexp(1.0, 50 - e);
      inv_scale = ldexp(1.0, e - 50);
    }
  }
  for (int64_t i0 = lo + tid; i0 < hi && finite; i0 += (int64_t)kThreads1d * kPpt1d) {
    CT xv[kPpt1d];
    cplx<T> cv[kPpt1d];
#pragma unroll
    for (int u = 0; u < kPpt1d; ++u) {  // all loads first
      const int64_t i = i0 + (int64_t)u * kThreads1d;
      xv[u] = i < hi ? static_cast<const CT*>(a.x)[i] : (CT)0;
      cv[u] = i < hi ? cT[i] : cplx<T>{(T)0, (T)0};
    }
#pragma unroll
    for (int u = 0; u < kPpt1d; ++u) {
      if (i0 + (int64_t)u * kThreads1d >= hi) break;
      const Folded f = fold_coord((double)xv[u], a.nf);
      const int s = support_start(f, NS / 2);
      const T t = (T)((double)s - f.xs);
      const double cre = (double)cv[u].re * scale, cim = (double)cv[u].im * scale;
#pragma unroll
      for (int k = 0; k < NS; ++k) {
        const double w = (double)es_phi(t + (T)k, a.es.beta_log2e, a.es.c);
        const int g = wrap1d(s + k, a.nf);
        if constexpr (kFixed) {
          atomicAdd(sre + g, TileAcc<float>::quant(cre, w));
          atomicAdd(sim + g, TileAcc<float>::quant(cim, w));
        } else {
          atomicAdd(sre + g, cre * w);
          atomicAdd(sim + g, cim * w);
        }
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < a.nf; i += kThreads1d) {
    T vr, vi;
    if constexpr (kFixed) {
      vr = finite ? (T)((double)(long long)sre[i] * inv_scale) : (T)NAN;
      vi = finite ? (T)((double)(long long)sim[i] * inv_scale) : (T)NAN;
    } else {
      vr = sre[i];
      vi = sim[i];
    }
    if (store) {
      fT[i] = cplx<T>{vr, vi};
    } else {
      if (vr != (T)0) atomic_add_global(&fT[i].re, vr);
      if (vi != (T)0) atomic_add_global(&fT[i].im, vi);
    }
  }
}

template <typename T, typename CT, int NS, bool LDS>
__global__ void __launch_bounds__(kThreads1d) k_interp1d(Args1d<T> a, const cplx<T>* __restrict__ fw,
                                                         cplx<T>* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem1d[];
  cplx<T>* tile = reinterpret_cast<cplx<T>*>(smem1d);
  const int tid = (int)threadIdx.x;
  const cplx<T>* fT = fw + (int64_t)blockIdx.y * a.nf;
  cplx<T>* oT = out + (int64_t)blockIdx.y * a.M;
  const int64_t lo = (int64_t)blockIdx.x * a.per_block, hi = min(a.M, lo + (int64_t)a.per_block);
  if constexpr (LDS) {
    for (int i = tid; i < a.nf; i += kThreads1d) tile[i] = fT[i];
    __syncthreads();
  }
  for (int64_t i = lo + tid; i < hi; i += kThreads1d) {
    const Folded f = fold_coord((double)static_cast<const CT*>(a.x)[i], a.nf);
    const int s = support_start(f, NS / 2);
    const T t = (T)((double)s - f.xs);
    const cplx<T>* src = LDS ? tile : fT;
    cplx<T> v[NS];
    if (s >= 0 && s + NS <= a.nf) {  // all but the points near the ends: adjacent cells
#pragma unroll
      for (int k = 0; k < NS; ++k) v[k] = src[s + k];
    } else {
#pragma unroll
      for (int k = 0; k < NS; ++k) v[k] = src[wrap1d(s + k, a.nf)];
    }
    cplx<T> sum = {(T)0, (T)0};
#pragma unroll
    for (int k = 0; k < NS; ++k) {
      const T w = es_phi(t + (T)k, a.es.beta_log2e, a.es.c);
      sum.re += v[k].re * w;
      sum.im += v[k].im * w;
    }
    oT[i] = sum;
  }
}

template <typename T>
Args1d<T> args1d(const GridOpArgs& ga, int per_block) {
  Args1d<T> a;
  a.x = ga.ps->coord[0];
  a.M = ga.ps->M;
  a.nf = ga.g->nf[0];
  a.per_block = per_block;
  const double log2e = 1.4426950408889634074;
  a.es.beta_log2e = std::is_same<T, float>::value ? (T)(ga.beta * log2e) : (T)ga.beta;
  a.es.beta = (T)ga.beta;
  a.es.c = (T)ga.c;
  return a;
}

// points per block: one step of every thread at least, at most `blocks` blocks
int points_per_block(int64_t M, int step, int64_t blocks) {
  const int64_t p = (M + blocks - 1) / blocks;
  return (int)((std::max<int64_t>(p, step) + kThreads1d - 1) / kThreads1d * kThreads1d);
}

template <typename T, typename CT>
hipError_t spread1d_run(const GridOpArgs& ga, const void* c, void* fw, hipStream_t s) {
  const int64_t M = ga.ps->M;
  // Up to one block's worth of points: the block stores the grid (no clear, no atomics).  All transforms together have
  // kBlocks1d blocks, two per CU: each adds a whole grid to memory with atomics, which 512 blocks for each of several
  // transforms spent most of their time on (8 FP64 transforms of 1M points, 4096 cells: 455 us, now 251; sorted 303).
  const int per = points_per_block(M, kThreads1d * kPpt1d, std::max<int64_t>(1, kBlocks1d / ga.n_trans));
  const unsigned nb = (unsigned)((M + per - 1) / per);
  const Args1d<T> a = args1d<T>(ga, per);
  const int store = nb == 1 && ga.zero_out ? 1 : 0;
  if (ga.zero_out && !store) {
    hipError_t e = launch_zero(fw, ga.n_trans * (int64_t)a.nf * (int64_t)sizeof(cplx<T>), s);
    if (e != hipSuccess) return e;
  }
  const size_t lds = (size_t)a.nf * 16;
  return dispatch_ns(ga.g->ns, [&](auto nsc) -> hipError_t {
    constexpr int NS = decltype(nsc)::value;
    auto kern = k_spread1d<T, CT, NS>;
    if (lds > 60000) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3(nb, (unsigned)ga.n_trans), dim3(kThreads1d), lds, s, a, static_cast<const cplx<T>*>(c),
                       static_cast<cplx<T>*>(fw), store);
    return hipGetLastError();
  });
}

template <typename T, typename CT>
hipError_t interp1d_run(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s) {
  const int64_t M = ga.ps->M;
  const bool lds = ga.g->nf[0] <= kInterp1dCells;
  // (a block that reads the grid from memory gains nothing from more points)
  const int per = lds ? points_per_block(M, kThreads1d, kBlocks1d) : kThreads1d;
  const unsigned nb = (unsigned)((M + per - 1) / per);
  const Args1d<T> a = args1d<T>(ga, per);
  const size_t bytes = lds ? (size_t)a.nf * sizeof(cplx<T>) : 0;
  return dispatch_ns(ga.g->ns, [&](auto nsc) -> hipError_t {
    constexpr int NS = decltype(nsc)::value;
    auto kern = lds ? k_interp1d<T, CT, NS, true> : k_interp1d<T, CT, NS, false>;
    if (bytes > 60000) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    hipLaunchKernelGGL(kern, dim3(nb, (unsigned)ga.n_trans), dim3(kThreads1d), bytes, s, a,
                       static_cast<const cplx<T>*>(fw), static_cast<cplx<T>*>(c));
    return hipGetLastError();
  });
}

}  // namespace

bool spread1d_direct(const Geometry& g) { return g.dim == 1 && g.nf[0] <= kSpread1dCells; }
bool interp1d_direct(const Geometry& g) { return g.dim == 1; }

hipError_t launch_spread1d(const GridOpArgs& ga, const void* c, void* fw, hipStream_t s) {
  if (ga.prec == kF32)
    return ga.ps->coord_f64 ? spread1d_run<float, double>(ga, c, fw, s) : spread1d_run<float, float>(ga, c, fw, s);
  return spread1d_run<double, double>(ga, c, fw, s);
}

hipError_t launch_interp1d(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s) {
  if (ga.prec == kF32)
    return ga.ps->coord_f64 ? interp1d_run<float, double>(ga, fw, c, s) : interp1d_run<float, float>(ga, fw, c, s);
  return interp1d_run<double, double>(ga, fw, c, s);
}

}  // namespace nufftx
