// Type-2 interpolation launchers (kernels in si_kernels.hpp and si_mfma.hpp).
#include <algorithm>
#include <cstdlib>

#include "si_mfma.hpp"
#include "si_gather3.hpp"
#include "si_win.hpp"

namespace nufftx {

namespace {

// 3D FP64: one wave per point straight from the grid instead of LDS tiles, whose FP64 cells leave one block of four
// waves per CU and whose halo is read again for every bin.  Whole type-2 calls, tiles -> waves: ns = 14 5990 -> 282 us
// (50k uniform points, 128^3 grid), 6280 -> 1145 (500k), 1119 -> 954 (500k points on 32^3); ns = 10 1407 -> 602 us (500k
// on 128^3) but 85 -> 94 (50k on 32^3) and 293 -> 461 (500k on 32^3); ns = 8 1205 -> 584 us (500k on 200^3) and 372 ->
// 394 (on 128^3); ns = 6 200 -> 128 us (50k on 128^3), 648 -> 537 (500k on 200^3) and 219 -> 359 (on 128^3).  So
// tiles pay from more points per cell the smaller the support is.
template <typename T, int D>
bool interp_by_wave(const Geometry& g, int64_t M) {
  if (D != 3 || !std::is_same<T, double>::value) return false;
  const int64_t cells = g.grid_cells();
  return g.ns >= 14 || M <= (g.ns >= 10 ? cells : g.ns == 8 ? cells / 8 : cells / 24);
}

// The 3D matrix-core gather: ns = 8, bins of whole 8 x 8 x 4 sub-bins (at most 16).  Whole type-2 calls, 32^3 .. 128^3
// modes, uniform and clustered, 0.003 .. 0.8 points per cell: 1.12 .. 1.19x faster than the thread-per-point gather (8M
// clustered points, 128^3: 1540 -> 1372 us; 20k points, 32^3: 70 -> 61).  At ns = 6 that one stays
// (0.79 .. 0.98x otherwise): its work falls with ns^3, that of the windows hardly.
bool gather3_applicable(const Geometry& g) {
  if (g.dim != 3 || g.ns != 8) return false;
  if (g.bs[0] % kW3SB || g.bs[1] % kW3SB || g.bs[2] % kW3SBZ) return false;
  if ((g.bs[0] / kW3SB) * (g.bs[1] / kW3SB) * (g.bs[2] / kW3SBZ) > 16) return false;
  for (int d = 0; d < 3; ++d)
    if (g.tile[d] > 127) return false;
  const Gather3Tile t = gather3_tile(g.bs, g.ns);
  return t.cells <= 4 * kG3Quads * kG3Threads && t.cells % 8 == 0 &&
         (size_t)t.cells * 8 + sizeof(Gather3Lds) + 256 <= (size_t)lds_device_max_bytes();
}

template <typename CT, int NS>
hipError_t launch_gather3(const GridOpArgs& ga, const SIArgs<float>& a, const void* fw, void* c, hipStream_t s) {
  auto kern = k_gather_win3<CT, NS, false>;
  if constexpr (NS == kEsPolyNs)
    if (a.poly.on) kern = k_gather_win3<CT, NS, true>;
  const size_t lds = (size_t)gather3_tile(ga.g->bs, NS).cells * 8;
  if (lds + sizeof(Gather3Lds) > 60000)
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  hipLaunchKernelGGL(kern, dim3(ga.ps->max_subprob, (unsigned)ga.n_trans), dim3(kG3Threads), lds, s, a,
                     static_cast<const cplx<float>*>(fw), static_cast<cplx<float>*>(c));
  return hipGetLastError();
}

template <typename T, typename CT, int D>
hipError_t interp_impl(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s) {
  const SIArgs<T> a = make_si_args<T>(ga);
  size_t lds = 0;
  const bool tiled = use_tiles(*ga.g, ga.prec, lds) && !interp_by_wave<T, D>(*ga.g, ga.ps->M);
  const PointSet& ps = *ga.ps;
  if constexpr (D == 3 && std::is_same<T, float>::value) {
    if (gather3_applicable(*ga.g)) return launch_gather3<CT, 8>(ga, a, fw, c, s);
  }
  GatherOut<T, D, false> o;
  o.val = static_cast<cplx<T>*>(c);
  o.P = nullptr;
  o.gcoord[0] = o.gcoord[1] = o.gcoord[2] = nullptr;
  o.store = false;
  return dispatch_ns(ga.g->ns, [&](auto nsc) -> hipError_t {
    constexpr int NS = decltype(nsc)::value;
    if (tiled) {
      if constexpr (std::is_same<T, float>::value && NS <= 8) {
        // 16-byte tile reads (k_gather_wide) unless NUFFTX_INTERP_WIDE=0; rows of an even
        // number of cells keep the reads aligned
        const char* ev = std::getenv("NUFFTX_INTERP_WIDE");
        const size_t lw = lds + 2 * sizeof(cplx<float>);  // the tile plus its two zero cells
        if ((a.tile[0] % 2) == 0 && lw <= (size_t)lds_device_max_bytes() && !(ev && std::atoi(ev) == 0)) {
          auto kw = k_gather_wide<CT, D, NS, false>;
          if constexpr (D == 2)
            if (a.crec) kw = k_gather_wide<CT, D, NS, true>;
          if constexpr (NS == kEsPolyNs)
            if (a.poly.on) {
              kw = k_gather_wide<CT, D, NS, false, true>;
              if constexpr (D == 2)
                if (a.crec) kw = k_gather_wide<CT, D, NS, true, true>;
            }
          if (lw > 65536) (void)hipFuncSetAttribute((const void*)kw, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lw);
          hipLaunchKernelGGL(kw, dim3(ps.max_subprob, (unsigned)ga.n_trans), dim3(256), lw, s, a,
                             static_cast<const cplx<float>*>(fw), static_cast<cplx<float>*>(c));
          return hipGetLastError();
        }
      }
      auto kern = k_gather_tiled<T, CT, D, NS, false>;
      if constexpr (D == 2 && std::is_same<T, float>::value)
        if (a.crec) kern = k_gather_tiled<T, CT, D, NS, false, true>;
      if (lds > 65536) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL(kern, dim3(ps.max_subprob, (unsigned)ga.n_trans), dim3(256), lds, s, a,
                         static_cast<const cplx<T>*>(fw), o);
    } else {
      const char* gw = std::getenv("NUFFTX_GLOBAL_WAVE");
      if (!(gw && gw[0] == '0')) {
        hipLaunchKernelGGL((k_gather_global_wave<T, CT, D, NS>), wave_grid(ps.M, ga.n_trans), dim3(256), 0, s, a,
                           static_cast<const cplx<T>*>(fw), static_cast<cplx<T>*>(c));
      } else {
        const unsigned nblk = (unsigned)((ps.M + 255) / 256);
        hipLaunchKernelGGL((k_gather_global<T, CT, D, NS, false>), dim3(nblk, (unsigned)ga.n_trans), dim3(256), 0, s,
                           a, static_cast<const cplx<T>*>(fw), o);
      }
    }
    return hipGetLastError();
  });
}

// The records-based matrix-core interpolation (needs the setpts point records).
bool interp_mfma(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s, hipError_t& err) {
  const PointSet& ps = *ga.ps;
  if (!ps.recs_subbin) return false;
  const SIArgs<float> a = make_si_args<float>(ga);
  auto launch = [&](auto nsc) -> bool {
    constexpr int NS = decltype(nsc)::value;
    const size_t lds = MfmaGeom<NS>::interp_lds();
    if (lds > (size_t)lds_device_max_bytes()) return false;
    auto kern = k_interp_mfma2d<NS>;
    if (lds > 65536) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3(ps.max_subprob, (unsigned)ga.n_trans), dim3(kMfmaThreads), lds, s, a, ps.recs,
                       ps.sub_off, static_cast<const cplx<float>*>(fw), static_cast<cplx<float>*>(c));
    err = hipGetLastError();
    return true;
  };
  switch (ga.g->ns) {
    case 2: return launch(std::integral_constant<int, 2>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    case 6: return launch(std::integral_constant<int, 6>{});
    case 8: return launch(std::integral_constant<int, 8>{});
  }
  return false;
}

// The matrix-core window interpolation (2D FP32, ns <= 8, window bins, compact records).
bool interp_win(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s, hipError_t& err) {
  const PointSet& ps = *ga.ps;
  if (!win2d_geometry(*ga.g, ga.prec, ps.maxsub) || !ps.has_crec || !win_interp_enabled()) return false;
  const SIArgs<float> a = make_si_args<float>(ga);
  if (!a.crec) return false;
  auto launch = [&](auto nsc) -> bool {
    constexpr int NS = decltype(nsc)::value;
    const size_t lds = wi_interp_lds<NS>(ps.maxsub);
    // static LDS (ordering counters) below 2.2 KB
    if (lds + 2304 > (size_t)lds_device_max_bytes()) return false;
    auto kern = k_interp_win2dh<NS>;
    if (lds > 65536) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(kern, dim3(ps.max_subprob, (unsigned)ga.n_trans), dim3(kWiThreads), lds, s, a, ps.maxsub,
                       static_cast<const cplx<float>*>(fw), static_cast<cplx<float>*>(c));
    err = hipGetLastError();
    return true;
  };
  switch (ga.g->ns) {
    case 2: return launch(std::integral_constant<int, 2>{});
    case 4: return launch(std::integral_constant<int, 4>{});
    case 6: return launch(std::integral_constant<int, 6>{});
    case 8: return launch(std::integral_constant<int, 8>{});
  }
  return false;
}

template <typename T, typename CT>
hipError_t interp_dim(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    hipError_t err = hipSuccess;
    if (mfma2d_applicable(*ga.g, ga.prec) && use_mfma() && interp_mfma(ga, fw, c, s, err)) return err;
    if (interp_win(ga, fw, c, s, err)) return err;
  }
  switch (ga.g->dim) {
    case 2: return interp_impl<T, CT, 2>(ga, fw, c, s);
    case 3: return interp_impl<T, CT, 3>(ga, fw, c, s);
  }
  return hipErrorInvalidValue;
}

template <typename CT, int D>
hipError_t interp_many_impl(const GridOpArgs* gas, int count, const void* const* fw, void* const* c, hipStream_t s) {
  size_t lmax = 0;
  GatherMany m;
  m.count = count;
  m.first[0] = 0;
  for (int i = 0; i < count; ++i) {
    size_t l = 0;
    if (!use_tiles(*gas[i].g, gas[i].prec, l)) return hipErrorNotSupported;
    lmax = std::max(lmax, l);
    m.a[i] = make_si_args<float>(gas[i]);
    m.fw[i] = static_cast<const cplx<float>*>(fw[i]);
    m.out[i] = static_cast<cplx<float>*>(c[i]);
    m.first[i + 1] = m.first[i] + std::max(0, gas[i].ps->max_subprob);
  }
  for (int i = count; i < kMaxMany; ++i) m.first[i + 1] = m.first[count];
  if (m.first[count] == 0) return hipSuccess;
  const bool rec = m.a[0].crec != nullptr;
  for (int i = 1; i < count; ++i)
    if ((m.a[i].crec != nullptr) != rec) return hipErrorNotSupported;
  return dispatch_ns(gas[0].g->ns, [&](auto nsc) -> hipError_t {
    constexpr int NS = decltype(nsc)::value;
    auto kern = k_gather_tiled_many<CT, D, NS, false>;
    if constexpr (D == 2)
      if (rec) kern = k_gather_tiled_many<CT, D, NS, true>;
    if (lmax > 65536) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lmax);
    hipLaunchKernelGGL(kern, dim3((unsigned)m.first[count], (unsigned)gas[0].n_trans), dim3(256), lmax, s, m);
    return hipGetLastError();
  });
}

}  // namespace

hipError_t launch_interp_many(const GridOpArgs* gas, int count, const void* const* fw, void* const* c, hipStream_t s) {
  if (count < 1 || count > kMaxMany) return hipErrorNotSupported;
  const GridOpArgs& g0 = gas[0];
  if (g0.prec != kF32 || g0.g->dim < 2 || use_mfma()) return hipErrorNotSupported;
  for (int i = 0; i < count; ++i) {
    const GridOpArgs& g = gas[i];
    if (g.prec != kF32 || g.g->dim != g0.g->dim || g.g->ns != g0.g->ns || g.n_trans != g0.n_trans ||
        g.ps->coord_f64 != g0.ps->coord_f64 || g.beta != g0.beta || g.c != g0.c || g.ps->M == 0 ||
        g.g->tile_cells != g0.g->tile_cells)  // one LDS size for the whole launch (see launch_spread_many)
      return hipErrorNotSupported;
  }
  const bool f64 = g0.ps->coord_f64;
  if (g0.g->dim == 2)
    return f64 ? interp_many_impl<double, 2>(gas, count, fw, c, s) : interp_many_impl<float, 2>(gas, count, fw, c, s);
  return f64 ? interp_many_impl<double, 3>(gas, count, fw, c, s) : interp_many_impl<float, 3>(gas, count, fw, c, s);
}

hipError_t launch_interp(const GridOpArgs& ga, const void* fw, void* c, hipStream_t s) {
  if (ga.ps->M == 0) return hipSuccess;
  if (interp1d_direct(*ga.g)) return launch_interp1d(ga, fw, c, s);
  if (ga.prec == kF32) {
    return ga.ps->coord_f64 ? interp_dim<float, double>(ga, fw, c, s) : interp_dim<float, float>(ga, fw, c, s);
  }
  return interp_dim<double, double>(ga, fw, c, s);
}

}  // namespace nufftx
