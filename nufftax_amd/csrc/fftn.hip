// Mixed-radix FFT of the fine grid fused with the deconvolution, mode truncation and shift (type 1) or zero
// padding (type 2), for the grids that fft2d.hip does not take: FP64, and FP32 grids that are not
// powers of two (grid sizes are 2-3-5-smooth, nufftax/utils/grid.py:6-58).  The DFT is that of
// nufftax/transforms/nufft1.py:81 and nufft2.py:74, the mode placement that of deconvolve.py:174-304.
//
// One pass per axis, each on the kept modes of the axes that are not transformed yet (type 2: z, y, x) or are
// already (type 1: x, y, z), so nothing is done for padding: a 3D type 2 with n of 2 n bins per axis
// moves (1/8 + 1/4) + (1/4 + 1/2) + (1/2 + 1) of the grid, where a library FFT after a padding pass moves 1/8 + 1 and
// 6, its strided axes at a fraction of the memory's rate (540^3 FP64, 2.5 GB, from 270^3 modes: rocFFT and the
// padding pass 5400 us; these passes 1600: x, y and z 3.8, 1.9 and 0.95 GB at 4.7, 3.9 and 3.3 TB/s, where a large copy
// reaches 4.8).  The x pass, the largest, reads and writes whole rows; y and z passes take S neighbouring x at once (runs
// of 128 bytes) and keep the order of the axes.  (An earlier form, contiguous reads and transposed writes on every axis,
// took 3440 us: its last pass wrote 64-byte runs over 540 planes.)  Axes longer than
// kMaxLen (1D) are split N = Na Nb (four-step, Bailey 1990): length-Na transforms over every Nb-th value, times
// exp(-2 pi i b n / N), then length-Nb ones.
//
// A sequence of N = R_1 R_2 .. points is transformed by Stockham passes (fft2d.hip describes the recurrence) of
// radix 2 .. 16, each thread taking one R-point column in registers (fft_dft.hpp), T = max N / R threads
// per sequence.  The first pass takes its column from memory and the last one stores it, so the data goes through
// LDS between passes only.  The factorisation with the fewest passes and then the largest smallest radix is
// taken (540 = 9 10 6, T = 90).  The inverse transform swaps real and imaginary parts on the way in and out.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "fft_dft.hpp"
#include "internal.hpp"

namespace nufftx {

namespace {

constexpr int kMaxLen = 4096;      // points per sequence
// threads per block, by the registers that a column of up to RMAX points needs without spilling
__host__ __device__ constexpr int fftn_threads(int real_bytes, int rmax) {
  return real_bytes == 8 || rmax > 10 ? 768 : 1024;
}
constexpr int kRowThreads = 256;   // aimed at where rows are short
constexpr int kMaxPasses = 8;
constexpr int kFftnBlocks = 4096;  // blocks of a pass: several rounds of what the CUs hold

// What one side of a pass holds: every value, the kept modes of the axis, these with deconvolution factors,
// or (output) every value times the twiddles of a split axis
enum { kValues, kModes, kFactors, kTwiddle };

struct FftnStep {     // one Stockham pass
  int R, ns, nr;      // radix, product of the earlier radices, N / R columns
  int tstep;          // twiddle step N / (ns R) of column residue 1
  unsigned magic;     // q / ns = umulhi(q, magic) for ns > 1 (q < 2^16)
};

template <typename T>
struct FftnPass {
  int N, T_seq, S, log_s, nsteps;
  FftnStep step[kMaxPasses];
  int nseq, D1, groups;             // sequence s = a D1 + b; blocks' worth of S sequences
  int64_t P1, P2, istride, Q1, Q2, ostride;  // a P1 + b P2 + value istride; the same for the output
  int64_t in_t, out_t;              // per transform
  int kmax, klow, c0, c1;           // bin -> mode: bin <= kmax: bin + c0, bin >= klow: bin + c1, else none
  int ib, is, ob, os;               // value i of sequence b is bin i ib + b is (in), i ob + b os (out)
  int64_t tw_n;                     // kTwiddle: output j of sequence b times exp(-2 pi i b j / tw_n)
  const T *facA, *facB, *facC;      // deconvolution factors of this axis' mode, of b and of a, or null
  const fcplx<T>* tw;               // exp(-2 pi i k / N), k < N
  int swap;                         // exponent sign +
};

// LDS length of a sequence stored in one piece (a pad slot per 16 values and an odd stride spread power-of-two
// strides over the banks); with runs, value n of sequence r is at n S + r instead
__host__ __device__ __forceinline__ int fftn_len(int n) { return (n + (n >> 4)) | 1; }

// LDS position of value n of the thread's sequence (base: r, or r times the sequence length)
template <bool INTERLEAVED>
__device__ __forceinline__ int fftn_at(int base, int log_s, int n) {
  return INTERLEAVED ? (n << log_s) + base : base + n + (n >> 4);
}

// What a thread needs on the global side: its sequence's first offset on each side and its factors.  Offsets are 32-bit
// byte offsets from the transform's uniform base (one register per address, no 64-bit arithmetic;
// fftn_applicable admits arrays below 4 GiB), and grow by uniform steps from value to value: the passes
// are bound by their instructions, most of them addresses.
template <typename T>
struct SeqIO {
  const char* in;
  char* out;
  unsigned in0, out0;
  int b;
  bool on;
  T fac;  // facB facC of the sequence
};

// v[r] = input value i0 + r di
template <typename T, int R, int IN>
__device__ __forceinline__ void fftn_load(const FftnPass<T>& P, const SeqIO<T>& io, int i0, int di, fcplx<T> (&v)[R]) {
  const unsigned step = (unsigned)(P.istride * (int64_t)sizeof(fcplx<T>));
  if constexpr (IN == kValues) {
    const unsigned at = io.in0 + (unsigned)i0 * step, d = (unsigned)di * step;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = *reinterpret_cast<const fcplx<T>*>(io.in + (at + r * d));
  } else {
    const int bin0 = i0 * P.ib + io.b * P.is, db = di * P.ib;
    const unsigned at = io.in0 + (unsigned)(bin0 + P.c0) * step, d = (unsigned)db * step, wrap = (unsigned)(P.c1 - P.c0) * step;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int bin = bin0 + r * db;
      const bool low = bin <= P.kmax;
      v[r] = {T(0), T(0)};
      if (low || bin >= P.klow) v[r] = *reinterpret_cast<const fcplx<T>*>(io.in + (at + r * d + (low ? 0u : wrap)));
    }
    if constexpr (IN == kFactors) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int bin = bin0 + r * db;
        const bool low = bin <= P.kmax;
        if (low || bin >= P.klow) {
          const T f = io.fac * P.facA[bin + (low ? P.c0 : P.c1)];
          v[r] = {v[r].x * f, v[r].y * f};
        }
      }
    }
  }
  if (P.swap) {
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = {v[r].y, v[r].x};
  }
}

// output value j0 + r dj = v[r]
template <typename T, int R, int OUT>
__device__ __forceinline__ void fftn_store(const FftnPass<T>& P, const SeqIO<T>& io, int j0, int dj, fcplx<T> (&v)[R]) {
  const unsigned step = (unsigned)(P.ostride * (int64_t)sizeof(fcplx<T>));
  if constexpr (OUT == kTwiddle) {
// exp(-2 pi i b (j0 + r dj) / n): two evaluations and a product per value, in FP64
    double s0, c0, s1, c1;
    sincospi(2.0 * (double)(((int64_t)io.b * j0) % P.tw_n) / (double)P.tw_n, &s0, &c0);
    sincospi(2.0 * (double)(((int64_t)io.b * dj) % P.tw_n) / (double)P.tw_n, &s1, &c1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      v[r] = fmul(v[r], fcplx<T>{(T)c0, (T)-s0});
      const double c = c0 * c1 - s0 * s1;
      s0 = s0 * c1 + c0 * s1;
      c0 = c;
    }
  }
  if (P.swap) {
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = {v[r].y, v[r].x};
  }
  if constexpr (OUT == kValues || OUT == kTwiddle) {
    const unsigned at = io.out0 + (unsigned)j0 * step, d = (unsigned)dj * step;
#pragma unroll
    for (int r = 0; r < R; ++r) *reinterpret_cast<fcplx<T>*>(io.out + (at + r * d)) = v[r];
  } else {
    const int bin0 = j0 * P.ob + io.b * P.os, db = dj * P.ob;
    const unsigned at = io.out0 + (unsigned)(bin0 + P.c0) * step, d = (unsigned)db * step, wrap = (unsigned)(P.c1 - P.c0) * step;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int bin = bin0 + r * db;
      const bool low = bin <= P.kmax;
      if (!low && bin < P.klow) continue;
      if constexpr (OUT == kFactors) {
        const T f = io.fac * P.facA[bin + (low ? P.c0 : P.c1)];
        v[r] = {v[r].x * f, v[r].y * f};
      }
      *reinterpret_cast<fcplx<T>*>(io.out + (at + r * d + (low ? 0u : wrap))) = v[r];
    }
  }
}

// One Stockham pass of radix R over the block's sequences (every read of LDS precedes every write of the pass).
template <typename T, int R, int IN, int OUT, bool RUNS>
__device__ __forceinline__ void fftn_radix(const FftnPass<T>& P, const SeqIO<T>& io, fcplx<T>* buf, int base,
                                           const fcplx<T>* tw, const FftnStep& st, int q, bool first, bool last) {
  // (the radices' code must not merge: shared address computations, hoisted out of the switch, and shared tails,
  // with every radix's column live at once, would take twice the registers)
  asm volatile("; radix %1" : "+v"(q) : "n"(R));
  const bool on = io.on && q < st.nr;
  fcplx<T> v[R];
  int d = q * R;
  if (on) {
    if (first) {
      fftn_load<T, R, IN>(P, io, q, st.nr, v);
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) v[r] = buf[fftn_at<RUNS>(base, P.log_s, q + r * st.nr)];
      if (st.ns > 1) {
        const int k = q - (int)__umulhi((unsigned)q, st.magic) * st.ns;
        d = (q - k) * R + k;
        const int w = k * st.tstep;  // k N / (ns R)
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = fmul(v[r], tw[r * w]);
      }
    }
    Dft<T, R>::run(v);
  }
  if (last) {
    if (on) fftn_store<T, R, OUT>(P, io, d, st.ns, v);
    asm volatile("; radix %0 stored" ::"n"(R));
    return;
  }
  if (!first) __syncthreads();
  if (on) {
#pragma unroll
    for (int r = 0; r < R; ++r) buf[fftn_at<RUNS>(base, P.log_s, d + r * st.ns)] = v[r];
  }
  asm volatile("; radix %0 done" ::"n"(R));
  __syncthreads();
}

// RMAX: largest radix of the axis (10 or 16).  RUNS: consecutive lanes take consecutive sequences (S a power of two),
// else consecutive values.
template <typename T, int RMAX, int IN, int OUT, bool RUNS>
__global__ void __launch_bounds__(fftn_threads(sizeof(T), RMAX)) k_fftn(FftnPass<T> P, const fcplx<T>* __restrict__ in,
                                                                      fcplx<T>* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char fftn_smem[];
  const int N = P.N, S = P.S, tid = (int)threadIdx.x, nt = (int)blockDim.x;
  fcplx<T>* stw = reinterpret_cast<fcplx<T>*>(fftn_smem);
  fcplx<T>* buf = stw + N;
  const fcplx<T>* inT = in + (int64_t)blockIdx.y * P.in_t;
  fcplx<T>* outT = out + (int64_t)blockIdx.y * P.out_t;
  if (P.nsteps > 1)
    for (int e = tid; e < N; e += nt) stw[e] = P.tw[e];
  const int PL = fftn_len(N);
  const int sq = RUNS ? tid & (S - 1) : tid / P.T_seq;
  const int q = RUNS ? tid >> P.log_s : tid - sq * P.T_seq;
  const int base = RUNS ? sq : sq * PL;
  SeqIO<T> io;
  io.in = reinterpret_cast<const char*>(inT);
  io.out = reinterpret_cast<char*>(outT);
  // Groups of runs that share lines (runs of 16 to 64 bytes on long axes) go to blocks of one XCD, i.e. one L2: block b
  // runs on XCD b mod 8 (the grid is a multiple of 8), and XCD k takes the k-th eighth of the groups in order.  In plain
  // order every L2 fetched and wrote back parts of the same lines (type 1 on a 2400 x 2400 FP32 grid 137 us, now 110;
  // 3000 x 3000 FP64 286, now 217).
  const int per = (P.groups + 7) / 8;
  for (int id = (int)blockIdx.x; id < (RUNS ? 8 * per : P.groups); id += (int)gridDim.x) {
    const int g = RUNS ? (id & 7) * per + (id >> 3) : id;
    if (g >= P.groups) continue;
    const int s0 = g * S;
    io.on = sq < S && q < P.T_seq && s0 + sq < P.nseq;
    const unsigned s = io.on ? (unsigned)(s0 + sq) : 0u, a = s / (unsigned)P.D1;
    io.b = (int)(s - a * (unsigned)P.D1);
    io.in0 = (unsigned)(((int64_t)a * P.P1 + (int64_t)io.b * P.P2) * (int64_t)sizeof(fcplx<T>));
    io.out0 = (unsigned)(((int64_t)a * P.Q1 + (int64_t)io.b * P.Q2) * (int64_t)sizeof(fcplx<T>));
    io.fac = (P.facB ? P.facB[io.b] : T(1)) * (P.facC ? P.facC[a] : T(1));
#pragma unroll 1
    for (int p = 0; p < P.nsteps; ++p) {
      const FftnStep st = P.step[p];
      const bool first = p == 0, last = p == P.nsteps - 1;
      switch (st.R) {  // uniform
#define FFTN_RADIX(r) fftn_radix<T, r, IN, OUT, RUNS>(P, io, buf, base, stw, st, q, first, last)
        case 2: FFTN_RADIX(2); break;
        case 3: FFTN_RADIX(3); break;
        case 4: FFTN_RADIX(4); break;
        case 5: FFTN_RADIX(5); break;
        case 6: FFTN_RADIX(6); break;
        case 8: FFTN_RADIX(8); break;
        case 9: FFTN_RADIX(9); break;
        case 10: FFTN_RADIX(10); break;
        default:
          if constexpr (RMAX > 10) {
            if (st.R == 12)
              FFTN_RADIX(12);
            else if (st.R == 15)
              FFTN_RADIX(15);
            else
              FFTN_RADIX(16);
          }
#undef FFTN_RADIX
      }
    }
    __syncthreads();  // the next group's first pass writes LDS
  }
}

// ---------------------------------------------------------------- host
constexpr int kRadices[] = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};

// radices with the fewest passes, then the largest smallest radix; false if n is not 2-3-5-smooth
bool factorise(int n, int most, std::vector<int>& best, std::vector<int>& cur, int from) {
  if (n == 1) {
    auto low = [](const std::vector<int>& v) { return v.empty() ? 1 : *std::min_element(v.begin(), v.end()); };
    if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && low(cur) > low(best))) best = cur;
    return true;
  }
  if ((int)cur.size() >= most) return false;
  bool any = false;
  for (int q = from; q < (int)(sizeof(kRadices) / sizeof(int)); ++q)
    if (n % kRadices[q] == 0) {
      cur.push_back(kRadices[q]);
      any |= factorise(n / kRadices[q], most, best, cur, q);
      cur.pop_back();
    }
  return any;
}

// Radices above 10 take the registers of some of the waves: FP32 axes use them where they leave two passes in 3D (type 1 of
// 500 points on 160^3: 88 us, 95 without; not in 2D, whose passes are short of waves: 4 transforms on 240 x 240 42.5,
// 39.4), or three on a long axis (1440 x 1440: 73.5, 77.1), not to save the fourth pass of a short one (type 2 on
// 375 x 375: 39.2, 37.0); FP64 axes never (2400 x 2400: 140, 129).
std::vector<int> radices_of(int n, int prec, int dim) {
  std::vector<int> best, cur;
  for (int most = 1; most <= kMaxPasses && best.empty() && n > 1; ++most) {
    factorise(n, most, best, cur, 3);  // up to 10
    if (best.empty() && prec == kF32 && ((most == 2 && dim == 3) || (most == 3 && n > 1024))) factorise(n, most, best, cur, 0);
  }
  // odd radices first: the first pass writes with a stride of its radix
  std::stable_partition(best.begin(), best.end(), [](int r) { return r % 2 != 0; });
  return best;
}

// Whether one pass transforms an axis of n points: its threads and its LDS (twiddles and one sequence) fit a block.
bool axis_fits(int n, int prec, int dim) {
  if (n < 2 || n > kMaxLen) return false;
  const std::vector<int> r = radices_of(n, prec, dim);
  if (r.empty()) return false;
  const int lo = *std::min_element(r.begin(), r.end()), hi = *std::max_element(r.begin(), r.end());
  const int real_bytes = prec == kF32 ? 4 : 8;
  return (n / lo + 63) / 64 * 64 <= fftn_threads(real_bytes, hi > 10 ? 16 : 10) &&
         (size_t)(n + fftn_len(n)) * 2 * real_bytes <= (size_t)lds_device_max_bytes();
}

// N = Na Nb, as near as can be, with axes that fit; 0 if there is none
int split_length(int n, int prec) {
  for (int a = (int)std::sqrt((double)n) + 1; a >= 2; --a)
    if (n % a == 0 && axis_fits(a, prec, 1) && axis_fits(n / a, prec, 1)) return a;
  return 0;
}

template <typename T>
hipError_t twiddle_table(void*& dst, int n) {
  std::vector<fcplx<T>> h((size_t)n);
  for (int k = 0; k < n; ++k) {
    const double ang = -2.0 * 3.14159265358979323846 * (double)k / (double)n;
    h[k] = {(T)std::cos(ang), (T)std::sin(ang)};
  }
  void* p = nullptr;
  hipError_t e = dev_malloc(&p, h.size() * sizeof(h[0]));
  if (e != hipSuccess) return e;
  if ((e = hipMemcpy(p, h.data(), h.size() * sizeof(h[0]), hipMemcpyHostToDevice)) != hipSuccess) {
    (void)hipFree(p);
    return e;
  }
  dst = p;
  return hipSuccess;
}

template <typename T>
struct Runner {
  const FftnPlan& fp;
  const DeconvArgs& a;
  hipStream_t s;
  bool swap;
  hipError_t err = hipSuccess;

  const T* fac(int d) const { return static_cast<const T*>(a.fac[d]); }

  // a pass over axis `axis` (twiddles and radices of entry `tab`)
  template <int IN, int OUT, bool RUNS>
  void pass(int axis, int tab, FftnPass<T> P, const void* in, void* out, int64_t n_trans) {
    if (err != hipSuccess) return;
    const FftnPlan::Axis& ax = fp.axis[tab];
    P.N = ax.n;
    P.nsteps = (int)ax.radix.size();
    P.T_seq = 1;
    for (int p = 0, ns = 1; p < P.nsteps; ns *= ax.radix[p], ++p) {
      FftnStep& st = P.step[p];
      st.R = ax.radix[p];
      st.ns = ns;
      st.nr = ax.n / st.R;
      st.tstep = st.nr / ns;
      st.magic = ns > 1 ? (unsigned)(((1ull << 32) + (unsigned)ns - 1) / (unsigned)ns) : 0u;
      P.T_seq = std::max(P.T_seq, st.nr);
    }
    P.tw = static_cast<const fcplx<T>*>(ax.tw);
    const int nm = a.nm[axis], nb = a.nf[axis];
    P.kmax = (nm - 1) / 2;
    P.klow = nb - nm / 2;
    P.c0 = a.modeord == 0 ? nm / 2 : 0;
    P.c1 = (a.modeord == 0 ? nm / 2 : nm) - nb;
    P.swap = swap ? 1 : 0;
    const bool big = *std::max_element(ax.radix.begin(), ax.radix.end()) > 10;
    const int most = fftn_threads(sizeof(T), big ? 16 : 10);
    auto lds = [&](int S) { return (size_t)(P.N + S * (RUNS ? P.N : fftn_len(P.N))) * sizeof(fcplx<T>); };
    if (RUNS) {
      // runs of 128 bytes, shorter where the LDS (two blocks per CU), the threads or a small grid asks for it
      P.S = 128 / (int)sizeof(fcplx<T>);
      while (P.S > 1 && (P.S * P.T_seq > most || lds(P.S) > 80 * 1024)) P.S /= 2;
      while (P.S > 4 && (P.nseq + P.S - 1) / P.S * n_trans < 512) P.S /= 2;
      while ((1 << P.log_s) < P.S) ++P.log_s;
    } else {
      // whole rows, up to 256 threads, several blocks per CU
      P.S = std::max(1, std::min(P.nseq, kRowThreads / P.T_seq));
      while (P.S > 1 && lds(P.S) > 40 * 1024) --P.S;
    }
    P.groups = (P.nseq + P.S - 1) / P.S;
    const int threads = std::max(64, (P.S * P.T_seq + 63) / 64 * 64);
    const size_t bytes = lds(P.S);
    if (threads > most || bytes > (size_t)lds_device_max_bytes()) {  // (axis_fits admits no such axis)
      err = hipErrorInvalidConfiguration;
      return;
    }
    auto kern = k_fftn<T, 10, IN, OUT, RUNS>;
    if constexpr (sizeof(T) == 4)
      if (big) kern = k_fftn<T, 16, IN, OUT, RUNS>;
    if (bytes > 65536) (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    // large passes: blocks that stay take several groups, for one load of the twiddles
    int64_t blocks = std::min<int64_t>(P.groups, std::max<int64_t>(1, kFftnBlocks / n_trans));
    if (RUNS) blocks = (blocks + 7) / 8 * 8;  // (see the kernel's order of groups)
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks, (unsigned)n_trans), dim3(threads), bytes, s, P,
                       static_cast<const fcplx<T>*>(in), static_cast<fcplx<T>*>(out));
    err = hipGetLastError();
  }

  // Transforms axis `axis` of an array [outer][len][inner] (inner = 1: rows), modes -> bins or bins -> modes.
  FftnPass<T> axis_pass(int axis, bool to_grid, int64_t outer, int64_t inner) {
    const int64_t ni = to_grid ? a.nm[axis] : a.nf[axis], no = to_grid ? a.nf[axis] : a.nm[axis];
    FftnPass<T> P{};
    P.nseq = (int)(outer * inner);
    P.D1 = (int)inner;
    P.P1 = ni * inner;
    P.Q1 = no * inner;
    P.P2 = P.Q2 = 1;
    P.istride = P.ostride = inner;
    P.in_t = outer * ni * inner;
    P.out_t = outer * no * inner;
    P.ib = P.ob = 1;
    return P;
  }

  // modes -> grid: z in the grid's memory, y in the intermediate
  void to_grid(const void* f, void* grid) {
    const int64_t n0 = a.nm[0], n1 = a.nm[1], f0 = a.nf[0], f1 = a.nf[1], f2 = a.nf[2];
    FftnPass<T> P;
    if (a.dim == 3) {
      P = axis_pass(2, true, 1, n1 * n0);  // sequence = m1 n0 + m0: factors of both
      P.D1 = (int)n0; P.P1 = P.Q1 = n0;
      P.facA = fac(2); P.facB = fac(0); P.facC = fac(1);
      pass<kFactors, kValues, true>(2, 2, P, f, grid, a.n_trans);
      pass<kModes, kValues, true>(1, 1, axis_pass(1, true, f2, n0), grid, fp.mid, a.n_trans);
      pass<kModes, kValues, false>(0, 0, axis_pass(0, true, f2 * f1, 1), fp.mid, grid, a.n_trans);
    } else if (a.dim == 2) {
      P = axis_pass(1, true, 1, n0);
      P.facA = fac(1); P.facB = fac(0);
      pass<kFactors, kValues, true>(1, 1, P, f, fp.mid, a.n_trans);
      pass<kModes, kValues, false>(0, 0, axis_pass(0, true, f1, 1), fp.mid, grid, a.n_trans);
    } else if (!fp.split) {  // the transforms are the rows
      P = axis_pass(0, true, a.n_trans, 1);
      P.facA = fac(0);
      pass<kFactors, kValues, false>(0, 0, P, f, grid, 1);
    } else {
      const int64_t na = fp.split, nb = f0 / na;
      P = axis_pass(0, true, 1, nb);  // value i of sequence b is bin i nb + b
      P.in_t = n0; P.P2 = 0; P.istride = 1; P.ib = (int)nb; P.is = 1; P.tw_n = f0; P.out_t = f0;
      P.facA = fac(0);
      pass<kFactors, kTwiddle, true>(0, 0, P, f, fp.mid, a.n_trans);
      P = axis_pass(0, false, 1, na);  // rows of nb values; output j of sequence b is bin j na + b
      P.P2 = nb; P.istride = 1; P.in_t = P.out_t = f0;
      pass<kValues, kValues, true>(0, 1, P, fp.mid, grid, a.n_trans);
    }
  }

  // grid -> modes: x in the intermediate, y in the grid's memory
  void to_modes(void* grid, void* f) {
    const int64_t n0 = a.nm[0], n1 = a.nm[1], f0 = a.nf[0], f1 = a.nf[1], f2 = a.nf[2];
    FftnPass<T> P;
    if (a.dim == 3) {
      pass<kValues, kModes, false>(0, 0, axis_pass(0, false, f2 * f1, 1), grid, fp.mid, a.n_trans);
      pass<kValues, kModes, true>(1, 1, axis_pass(1, false, f2, n0), fp.mid, grid, a.n_trans);
      P = axis_pass(2, false, 1, n1 * n0);
      P.D1 = (int)n0; P.P1 = P.Q1 = n0;
      P.facA = fac(2); P.facB = fac(0); P.facC = fac(1);
      pass<kValues, kFactors, true>(2, 2, P, grid, f, a.n_trans);
    } else if (a.dim == 2) {
      pass<kValues, kModes, false>(0, 0, axis_pass(0, false, f1, 1), grid, fp.mid, a.n_trans);
      P = axis_pass(1, false, 1, n0);
      P.facA = fac(1); P.facB = fac(0);
      pass<kValues, kFactors, true>(1, 1, P, fp.mid, f, a.n_trans);
    } else if (!fp.split) {
      P = axis_pass(0, false, a.n_trans, 1);
      P.facA = fac(0);
      pass<kValues, kFactors, false>(0, 0, P, grid, f, 1);
    } else {
      const int64_t na = fp.split, nb = f0 / na;
      P = axis_pass(0, false, 1, nb);
      P.tw_n = f0; P.in_t = P.out_t = f0;
      pass<kValues, kTwiddle, true>(0, 0, P, grid, fp.mid, a.n_trans);
      P = axis_pass(0, false, 1, na);
      P.P2 = nb; P.istride = 1; P.in_t = f0;
      P.Q2 = 0; P.ostride = 1; P.ob = (int)na; P.os = 1; P.out_t = n0;
      P.facA = fac(0);
      pass<kValues, kFactors, true>(0, 1, P, fp.mid, f, a.n_trans);
    }
  }
};

template <typename T>
hipError_t fftn_run(FftnPlan& fp, const DeconvArgs& a, bool to_grid, const void* src, void* dst, int isign, hipStream_t s) {
  Runner<T> r{fp, a, s, isign > 0};
  if (to_grid)
    r.to_grid(src, dst);
  else
    r.to_modes(const_cast<void*>(src), dst);
  return r.err;
}

}  // namespace

// Whether every axis is 2-3-5-smooth and fits a pass (1D: or two), and offsets fit 32 bits.
bool fftn_applicable(const DeconvArgs& a) {
  if (a.dim < 1 || a.dim > 3 || a.from_phihat) return false;
  // small 3D FP64 grids stay with rocFFT, which transforms two short axes in one launch (type 1 of 2000 points: 64^3 grid
  // 65 us, 77 with three passes; 80^3 87, 91; 96^3 106, 102)
  if (a.dim == 3 && a.prec == kF64 && (int64_t)a.nf[0] * a.nf[1] * a.nf[2] < 700000) return false;
  double bytes = a.prec == kF32 ? 8.0 : 16.0;
  for (int d = 0; d < a.dim; ++d) bytes *= a.nf[d];
  if (bytes * (a.dim == 1 ? a.n_trans : 1) > 4294967295.0) return false;
  for (const char* name : {a.dim == 3 ? "NUFFTX_FFT3_FUSED" : "", a.dim == 1 ? "NUFFTX_FFT1_FUSED" : ""})
    if (name[0])
      if (const char* e = std::getenv(name))
        if (e[0] == '0') return false;
  // 1D FP32 beyond 8M cells stays with rocFFT: both halves of the split have some 3000 points there, whose sequences leave
  // runs of 8 and 16 bytes (type 1 of 500 points: 8M cells 183 us, rocFFT 195; 9M 253, 220; 12M 328, 276.  FP64 12M 520, 555)
  if (a.dim == 1 && a.prec == kF32 && a.nf[0] > 8000000) return false;
  for (int d = 0; d < a.dim; ++d) {
    if (a.nf[d] < 2 || a.nm[d] > a.nf[d]) return false;
    if (!axis_fits(a.nf[d], a.prec, a.dim) && (a.dim > 1 || split_length(a.nf[d], a.prec) == 0)) return false;
  }
  return true;
}

int64_t fftn_mid_bytes(const DeconvArgs& a) {
  const int64_t n0 = a.nm[0], f0 = a.nf[0], f1 = a.nf[1], f2 = a.nf[2];
  const int64_t cells = a.dim == 1 ? (axis_fits(a.nf[0], a.prec, 1) ? 0 : f0) : a.dim == 2 ? f1 * n0 : f2 * f1 * n0;
  return cells * a.n_trans * (a.prec == kF32 ? 8 : 16);
}

hipError_t fftn_plan_init(FftnPlan& fp, const DeconvArgs& a) {
  hipError_t e;
  int len[3] = {a.nf[0], a.nf[1], a.nf[2]}, n = a.dim;
  if (a.dim == 1 && !axis_fits(a.nf[0], a.prec, 1)) {
    fp.split = split_length(a.nf[0], a.prec);
    len[0] = fp.split;
    len[1] = a.nf[0] / fp.split;
    n = 2;
  }
  for (int d = 0; d < n; ++d) {
    fp.axis[d].n = len[d];
    fp.axis[d].radix = radices_of(len[d], a.prec, a.dim);
    e = a.prec == kF32 ? twiddle_table<float>(fp.axis[d].tw, len[d]) : twiddle_table<double>(fp.axis[d].tw, len[d]);
    if (e != hipSuccess) return e;
  }
  const int64_t bytes = fftn_mid_bytes(a);
  return bytes > 0 ? dev_malloc(&fp.mid, (size_t)bytes) : hipSuccess;
}

void fftn_plan_free(FftnPlan& fp) {
  for (FftnPlan::Axis& ax : fp.axis) {
    if (ax.tw) (void)hipFree(ax.tw);
    ax.tw = nullptr;
  }
  if (fp.mid) (void)hipFree(fp.mid);
  fp.mid = nullptr;
}

hipError_t fftn_to_modes(FftnPlan& fp, const DeconvArgs& a, void* grid, void* f, int isign, hipStream_t s) {
  return a.prec == kF32 ? fftn_run<float>(fp, a, false, grid, f, isign, s) : fftn_run<double>(fp, a, false, grid, f, isign, s);
}

hipError_t fftn_to_grid(FftnPlan& fp, const DeconvArgs& a, const void* f, void* grid, int isign, hipStream_t s) {
  return a.prec == kF32 ? fftn_run<float>(fp, a, true, f, grid, isign, s) : fftn_run<double>(fp, a, true, f, grid, isign, s);
}

}  // namespace nufftx
