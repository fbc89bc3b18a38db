// k_mixfft.hip -- the pruned FFT passes of k_fft.hip on grids that are not
// powers of two (Nt = 2 ceil(sigma N / 2) of an ordinary image size: 640, 300,
// 250, ...), with the deconvolution fused into the dimension-1 pass.
//
// Same passes and the same pruning as k_fft.hip (which lines are zero or
// discarded, which positions of a line are read or written); the line FFTs
// are Stockham passes in LDS whose radices come from a per-plan list
// (MixLine) instead of template parameters.  A pass branches once, on a
// uniform radix, to code for that radix; a thread holds all butterflies it
// owns (8 points, rounded up to whole butterflies) in registers between the
// reads and the writes of a pass, so that one LDS copy of the lines suffices.
// The first pass takes its points from global memory and the last one
// writes its results there.  Divisions are by multiply-high.
//
// What bounds it: HBM where the grid exceeds the caches (the LDS work of a
// line of 3 passes is about a third of its HBM time); the line latency on
// small images, hence few lines per workgroup there (mix_shape).
// The radices and the threads per line are those with the fewest exchanges
// and idle butterfly slots (best_threads); lines with a prime factor above 13
// keep rocFFT.
//
// Measured (us of the whole FFT stage with the deconvolution, forward /
// adjoint, against rocFFT with separate deconvolution): 300 x 288 x 250 FP32
// 129 / 119 against 495 / 477, 192^3 FP64 72 / 71 against 179 / 169, 640^2 FP64
// 23 / 22 against 37 / 36, 32 slices of 480^2 FP32 53 / 50 against 896 / 870.
// (Ordinary FP32 plans keep rocFFT in the forward direction: plan.cpp,
// mix_forward.)
//
// Lines of the strided passes are lpb consecutive x positions: every load and
// store row is a contiguous run of lpb elements.  Rows of a grid whose width
// is not a multiple of the cache line start anywhere in one, and neighbouring
// workgroups share the line at their border, so consecutive chunks go to one
// XCD (one L2).
#include <algorithm>

#include "fft_line.hpp"
#include "mixfft.hpp"

namespace nfftm {

namespace {

using namespace lf;

// (cos, sin)(2 pi k / N) at compile time: Taylor series after reduction to
// the first octant.
struct CS {
  double c, s;
};
constexpr CS octant(double x) {
  double c = 1.0, s = x, t = 1.0;
  for (int i = 1; i < 20; ++i) {
    t = t * x / i;
    if (i % 4 == 2) c -= t;
    if (i % 4 == 0) c += t;
    if (i % 4 == 3) s -= t;
    if (i % 4 == 1 && i > 1) s += t;
  }
  return CS{c, s};
}
constexpr CS unit_root(int k, int N) {
  k %= N;
  // angle = (q + f) quarter turns, 0 <= f < 1
  const int q = 4 * k / N, num = 4 * k - q * N;  // f = num / N
  constexpr double H = 1.57079632679489661923;
  CS a = 2 * num <= N ? octant(H * num / N) : CS{octant(H * (N - num) / N).s, octant(H * (N - num) / N).c};
  if (q == 0) return a;
  if (q == 1) return CS{-a.s, a.c};
  if (q == 2) return CS{-a.c, -a.s};
  return CS{a.s, -a.c};
}

// x * exp(-+2 pi i K / N)
template <typename R, int N, int K, bool INV, typename C>
__device__ __forceinline__ C croot(C x) {
  if constexpr (K % N == 0) {
    return x;
  } else {
    constexpr CS w = unit_root(K, N);
    return tmul<INV>(x, C{(R)w.c, (R)w.s});
  }
}

// DFT of an odd number of points: with a_j = v_j + v_{N-j}, b_j = v_j - v_{N-j},
// X_k and X_{N-k} = v_0 + sum_j a_j cos(2 pi j k / N) -+ i sum_j b_j sin(2 pi j k / N).
template <typename R, int N, int K, int J, typename C>
__device__ __forceinline__ void odd_terms(C* t, C* u, const C* a, const C* b) {
  if constexpr (J <= N / 2) {
    constexpr CS w = unit_root(J * K, N);
    const R c = (R)w.c, s = (R)w.s;
    t->x = fma(c, a[J - 1].x, t->x);
    t->y = fma(c, a[J - 1].y, t->y);
    u->x = fma(s, b[J - 1].x, u->x);
    u->y = fma(s, b[J - 1].y, u->y);
    odd_terms<R, N, K, J + 1>(t, u, a, b);
  }
}
template <typename R, int N, int K, bool INV, typename C>
__device__ __forceinline__ void odd_outputs(C* v, C v0, const C* a, const C* b) {
  if constexpr (K <= N / 2) {
    C t = v0, u = C{0, 0};
    odd_terms<R, N, K, 1>(&t, &u, a, b);
    const C iu = INV ? C{-u.y, u.x} : C{u.y, -u.x};
    v[K] = cadd(t, iu);
    v[N - K] = csub(t, iu);
    odd_outputs<R, N, K + 1, INV>(v, v0, a, b);
  }
}
template <typename R, int N, bool INV, typename C>
__device__ __forceinline__ void dft_odd(C* v) {
  C a[N / 2], b[N / 2];
  const C v0 = v[0];
#pragma unroll
  for (int j = 1; j <= N / 2; ++j) {
    a[j - 1] = cadd(v[j], v[N - j]);
    b[j - 1] = csub(v[j], v[N - j]);
  }
  C s = v0;
#pragma unroll
  for (int j = 0; j < N / 2; ++j) s = cadd(s, a[j]);
  v[0] = s;
  odd_outputs<R, N, 1, INV>(v, v0, a, b);
}

template <typename R, int N, bool INV, typename C>
__device__ __forceinline__ void mdft(C* v);

// DFT of A B points: B DFTs of A points over n = B a + b, twiddles
// W^(b k1), A DFTs of B points into k1 + A k2.
template <typename R, int A, int B, int IB, int K1, bool INV, typename C>
__device__ __forceinline__ void comp_twiddle(C* y) {
  if constexpr (K1 < A) {
    y[K1] = croot<R, A * B, IB * K1, INV>(y[K1]);
    comp_twiddle<R, A, B, IB, K1 + 1, INV>(y);
  }
}
template <typename R, int A, int B, int IB, bool INV, typename C>
__device__ __forceinline__ void comp_inner(const C* v, C (*y)[A]) {
  if constexpr (IB < B) {
#pragma unroll
    for (int a = 0; a < A; ++a) y[IB][a] = v[B * a + IB];
    mdft<R, A, INV>(y[IB]);
    comp_twiddle<R, A, B, IB, 1, INV>(y[IB]);
    comp_inner<R, A, B, IB + 1, INV>(v, y);
  }
}
template <typename R, int A, int B, bool INV, typename C>
__device__ __forceinline__ void dft_comp(C* v) {
  C y[B][A];
  comp_inner<R, A, B, 0, INV>(v, y);
#pragma unroll
  for (int k1 = 0; k1 < A; ++k1) {
    C z[B];
#pragma unroll
    for (int b = 0; b < B; ++b) z[b] = y[b][k1];
    mdft<R, B, INV>(z);
#pragma unroll
    for (int k2 = 0; k2 < B; ++k2) v[k1 + A * k2] = z[k2];
  }
}

template <typename R, int N, bool INV, typename C>
__device__ __forceinline__ void mdft(C* v) {
  if constexpr (N == 2 || N == 4 || N == 8 || N == 16) dft<R, N, INV>(v);
  else if constexpr (N % 2 == 1 && N != 9) dft_odd<R, N, INV>(v);
  else if constexpr (N == 9) dft_comp<R, 3, 3, INV>(v);
  else if constexpr (N == 12) dft_comp<R, 4, 3, INV>(v);
  else dft_comp<R, 2, N / 2, INV>(v);  // 6, 10
}

// LDS element of point i of line l: strided passes keep the lines of one
// point together (row stride lpb + 1), dimension-1 passes the points of one
// line (one pad element per 16 points), so that the power-of-two strides of
// the Stockham writes spread over the banks.
template <bool COL>
__device__ __forceinline__ int lds_at(const MixArgs& a, int l, int i) {
  if constexpr (COL) return i * (a.lpb + 1) + l;
  return l * (a.ln.L + (a.ln.L >> 4) + 1) + i + (i >> 4);
}

// The thread's line and first butterfly, and the threads per line: a thread
// works on one line throughout, on butterflies j0, j0 + tpl, ... of it;
// consecutive threads on consecutive lines (strided passes) or consecutive
// butterflies.
struct Own {
  int l, j0, tpl;
};
template <bool COL>
__device__ __forceinline__ Own own_of(const MixArgs& a) {
  Own o;
  o.tpl = a.ln.tpl;
  if constexpr (COL) {
    o.l = (int)threadIdx.x & (a.lpb - 1);
    o.j0 = (int)threadIdx.x >> a.lsh;
  } else {
    o.l = (int)fdiv(threadIdx.x, a.ln.dtpl);
    o.j0 = (int)threadIdx.x - o.l * o.tpl;
  }
  // threads past the last line own no butterfly
  if (o.l >= a.lpb || o.j0 >= o.tpl) o.l = 0, o.j0 = 1 << 20;
  return o;
}

// One pass of radix RAD.
template <typename R, int RAD, bool INV, bool COL, typename C, typename Ld, typename St>
__device__ __forceinline__ void mix_pass(const MixArgs& a, const Own& o, int ip, C* buf, const C* tw, Ld& load,
                                         St& store) {
  constexpr int NB = mix_butterflies(RAD);
  const MixPass q = a.ln.p[ip];
  const int M = q.M(), NS = q.NS();
  const FastDiv dNS = q.dNS();
  const bool last = ip == a.ln.npass - 1;
  C v[NB][RAD];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (b * o.tpl >= M) break;  // uniform
    const int j = o.j0 + b * o.tpl;
    const bool ok = j < M;
    const int jj = ok ? j : 0;
    if (ip == 0) {
#pragma unroll
      for (int u = 0; u < RAD; ++u) v[b][u] = load(jj + u * M, ok);
    } else {
#pragma unroll
      for (int u = 0; u < RAD; ++u) v[b][u] = buf[lds_at<COL>(a, o.l, jj + u * M)];
    }
  }
  if (ip > 0 && !last) __syncthreads();
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (b * o.tpl >= M) break;
    const int j = o.j0 + b * o.tpl;
    if (j < M) {
      const int jd = (int)fdiv((uint32_t)j, dNS), jm = j - jd * NS;
      if (ip > 0) {
        const int e = jm * q.ts();
#pragma unroll
        for (int u = 1; u < RAD; ++u) v[b][u] = tmul<INV>(v[b][u], tw[e * u]);
      }
      mdft<R, RAD, INV>(v[b]);
      const int i0 = jd * NS * RAD + jm;
      if (last) {
#pragma unroll
        for (int u = 0; u < RAD; ++u) store(i0 + u * NS, v[b][u]);
      } else {
#pragma unroll
        for (int u = 0; u < RAD; ++u) buf[lds_at<COL>(a, o.l, i0 + u * NS)] = v[b][u];
      }
    }
  }
  if (!last) __syncthreads();
}

// The FFT of the workgroup's lines: load(point, valid) gives the input of
// the thread's line, store(point, value) takes the output.
template <typename R, bool INV, bool COL, typename C, typename Ld, typename St>
__device__ __forceinline__ void mix_lines(const MixArgs& a, const Own& o, C* buf, const C* tw, Ld load, St store) {
  for (int ip = 0; ip < a.ln.npass; ++ip) {
    switch (a.ln.p[ip].r()) {
#define NFFTM_MR(RR) \
  case RR:           \
    mix_pass<R, RR, INV, COL>(a, o, ip, buf, tw, load, store); \
    break;
      NFFTM_MR(2) NFFTM_MR(3) NFFTM_MR(4) NFFTM_MR(5) NFFTM_MR(6) NFFTM_MR(7) NFFTM_MR(8) NFFTM_MR(9) NFFTM_MR(10)
      NFFTM_MR(11) NFFTM_MR(12) NFFTM_MR(13) NFFTM_MR(16)
#undef NFFTM_MR
    }
  }
}

template <typename R>
struct MixBlock {  // most threads of a workgroup (register budget of the radix code)
  static constexpr int NT = sizeof(R) == 4 ? 1024 : 512;
};

// Workgroup -> position in the pass, consecutive ones on one XCD; -1: none.
__device__ __forceinline__ int mix_id(int total) {
  const int per = (total + 7) >> 3;
  const int id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  return (int)(blockIdx.x >> 3) < per && id < total ? id : -1;
}

__device__ __forceinline__ size_t slice_start(const MixArgs& a) {
  return (size_t)slice_off(a.s0 + (int)blockIdx.y, a.Bsl, a.P);
}
__device__ __forceinline__ size_t slice_grid(const MixArgs& a) {
  return (size_t)(a.nsl - 1 - (int)blockIdx.y) * (size_t)a.Q;
}

// A line of the dimension-1 pass: whether there is one, its start in the
// grid and the product of its outer deconvolution factors.
struct XLine {
  bool ok;
  size_t g;
  double fac;
};
__device__ __forceinline__ XLine x_line(const MixArgs& a, int q) {
  XLine x;
  x.ok = q < a.nlines;
  const int qq = x.ok ? q : 0;
  const int iz = (int)fdiv((uint32_t)qq, a.dN1), iy = qq - iz * a.N1;
  x.g = (size_t)grid_pos(iz, a.N2, a.L2, a.Na2) * a.st2 + (size_t)grid_pos(iy, a.N1, a.L1, a.Na1) * a.st1;
  x.fac = 1.0;
  if (a.fac[1]) x.fac *= a.fac[1][iy];
  if (a.fac[2]) x.fac *= a.fac[2][iz];
  return x;
}

// Dimension 1, forward: f deconvolved into lines (y, z) in S_y x S_z.
template <typename R>
__global__ __launch_bounds__(MixBlock<R>::NT) void k_mix_x_fwd(MixArgs a, const typename cpx<R>::T* __restrict__ f,
                                                              typename cpx<R>::T* __restrict__ grid) {
  using C = typename cpx<R>::T;
  extern __shared__ __align__(16) char smem[];
  C* tw = (C*)smem;
  C* buf = tw + a.ln.L;
  const int id = mix_id(a.total);
  if (id < 0) return;
  for (int i = threadIdx.x; i < a.ln.L; i += blockDim.x) tw[i] = ((const C*)a.tw)[i];
  const Own o = own_of<false>(a);
  const int q = id * a.lpb + o.l;
  const XLine x = x_line(a, q);
  const C* img = f + slice_start(a) + (size_t)(x.ok ? q : 0) * a.N * a.ist;
  C* g = grid + slice_grid(a) + x.g;
  const double fr = x.fac * a.oscale;
  mix_lines<R, false, false>(
      a, o, buf, tw,
      [&](int i, bool ok) {
        const int ix = image_idx(i, a.N, a.ln.L, a.Na);
        C v{0, 0};
        if (ok && x.ok && ix >= 0) {
          const double s = a.fac[0][ix] * fr;
          v = img[(size_t)(unsigned)ix * (unsigned)a.ist];
          v = C{(R)((double)v.x * s), (R)((double)v.y * s)};
        }
        return v;
      },
      [&](int i, C v) {
        if (x.ok) g[i] = v;
      });
}

// Dimension 1, adjoint: lines (y, z) in S_y x S_z to the image, transposed
// deconvolution fused.
template <typename R>
__global__ __launch_bounds__(MixBlock<R>::NT) void k_mix_x_adj(MixArgs a, const typename cpx<R>::T* __restrict__ grid,
                                                              typename cpx<R>::T* __restrict__ f) {
  using C = typename cpx<R>::T;
  extern __shared__ __align__(16) char smem[];
  C* tw = (C*)smem;
  C* buf = tw + a.ln.L;
  const int id = mix_id(a.total);
  if (id < 0) return;
  for (int i = threadIdx.x; i < a.ln.L; i += blockDim.x) tw[i] = ((const C*)a.tw)[i];
  const Own o = own_of<false>(a);
  const int q = id * a.lpb + o.l;
  const XLine x = x_line(a, q);
  C* img = f + slice_start(a) + (size_t)(x.ok ? q : 0) * a.N * a.ist;
  const C* g = grid + slice_grid(a) + x.g;
  const double fr = x.fac * a.oscale;
  mix_lines<R, true, false>(
      a, o, buf, tw,
      [&](int i, bool ok) {
        C v{0, 0};
        if (ok && x.ok) v = g[i];
        return v;
      },
      [&](int i, C v) {
        const int ix = image_idx(i, a.N, a.ln.L, a.Na);
        if (x.ok && ix >= 0) {
          const double s = a.fac[0][ix] * fr;
          img[(size_t)(unsigned)ix * (unsigned)a.ist] = C{(R)((double)v.x * s), (R)((double)v.y * s)};
        }
      });
}

// Strided pass along dimension 2 or 3, in place: forward reads only the
// image positions of a line (the rest is zero), adjoint writes only those.
// Grid offsets fit 32 bits (grids of less than 2^31 points).
template <typename R, bool INV>
__global__ __launch_bounds__(MixBlock<R>::NT) void k_mix_col(MixArgs a, typename cpx<R>::T* __restrict__ grid) {
  using C = typename cpx<R>::T;
  extern __shared__ __align__(16) char smem[];
  C* tw = (C*)smem;
  C* buf = tw + a.ln.L;
  const int id = mix_id(a.total);
  if (id < 0) return;
  for (int i = threadIdx.x; i < a.ln.L; i += blockDim.x) tw[i] = ((const C*)a.tw)[i];
  const Own o = own_of<true>(a);
  const int c = (int)fdiv((uint32_t)id, a.dchunk), x = (id - c * a.nchunk) * a.lpb + o.l;
  const int gc = a.oall ? c : grid_pos(c, a.oN, a.oL, a.oNa);
  const bool xin = x < a.nx;
  C* g = grid + slice_grid(a) + (size_t)gc * a.ost + (xin ? x : 0);
  const unsigned st = (unsigned)a.st;
  mix_lines<R, INV, true>(
      a, o, buf, tw,
      [&](int i, bool ok) {
        C v{0, 0};
        if (ok && xin && (INV || image_idx(i, a.N, a.ln.L, a.Na) >= 0)) v = g[(unsigned)i * st];
        return v;
      },
      [&](int i, C v) {
        if (xin && (!INV || image_idx(i, a.N, a.ln.L, a.Na) >= 0)) g[(unsigned)i * st] = v;
      });
}

// The strided pass of the last dimension in both directions with a product
// between (the Toeplitz embedding: FFT, eigenvalues, inverse FFT): the line
// stays in LDS, where separate passes would write, multiply and read the grid
// once more each.  The transformed line goes to a second LDS area, since other
// threads still read the first one.
template <typename R>
__global__ __launch_bounds__(MixBlock<R>::NT) void k_mix_mul(MixArgs a, typename cpx<R>::T* __restrict__ grid) {
  using C = typename cpx<R>::T;
  extern __shared__ __align__(16) char smem[];
  C* tw = (C*)smem;
  C* buf = tw + a.ln.L;
  C* res = buf + a.ln.L * (a.lpb + 1);
  const int id = mix_id(a.total);
  if (id < 0) return;
  for (int i = threadIdx.x; i < a.ln.L; i += blockDim.x) tw[i] = ((const C*)a.tw)[i];
  const Own o = own_of<true>(a);
  const int c = (int)fdiv((uint32_t)id, a.dchunk), x = (id - c * a.nchunk) * a.lpb + o.l;
  const bool xin = x < a.nx;
  const size_t base = (size_t)(a.oall ? c : grid_pos(c, a.oN, a.oL, a.oNa)) * a.ost + (xin ? x : 0);
  C* g = grid + base;
  const C* lam = (const C*)a.lam + base;
  const unsigned st = (unsigned)a.st;
  mix_lines<R, false, true>(
      a, o, buf, tw,
      [&](int i, bool ok) {
        C v{0, 0};
        if (ok && xin && image_idx(i, a.N, a.ln.L, a.Na) >= 0) v = g[(unsigned)i * st];
        return v;
      },
      [&](int i, C v) {
        C f{0, 0};
        if (xin) f = lam[(unsigned)i * st];
        res[lds_at<true>(a, o.l, i)] = C{v.x * f.x - v.y * f.y, v.x * f.y + v.y * f.x};
      });
  __syncthreads();
  mix_lines<R, true, true>(
      a, o, buf, tw, [&](int i, bool) { return res[lds_at<true>(a, o.l, i)]; },
      [&](int i, C v) {
        if (xin && image_idx(i, a.N, a.ln.L, a.Na) >= 0) g[(unsigned)i * st] = v;
      });
}

inline int mix_threads(const MixArgs& a) { return (a.lpb * a.ln.tpl + 63) / 64 * 64; }

template <typename R>
hipError_t x_go(bool fwd, const MixArgs& a, hipStream_t s, const void* in, void* out) {
  using C = typename cpx<R>::T;
  const size_t lds = mix_lds_bytes(sizeof(R) == 8, false, a.ln, a.lpb);
  const dim3 g((unsigned)(8 * ((a.total + 7) / 8)), (unsigned)a.nsl), b((unsigned)mix_threads(a));
  auto k = fwd ? k_mix_x_fwd<R> : k_mix_x_adj<R>;
  if (lds > 65536 &&
      hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(k, g, b, lds, s, a, (const C*)in, (C*)out);
  return hipGetLastError();
}

template <typename R>
hipError_t col_go(bool fwd, const MixArgs& a, hipStream_t s, void* grid) {
  using C = typename cpx<R>::T;
  const size_t lds = mix_lds_bytes(sizeof(R) == 8, true, a.ln, a.lpb);
  const dim3 g((unsigned)(8 * ((a.total + 7) / 8)), (unsigned)a.nsl), b((unsigned)mix_threads(a));
  auto k = fwd ? k_mix_col<R, false> : k_mix_col<R, true>;
  if (lds > 65536 &&
      hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(k, g, b, lds, s, a, (C*)grid);
  return hipGetLastError();
}

constexpr int RADICES[] = {16, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// Time of one thread's butterfly of radix r in units of one LDS exchange of a
// point: its exchanges, twiddles and additions.
double butterfly_cost(int r) {
  double c = 2.0 * r;
  for (int n = r; n > 1;) {
    int p = 2;
    while (n % p) ++p;
    c += 0.12 * r * p;
    n /= p;
  }
  return c;
}

// Threads per line for the radices r[0 .. n) of a line of L points: the
// fewest idle butterfly slots, at most mix_butterflies(r) per thread.
// Returns the cost per point.
double best_threads(int L, const int* r, int n, int most, int* tpl) {
  int lo = 1;
  for (int i = 0; i < n; ++i) {
    const int cap = mix_butterflies(r[i]);
    lo = std::max(lo, (L / r[i] + cap - 1) / cap);
  }
  double best = 1e30;
  for (int t = lo; t <= std::min(most, std::max(lo, L / 4)); ++t) {
    double c = 0;
    for (int i = 0; i < n; ++i) c += (double)((L / r[i] + t - 1) / t) * t * butterfly_cost(r[i]) / L + 1.0;
    if (c < best) {
      best = c;
      *tpl = t;
    }
  }
  return best;
}

// The radices of a line of L points: least cost.
struct Search {
  int L, most, rmax;
  int cur[MIX_PASSES], best[MIX_PASSES], nb, tpl;
  double cost;
  void go(int n, int nc) {
    if (n == 1) {
      int t = 0;
      const double c = best_threads(L, cur, nc, most, &t);
      if (c < cost) {
        cost = c;
        nb = nc;
        tpl = t;
        std::copy(cur, cur + nc, best);
      }
      return;
    }
    if (nc >= MIX_PASSES) return;
    for (int r : RADICES)
      if (n % r == 0 && r <= (nc == 0 ? rmax : cur[nc - 1])) {
        cur[nc] = r;
        go(n / r, nc + 1);
      }
  }
};

// most threads and points of a workgroup
constexpr int max_threads(bool dbl) { return dbl ? 512 : 1024; }
constexpr int max_points(bool dbl) { return dbl ? 8192 : 16384; }

}  // namespace

bool mix_factor(int64_t L, bool dbl, bool only, MixLine* ln, int rmax) {
  // the strided passes want rows of at least 32 bytes within the LDS
  if (L < 16 || L % 2 || L > (only ? max_points(dbl) / 2 : 2048)) return false;
  Search se;
  se.L = (int)L;
  se.rmax = rmax;
  se.most = max_threads(dbl) / (only ? 1 : dbl ? 2 : 4);
  se.cost = 1e30;
  se.go(se.L, 0);
  if (se.cost > 1e29) return false;
  ln->L = (int)L;
  ln->npass = se.nb;
  ln->tpl = se.tpl;
  ln->dtpl = make_fastdiv((uint32_t)se.tpl);
  int ns = 1;
  for (int i = 0; i < ln->npass; ++i) {
    const int r = se.best[i];
    const FastDiv d = make_fastdiv((uint32_t)ns);
    ln->p[i].r_sh_ns = (uint32_t)r | d.shift << 8 | (uint32_t)ns << 16;
    ln->p[i].m_ts = (uint32_t)(L / r) | (uint32_t)(L / (ns * r)) << 16;
    ln->p[i].mul = d.mul;
    ns *= r;
  }
  return true;
}

int mix_shape(bool dbl, bool col, const MixLine& ln, long long lines, long long outer) {
  // Strided passes: rows of 8 lines (64 bytes in FP32; 4, 16 and 32 lines
  // took 6-20 % longer on 300 x 288 x 250, the same in FP64 on 192^3).
  // Dimension 1: about 2048 points (1024 and 4096: up to 30 % longer).  More
  // lines where that leaves a workgroup small, fewer where there are not
  // lines enough for two workgroups per CU.
  const int mp = max_points(dbl), least = col ? (dbl ? 2 : 4) : 1;
  int l = col ? 8 : 1;
  while (l * 2 * ln.L <= 2048) l *= 2;
  while (l > least && (l * ln.tpl > max_threads(dbl) || l * ln.L > mp || mix_lds_bytes(dbl, col, ln, l) > 163840 ||
                       (lines + l - 1) / l * outer < 512))
    l /= 2;
  return l;
}

size_t mix_lds_bytes(bool dbl, bool col, const MixLine& ln, int lpb) {
  const size_t L = (size_t)ln.L;
  const size_t n = L + (col ? L * (lpb + 1) : (size_t)lpb * (L + (L >> 4) + 1));
  return n * (dbl ? 16 : 8);
}

size_t mix_mul_lds_bytes(bool dbl, const MixLine& ln, int lpb) {
  return mix_lds_bytes(dbl, true, ln, lpb) + (size_t)ln.L * (lpb + 1) * (dbl ? 16 : 8);
}

template <typename R>
static hipError_t mul_go(const MixArgs& a, hipStream_t s, void* grid) {
  const size_t lds = mix_mul_lds_bytes(sizeof(R) == 8, a.ln, a.lpb);
  auto k = k_mix_mul<R>;
  if (lds > 65536 &&
      hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(k, dim3((unsigned)(8 * ((a.total + 7) / 8))), dim3((unsigned)mix_threads(a)), lds, s, a,
                     (typename cpx<R>::T*)grid);
  return hipGetLastError();
}

hipError_t launch_mix_mul(bool dbl, const MixArgs& a, hipStream_t s, void* grid) {
  return dbl ? mul_go<double>(a, s, grid) : mul_go<float>(a, s, grid);
}

hipError_t launch_mix_x(bool dbl, bool fwd, const MixArgs& a, hipStream_t s, const void* in, void* out) {
  return dbl ? x_go<double>(fwd, a, s, in, out) : x_go<float>(fwd, a, s, in, out);
}

hipError_t launch_mix_col(bool dbl, bool fwd, const MixArgs& a, hipStream_t s, void* grid) {
  return dbl ? col_go<double>(fwd, a, s, grid) : col_go<float>(fwd, a, s, grid);
}

}  // namespace nfftm
