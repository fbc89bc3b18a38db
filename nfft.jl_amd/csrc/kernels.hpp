// kernels.hpp -- device code of the gfx950 NFFT gridding path.
//
// Spreading (convolve_transpose!, src/convolution.jl:115-149) and
// interpolation (convolve!, src/convolution.jl:20-45) over nodes that the host
// has bin-sorted into tiles of the oversampled grid.  One workgroup owns one
// work item = (tile, contiguous range of that tile's nodes).  The tile plus
// its stencil halo ("padded tile", extent T + 2m - 1 per dimension) lives in
// LDS:
//   * spreading accumulates every node's (2m)^D footprint into the padded tile
//     with LDS atomics, then writes the padded tile with plain coalesced
//     stores to a per-item scratch slot; a fold kernel then sums the (at most
//     2^D, or 3^D for narrow tiles) padded tiles covering each grid point and
//     writes every grid point once.  FP32 accumulates packed 32+32-bit
//     fixed-point (re, im) pairs with one 64-bit integer LDS add per tap (on
//     gfx950 the FP32 LDS float add costs ~40x an integer add); the scale is a
//     power of two per work item from the strict bound sum_j |f_j| max(w)^D,
//     so sums are exact integers, independent of order.  FP64 accumulates
//     with the FP64 LDS add.
//   * interpolation stages the padded tile from HBM once, then gathers every
//     node's footprint from LDS.
// Per node and dimension the FP64 index reduction of the reference
// (src/precomputation.jl:524-554) gives the cell and the window argument; the
// 2m window values come from the LINEAR table (src/precomputation.jl:179-201),
// the polynomial of TENSOR/POLYNOMIAL (src/precomputation.jl:215-222,
// 556-591) or the exact Kaiser-Bessel window of FULL
// (src/windowFunctions.jl:21-34).
//
// Lane layout (64-wide wavefronts):
//   D = 3: one node per wavefront step, lane = (lx, ly) of the footprint, each
//          lane walks lz.  With row stride Sx = 8 (mod 16) the 64 lanes of a
//          W = 8 footprint hit 64 distinct LDS banks.
//   D = 2: Wp = pow2ceil(2m) lanes per node (lx), 64/Wp nodes per step, each
//          lane walks ly.
//   D = 1: Wp lanes per node, one tap per lane.
// Interpolation reduces per-lane partial sums with DPP row operations.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace nfftm {

constexpr int MAXD = 8;
enum { WIN_LINEAR = 0, WIN_POLY = 1, WIN_EXACT = 2 };

template <typename R>
struct cpx;
template <>
struct cpx<float> {
  using T = float2;
};
template <>
struct cpx<double> {
  using T = double2;
};

// Division of non-negative 32-bit integers (< 2^31) by a fixed divisor via a
// multiply-high (Granlund & Montgomery 1994, fig. 4.1).
struct FastDiv {
  uint32_t d, mul, shift;
};

__host__ inline FastDiv make_fastdiv(uint32_t d) {
  FastDiv f;
  f.d = d;
  uint32_t l = 0;
  while ((1ull << l) < d) ++l;
  f.shift = l;
  f.mul = (uint32_t)((((1ull << l) - d) << 32) / d + 1);
  return f;
}

__device__ __forceinline__ uint32_t fdiv(uint32_t x, const FastDiv& f) {
  return (__umulhi(x, f.mul) + x) >> f.shift;
}

struct KArgs {
  int D, m, W, mode;
  int M;                 // number of nodes
  long long fst;         // element stride of the node values (directional plans: the product of the
                         // sizes of the axes before the transformed ones; otherwise 1)
  int Nt[MAXD];          // oversampled grid size per dim
  double Ntd[MAXD];
  long long gstr[MAXD];  // grid strides (dim 1 fastest)
  // tiling (D <= 3)
  int T[3];        // tile extent per dim
  int ntiles[3];   // tiles per dim
  int Pd[3];       // padded extent T + W - 1
  int Sx, Sxy;     // LDS strides of the padded tile (elements)
  int tileElems;   // elements of one LDS plane
  int padCells;    // Pd[0]*Pd[1]*Pd[2]
  FastDiv divP0, divT0;
  // window
  const void* lut;  // R[LUTSize + 2]
  long long scale;  // LUTSize / m, a power of two
  const void* poly; // R[(2m+1) * 2m], column l holds coefficients of tap l
  const double* polyd;  // the same coefficients in FP64 (node gradient)
  double b;         // Kaiser-Bessel shape pi*(2 - 1/sigma)
  int win;          // window id (NFFTM_KAISER_BESSEL .. NFFTM_COSH_TYPE) of the exact (FULL) mode
  double wscale;    // power-of-two window normalisation
  double oscale;    // output scale: 1 inside a transform; wscale^-D for the
                    // standalone convolve!/convolve_transpose! entry points
  // nodes
  const double* ks;   // ks[d * M + j], shifted into [0, 1)
  const int* perm;    // sorted position -> caller's node index
  void* fsort;        // interpolation results in sorted order (D = 1 polynomial
                      // kernels; null: stored at the caller's positions)
  const int4* items;  // {tile, begin, end, 0}
  int nitems;
  const char* rec;    // node records in sorted order (NodeRec layout), tiled plans
  int recBytes;
  int blocked3;       // 3-D scratch slots stored as 27 halo/interior blocks (1: whole tiles, 2: some
                      // partial); 2-D: every grid point is covered by its own tile and neighbouring
                      // ones only (k_fold2)
  int tvar;           // 3-D tile geometry variant (compile-time tile edge)
  int fix2;           // FP32 2-D spreading accumulates packed fixed point (one
                      // 64-bit LDS atomic per tap) instead of two FP64 planes
  // spreading
  double wmaxD;        // bound of any product of D window values
  void* scratch;       // nitems padded tiles (dense, px fastest)
  const int* tstart;   // items of tile t: [tstart[t], tstart[t+1])
  int ntile_all;       // product of ntiles
  // slices s0 .. s0 + nsl - 1 of a directional plan in one launch (1-D and 2-D
  // tile kernels and their fold; otherwise s0 = 0, nsl = 1): the node values
  // of slice s start at element s % Bsl + (s / Bsl) Bsl M, its grid is slot
  // nsl - 1 - (s - s0) of consecutive grids of Q points (the last slice in
  // slot 0, the plan's grid), its scratch slots follow those of s - 1
  int s0, nsl;
  long long Bsl, Q;
  // density compensation on 2-D tiled plans, fused (null otherwise): k_fold2
  // divides the grid by gdiv[0]; interpolation, instead of storing its
  // result, divides the real weights wdiv of the nodes by its real part over
  // gdiv[0] and flags results that are not positive
  const double* gdiv;
  void* wdiv;
  int* wbad;
};

// (Bsl < 2^31; slice 0, the only one of an ordinary plan, needs no division)
__host__ __device__ __forceinline__ long long slice_off(int s, long long Bsl, long long len) {
  if (s == 0) return 0;
  const unsigned q = (unsigned)s / (unsigned)Bsl;
  return (long long)((unsigned)s - q * (unsigned)Bsl) + (long long)q * Bsl * len;
}
// i = the launch's slice index (a block index)
__device__ __forceinline__ long long slice_nodes(const KArgs& a, int i) { return slice_off(a.s0 + i, a.Bsl, a.M); }
__device__ __forceinline__ size_t slice_slot(const KArgs& a, int i) {
  return (size_t)(a.nsl - 1 - i) * (size_t)a.Q;
}
__device__ __forceinline__ size_t slice_scratch(const KArgs& a, int i) {
  return (size_t)i * (size_t)a.nitems * (size_t)a.padCells;
}

// k * Ntilde rounded to FP64 before any further use, as the reference
// computes kscale (src/precomputation.jl:538): kept out of a fused multiply-add
// with the following subtraction, which at Ntilde ~ 2e7 would move the window
// argument by ~1e-9 grid units.
__device__ __forceinline__ double scaled_node(double ksv, double Ntd) {
#pragma clang fp contract(off)
  return ksv * Ntd;
}

// Window values of one node along dimension d.  Returns the wrapped cell
// floor(k * Ntilde) (in [0, Ntilde)); t = kscale - off with
// off = cell - m + 1 exactly as src/precomputation.jl:537-545.
// I0 by its positive power series, to the precision of R.
template <typename R>
__device__ __forceinline__ R i0_dev(R x) {
  const R y = (R)0.25 * x * x;
  R t = 1, s = 1;
  for (int k = 1; k < 200 && t > (sizeof(R) == 4 ? (R)1e-8 : (R)1e-17) * s; ++k) {
    t = t * y / (R)(k * k);
    s += t;
  }
  return s;
}

// Exact window psi(u), u in grid units, of window a.win (src/windowFunctions.jl:
// 21-134): Kaiser-Bessel, Gaussian, cardinal B-spline of order W = 2m
// (Cox-de Boor), reversed Kaiser-Bessel, cosh type.
template <typename R, int W>
__device__ __forceinline__ R window_exact(const KArgs& a, R u) {
  const R m = (R)a.m, b = (R)a.b, au = u < 0 ? -u : u;
  switch (a.win) {
    case 1: {  // gauss, b_g = m / pi
      const R bg = m / (R)M_PI;
      return au < m ? exp(-u * u / bg) / sqrt((R)M_PI * bg) : (R)0;
    }
    case 2: {  // spline: M_W(u + m)
      if (!(au < m)) return 0;
      const R x = u + m;
      R v[W];
#pragma unroll
      for (int s = 0; s < W; ++s) v[s] = (x - (R)s >= 0 && x - (R)s < 1) ? (R)1 : (R)0;
#pragma unroll
      for (int k = 2; k <= W; ++k) {
#pragma unroll
        for (int s = 0; s + k <= W; ++s) v[s] = ((x - (R)s) * v[s] + ((R)k - (x - (R)s)) * v[s + 1]) / (R)(k - 1);
      }
      return v[0];
    }
    case 3: {  // kaiser_bessel_rev
      if (!(au < m)) return 0;
      const R r = u / m;
      return (R)0.5 / m * i0_dev<R>(m * b * sqrt((R)1 - r * r));
    }
    case 4: {  // cosh_type, beta = m b
      if (!(au < m)) return 0;
      const R r = u / m, al = sqrt((R)1 - r * r), beta = m * b;
      return (cosh(beta * al) - (R)1) / ((cosh(beta) - (R)1) * al);
    }
    default: {  // kaiser_bessel
      if (au < m) {
        const R arg = sqrt(m * m - u * u);
        return sinh(b * arg) / (arg * (R)M_PI);
      }
      return au > m ? (R)0 : b / (R)M_PI;
    }
  }
}

// The 2m fitted window polynomials at x = t - m + 1/2 (evalpoly per tap,
// src/precomputation.jl:203-218): column l of P holds the 2m + 1 coefficients
// of tap l, lowest degree first; Horner in the data precision.
template <typename R, int W, typename PT = const R*>
__device__ __forceinline__ void poly_taps(PT P, R x, R* w) {
  constexpr int NC = W + 1;
#pragma unroll
  for (int l = 0; l < W; ++l) {
    R s = P[l * NC + NC - 1];
#pragma unroll
    for (int i = NC - 2; i >= 0; --i) s = fma(x, s, P[l * NC + i]);
    w[l] = s;
  }
}

template <typename R, int W>
__device__ __forceinline__ int node_weights(const KArgs& a, int d, double ksv, R* w) {
  const double kscale = scaled_node(ksv, a.Ntd[d]);
  const long long c = (long long)kscale;  // unsafe_trunc, kscale >= 0
  const long long off = c - a.m + 1;
  const double t = kscale - (double)off;  // in [m-1, m), exact
  if (a.mode == WIN_LINEAR) {
    const R* lut = (const R*)a.lut;
    const double idx = t * (double)a.scale;  // (kscale - off) * (LUTSize / m)
    const long long ii = (long long)floor(idx);
    const R alpha = (R)(idx - (double)ii);
#pragma unroll
    for (int l = 0; l < W; ++l) {
      long long v = ii - (long long)l * a.scale;
      long long i1 = v < 0 ? -v : v;
      long long i2 = (v + 1) < 0 ? -(v + 1) : (v + 1);
      R y1 = lut[i1], y2 = lut[i2];
      w[l] = y1 + alpha * (y2 - y1);
    }
  } else if (a.mode == WIN_POLY) {
    poly_taps<R, W>((const R*)a.poly, (R)(t - (double)a.m + 1.0 - 0.5), w);
  } else {
#pragma unroll
    for (int l = 0; l < W; ++l) w[l] = window_exact<R, W>(a, (R)(t - (double)l)) * (R)a.wscale;
  }
  return (int)(c >= a.Nt[d] ? c - a.Nt[d] : c);
}

__device__ __forceinline__ long long wrapidx(long long x, long long n) {
  while (x < 0) x += n;
  while (x >= n) x -= n;
  return x;
}

// Workgroup -> work item, XCD-aware: the dispatcher deals workgroups to the 8
// XCDs round-robin, so consecutive items (neighbouring tiles sharing halo
// lines) are given to the same XCD and its L2.
__device__ __forceinline__ int xcd_item(int nitems) {
  const int per = (nitems + 7) >> 3;
  return (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
}

// ---------------------------------------------------------------------------
// DPP reductions (all 64 lanes must be active)
// ---------------------------------------------------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  int2 u = *reinterpret_cast<int2*>(&v);
  u.x = __builtin_amdgcn_update_dpp(0, u.x, CTRL, 0xF, 0xF, false);
  u.y = __builtin_amdgcn_update_dpp(0, u.y, CTRL, 0xF, 0xF, false);
  return *reinterpret_cast<double*>(&u);
}
// DPP move restricted to the rows of ROWMASK (other lanes read 0).
template <int CTRL, int ROWMASK>
__device__ __forceinline__ float dpp_rows(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWMASK, 0xF, false));
}
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_rows(double v) {
  int2 u = *reinterpret_cast<int2*>(&v);
  u.x = __builtin_amdgcn_update_dpp(0, u.x, CTRL, ROWMASK, 0xF, false);
  u.y = __builtin_amdgcn_update_dpp(0, u.y, CTRL, ROWMASK, 0xF, false);
  return *reinterpret_cast<double*>(&u);
}
// Lane L of each aligned group of G lanes (2, 4, 8 or 16; L < G), in all lanes of
// the group: quad permutation, or a broadcast within rows of 16 (in two halves
// for G = 8).
template <int G, int L>
__device__ __forceinline__ int group_lane(int v) {
  if constexpr (G <= 4) {
    constexpr int q = G == 4 ? L * 0x55 : L * 0x55 + 0xA0;  // quad_perm(L, L, L, L) or (L, L, 2 + L, 2 + L)
    return __builtin_amdgcn_update_dpp(0, v, q, 0xF, 0xF, false);
  } else {
    const int u = __builtin_amdgcn_update_dpp(0, v, 0x150 + L, 0xF, 0xF, false);  // row_newbcast
    if constexpr (G == 16) return u;
    return __builtin_amdgcn_update_dpp(u, v, 0x150 + (L + 8) % 16, 0xF, 0xC, false);
  }
}
template <int G, int L>
__device__ __forceinline__ float group_lane(float v) {
  return __int_as_float(group_lane<G, L>(__float_as_int(v)));
}
template <int G, int L>
__device__ __forceinline__ double group_lane(double v) {
  return __hiloint2double(group_lane<G, L>(__double2hiint(v)), group_lane<G, L>(__double2loint(v)));
}
__device__ __forceinline__ float readlane(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double readlane(double v, int l) {
  int2 u = *reinterpret_cast<int2*>(&v);
  u.x = __builtin_amdgcn_readlane(u.x, l);
  u.y = __builtin_amdgcn_readlane(u.y, l);
  return *reinterpret_cast<double*>(&u);
}

// Sum over aligned groups of G lanes (G in 1,2,4,8,16,64); every lane of the
// group ends with the group sum.
template <int G, typename R>
__device__ __forceinline__ R group_sum(R v) {
  if (G >= 2) v += dpp<0xB1>(v);   // quad_perm(1,0,3,2)
  if (G >= 4) v += dpp<0x4E>(v);   // quad_perm(2,3,0,1)
  if (G >= 8) v += dpp<0x141>(v);  // row_half_mirror
  if (G >= 16) v += dpp<0x140>(v); // row_mirror
  if (G == 64) v = readlane(v, 0) + readlane(v, 16) + readlane(v, 32) + readlane(v, 48);
  return v;
}

template <int W>
struct LanesPerNode {
  static constexpr int value = W <= 2 ? 2 : W <= 4 ? 4 : W <= 8 ? 8 : 16;
};

template <typename R>
__device__ __forceinline__ void lds_add(R* p, R v) {
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <typename R>
__device__ __forceinline__ void gbl_add(R* p, R v) {
  unsafeAtomicAdd(p, v);
}

// ---------------------------------------------------------------------------
// Node records and the LDS layout of the tile kernels
// ---------------------------------------------------------------------------
// Node record, one per node in tile order, built once per node set: the
// window weights of every dimension (D x W values of R), the node's cell
// relative to its tile origin (D <= 2: packed in 32 / D bits per dimension;
// D = 3: the LDS element index x + Sx y + Sxy z of that cell in the padded
// tile), and the caller's index of the node.  16-byte aligned for block
// copies.
template <typename R, int D, int W>
struct NodeRec {
  static constexpr int WBYTES = D * W * (int)sizeof(R);
  static constexpr int BYTES = (WBYTES + 8 + 15) & ~15;
  static constexpr int LOCBITS = 32 / D;
};
__host__ inline int node_rec_bytes(int D, size_t sizeofR, int W) {
  return (int)((D * W * sizeofR + 8 + 15) & ~(size_t)15);
}

// LDS layout of the D <= 2 tile kernels: the tile (spreading: FP64 planes or
// packed fixed point, in both precisions at most two doubles per cell), then
// the node values of one batch (spreading).
constexpr int NBV = 512;  // node values of a batch at most
__host__ __device__ __forceinline__ size_t tile_fv_off(int tileElems) {
  return (2 * (size_t)tileElems * sizeof(double) + 15) & ~(size_t)15;
}
__host__ inline size_t tile_layout_bytes(size_t sizeofR, int tileElems) {
  return tile_fv_off(tileElems) + NBV * 2 * sizeofR;
}

// Nodes of one 3-D work item at most (items are chunks of one tile's nodes).
constexpr int ITEM3 = 1024;

__device__ __forceinline__ void tile_origin(const KArgs& a, int D, int tile, int* t0) {
  int r = tile;
  for (int d = 0; d < D; ++d) {
    int td = r % a.ntiles[d];
    r /= a.ntiles[d];
    t0[d] = td * a.T[d];
  }
}

// Node records, one thread per node in sorted order: weights from
// node_weights, the cell relative to the origin of the node's tile, the
// caller's index; assembled in registers and stored as 16-byte words (4-byte
// stores at the record stride, one workgroup per work item: 32 us for 2 10^5
// nodes of a 2-D FP32 plan).
template <typename R, int D, int W>
__global__ __launch_bounds__(256) void k_node_records(KArgs a, char* __restrict__ rec) {
  using N = NodeRec<R, D, W>;
  const long long j = (long long)blockIdx.x * 256 + threadIdx.x;
  if (j >= a.M) return;
  unsigned u[N::BYTES / 4];
#pragma unroll
  for (int i = N::WBYTES / 4; i < N::BYTES / 4; ++i) u[i] = 0;
  unsigned pk = 0;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    R wd[W];
    const int cw = node_weights<R, W>(a, d, a.ks[(size_t)d * a.M + j], wd);
#pragma unroll
    for (int l = 0; l < W; ++l) {
      if constexpr (sizeof(R) == 4) {
        u[d * W + l] = __float_as_uint(wd[l]);
      } else {
        u[2 * (d * W + l)] = (unsigned)__double2loint(wd[l]);
        u[2 * (d * W + l) + 1] = (unsigned)__double2hiint(wd[l]);
      }
    }
    const unsigned loc = (unsigned)cw % (unsigned)a.T[d];
    if (D == 3) pk += loc * (unsigned)(d == 0 ? 1 : d == 1 ? a.Sx : a.Sxy);
    else pk |= loc << (N::LOCBITS * d);
  }
  u[N::WBYTES / 4] = pk;
  u[N::WBYTES / 4 + 1] = (unsigned)a.perm[j];
  uint4* out = (uint4*)(rec + (size_t)j * N::BYTES);
#pragma unroll
  for (int i = 0; i < N::BYTES / 16; ++i) out[i] = make_uint4(u[4 * i], u[4 * i + 1], u[4 * i + 2], u[4 * i + 3]);
}

// The record of one node as a lane of its group holds it (D <= 2): the
// dimension-1 weight of the lane's column, the dimension-2 weights, the packed
// cell and the caller's index.  Read straight from global memory, one step
// ahead of its use: the lanes of a group read the same words, a wavefront's
// groups consecutive records.  (Copying the records through LDS took a block
// copy, a barrier and, per node, as many LDS reads as the taps have adds; two
// or four steps ahead: more registers, the same or a longer time.)
// OWN (interpolation with more than 32 bytes of dimension-2 weights): one of
// them per lane, passed round the group (group_lane), where all W in every lane
// bound crowded tiles by the loads: 256^2, 16 nodes per pixel, us of
// interpolation, FP64 m = 3 43 -> 40, m = 5 88 -> 77, FP32 m = 5 49 -> 47
// (records through LDS: 39, 76, 47).  FP32 m = 4 is no faster by it alone and
// slower in a batch (165 -> 176).
template <typename R, int D, int W, bool OWN = false>
struct NodeTaps {
  static constexpr int N2 = D == 2 && !OWN ? W : 1;
  R w1, w2[N2];
  unsigned pk;
  int pj;
  __device__ __forceinline__ void load(const char* __restrict__ rec, long long j, int lx) {
    using N = NodeRec<R, D, W>;
    const char* r = rec + (size_t)j * N::BYTES;
    w1 = ((const R*)r)[lx];
    if constexpr (D == 2) {
#pragma unroll
      for (int l = 0; l < N2; ++l) w2[l] = ((const R*)r)[W + (OWN ? lx : l)];
    }
    const int2 q = *(const int2*)(r + N::WBYTES);
    pk = (unsigned)q.x;
    pj = q.y;
  }
};

// Taps of one column of a node's footprint: rows L .. W - 1, the weight of row
// L from lane L of the group.
template <int L, int W, int G, typename R, typename C>
__device__ __forceinline__ void interp_rows(const C* col, int Sx, R w2, R* ar, R* ai) {
  if constexpr (L < W) {
    const R w = group_lane<G, L>(w2);
    const C v = col[Sx * L];
    *ar = fma(w, v.x, *ar);
    *ai = fma(w, v.y, *ai);
    interp_rows<L + 1, W, G>(col, Sx, w2, ar, ai);
  }
}

// Fields of a record in LDS.
template <typename R, int D, int W>
__device__ __forceinline__ const R* rec_w(const char* lrec, int n) {
  return (const R*)(lrec + n * NodeRec<R, D, W>::BYTES);
}
template <typename R, int D, int W>
__device__ __forceinline__ unsigned rec_loc(const char* lrec, int n) {
  return ((const unsigned*)(lrec + n * NodeRec<R, D, W>::BYTES + NodeRec<R, D, W>::WBYTES))[0];
}
template <typename R, int D, int W>
__device__ __forceinline__ int rec_pj(const char* lrec, int n) {
  return ((const int*)(lrec + n * NodeRec<R, D, W>::BYTES + NodeRec<R, D, W>::WBYTES))[1];
}

// ---------------------------------------------------------------------------
// Spreading
// ---------------------------------------------------------------------------
// Packed fixed-point term: the 64-bit integer im * 2^32 + re (re, im signed
// 32-bit).  Sums of such terms decode exactly while |sum re|, |sum im| < 2^31.
__device__ __forceinline__ unsigned long long pack_term(float vr, float vi) {
  const int re = __float2int_rn(vr), im = __float2int_rn(vi);
  return ((unsigned long long)(unsigned)(im + (re >> 31)) << 32) | (unsigned)re;
}

template <typename R>
struct SpreadCell;
template <>
struct SpreadCell<float> {  // one 64-bit integer per cell
  static __device__ __forceinline__ void add(char* tile, int te, int idx, float vr, float vi) {
    __hip_atomic_fetch_add(&((unsigned long long*)tile)[idx], pack_term(vr, vi), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  static __device__ __forceinline__ float2 get(const char* tile, int te, int idx, float inv) {
    const long long s = (long long)((const unsigned long long*)tile)[idx];
    const int re = (int)(unsigned)s;
    const int im = (int)((s - (long long)re) >> 32);
    return float2{(float)re * inv, (float)im * inv};
  }
};
template <>
struct SpreadCell<double> {  // two FP64 planes
  static __device__ __forceinline__ void add(char* tile, int te, int idx, double vr, double vi) {
    double* t = (double*)tile;
    __hip_atomic_fetch_add(&t[idx], vr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(&t[te + idx], vi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  static __device__ __forceinline__ double2 get(const char* tile, int te, int idx, double) {
    const double* t = (const double*)tile;
    return double2{t[idx], t[te + idx]};
  }
};

// One work item (<= CH nodes of one tile, D <= 2) of spreading: the padded
// tile is accumulated in LDS -- FP64 adds of the data-precision products, one
// rounding per term, or packed fixed point -- and written to the item's slot
// of `scratch`.  W lanes per node (one per dimension-1 column, 64 / W nodes
// per wavefront step), each walking dimension 2.
//
// A plan of ordinary size has about one item per resident workgroup, so the
// time of an item is the chain of its memory latencies: item, then (caller
// index, node value) beside (first records), one barrier, taps, flush.  2 10^5
// radial nodes on 512^2 points, FP32, m = 4: 16.2 -> 13.2 us; 32 slices of
// 1.2 10^5 nodes: 171 -> 150 us.  FP64 is bound by its two LDS adds per tap.
template <typename R, int D, int W, int NT>
__device__ __forceinline__ void spread_tile_item(const KArgs& a, int item,
                                                 const typename cpx<R>::T* __restrict__ fhat,
                                                 typename cpx<R>::T* __restrict__ scratch) {
  static_assert(D <= 2, "3-D spreading lives in k_tile3.hip");
  using C = typename cpx<R>::T;
  using A = double;
  constexpr int NW = NT / 64, NB = NT < NBV ? NT : NBV;
  // FP32 2-D: the values of all nodes of an item (at most 2048) in registers,
  // for the fixed-point bound; otherwise one batch ahead
  constexpr bool HOLD = sizeof(R) == 4 && D == 2;
  constexpr int HPT = HOLD ? 2048 / NB : 1;
  constexpr unsigned LM = NodeRec<R, D, W>::LOCBITS >= 32 ? 0xFFFFFFFFu : (1u << NodeRec<R, D, W>::LOCBITS) - 1u;
  constexpr int NPW = 64 / W;
  extern __shared__ __align__(16) char smem[];
  const int4 it = a.items[item];
  char* tile = smem;
  C* fv = (C*)(smem + tile_fv_off(a.tileElems));
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int slot = lane / W, lx = lane - slot * W;
  const bool lane_on = slot < NPW;
  const int tid = threadIdx.x;

  R hre[HPT], him[HPT];
#pragma unroll
  for (int h = 0; h < HPT; ++h) {
    const int j = it.y + tid + h * NB;
    C v{0, 0};
    if (tid < NB && j < it.z) v = fhat[(long long)a.perm[j] * a.fst];
    hre[h] = v.x;
    him[h] = v.y;
  }
  int n = it.y + wave * NPW + slot;  // the lane's node
  NodeTaps<R, D, W> nx;
  nx.load(a.rec, lane_on && n < it.z ? n : it.y, lane_on ? lx : 0);

  // FP32 2-D with fix2: packed 32+32-bit fixed point in the first tileElems
  // 64-bit words, scale s = 2^(30 - e) from a strict bound of the item's
  // sums, B = sum_j |f_j|_inf * wmaxD < 2^e (as the 3-D FP32 kernel); one
  // ds_add_u64 per tap instead of two ds_add_f64
  const bool fix = HOLD && a.fix2;
  {
    const int nz = fix ? a.tileElems : 2 * a.tileElems;
    for (int i = tid; i < nz; i += NT) ((A*)tile)[i] = 0;
  }
  R fscale = 1, inv = 1;
  if (fix) {
    R part = 0;
#pragma unroll
    for (int h = 0; h < HPT; ++h) part += fmax(fabs(hre[h]), fabs(him[h]));
    part = group_sum<64>(part);
    R* red = (R*)fv;
    if (lane == 0) red[wave] = part;
    __syncthreads();
    double B = 0;
    for (int w = 0; w < NW; ++w) B += (double)red[w];
    B *= a.oscale * a.wmaxD * 1.0000001;
    int e = 0;
    if (B > 0) (void)frexp(B, &e);
    // both powers stay normal floats; a non-finite bound (Inf or NaN data)
    // spreads zeros and turns the slot into NaN at the flush
    e = max(e, -96);
    fscale = (R)ldexp(1.0, 30 - e);
    inv = (R)ldexp(1.0, e - 30);
    if (!(B <= 1.0e300)) {
      fscale = 0;
      inv = (R)NAN;
    }
    __syncthreads();  // before fv takes the values
  }
  const R sc = (R)a.oscale * fscale;

#pragma unroll(HOLD ? HPT : 1)
  for (int h = 0; h < (HOLD ? HPT : 1 << 20); ++h) {
    const int b0 = it.y + h * NB;
    if (b0 >= it.z) break;
    const int b1 = min(b0 + NB, it.z);
    if (tid < NB) fv[tid] = C{hre[HOLD ? h : 0] * sc, him[HOLD ? h : 0] * sc};
    __syncthreads();
    if constexpr (!HOLD) {  // the next batch's values
      const int j = b0 + NB + tid;
      C v{0, 0};
      if (tid < NB && j < it.z) v = fhat[(long long)a.perm[j] * a.fst];
      hre[0] = v.x;
      him[0] = v.y;
    }
    for (int n0 = b0 + wave * NPW; n0 < b1; n0 += NW * NPW) {
      n = n0 + slot;
      const bool on = lane_on && n < b1;
      const NodeTaps<R, D, W> c = nx;
      // the next step's node: in this batch, or the wavefront's first of the
      // next one
      const int m0 = n0 + NW * NPW < b1 ? n0 + NW * NPW : b0 + NB + wave * NPW;
      const int m = m0 + slot;
      nx.load(a.rec, lane_on && m < it.z ? m : it.y, lane_on ? lx : 0);
      if (on) {
        const C f = fv[n - b0];
        const R vr = f.x * c.w1, vi = f.y * c.w1;
        if constexpr (D == 2) {
          const int base = ((int)(c.pk & LM) + lx) + a.Sx * (int)(c.pk >> 16);
          if (fix) {
#pragma unroll
            for (int ly = 0; ly < W; ++ly)
              SpreadCell<float>::add(tile, a.tileElems, base + a.Sx * ly, (float)(vr * c.w2[ly]),
                                     (float)(vi * c.w2[ly]));
          } else {
#pragma unroll
            for (int ly = 0; ly < W; ++ly)
              SpreadCell<A>::add(tile, a.tileElems, base + a.Sx * ly, (A)(vr * c.w2[ly]), (A)(vi * c.w2[ly]));
          }
        } else {
          SpreadCell<A>::add(tile, a.tileElems, (int)c.pk + lx, (A)vr, (A)vi);
        }
      }
    }
    __syncthreads();
  }
  if (it.y >= it.z) __syncthreads();

  // padded tile -> this item's scratch slot (dense, px fastest), plain stores
  C* out = scratch + (size_t)item * a.padCells;
  for (int i = threadIdx.x; i < a.padCells; i += NT) {
    int px = i, py = 0;
    if (D >= 2) {
      const int q = (int)fdiv((uint32_t)i, a.divP0);
      px = i - q * a.Pd[0];
      py = q;
    }
    if (fix) {
      const float2 v = SpreadCell<float>::get(tile, a.tileElems, px + a.Sx * py, (float)inv);
      out[i] = C{(R)v.x, (R)v.y};
    } else {
      const auto v = SpreadCell<A>::get(tile, a.tileElems, px + a.Sx * py, 1.0);
      out[i] = C{(R)v.x, (R)v.y};
    }
  }
}

template <typename R, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_spread_tile(KArgs a, const typename cpx<R>::T* __restrict__ fhat,
                                                    typename cpx<R>::T* __restrict__ unused) {
  // items round robin over the XCDs: where nodes cluster, the items of one
  // region are much heavier than the rest, and contiguous item ranges per
  // XCD (xcd_item) leave the XCDs unevenly loaded
  const int item = blockIdx.x;
  if (item >= a.nitems) return;
  spread_tile_item<R, D, W, NT>(a, item, fhat + slice_nodes(a, blockIdx.y),
                                (typename cpx<R>::T*)a.scratch + slice_scratch(a, blockIdx.y));
}

// Fold: grid point x sums, over the padded tiles covering it, the scratch
// slots of every work item of those tiles.  Tile t's padded range is
// [tT - m + 1, tT + T + m - 1] modulo Ntilde; with that range no longer than
// Ntilde and 2T >= 2m - 1 (checked by the host) a point has at most 3
// covering (tile, offset) pairs per dimension.
// Covering pairs in the order of the images y = x - Nt, x, x + Nt and
// ascending tile: tile 0 (y = x - Nt, its left halo wrapped), tiles t - 1,
// t, t + 1 of x's own tile t (y = x), the last two tiles (y = x + Nt, a
// right halo wrapped).  With T >= m no other tile can cover x, so one
// division per point suffices.
__device__ __forceinline__ int cover_pairs(const KArgs& a, int d, int x, int* tl, int* pl) {
  const int T = a.T[d], P = a.Pd[d], Nt = a.Nt[d], nt = a.ntiles[d], m1 = a.m - 1;
  const int t = x / T;
  const int cu[6] = {0, t - 1, t, t + 1, nt - 2, nt - 1};
  const int cy[6] = {x - Nt, x, x, x, x + Nt, x + Nt};
  int n = 0;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const int u = cu[q];
    const int p = cy[q] - u * T + m1;
    if (u >= 0 && u < nt && p >= 0 && p < P && n < 3) {
      tl[n] = u;
      pl[n] = p;
      ++n;
    }
  }
  return n;
}

// Sum at grid point x (dimension 1) of the scratch slots covering it, given
// the covering (tile, offset) pairs of dimensions 2 and 3.
template <typename R, int D>
__device__ __forceinline__ typename cpx<R>::T fold_sum(const KArgs& a, const typename cpx<R>::T* __restrict__ scr,
                                                       int x, int n1, const int* t1, const int* p1, int n2,
                                                       const int* t2, const int* p2) {
  using C = typename cpx<R>::T;
  int t0[3] = {0, 0, 0}, p0[3] = {0, 0, 0};
  const int n0 = cover_pairs(a, 0, x, t0, p0);
  R sr = 0, si = 0;
#pragma unroll
  for (int c2 = 0; c2 < 3; ++c2) {
    if (c2 >= n2) break;
#pragma unroll
    for (int c1 = 0; c1 < 3; ++c1) {
      if (c1 >= n1) break;
#pragma unroll
      for (int c0 = 0; c0 < 3; ++c0) {
        if (c0 >= n0) break;
        const int t = t0[c0] + a.ntiles[0] * (t1[c1] + a.ntiles[1] * t2[c2]);
        const int off = p0[c0] + a.Pd[0] * (p1[c1] + a.Pd[1] * p2[c2]);
        for (int itm = a.tstart[t]; itm < a.tstart[t + 1]; ++itm) {
          const C v = scr[(size_t)itm * a.padCells + off];
          sr += v.x;
          si += v.y;
        }
      }
    }
  }
  return C{sr, si};
}

template <typename R, int D>
__global__ __launch_bounds__(256) void k_fold(KArgs a, typename cpx<R>::T* __restrict__ grid) {
  using C = typename cpx<R>::T;
  const C* scr = (const C*)a.scratch + slice_scratch(a, blockIdx.z);
  grid += slice_slot(a, blockIdx.z);
  const int x = blockIdx.x * 256 + threadIdx.x;
  const int ny = D >= 2 ? a.Nt[1] : 1;
  const int nrows = (D >= 2 ? a.Nt[1] : 1) * (D == 3 ? a.Nt[2] : 1);
  int t1[3] = {0, 0, 0}, p1[3] = {0, 0, 0}, t2[3] = {0, 0, 0}, p2[3] = {0, 0, 0};
  int n1 = 1, n2 = 1;
  for (int row = blockIdx.y; row < nrows; row += gridDim.y) {
    const int y = row % ny, z = row / ny;
    if (D >= 2) n1 = cover_pairs(a, 1, y, t1, p1);
    if (D == 3) n2 = cover_pairs(a, 2, z, t2, p2);
    if (x >= a.Nt[0]) continue;
    grid[(long long)row * a.Nt[0] + x] = fold_sum<R, D>(a, scr, x, n1, t1, p1, n2, t2, p2);
  }
}

// 2-D fold where every tile has at least m cells per dimension: a point is
// covered by its own tile and the eight around it only.  One workgroup per
// tile, a thread per point: the item ranges of the nine tiles are uniform and
// read together, then the covering values together (four at most where the
// tiles have 2m - 1 cells or more, up to nine on smaller ones), where fold_sum walks the covering pairs one dependent load after the other
// (512^2 points, FP32, radial nodes: 12.9 -> 9 us).
template <typename R>
__device__ __forceinline__ void fold2_point(const KArgs& a, const typename cpx<R>::T* __restrict__ scr,
                                            typename cpx<R>::T* __restrict__ grid, int tile, int c) {
  using C = typename cpx<R>::T;
  const int ntx = a.ntiles[0], nty = a.ntiles[1], oy = tile / ntx, ox = tile - oy * ntx;
  const int ly = (int)fdiv((uint32_t)c, a.divT0), lx = c - ly * a.T[0];
  const int x = ox * a.T[0] + lx, y = oy * a.T[1] + ly;
  const bool in = ly < a.T[1] && x < a.Nt[0] && y < a.Nt[1];
  int i0[9], i1[9], off[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const int dx = q % 3 - 1, dy = q / 3 - 1;
    int ux = ox + dx, uy = oy + dy, ix = x, iy = y;
    if (ux < 0) ux += ntx, ix += a.Nt[0];
    if (ux >= ntx) ux -= ntx, ix -= a.Nt[0];
    if (uy < 0) uy += nty, iy += a.Nt[1];
    if (uy >= nty) uy -= nty, iy -= a.Nt[1];
    const int t = ux + ntx * uy;
    i0[q] = a.tstart[t];
    i1[q] = a.tstart[t + 1];
    const int px = ix - ux * a.T[0] + a.m - 1, py = iy - uy * a.T[1] + a.m - 1;
    off[q] = in && px >= 0 && px < a.Pd[0] && py >= 0 && py < a.Pd[1] ? px + a.Pd[0] * py : -1;
  }
  C v[9];
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    v[q] = C{0, 0};
    if (i1[q] > i0[q] && off[q] >= 0) v[q] = scr[(size_t)i0[q] * a.padCells + off[q]];
  }
  R sr = 0, si = 0;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    sr += v[q].x;
    si += v[q].y;
    for (int itm = i0[q] + 1; itm < i1[q]; itm += 8) {  // crowded tiles, eight items in flight
      C w[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        w[u] = C{0, 0};
        if (itm + u < i1[q] && off[q] >= 0) w[u] = scr[(size_t)(itm + u) * a.padCells + off[q]];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        sr += w[u].x;
        si += w[u].y;
      }
    }
  }
  if (a.gdiv) {
    const R d = (R)a.gdiv[0];
    sr /= d;
    si /= d;
  }
  if (in) grid[(long long)y * a.Nt[0] + x] = C{sr, si};
}

template <typename R>
__global__ __launch_bounds__(256) void k_fold2(KArgs a, typename cpx<R>::T* __restrict__ grid) {
  using C = typename cpx<R>::T;
  fold2_point<R>(a, (const C*)a.scratch + slice_scratch(a, blockIdx.z), grid + slice_slot(a, blockIdx.z),
                 (int)blockIdx.x, (int)(blockIdx.y * 256 + threadIdx.x));
}

// ---------------------------------------------------------------------------
// Interpolation
// ---------------------------------------------------------------------------
// One work item of interpolation (D <= 2): stage the padded tile, gather
// every node with G lanes per node (one per dimension-1 column); the first
// records are read while the tile is staged, each later one a step ahead
// (32 slices of 1.2 10^5 nodes, FP32, m = 4: 130 -> 121 us).
//
// Every lane of a group has the sums of its node: lane s keeps those of step s,
// and the lanes store together after KEEP steps, ahead of the next loads.  With a
// store in every step each wait for a record, which counts stores as well, was
// one for the store just issued (us of interpolation: 100^2 image, 50 nodes per
// pixel, FP32 m = 3 26.8 -> 20.8, m = 5 49 -> 42, FP64 m = 3 36 -> 33; 64^2, 50 per
// pixel, FP64 m = 5 53 -> 41; 256^2, 16 per pixel, FP64 m = 3 39.0 -> 35.5).  FP32
// keeps four: eight scattered stores of a group together took longer where the
// results exceed the caches (256^2, 4 10^6 nodes, m = 4: 149 against 143).
template <typename R, int D, int W, int NT>
__device__ __forceinline__ void interp_tile_item(const KArgs& a, int item,
                                                 const typename cpx<R>::T* __restrict__ grid,
                                                 typename cpx<R>::T* __restrict__ fhat) {
  static_assert(D <= 2, "3-D interpolation lives in k_tile3.hip");
  using C = typename cpx<R>::T;
  constexpr int NW = NT / 64;
  constexpr unsigned LM = NodeRec<R, D, W>::LOCBITS >= 32 ? 0xFFFFFFFFu : (1u << NodeRec<R, D, W>::LOCBITS) - 1u;
  constexpr int G = LanesPerNode<W>::value;
  constexpr int NPW = 64 / G;
  extern __shared__ __align__(16) char smem[];
  const int4 it = a.items[item];
  // a batch has its KArgs in global memory: fields used among the stores of the
  // node loop are read once, here
  const char* const rec = a.rec;
  const long long fst = a.fst;
  const int Sx = a.Sx;
  C* const wdiv = (C*)a.wdiv;
  int* const wbad = a.wbad;
  C* tile = (C*)smem;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int slot = lane / G, lx = lane & (G - 1), lw = min(lx, W - 1);
  constexpr bool OWN = D == 2 && W * sizeof(R) > 32;
  NodeTaps<R, D, W, OWN> nx;
  {
    const int n = it.y + wave * NPW + slot;
    nx.load(rec, n < it.z ? n : it.y, lw);
  }
  int t0[3] = {0, 0, 0};
  tile_origin(a, D, it.x, t0);

  // stage the padded tile (within one period: at most one wrap per index),
  // ST cells per thread in flight
  constexpr int ST = 2;
  for (int i0 = threadIdx.x; i0 < a.padCells; i0 += ST * NT) {
    C v[ST];
    int li[ST];
#pragma unroll
    for (int u = 0; u < ST; ++u) {
      const int i = i0 + u * NT;
      const bool ok = i < a.padCells;
      int px = ok ? i : 0, py = 0;
      if (D >= 2) {
        const int q = (int)fdiv((uint32_t)px, a.divP0);
        px -= q * a.Pd[0];
        py = q;
      }
      int gx = t0[0] - a.m + 1 + px;
      gx += gx < 0 ? a.Nt[0] : 0;
      gx -= gx >= a.Nt[0] ? a.Nt[0] : 0;
      long long gi = gx;
      if (D >= 2) {
        int gy = t0[1] - a.m + 1 + py;
        gy += gy < 0 ? a.Nt[1] : 0;
        gy -= gy >= a.Nt[1] ? a.Nt[1] : 0;
        gi += (long long)gy * a.Nt[0];
      }
      v[u] = grid[gi];
      li[u] = ok ? px + a.Sx * py : -1;
    }
#pragma unroll
    for (int u = 0; u < ST; ++u)
      if (li[u] >= 0) tile[li[u]] = v[u];
  }
  __syncthreads();

  const R osc = (R)a.oscale, gd = D == 2 && wdiv ? (R)a.gdiv[0] : (R)1;
  R kr = 0, ki = 0;  // the lane's results and their index (-1: none)
  int kj = -1, step = 0;
  constexpr int KEEP = sizeof(R) == 4 && G > 4 ? 4 : G;
  auto store = [&]() {
    if (kj < 0) return;
    C* o = fhat + (long long)kj * fst;
    C v{kr * osc, ki * osc};
    if (D == 2 && wdiv) {
      const R t = v.x / gd;
      if (!(t > (R)0)) wbad[0] = 1;
      o = wdiv + kj;
      v = C{o->x / t, (R)0};
    }
    *o = v;
    kj = -1;
  };
  for (int n0 = it.y + wave * NPW; n0 < it.z; n0 += NW * NPW) {
    const int n = n0 + slot;
    const bool on = n < it.z;
    const NodeTaps<R, D, W, OWN> c = nx;
    if (step == KEEP) {
      store();
      step = 0;
    }
    const int m = n + NW * NPW;
    nx.load(rec, m < it.z ? m : it.y, lw);
    R ar = 0, ai = 0;
    if (on && lx < W) {
      if constexpr (D == 2) {
        const int base = ((int)(c.pk & LM) + lx) + Sx * (int)(c.pk >> 16);
        if constexpr (OWN) {
          interp_rows<0, W, G>(tile + base, Sx, c.w2[0], &ar, &ai);
        } else {
#pragma unroll
          for (int ly = 0; ly < W; ++ly) {
            const C v = tile[base + Sx * ly];
            ar = fma(c.w2[ly], v.x, ar);
            ai = fma(c.w2[ly], v.y, ai);
          }
        }
        ar *= c.w1;
        ai *= c.w1;
      } else {
        const C v = tile[(int)c.pk + lx];
        ar = c.w1 * v.x;
        ai = c.w1 * v.y;
      }
    }
    ar = group_sum<G>(ar);
    ai = group_sum<G>(ai);
    if (lx == step && on) {
      kr = ar;
      ki = ai;
      kj = c.pj;
    }
    ++step;
  }
  store();
}

template <typename R, int D, int W, int NT>
__global__ __launch_bounds__(NT) void k_interp_tile(KArgs a, const typename cpx<R>::T* __restrict__ grid,
                                                    typename cpx<R>::T* __restrict__ fhat) {
  const int item = blockIdx.x;  // round robin over the XCDs (k_spread_tile)
  if (item >= a.nitems) return;
  interp_tile_item<R, D, W, NT>(a, item, grid + slice_slot(a, blockIdx.y), fhat + slice_nodes(a, blockIdx.y));
}

}  // namespace nfftm
