// mixfft.hpp -- the pruned FFT passes on grids that are not powers of two
// (k_mixfft.hip): line FFTs whose radices are chosen per plan.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.hpp"

namespace nfftm {

constexpr int MIX_PASSES = 6;

// One Stockham pass: radix r, NS the product of the radices before it,
// M = L / r butterflies per line, twiddle step ts = L / (NS r), and the
// multiplier and shift of the division by NS.  Packed, so that the passes of
// a line take one or two cache lines of the kernel arguments (unpacked
// descriptors were fetched one after the other, a miss each, as the passes
// reached them).
struct MixPass {
  uint32_t r_sh_ns, m_ts, mul;
  __host__ __device__ int r() const { return (int)(r_sh_ns & 255u); }
  __host__ __device__ int NS() const { return (int)(r_sh_ns >> 16); }
  __host__ __device__ int M() const { return (int)(m_ts & 65535u); }
  __host__ __device__ int ts() const { return (int)(m_ts >> 16); }
  __host__ __device__ FastDiv dNS() const { return FastDiv{(uint32_t)NS(), mul, (r_sh_ns >> 8) & 255u}; }
};

// Butterflies of radix r that a thread holds at most.
constexpr __host__ __device__ int mix_butterflies(int r) { return (8 + r - 1) / r; }

// Radices of a line of L points and the threads that share it.
struct MixLine {
  int L, npass, tpl;
  FastDiv dtpl;
  MixPass p[MIX_PASSES];
};

// Arguments of one pass over the lines of one dimension d of a grid (and of
// the slices of a directional plan).
struct MixArgs {
  MixLine ln;
  const void* tw;      // (cos, sin)(2 pi k / L), k < L, in the data precision
  int N, Na;           // image size along d and N / 2
  int lpb, lsh;        // lines per workgroup (power of two in the strided passes: 1 << lsh)
  int nlines;          // dimension 1: lines (N_2 N_3)
  int nx, nchunk;      // strided passes: lines along x, and their chunks of lpb
  FastDiv dchunk, dN1; // divisions by nchunk and by the image size along dimension 2
  int total;           // workgroups per slice
  int oall, oN, oL, oNa;  // strided passes: the remaining dimension (all its positions, or the image's)
  long long st, ost;      // grid strides along d and along the remaining dimension
  int N1, L1, Na1, N2, L2, Na2;  // dimension 1: placement of the lines (y, z)
  long long st1, st2;
  const double* fac[3];  // deconvolution factors (dimension-1 passes)
  double oscale;
  long long ist;         // element stride of the image
  // slices of a directional plan: the image of slice s starts at element
  // s % Bsl + (s / Bsl) Bsl P, its grid is slot nsl - 1 - (s - s0)
  int s0, nsl;
  long long Bsl, P, Q;
  const void* lam;  // launch_mix_mul: the grid-sized factor
};

// Radices of a line of L points; false where the passes are not built for it
// (only: the line is the whole 1-D grid, no strided pass follows; rmax: largest
// radix).
bool mix_factor(int64_t L, bool dbl, bool only, MixLine* ln, int rmax = 16);
// Lines per workgroup of the dimension-1 pass (col = false) or of a strided
// pass, for `lines` lines at each of `outer` positions.
int mix_shape(bool dbl, bool col, const MixLine& ln, long long lines, long long outer);
size_t mix_lds_bytes(bool dbl, bool col, const MixLine& ln, int lpb);
hipError_t launch_mix_x(bool dbl, bool fwd, const MixArgs& a, hipStream_t s, const void* in, void* out);
hipError_t launch_mix_col(bool dbl, bool fwd, const MixArgs& a, hipStream_t s, void* grid);
// Strided pass along the last dimension in place: forward FFT of the image
// positions, product with lam, inverse FFT, image positions written.
size_t mix_mul_lds_bytes(bool dbl, const MixLine& ln, int lpb);
hipError_t launch_mix_mul(bool dbl, const MixArgs& a, hipStream_t s, void* grid);

}  // namespace nfftm
