// k_bin.hip -- node binning on the device for nodes! (src/implementation.jl:
// 108-141): the shift into [0, 1) of shiftNodes! (src/utils.jl:32-44) and the
// binning of src/precomputation.jl:459-520 (_precomputeBlocks), here at tile
// granularity:
//   1. k_bin_keys: tile index of every node (FP64 k * Ntilde, truncated, as
//      the reference's floor of the shifted node), a histogram of the tiles;
//   2. a stable radix sort of (tile, caller index) pairs over the key bits:
//      within a tile the nodes keep the caller's order, so the binning is
//      deterministic;
//   3. k_bin_scan: tile offsets and work-item offsets (chunks of at most CH
//      nodes of one tile), one workgroup;
//   4. k_bin_items: the work items and per-tile item ranges;
//   5. k_bin_ks: the shifted coordinates in sorted order.
#include <rocprim/device/device_radix_sort.hpp>

#include "launch.hpp"

namespace nfftm {

namespace {

constexpr int BT = 256;  // threads of the elementwise binning kernels

// shiftNodes! (src/utils.jl:32-44): k < 0 moves up by 1, and a result of
// exactly 1 (a negative k that rounds to 1 - k == 1) is pulled below 1 by
// eps(Float64).
__device__ __forceinline__ double shifted(double x) {
  if (x < 0.0) x += 1.0;
  if (x == 1.0) x -= 2.220446049250313e-16;  // eps(Float64)
  return x;
}

// Tile of node j (k in the caller's layout).  A coordinate outside
// [-1/2, 1/2] (or NaN) is flagged and taken as 0: the host reads the flag
// before anything of the plan changes.
__device__ __forceinline__ int node_tile(const BinArgs& a, const double* __restrict__ k, long long j, int* bad) {
  int t = 0, str = 1;
  for (int d = 0; d < a.D; ++d) {
    double x = k[d * a.sd + j * a.sj];
    if (!(fabs(x) <= 0.5)) {
      *bad = 1;
      x = 0;
    }
    const double kscale = shifted(x) * (double)a.Nt[d];
    int c = (int)kscale;
    if (c >= a.Nt[d]) c -= a.Nt[d];
    t += (int)((unsigned)c / (unsigned)a.T[d]) * str;
    str *= a.ntiles[d];
  }
  return t;
}

__global__ __launch_bounds__(BT) void k_bin_keys(BinArgs a, const double* __restrict__ k, int* __restrict__ key,
                                                 int* __restrict__ idx, int* __restrict__ cnt) {
  const long long j = (long long)blockIdx.x * BT + threadIdx.x;
  if (j >= a.M) return;
  const int t = node_tile(a, k, j, &cnt[a.ntile]);
  key[j] = t;
  idx[j] = (int)j;
  atomicAdd(&cnt[t], 1);
}

// The same with the histogram of each workgroup's nodes in LDS first (at most
// HIST tiles): crowded tiles (thousands of nodes in one tile) then cost one
// global atomic per workgroup instead of one per node.
constexpr int HIST = 16384;
constexpr int HIST_BLOCKS = 512;
__global__ __launch_bounds__(BT) void k_bin_keys_lds(BinArgs a, const double* __restrict__ k, int* __restrict__ key,
                                                     int* __restrict__ idx, int* __restrict__ cnt) {
  __shared__ int hist[HIST];
  for (int i = threadIdx.x; i < a.ntile; i += BT) hist[i] = 0;
  __syncthreads();
  for (long long j = (long long)blockIdx.x * BT + threadIdx.x; j < a.M; j += (long long)gridDim.x * BT) {
    const int t = node_tile(a, k, j, &cnt[a.ntile]);
    key[j] = t;
    idx[j] = (int)j;
    atomicAdd(&hist[t], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < a.ntile; i += BT)
    if (hist[i]) atomicAdd(&cnt[i], hist[i]);
}

// One workgroup: off = exclusive scan of cnt (ntile + 1 entries), ioff =
// exclusive scan of ceil(cnt / CH) (work items per tile); stats[0] = number
// of work items, stats[1] = tiles of more than one, stats[2] = 0 (the counter
// of k_bin_items), stats[3] = the bad-node flag cnt[ntile].  Each thread sums
// its run of tiles, the 1024 sums are scanned by wavefront shuffles (by one
// thread they took 20 of 27 us).
constexpr int ST = 1024;
__device__ __forceinline__ int3 wave_scan(int3 v) {  // inclusive
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int x = __shfl_up(v.x, o), y = __shfl_up(v.y, o), z = __shfl_up(v.z, o);
    if ((int)(threadIdx.x & 63) >= o) v.x += x, v.y += y, v.z += z;
  }
  return v;
}
__global__ __launch_bounds__(ST) void k_bin_scan(BinArgs a, const int* __restrict__ cnt, int* __restrict__ off,
                                                 int* __restrict__ ioff, int* __restrict__ stats) {
  __shared__ int3 s_wave[ST / 64];
  const int n = a.ntile;
  const int per = (n + ST - 1) / ST;
  const int b = min(n, (int)threadIdx.x * per), e = min(n, b + per);
  int3 s{0, 0, 0};  // nodes, items, tiles of several items
  for (int t = b; t < e; ++t) {
    const int c = cnt[t];
    const int it = (c + a.CH - 1) / a.CH;
    s.x += c;
    s.y += it;
    s.z += it > 1;
  }
  int3 inc = wave_scan(s);
  if ((threadIdx.x & 63) == 63) s_wave[threadIdx.x >> 6] = inc;
  __syncthreads();
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) {
    inc.x += s_wave[w].x;
    inc.y += s_wave[w].y;
    inc.z += s_wave[w].z;
  }
  if (threadIdx.x == ST - 1) {
    off[n] = inc.x;
    ioff[n] = inc.y;
    stats[0] = inc.y;
    stats[1] = inc.z;
    stats[2] = 0;
    stats[3] = cnt[n];
  }
  int an = inc.x - s.x, ai = inc.y - s.y;
  for (int t = b; t < e; ++t) {
    const int c = cnt[t];
    off[t] = an;
    ioff[t] = ai;
    an += c;
    ai += (c + a.CH - 1) / a.CH;
  }
}

// Work items of tile t: {t, begin, end, 0} for chunks of at most CH nodes;
// tstart[t] = first item of tile t (tstart[ntile] = number of items); the
// tiles of several items are listed in multi (in any order).
__global__ __launch_bounds__(BT) void k_bin_items(BinArgs a, const int* __restrict__ off, const int* __restrict__ ioff,
                                                  int4* __restrict__ items, int* __restrict__ tstart,
                                                  int* __restrict__ multi, int* __restrict__ nmulti) {
  const long long t = (long long)blockIdx.x * BT + threadIdx.x;
  if (t > a.ntile) return;
  tstart[t] = ioff[t];
  if (t == a.ntile) return;
  const int b0 = off[t], e0 = off[t + 1];
  int q = ioff[t];
  if (ioff[t + 1] - q > 1) multi[atomicAdd(nmulti, 1)] = (int)t;
  for (int s = b0; s < e0; s += a.CH) items[q++] = int4{(int)t, s, min(e0, s + a.CH), 0};
}

// ks[d * M + s] = shifted k of node perm[s] (perm == nullptr: caller order).
__global__ __launch_bounds__(BT) void k_bin_ks(BinArgs a, const double* __restrict__ k, const int* __restrict__ perm,
                                               double* __restrict__ ks) {
  const long long s = (long long)blockIdx.x * BT + threadIdx.x;
  if (s >= a.M) return;
  const long long j = perm ? perm[s] : s;
  for (int d = 0; d < a.D; ++d) ks[(long long)d * a.M + s] = shifted(k[d * a.sd + j * a.sj]);
}

// flag[0] = 1 if some coordinate is outside [-1/2, 1/2] or NaN.
__global__ __launch_bounds__(BT) void k_check(const double* __restrict__ k, long long n, int* __restrict__ flag) {
  const long long i = (long long)blockIdx.x * BT + threadIdx.x;
  if (i < n && !(fabs(k[i]) <= 0.5)) flag[0] = 1;
}

__global__ __launch_bounds__(BT) void k_iota(int* __restrict__ p, long long n) {
  const long long i = (long long)blockIdx.x * BT + threadIdx.x;
  if (i < n) p[i] = (int)i;
}

inline unsigned blocks(long long n) { return (unsigned)((n + BT - 1) / BT); }

}  // namespace

// The radix passes for every M: up to 2^20 nodes rocPRIM would take its merge
// sort, 17 launches and 91 us for 2 10^5 nodes.
using SortConfig =
    rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config, rocprim::default_config, 0>;

size_t bin_sort_temp_bytes(long long M, int key_bits) {
  size_t bytes = 0;
  if (rocprim::radix_sort_pairs<SortConfig>(nullptr, bytes, (int*)nullptr, (int*)nullptr, (int*)nullptr, (int*)nullptr,
                                (size_t)M, 0, key_bits) != hipSuccess)
    return 0;
  return std::max<size_t>(bytes, 16);
}

hipError_t launch_bin_keys(const BinArgs& a, const double* k, int* key, int* idx, int* cnt, hipStream_t s) {
  hipError_t e = launch_fill0(cnt, sizeof(int) * ((size_t)a.ntile + 1), s);
  if (e != hipSuccess || a.M == 0) return e;
  if (a.ntile <= HIST) {
    const unsigned nb = (unsigned)std::min<long long>(HIST_BLOCKS, (a.M + BT - 1) / BT);
    hipLaunchKernelGGL(k_bin_keys_lds, dim3(nb), dim3(BT), 0, s, a, k, key, idx, cnt);
  } else {
    hipLaunchKernelGGL(k_bin_keys, dim3(blocks(a.M)), dim3(BT), 0, s, a, k, key, idx, cnt);
  }
  return hipGetLastError();
}

hipError_t launch_bin_sort(const BinArgs& a, void* temp, size_t temp_bytes, int* key_in, int* key_out, int* idx_in,
                           int* idx_out, hipStream_t s) {
  if (a.M == 0) return hipSuccess;
  return rocprim::radix_sort_pairs<SortConfig>(temp, temp_bytes, key_in, key_out, idx_in, idx_out, (size_t)a.M, 0, a.key_bits,
                                   s);
}

hipError_t launch_bin_scan(const BinArgs& a, const int* cnt, int* off, int* ioff, int* stats, hipStream_t s) {
  hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(ST), 0, s, a, cnt, off, ioff, stats);
  return hipGetLastError();
}

hipError_t launch_bin_items(const BinArgs& a, const int* off, const int* ioff, int4* items, int* tstart, int* multi,
                            int* nmulti, hipStream_t s) {
  hipLaunchKernelGGL(k_bin_items, dim3(blocks((long long)a.ntile + 1)), dim3(BT), 0, s, a, off, ioff, items, tstart,
                     multi, nmulti);
  return hipGetLastError();
}

hipError_t launch_bin_ks(const BinArgs& a, const double* k, const int* perm, double* ks, hipStream_t s) {
  if (a.M == 0) return hipSuccess;
  hipLaunchKernelGGL(k_bin_ks, dim3(blocks(a.M)), dim3(BT), 0, s, a, k, perm, ks);
  return hipGetLastError();
}

hipError_t launch_check_nodes(const double* k, long long n, int* flag, hipStream_t s) {
  const hipError_t e = launch_fill0(flag, sizeof(int), s);
  if (e != hipSuccess || n == 0) return e;
  hipLaunchKernelGGL(k_check, dim3(blocks(n)), dim3(BT), 0, s, k, n, flag);
  return hipGetLastError();
}

hipError_t launch_iota(int* p, long long n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_iota, dim3(blocks(n)), dim3(BT), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace nfftm
