// Block kernels: several right-hand sides of one hierarchy in one launch.
//
// k independent integer solves on the same hierarchy (INTAMG.hpp:269-293
// applied to k vectors) share every matrix, factor and level schedule, so a
// kernel loads each entry once and applies it to all of them.  Vectors of a
// block are stored in groups of four right-hand sides: element (row i,
// right-hand side r) sits at ((r / 4) * n + i) * 4 + r % 4, so the four
// values of a row form one 16-byte word.  Every operation is integer and
// per element (the sums of a row are order-free), so each right-hand side's
// values are those its own single solve computes, bit for bit.
#include <type_traits>

#include "dev_common.hpp"
#include "launch.hpp"
#include "tri_common.hpp"

namespace sc23ad::dev {

namespace {

constexpr int kBk = 256;
constexpr int kSellBlkRows = 256 * kBk;  // a workgroup for every CU

__device__ __forceinline__ int32_t lane_of(const int4& v, int c) {
  return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
}

__device__ __forceinline__ int4 fin4(const uint64_t* acc, int bit, int mode, int4 z) {
  int4 y;
  int32_t s[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) s[c] = low32(as_i64(acc[c]) >> bit);
  if (mode == 0) {
    y = make_int4(s[0], s[1], s[2], s[3]);
  } else if (mode == 1) {
    y = make_int4(sub32(z.x, s[0]), sub32(z.y, s[1]), sub32(z.z, s[2]), sub32(z.w, s[3]));
  } else {
    y = make_int4(add32(z.x, s[0]), add32(z.y, s[1]), add32(z.z, s[2]), add32(z.w, s[3]));
  }
  return y;
}

__device__ __forceinline__ void mac4(uint64_t* acc, int32_t v, const int4& x) {
  acc[0] += prod64(v, x.x);
  acc[1] += prod64(v, x.y);
  acc[2] += prod64(v, x.z);
  acc[3] += prod64(v, x.w);
}

// ---- permutation into / out of a level's smoother order -------------------
template <bool kGather>
__global__ __launch_bounds__(kBk) void k_permute_blk(int n, int groups, const int* __restrict__ perm,
                                                     const int4* __restrict__ src,
                                                     int4* __restrict__ dst) {
  const long long t = static_cast<long long>(blockIdx.x) * kBk + threadIdx.x;
  if (t >= static_cast<long long>(n) * groups) return;
  const int g = static_cast<int>(t / n), k = static_cast<int>(t % n);
  const size_t base = static_cast<size_t>(g) * n;
  if (kGather) dst[base + k] = src[base + perm[k]];
  else dst[base + perm[k]] = src[base + k];
}

__global__ __launch_bounds__(kBk) void k_copy_blk(size_t n4, const int4* __restrict__ src,
                                                  int4* __restrict__ dst) {
  for (size_t i = blockIdx.x * static_cast<size_t>(kBk) + threadIdx.x; i < n4;
       i += static_cast<size_t>(gridDim.x) * kBk)
    dst[i] = src[i];
}

// One right-hand side of a block <-> a plain vector.
template <bool kGet>
__global__ __launch_bounds__(kBk) void k_blk_column(int n, int r, int32_t* __restrict__ blk,
                                                   int32_t* __restrict__ col) {
  const int i = blockIdx.x * kBk + threadIdx.x;
  if (i >= n) return;
  const size_t at = (static_cast<size_t>(r >> 2) * n + i) * 4 + (r & 3);
  if (kGet) col[i] = blk[at];
  else blk[at] = col[i];
}

// ---- SpMV: y_r = (int32)((A x_r) >> bit) for every right-hand side r -----
// CSR: kGroups x kSlots lanes per row; lane (g, slot) adds the row's entries
// slot, slot + kSlots, ... for the four right-hand sides of group g, four
// entries per round with every load unconditional (clamped; their value is
// then zero), and the slots' sums are added with DPP moves (64-bit sums are
// order-free).  MODE 1 / 2 fuse y = z - A x / y = z + A x.
template <int MODE, int kGroups, int kSlots>
__global__ __launch_bounds__(kBk) void k_spmv_blk_csr(int n, int m, const int* __restrict__ rptr,
                                                      const int* __restrict__ cind,
                                                      const int32_t* __restrict__ val, int bit,
                                                      const int4* __restrict__ x,
                                                      const int4* z, int4* y) {
  constexpr int kLanes = kGroups * kSlots;
  const int t = threadIdx.x;
  const int row = blockIdx.x * (kBk / kLanes) + t / kLanes;
  const int slot = t % kSlots, g = t / kSlots % kGroups;
  uint64_t acc[4] = {0, 0, 0, 0};
  const size_t at = static_cast<size_t>(g) * n + row;
  int4 zv = make_int4(0, 0, 0, 0);
  if (row < n) {
    const int4* xg = x + static_cast<size_t>(g) * m;
    const int rb = rptr[row], re = rptr[row + 1];
    if (MODE != 0) zv = z[at];
    for (int p0 = rb + slot; p0 < re; p0 += 4 * kSlots) {
      int cc[4];
      int32_t vv[4];
      int4 xx[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = p0 + j * kSlots < re ? p0 + j * kSlots : p0;
        cc[j] = cind[p];
        vv[j] = val[p];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) xx[j] = xg[cc[j]];
#pragma unroll
      for (int j = 0; j < 4; ++j) mac4(acc, p0 + j * kSlots < re ? vv[j] : 0, xx[j]);
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = group_sum<kSlots>(acc[c]);
  if (row < n && slot == 0) y[at] = fin4(acc, bit, MODE, zv);
}

template <int MODE, int kGroups>
__global__ __launch_bounds__(kBk) void k_spmv_blk_sell(int n, int m,
                                                       const long long* __restrict__ soff,
                                                       const int* __restrict__ scol,
                                                       const int32_t* __restrict__ sval,
                                                       const int* __restrict__ srow, int bit,
                                                       const int4* __restrict__ x,
                                                       const int4* z, int4* y) {
  const int row = blockIdx.x * kBk + threadIdx.x;
  if (row >= n) return;
  const int orow = srow ? srow[row] : row;
  const long long b = soff[row >> 6];
  const int w = static_cast<int>((soff[(row >> 6) + 1] - b) >> 6);
  const int* c = scol + b + (row & 63);
  const int32_t* v = sval + b + (row & 63);
  uint64_t acc[kGroups][4];
#pragma unroll
  for (int g = 0; g < kGroups; ++g)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[g][q] = 0;
  for (int k0 = 0; k0 < w; k0 += 8) {
    int cc[8];
    int32_t vv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < w ? k0 + j : k0;
      const int col = c[64 * k];
      cc[j] = col < 0 ? 0 : col;
      vv[j] = (k0 + j < w && col >= 0) ? v[64 * k] : 0;
    }
#pragma unroll
    for (int g = 0; g < kGroups; ++g) {
      int4 xx[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) xx[j] = x[static_cast<size_t>(g) * m + cc[j]];
#pragma unroll
      for (int j = 0; j < 8; ++j) mac4(acc[g], vv[j], xx[j]);
    }
  }
#pragma unroll
  for (int g = 0; g < kGroups; ++g) {
    const size_t at = static_cast<size_t>(g) * n + orow;
    const int4 zv = MODE != 0 ? z[at] : make_int4(0, 0, 0, 0);
    y[at] = fin4(acc[g], bit, MODE, zv);
  }
}

}  // namespace

hipError_t launch_permute_blk(int n, int groups, const int* perm, const void* src, void* dst,
                              bool gather, hipStream_t s) {
  const long long tot = static_cast<long long>(n) * groups;
  if (tot <= 0) return hipSuccess;
  const int grid = static_cast<int>((tot + kBk - 1) / kBk);
  if (gather)
    hipLaunchKernelGGL(k_permute_blk<true>, dim3(grid), dim3(kBk), 0, s, n, groups, perm,
                       static_cast<const int4*>(src), static_cast<int4*>(dst));
  else
    hipLaunchKernelGGL(k_permute_blk<false>, dim3(grid), dim3(kBk), 0, s, n, groups, perm,
                       static_cast<const int4*>(src), static_cast<int4*>(dst));
  return hipGetLastError();
}

hipError_t launch_copy_blk(int n, int groups, const void* src, void* dst, hipStream_t s) {
  const size_t n4 = static_cast<size_t>(n) * groups;
  if (n4 == 0) return hipSuccess;
  const int grid = static_cast<int>(std::min<size_t>((n4 + kBk - 1) / kBk, 8192));
  hipLaunchKernelGGL(k_copy_blk, dim3(grid), dim3(kBk), 0, s, n4, static_cast<const int4*>(src),
                     static_cast<int4*>(dst));
  return hipGetLastError();
}

hipError_t launch_blk_column(int n, int r, void* blk, void* col, bool get, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const int grid = (n + kBk - 1) / kBk;
  if (get)
    hipLaunchKernelGGL(k_blk_column<true>, dim3(grid), dim3(kBk), 0, s, n, r,
                       static_cast<int32_t*>(blk), static_cast<int32_t*>(col));
  else
    hipLaunchKernelGGL(k_blk_column<false>, dim3(grid), dim3(kBk), 0, s, n, r,
                       static_cast<int32_t*>(blk), static_cast<int32_t*>(col));
  return hipGetLastError();
}

template <int MODE, int kGroups>
static hipError_t spmv_blk_go(const DCsr& a, const void* x, const void* z, void* y,
                              hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  const int4* xv = static_cast<const int4*>(x);
  const int4* zv = static_cast<const int4*>(z);
  int4* yv = static_cast<int4*>(y);
  // SELL (one lane per row) where its rows fill the chip: 96^3 inclusions, 16
  // right-hand sides, 28,160 rows on 110 workgroups took 53 us
  if (a.soff && a.scol && a.n >= kSellBlkRows) {
    hipLaunchKernelGGL((k_spmv_blk_sell<MODE, kGroups>), dim3((a.n + kBk - 1) / kBk), dim3(kBk),
                       0, s, a.n, a.m, a.soff, a.scol, static_cast<const int32_t*>(a.sval),
                       a.srow, a.bit, xv, zv, yv);
    return hipGetLastError();
  }
  auto go = [&](auto slots) -> hipError_t {
    constexpr int kSlots = decltype(slots)::value;
    constexpr int kRows = kBk / (kGroups * kSlots);
    hipLaunchKernelGGL((k_spmv_blk_csr<MODE, kGroups, kSlots>), dim3((a.n + kRows - 1) / kRows),
                       dim3(kBk), 0, s, a.n, a.m, a.rptr, a.cind,
                       static_cast<const int32_t*>(a.val), a.bit, xv, zv, yv);
    return hipGetLastError();
  };
  // about eight entries per lane: at 4 per lane 120,000 rows of 60 entries
  // took 122 us instead of 92, at one lane per row 131-340 us on the coarse
  // levels (96^3 inclusions, 16 right-hand sides), now 23-92 us
  const double avg = static_cast<double>(a.nnz) / a.n;
  if (avg <= 8) return go(std::integral_constant<int, 1>{});
  if (avg <= 16) return go(std::integral_constant<int, 2>{});
  if (avg <= 32) return go(std::integral_constant<int, 4>{});
  if (avg <= 64) return go(std::integral_constant<int, 8>{});
  return go(std::integral_constant<int, 16>{});
}

template <int MODE>
static hipError_t spmv_blk_mode(const DCsr& a, int groups, const void* x, const void* z,
                                void* y, hipStream_t s) {
  // four, two or one groups per launch
  for (int g0 = 0, gs = 0; g0 < groups; g0 += gs) {
    gs = groups - g0 >= 4 ? 4 : groups - g0 >= 2 ? 2 : 1;
    const size_t xo = static_cast<size_t>(g0) * a.m, yo = static_cast<size_t>(g0) * a.n;
    const int4* xx = static_cast<const int4*>(x) + xo;
    const int4* zz = z ? static_cast<const int4*>(z) + yo : nullptr;
    int4* yy = static_cast<int4*>(y) + yo;
    hipError_t e;
    switch (gs) {
      case 1: e = spmv_blk_go<MODE, 1>(a, xx, zz, yy, s); break;
      case 2: e = spmv_blk_go<MODE, 2>(a, xx, zz, yy, s); break;
      default: e = spmv_blk_go<MODE, 4>(a, xx, zz, yy, s); break;
    }
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_spmv_blk(const DCsr& a, int groups, SpmvMode mode, const void* x,
                           const void* z, void* y, hipStream_t s) {
  if (mode == SpmvMode::kPlain) return spmv_blk_mode<0>(a, groups, x, z, y, s);
  if (mode == SpmvMode::kSub) return spmv_blk_mode<1>(a, groups, x, z, y, s);
  return spmv_blk_mode<2>(a, groups, x, z, y, s);
}


}  // namespace sc23ad::dev
