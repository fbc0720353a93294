// Sparse matrix-vector products and level-scheduled triangular solves.
//
// Integer kernels (CSR int32 values, int64 accumulation, arithmetic shift;
// Library/matrix/spmat.hpp:77-86,128-137) are order-free, so a row may be
// split across lanes.  FP kernels (CSR<T>::SpMV spmat.hpp:43-52 and the
// triangular solves) keep each row's sum strictly in column order, one thread
// per row, so that the device rounds exactly like the CPU.
#include <hip/hip_ext.h>

#include <cstdlib>
#include <type_traits>

#include "dev_common.hpp"
#include "launch.hpp"
#include "tri_common.hpp"

namespace sc23ad::dev {

namespace {
thread_local DispatchEvents t_armed;
}  // namespace

void arm_dispatch_events(hipEvent_t start, hipEvent_t stop) { t_armed = {start, stop}; }

DispatchEvents take_dispatch_events() {
  const DispatchEvents e = t_armed;
  t_armed = {};
  return e;
}

namespace {

constexpr int kBlock = 256;

// SpMV workgroups renumbered per XCD (xcd_block) when SC23AD_XCD_REMAP=1.
// Off by default: the fine-level SpMV ran 4 % slower with it.  The SpMV
// tuner also tries it per matrix on the row-sorted SELL copies (restriction,
// prolongation), whose scattered rows of one window then stay under one L2
// (at 128^3 their HBM fetches fell 30-45 %).
int xcd_remap() {
  static const int on = [] {
    const char* e = std::getenv("SC23AD_XCD_REMAP");
    return (e && e[0] == '1') ? 1 : 0;
  }();
  return on;
}

// A launch that honours armed dispatch events (arm_dispatch_events).
template <typename F, typename... A>
void launch_timed(F kern, dim3 grid, dim3 block, uint32_t lds, hipStream_t s, A... args) {
  const DispatchEvents ev = take_dispatch_events();
  if (ev.start)
    hipExtLaunchKernelGGL(kern, grid, block, lds, s, ev.start, ev.stop, 0u, args...);
  else
    hipLaunchKernelGGL(kern, grid, block, lds, s, args...);
}

// CSR integer SpMV, G lanes per row.  Each lane takes the row's entries
// lane, lane + G, ... eight at a time with every load unconditional (clamped
// to the chunk's first entry), so a chunk costs two memory latencies (entries,
// then the gathered x values) instead of two per entry.
template <int G, int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_int(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind,
    const int32_t* __restrict__ val, int bit, const int32_t* __restrict__ x,
    const int32_t* z, int32_t* y, int remap) {
  const int blk = remap ? xcd_block() : static_cast<int>(blockIdx.x);
  const int gid = blk * kBlock + threadIdx.x;
  const int row = gid / G;
  const int lane = gid & (G - 1);
  uint64_t acc = 0;
  int32_t zv = 0;
  if (row < n) {
    if (MODE != 0 && lane == 0) zv = z[row];
    const int rb = rptr[row], re = rptr[row + 1];
    for (int p0 = rb + lane; p0 < re; p0 += 8 * G) {
      int cc[8];
      int32_t vv[8], xx[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int p = p0 + j * G < re ? p0 + j * G : p0;
        cc[j] = cind[p];
        vv[j] = val[p];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) xx[j] = x[cc[j]];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (p0 + j * G < re) acc += prod64(vv[j], xx[j]);
    }
  }
#pragma unroll
  for (int m = G / 2; m > 0; m >>= 1) acc += shfl_xor_u64(acc, m);
  if (row < n && lane == 0) {
    const int32_t s = low32(as_i64(acc) >> bit);
    if (MODE == 0) y[row] = s;
    else if (MODE == 1) y[row] = sub32(zv, s);
    else y[row] = add32(zv, s);
  }
}

// CSR integer SpMV streamed through LDS: a workgroup owns kRows consecutive
// rows, reads their entries coalesced in tiles of 8 per thread, whatever the
// row lengths, leaves the products in LDS, and kBlock / kRows lanes per row add
// them (the next tile's entries are already in flight).  The lanes-per-row
// kernel above reads short pieces of many rows per instruction and repeats its
// clamped loads where a row is shorter than 8 G: with 8 lanes per row 79 us on
// the 95^3 27-point operator and 134 us on the 128^3 7-point one, against 43
// and 35 us here with 128 rows (4.5 and 4.1 TB/s).
//
// kLong (rows of unknown lengths): a row of more than 32 entries per lane would
// hold up its workgroup, one LDS read after another by few lanes (65,536 rows
// of 300: 140 us at two lanes per row; 100 rows of 50,000: 1,974).  A workgroup
// that has one shares every tile's products among the rows that the tile
// holds, up to all its lanes for one row, and adds the parts to the rows' sums
// in LDS (60 and 175 us).
template <int kRows, int MODE, bool kLong>
__global__ __launch_bounds__(kBlock) void k_spmv_stream_int(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind,
    const int32_t* __restrict__ val, int bit, const int32_t* __restrict__ x,
    const int32_t* z, int32_t* y) {
  constexpr int kPer = 8, kTile = kBlock * kPer, kLanes = kBlock / kRows;
  __shared__ uint64_t prod[kTile];
  __shared__ int rp[kRows + 1];
  __shared__ unsigned long long sums[kLong ? kRows : 1];
  __shared__ int long_in[kBlock / 64];
  const int t = threadIdx.x;
  const int r0 = blockIdx.x * kRows, nr = min(kRows, n - r0);
  if constexpr (kLong) {
    static_assert(kRows <= kBlock, "a row per thread");
    bool mine = false;
    if (t < nr) {
      const int rb = rptr[r0 + t], re = rptr[r0 + t + 1];
      rp[t] = rb;
      if (t == nr - 1) rp[nr] = re;
      sums[t] = 0;
      mine = re - rb > 32 * kLanes;
    }
    const bool any = __any(mine);
    if ((t & 63) == 0) long_in[t >> 6] = any;
  } else {
    for (int k = t; k <= nr; k += kBlock) rp[k] = rptr[r0 + k];
  }
  const int row = t / kLanes, lane = t % kLanes;
  const int32_t zv = MODE != 0 && row < nr && lane == 0 ? z[r0 + row] : 0;
  __syncthreads();
  const int e0 = rp[0], e1 = rp[nr];
  const int b = row < nr ? rp[row] : e0, e = row < nr ? rp[row + 1] : e0;
  uint64_t acc = 0;
  int cc[kPer];
  int32_t vv[kPer];
  auto load = [&](int p0) {  // p0 < e1; no sum passes e1, so none overflows
    const int left = e1 - p0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int p = t + kBlock * j < left ? p0 + t + kBlock * j : e0;
      cc[j] = cind[p];
      vv[j] = val[p];
    }
  };
  if (e0 < e1) load(e0);
  bool any_long = false;
  if constexpr (kLong) {
    int any = 0;
#pragma unroll
    for (int k = 0; k < kBlock / 64; ++k) any |= long_in[k];
    any_long = __builtin_amdgcn_readfirstlane(any) != 0;
  }
  bool more = e0 < e1;
  for (int p0 = e0; more; p0 += kTile) {
    more = e1 - p0 > kTile;
    int32_t xx[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) xx[j] = x[cc[j]];
#pragma unroll
    for (int j = 0; j < kPer; ++j) prod[t + kBlock * j] = prod64(vv[j], xx[j]);
    if (more) load(p0 + kTile);
    lds_barrier();
    if (!kLong || !any_long) {
      const int lo = max(b - p0, 0), hi = min(e - p0, kTile);
      for (int q = lo + lane; q < hi; q += kLanes) acc += prod[q];
    } else {
      // rows that end after p0 from the first on, and those that begin in the tile
      int first = 0, last = 0;
#pragma unroll
      for (int k = 0; k < kRows; k += 64) {
        const int r = min(k + (t & 63), nr - 1);
        const bool mine = k + (t & 63) < nr;
        first += __popcll(__ballot(mine && rp[r + 1] <= p0));
        last += __popcll(__ballot(mine && rp[r] - p0 < kTile));
      }
      // 2^lg lanes for each of them (at least kLanes: there are kRows at most;
      // one or more, unless the row pointers do not ascend)
      const int lg = 31 - __clz(kBlock / max(last - first, 1));
      const int g = t >> lg, part = t & ((1 << lg) - 1);
      const int mine = min(first + g, nr - 1);
      const int lo = max(rp[mine] - p0, 0);
      const int hi = first + g < last ? min(rp[mine + 1] - p0, kTile) : 0;
      uint64_t s = 0;
      for (int q = lo + part; q < hi; q += 1 << lg) s += prod[q];
      for (int o = 1; o < min(1 << lg, 64); o *= 2) s += __shfl_xor(s, o, 64);
      if ((part & 63) == 0 && lo < hi) atomicAdd(&sums[mine], s);
    }
    lds_barrier();
  }
  if (kLong && any_long) acc = lane == 0 && row < nr ? sums[row] : 0;
  acc = group_sum<(kLanes < 16 ? kLanes : 16)>(acc);
#pragma unroll
  for (int o = 16; o < kLanes; o *= 2) acc += __shfl_xor(acc, o, 64);
  if (row < nr && lane == 0) {
    const int32_t s = low32(as_i64(acc) >> bit);
    if (MODE == 0) y[r0 + row] = s;
    else if (MODE == 1) y[r0 + row] = sub32(zv, s);
    else y[r0 + row] = add32(zv, s);
  }
}

// SELL-64 SpMV, one thread per row.  Entries are read eight at a time with
// clamped indices (every load unconditional), padding contributes nothing.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_sell_int(
    int n, const long long* __restrict__ soff, const int* __restrict__ scol,
    const int32_t* __restrict__ sval, const int* __restrict__ srow, int bit,
    const int32_t* __restrict__ x, const int32_t* z, int32_t* y, int remap) {
  const int row = (remap ? xcd_block() : static_cast<int>(blockIdx.x)) * kBlock + threadIdx.x;
  if (row >= n) return;
  const int orow = srow ? srow[row] : row;
  const int32_t zv = MODE != 0 ? z[orow] : 0;  // issued before the entries
  const long long b = soff[row >> 6];
  const int w = static_cast<int>((soff[(row >> 6) + 1] - b) >> 6);
  const int* c = scol + b + (row & 63);
  const int32_t* v = sval + b + (row & 63);
  uint64_t acc = 0;
  for (int k0 = 0; k0 < w; k0 += 8) {
    int cc[8];
    int32_t vv[8], xx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < w ? k0 + j : k0;
      cc[j] = c[64 * k];
      vv[j] = v[64 * k];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) xx[j] = x[cc[j] < 0 ? 0 : cc[j]];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < w) acc += prod64(vv[j], xx[j]);
  }
  const int32_t s = low32(as_i64(acc) >> bit);
  if (MODE == 0) y[orow] = s;
  else if (MODE == 1) y[orow] = sub32(zv, s);
  else y[orow] = add32(zv, s);
}

// SELL-64 integer SpMV with 16-bit column offsets: entry k of row r holds
// col - r (square matrices whose entries all lie within 32767 of the
// diagonal; padding is offset 0 with value 0, an exact zero product).  Six
// bytes per entry instead of eight.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_sell16_int(
    int n, const long long* __restrict__ soff, const int16_t* __restrict__ scol,
    const int32_t* __restrict__ sval, int bit, const int32_t* __restrict__ x, const int32_t* z,
    int32_t* y, int remap) {
  const int row = (remap ? xcd_block() : static_cast<int>(blockIdx.x)) * kBlock + threadIdx.x;
  if (row >= n) return;
  const int32_t zv = MODE != 0 ? z[row] : 0;  // issued before the entries
  const long long b = soff[row >> 6];
  const int w = static_cast<int>((soff[(row >> 6) + 1] - b) >> 6);
  const int16_t* c = scol + b + (row & 63);
  const int32_t* v = sval + b + (row & 63);
  uint64_t acc = 0;
  for (int k0 = 0; k0 < w; k0 += 8) {
    int cc[8];
    int32_t vv[8], xx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < w ? k0 + j : k0;
      cc[j] = row + c[64 * k];
      vv[j] = v[64 * k];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) xx[j] = x[cc[j]];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < w) acc += prod64(vv[j], xx[j]);
  }
  const int32_t s = low32(as_i64(acc) >> bit);
  if (MODE == 0) y[row] = s;
  else if (MODE == 1) y[row] = sub32(zv, s);
  else y[row] = add32(zv, s);
}

// FP SELL-64 SpMV: the row's products are added in stored (column) order,
// as the CSR kernel adds them; padding is skipped, not added.
template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_sell_fp(
    int n, const long long* __restrict__ soff, const int* __restrict__ scol,
    const T* __restrict__ sval, const int* __restrict__ srow, const T* __restrict__ x,
    const T* z, T* y, int remap) {
  const int row = (remap ? xcd_block() : static_cast<int>(blockIdx.x)) * kBlock + threadIdx.x;
  if (row >= n) return;
  const int orow = srow ? srow[row] : row;
  const T zv = MODE != 0 ? z[orow] : T(0);  // issued before the entries
  const long long b = soff[row >> 6];
  const int w = static_cast<int>((soff[(row >> 6) + 1] - b) >> 6);
  const int* c = scol + b + (row & 63);
  const T* v = sval + b + (row & 63);
  T t = 0;
  for (int k0 = 0; k0 < w; k0 += 8) {
    int cc[8];
    T vv[8], xx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int k = k0 + j < w ? k0 + j : k0;
      cc[j] = c[64 * k];
      vv[j] = v[64 * k];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) xx[j] = x[cc[j] < 0 ? 0 : cc[j]];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (k0 + j < w && cc[j] >= 0) t += vv[j] * xx[j];
  }
  if (MODE == 0) y[orow] = t;
  else if (MODE == 1) y[orow] = zv - t;
  else y[orow] = zv + t;
}

template <typename T, int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_fp(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind,
    const T* __restrict__ val, const T* __restrict__ x, const T* z, T* y, int remap) {
  const int row = (remap ? xcd_block() : static_cast<int>(blockIdx.x)) * kBlock + threadIdx.x;
  if (row >= n) return;
  T t = 0;
  const int rb = rptr[row], re = rptr[row + 1];
  // Eight entries at a time, every load unconditional (clamped), so that a
  // chunk costs two memory latencies; the sum keeps the stored order.
  for (int p0 = rb; p0 < re; p0 += 8) {
    int cc[8];
    T vv[8], xx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = p0 + j < re ? p0 + j : p0;
      cc[j] = cind[p];
      vv[j] = val[p];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) xx[j] = x[cc[j]];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (p0 + j < re) t += vv[j] * xx[j];
  }
  if (MODE == 0) y[row] = t;
  else if (MODE == 1) y[row] = z[row] - t;
  else y[row] = z[row] + t;
}

// FP CSR SpMV streamed through LDS: as k_spmv_stream_int, with one lane per row
// adding the row's products in stored order (16 read ahead of the additions);
// the rows are dealt over the four waves.  Two product tiles, so that the
// waves fill the next one while rows are still being added.  One lane per row
// reading its own entries (k_spmv_fp) waits for two dependent loads per eight
// entries: 3,520 rows of 440 entries took 153 us in FP64.
template <typename T, int kRows, int MODE>
__global__ __launch_bounds__(kBlock) void k_spmv_stream_fp(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind,
    const T* __restrict__ val, const T* __restrict__ x, const T* z, T* y) {
  constexpr int kPer = 8, kTile = kBlock * kPer, kRowsPerWave = kRows / 4, kAhead = 16;
  __shared__ T prod[2][kTile + kAhead];
  __shared__ int rp[kRows + 1];
  const int t = threadIdx.x;
  const int r0 = blockIdx.x * kRows, nr = min(kRows, n - r0);
  for (int k = t; k <= nr; k += kBlock) rp[k] = rptr[r0 + k];
  const int row = (t & 63) < kRowsPerWave ? (t >> 6) * kRowsPerWave + (t & 63) : kRows;
  const T zv = MODE != 0 && row < nr ? z[r0 + row] : T(0);
  __syncthreads();
  const int e0 = rp[0], e1 = rp[nr];
  const int b = row < nr ? rp[row] : e0, e = row < nr ? rp[row + 1] : e0;
  T sum = 0;
  int cc[kPer];
  T vv[kPer];
  auto load = [&](int p0) {  // p0 < e1; no sum passes e1, so none overflows
    const int left = e1 - p0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      const int p = t + kBlock * j < left ? p0 + t + kBlock * j : e0;
      cc[j] = cind[p];
      vv[j] = val[p];
    }
  };
  if (e0 < e1) load(e0);
  bool more = e0 < e1;
  int half = 0;
  for (int p0 = e0; more; p0 += kTile, half ^= 1) {
    more = e1 - p0 > kTile;
    T* pr = prod[half];
    T xx[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) xx[j] = x[cc[j]];
#pragma unroll
    for (int j = 0; j < kPer; ++j) pr[t + kBlock * j] = vv[j] * xx[j];
    if (more) load(p0 + kTile);
    // the other tile's rows were added before this barrier was reached
    lds_barrier();
    int q = max(b - p0, 0);
    const int hi = min(e - p0, kTile);
    T v[kAhead];
    if (q < hi) {
#pragma unroll
      for (int j = 0; j < kAhead; ++j) v[j] = pr[q + j];
      for (; q + kAhead <= hi; q += kAhead) {
        T w[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) w[j] = pr[min(q + kAhead, kTile) + j];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) sum = sum + v[j];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) v[j] = w[j];
      }
#pragma unroll
      for (int j = 0; j < kAhead; ++j) sum = q + j < hi ? sum + v[j] : sum;
    }
  }
  if (row < nr) {
    if (MODE == 0) y[r0 + row] = sum;
    else if (MODE == 1) y[r0 + row] = zv - sum;
    else y[r0 + row] = zv + sum;
  }
}

template <int G, int MODE>
hipError_t spmv_int_g(const DCsr& a, const void* x, const void* z, void* y,
                      hipStream_t s) {
  const long long threads = static_cast<long long>(a.n) * G;
  const int grid = static_cast<int>((threads + kBlock - 1) / kBlock);
  if (grid == 0) return hipSuccess;
  launch_timed(&k_spmv_int<G, MODE>, dim3(grid), dim3(kBlock), 0, s, a.n, a.rptr, a.cind,
               static_cast<const int32_t*>(a.val), a.bit, static_cast<const int32_t*>(x),
               static_cast<const int32_t*>(z), static_cast<int32_t*>(y), xcd_remap());
  return hipGetLastError();
}

template <int R, int MODE, bool kLong = false>
hipError_t spmv_stream_go(const DCsr& a, const void* x, const void* z, void* y, hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  launch_timed(&k_spmv_stream_int<R, MODE, kLong>, dim3((a.n + R - 1) / R), dim3(kBlock), 0, s, a.n,
               a.rptr, a.cind, static_cast<const int32_t*>(a.val), a.bit,
               static_cast<const int32_t*>(x), static_cast<const int32_t*>(z),
               static_cast<int32_t*>(y));
  return hipGetLastError();
}

template <int MODE>
hipError_t spmv_int_mode(const DCsr& a, const void* x, const void* z, void* y,
                         hipStream_t s) {
  switch (a.stream) {
    case 0: break;
    case 16: return spmv_stream_go<16, MODE>(a, x, z, y, s);
    case 32: return spmv_stream_go<32, MODE>(a, x, z, y, s);
    case 64: return spmv_stream_go<64, MODE>(a, x, z, y, s);
    case 128: return spmv_stream_go<128, MODE>(a, x, z, y, s);
    case 256: return spmv_stream_go<256, MODE>(a, x, z, y, s);
    default: return hipErrorInvalidValue;
  }
  switch (a.group) {
    case 1: return spmv_int_g<1, MODE>(a, x, z, y, s);
    case 2: return spmv_int_g<2, MODE>(a, x, z, y, s);
    case 4: return spmv_int_g<4, MODE>(a, x, z, y, s);
    case 8: return spmv_int_g<8, MODE>(a, x, z, y, s);
    case 16: return spmv_int_g<16, MODE>(a, x, z, y, s);
    case 32: return spmv_int_g<32, MODE>(a, x, z, y, s);
    default: return spmv_int_g<64, MODE>(a, x, z, y, s);
  }
}

template <typename T, int R, int MODE>
hipError_t spmv_stream_fp_go(const DCsr& a, const void* x, const void* z, void* y,
                             hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  launch_timed(&k_spmv_stream_fp<T, R, MODE>, dim3((a.n + R - 1) / R), dim3(kBlock), 0, s, a.n,
               a.rptr, a.cind, static_cast<const T*>(a.val), static_cast<const T*>(x),
               static_cast<const T*>(z), static_cast<T*>(y));
  return hipGetLastError();
}

template <typename T, int MODE>
hipError_t spmv_fp(const DCsr& a, const void* x, const void* z, void* y,
                   hipStream_t s) {
  switch (a.stream) {
    case 0: break;
    case 8: return spmv_stream_fp_go<T, 8, MODE>(a, x, z, y, s);
    case 16: return spmv_stream_fp_go<T, 16, MODE>(a, x, z, y, s);
    case 32: return spmv_stream_fp_go<T, 32, MODE>(a, x, z, y, s);
    case 64: return spmv_stream_fp_go<T, 64, MODE>(a, x, z, y, s);
    case 128: return spmv_stream_fp_go<T, 128, MODE>(a, x, z, y, s);
    default: return hipErrorInvalidValue;
  }
  const int grid = (a.n + kBlock - 1) / kBlock;
  if (grid == 0) return hipSuccess;
  launch_timed(&k_spmv_fp<T, MODE>, dim3(grid), dim3(kBlock), 0, s, a.n, a.rptr, a.cind,
               static_cast<const T*>(a.val), static_cast<const T*>(x),
               static_cast<const T*>(z), static_cast<T*>(y), xcd_remap());
  return hipGetLastError();
}

constexpr int kChainBlock = 512;

// ---- blocked single-workgroup solve for the coarsest grid ------------------
//
// The coarsest factors (n <= a few thousand, dense-ish after the complete LU)
// form one long dependency chain.  One workgroup keeps the solution and the
// row accumulators in LDS and walks 64-column blocks: the block's diagonal
// tile is solved by one wave as a column sweep (lane r owns row r; after
// column c is final it is broadcast and every dependent row subtracts its
// term), then all waves subtract the block's contributions from the rows
// still to come.  Each row thus receives its terms in the same column order
// as the sequential solve (ascending for L / LD, descending for DU), so FP
// results round exactly as the CPU's; integer sums are order-free anyway.
// bptr[i * (nb + 1) + b] is the first dependency entry of row i whose column
// is >= 64 b.

// Broadcast lane `src` (wave-uniform) to the whole wave with v_readlane.
template <typename T>
__device__ __forceinline__ T bcast_lane(T v, int src) {
  if constexpr (sizeof(T) == 4) {
    int x;
    __builtin_memcpy(&x, &v, 4);
    x = __builtin_amdgcn_readlane(x, src);
    T r;
    __builtin_memcpy(&r, &x, 4);
    return r;
  } else {
    int x[2];
    __builtin_memcpy(x, &v, 8);
    x[0] = __builtin_amdgcn_readlane(x[0], src);
    x[1] = __builtin_amdgcn_readlane(x[1], src);
    T r;
    __builtin_memcpy(&r, x, 8);
    return r;
  }
}

template <typename T, TriKind K>
__global__ __launch_bounds__(kBlkThreads) void k_tri_blocked(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind, const void* valv,
    int bit, int dbit, const int* __restrict__ bptr, int nb, const T* __restrict__ in,
    T* __restrict__ out) {
  using Acc = typename AccOf<T>::type;
  extern __shared__ __align__(16) unsigned char smem[];
  Acc* acc = reinterpret_cast<Acc*>(smem);
  T* xs = reinterpret_cast<T*>(acc + n);
  T* dinv = xs + n;
  uint64_t* msk = reinterpret_cast<uint64_t*>(
      (reinterpret_cast<uintptr_t>(dinv + n) + 15) & ~static_cast<uintptr_t>(15));
  T* tile = reinterpret_cast<T*>(msk + kTB);
  const T* val = static_cast<const T*>(valv);
  constexpr bool fwd = (K != TriKind::kDU);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  constexpr int nw = kBlkThreads / 64;
  const int stride_b = nb + 1;
  for (int i = tid; i < n; i += kBlkThreads) {
    acc[i] = acc_init<T>(in[i], bit);
    if (K == TriKind::kLD) dinv[i] = val[rptr[i + 1] - 1];
    if (K == TriKind::kDU) dinv[i] = val[rptr[i]];
  }
  __syncthreads();
  for (int q = 0; q < nb; ++q) {
    const int b = fwd ? q : nb - 1 - q;
    const int r0 = b * kTB;
    const int r1 = min(r0 + kTB, n);
    const int rows = r1 - r0;
    // (a) the diagonal tile: dependency entries of rows r0..r1-1 in block b
    for (int rr = wid; rr < rows; rr += nw) {
      const int i = r0 + rr;
      const int pb = bptr[i * stride_b + b], pe = bptr[i * stride_b + b + 1];
      const int p = pb + lane;
      uint64_t bitv = 0;
      if (p < pe) {
        const int c = cind[p] - r0;
        tile[c * kTB + rr] = val[p];
        bitv = 1ull << c;
      }
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) bitv |= shfl_xor_u64(bitv, m);
      if (lane == 0) msk[rr] = bitv;
    }
    __syncthreads();
    // (b) one wave: column sweep over the tile
    if (wid == 0) {
      Acc t = lane < rows ? acc[r0 + lane] : Acc(0);
      const uint64_t mine = lane < rows ? msk[lane] : 0;
      const T dv = lane < rows ? dinv[r0 + lane] : T(0);
      T xv = 0;
      for (int st = 0; st < rows; ++st) {
        const int c = fwd ? st : rows - 1 - st;
        T xl = 0;
        if (lane == c) {
          xl = acc_final<T, K>(t, dv, bit, dbit);
          xv = xl;
        }
        const T xc = bcast_lane<T>(xl, c);
        if ((mine >> c) & 1ull) t = acc_sub<T>(t, tile[c * kTB + lane], xc);
      }
      if (lane < rows) {
        xs[r0 + lane] = xv;
        out[r0 + lane] = xv;
      }
    }
    __syncthreads();
    // (c) all waves: rows still to come take block b's terms
    const int lo = fwd ? r1 : 0;
    const int hi = fwd ? n : r0;
    for (int i = lo + tid; i < hi; i += kBlkThreads) {
      const int pb = bptr[i * stride_b + b], pe = bptr[i * stride_b + b + 1];
      if (pb == pe) continue;
      Acc t = acc[i];
      // batches of kBatch independent loads, applied in the row's order
      constexpr int kBatch = 8;
      const int cnt = pe - pb;
      for (int q0 = 0; q0 < cnt; q0 += kBatch) {
        T vv[kBatch];
        int cc[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          const int q = q0 + u;
          if (q < cnt) {
            const int p = fwd ? pb + q : pe - 1 - q;
            vv[u] = val[p];
            cc[u] = cind[p];
          }
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
          if (q0 + u < cnt) t = acc_sub<T>(t, vv[u], xs[cc[u]]);
      }
      acc[i] = t;
    }
    __syncthreads();
  }
}

// Integer version of the blocked solve.  Integer row sums are order-free, so
// (i) the sweeping wave keeps its row's 64 tile values in registers and the
// 64-step sweep is fully unrolled, and (ii) the off-block update gives each
// row a whole wave: lane q takes the row's q-th entry in the block and the
// wave sums the products.
template <TriKind K>
__global__ __launch_bounds__(kBlkThreads) void k_tri_blocked_int(
    int n, const int* __restrict__ rptr, const int* __restrict__ cind,
    const int32_t* __restrict__ val, int bit, int dbit, const int* __restrict__ bptr,
    int nb, const int32_t* __restrict__ in, int32_t* __restrict__ out) {
  extern __shared__ __align__(16) unsigned char smem[];
  uint64_t* acc = reinterpret_cast<uint64_t*>(smem);
  int32_t* xs = reinterpret_cast<int32_t*>(acc + n);
  int32_t* dinv = xs + n;
  int32_t* tile = reinterpret_cast<int32_t*>(
      (reinterpret_cast<uintptr_t>(dinv + n) + 15) & ~static_cast<uintptr_t>(15));
  constexpr bool fwd = (K != TriKind::kDU);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  constexpr int nw = kBlkThreads / 64;
  const int stride_b = nb + 1;
  for (int i = tid; i < n; i += kBlkThreads) {
    acc[i] = static_cast<uint64_t>(static_cast<int64_t>(in[i])) << bit;
    if (K == TriKind::kLD) dinv[i] = val[rptr[i + 1] - 1];
    if (K == TriKind::kDU) dinv[i] = val[rptr[i]];
  }
  __syncthreads();
  for (int q = 0; q < nb; ++q) {
    const int b = fwd ? q : nb - 1 - q;
    const int r0 = b * kTB;
    const int r1 = min(r0 + kTB, n);
    const int rows = r1 - r0;
    // (a) the diagonal tile, column-major, zero where no entry
    for (int idx = tid; idx < kTB * kTB; idx += kBlkThreads) tile[idx] = 0;
    __syncthreads();
    for (int rr = wid; rr < rows; rr += nw) {
      const int i = r0 + rr;
      const int pb = bptr[i * stride_b + b], pe = bptr[i * stride_b + b + 1];
      const int p = pb + lane;
      if (p < pe) tile[(cind[p] - r0) * kTB + rr] = val[p];
    }
    __syncthreads();
    // (b) one wave sweeps the tile with its operands in registers
    if (wid == 0) {
      int32_t reg[kTB];
#pragma unroll
      for (int c = 0; c < kTB; ++c) reg[c] = tile[c * kTB + lane];
      uint64_t t = lane < rows ? acc[r0 + lane] : 0;
      const int32_t dv = lane < rows ? dinv[r0 + lane] : 0;
      int32_t xv = 0;
#pragma unroll
      for (int st = 0; st < kTB; ++st) {
        const int c = fwd ? st : kTB - 1 - st;
        if (c < rows) {
          const int32_t mine = acc_final<int32_t, K>(t, dv, bit, dbit);
          if (lane == c) xv = mine;
          const int32_t xc = __builtin_amdgcn_readlane(mine, c);
          t -= prod64(reg[c], xc);
        }
      }
      if (lane < rows) {
        xs[r0 + lane] = xv;
        out[r0 + lane] = xv;
      }
    }
    __syncthreads();
    // (c) one wave per remaining row
    const int lo = fwd ? r1 : 0;
    const int hi = fwd ? n : r0;
    for (int i = lo + wid; i < hi; i += nw) {
      const int pb = bptr[i * stride_b + b], pe = bptr[i * stride_b + b + 1];
      if (pb == pe) continue;
      const int p = pb + lane;
      uint64_t prod = 0;
      if (p < pe) prod = prod64(val[p], xs[cind[p]]);
      prod = wave_sum_u64(prod);
      if (lane == 0) acc[i] -= prod;
    }
    __syncthreads();
  }
}

// low32(mul_wrap(t >> bit, dinv) >> dbit) for shifts 0..31.  With q = t >> bit
// as words qhi:qlo and dinv read as unsigned u = dinv + 2^32 [dinv < 0], the
// low 64 bits of q dinv are qlo u plus, in the high word, qhi u - qlo
// [dinv < 0]; the two products and the correction do not wait for each other.
__device__ __forceinline__ int32_t rp_finish(uint64_t t, int32_t dinv, int bit, int dbit) {
  const unsigned lo = static_cast<unsigned>(t), hi = static_cast<unsigned>(t >> 32);
  const unsigned neg = static_cast<unsigned>(dinv >> 31);
  const unsigned qlo = __builtin_amdgcn_alignbit(hi, lo, static_cast<unsigned>(bit));
  const unsigned qhi = static_cast<unsigned>(static_cast<int>(hi) >> bit);
  unsigned m;  // opaque: folded into the other product it would wait for it
  asm("v_mul_lo_u32 %0, %1, %2" : "=v"(m) : "v"(qhi), "v"(dinv));
  const uint64_t p = static_cast<uint64_t>(qlo) * static_cast<unsigned>(dinv);
  const unsigned ph = static_cast<unsigned>(p >> 32) + m + ((0u - qlo) & neg);
  return static_cast<int32_t>(
      __builtin_amdgcn_alignbit(ph, static_cast<unsigned>(p), static_cast<unsigned>(dbit)));
}

// Tiled coarse solve (integer and FP), one wave per 64-row block, kB
// consecutive blocks per workgroup.  A block's factor entries are stored as
// dense 64 x 64 tiles, column-major (entry (row r, column c) of a tile at c *
// 64 + r), in processing order: the off-diagonal tiles of the blocks it
// depends on (forward: 0 .. b-1; backward: nb-1 .. b+1), then its diagonal
// tile.  Lane r owns row r and subtracts its terms column by column in that
// order, the sequential solve's (ascending columns for L, descending for DU),
// so FP sums round as the CPU's; integer sums are order-free.  FP: the product
// of an entry absent from the factor (a clear bit of the row's 64-bit mask per
// tile) is masked to +0, which leaves the sum unchanged, so only the
// subtractions form a chain.
//
// A solved row is published as one 64-bit word {epoch, value} (FP64: two, for
// the value's halves) in xp, an agent-scope atomic store, so a consumer learns
// that a value is ready and reads it in the same load; two polls are in flight,
// so the words are seen about half a round trip sooner.  Inside a workgroup
// the values go through LDS: wave q sweeps its diagonal tile (at step c lane c
// finishes its row and the value is broadcast), then the later waves subtract
// its block's terms; the tiles among a workgroup's blocks wait in LDS.  The
// tile of the next outside dependency is loaded into the registers of the
// columns just used, so its latency is covered by the wait.
//
// What bounds it is the chain: per block the sweep's 64 dependent steps and a
// tile product, plus per workgroup one hand-off through memory.  With a
// workgroup per block, its four waves sharing the products, every block paid
// the hand-off (integer, 128^3: 83 + 105 us per solve, now 60 + 82; FP64, 96^3: 30
// blocks, 187 + 190 us, now 92 + 93; FP32, 48^3: 89 + 89, now 43 + 43).
//
// Workgroups take their blocks (and right-hand side) from a ticket counter in
// processing order, so a workgroup only ever waits for workgroups that started
// before it, whatever order the hardware starts them in and whatever else
// shares the GPU.  A launch that runs out of its wait budget (tile_wait_over)
// records an error and gives up instead of hanging.
template <typename T>
__device__ __forceinline__ T readlane_of(T v, int src);
template <>
__device__ __forceinline__ double readlane_of<double>(double v, int src) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned long long>(b)), src);
  const int hi = __builtin_amdgcn_readlane(static_cast<int>(static_cast<unsigned long long>(b) >> 32), src);
  return __longlong_as_double(static_cast<long long>(
      (static_cast<unsigned long long>(static_cast<unsigned>(hi)) << 32) | static_cast<unsigned>(lo)));
}
template <>
__device__ __forceinline__ float readlane_of<float>(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}
template <>
__device__ __forceinline__ int32_t readlane_of<int32_t>(int32_t v, int src) {
  return __builtin_amdgcn_readlane(v, src);
}

// t - v x where bit `c` of the row's mask is set (FP); integer tiles hold
// negated values, zero where the factor has no entry: t + v x
__device__ __forceinline__ uint64_t tile_sub(uint64_t t, int32_t v, int32_t x, uint64_t, int) {
  return t + prod64(v, x);
}
__device__ __forceinline__ float tile_sub(float t, float v, float x, uint64_t mask, int c) {
  const unsigned w = static_cast<unsigned>(c < 32 ? mask : mask >> 32);
  const int m = __builtin_amdgcn_sbfe(static_cast<int>(w), c % 32, 1);
  return t - __int_as_float(__float_as_int(v * x) & m);
}
__device__ __forceinline__ double tile_sub(double t, double v, double x, uint64_t mask, int c) {
  const unsigned w = static_cast<unsigned>(c < 32 ? mask : mask >> 32);
  const int m = __builtin_amdgcn_sbfe(static_cast<int>(w), c % 32, 1);
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v * x));
  const unsigned lo = static_cast<unsigned>(b) & m, hi = static_cast<unsigned>(b >> 32) & m;
  return t - __longlong_as_double(
                 static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// The row's value; kShort: integer shifts of 0..31 (a shorter chain).
template <typename T, TriKind K, bool kShort>
__device__ __forceinline__ T tile_finish(typename AccOf<T>::type t, T dinv, int bit, int dbit) {
  if constexpr (std::is_same_v<T, int32_t> && kShort) {
    if constexpr (K == TriKind::kL)
      return static_cast<int32_t>(__builtin_amdgcn_alignbit(
          static_cast<unsigned>(t >> 32), static_cast<unsigned>(t), static_cast<unsigned>(bit)));
    else
      return rp_finish(t, dinv, bit, dbit);
  } else {
    return acc_final<T, K>(t, dinv, bit, dbit);
  }
}

// kS: 1 for plain vectors; 4 for a block of nrhs right-hand sides (element
// (row i, right-hand side r) at ((r / 4) n + i) 4 + r % 4).
template <typename T, TriKind K, bool kShort, int kS, int kB>
__global__ __launch_bounds__(64 * kB) void k_tri_tiles(
    int n, int nb, int nrhs, const T* __restrict__ tiles, const long long* __restrict__ toff,
    const uint64_t* __restrict__ tmask, const T* __restrict__ dinv_g, int bit, int dbit,
    const T* __restrict__ in_all, T* out_all, unsigned long long* xp_all, int epoch, int* err,
    unsigned* tickets) {
  constexpr bool fwd = (K != TriKind::kDU), kFp = !std::is_same_v<T, int32_t>;
  constexpr int kW = sizeof(T) / 4;  // published words per row
  // wave w's tiles against the workgroup's blocks 0 .. w (its diagonal tile
  // last), column-major: lane r reads only row r's values
  extern __shared__ __align__(16) unsigned char smem_t[];
  __shared__ T xs[kB][kTB];
  __shared__ int ticket_sh;
  const long long t0 = wall_clock64();
  const int ticket = tile_ticket(tickets, &ticket_sh);
  const int group = ticket / nrhs, r = ticket % nrhs;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int first = group * kB;  // dependencies of earlier workgroups
  const int pb = first + w;      // place in processing order = dependencies
  const bool valid = pb < nb;
  const int b = !valid ? 0 : fwd ? pb : nb - 1 - pb;
  const size_t off = kS == 1 ? 0 : static_cast<size_t>(r >> 2) * n * 4 + (r & 3);
  const T* in = in_all + off;
  T* out = out_all + off;
  unsigned long long* xp = xp_all + static_cast<size_t>(r) * n * kW;
  const int r0 = b * kTB;
  const int rows = valid ? min(kTB, n - r0) : 0;
  const T* Tb = tiles + toff[b];
  const uint64_t* Mb = kFp ? tmask + toff[b] / kTB : nullptr;  // one mask per tile row
  T* mine_lds = reinterpret_cast<T*>(smem_t) + static_cast<size_t>(w * (w + 1) / 2) * (kTB * kTB);
  uint64_t mi[kB];  // masks of the tiles in LDS
#pragma unroll
  for (int q = 0; q < kB; ++q) mi[q] = 0;
  if (valid) {
#pragma unroll
    for (int q = 0; q < kB; ++q)
      if (q <= w) {
        const T* Tq = Tb + static_cast<size_t>(first + q) * (kTB * kTB);
#pragma unroll 16
        for (int c = 0; c < kTB; ++c)
          mine_lds[(q * kTB + c) * kTB + lane] = Tq[c * kTB + lane];
        if (kFp) mi[q] = Mb[static_cast<size_t>(first + q) * kTB + lane];
      }
  }
  const T dv = (K != TriKind::kL && lane < rows) ? dinv_g[r0 + lane] : T(0);
  typename AccOf<T>::type t =
      acc_init<T>(lane < rows ? in[static_cast<size_t>(r0 + lane) * kS] : T(0), bit);
  // vk: the current outside dependency's tile (without one: any, unused)
  T vk[kTB];
#pragma unroll
  for (int c = 0; c < kTB; ++c) vk[c] = Tb[c * kTB + lane];
  uint64_t mk = kFp ? Mb[lane] : 0;
  const unsigned long long tag = static_cast<unsigned long long>(static_cast<unsigned>(epoch))
                                 << 32;
  for (int k = 0; k < (valid ? first : 0); ++k) {
    // every lane loads (rows past the end the last row's words, which no entry
    // names): a load under a divergent branch would make the compiler wait
    // for both polls where the paths join
    const int row = min((fwd ? k : nb - 1 - k) * kTB + lane, n - 1);
    struct Words {
      unsigned long long w[kW];
    };
    auto poll = [&]() {
      Words u;
#pragma unroll
      for (int q = 0; q < kW; ++q)
        u.w[q] = __hip_atomic_load(&xp[kW * row + q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return u;
    };
    auto ready = [&](const Words& u) {
      bool ok = true;
#pragma unroll
      for (int q = 0; q < kW; ++q) ok = ok && (u.w[q] >> 32) == (tag >> 32);
      return __all(ok);
    };
    Words v, va = poll();
    int spins = 0;
    while (true) {
      __builtin_amdgcn_s_sleep(1);
      const Words vb = poll();
      if (ready(va)) {
        v = va;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
      va = poll();
      if (ready(vb)) {
        v = vb;
        break;
      }
      if ((++spins & 15) == 0 && tile_wait_over(t0, err)) {
        if (lane == 0) atomicAdd(err, 1);
        v = vb;
        break;
      }
    }
    T x;
    if constexpr (kW == 2)
      x = __longlong_as_double(
          static_cast<long long>((v.w[1] << 32) | static_cast<unsigned>(v.w[0])));
    else if constexpr (kFp)
      x = __uint_as_float(static_cast<unsigned>(v.w[0]));
    else
      x = static_cast<int32_t>(static_cast<unsigned>(v.w[0]));
    // the terms of dependency k; the next one's tile replaces this one's
    const size_t nx = static_cast<size_t>(min(k + 1, first - 1));
    const T* Tn = Tb + nx * (kTB * kTB);
    const uint64_t mn = kFp ? Mb[nx * kTB + lane] : 0;
#pragma unroll
    for (int st = 0; st < kTB; ++st) {
      const int c = fwd ? st : kTB - 1 - st;
      t = tile_sub(t, vk[c], readlane_of<T>(x, c), mk, c);
      vk[c] = Tn[c * kTB + lane];
    }
    mk = mn;
  }
#pragma unroll
  for (int q = 0; q < kB; ++q) {
    if (w == q && valid) {
#pragma unroll
      for (int st = 0; st < kTB; ++st) {
        // no test for rows past the end, whose values are zero and which no
        // entry names: a branch per step would keep the tile's LDS reads from
        // being issued ahead
        const int c = fwd ? st : kTB - 1 - st;
        const T mine = tile_finish<T, K, kShort>(t, dv, bit, dbit);
        t = tile_sub(t, mine_lds[(q * kTB + c) * kTB + lane], readlane_of<T>(mine, c), mi[q], c);
      }
      // a row has no entries at its own step or later: its sum still stands
      const T xv = tile_finish<T, K, kShort>(t, dv, bit, dbit);
      xs[q][lane] = xv;
      if (lane < rows) {
        unsigned long long bits;
        if constexpr (kW == 2) bits = static_cast<unsigned long long>(__double_as_longlong(xv));
        else if constexpr (kFp) bits = __float_as_uint(xv);
        else bits = static_cast<uint32_t>(xv);
#pragma unroll
        for (int h = 0; h < kW; ++h)
          __hip_atomic_store(&xp[kW * (r0 + lane) + h],
                             tag | static_cast<uint32_t>(bits >> (32 * h)), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        out[static_cast<size_t>(r0 + lane) * kS] = xv;
      }
    }
    if (q + 1 == kB) break;
    lds_barrier();
    if (w > q && valid) {
      const T x = xs[q][lane];
#pragma unroll
      for (int st = 0; st < kTB; ++st) {
        const int c = fwd ? st : kTB - 1 - st;
        t = tile_sub(t, mine_lds[(q * kTB + c) * kTB + lane], readlane_of<T>(x, c), mi[q], c);
      }
    }
  }
  tile_done(tickets, (nb + kB - 1) / kB * nrhs);
}

template <typename T, TriKind K>
hipError_t tri_blocked(const DCsr& a, const int* bptr, int nb, const void* in, void* out,
                       hipStream_t s) {
  if (a.n <= 0) return hipSuccess;
  if constexpr (std::is_same_v<T, int32_t>) {
    const size_t lds = tri_blocked_lds(a.n, 4, 8);
    static bool attr_i = false;
    if (!attr_i) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tri_blocked_int<K>),
                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                         static_cast<int>(kTriBlockedMaxLds));
      if (e != hipSuccess) return e;
      attr_i = true;
    }
    hipLaunchKernelGGL((k_tri_blocked_int<K>), dim3(1), dim3(kBlkThreads), lds, s, a.n,
                       a.rptr, a.cind, static_cast<const int32_t*>(a.val), a.bit, a.dbit,
                       bptr, nb, static_cast<const int32_t*>(in), static_cast<int32_t*>(out));
    return hipGetLastError();
  }
  const size_t lds = tri_blocked_lds(a.n, sizeof(T), sizeof(typename AccOf<T>::type));
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tri_blocked<T, K>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(kTriBlockedMaxLds));
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL((k_tri_blocked<T, K>), dim3(1), dim3(kBlkThreads), lds, s, a.n, a.rptr,
                     a.cind, a.val, a.bit, a.dbit, bptr, nb, static_cast<const T*>(in),
                     static_cast<T*>(out));
  return hipGetLastError();
}

// ---- level-ordered chain solve with prefetch ---------------------------------
//
// The factor is re-laid out in level order: position idx holds row lrow[idx]
// with its dependency entries lcol/lval[lbeg[idx] .. lbeg[idx+1]) in the order
// the sequential solve subtracts them, and its stored inverse diagonal in
// ldiag[idx].  One workgroup walks the levels of one chain; while level L is
// being computed, the row data of level L+1 (which does not depend on the
// solution) is already loaded into registers, so the only loads left on the
// critical path are the solution values of earlier levels.  When the chain's
// rows fit, its solution is also kept in LDS.

constexpr int kPre = 8;  // dependency entries held in registers per row

// The first kPre dependency entries of position idx are also stored with a
// fixed stride (ecol / eval[idx * kPre + q]), so every load of a row's data
// depends only on idx; entries beyond kPre are read from lcol / lval.
template <typename T>
struct PreRow {
  int row = -1, beg = 0, end = 0;
  T in = 0, dinv = 0;
  int col[kPre];
  T val[kPre];
};

template <typename T, TriKind K>
__device__ __forceinline__ void pre_meta(PreRow<T>& r, int idx, int lim,
                                         const int* __restrict__ lrow,
                                         const int* __restrict__ lbeg,
                                         const int* __restrict__ ecol,
                                         const T* __restrict__ eval,
                                         const T* __restrict__ ldiag) {
  if (idx >= lim) {
    r.row = -1;
    return;
  }
  r.row = lrow[idx];
  r.beg = lbeg[idx];
  r.end = lbeg[idx + 1];
  if (K != TriKind::kL) r.dinv = ldiag[idx];
#pragma unroll
  for (int q = 0; q < kPre; ++q) {
    r.col[q] = ecol[static_cast<size_t>(idx) * kPre + q];
    r.val[q] = eval[static_cast<size_t>(idx) * kPre + q];
  }
}

template <typename T>
__device__ __forceinline__ void pre_in(PreRow<T>& r, const T* __restrict__ in) {
  if (r.row >= 0) r.in = in[r.row];
}

template <typename T, TriKind K, bool kRing>
__device__ __forceinline__ T pre_eval(const PreRow<T>& r, int bit, int dbit,
                                      const int* __restrict__ lcol,
                                      const T* __restrict__ lval, const T* out,
                                      const T* ring, int rmask) {
  using Acc = typename AccOf<T>::type;
  Acc t = acc_init<T>(r.in, bit);
  // kRing: entries name dependency positions, whose values sit in the LDS ring
  auto X = [&](int c) -> T { return kRing ? ring[c & rmask] : out[c]; };
  const int cnt = r.end - r.beg;
#pragma unroll
  for (int q = 0; q < kPre; ++q)
    if (q < cnt) t = acc_sub<T>(t, r.val[q], X(r.col[q]));
  for (int p = r.beg + kPre; p < r.end; ++p) t = acc_sub<T>(t, lval[p], X(lcol[p]));
  return acc_final<T, K>(t, r.dinv, bit, dbit);
}


// kRing: dependency entries hold level-ordered positions; the values of the
// last rmask+1 positions of the chain live in an LDS ring (the host checks
// that no dependency reaches further back than that).  Otherwise entries hold
// row indices and values are read back from `out` after a full barrier.
template <typename T, TriKind K, bool kRing>
__global__ __launch_bounds__(kChainBlock) void k_tri_chain_pre(
    const int* __restrict__ lrow, const int* __restrict__ lbeg,
    const int* __restrict__ lcol, const T* __restrict__ lval,
    const int* __restrict__ ecol, const T* __restrict__ eval,
    const T* __restrict__ ldiag, int bit, int dbit, const int* __restrict__ lev_ptr,
    const int* __restrict__ chain_lev, int rmask, const T* __restrict__ in, T* out) {
  extern __shared__ __align__(16) unsigned char smem_c[];
  T* ring = reinterpret_cast<T*>(smem_c);
  const int lb = chain_lev[2 * blockIdx.x], le = chain_lev[2 * blockIdx.x + 1];
  const int tid = threadIdx.x;
  // pipeline: nxt = level L+1 (metadata and input), far = level L+2 (metadata)
  PreRow<T> nxt, far;
  if (lb < le) {
    pre_meta<T, K>(nxt, lev_ptr[lb] + tid, lev_ptr[lb + 1], lrow, lbeg, ecol, eval, ldiag);
    pre_in<T>(nxt, in);
  }
  if (lb + 1 < le)
    pre_meta<T, K>(far, lev_ptr[lb + 1] + tid, lev_ptr[lb + 2], lrow, lbeg, ecol, eval,
                   ldiag);
  for (int L = lb; L < le; ++L) {
    const PreRow<T> cur = nxt;
    const int s = lev_ptr[L], e = lev_ptr[L + 1];
    if (L + 1 < le) {
      nxt = far;
      pre_in<T>(nxt, in);
    }
    if (L + 2 < le)
      pre_meta<T, K>(far, lev_ptr[L + 2] + tid, lev_ptr[L + 3], lrow, lbeg, ecol, eval,
                     ldiag);
    if (cur.row >= 0) {
      const T v = pre_eval<T, K, kRing>(cur, bit, dbit, lcol, lval, out, ring, rmask);
      out[cur.row] = v;
      if (kRing) ring[(s + tid) & rmask] = v;
    }
    // rows beyond one per thread (large levels)
    for (int idx = s + kChainBlock + tid; idx < e; idx += kChainBlock) {
      PreRow<T> r;
      pre_meta<T, K>(r, idx, e, lrow, lbeg, ecol, eval, ldiag);
      pre_in<T>(r, in);
      const T v = pre_eval<T, K, kRing>(r, bit, dbit, lcol, lval, out, ring, rmask);
      out[r.row] = v;
      if (kRing) ring[idx & rmask] = v;
    }
    if (kRing)
      lds_barrier();
    else
      __syncthreads();
  }
}

// ---- entry-parallel chain solve (integer factors, LDS ring) -------------------
//
// For integer factors a row's sum is order-free, so the dependency entries of
// a whole level (contiguous in the level-ordered layout) are spread over the
// lanes: each lane multiplies its entries by solution values and adds the
// products into the row's LDS accumulator with 64-bit LDS atomics; then one
// lane per row finishes the row.  The factor is numbered in level order (row
// = position), so a level's right-hand sides, inverse diagonals and results
// are contiguous.
//
// Entries are packed as int4 {dep, val, slot, 0}: dep >= 0 is the position of
// a dependency whose value sits in the LDS ring; dep < 0 (kFar kernels only)
// names position -dep-1, a dependency at least kEpFarLevels levels back that
// the ring cannot hold, read from `out` in global memory.  A full workgroup
// fence every kEpFence levels makes such values visible before any load of
// them is issued.  The chain's level offsets are staged in LDS, so the loads
// of a level depend only on LDS data: entries, right-hand sides and inverse
// diagonals of level L + kD are loaded once level L is done (into the
// registers it has just freed), far values of level L + kEpFarAhead (whose
// addresses need the entries) at the start of level L.  Every load is issued
// unconditionally (lanes past a level's end read element 0 and ignore it):
// loads under divergent branches make the compiler wait for all outstanding
// loads at the join.

// Prefetch distance kD in levels: 4 for the wide register layout (8 entries,
// 2 rows per lane), 8 for the narrow one (4 entries, 1 row), whose buffers
// are half the size.  A level costs at least the global-load latency / kD.
constexpr int kEpFarAhead = 2;  // far-value distance in levels
constexpr int kEpFence = 32;    // full fence period in levels (kFar kernels)
static_assert(kEpFarAhead < 4, "far values need their entries loaded first");
static_assert(kEpFarLevels >= kEpFarAhead + kEpFence,
              "far dependencies must be fenced before their values are loaded");

template <int kE, int kR>
struct EpPre {
  int2 lo, hi;  // the level's {position, entry} bounds
  int dep[kE];
  int32_t val[kE];
  int slot[kE];
  int32_t xfar[kE];
  int32_t dinv[kR];
  int32_t in[kR];
};

template <int kThreads, int kE, int kR>
__device__ __forceinline__ void ep_load(EpPre<kE, kR>& r, int2 lo, int2 hi,
                                        const int4* __restrict__ lent,
                                        const int32_t* __restrict__ dinv,
                                        const int32_t* __restrict__ in) {
  const int t = threadIdx.x;
  r.lo = lo;
  r.hi = hi;
#pragma unroll
  for (int q = 0; q < kE; ++q) {
    const int p = lo.y + t + q * kThreads;
    const int4 w = lent[p < hi.y ? p : 0];
    r.dep[q] = w.x;
    r.val[q] = w.y;
    r.slot[q] = w.z;
  }
#pragma unroll
  for (int q = 0; q < kR; ++q) {
    const int idx = lo.x + t + q * kThreads;
    const int id = idx < hi.x ? idx : 0;
    r.dinv[q] = dinv[id];
    r.in[q] = in[id];
  }
}

template <int kThreads, int kE, int kR>
__device__ __forceinline__ void ep_far(EpPre<kE, kR>& r, const int32_t* out) {
  const int t = threadIdx.x;
#pragma unroll
  for (int q = 0; q < kE; ++q) {
    const int p = r.lo.y + t + q * kThreads;
    const int d = r.dep[q];
    r.xfar[q] = out[(p < r.hi.y && d < 0) ? -d - 1 : 0];
  }
}


struct EpShared {
  const int2* lvo;  // level offsets {position, entry}, LDS
  uint64_t* acc;    // accumulators, then kEpDummy slots for lanes past a level's end
  int32_t* ring;
  int rmask;
  int dummy;        // index of the first dummy slot
};

// One level of the chain; `cur` holds the level's prefetched data, `ahead`
// the buffer of level L + kEpFarAhead.  Level indices past the chain's end
// are clamped to an empty level.  kC accumulator copies per row: lane t adds
// into copy t % kC of its entry's row; the row's thread sums the copies.
template <TriKind K, int kWaves, bool kFar, int kE, int kR, int kC, int kD>
__device__ __forceinline__ void ep_level(EpPre<kE, kR>& cur, EpPre<kE, kR>& ahead, int L,
                                         int nl, const EpShared& sh,
                                         const int4* __restrict__ lent,
                                         const int32_t* __restrict__ dinv,
                                         const int32_t* __restrict__ in, int32_t* out, int bit,
                                         int dbit) {
  constexpr int kThreads = 64 * kWaves;
  const int t = threadIdx.x;
  const int s = cur.lo.x, e = cur.hi.x, e0 = cur.lo.y, e1 = cur.hi.y;
  uint64_t* acc = sh.acc;
  int32_t* ring = sh.ring;
  const int rmask = sh.rmask;
  const int cp = t & (kC - 1);
  // Offsets of the level prefetched at the end of this one, read now so
  // their LDS latency overlaps this level's work.
  const int Lp = min(L + kD, nl);
  const int2 plo = sh.lvo[Lp], phi = sh.lvo[min(Lp + 1, nl)];
  if (kFar) ep_far<kThreads>(ahead, out);
  // All ring reads first (lanes past the level's end read a valid, unused
  // slot), then the atomics: one LDS round trip for the whole level.
  int32_t xv[kE];
#pragma unroll
  for (int q = 0; q < kE; ++q) xv[q] = ring[cur.dep[q] & rmask];
  if (kFar) {
    // Far values are rare; waiting for their loads only where a lane of
    // the wave has one keeps the other levels off the global-load latency.
#pragma unroll
    for (int q = 0; q < kE; ++q)
      if (__any(cur.dep[q] < 0)) xv[q] = cur.dep[q] < 0 ? cur.xfar[q] : xv[q];
  }
  // Unconditional atomics: lanes past the level's end add into a dummy slot
  // of their own, which keeps the LDS traffic free of branches and waits.
#pragma unroll
  for (int q = 0; q < kE; ++q) {
    const int p = e0 + t + q * kThreads;
    const int a = p < e1 ? cur.slot[q] * kC + cp : sh.dummy + (t & (kEpDummy - 1));
    atomicAdd(reinterpret_cast<unsigned long long*>(&acc[a]),
              static_cast<unsigned long long>(prod64(cur.val[q], xv[q])));
  }
  for (int p = e0 + t + kE * kThreads; p < e1; p += kThreads) {
    const int4 w = lent[p];
    const int32_t x = (kFar && w.x < 0) ? out[-w.x - 1] : ring[w.x & rmask];
    atomicAdd(reinterpret_cast<unsigned long long*>(&acc[w.z * kC + cp]),
              static_cast<unsigned long long>(prod64(w.y, x)));
  }
  ep_sync<kWaves>();
  uint64_t av[kR];
  if (kC == 1) {
#pragma unroll
    for (int q = 0; q < kR; ++q) av[q] = acc[t + q * kThreads];
  } else {
#pragma unroll
    for (int q = 0; q < kR; ++q) {
      const int k = t + q * kThreads;
      uint64_t sum = 0;
      if (s + k < e) {
#pragma unroll
        for (int c = 0; c < kC; ++c) {
          sum += acc[k * kC + c];
          acc[k * kC + c] = 0;
        }
      }
      av[q] = sum;
    }
  }
#pragma unroll
  for (int q = 0; q < kR; ++q) {
    const int k = t + q * kThreads;
    if (s + k < e) {
      const uint64_t tt =
          (static_cast<uint64_t>(static_cast<int64_t>(cur.in[q])) << bit) - av[q];
      if (kC == 1) acc[k] = 0;
      const int32_t v = acc_final<int32_t, K>(tt, cur.dinv[q], bit, dbit);
      ring[(s + k) & rmask] = v;
      out[s + k] = v;
    }
  }
  for (int k = t + kR * kThreads; s + k < e; k += kThreads) {
    uint64_t sum = 0;
    for (int c = 0; c < kC; ++c) {
      sum += acc[k * kC + c];
      acc[k * kC + c] = 0;
    }
    const uint64_t tt = (static_cast<uint64_t>(static_cast<int64_t>(in[s + k])) << bit) - sum;
    const int32_t v = acc_final<int32_t, K>(tt, dinv[s + k], bit, dbit);
    ring[(s + k) & rmask] = v;
    out[s + k] = v;
  }
  if (kFar && (L % kEpFence) == kEpFence - 1)
    __syncthreads();  // full fence: global results visible to later loads
  else
    ep_sync<kWaves>();
  ep_load<kThreads>(cur, plo, phi, lent, dinv, in);
}

// LDS: acc_slots uint64 accumulators (kC per row of the widest level), the
// ring, then the chain's level offsets (max_levels + 1 int2).
template <TriKind K, int kWaves, bool kFar, int kE, int kR, int kC, int kD>
__global__ __launch_bounds__(64 * kWaves) void k_tri_chain_ep(
    const int4* __restrict__ lent, const int32_t* __restrict__ dinv,
    const int* __restrict__ lev_ptr, const int* __restrict__ lev_eptr,
    const int* __restrict__ chain_lev, int rmask, int acc_slots, int bit, int dbit,
    const int32_t* __restrict__ in, int32_t* out) {
  constexpr int kThreads = 64 * kWaves;
  extern __shared__ __align__(16) unsigned char smem_e[];
  EpShared sh;
  sh.acc = reinterpret_cast<uint64_t*>(smem_e);
  sh.dummy = acc_slots;
  sh.ring = reinterpret_cast<int32_t*>(sh.acc + acc_slots + kEpDummy);
  sh.rmask = rmask;
  int2* lvo = reinterpret_cast<int2*>(sh.ring + rmask + 1);
  sh.lvo = lvo;
  const int t = threadIdx.x;
  const int lb = chain_lev[2 * blockIdx.x], le = chain_lev[2 * blockIdx.x + 1];
  const int nl = le - lb;
  for (int k = t; k < acc_slots; k += kThreads) sh.acc[k] = 0;
  for (int k = t; k <= nl; k += kThreads) lvo[k] = make_int2(lev_ptr[lb + k], lev_eptr[lb + k]);
  __syncthreads();
  EpPre<kE, kR> buf[kD];
#pragma unroll
  for (int d = 0; d < kD; ++d) {
    const int Lc = min(d, nl);
    ep_load<kThreads>(buf[d], lvo[Lc], lvo[min(Lc + 1, nl)], lent, dinv, in);
  }
  // Dependencies stay inside a chain, so its first kEpFarLevels levels have
  // no far entries: the first far loads are issued from the loop.
  int L0 = 0;
  for (; L0 + kD <= nl; L0 += kD) {
#pragma unroll
    for (int d = 0; d < kD; ++d)
      ep_level<K, kWaves, kFar, kE, kR, kC, kD>(buf[d], buf[(d + kEpFarAhead) % kD], L0 + d, nl,
                                                sh, lent, dinv, in, out, bit, dbit);
  }
#pragma unroll
  for (int d = 0; d < kD; ++d)
    if (L0 + d < nl)
      ep_level<K, kWaves, kFar, kE, kR, kC, kD>(buf[d], buf[(d + kEpFarAhead) % kD], L0 + d, nl,
                                                sh, lent, dinv, in, out, bit, dbit);
}

template <TriKind K, int kWaves, bool kFar, int kE, int kR, int kC, int kD>
hipError_t tri_ep_go(const TriLayout& L, const TriSegment& seg, int bit, int dbit,
                     const int32_t* in, int32_t* out, hipStream_t s) {
  const size_t lds = ep_lds_bytes(L.ring, L.ep_maxlev, L.ep_acc);
  if (lds > static_cast<size_t>(kTriBlockedMaxLds) || L.ep_acc < kC) return hipErrorInvalidValue;
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&k_tri_chain_ep<K, kWaves, kFar, kE, kR, kC, kD>),
        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kTriBlockedMaxLds));
    if (e != hipSuccess) return e;
    attr = true;
  }
  launch_timed(&k_tri_chain_ep<K, kWaves, kFar, kE, kR, kC, kD>, dim3(seg.nchain),
               dim3(64 * kWaves), static_cast<uint32_t>(lds), s,
               reinterpret_cast<const int4*>(L.lent), static_cast<const int32_t*>(L.ldiag),
               L.lev_ptr, L.lev_eptr, seg.chain_lev, L.ring - 1, L.ep_acc, bit, dbit, in, out);
  return hipGetLastError();
}

template <TriKind K, int kWaves, int kC>
hipError_t tri_ep_launch_c(const TriLayout& L, const TriSegment& seg, int bit, int dbit,
                           const int32_t* in, int32_t* out, hipStream_t s) {
  if (L.ep_far) return tri_ep_go<K, kWaves, true, 8, 2, kC, 4>(L, seg, bit, dbit, in, out, s);
  if (L.ep_narrow)
    return tri_ep_go<K, kWaves, false, 4, 1, kC, 8>(L, seg, bit, dbit, in, out, s);
  return tri_ep_go<K, kWaves, false, 8, 2, kC, 4>(L, seg, bit, dbit, in, out, s);
}

// Accumulator copies only for the smoother's LD factors (rows with many
// entries on coarse levels).
template <TriKind K, int kWaves>
hipError_t tri_ep_launch(const TriLayout& L, const TriSegment& seg, int bit, int dbit,
                         const int32_t* in, int32_t* out, hipStream_t s) {
  if constexpr (K == TriKind::kLD) {
    if (L.ep_copies == kEpCopies)
      return tri_ep_launch_c<K, kWaves, kEpCopies>(L, seg, bit, dbit, in, out, s);
  }
  return tri_ep_launch_c<K, kWaves, 1>(L, seg, bit, dbit, in, out, s);
}

// ---------------------------------------------------------------------------
// Row-parallel integer LD solve: the chains, levels, LDS ring and far
// dependencies of k_tri_chain_ep, for factors whose rows hold at most kG * kE
// dependency entries.  kG lanes serve one row; each lane keeps kE entries of
// its row, padded with zero values, in registers.  The integer sum is
// order-free (wrap-around), so the result equals the sequential one bit for
// bit.
//
// What bounds it: a chain is one workgroup of 1-8 waves that walks its levels
// one after another, so a level costs the instructions its waves issue (one
// per four cycles and wave) plus one LDS round trip, whatever the bandwidth.
// Everything that does not depend on the previous level is therefore computed
// once on the host or kept off the vector unit:
//  * an entry {code, val} holds the byte offset of its ring slot (no masking,
//    no address arithmetic) and the negated value, so a row's sum starts from
//    in * 2^bit and only adds products; a far entry (the first kFq slots of a
//    row at most) holds ~(4 * position) instead;
//  * entries, inverse diagonals, right-hand sides and results are buffers of
//    exactly their bytes, addressed by a lane's place in the level plus the
//    level's start; lanes past a level's end load what follows (past the
//    buffer's end: 0) and never store.  The sum is the instruction's vector
//    offset, the one that the hardware compares with the buffer's size: with
//    the level's start as its scalar offset, which that comparison does not
//    count (or subtracts from the size, where it may pass it), the rows past
//    the last one would be read from beyond the buffer;
//  * the loads of level L + kD - 1 are issued into the buffer that level L - 1
//    has freed, between this level's ring reads and their first use;
//  * shifts by bit and dbit (0..30) are single 32-bit funnel shifts, and the
//    finish takes one 32 x 32 product and one low product.
// Measured per solve against the form that masked ring positions and computed
// addresses per level (128^3 BlockSOR, levels 0-4: 87 / 83 / 78 / 92 / 43 us,
// now 80 / 82 / 57 / 55 / 27; with scalar offsets 82 / 80 / 64 / 62 / 29) and
// against the entry-parallel kernel and one launch per wide level (63^3 SOR,
// whole V-cycle: 5.27 -> 2.50 ms).
// A block of right-hand sides runs one workgroup per chain and right-hand side
// (a chain leaves most of the chip idle: 40 chains, 256 CUs), all of one chain
// on one XCD when the chain count is a multiple of 8; four right-hand sides
// per workgroup, which loads each entry once, took 1.9 ms of LD solves per
// 16-vector V-cycle of the 96^3 inclusions system, against 0.95 ms.
using RpWord4 = __attribute__((ext_vector_type(4))) unsigned;
template <int kE, int kFq>
struct RpPre {
  int lo, cnt;            // first position and rows of the level (scalars)
  RpWord4 ent[kE / 2];    // {code, -val, code, -val}
  int32_t xfar[kFq > 0 ? kFq : 1];
  int32_t dinv, in;
};

struct RpArgs {
  __amdgpu_buffer_rsrc_t rent, dinv, in, out;
  unsigned ring_mask;     // ring size in bytes - 1
  int bit, dbit;
  int fence_mask;
};

// Constants of a lane.
struct RpLane {
  unsigned ent_off;       // its entries' byte offset from the level's first row's
  unsigned row4;          // 4 * its row in the level
  int owner;              // its row for the row's first lane, else INT32_MAX
  int32_t scale;          // 2^bit for the row's first lane, else 0
};

// A buffer of `bytes` bytes; loads whose vector offset is past its end return 0.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rp_buffer(const void* p, unsigned bytes) {
  constexpr int kRaw32 = 0x00020000;  // untyped, 32-bit elements
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes),
                                           kRaw32);
}

// LDS word at a byte offset: the ring begins the kernel's only LDS array, at
// address 0.
using LdsWord = __attribute__((address_space(3))) int32_t;
__device__ __forceinline__ LdsWord* rp_lds(unsigned off) {
  return reinterpret_cast<LdsWord*>(off);
}

template <int kG, int kE, int kS, int kFq>
__device__ __forceinline__ void rp_load(RpPre<kE, kFq>& r, int lo, int hi, const RpArgs& a,
                                        const RpLane& ln) {
  r.lo = lo;
  r.cnt = hi - lo;
  const unsigned pos4 = 4u * static_cast<unsigned>(lo) + ln.row4;
  const unsigned ent = static_cast<unsigned>(lo) * (kG * kE * 8) + ln.ent_off;
#pragma unroll
  for (int h = 0; h < kE / 2; ++h)
    r.ent[h] = __builtin_amdgcn_raw_buffer_load_b128(a.rent, static_cast<int>(ent) + 16 * h, 0, 0);
  r.dinv = static_cast<int>(
      __builtin_amdgcn_raw_buffer_load_b32(a.dinv, static_cast<int>(pos4), 0, 0));
  r.in = static_cast<int>(
      __builtin_amdgcn_raw_buffer_load_b32(a.in, static_cast<int>(kS * pos4), 0, 0));
}

// acc + dpp(acc) on 64-bit values, one stage of a group sum: the low words'
// sum sets the carry that the high words' takes.  A DPP operand written by
// the two instructions before it needs two wait states.
#define SC23AD_DPP_ADD64(NAME, CTRL)                                                    \
  __device__ __forceinline__ uint64_t NAME(uint64_t v) {                                \
    unsigned lo, hi;                                                                    \
    asm("s_nop 1\n\t"                                                                   \
        "v_add_co_u32_dpp %0, vcc, %2, %2 " CTRL " row_mask:0xf bank_mask:0xf\n\t"      \
        "v_addc_co_u32_dpp %1, vcc, %3, %3, vcc " CTRL " row_mask:0xf bank_mask:0xf"    \
        : "=&v"(lo), "=&v"(hi)                                                          \
        : "v"(static_cast<unsigned>(v)), "v"(static_cast<unsigned>(v >> 32))            \
        : "vcc");                                                                       \
    return (static_cast<uint64_t>(hi) << 32) | lo;                                      \
  }
SC23AD_DPP_ADD64(dpp_add_swap1, "quad_perm:[1,0,3,2]")
SC23AD_DPP_ADD64(dpp_add_swap2, "quad_perm:[2,3,0,1]")
SC23AD_DPP_ADD64(dpp_add_half_mirror, "row_half_mirror")
SC23AD_DPP_ADD64(dpp_add_mirror, "row_mirror")
#undef SC23AD_DPP_ADD64

// Sum over aligned groups of kG lanes, every lane ending with its group's;
// all lanes must be active.  Groups of 32 and 64 exchange rows of 16 and
// halves of the wave with gfx950's permlane swaps: two equal inputs come back
// as the two parts side by side.
__device__ __forceinline__ uint64_t permlane_add(uint64_t v, bool halves) {
  const unsigned lo = static_cast<unsigned>(v), hi = static_cast<unsigned>(v >> 32);
  auto l = halves ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                  : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  auto h = halves ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                  : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return ((static_cast<uint64_t>(h[0]) << 32) | l[0]) +
         ((static_cast<uint64_t>(h[1]) << 32) | l[1]);
}
template <int kG>
__device__ __forceinline__ uint64_t group_sum_dpp(uint64_t v) {
  static_assert(kG >= 1 && kG <= 64 && (kG & (kG - 1)) == 0, "groups of 1-64 lanes");
  if (kG >= 2) v = dpp_add_swap1(v);
  if (kG >= 4) v = dpp_add_swap2(v);
  if (kG >= 8) v = dpp_add_half_mirror(v);
  if (kG >= 16) v = dpp_add_mirror(v);
  if (kG >= 32) v = permlane_add(v, false);
  if (kG >= 64) v = permlane_add(v, true);
  return v;
}

// Level L (buffer cur).  nxt: the buffer level L - 1 has freed, filled for
// level L + kD - 1, whose bounds `pend` holds; `ahead`: level L + kA's buffer.
template <bool kTail, int kMaxWaves, bool kFar, int kG, int kE, int kS, int kD, int kA, int kFq>
__device__ __forceinline__ void rp_level(RpPre<kE, kFq>& cur, RpPre<kE, kFq>& nxt,
                                         RpPre<kE, kFq>& ahead, int L, int2& pend,
                                         const int* lvo, const RpArgs& a,
                                         const RpLane& ln) {
  int32_t xv[kE];
#pragma unroll
  for (int q = 0; q < kE; ++q) {
    int c = static_cast<int>(q % 2 ? cur.ent[q / 2].z : cur.ent[q / 2].x);
    if (kFar && q < kFq) c = max(c, 0);
    xv[q] = *rp_lds(static_cast<unsigned>(c));
  }
  int plo = 0, phi = 0;
  if (!kTail) {
    plo = __builtin_amdgcn_readfirstlane(pend.x);
    phi = __builtin_amdgcn_readfirstlane(pend.y);
  }
  // every ring read is issued before the loads and the first product, so the
  // level pays one LDS round trip, covered in part by issuing the loads
  __builtin_amdgcn_sched_barrier(0);
  if (!kTail) rp_load<kG, kE, kS, kFq>(nxt, plo, phi, a, ln);
  if (kFar) {
#pragma unroll
    for (int q = 0; q < kFq; ++q) {
      // ~code is 4 * position for a far entry, else past the buffer's end
      const unsigned c = q % 2 ? ahead.ent[q / 2].z : ahead.ent[q / 2].x;
      ahead.xfar[q] = static_cast<int>(
          __builtin_amdgcn_raw_buffer_load_b32(a.out, static_cast<int>(kS * ~c), 0, 0));
    }
  }
  if (!kTail) {
    pend.x = lvo[L + kD];
    pend.y = lvo[L + kD + 1];
  }
  __builtin_amdgcn_sched_barrier(0);
  if (kFar) {
    // waits for a far value only where a lane of the wave has one
#pragma unroll
    for (int q = 0; q < kFq; ++q) {
      const int c = static_cast<int>(q % 2 ? cur.ent[q / 2].z : cur.ent[q / 2].x);
      if (__any(c < 0)) xv[q] = c < 0 ? cur.xfar[q] : xv[q];
    }
  }
  uint64_t acc = prod64(cur.in, ln.scale), acc2 = 0;  // two chains of multiply-adds
#pragma unroll
  for (int h = 0; h < kE / 2; ++h) {
    acc += prod64(static_cast<int>(cur.ent[h].y), xv[2 * h]);
    acc2 += prod64(static_cast<int>(cur.ent[h].w), xv[2 * h + 1]);
  }
  // opaque ends keep the two chains apart (the compiler would otherwise
  // fold them into one chain of dependent multiply-adds)
  asm volatile("" : "+v"(acc));
  asm volatile("" : "+v"(acc2));
  acc = group_sum_dpp<kG>(acc + acc2);
  const int32_t v = rp_finish(acc, cur.dinv, a.bit, a.dbit);
  if (ln.owner < cur.cnt) {
    const unsigned pos4 = 4u * static_cast<unsigned>(cur.lo) + ln.row4;
    *rp_lds(pos4 & a.ring_mask) = v;
    __builtin_amdgcn_raw_buffer_store_b32(static_cast<unsigned>(v), a.out,
                                          static_cast<int>(kS * pos4), 0, 0);
  }
  // a full fence every fence_mask + 1 levels makes far values visible before
  // any load of them; it also drains the loads in flight, so the plan makes
  // the period as long as the nearest far dependency allows
  if (kFar && (L & a.fence_mask) == a.fence_mask)
    __syncthreads();
  else
    ep_sync<kMaxWaves>();
}

// The last nl - L0 < kD levels, nested so that no paths join between them.
template <int kFirst, int kMaxWaves, bool kFar, int kG, int kE, int kS, int kD, int kA, int kFq>
__device__ __forceinline__ void rp_tail(RpPre<kE, kFq> (&buf)[kD], int L0, int nl, int2& pend,
                                        const int* lvo, const RpArgs& a, const RpLane& ln) {
  if constexpr (kFirst < kD - 1) {
    if (L0 + kFirst < nl) {
      rp_level<true, kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>(
          buf[kFirst], buf[(kFirst + kD - 1) % kD], buf[(kFirst + kA) % kD], L0 + kFirst, pend,
          lvo, a, ln);
      rp_tail<kFirst + 1, kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>(buf, L0, nl, pend, lvo, a, ln);
    }
  }
}

// LDS: the ring, then the chain's level offsets (max_levels + 1 ints and
// kRpPadLevels more that repeat the last one).  Far values of level L + kA
// are loaded in level L, from entries loaded kD - 1 - kA levels before that.
template <int kMaxWaves, bool kFar, int kG, int kE, int kS, int kD, int kA, int kFq>
__global__ __launch_bounds__(64 * kMaxWaves) void k_tri_chain_rp(
    const void* __restrict__ rent, const int32_t* __restrict__ dinv,
    const int* __restrict__ lev_ptr, const int* __restrict__ chain_lev, int n, int ring4, int bit,
    int dbit, int fence, const int32_t* __restrict__ in, int32_t* out) {
  static_assert(!kFar || (kA >= 1 && kA < kD - 1), "far values need their entries loaded first");
  static_assert(kA <= kRpMaxAhead, "the plan's fence period allows for kRpMaxAhead");
  static_assert(kD + 1 <= kRpPadLevels, "level offsets are read kD + 1 past the end");
  extern __shared__ __align__(16) unsigned char smem_r[];
  int* lvo = reinterpret_cast<int*>(smem_r + ring4);
  const int t = threadIdx.x;
  const int threads = kMaxWaves == 1 ? 64 : static_cast<int>(blockDim.x);
  const int lb = chain_lev[2 * blockIdx.x], le = chain_lev[2 * blockIdx.x + 1];
  const int nl = le - lb;
  for (int k = t; k <= nl + kD + 1; k += threads) lvo[k] = lev_ptr[lb + min(k, nl)];
  __syncthreads();
  const unsigned n4 = 4u * static_cast<unsigned>(n);
  // kS = 1: a plain vector.  kS = 4: right-hand side blockIdx.y of a block
  // (four values of a row in one 16-byte word, groups of four one after another)
  const unsigned r = kS == 1 ? 0u : blockIdx.y & 3u;
  const size_t off = kS == 1 ? 0 : static_cast<size_t>(blockIdx.y >> 2) * n * 4 + r;
  const unsigned vec_bytes = kS * n4 - 4u * r;
  const RpArgs a{rp_buffer(rent, n4 * (kG * kE * 2)), rp_buffer(dinv, n4),
                 rp_buffer(in + off, vec_bytes), rp_buffer(out + off, vec_bytes), static_cast<unsigned>(ring4) - 1u, bit, dbit, fence - 1};
  RpLane ln;
  ln.ent_off = static_cast<unsigned>(t) * (kE * 8);
  ln.row4 = 4u * static_cast<unsigned>(t / kG);
  ln.owner = t % kG == 0 ? t / kG : INT32_MAX;
  ln.scale = t % kG == 0 ? 1 << bit : 0;
  RpPre<kE, kFq> buf[kD];
#pragma unroll
  for (int d = 0; d < kD - 1; ++d)
    rp_load<kG, kE, kS, kFq>(buf[d], __builtin_amdgcn_readfirstlane(lvo[d]),
                         __builtin_amdgcn_readfirstlane(lvo[d + 1]), a, ln);
  int2 pend = make_int2(lvo[kD - 1], lvo[kD]);
  // Whole rounds of kD levels, then the tail, which loads nothing ahead, in a
  // copy of the body.  (One body for all levels measured slower: with a test
  // around each level the compiler waits for every outstanding load where the
  // paths join, and without one the last round runs up to kD - 1 empty levels.)
  int L0 = 0;
  for (; L0 + kD <= nl; L0 += kD) {
#pragma unroll
    for (int d = 0; d < kD; ++d)
      rp_level<false, kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>(buf[d], buf[(d + kD - 1) % kD],
                                                       buf[(d + kA) % kD], L0 + d, pend, lvo, a,
                                                       ln);
  }
  rp_tail<0, kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>(buf, L0, nl, pend, lvo, a, ln);
}

template <int kMaxWaves, bool kFar, int kG, int kE, int kS, int kD, int kA, int kFq = kFar ? kE : 0>
hipError_t tri_rp_go(const TriLayout& L, int nrhs, int bit, int dbit, const int32_t* in,
                     int32_t* out, hipStream_t s) {
  const size_t lds = rp_lds_bytes(L.rp_ring, L.rp_maxlev);
  if (lds > static_cast<size_t>(kTriBlockedMaxLds) || L.n <= 0 || bit < 0 || bit > 30 ||
      dbit < 0 || dbit > 30 || L.rp_fence < 1 ||
      static_cast<uint64_t>(L.n) * (kG * kE * 8) > kRpMaxBytes)
    return hipErrorInvalidValue;
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&k_tri_chain_rp<kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>),
        hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kTriBlockedMaxLds));
    if (e != hipSuccess) return e;
    attr = true;
  }
  launch_timed(&k_tri_chain_rp<kMaxWaves, kFar, kG, kE, kS, kD, kA, kFq>, dim3(L.rp_nchain, nrhs),
               dim3(64 * L.rp_waves), static_cast<uint32_t>(lds), s,
               L.rent, static_cast<const int32_t*>(L.ldiag), L.rp_lev, L.rp_chain, L.n,
               4 * L.rp_ring, bit, dbit, L.rp_fence, in, out);
  return hipGetLastError();
}

// Register layouts and prefetch distances: a level takes 0.1-0.3 us and its
// entries come from HBM, so the loads run several levels ahead, as far as the
// 256 registers of a lane allow.
template <int kMaxWaves, int kS, bool kFar>
hipError_t tri_rp_layout(const TriLayout& L, int nrhs, int bit, int dbit, const int32_t* in,
                         int32_t* out, hipStream_t s) {
  constexpr int kD8 = kFar ? 6 : 8, kD10 = kFar ? 5 : 8, kD12 = kFar ? 5 : 6;
  constexpr int kA8 = kFar ? 3 : 1, kA10 = kFar ? 2 : 1;
  if (L.rp_lanes <= 1) {
    if (L.rp_e == 4) {
      if (kFar && L.rp_farq == 1)  // one far entry at most, stored first
        return tri_rp_go<kMaxWaves, kFar, 1, 4, kS, 10, 4, 1>(L, nrhs, bit, dbit, in, out, s);
      return tri_rp_go<kMaxWaves, kFar, 1, 4, kS, 10, 4>(L, nrhs, bit, dbit, in, out, s);
    }
    if (L.rp_e == 8) return tri_rp_go<kMaxWaves, kFar, 1, 8, kS, kD8, kA8>(L, nrhs, bit, dbit, in, out, s);
    if (L.rp_e == 10)
      return tri_rp_go<kMaxWaves, kFar, 1, 10, kS, kD10, kA10>(L, nrhs, bit, dbit, in, out, s);
    if (L.rp_e == 12)
      return tri_rp_go<kMaxWaves, kFar, 1, 12, kS, kD12, kA10>(L, nrhs, bit, dbit, in, out, s);
    return hipErrorInvalidValue;
  }
  if constexpr (kFar) {
    // far entries dealt over the lanes, slot 0 of each lane first: up to
    // kRpFarSlots per lane
    auto lanes = [&](auto e_tag) -> hipError_t {
      constexpr int E = decltype(e_tag)::value, Q = kRpFarSlots;
      switch (L.rp_lanes) {
        case 2: return tri_rp_go<kMaxWaves, true, 2, E, kS, 5, 2, Q>(L, nrhs, bit, dbit, in, out, s);
        case 4: return tri_rp_go<kMaxWaves, true, 4, E, kS, 5, 2, Q>(L, nrhs, bit, dbit, in, out, s);
        case 8: return tri_rp_go<kMaxWaves, true, 8, E, kS, 5, 2, Q>(L, nrhs, bit, dbit, in, out, s);
        default: return hipErrorInvalidValue;
      }
    };
    using std::integral_constant;
    if (L.rp_e == 8) return lanes(integral_constant<int, 8>{});
    if (L.rp_e == 10) return lanes(integral_constant<int, 10>{});
    if (L.rp_e == 12) return lanes(integral_constant<int, 12>{});
  }
  if constexpr (!kFar) {
    auto lanes = [&](auto e_tag, auto d_tag) -> hipError_t {
      constexpr int E = decltype(e_tag)::value, D = decltype(d_tag)::value;
      switch (L.rp_lanes) {
        case 2: return tri_rp_go<kMaxWaves, false, 2, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        case 4: return tri_rp_go<kMaxWaves, false, 4, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        case 8: return tri_rp_go<kMaxWaves, false, 8, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        case 16: return tri_rp_go<kMaxWaves, false, 16, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        case 32: return tri_rp_go<kMaxWaves, false, 32, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        case 64: return tri_rp_go<kMaxWaves, false, 64, E, kS, D, 1>(L, nrhs, bit, dbit, in, out, s);
        default: return hipErrorInvalidValue;
      }
    };
    using std::integral_constant;
    if (L.rp_e == 4) return lanes(integral_constant<int, 4>{}, integral_constant<int, 10>{});
    if (L.rp_e == 6) return lanes(integral_constant<int, 6>{}, integral_constant<int, 8>{});
    if (L.rp_e == 8) return lanes(integral_constant<int, 8>{}, integral_constant<int, 8>{});
    if (L.rp_e == 10) return lanes(integral_constant<int, 10>{}, integral_constant<int, 8>{});
    if (L.rp_e == 12) return lanes(integral_constant<int, 12>{}, integral_constant<int, 6>{});
  }
  return hipErrorInvalidValue;
}

template <int kMaxWaves, int kS>
hipError_t tri_rp_far(const TriLayout& L, int nrhs, int bit, int dbit, const int32_t* in,
                         int32_t* out, hipStream_t s) {
  if (L.rp_farq > 0) return tri_rp_layout<kMaxWaves, kS, true>(L, nrhs, bit, dbit, in, out, s);
  return tri_rp_layout<kMaxWaves, kS, false>(L, nrhs, bit, dbit, in, out, s);
}

// 9-16 waves (128 registers per lane): one lane of 4 entries per row.
template <int kS>
hipError_t tri_rp_wide(const TriLayout& L, int nrhs, int bit, int dbit, const int32_t* in,
                         int32_t* out, hipStream_t s) {
  if (L.rp_lanes != 1 || L.rp_e != 4) return hipErrorInvalidValue;
  if (L.rp_farq == 0) return tri_rp_go<16, false, 1, 4, kS, 8, 1>(L, nrhs, bit, dbit, in, out, s);
  if (L.rp_farq == 1) return tri_rp_go<16, true, 1, 4, kS, 8, 4, 1>(L, nrhs, bit, dbit, in, out, s);
  return tri_rp_go<16, true, 1, 4, kS, 6, 2>(L, nrhs, bit, dbit, in, out, s);
}

// Row-parallel FP LD solve (solvers 0 and 1): the chains, pieces, LDS ring,
// far rule and buffer addressing of k_tri_chain_rp, with a row's products
// subtracted one at a time in stored order, as the sequential solve does, so
// the result is the reference's bit for bit.
//
// 2^lg lanes form the products of a row, kE consecutive entries each.  With
// one lane they are subtracted as they come.  With several they go through
// LDS: every lane writes its products to the row's slots and all lanes of the
// row (one wave, whose LDS accesses stay in order) read them back, 16 bytes
// at a time, two blocks of 8 ahead of the subtractions; a piece subtracts as
// many as its longest row has, rounded up to 8.  An absent entry names the
// zero slot behind the ring and has the value +0, so its product is +0, and
// t - (+0) is t for every t: no count is checked.  What bounds a level is that
// chain of subtractions and the instructions a wave issues.
// Against the form that shuffled every product to the row's lanes and
// selected by the row's count, several rows' worth of steps per level
// whatever their length: 96^3 FP64 solve 45.7 -> 24.3 ms, 48^3 27-point FP32
// solve 70.4 -> 37.8 ms.
template <typename T>
struct FpWords;
template <>
struct FpWords<float> {
  static constexpr int k16 = 4;  // values in 16 bytes
  static __device__ __forceinline__ float load(__amdgpu_buffer_rsrc_t b, int v) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, v, 0, 0));
  }
  static __device__ __forceinline__ void store(float x, __amdgpu_buffer_rsrc_t b, int v) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), b, v, 0, 0);
  }
};
using RpWord2 = __attribute__((ext_vector_type(2))) unsigned;
template <>
struct FpWords<double> {
  static constexpr int k16 = 2;
  static __device__ __forceinline__ double load(__amdgpu_buffer_rsrc_t b, int v) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(b, v, 0, 0));
  }
  static __device__ __forceinline__ void store(double x, __amdgpu_buffer_rsrc_t b, int v) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(RpWord2, x), b, v, 0, 0);
  }
};
template <typename T>
using FpVec16 = __attribute__((ext_vector_type(16 / sizeof(T)))) T;
template <typename T>
using LdsOf = __attribute__((address_space(3))) T;
template <typename T>
__device__ __forceinline__ LdsOf<T>* fp_lds(unsigned off) {  // as rp_lds
  return reinterpret_cast<LdsOf<T>*>(off);
}

template <typename T, int kE, int kFq>
struct RpfPre {
  int lo, cnt, steps;     // first position, rows, subtractions per row (scalars)
  RpWord4 code[kE / 4];
  FpVec16<T> val[kE * sizeof(T) / 16];
  T xfar[kFq > 0 ? kFq : 1];
  T dinv, in;
};

struct RpfArgs {
  __amdgpu_buffer_rsrc_t code, val, dinv, in, out;
  unsigned ring_mask;     // ring size in bytes - 1
  int lg;                 // log2 of the lanes per row
  int fence_mask;
};

struct RpfLane {
  unsigned slot;          // its first entry's place from the piece's first row's
  unsigned row_off;       // its row's byte offset from the piece's first row's
  int owner;              // its row for the row's first lane, else INT32_MAX
  unsigned put, get;      // LDS offsets: its products, the row's products
};

template <typename T, int kE, int kFq>
__device__ __forceinline__ T rpf_val(const RpfPre<T, kE, kFq>& r, int q) {
  constexpr int k = FpWords<T>::k16;
  return r.val[q / k][q % k];
}

template <typename T, int kE, int kFq>
__device__ __forceinline__ void rpf_load(RpfPre<T, kE, kFq>& r, int lo, int hi, int steps,
                                         const RpfArgs& a, const RpfLane& ln) {
  constexpr int kT = sizeof(T);
  r.lo = lo;
  r.cnt = hi - lo;
  r.steps = steps;
  // vector offsets, as in rp_load
  const unsigned e = (static_cast<unsigned>(lo) << a.lg) * kE + ln.slot;
  const int ce = static_cast<int>(e * 4), ve = static_cast<int>(e * kT);
  const int row = static_cast<int>(static_cast<unsigned>(lo) * kT + ln.row_off);
#pragma unroll
  for (int h = 0; h < kE / 4; ++h)
    r.code[h] = __builtin_amdgcn_raw_buffer_load_b128(a.code, ce + 16 * h, 0, 0);
#pragma unroll
  for (int h = 0; h < kE * kT / 16; ++h)
    r.val[h] = __builtin_bit_cast(
        FpVec16<T>, __builtin_amdgcn_raw_buffer_load_b128(a.val, ve + 16 * h, 0, 0));
  r.dinv = FpWords<T>::load(a.dinv, row);
  r.in = FpWords<T>::load(a.in, row);
}

template <typename T>
struct FpBlock8 {
  FpVec16<T> v[8 * sizeof(T) / 16];
};
template <typename T>
__device__ __forceinline__ FpBlock8<T> rpf_get8(unsigned off) {
  FpBlock8<T> b;
#pragma unroll
  for (int h = 0; h < static_cast<int>(8 * sizeof(T) / 16); ++h)
    b.v[h] = *fp_lds<FpVec16<T>>(off + 16 * h);
  return b;
}
template <typename T>
__device__ __forceinline__ T rpf_sub8(T t, const FpBlock8<T>& b) {
  constexpr int k = FpWords<T>::k16;
#pragma unroll
  for (int q = 0; q < 8; ++q) t = t - b.v[q / k][q % k];
  return t;
}

template <typename T, bool kTail, int kMaxWaves, bool kLanes, int kE, int kD, int kA, int kFq>
__device__ __forceinline__ void rpf_level(RpfPre<T, kE, kFq>& cur, RpfPre<T, kE, kFq>& nxt,
                                          RpfPre<T, kE, kFq>& ahead, int L, int (&pend)[3],
                                          const int2* lvo, const RpfArgs& a, const RpfLane& ln) {
  constexpr int kT = sizeof(T);
  T xv[kE];
#pragma unroll
  for (int q = 0; q < kE; ++q) {
    int c = static_cast<int>(cur.code[q / 4][q % 4]);
    if (q < kFq) c = max(c, 0);
    xv[q] = *fp_lds<T>(static_cast<unsigned>(c));
  }
  int plo = 0, phi = 0, pst = 0;
  if (!kTail) {
    plo = __builtin_amdgcn_readfirstlane(pend[0]);
    phi = __builtin_amdgcn_readfirstlane(pend[1]);
    pst = __builtin_amdgcn_readfirstlane(pend[2]);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (!kTail) rpf_load<T, kE, kFq>(nxt, plo, phi, pst, a, ln);
  if (kFq > 0) {
#pragma unroll
    for (int q = 0; q < kFq; ++q) {
      // ~code is the byte offset of a far entry's value, else past the end
      const unsigned c = ahead.code[q / 4][q % 4];
      ahead.xfar[q] = FpWords<T>::load(a.out, static_cast<int>(~c));
    }
  }
  if (!kTail) {
    const int2 p = lvo[L + kD];
    pend[0] = p.x;
    pend[2] = p.y;
    pend[1] = lvo[L + kD + 1].x;
  }
  __builtin_amdgcn_sched_barrier(0);
  if (kFq > 0) {
#pragma unroll
    for (int q = 0; q < kFq; ++q) {
      const int c = static_cast<int>(cur.code[q / 4][q % 4]);
      if (__any(c < 0)) xv[q] = c < 0 ? cur.xfar[q] : xv[q];
    }
  }
  T t = cur.in;
  if constexpr (!kLanes) {
#pragma unroll
    for (int q = 0; q < kE; ++q) t = t - rpf_val<T, kE, kFq>(cur, q) * xv[q];
  } else {
    constexpr int k = FpWords<T>::k16;
#pragma unroll
    for (int h = 0; h < kE * kT / 16; ++h) {
      FpVec16<T> p;
#pragma unroll
      for (int q = 0; q < k; ++q) p[q] = cur.val[h][q] * xv[h * k + q];
      *fp_lds<FpVec16<T>>(ln.put + 16 * h) = p;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    // steps is a multiple of 8; blocks read past it are not subtracted (the
    // offsets stay inside the array: kRpfReadAhead bytes follow the last row)
    FpBlock8<T> b0 = rpf_get8<T>(ln.get), b1 = rpf_get8<T>(ln.get + 8 * kT), b2;
    unsigned g = ln.get + 16 * kT;
    for (int left = cur.steps;;) {
      b2 = rpf_get8<T>(g);
      t = rpf_sub8(t, b0);
      if (left <= 8) break;
      b0 = rpf_get8<T>(g + 8 * kT);
      t = rpf_sub8(t, b1);
      if (left <= 16) break;
      b1 = rpf_get8<T>(g + 16 * kT);
      t = rpf_sub8(t, b2);
      if (left <= 24) break;
      left -= 24;
      g += 24 * kT;
    }
  }
  const T v = t * cur.dinv;
  if (ln.owner < cur.cnt) {
    const unsigned row = static_cast<unsigned>(cur.lo) * kT + ln.row_off;
    *fp_lds<T>(row & a.ring_mask) = v;
    FpWords<T>::store(v, a.out, static_cast<int>(row));
  }
  // as in rp_level
  if (kFq > 0 && (L & a.fence_mask) == a.fence_mask)
    __syncthreads();
  else
    ep_sync<kMaxWaves>();
}

template <typename T, int kFirst, int kMaxWaves, bool kLanes, int kE, int kD, int kA, int kFq>
__device__ __forceinline__ void rpf_tail(RpfPre<T, kE, kFq> (&buf)[kD], int L0, int nl,
                                         int (&pend)[3], const int2* lvo, const RpfArgs& a,
                                         const RpfLane& ln) {
  if constexpr (kFirst < kD - 1) {
    if (L0 + kFirst < nl) {
      rpf_level<T, true, kMaxWaves, kLanes, kE, kD, kA, kFq>(
          buf[kFirst], buf[(kFirst + kD - 1) % kD], buf[(kFirst + kA) % kD], L0 + kFirst, pend,
          lvo, a, ln);
      rpf_tail<T, kFirst + 1, kMaxWaves, kLanes, kE, kD, kA, kFq>(buf, L0, nl, pend, lvo, a, ln);
    }
  }
}

// LDS: the ring, 16 bytes of zeros, the rows' products (kLanes), then the
// chain's {first position, steps} per piece (as in k_tri_chain_rp).
template <typename T, int kMaxWaves, bool kLanes, int kE, int kD, int kA, int kFq>
__global__ __launch_bounds__(64 * kMaxWaves) void k_tri_chain_rpf(
    const int* __restrict__ code, const T* __restrict__ val, const T* __restrict__ dinv,
    const int* __restrict__ lev_ptr, const int* __restrict__ lev_steps,
    const int* __restrict__ chain_lev, int n, int ring_bytes, int lg, int fence,
    const T* __restrict__ in, T* out) {
  constexpr int kT = sizeof(T);
  static_assert(kFq == 0 || (kA >= 1 && kA < kD - 1), "far values need their entries first");
  static_assert(kA <= kRpMaxAhead, "the plan's fence period allows for kRpMaxAhead");
  static_assert(kD + 1 <= kRpPadLevels, "level offsets are read kD + 1 past the end");
  extern __shared__ __align__(16) unsigned char smem_f[];
  const int t = threadIdx.x;
  const int threads = kMaxWaves == 1 ? 64 : static_cast<int>(blockDim.x);
  const int lanes = 1 << lg;
  const int row_bytes = lanes * kE * kT + 16;  // rows on different banks
  const int stage = ring_bytes + 16;
  const int stage_bytes = kLanes ? (threads >> lg) * row_bytes + kRpfReadAhead : 0;
  int2* lvo = reinterpret_cast<int2*>(smem_f + stage + stage_bytes);
  const int lb = chain_lev[2 * blockIdx.x], le = chain_lev[2 * blockIdx.x + 1];
  const int nl = le - lb;
  // a slot that nothing has been written to yet holds no leftover bits
  for (int k = 4 * t; k < stage; k += 4 * threads) *fp_lds<int>(k) = 0;
  for (int k = t; k <= nl + kD + 1; k += threads)
    lvo[k] = make_int2(lev_ptr[lb + min(k, nl)], k < nl ? lev_steps[lb + k] : 8);
  __syncthreads();
  const unsigned nb = static_cast<unsigned>(n) * kT;
  const unsigned slots = (static_cast<unsigned>(n) << lg) * kE;
  const RpfArgs a{rp_buffer(code, slots * 4), rp_buffer(val, slots * kT), rp_buffer(dinv, nb),
                  rp_buffer(in, nb), rp_buffer(out, nb), static_cast<unsigned>(ring_bytes) - 1u,
                  lg, fence - 1};
  const int row = t >> lg, lane = t & (lanes - 1);
  RpfLane ln;
  ln.slot = static_cast<unsigned>(t) * kE;
  ln.row_off = static_cast<unsigned>(row) * kT;
  ln.owner = lane == 0 ? row : INT32_MAX;
  ln.get = static_cast<unsigned>(stage + row * row_bytes);
  ln.put = ln.get + static_cast<unsigned>(lane * kE * kT);
  RpfPre<T, kE, kFq> buf[kD];
#pragma unroll
  for (int d = 0; d < kD - 1; ++d)
    rpf_load<T, kE, kFq>(buf[d], __builtin_amdgcn_readfirstlane(lvo[d].x),
                         __builtin_amdgcn_readfirstlane(lvo[d + 1].x),
                         __builtin_amdgcn_readfirstlane(lvo[d].y), a, ln);
  int pend[3] = {lvo[kD - 1].x, lvo[kD].x, lvo[kD - 1].y};
  int L0 = 0;
  for (; L0 + kD <= nl; L0 += kD) {
#pragma unroll
    for (int d = 0; d < kD; ++d)
      rpf_level<T, false, kMaxWaves, kLanes, kE, kD, kA, kFq>(
          buf[d], buf[(d + kD - 1) % kD], buf[(d + kA) % kD], L0 + d, pend, lvo, a, ln);
  }
  rpf_tail<T, 0, kMaxWaves, kLanes, kE, kD, kA, kFq>(buf, L0, nl, pend, lvo, a, ln);
}

template <typename T, int kMaxWaves, bool kLanes, int kE, int kD, int kA, int kFq>
hipError_t tri_rpf_go(const TriLayout& L, const T* in, T* out, hipStream_t s) {
  const size_t lds = rpf_lds_bytes(sizeof(T), L.rp_ring, L.rp_waves, L.rp_lanes, kE, L.rp_maxlev);
  int lg = 0;
  while ((1 << lg) < L.rp_lanes) ++lg;
  if (lds > static_cast<size_t>(kTriBlockedMaxLds) || L.n <= 0 || L.rp_fence < 1 ||
      (1 << lg) != L.rp_lanes || (L.rp_lanes > 1) != kLanes ||
      static_cast<uint64_t>(L.n) * L.rp_lanes * kE * sizeof(T) > kRpMaxBytes)
    return hipErrorInvalidValue;
  auto kern = &k_tri_chain_rpf<T, kMaxWaves, kLanes, kE, kD, kA, kFq>;
  static bool attr = false;
  if (!attr) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(kTriBlockedMaxLds));
    if (e != hipSuccess) return e;
    attr = true;
  }
  hipLaunchKernelGGL(kern, dim3(L.rp_nchain), dim3(64 * L.rp_waves), static_cast<uint32_t>(lds),
                     s, L.rpf_dep, static_cast<const T*>(L.rpf_val),
                     static_cast<const T*>(L.ldiag), L.rp_lev, L.rp_steps, L.rp_chain, L.n,
                     L.rp_ring * static_cast<int>(sizeof(T)), lg, L.rp_fence, in, out);
  return hipGetLastError();
}

// Prefetch distances as far as 256 registers allow.  Far values: the leading
// slots that can hold one with one lane per row (the 7-point factor's only
// far entry is its first), else every slot.
template <typename T, int kMaxWaves, bool kLanes>
hipError_t tri_rpf_layout(const TriLayout& L, const T* in, T* out, hipStream_t s) {
  constexpr bool kD64 = sizeof(T) == 8;
  if (L.rp_e == 4) {
    if (L.rp_farq == 0) return tri_rpf_go<T, kMaxWaves, kLanes, 4, kD64 ? 8 : 10, 1, 0>(L, in, out, s);
    if constexpr (!kLanes) {
      if (L.rp_farq == 1) return tri_rpf_go<T, kMaxWaves, kLanes, 4, 8, 3, 1>(L, in, out, s);
    }
    return tri_rpf_go<T, kMaxWaves, kLanes, 4, kD64 ? 6 : 8, 2, 4>(L, in, out, s);
  }
  if (L.rp_e == 8) {
    if (L.rp_farq == 0) return tri_rpf_go<T, kMaxWaves, kLanes, 8, kD64 ? 5 : 8, 1, 0>(L, in, out, s);
    return tri_rpf_go<T, kMaxWaves, kLanes, 8, kD64 ? 4 : 6, 2, 8>(L, in, out, s);
  }
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t tri_rpf(const TriLayout& L, const T* in, T* out, hipStream_t s) {
  if (L.rp_waves < 1 || L.rp_waves > kRpfMaxWaves) return hipErrorInvalidValue;
  if (L.rp_lanes > 1)
    return L.rp_waves == 1 ? tri_rpf_layout<T, 1, true>(L, in, out, s)
                           : tri_rpf_layout<T, 8, true>(L, in, out, s);
  return L.rp_waves == 1 ? tri_rpf_layout<T, 1, false>(L, in, out, s)
                         : tri_rpf_layout<T, 8, false>(L, in, out, s);
}

// One level, many workgroups, level-ordered layout.
template <typename T, TriKind K>
__global__ __launch_bounds__(kBlock) void k_tri_level_pre(
    const int* __restrict__ lrow, const int* __restrict__ lbeg,
    const int* __restrict__ lcol, const T* __restrict__ lval,
    const int* __restrict__ ecol, const T* __restrict__ eval,
    const T* __restrict__ ldiag, int bit, int dbit, int row_begin, int row_end,
    const T* __restrict__ in, T* out) {
  const int idx = row_begin + blockIdx.x * kBlock + threadIdx.x;
  if (idx >= row_end) return;
  PreRow<T> r;
  pre_meta<T, K>(r, idx, row_end, lrow, lbeg, ecol, eval, ldiag);
  pre_in<T>(r, in);
  out[r.row] = pre_eval<T, K, false>(r, bit, dbit, lcol, lval, out, nullptr, 0);
}

// One level of an integer factor, `G` lanes per row: each lane sums a
// strided share of the row's entries (integer sums are order-free), the
// group reduces with shuffles and its first lane finishes the row.
template <TriKind K, int G>
__global__ __launch_bounds__(kBlock) void k_tri_level_g(
    const int* __restrict__ lrow, const int* __restrict__ lbeg, const int* __restrict__ lcol,
    const int32_t* __restrict__ lval, const int32_t* __restrict__ ldiag, int bit, int dbit,
    int row_begin, int row_end, const int32_t* __restrict__ in, int32_t* out) {
  const int gid = blockIdx.x * kBlock + threadIdx.x;
  const int idx = row_begin + gid / G;
  const int lane = gid & (G - 1);
  uint64_t acc = 0;
  if (idx < row_end) {
    const int pb = lbeg[idx], pe = lbeg[idx + 1];
    for (int p = pb + lane; p < pe; p += G) acc += prod64(lval[p], out[lcol[p]]);
  }
#pragma unroll
  for (int m = G / 2; m > 0; m >>= 1) acc += shfl_xor_u64(acc, m);
  if (idx < row_end && lane == 0) {
    const int row = lrow[idx];
    const uint64_t tt = (static_cast<uint64_t>(static_cast<int64_t>(in[row])) << bit) - acc;
    out[row] = acc_final<int32_t, K>(tt, ldiag[idx], bit, dbit);
  }
}

template <TriKind K>
hipError_t tri_level_group(const TriLayout& L, const TriSegment& seg, int bit, int dbit,
                           const int32_t* in, int32_t* out, hipStream_t s) {
  const long long threads = static_cast<long long>(seg.row_end - seg.row_begin) * seg.group;
  const int grid = static_cast<int>((threads + kBlock - 1) / kBlock);
  if (grid <= 0) return hipSuccess;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, s, L.lrow, L.lbeg, L.lcol,
                       static_cast<const int32_t*>(L.lval),
                       static_cast<const int32_t*>(L.ldiag), bit, dbit, seg.row_begin,
                       seg.row_end, in, out);
    return hipGetLastError();
  };
  switch (seg.group) {
    case 2: return go(&k_tri_level_g<K, 2>);
    case 4: return go(&k_tri_level_g<K, 4>);
    case 8: return go(&k_tri_level_g<K, 8>);
    case 16: return go(&k_tri_level_g<K, 16>);
    case 32: return go(&k_tri_level_g<K, 32>);
    case 64: return go(&k_tri_level_g<K, 64>);
    default: return hipErrorInvalidValue;
  }
}

template <typename T, TriKind K>
hipError_t tri_pre_seg(const TriLayout& L, const TriSegment& seg, int bit, int dbit,
                       const void* in, void* out, hipStream_t s) {
  if constexpr (std::is_same_v<T, int32_t>) {
    if (!seg.chain_kernel && seg.group > 1)
      return tri_level_group<K>(L, seg, bit, dbit, static_cast<const int32_t*>(in),
                                static_cast<int32_t*>(out), s);
  }
  const T* vin = static_cast<const T*>(in);
  T* vout = static_cast<T*>(out);
  const T* lval = static_cast<const T*>(L.lval);
  const T* eval = static_cast<const T*>(L.eval);
  const T* ldiag = static_cast<const T*>(L.ldiag);
  if (seg.chain_kernel) {
    if (seg.nchain <= 0) return hipSuccess;
    if (L.ring > 0) {
      const size_t lds = sizeof(T) * static_cast<size_t>(L.ring);
      static bool attr = false;
      if (!attr) {
        hipError_t e = hipFuncSetAttribute(
            reinterpret_cast<const void*>(&k_tri_chain_pre<T, K, true>),
            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kTriBlockedMaxLds));
        if (e != hipSuccess) return e;
        attr = true;
      }
      hipLaunchKernelGGL((k_tri_chain_pre<T, K, true>), dim3(seg.nchain), dim3(kChainBlock),
                         lds, s, L.lrow, L.lbeg, L.lpos, lval, L.epos, eval, ldiag, bit, dbit,
                         L.lev_ptr, seg.chain_lev, L.ring - 1, vin, vout);
    } else {
      hipLaunchKernelGGL((k_tri_chain_pre<T, K, false>), dim3(seg.nchain),
                         dim3(kChainBlock), 0, s, L.lrow, L.lbeg, L.lcol, lval, L.ecol, eval,
                         ldiag, bit, dbit, L.lev_ptr, seg.chain_lev, 0, vin, vout);
    }
  } else {
    const int rows = seg.row_end - seg.row_begin;
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_tri_level_pre<T, K>), dim3((rows + kBlock - 1) / kBlock),
                       dim3(kBlock), 0, s, L.lrow, L.lbeg, L.lcol, lval, L.ecol, eval, ldiag,
                       bit, dbit, seg.row_begin, seg.row_end, vin, vout);
  }
  return hipGetLastError();
}

}  // namespace

template <typename T, int MODE>
hipError_t spmv_sell(const DCsr& a, const void* x, const void* z, void* y, hipStream_t s) {
  const int grid = (a.n + kBlock - 1) / kBlock;
  if (grid == 0) return hipSuccess;
  const int remap = a.remap >= 0 ? a.remap : xcd_remap();
  if constexpr (std::is_same_v<T, int32_t>) {
    if (a.scol16) {
      launch_timed(&k_spmv_sell16_int<MODE>, dim3(grid), dim3(kBlock), 0, s, a.n, a.soff,
                   a.scol16, static_cast<const int32_t*>(a.sval), a.bit,
                   static_cast<const int32_t*>(x), static_cast<const int32_t*>(z),
                   static_cast<int32_t*>(y), remap);
      return hipGetLastError();
    }
    launch_timed(&k_spmv_sell_int<MODE>, dim3(grid), dim3(kBlock), 0, s, a.n, a.soff, a.scol,
                 static_cast<const int32_t*>(a.sval), a.srow, a.bit,
                 static_cast<const int32_t*>(x),
                 static_cast<const int32_t*>(z), static_cast<int32_t*>(y), remap);
  } else {
    launch_timed(&k_spmv_sell_fp<T, MODE>, dim3(grid), dim3(kBlock), 0, s, a.n, a.soff, a.scol,
                 static_cast<const T*>(a.sval), a.srow, static_cast<const T*>(x),
                 static_cast<const T*>(z), static_cast<T*>(y), remap);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t spmv_sell_mode(const DCsr& a, int md, const void* x, const void* z, void* y,
                          hipStream_t s) {
  if (md == 0) return spmv_sell<T, 0>(a, x, z, y, s);
  if (md == 1) return spmv_sell<T, 1>(a, x, z, y, s);
  return spmv_sell<T, 2>(a, x, z, y, s);
}

hipError_t launch_spmv_rows_unknown(const DCsr& a, const void* x, void* y, hipStream_t s) {
  if (a.n >= 128 * 512) return spmv_stream_go<128, 0, true>(a, x, nullptr, y, s);
  if (a.n >= 32 * 512) return spmv_stream_go<32, 0, true>(a, x, nullptr, y, s);
  if (a.n >= 1024) return spmv_stream_go<16, 0, true>(a, x, nullptr, y, s);
  return spmv_stream_go<4, 0, true>(a, x, nullptr, y, s);
}

hipError_t launch_spmv(Elem e, const DCsr& a, SpmvMode mode, const void* x,
                       const void* z, void* y, hipStream_t s) {
  const int md = static_cast<int>(mode);
  if (a.soff) {
    if (e == Elem::kI32) return spmv_sell_mode<int32_t>(a, md, x, z, y, s);
    if (e == Elem::kF64) return spmv_sell_mode<double>(a, md, x, z, y, s);
    return spmv_sell_mode<float>(a, md, x, z, y, s);
  }
  if (e == Elem::kI32) {
    if (md == 0) return spmv_int_mode<0>(a, x, z, y, s);
    if (md == 1) return spmv_int_mode<1>(a, x, z, y, s);
    return spmv_int_mode<2>(a, x, z, y, s);
  }
  if (e == Elem::kF64) {
    if (md == 0) return spmv_fp<double, 0>(a, x, z, y, s);
    if (md == 1) return spmv_fp<double, 1>(a, x, z, y, s);
    return spmv_fp<double, 2>(a, x, z, y, s);
  }
  if (md == 0) return spmv_fp<float, 0>(a, x, z, y, s);
  if (md == 1) return spmv_fp<float, 1>(a, x, z, y, s);
  return spmv_fp<float, 2>(a, x, z, y, s);
}

size_t tri_blocked_lds(int n, size_t elem, size_t acc) {
  size_t b = acc * n + 2 * elem * n;
  b = (b + 15) & ~static_cast<size_t>(15);
  return b + 8 * kTB + elem * kTB * kTB;
}

// Blocks per workgroup: the most whose tiles fit in LDS with one workgroup per
// CU (kB (kB + 1) / 2 of them); one for a block of right-hand sides, whose many
// workgroups share the CUs with other systems' kernels.
template <typename T, bool kShort, int kS>
static hipError_t tri_tiles_go(TriKind kind, int n, int nb, int nrhs, const void* tiles,
                               const long long* toff, const uint64_t* tmask, const void* dinv,
                               int bit, int dbit, const void* in, void* out,
                               unsigned long long* xp, int epoch, int* err, unsigned* tickets,
                               hipStream_t s) {
  if (n <= 0 || nrhs <= 0) return hipSuccess;
  if (nb > kTileMaxBlocks) return hipErrorInvalidValue;
  constexpr int kB = kS > 1 ? 1 : sizeof(T) == 8 ? 2 : 3;
  constexpr size_t lds = sizeof(T) * kTB * kTB * kB * (kB + 1) / 2;
  auto go = [&](auto kern, bool& attr) -> hipError_t {
    if (!attr) {
      const hipError_t e =
          hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                              hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
      if (e != hipSuccess) return e;
      attr = true;
    }
    hipLaunchKernelGGL(kern, dim3((nb + kB - 1) / kB * nrhs), dim3(64 * kB), lds, s, n, nb, nrhs, static_cast<const T*>(tiles),
                       toff, tmask, static_cast<const T*>(dinv), bit, dbit,
                       static_cast<const T*>(in), static_cast<T*>(out), xp, epoch, err, tickets);
    return hipGetLastError();
  };
  static bool attr_l = false, attr_du = false;
  if (kind == TriKind::kL) return go(&k_tri_tiles<T, TriKind::kL, kShort, kS, kB>, attr_l);
  if (kind == TriKind::kDU) return go(&k_tri_tiles<T, TriKind::kDU, kShort, kS, kB>, attr_du);
  return hipErrorInvalidValue;  // only the coarse factors are tiled
}

hipError_t launch_trsv_tiles(Elem e, TriKind kind, int n, int nb, const void* tiles,
                             const long long* toff, const uint64_t* tmask, const void* dinv,
                             int bit, int dbit, const void* in, void* out,
                             unsigned long long* xp, int epoch, int* err, unsigned* tickets,
                             hipStream_t s) {
  if (e == Elem::kF64)
    return tri_tiles_go<double, false, 1>(kind, n, nb, 1, tiles, toff, tmask, dinv, 0, 0, in, out,
                                          xp, epoch, err, tickets, s);
  if (e == Elem::kF32)
    return tri_tiles_go<float, false, 1>(kind, n, nb, 1, tiles, toff, tmask, dinv, 0, 0, in, out,
                                         xp, epoch, err, tickets, s);
  const bool in_word = bit >= 0 && bit < 32 && (kind == TriKind::kL || (dbit >= 0 && dbit < 32));
  return in_word ? tri_tiles_go<int32_t, true, 1>(kind, n, nb, 1, tiles, toff, nullptr, dinv, bit,
                                                  dbit, in, out, xp, epoch, err, tickets, s)
                 : tri_tiles_go<int32_t, false, 1>(kind, n, nb, 1, tiles, toff, nullptr, dinv,
                                                   bit, dbit, in, out, xp, epoch, err, tickets, s);
}

hipError_t launch_trsv_tiles_blk(TriKind kind, int n, int nb, int groups, const int32_t* tiles,
                                 const long long* toff, const int32_t* dinv, int bit, int dbit,
                                 const void* in, void* out, unsigned long long* xp, int epoch,
                                 int* err, unsigned* tickets, hipStream_t s) {
  const bool in_word = bit >= 0 && bit < 32 && (kind == TriKind::kL || (dbit >= 0 && dbit < 32));
  return in_word
             ? tri_tiles_go<int32_t, true, 4>(kind, n, nb, 4 * groups, tiles, toff, nullptr, dinv,
                                              bit, dbit, in, out, xp, epoch, err, tickets, s)
             : tri_tiles_go<int32_t, false, 4>(kind, n, nb, 4 * groups, tiles, toff, nullptr,
                                               dinv, bit, dbit, in, out, xp, epoch, err, tickets,
                                               s);
}

hipError_t launch_trsv_blocked(Elem e, TriKind kind, const DCsr& a, const int* bptr,
                               int nb, const void* in, void* out, hipStream_t s) {
  if (e == Elem::kI32) {
    if (kind == TriKind::kL) return tri_blocked<int32_t, TriKind::kL>(a, bptr, nb, in, out, s);
    if (kind == TriKind::kLD) return tri_blocked<int32_t, TriKind::kLD>(a, bptr, nb, in, out, s);
    return tri_blocked<int32_t, TriKind::kDU>(a, bptr, nb, in, out, s);
  }
  if (e == Elem::kF64) {
    if (kind == TriKind::kL) return tri_blocked<double, TriKind::kL>(a, bptr, nb, in, out, s);
    if (kind == TriKind::kLD) return tri_blocked<double, TriKind::kLD>(a, bptr, nb, in, out, s);
    return tri_blocked<double, TriKind::kDU>(a, bptr, nb, in, out, s);
  }
  if (kind == TriKind::kL) return tri_blocked<float, TriKind::kL>(a, bptr, nb, in, out, s);
  if (kind == TriKind::kLD) return tri_blocked<float, TriKind::kLD>(a, bptr, nb, in, out, s);
  return tri_blocked<float, TriKind::kDU>(a, bptr, nb, in, out, s);
}

hipError_t launch_trsv_layout(Elem e, TriKind kind, const TriLayout& L,
                              const TriSegment& seg, int bit, int dbit, const void* in,
                              void* out, hipStream_t s) {
  if (e == Elem::kI32) {
    if (kind == TriKind::kL) return tri_pre_seg<int32_t, TriKind::kL>(L, seg, bit, dbit, in, out, s);
    if (kind == TriKind::kLD) return tri_pre_seg<int32_t, TriKind::kLD>(L, seg, bit, dbit, in, out, s);
    return tri_pre_seg<int32_t, TriKind::kDU>(L, seg, bit, dbit, in, out, s);
  }
  if (e == Elem::kF64) {
    if (kind == TriKind::kL) return tri_pre_seg<double, TriKind::kL>(L, seg, bit, dbit, in, out, s);
    if (kind == TriKind::kLD) return tri_pre_seg<double, TriKind::kLD>(L, seg, bit, dbit, in, out, s);
    return tri_pre_seg<double, TriKind::kDU>(L, seg, bit, dbit, in, out, s);
  }
  if (kind == TriKind::kL) return tri_pre_seg<float, TriKind::kL>(L, seg, bit, dbit, in, out, s);
  if (kind == TriKind::kLD) return tri_pre_seg<float, TriKind::kLD>(L, seg, bit, dbit, in, out, s);
  return tri_pre_seg<float, TriKind::kDU>(L, seg, bit, dbit, in, out, s);
}

hipError_t launch_trsv_ep(TriKind kind, const TriLayout& L, const TriSegment& seg, int bit,
                          int dbit, const void* in_v, void* out_v, hipStream_t s) {
  const int32_t* in = static_cast<const int32_t*>(in_v);
  int32_t* o = static_cast<int32_t*>(out_v);
  const int w = L.ep_waves;
  if (kind == TriKind::kLD) {
    if (w <= 1) return tri_ep_launch<TriKind::kLD, 1>(L, seg, bit, dbit, in, o, s);
    if (w <= 2) return tri_ep_launch<TriKind::kLD, 2>(L, seg, bit, dbit, in, o, s);
    if (w <= 4) return tri_ep_launch<TriKind::kLD, 4>(L, seg, bit, dbit, in, o, s);
    return tri_ep_launch<TriKind::kLD, 8>(L, seg, bit, dbit, in, o, s);
  }
  if (kind == TriKind::kL) {
    if (w <= 1) return tri_ep_launch<TriKind::kL, 1>(L, seg, bit, dbit, in, o, s);
    if (w <= 2) return tri_ep_launch<TriKind::kL, 2>(L, seg, bit, dbit, in, o, s);
    if (w <= 4) return tri_ep_launch<TriKind::kL, 4>(L, seg, bit, dbit, in, o, s);
    return tri_ep_launch<TriKind::kL, 8>(L, seg, bit, dbit, in, o, s);
  }
  if (w <= 1) return tri_ep_launch<TriKind::kDU, 1>(L, seg, bit, dbit, in, o, s);
  if (w <= 2) return tri_ep_launch<TriKind::kDU, 2>(L, seg, bit, dbit, in, o, s);
  if (w <= 4) return tri_ep_launch<TriKind::kDU, 4>(L, seg, bit, dbit, in, o, s);
  return tri_ep_launch<TriKind::kDU, 8>(L, seg, bit, dbit, in, o, s);
}

template <int kS>
static hipError_t trsv_rp_waves(const TriLayout& L, int nrhs, int bit, int dbit,
                                const int32_t* in, int32_t* out, hipStream_t s) {
  if (L.rp_waves <= 1) return tri_rp_far<1, kS>(L, nrhs, bit, dbit, in, out, s);
  if (L.rp_waves <= 8) return tri_rp_far<8, kS>(L, nrhs, bit, dbit, in, out, s);
  return tri_rp_wide<kS>(L, nrhs, bit, dbit, in, out, s);
}

hipError_t launch_trsv_rp(const TriLayout& L, int bit, int dbit, const void* in, void* out,
                          hipStream_t s) {
  return trsv_rp_waves<1>(L, 1, bit, dbit, static_cast<const int32_t*>(in),
                          static_cast<int32_t*>(out), s);
}

bool trsv_rp_blk_supported(const TriLayout& L) {
  return L.rp_waves > 0 && L.n < (1 << 27);  // 32-bit byte offsets into 16 n bytes
}

hipError_t launch_trsv_rp_blk(const TriLayout& L, int groups, int bit, int dbit, const void* in,
                              void* out, hipStream_t s) {
  if (!trsv_rp_blk_supported(L)) return hipErrorInvalidValue;
  // a right-hand side per workgroup in y, whose grids have at most 65,535
  constexpr int kSlice = 65535 / 4;
  for (int g0 = 0; g0 < groups; g0 += kSlice) {
    const size_t off = static_cast<size_t>(g0) * L.n * 4;
    const hipError_t e =
        trsv_rp_waves<4>(L, 4 * std::min(kSlice, groups - g0), bit, dbit,
                         static_cast<const int32_t*>(in) + off, static_cast<int32_t*>(out) + off, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_trsv_rpf(Elem e, const TriLayout& L, const void* in, void* out,
                           hipStream_t s) {
  if (e == Elem::kF64)
    return tri_rpf<double>(L, static_cast<const double*>(in), static_cast<double*>(out), s);
  if (e == Elem::kF32)
    return tri_rpf<float>(L, static_cast<const float*>(in), static_cast<float*>(out), s);
  return hipErrorInvalidValue;
}

}  // namespace sc23ad::dev
