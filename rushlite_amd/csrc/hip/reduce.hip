// Keep-dims reductions over the middle axis of a contiguous [outer, len,
// inner] view (Lamp3: cpu/reduct.cpp:7-49 for the semantics, reduct.cu:213-260
// for the CUDA dispatcher this replaces).
//
// Row case (inner == 1, e.g. sum/max over dim 1 of [16384,16384]):
//   long fp32 rows  -> one 256-thread workgroup per row segment, 128-bit
//                      loads, 16 independent accumulators per lane, wave64
//                      butterfly (DPP lane swaps) then LDS across the 4 waves;
//                      a row is split over several workgroups only when
//                      there are too few rows to fill 256 CUs, and the
//                      partials are folded by a second pass in fixed order.
//   other long rows -> (odd lengths, other types) the same with units of
//                      one value, or of 16 bytes where the type, length and
//                      alignment allow, in longer parts whose results are a row
//                      of their own to reduce.
//   short rows      -> one wave per row (softmax/loss rows like [512,1000]),
//                      float4 loads when rows are 16-byte multiples, four
//                      loads in flight per lane; rows of at most 32 units
//                      share a wave, 8 to 32 lanes each.
// Column case (inner > 1, e.g. sum over dim 0, the bias-gradient reduction):
//   units of 16 bytes along the columns where the type, inner extent and
//   alignment allow, one value otherwise.  A workgroup owns a strip of up to
//   1 KiB of one outer slice (the strips of a slice evenly wide) and a chunk
//   of the reduced axis; its 256 lanes are row groups that take every rg-th row
//   (8 loads in flight per lane) and combine in LDS by halving in fixed order.
//   The axis is cut into S chunks so the grid holds about four workgroups per
//   CU; the same kernel folds the chunk partials [outer, S, inner].  A short
//   axis that would need chunks (bias gradients: [batch, out] with a batch of a
//   few hundred) takes narrower strips instead, down to 64 bytes, so there is
//   no second launch.
//   Slices of a few units, and short axes of many outputs, take a lane per
//   output.  No atomics: results are deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "common.hpp"
#include "ops.hpp"
#include "row_split.hpp"

namespace lmp_hip {

typedef float v4f __attribute__((ext_vector_type(4)));

namespace {

constexpr int kBlock = kRowLanes;
constexpr int kWaves = kBlock / 64;

#define LMP_WAVE_SWAP_SRC(...) __VA_ARGS__
#include "wave_swap.inc"
#undef LMP_WAVE_SWAP_SRC

// Butterfly over the 64 lanes in the order 1, 2, 4, 8, 16, 32; lane 0 holds
// the result.
template <int OP, typename T>
__device__ __forceinline__ T wave_reduce(T v) {
  using R = Reducer<OP, T>;
  v = R::combine(v, lmp_swap<1>(v));
  v = R::combine(v, lmp_swap<2>(v));
  v = R::combine(v, lmp_swap<4>(v));
  v = R::combine(v, lmp_swap<8>(v));
  v = R::combine(v, lmp_swap<16>(v));
  v = R::combine(v, lmp_swap<32>(v));
  return v;
}

template <int OP>
__device__ __forceinline__ v4f combine4(v4f a, v4f b) {
  v4f r;
  r.x = Reducer<OP, float>::combine(a.x, b.x);
  r.y = Reducer<OP, float>::combine(a.y, b.y);
  r.z = Reducer<OP, float>::combine(a.z, b.z);
  r.w = Reducer<OP, float>::combine(a.w, b.w);
  return r;
}

// Inputs of kStreamBytes or more are read with the nontemporal hint.
template <bool NT>
__device__ __forceinline__ v4f load4(const v4f* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// V consecutive values, loaded and stored at once.
template <typename T, int V>
struct alignas(sizeof(T) * V) Pack {
  T x[V];
};
template <int OP, typename T, int V>
__device__ __forceinline__ Pack<T, V> combine_pack(Pack<T, V> a, const Pack<T, V>& b) {
#pragma unroll
  for (int i = 0; i < V; ++i) a.x[i] = Reducer<OP, T>::combine(a.x[i], b.x[i]);
  return a;
}
template <int OP, typename T, int V>
__device__ __forceinline__ Pack<T, V> identity_pack() {
  Pack<T, V> p;
#pragma unroll
  for (int i = 0; i < V; ++i) p.x[i] = Reducer<OP, T>::identity();
  return p;
}
template <bool NT, typename T, int V>
__device__ __forceinline__ Pack<T, V> load_pack(const Pack<T, V>* p) {
  if constexpr (NT) {
    const v4f v = __builtin_nontemporal_load(reinterpret_cast<const v4f*>(p));
    return __builtin_bit_cast(Pack<T, V>, v);
  } else {
    return *p;
  }
}

// Block (row, part) reduces float4 [part*seg4, min(len4, (part+1)*seg4)) of
// its row and writes one value to out[row * parts + part].
template <int OP, bool NT>
__global__ __launch_bounds__(kBlock) void row_reduce_f32(
    float* __restrict__ out, const float* __restrict__ in, uint32_t len4,
    uint32_t seg4, FastDiv parts) {
  using R = Reducer<OP, float>;
  const uint32_t row = parts.div(blockIdx.x);
  const uint32_t part = blockIdx.x - row * parts.d;
  const v4f* src = reinterpret_cast<const v4f*>(in) + uint64_t(row) * len4;
  const uint32_t beg = part * seg4;
  const uint32_t end = min(len4, beg + seg4);
  const v4f id = v4f(R::identity());
  v4f acc0 = id, acc1 = id, acc2 = id, acc3 = id;
  uint32_t i = beg + threadIdx.x;
  for (; i + 3 * kBlock < end; i += 4 * kBlock) {
    v4f x0 = load4<NT>(src + i), x1 = load4<NT>(src + i + kBlock),
        x2 = load4<NT>(src + i + 2 * kBlock), x3 = load4<NT>(src + i + 3 * kBlock);
    acc0 = combine4<OP>(acc0, x0);
    acc1 = combine4<OP>(acc1, x1);
    acc2 = combine4<OP>(acc2, x2);
    acc3 = combine4<OP>(acc3, x3);
  }
  for (; i < end; i += kBlock) acc0 = combine4<OP>(acc0, load4<NT>(src + i));
  v4f acc = combine4<OP>(combine4<OP>(acc0, acc1), combine4<OP>(acc2, acc3));
  float v = R::combine(R::combine(acc.x, acc.y), R::combine(acc.z, acc.w));
  v = wave_reduce<OP, float>(v);
  __shared__ float lds[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    float r = lds[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) r = R::combine(r, lds[w]);
    out[blockIdx.x] = r;
  }
}

// One wave per row, any dtype, any length.  Four loads per lane are issued
// before they are combined (four accumulators), so a short row costs one
// memory latency rather than one per 64 elements.
template <int OP, typename T>
__global__ __launch_bounds__(kBlock) void row_reduce_wave(
    T* __restrict__ out, const T* __restrict__ in, uint64_t rows,
    uint64_t len) {
  using R = Reducer<OP, T>;
  const uint64_t row = uint64_t(blockIdx.x) * kWaves + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const T* src = in + row * len;
  T a0 = R::identity(), a1 = a0, a2 = a0, a3 = a0;
  uint64_t j = lane;
  for (; j + 192 < len; j += 256) {
    const T x0 = src[j], x1 = src[j + 64], x2 = src[j + 128], x3 = src[j + 192];
    a0 = R::combine(a0, x0);
    a1 = R::combine(a1, x1);
    a2 = R::combine(a2, x2);
    a3 = R::combine(a3, x3);
  }
  // At most three elements per lane remain (j + 192 >= len): their loads go
  // out together, then a0 takes them in index order as a loop would.
  {
    const bool t0 = j < len, t1 = j + 64 < len, t2 = j + 128 < len;
    T y0 = a0, y1 = a0, y2 = a0;
    if (t0) y0 = src[j];
    if (t1) y1 = src[j + 64];
    if (t2) y2 = src[j + 128];
    if (t0) a0 = R::combine(a0, y0);
    if (t1) a0 = R::combine(a0, y1);
    if (t2) a0 = R::combine(a0, y2);
  }
  T acc = R::combine(R::combine(a0, a1), R::combine(a2, a3));
  acc = wave_reduce<OP, T>(acc);
  if (lane == 0) out[row] = acc;
}

// One wave per fp32 row with 16-byte rows (len % 4 == 0): float4 loads, four
// in flight per lane.
template <int OP>
__global__ __launch_bounds__(kBlock) void row_reduce_wave_f32(
    float* __restrict__ out, const float* __restrict__ in, uint64_t rows,
    uint32_t len4) {
  using R = Reducer<OP, float>;
  const uint64_t row = uint64_t(blockIdx.x) * kWaves + (threadIdx.x >> 6);
  if (row >= rows) return;
  const uint32_t lane = threadIdx.x & 63;
  const v4f* src = reinterpret_cast<const v4f*>(in) + row * len4;
  const v4f id = v4f(R::identity());
  v4f a0 = id, a1 = id, a2 = id, a3 = id;
  uint32_t j = lane;
  for (; j + 192 < len4; j += 256) {
    const v4f x0 = src[j], x1 = src[j + 64], x2 = src[j + 128], x3 = src[j + 192];
    a0 = combine4<OP>(a0, x0);
    a1 = combine4<OP>(a1, x1);
    a2 = combine4<OP>(a2, x2);
    a3 = combine4<OP>(a3, x3);
  }
  // At most three float4 per lane remain (j + 192 >= len4): their loads go
  // out together, then a0 takes them in index order as a loop would.
  {
    const bool t0 = j < len4, t1 = j + 64 < len4, t2 = j + 128 < len4;
    v4f y0 = id, y1 = id, y2 = id;
    if (t0) y0 = src[j];
    if (t1) y1 = src[j + 64];
    if (t2) y2 = src[j + 128];
    if (t0) a0 = combine4<OP>(a0, y0);
    if (t1) a0 = combine4<OP>(a0, y1);
    if (t2) a0 = combine4<OP>(a0, y2);
  }
  const v4f a = combine4<OP>(combine4<OP>(a0, a1), combine4<OP>(a2, a3));
  float v = R::combine(R::combine(a.x, a.y), R::combine(a.z, a.w));
  v = wave_reduce<OP, float>(v);
  if (lane == 0) out[row] = v;
}

// Long rows of any type: row_reduce_f32 with units of V values (len, a multiple
// of V, counted in units), the waves' results in pairs.  [2048, 10001] fp32 (one
// wave a row before) 23.5 -> 15.3 us, 5.35 TB/s.
template <int OP, typename T, int V>
__global__ __launch_bounds__(kBlock) void row_reduce_block(T* __restrict__ out,
                                                           const T* __restrict__ in, uint32_t units,
                                                           uint32_t seg, FastDiv parts) {
  using R = Reducer<OP, T>;
  using P = Pack<T, V>;
  const uint32_t row = parts.div(blockIdx.x);
  const uint32_t part = blockIdx.x - row * parts.d;
  const P* src = reinterpret_cast<const P*>(in) + uint64_t(row) * units;
  const uint32_t end = min(units, (part + 1) * seg);
  P acc[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) acc[u] = identity_pack<OP, T, V>();
  uint32_t i = part * seg + threadIdx.x;
  for (; i + 3 * kBlock < end; i += 4 * kBlock) {
    P x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = src[i + u * kBlock];
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] = combine_pack<OP>(acc[u], x[u]);
  }
  {  // at most three units per lane remain: their loads go out together
    P x[3];
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      x[u] = identity_pack<OP, T, V>();
      if (i + u * kBlock < end) x[u] = src[i + u * kBlock];
    }
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (i + u * kBlock < end) acc[0] = combine_pack<OP>(acc[0], x[u]);
  }
  P a = combine_pack<OP>(combine_pack<OP>(acc[0], acc[1]), combine_pack<OP>(acc[2], acc[3]));
#pragma unroll
  for (int w = 1; w < V; w *= 2)
#pragma unroll
    for (int j = 0; j + w < V; j += 2 * w) a.x[j] = R::combine(a.x[j], a.x[j + w]);
  const T v = wave_reduce<OP, T>(a.x[0]);
  __shared__ T lds[kWaves];
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  static_assert(kWaves == 4, "two pairs");
  if (threadIdx.x == 0)
    out[blockIdx.x] = R::combine(R::combine(lds[0], lds[1]), R::combine(lds[2], lds[3]));
}

// Rows of at most 32 units, G = 8, 16 or 32 lanes each (64 / G rows per wave):
// a lane holds at most one unit, so the butterfly's first steps, which stay
// inside the G lanes, give the bits of the one-wave kernels (whose other lanes
// hold the identity).  [65536, 8] fp32: 8.3 -> 3.7 us.
template <int OP, typename T, int V, int G>
__global__ __launch_bounds__(kBlock) void row_reduce_small(T* __restrict__ out,
                                                           const T* __restrict__ in, uint64_t rows,
                                                           uint32_t units) {
  using R = Reducer<OP, T>;
  const uint64_t row = (uint64_t(blockIdx.x) * kBlock + threadIdx.x) / G;
  const uint32_t lane = threadIdx.x % G;
  Pack<T, V> a = identity_pack<OP, T, V>();
  if (row < rows && lane < units)
    a = combine_pack<OP>(a, reinterpret_cast<const Pack<T, V>*>(in)[row * units + lane]);
#pragma unroll
  for (int w = 1; w < V; w *= 2)
#pragma unroll
    for (int j = 0; j + w < V; j += 2 * w) a.x[j] = R::combine(a.x[j], a.x[j + w]);
  T v = a.x[0];
  v = R::combine(v, lmp_swap<1>(v));
  v = R::combine(v, lmp_swap<2>(v));
  v = R::combine(v, lmp_swap<4>(v));
  if constexpr (G > 8) v = R::combine(v, lmp_swap<8>(v));
  if constexpr (G > 16) v = R::combine(v, lmp_swap<16>(v));
  if (lane == 0 && row < rows) out[row] = v;
}

// Fold `parts` consecutive partials per output in order.
template <int OP>
__global__ __launch_bounds__(kBlock) void fold_parts(float* __restrict__ out,
                                                     const float* __restrict__ part,
                                                     uint64_t n,
                                                     uint32_t parts) {
  using R = Reducer<OP, float>;
  const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i >= n) return;
  float acc = R::identity();
  for (uint32_t p = 0; p < parts; ++p) acc = R::combine(acc, part[i * parts + p]);
  out[i] = acc;
}

// Column reduction, V values per unit.  Workgroup (o, s, b) owns units
// [b * cw, b * cw + cw) of slice o and rows [s * chunk, s * chunk + chunk);
// lane t takes unit t % cw and, of rg = 256 / cw row groups, rows t / cw +
// rg * i, eight loads in flight.  dst layout [outer, S, units] (S == 1 writes
// the final result).  HBM-bound: sum over the middle axis of [256, 197, 768]
// 51.6 -> 28.8 us (5.4 TB/s; fp32 strips were sized without the outer extent:
// 64-byte rows), over dim 0 of [16384, 16384] 158.5 us (6.8 TB/s; 159 before), float64
// 352 -> 317 us and int32 184 -> 164 us (units of one value before), of
// [200000, 64] fp32 59 -> 14 us, float64 272 -> 21 us (the partials folded by one
// lane per column), [16384, 3] 27.6 -> 6.5 us (three lanes of 256).
constexpr int kColUnroll = 8;
template <int OP, typename T, int V, bool NT>
__global__ __launch_bounds__(kBlock) void col_reduce_tile(T* __restrict__ dst,
                                                          const T* __restrict__ in, uint32_t units,
                                                          uint32_t len, uint32_t chunk, FastDiv cw,
                                                          FastDiv strips, FastDiv S) {
  using P = Pack<T, V>;
  const uint32_t q = strips.div(blockIdx.x), b = blockIdx.x - q * strips.d;
  const uint32_t o = S.div(q), s = q - o * S.d;
  const uint32_t g = cw.div(threadIdx.x), col = threadIdx.x - g * cw.d;
  const uint32_t rg = cw.div(uint32_t(kBlock)), c = b * cw.d + col;
  const uint32_t r1 = min(len, (s + 1) * chunk);
  P acc[kColUnroll];
#pragma unroll
  for (int u = 0; u < kColUnroll; ++u) acc[u] = identity_pack<OP, T, V>();
  if (c < units && g < rg) {
    const P* src = reinterpret_cast<const P*>(in) + uint64_t(o) * len * units + c;
    uint32_t r = s * chunk + g;
    for (; r + rg * (kColUnroll - 1) < r1; r += rg * kColUnroll) {
      P x[kColUnroll];
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u) x[u] = load_pack<NT>(src + uint64_t(r + rg * u) * units);
#pragma unroll
      for (int u = 0; u < kColUnroll; ++u) acc[u] = combine_pack<OP>(acc[u], x[u]);
    }
    if (r < r1) {  // at most seven rows remain: their loads go out together too
      P x[kColUnroll - 1];
#pragma unroll
      for (int u = 0; u < kColUnroll - 1; ++u) {
        x[u] = identity_pack<OP, T, V>();
        if (r + rg * u < r1) x[u] = load_pack<NT>(src + uint64_t(r + rg * u) * units);
      }
#pragma unroll
      for (int u = 0; u < kColUnroll - 1; ++u) acc[u] = combine_pack<OP>(acc[u], x[u]);
    }
  }
#pragma unroll
  for (int w = kColUnroll / 2; w >= 1; w /= 2)
#pragma unroll
    for (int u = 0; u < w; ++u) acc[u] = combine_pack<OP>(acc[u], acc[u + w]);
  P a = acc[0];
  __shared__ P lds[kBlock];
  lds[threadIdx.x] = a;
  for (uint32_t n = rg; n > 1;) {
    const uint32_t half = (n + 1) / 2;
    __syncthreads();
    if (g < n - half) {
      a = combine_pack<OP>(a, lds[threadIdx.x + half * cw.d]);
      lds[threadIdx.x] = a;
    }
    n = half;
  }
  if (g == 0 && c < units)
    reinterpret_cast<P*>(dst)[(uint64_t(o) * S.d + s) * units + c] = a;
}

// One lane per output unit of [outer, units]: short slices, or an axis whose
// outputs alone fill the chip.  Eight accumulators as above.
template <int OP, typename T, int V>
__global__ __launch_bounds__(kBlock) void col_reduce_lane(T* __restrict__ out,
                                                          const T* __restrict__ in, uint64_t n,
                                                          FastDiv by_units, uint32_t len) {
  using P = Pack<T, V>;
  const uint32_t i = blockIdx.x * kBlock + threadIdx.x;  // below 2^32: the launch's threads
  if (i >= n) return;
  const uint32_t units = by_units.d, o = by_units.div(i), c = i - o * units;
  const P* src = reinterpret_cast<const P*>(in) + uint64_t(o) * len * units + c;
  P acc[kColUnroll];
#pragma unroll
  for (int u = 0; u < kColUnroll; ++u) acc[u] = identity_pack<OP, T, V>();
  uint32_t r = 0;
  for (; r + kColUnroll <= len; r += kColUnroll) {
    P x[kColUnroll];
#pragma unroll
    for (int u = 0; u < kColUnroll; ++u) x[u] = src[uint64_t(r + u) * units];
#pragma unroll
    for (int u = 0; u < kColUnroll; ++u) acc[u] = combine_pack<OP>(acc[u], x[u]);
  }
  for (; r < len; ++r) acc[0] = combine_pack<OP>(acc[0], src[uint64_t(r) * units]);
#pragma unroll
  for (int w = kColUnroll / 2; w >= 1; w /= 2)
#pragma unroll
    for (int u = 0; u < w; ++u) acc[u] = combine_pack<OP>(acc[u], acc[u + w]);
  reinterpret_cast<P*>(out)[i] = acc[0];
}

// Column reduction with one lane per output element (o, c) of [outer, inner],
// grid-striding over them: the axis is folded sequentially from the identity
// (eight loads in flight, combined in row order).  For more than 65535 outer
// slices, whose results are the sequential fold's bit for bit, as
// cpu/reduct.cpp:15-19 forms them, and for what the kernels above do not count:
// extents of 2^31 or more, or more workgroups than a grid holds
// (reduct.cu:166-182 grid-strides over any output count too).
template <int OP, typename T>
__global__ __launch_bounds__(kBlock) void col_reduce_flat(T* __restrict__ out,
                                                          const T* __restrict__ in,
                                                          uint64_t outer, uint64_t len,
                                                          uint64_t inner) {
  using R = Reducer<OP, T>;
  const uint64_t n = outer * inner;
  const uint64_t stride = uint64_t(gridDim.x) * kBlock;
  for (uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
    const uint64_t o = i / inner, c = i - o * inner;
    const T* src = in + o * len * inner + c;
    T acc = R::identity();
    uint64_t r = 0;
    for (; r + 8 <= len; r += 8, src += 8 * inner) {
      T x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = src[u * inner];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = R::combine(acc, x[u]);
    }
    for (; r < len; ++r, src += inner) acc = R::combine(acc, *src);
    out[i] = acc;
  }
}

bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

constexpr uint64_t kStripMaxLen = 4096;

uint32_t blocks_for(uint64_t n) { return uint32_t((n + kBlock - 1) / kBlock); }

// The float4 row and column kernels index within a row or a column with
// 32-bit counters that run up to a few hundred past the extent (and a chunk
// start plus a chunk length): extents of 2^31 float4 (rows) or 2^31 rows
// (columns) or more take the 64-bit kernels instead.
constexpr uint64_t kMaxU32Extent = 0x7fffffffull;

// Units of 16 bytes where the type, the contiguous extent and the address
// allow, else of one value.
template <typename T>
constexpr int kPackOf = sizeof(T) >= 2 ? int(16 / sizeof(T)) : 1;
template <typename T>
bool packs(const void* p, uint64_t extent) {
  return kPackOf<T> > 1 && extent % kPackOf<T> == 0 && aligned16(p);
}

template <int OP, typename T, int V, int G>
int launch_small_rows(Runtime* rt, T* out, const T* in, uint64_t rows, uint64_t units) {
  hipLaunchKernelGGL((row_reduce_small<OP, T, V, G>), dim3(blocks_for(rows * G)), dim3(kBlock), 0,
                     rt->stream, out, in, rows, uint32_t(units));
  LMP_LAUNCH_CHECK("row_reduce_small");
  return LMP_OK;
}

template <int OP, typename T>
int reduce_rows(Runtime* rt, T* out, const T* in, uint64_t rows, uint64_t len);

// Rows of V-value units: short ones several to a wave, long ones a workgroup
// (or several) each; *done false where neither applies.
template <int OP, typename T, int V>
int reduce_rows_as(Runtime* rt, T* out, const T* in, uint64_t rows, uint64_t len, bool* done) {
  const uint64_t units = len / V;
  *done = true;
  if (units <= 32 && rows <= 0x7fffffffull) {
    if (units <= 8) return launch_small_rows<OP, T, V, 8>(rt, out, in, rows, units);
    if (units <= 16) return launch_small_rows<OP, T, V, 16>(rt, out, in, rows, units);
    return launch_small_rows<OP, T, V, 32>(rt, out, in, rows, units);
  }
  if (len >= kLongRow && units <= kMaxU32Extent) {
    constexpr bool kFloat4 = std::is_same_v<T, float> && V == 4;
    const uint64_t parts = row_parts(uint64_t(rt->cu_count), rows, units,
                                     kFloat4 ? RowUnits::Float4 : RowUnits::Other);
    const uint64_t seg = (units + parts - 1) / parts;
    if (rows * parts > 0x7fffffffull) return fail(LMP_ERR_UNSUPPORTED, "reduce: too many rows");
    T* dst = out;
    T* tmp = nullptr;
    if (parts > 1) {
      tmp = static_cast<T*>(scratch_alloc(rows * parts * sizeof(T)));
      if (!tmp) return LMP_ERR_OOM;
      dst = tmp;
    }
    const dim3 grid{uint32_t(rows * parts)};
    if constexpr (kFloat4) {
      // Enough workgroups in flight, and the nontemporal hint for inputs that
      // cannot stay in the MALL.
      if (rows * len * sizeof(T) >= kStreamBytes)
        hipLaunchKernelGGL((row_reduce_f32<OP, true>), grid, dim3(kBlock), 0, rt->stream, dst, in,
                           uint32_t(units), uint32_t(seg), FastDiv(uint32_t(parts)));
      else
        hipLaunchKernelGGL((row_reduce_f32<OP, false>), grid, dim3(kBlock), 0, rt->stream, dst,
                           in, uint32_t(units), uint32_t(seg), FastDiv(uint32_t(parts)));
      LMP_LAUNCH_CHECK("row_reduce_f32");
    } else {
      hipLaunchKernelGGL((row_reduce_block<OP, T, V>), grid, dim3(kBlock), 0, rt->stream, dst, in,
                         uint32_t(units), uint32_t(seg), FastDiv(uint32_t(parts)));
      LMP_LAUNCH_CHECK("row_reduce_block");
    }
    if (parts > 1) {
      int rc = LMP_OK;
      if constexpr (kFloat4) {
        hipLaunchKernelGGL((fold_parts<OP>), dim3(blocks_for(rows)), dim3(kBlock), 0, rt->stream,
                           out, tmp, rows, uint32_t(parts));
        LMP_LAUNCH_CHECK("fold_parts");
      } else {
        // Parts of many rounds: few enough for a row reduction of their own (one
        // lane adding 976 of them took 60 of the 64 us of [1, 1000001]).
        rc = reduce_rows<OP, T>(rt, out, tmp, rows, parts);
      }
      scratch_free(tmp);  // stream-ordered: the second pass reads it first
      return rc;
    }
    return LMP_OK;
  }
  *done = false;
  return LMP_OK;
}

template <int OP, typename T>
int reduce_rows(Runtime* rt, T* out, const T* in, uint64_t rows, uint64_t len) {
  // A wave (long rows: a workgroup) per row, 2^31 threads a launch at most.
  if ((rows + kWaves - 1) / kWaves > 0x7fffffffull)
    return fail(LMP_ERR_UNSUPPORTED, "reduce: too many rows");
  const uint64_t most = uint64_t(1) << (len >= kLongRow ? 23 : 25);
  if (rows > most) {
    const uint64_t launches = (rows + most - 1) / most, per = (rows + launches - 1) / launches;
    for (uint64_t r = 0; r < rows; r += per) {
      const int rc = reduce_rows<OP, T>(rt, out + r, in + r * len, std::min(per, rows - r), len);
      if (rc != LMP_OK) return rc;
    }
    return LMP_OK;
  }
  // Short float64 rows stay in units of one value, as the fused row kernels
  // take them.
  bool done = false;
  const bool pack = packs<T>(in, len) && !(std::is_same_v<T, double> && len < kLongRow);
  const int rc = pack ? reduce_rows_as<OP, T, kPackOf<T>>(rt, out, in, rows, len, &done)
                      : reduce_rows_as<OP, T, 1>(rt, out, in, rows, len, &done);
  if (done) return rc;
  const uint64_t blocks = (rows + kWaves - 1) / kWaves;
  if constexpr (std::is_same_v<T, float>) {
    if (len % 4 == 0 && aligned16(in) && len / 4 <= kMaxU32Extent) {
      hipLaunchKernelGGL((row_reduce_wave_f32<OP>), dim3(uint32_t(blocks)), dim3(kBlock), 0,
                         rt->stream, out, in, rows, uint32_t(len / 4));
      LMP_LAUNCH_CHECK("row_reduce_wave_f32");
      return LMP_OK;
    }
  }
  hipLaunchKernelGGL((row_reduce_wave<OP, T>), dim3(uint32_t(blocks)),
                     dim3(kBlock), 0, rt->stream, out, in, rows, len);
  LMP_LAUNCH_CHECK("row_reduce_wave");
  return LMP_OK;
}

// One lane per output element, grid-striding, the axis folded in row order.
template <int OP, typename T>
int reduce_cols_flat(Runtime* rt, T* out, const T* in, uint64_t outer, uint64_t len,
                     uint64_t inner) {
  const uint64_t cap = uint64_t(rt->cu_count) * 64;
  const uint64_t blocks = std::min<uint64_t>((outer * inner + kBlock - 1) / kBlock, cap);
  hipLaunchKernelGGL((col_reduce_flat<OP, T>), dim3(uint32_t(blocks)), dim3(kBlock), 0, rt->stream,
                     out, in, outer, len, inner);
  LMP_LAUNCH_CHECK("col_reduce_flat");
  return LMP_OK;
}

template <int OP, typename T, int V>
int reduce_cols_as(Runtime* rt, T* out, const T* in, uint64_t outer, uint64_t len,
                   uint64_t inner, bool second = false) {
  constexpr uint64_t kUnit = sizeof(T) * V;
  const uint64_t units = inner / V, cus = uint64_t(rt->cu_count);
  const uint64_t n = outer * units;
  // A lane per output where a slice is too short to share a workgroup ([30000, 16,
  // 16] fp32 34.6 -> 6.0 us, [5912, 21, 16] float64 8.3 -> 4.2) and there are many
  // ([49, 21, 48] is 588 lanes: 3 us longer so), or where the outputs give every CU
  // two workgroups of lanes, rows are 128 bytes or more and the axis is short: 64
  // values of 4 bytes ([60000, 8, 50] fp32 35.6 us in strips, 18.3 so), but for
  // slices of one strip that give a workgroup over three values a lane ([10000,
  // 20, 250] 29.9 us in strips, 35.8 by lanes, [25600, 16, 62] 17.7 and 18.5, [4096,
  // 64, 33] 6.2 and 7.1; [20000, 24, 34] 14.3 and 12.2), or 16 units of other sizes
  // ([64, 1, 151296] float64 63 us in strips, 25.3 so).
  const bool lanes = (len * units <= (len <= 32 ? 256 : 128) && n >= 8192) ||
                     (n >= cus * 2 * kBlock && units * kUnit >= 128 &&
                      len <= (kUnit == 4 ? 64 : 16) &&
                      (kUnit != 4 || units > kBlock || len * units <= 7 * kBlock / 2));
  if (lanes && n <= kMaxGridThreads - kBlock) {
    hipLaunchKernelGGL((col_reduce_lane<OP, T, V>), dim3(blocks_for(n)), dim3(kBlock), 0,
                       rt->stream, out, in, n, FastDiv(uint32_t(units)), uint32_t(len));
    LMP_LAUNCH_CHECK("col_reduce_lane");
    return LMP_OK;
  }
  // Strips of equal width, 1 KiB and 256 units at most.  Strips of 16-byte units
  // may be narrower for an axis of 128 rows or more until there are four
  // workgroups per CU ([16384,16384]: 176 us at 4/CU, 196 us at 8/CU; [256, 197,
  // 768] at 3/CU 31.7 us, at 4/CU 28.8; but [64, 151296] 7.5 us at 2.3/CU, 8.2 at
  // 4/CU), where rows are a whole number of 256 bytes ([10000, 10000] fp32 68.1 us
  // in strips of 1 KiB, 77.5 narrower ones lying across lines, [20000, 3000] 40.9
  // and 51.7).  512 bytes are the least: [256, 65536] 11.9 us (256 bytes: 15.7),
  // [192, 28928] 6.0 (10.3), [16384, 16384] 158 to 161 us wherever it starts (157
  // to 169; 1 KiB: 161 to 168); 256 bytes below 256 MiB where rows are 8 KiB or
  // less or there are four slices ([16384, 1024] 15.3 us, 17.6 with 512; [28, 145,
  // 1984] 6.0 and 7.1, [8, 252, 2240] 4.3 and 6.5).  Where rows are whole 128-byte
  // lines, strips longer than one start on them ([205, 128, 1152] fp32 19.8 -> 18.5
  // us, [25, 314, 1344] float64 18.1 -> 14.0; else that only leaves lanes idle:
  // [49, 7692, 48] fp32 15.1 us, 17.9 so).  They are a power of two wide where that
  // divides the row, so that the row groups meet in even pairs ([256, 197, 768]
  // 3.95e-8 -> 3.81e-8 from float64).
  // Strips of single values stay 1 KiB: [16, 576, 3135] fp32 27.5 -> 22.8 us, [15,
  // 7424, 67] 12.8 -> 7.6, [14, 1004, 1269] float64 33.4 -> 25.9 against 256 bytes.
  const uint64_t target = cus * 4, bytes = outer * len * inner * sizeof(T);
  const uint64_t widest = std::min<uint64_t>(kBlock, 1024 / kUnit);  // a lane per unit at least
  const uint64_t slim =
      (outer >= 4 || units * kUnit <= (8 << 10)) && bytes < kStreamBytes ? 256 : 512;
  const auto width = [&](uint64_t count) { return (units + count - 1) / count; };
  uint64_t strips = (units + widest - 1) / widest, S = 1;
  if (kUnit == 16 && len >= 128 && units % 16 == 0)
    while (strips * outer < target && width(strips + 1) * kUnit >= slim) ++strips;
  uint64_t cw = width(strips);
  if (kUnit == 16 && cw > 8) {
    const uint64_t lines = std::min(widest, (cw + 7) / 8 * 8), last = units % lines;
    if (units % 8 == 0 && (last == 0 || last >= lines / 2)) cw = lines;  // no nearly empty last strip
    uint64_t p = 16;
    while (p * 2 <= cw) p *= 2;
    if (p <= cw && units % p == 0) cw = p;
  }
  strips = (units + cw - 1) / cw;
  if (strips * outer < target) {
    // One pass for an axis of at most 4096 rows, with strips of 64 bytes or
    // more until there are 128 workgroups, while a workgroup reads at most 128
    // KiB (more than that costs more than a second launch: [4096, 4096] 25 us
    // in one pass, 15 us in two), or 256 KiB where there is one for every CU or
    // the whole is 16 MiB at most ([3000, 256] fp32 7.4 us in two passes, 5.3 in
    // one; [3111, 1024] 7.9 and 5.9), down to a line per row ([896, 8192] 8.2 us
    // in two passes, 5.9 in one) or to two lines' length where rows are no whole
    // lines ([3, 500, 5000] float64 14.2 and 12.3); the partials of a first pass
    // always.
    uint64_t narrow = cw;
    constexpr uint64_t least = 64 / kUnit, line = 128 / kUnit;
    const auto groups = [&] { return (units + narrow - 1) / narrow * outer; };
    const bool lined = units % 8 == 0;
    const auto fits = [&] {
      const bool more = groups() >= cus || bytes <= (16 << 20);
      return groups() >= target || len * narrow * kUnit <= (more ? 256u << 10 : 128u << 10);
    };
    while (narrow > least && groups() < 128) narrow = std::max(least, (narrow + 1) / 2);
    while (kUnit == 16 && narrow >= (lined ? 2 : 4) * line && !fits())
      narrow = lined ? (narrow / 2 + line - 1) / line * line : (narrow + 1) / 2;
    if (second || (len <= kStripMaxLen && fits())) {
      cw = narrow;
      strips = (units + cw - 1) / cw;
    } else {
      // Chunks of at least 64 rows and 16 KiB.
      const uint64_t base = strips * outer;
      S = std::min({(target + base - 1) / base, std::max<uint64_t>(1, len / 64),
                    std::max<uint64_t>(1, len * cw * kUnit / (16 << 10))});
    }
  }
  const uint64_t chunk = (len + S - 1) / S;
  S = (len + chunk - 1) / chunk;
  const uint64_t blocks = strips * outer * S;
  if (blocks > kMaxGridThreads / kBlock)
    return reduce_cols_flat<OP, T>(rt, out, in, outer, len, inner);
  T* dst = out;
  T* tmp = nullptr;
  if (S > 1) {
    tmp = static_cast<T*>(scratch_alloc(outer * S * inner * sizeof(T)));
    if (!tmp) return LMP_ERR_OOM;
    dst = tmp;
  }
  const FastDiv dcw{uint32_t(cw)}, dst_strips{uint32_t(strips)}, dS{uint32_t(S)};
  bool nt = false;
  if constexpr (kUnit == 16) {
    nt = bytes >= kStreamBytes;
    if (nt)
      hipLaunchKernelGGL((col_reduce_tile<OP, T, V, true>), dim3(uint32_t(blocks)), dim3(kBlock),
                         0, rt->stream, dst, in, uint32_t(units), uint32_t(len), uint32_t(chunk),
                         dcw, dst_strips, dS);
  }
  if (!nt)
    hipLaunchKernelGGL((col_reduce_tile<OP, T, V, false>), dim3(uint32_t(blocks)), dim3(kBlock), 0,
                       rt->stream, dst, in, uint32_t(units), uint32_t(len), uint32_t(chunk), dcw,
                       dst_strips, dS);
  LMP_LAUNCH_CHECK("col_reduce_tile");
  if (S > 1) {
    const int rc = reduce_cols_as<OP, T, V>(rt, out, tmp, outer, S, inner, true);
    scratch_free(tmp);  // stream-ordered: the second pass reads it first
    return rc;
  }
  return LMP_OK;
}

template <int OP, typename T>
int reduce_cols(Runtime* rt, T* out, const T* in, uint64_t outer, uint64_t len,
                uint64_t inner) {
  // A short axis whose outputs give every CU two to eight workgroups of lanes:
  // a lane per 4-byte value ([64, 151296] int32 7.1 us, 7.6 in strips of 16-byte
  // units).
  const uint64_t per_cu = outer * inner / kBlock / uint64_t(rt->cu_count);
  const bool lanes = sizeof(T) == 4 && len <= 64 && inner >= 32 && per_cu >= 2 && per_cu < 8;
  const bool pack = !lanes && packs<T>(in, inner) && aligned16(out);
  const uint64_t units = pack ? inner / kPackOf<T> : inner;
  // Extents past the tile kernel's 32-bit counters; more than 65535 outer slices
  // (in row order, which callers can hold against the sequential fold).
  if (units > kMaxU32Extent || len > kMaxU32Extent || outer > 65535)
    return reduce_cols_flat<OP, T>(rt, out, in, outer, len, inner);
  return pack ? reduce_cols_as<OP, T, kPackOf<T>>(rt, out, in, outer, len, inner)
              : reduce_cols_as<OP, T, 1>(rt, out, in, outer, len, inner);
}

// An empty reduced axis leaves every output at the functor's identity
// (cpu/reduct.cpp:15-19 folds nothing into it).
template <int OP, typename T>
__global__ __launch_bounds__(kBlock) void fill_identity(T* __restrict__ out, uint64_t n) {
  const uint64_t stride = uint64_t(gridDim.x) * kBlock;
  for (uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride)
    out[i] = Reducer<OP, T>::identity();
}

template <int OP, typename T>
int reduce_any(Runtime* rt, T* out, const T* in, uint64_t outer, uint64_t len,
               uint64_t inner) {
  if (len == 0) {
    const uint64_t n = outer * inner;
    hipLaunchKernelGGL((fill_identity<OP, T>),
                       dim3(uint32_t(std::min<uint64_t>((n + kBlock - 1) / kBlock, 65536))),
                       dim3(kBlock), 0, rt->stream, out, n);
    LMP_LAUNCH_CHECK("fill_identity");
    return LMP_OK;
  }
  return inner == 1 ? reduce_rows<OP, T>(rt, out, in, outer, len)
                    : reduce_cols<OP, T>(rt, out, in, outer, len, inner);
}

template <typename T>
int dispatch_reduce(int op, Runtime* rt, T* out, const T* in, uint64_t outer,
                    uint64_t len, uint64_t inner) {
  switch (op) {
#define LMP_CASE(OPV) \
  case OPV:           \
    return reduce_any<OPV, T>(rt, out, in, outer, len, inner);
    LMP_CASE(LMP_RED_SUM)
    LMP_CASE(LMP_RED_MAX)
    LMP_CASE(LMP_RED_MIN)
    LMP_CASE(LMP_RED_PROD)
#undef LMP_CASE
    default:
      return fail(LMP_ERR_INVALID, "lmp_k_reduce: unknown op " + std::to_string(op));
  }
}

}  // namespace
}  // namespace lmp_hip

using namespace lmp_hip;

extern "C" int lmp_k_reduce(int op, int dtype, void* out, const void* in,
                            size_t outer, size_t len, size_t inner) {
  if (outer == 0 || inner == 0) return LMP_OK;
  if (!out || (!in && len)) return fail(LMP_ERR_INVALID, "lmp_k_reduce: null buffer");
  LMP_RUNTIME_OR_FAIL(rt);
  switch (dtype) {
    case LMP_FLOAT32:
      return dispatch_reduce<float>(op, rt, static_cast<float*>(out),
                                    static_cast<const float*>(in), outer, len, inner);
    case LMP_FLOAT64:
      return dispatch_reduce<double>(op, rt, static_cast<double*>(out),
                                     static_cast<const double*>(in), outer, len, inner);
    case LMP_INT32:
      return dispatch_reduce<int32_t>(op, rt, static_cast<int32_t*>(out),
                                      static_cast<const int32_t*>(in), outer, len, inner);
    case LMP_INT64:
      return dispatch_reduce<int64_t>(op, rt, static_cast<int64_t*>(out),
                                      static_cast<const int64_t*>(in), outer, len, inner);
    case LMP_INT16:
      return dispatch_reduce<int16_t>(op, rt, static_cast<int16_t*>(out),
                                      static_cast<const int16_t*>(in), outer, len, inner);
    case LMP_BOOL:
      return dispatch_reduce<bool>(op, rt, static_cast<bool*>(out),
                                   static_cast<const bool*>(in), outer, len, inner);
    default:
      return fail(LMP_ERR_UNSUPPORTED,
                  std::string("lmp_k_reduce: dtype ") + dtype_name(dtype));
  }
}
