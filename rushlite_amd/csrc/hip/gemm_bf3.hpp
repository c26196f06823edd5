// fp32 GEMM on the bf16 matrix cores, each operand split into three bf16 parts.
//
// Why.  v_mfma_f32_32x32x2_f32 does 64 flop per cycle and SIMD (157 TFLOP/s on
// the chip); v_mfma_f32_32x32x16_bf16 does 1024.  An fp32 value x scaled by
// 2^24 is h + m + l exactly (h = bf16(x), m = bf16(x - h), l = x - h - m: 8
// bits each, round to nearest), so
//   a*b = ah*bh + ah*bm + am*bh + am*bm + ah*bl + al*bh + (am*bl + al*bm + al*bl)
// takes six bf16 MFMAs with fp32 accumulation: 2.5 PFLOP/s / 6 = 419 TFLOP/s.
//
// Error.  The terms left out are 2^-24 of a product at most (a = b = 1 + 2^-8 -
// 2^-17 leaves out 2^-24.01, with one sign), 2^-26.5 rms.  The leading products
// ah*bh accumulate apart from the five small ones, whose roundings are 2^-8 of
// theirs, and the two sums meet at the end: one rounding of the sum per 16
// values of k where an fp32 MFMA rounds once per value or two.  A single
// product (a diagonal operand) is one rounding and the terms left out: rms
// 2.6e-8, at most 2^-23, where an fp32 product has 2.5e-8 and 2^-24.  The
// 256 x 256 tile has no registers for a second sum and adds all six to one, the
// leading product last (first, a single product was 5.3e-8 rms off, at most
// 2.8e-7; last 3.3e-8 and 1.6e-7).  Relative 2-norm of the error against
// float64, fp32 MFMAs / this, K unsplit unless marked (splits fp32 / this):
//                              normal           positive         one term 2^12
//   512 x 512 x 33             1.0e-7  3.9e-8   8.7e-8  4.2e-8   1.0e-7  7.0e-8
//   512 x 512 x 128            2.0e-7  6.5e-8   1.6e-7  6.2e-8   2.1e-7  9.1e-8
//   1000 x 2047 x 1531 (1/2)   7.0e-7  1.6e-7   5.9e-7  1.1e-7   7.0e-7  1.8e-7
//   512 x 4096 x 4096 (4/2)    5.7e-7  2.7e-7   2.2e-7  1.6e-7   5.8e-7  3.0e-7
//   4096^3 (one sum)           1.2e-6  1.0e-6
//
// Range.  The scaling makes the split exact for every finite fp32 value,
// subnormals included (the last bit of one, 2^-149, becomes 2^-125, a normal
// bf16), up to 2^103 for operands and 2^80 for results.  Whatever exceeds
// that, and every infinity and NaN of the operands, leaves a non-finite value
// in the accumulator (an infinite h has m = NaN), so a workgroup that finds
// one after its K loop computes its tile again with fp32 MFMAs on the
// unscaled operands, staged through the same LDS (fallback below): infinities,
// NaN and overflow come out as fp32 products give them, and no other value takes
// that path unnoticed.  A tile that takes it costs both products: with every
// operand NaN 4096^3 takes 1440-1530 us and 512 x 4096 x 4096 227 (fp32 MFMAs
// alone 950 and 139; 2120-3140 and 740 with the second product's operands read
// straight from memory).  Looking for non-finite operands in the first step
// instead (1070 and 158) cost finite ones 1-5%.
//
// What bounds it: power.  4096^3 takes 555-640 us on normal operands (215-248
// TFLOP/s = 1.29-1.49 PFLOP/s of bf16, where a bf16 product of 8192^3 through
// the vendor library reached 1.26) and 395-470 us on zeros: the clock falls
// under the MFMAs of random operands.  The fp32 MFMA kernel it replaced took
// 965 us (143 TFLOP/s); a Linear's backward of 1000 x 2047 x 1531 (odd rows,
// register-staged fp32 tiles and a separate column reduction) 211 -> 84 us;
// the two backward products of 512 x 4096 x 4096 268 -> 182 us.
//
// Structure.  A workgroup owns a BM x BN tile of C, its waves TM x TN blocks
// of 32 x 32 each; K advances 16 at a time through two LDS stages with one
// barrier per step.  Loads go through registers (any alignment, any
// orientation, one step ahead), are split there and stored to LDS as three
// planes of 16-byte octets, [plane][k / 8][row], in which a fragment of one
// MFMA is one conflict-free 128-bit read per lane; 64 bytes between the two
// octets keep the stores of k-contiguous operands off each other's banks.
// Each operand value is converted once per workgroup (13 VALU operations per
// pair, spread over the MFMAs by hand: a pair, then MPC MFMAs), and a fragment
// feeds TN (or TM) x 2 MFMAs per plane, so neither the VALU nor the LDS is
// near its limit.  The leading product is held past the barrier: it reads
// registers only and covers the first fragment reads of the next step.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

namespace lmp_hip {
namespace {

typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr float kBf3Scale = 16777216.0f;                // 2^24, on each operand
constexpr float kBf3Unscale = 3.552713678800501e-15f;   // 2^-48, on the result

// Kept out of the templates, as lds_dma16 is: a target builtin inside a kernel
// template keeps the host pass from emitting the kernel's launch stub.
__device__ __forceinline__ v16f mfma_bf16(bf8 a, bf8 b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v16f mfma_f32(float a, float b, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{x, y}, bf2));
}
__device__ __forceinline__ float bf16_low(uint32_t u) {
  return __builtin_bit_cast(float, u << 16);
}
__device__ __forceinline__ float bf16_high(uint32_t u) {
  return __builtin_bit_cast(float, u & 0xffff0000u);
}
// Two values into the three parts, packed.
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& h, uint32_t& m,
                                           uint32_t& l) {
  const float xs = x * kBf3Scale, ys = y * kBf3Scale;
  h = pack_bf16(xs, ys);
  const float xr = xs - bf16_low(h), yr = ys - bf16_high(h);
  m = pack_bf16(xr, yr);
  l = pack_bf16(xr - bf16_low(m), yr - bf16_high(m));
}

// A sum and the rounding errors of its additions (Knuth's TwoSum; The Art of
// Computer Programming, vol. 2, 4.2.2).
template <typename T>
struct TwoSum {
  T s, err;
  __device__ __forceinline__ void add(T x) {
    const T t = s + x, of_x = t - s;
    err = err + ((s - (t - of_x)) + (x - of_x));
    s = t;
  }
};
// Their total; an infinite or NaN sum as it is (its errors are NaN).
__device__ __forceinline__ float sum_of(const TwoSum<float>& a) {
  const bool finite = (__builtin_bit_cast(uint32_t, a.s) & 0x7fffffffu) < 0x7f800000u;
  return finite ? a.s + a.err : a.s;
}

// DEPTH: steps of loads in flight ahead of the one being split.  APART: the five
// small products of a step accumulate apart from the leading one.
template <int WM_, int WN_, int TM_, int TN_, int DEPTH_, int MINB_, bool APART_>
struct Bf3Cfg {
  static constexpr int WM = WM_, WN = WN_, TM = TM_, TN = TN_, DEPTH = DEPTH_, MINB = MINB_;
  static constexpr bool APART = APART_;
  static constexpr int NW = WM * WN, THREADS = 64 * NW;
  static constexpr int BM = WM * TM * 32, BN = WN * TN * 32;
  static constexpr int A_OCT = BM * 16 + 64, B_OCT = BN * 16 + 64;  // bytes
  static constexpr int A_PLANE = 2 * A_OCT, B_PLANE = 2 * B_OCT;
  static constexpr int STAGE = 3 * (A_PLANE + B_PLANE);
  static constexpr int SMEM = 2 * STAGE + 16;  // the stages and the fallback's flag
  static_assert(2 * STAGE >= NW * 32 * 36 * 4, "the epilogue's wave tiles fit");
};

// One operand's panel of R rows (of m or n) x 16 k on its way from memory to
// LDS.  A thread holds ITEMS items of W consecutive k values of one row, in
// SETS register sets (steps in flight).  KMAJOR: k is contiguous in memory.
// Rows past the matrix read its last row (their results are never stored).
template <int R, int THREADS, bool KMAJOR, int SETS>
struct Bf3Panel {
  static constexpr int W = R * 2 >= THREADS ? 8 : 4;
  static constexpr int PER_ROW = kBf3K / W;
  static constexpr int ITEMS = R * PER_ROW / THREADS;
  static constexpr int PAIRS = ITEMS * (W / 2);  // of this thread, per step
  static_assert(ITEMS * THREADS == R * PER_ROW, "items split evenly over the threads");
  const float* p[ITEMS];
  int ld, k[ITEMS], off[ITEMS];
  float v[SETS][ITEMS][W];
  TwoSum<float> cs[ITEMS];  // column sums (bias gradient), where they are asked for

  // `k0`: the first k that load() reads.
  __device__ __forceinline__ void init(const float* base, int ld_, int r0, int rows, int k0,
                                       int oct_bytes) {
    ld = ld_;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int q = int(threadIdx.x) + i * THREADS;
      const int row = KMAJOR ? q / PER_ROW : q % R;
      k[i] = W * (KMAJOR ? q % PER_ROW : q / R);
      const int64_t r = min(r0 + row, rows - 1);
      p[i] = base + (KMAJOR ? r * ld + (k0 + k[i]) : int64_t(k0 + k[i]) * ld + r);
      off[i] = (k[i] / 8) * oct_bytes + row * 16 + (k[i] % 8) * 2;
      cs[i] = TwoSum<float>{0.0f, 0.0f};
    }
  }
  // The item's values of a whole step; the next load reads `advance` k on.
  __device__ __forceinline__ void load(int set, int i, int advance) {
    if constexpr (KMAJOR) {
#pragma unroll
      for (int j = 0; j < W; j += 4) {
        const v4f_any x = *reinterpret_cast<const v4f_any*>(p[i] + j);
        v[set][i][j] = x.x; v[set][i][j + 1] = x.y; v[set][i][j + 2] = x.z; v[set][i][j + 3] = x.w;
      }
      p[i] += advance;
    } else {
#pragma unroll
      for (int j = 0; j < W; ++j) v[set][i][j] = p[i][int64_t(j) * ld];
      p[i] += int64_t(advance) * ld;
    }
  }
  __device__ __forceinline__ void load_all(int set, int advance) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) load(set, i, advance);
  }
  // A step of `left` values of k that starts `at` k past the pointers, zeros
  // after them.
  __device__ __forceinline__ void load_tail(int set, int at, int left) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j) {
        v[set][i][j] = 0.0f;
        if (k[i] + j < left)
          v[set][i][j] = KMAJOR ? p[i][at + j] : p[i][int64_t(at + j) * ld];
      }
  }
  // A step's values add in pairs and the running sum keeps its rounding errors:
  // a plain sum of every value of K was 4.0e-7 from float64 over 2048 normal rows
  // and 3.1e-7 over 4096 (in two splits), this is 6.1e-8 and 6.6e-8, the dim-0
  // reduction 9.6e-8 and 1.1e-7; no difference in time.
  __device__ __forceinline__ void add_cs(int set) {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      float x[W];
#pragma unroll
      for (int j = 0; j < W; ++j) x[j] = v[set][i][j];
#pragma unroll
      for (int w = 1; w < W; w *= 2)
#pragma unroll
        for (int j = 0; j < W; j += 2 * w) x[j] = x[j] + x[j + w];
      cs[i].add(x[0]);
    }
  }
  // Stores an item's parts (h, m, l: W / 2 packed pairs) into the three planes.
  __device__ __forceinline__ void put(int i, char* lds, int plane, const uint32_t (&h)[4],
                                      const uint32_t (&m)[4], const uint32_t (&l)[4]) const {
    char* q = lds + off[i];
    if constexpr (W == 8) {
      *reinterpret_cast<u4*>(q) = u4{h[0], h[1], h[2], h[3]};
      *reinterpret_cast<u4*>(q + plane) = u4{m[0], m[1], m[2], m[3]};
      *reinterpret_cast<u4*>(q + 2 * plane) = u4{l[0], l[1], l[2], l[3]};
    } else {
      *reinterpret_cast<u2*>(q) = u2{h[0], h[1]};
      *reinterpret_cast<u2*>(q + plane) = u2{m[0], m[1]};
      *reinterpret_cast<u2*>(q + 2 * plane) = u2{l[0], l[1]};
    }
  }
  // Stores the values themselves, [k][row] with R + 4 values per k.
  __device__ __forceinline__ void store_values(float* lds) const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const int q = int(threadIdx.x) + i * THREADS, row = KMAJOR ? q / PER_ROW : q % R;
#pragma unroll
      for (int j = 0; j < W; ++j) lds[(k[i] + j) * (R + 4) + row] = v[0][i][j];
    }
  }
  __device__ __forceinline__ void store_all(int set, char* lds, int plane) const {
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      uint32_t h[4], m[4], l[4];
#pragma unroll
      for (int j = 0; j < W / 2; ++j)
        split_pair(v[set][i][2 * j], v[set][i][2 * j + 1], h[j], m[j], l[j]);
      put(i, lds, plane, h, m, l);
    }
  }
};

struct Bf3Args {
  GemmArgs g;
  int splits, steps_per_split;  // K splits, and 16-wide k steps in each
  // Partials of split s (splits > 1): C's m * n values at part + s *
  // part_stride and, with column sums, their n values cs_at after it; both
  // start on 16 bytes.
  float* part;
  int64_t part_stride, cs_at;
};

// Work item `id` of the product (in [0, tiles * splits)) for this workgroup.
template <class C, bool TA, bool TB>
__device__ __forceinline__ void gemm_bf3_tile(const Bf3Args& args, int id, char* smem) {
  const GemmArgs& g = args.g;
  constexpr int TM = C::TM, TN = C::TN, MM = TM * TN;
  // Consecutive ids go round the eight XCDs: give each XCD a contiguous run of
  // (split, tile), so its L2 sees one range of k and neighbouring tiles.
  const int ntiles = g.tiles_m * g.tiles_n, total = ntiles * args.splits;
  {
    const int q = total / 8, r = total % 8, x = id % 8;
    id = x * q + min(x, r) + id / 8;
  }
  const int split = id / ntiles, tile = id - split * ntiles;
  constexpr int kGroup = 8;  // tile rows walked together
  const int per_group = kGroup * g.tiles_n, group = tile / per_group;
  const int gsize = min(g.tiles_m - group * kGroup, kGroup);
  const int in_group = tile - group * per_group;
  const int tile_m = group * kGroup + in_group % gsize;
  const int m0 = tile_m * C::BM, n0 = (in_group / gsize) * C::BN;

  const int k_begin = split * args.steps_per_split * kBf3K;
  const int k_len = min(g.k - k_begin, args.steps_per_split * kBf3K);
  const int full = k_len / kBf3K, left = k_len % kBf3K, steps = full + (left ? 1 : 0);
  const bool partial = args.splits > 1;
  int* flag = reinterpret_cast<int*>(smem + 2 * C::STAGE);
  if (threadIdx.x == 0) *flag = 0;  // set after the K loop's barriers
  const bool do_cs = !TB && g.colsum != nullptr && tile_m == 0;  // uniform

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int li = lane & 31, lh = lane >> 5;

  using PA = Bf3Panel<C::BM, C::THREADS, !TA, C::DEPTH>;
  using PB = Bf3Panel<C::BN, C::THREADS, TB, C::DEPTH>;
  PA pa;
  PB pb;
  // Loads past the last whole step repeat it (and are not used); a split
  // without a whole step reads the 16 k before the end of K for them (K > 32).
  const int k_load = min(k_begin, g.k - kBf3K);
  pa.init(g.a, g.lda, m0, g.m, k_load, C::A_OCT);
  pb.init(g.b, g.ldb, n0, g.n, k_load, C::B_OCT);

  // The leading products, and (APART) the small ones.
  v16f acc[TM][TN], low[C::APART ? TM : 1][C::APART ? TN : 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = v16f(0.0f);
      if constexpr (C::APART) low[i][j] = v16f(0.0f);
    }

  const int a_at = lh * C::A_OCT + (wm * TM * 32 + li) * 16;
  const int b_at = 3 * C::A_PLANE + lh * C::B_OCT + (wn * TN * 32 + li) * 16;
  bf8 fa[3][TM], fb[3][TN];
  auto read_a = [&](const char* s, int p) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      fa[p][i] = *reinterpret_cast<const bf8*>(s + p * C::A_PLANE + a_at + i * 512);
  };
  auto read_b = [&](const char* s, int p) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
      fb[p][j] = *reinterpret_cast<const bf8*>(s + p * C::B_PLANE + b_at + j * 512);
  };
  auto mma_leading = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma_bf16(fa[0][i], fb[0][j], acc[i][j]);
  };

  // The step with the end of K first (when 16 does not divide it), then the
  // whole ones.  Stage t % 2 holds step t, the register sets the DEPTH steps
  // after it: step u in set u % DEPTH.
  int ahead = full;  // whole steps not loaded yet
  auto advance = [&]() { return ahead > 1 ? kBf3K : 0; };
  if (left) {
    pa.load_tail(0, k_begin - k_load + full * kBf3K, left);
    pb.load_tail(0, k_begin - k_load + full * kBf3K, left);
  } else {
    pa.load_all(0, advance());
    pb.load_all(0, advance());
    --ahead;
  }
  // A tile that meets an infinity or a NaN in its first step goes to the fallback
  // at once (a diverged run's operands are NaN throughout).
  if constexpr (!TB)
    if (do_cs) pb.add_cs(0);
  pa.store_all(0, smem, C::A_PLANE);
  pb.store_all(0, smem + 3 * C::A_PLANE, C::B_PLANE);
#pragma unroll
  for (int d = 1; d <= C::DEPTH; ++d) {
    const int adv = advance();
    pa.load_all(d % C::DEPTH, adv);
    pb.load_all(d % C::DEPTH, adv);
    --ahead;
  }
  // The leading product of the step before is held past the barrier; zeros at
  // first.
#pragma unroll
  for (int i = 0; i < TM; ++i) fa[0][i] = bf8(0);
#pragma unroll
  for (int j = 0; j < TN; ++j) fb[0][j] = bf8(0);
  constexpr int PA_OF[5] = {1, 1, 0, 0, 2}, PB_OF[5] = {1, 0, 1, 2, 0};
  constexpr int PAIRS = PA::PAIRS + PB::PAIRS;
  constexpr int MPC = (5 * MM - MM / 2) / PAIRS > 0 ? (5 * MM - MM / 2) / PAIRS : 1;
  // One step: STAGE holds it, SET the next one.
  auto step = [&](auto stage_c, auto set_c, int t) {
    constexpr int stage = decltype(stage_c)::value, set = decltype(set_c)::value;
    const char* s = smem + stage * C::STAGE;
    char* d = smem + (stage ^ 1) * C::STAGE;
    __syncthreads();
    if constexpr (!TB)
      if (do_cs && t + 1 < steps) pb.add_cs(set);
    const int adv = advance();
    --ahead;
    read_a(s, 1);
    read_b(s, 1);
    __builtin_amdgcn_sched_barrier(0);
    mma_leading();
    __builtin_amdgcn_sched_barrier(0);
    read_b(s, 0);
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int c = 0; c < PAIRS; ++c) {
      // The next product's fragments, half a product or more ahead of it.
      const int q0 = c * MPC, q1 = c == PAIRS - 1 ? 5 * MM : q0 + MPC;
      auto covers = [&](int q) { return q0 <= q && q < q1; };
      if (covers(MM / 2)) read_a(s, 0);
      if (covers(MM + MM / 2)) read_b(s, 2);
      if (covers(3 * MM - 1)) read_a(s, 2);
      const bool of_a = c < PA::PAIRS;
      const int ca = of_a ? c : c - PA::PAIRS;
      const int it = of_a ? ca / (PA::W / 2) : ca / (PB::W / 2);
      const int pr = of_a ? ca % (PA::W / 2) : ca % (PB::W / 2);
      if (of_a)
        split_pair(pa.v[set][it][2 * pr], pa.v[set][it][2 * pr + 1], h[pr], m[pr], l[pr]);
      else
        split_pair(pb.v[set][it][2 * pr], pb.v[set][it][2 * pr + 1], h[pr], m[pr], l[pr]);
#pragma unroll
      for (int q = q0; q < q1; ++q)
        if (q < 5 * MM) {
          const int pp = q / MM, i = (q % MM) / TN, j = q % TN;
          v16f& sum = [&]() -> v16f& {
            if constexpr (C::APART) return low[i][j];
            else return acc[i][j];
          }();
          sum = mfma_bf16(fa[PA_OF[pp]][i], fb[PB_OF[pp]][j], sum);
        }
      if (of_a && pr == PA::W / 2 - 1) {
        pa.put(it, d, C::A_PLANE, h, m, l);
        pa.load(set, it, adv);
      }
      if (!of_a && pr == PB::W / 2 - 1) {
        pb.put(it, d + 3 * C::A_PLANE, C::B_PLANE, h, m, l);
        pb.load(set, it, adv);
      }
      // Masks: 0x8 MFMA, 0x100 LDS read, 0x2 VALU.
#pragma unroll
      for (int q = 0; q < MPC; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (13 + MPC - 1) / MPC, 0);
      }
      if (c < PAIRS - 1) __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr int D = C::DEPTH;
  static_assert(D == 1 || D == 2, "steps are unrolled by two");
#define LMP_BF3_STEP(U) \
  step(std::integral_constant<int, (U) % 2>{}, std::integral_constant<int, ((U) + 1) % D>{}, t)
  // (One way out of the loop: with two the compiler holds both accumulators
  // twice.)
  int t = 0;
  while (t + 1 < steps) {
    LMP_BF3_STEP(0);
    ++t;
    LMP_BF3_STEP(1);
    ++t;
  }
  if (t < steps) LMP_BF3_STEP(0);
#undef LMP_BF3_STEP
  mma_leading();
  __syncthreads();

  // Column sums: the parts of a column (its items' k ranges) in k order.
  if constexpr (!TB) {
    if (do_cs) {
      float* sums = reinterpret_cast<float*>(smem);
#pragma unroll
      for (int i = 0; i < PB::ITEMS; ++i) sums[int(threadIdx.x) + i * C::THREADS] = sum_of(pb.cs[i]);
      __syncthreads();
      for (int c = threadIdx.x; c < C::BN; c += C::THREADS) {
        float v = sums[c];
#pragma unroll
        for (int q = 1; q < PB::PER_ROW; ++q) v += sums[q * C::BN + c];
        const int col = n0 + c;
        if (col < g.n) {
          if (partial)
            args.part[split * args.part_stride + args.cs_at + col] = v;
          else
            g.colsum[col] = g.colsum_acc ? g.colsum[col] + v : v;
        }
      }
      __syncthreads();
    }
  }

  // A sum that is not finite sends the workgroup to the fallback.
  if constexpr (C::APART) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = acc[i][j] + low[i][j];
  }
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        top = max(top, __builtin_bit_cast(uint32_t, float(acc[i][j][r])) & 0x7fffffffu);
  if (top >= 0x7f800000u) *flag = 1;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = acc[i][j] * kBf3Unscale;
  __syncthreads();
  if (*flag) {
    // fp32 MFMAs on the unscaled values, staged through the same LDS.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = v16f(0.0f);
    Bf3Panel<C::BM, C::THREADS, !TA, 1> qa;
    Bf3Panel<C::BN, C::THREADS, TB, 1> qb;
    qa.init(g.a, g.lda, m0, g.m, k_load, C::A_OCT);
    qb.init(g.b, g.ldb, n0, g.n, k_load, C::B_OCT);
    int whole = full;  // whole steps not loaded yet
    if (left) {
      qa.load_tail(0, k_begin - k_load + full * kBf3K, left);
      qb.load_tail(0, k_begin - k_load + full * kBf3K, left);
    } else {
      --whole;
      qa.load_all(0, whole > 0 ? kBf3K : 0);
      qb.load_all(0, whole > 0 ? kBf3K : 0);
    }
    constexpr int PITCH_A = C::BM + 4, PITCH_B = C::BN + 4;
    static_assert(kBf3K * (PITCH_A + PITCH_B) * 4 <= C::STAGE, "a stage holds a step's values");
#pragma unroll 1
    for (int t = 0; t < steps; ++t) {
      float* sa = reinterpret_cast<float*>(smem + (t & 1) * C::STAGE);
      float* sb = sa + kBf3K * PITCH_A;
      qa.store_values(sa);
      qb.store_values(sb);
      __syncthreads();
      if (whole > 0) {
        --whole;
        qa.load_all(0, whole > 0 ? kBf3K : 0);
        qb.load_all(0, whole > 0 ? kBf3K : 0);
      }
#pragma unroll
      for (int k = 0; k < kBf3K; k += 2) {
        float xa[TM], xb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) xa[i] = sa[(k + lh) * PITCH_A + (wm * TM + i) * 32 + li];
#pragma unroll
        for (int j = 0; j < TN; ++j) xb[j] = sb[(k + lh) * PITCH_B + (wn * TN + j) * 32 + li];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = mfma_f32(xa[i], xb[j], acc[i][j]);
      }
    }
    __syncthreads();  // the epilogue writes over the stages
  }

  float* out = partial ? args.part + split * args.part_stride : g.c;
  const int64_t ld = partial ? g.n : g.ldc;
  const float* bias = partial ? nullptr : g.bias;
  const bool acc_out = !partial && g.accumulate;
  if (g.vec_out) {
    // Whole float4s of C's rows through a wave-private 32 x 36 LDS tile (LDS
    // requests of one wave complete in order).  Every wave is past its reads of
    // the stages (the flag's barrier).
    float* w = reinterpret_cast<float*>(smem) + wave * (32 * 36);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          w[((r / 4) * 8 + lh * 4 + (r % 4)) * 36 + li] = acc[i][j][r];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        const int row0 = m0 + (wm * TM + i) * 32, col0 = n0 + (wn * TN + j) * 32;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int at = lane + 64 * q, rr = at >> 3, cc = (at & 7) * 4;
          const v4f v = *reinterpret_cast<const v4f*>(w + rr * 36 + cc);
          const int row = row0 + rr, col = col0 + cc;
          if (row < g.m && col < g.n) {
            v4f* p = reinterpret_cast<v4f*>(out + row * ld + col);
            if (acc_out) *p = *p + v;
            else if (bias) *p = lin_epi4(v, *reinterpret_cast<const v4f*>(bias + col), g.relu);
            else *p = v;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + (wn * TN + j) * 32 + li;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = m0 + (wm * TM + i) * 32 + (r / 4) * 8 + lh * 4 + (r % 4);
        if (row < g.m && col < g.n) {
          float* p = out + row * ld + col;
          const float v = acc[i][j][r];
          if (acc_out) *p = *p + v;
          else if (bias) *p = lin_epi(v, bias[col], g.relu);
          else *p = v;
        }
      }
    }
}

template <int NT, int MINB, class C, bool TA, bool TB>
__global__ __launch_bounds__(NT, MINB) void gemm_bf3(Bf3Args args) {
  static_assert(NT == C::THREADS, "one lane per thread of the configuration");
  __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
  gemm_bf3_tile<C, TA, TB>(args, int(blockIdx.x), smem);
}

// A Linear's weight gradient (`w`: A transposed) and input gradient (`x`: B
// transposed) in one grid, the first product's workgroups first: the CUs it
// frees start the second's first loads while its last stores drain, and the
// bits are those of two launches.
template <int NT, int MINB, class CW, class CX>
__global__ __launch_bounds__(NT, MINB) void gemm_bf3_pair(Bf3Args w, Bf3Args x) {
  static_assert(NT == CW::THREADS && NT == CX::THREADS, "one workgroup size for both");
  __shared__ __attribute__((aligned(1024))) char smem[CW::SMEM > CX::SMEM ? CW::SMEM : CX::SMEM];
  const int of_w = w.g.tiles_m * w.g.tiles_n * w.splits;
  const int id = int(blockIdx.x);
  if (id < of_w) gemm_bf3_tile<CW, true, false>(w, id, smem);
  else gemm_bf3_tile<CX, false, true>(x, id - of_w, smem);
}

// C (and the column sums) from the partials of one product, or of two (`b`,
// from workgroup `blocks_a` on), added in split order, with the epilogue of
// the final output.  Four consecutive values per lane, counted through C as
// one run of m * n: the loads are 128-bit whatever n is, and so are the stores
// when C's rows are contiguous or all 16-byte aligned (g.vec_out).  The last
// workgroups of a product add its column sums.
struct Bf3Fold {
  Bf3Args a;
  int blocks_c, blocks;  // workgroups for C, and with the column sums
};

__device__ __forceinline__ void fold_bf3_block(const Bf3Args& a, int block, int blocks_c) {
  const GemmArgs& g = a.g;
  const bool is_cs = block >= blocks_c;
  const int count = is_cs ? g.n : g.m * g.n;  // below 2^23: the partials are bounded
  const int i = 4 * ((block - (is_cs ? blocks_c : 0)) * 256 + int(threadIdx.x));
  if (i >= count) return;
  const float* src = a.part + (is_cs ? a.cs_at : 0) + i;
  v4f v = *reinterpret_cast<const v4f*>(src);
  if (is_cs) {
    TwoSum<v4f> t{v, v4f(0.0f)};
    for (int s = 1; s < a.splits; ++s)
      t.add(*reinterpret_cast<const v4f*>(src + s * a.part_stride));
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i + e < count) {
        const float x = sum_of(TwoSum<float>{t.s[e], t.err[e]});
        g.colsum[i + e] = g.colsum_acc ? g.colsum[i + e] + x : x;
      }
    return;
  }
  int s = 1;
  for (; s + 4 <= a.splits; s += 4) {
    v4f x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = *reinterpret_cast<const v4f*>(src + (s + u) * a.part_stride);
#pragma unroll
    for (int u = 0; u < 4; ++u) v = v + x[u];
  }
  for (; s < a.splits; ++s) v = v + *reinterpret_cast<const v4f*>(src + s * a.part_stride);
  int row = i / g.n, col = i - row * g.n;
  if (g.vec_out) {
    v4f* p = reinterpret_cast<v4f*>(g.c + int64_t(row) * g.ldc + col);
    if (g.accumulate) *p = *p + v;
    else *p = g.bias ? lin_epi4(v, *reinterpret_cast<const v4f*>(g.bias + col), g.relu) : v;
    return;
  }
  if (g.ldc == g.n && !g.accumulate && i + 4 <= count) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (g.bias) v[e] = lin_epi(v[e], g.bias[col], g.relu);
      if (++col == g.n) col = 0;
    }
    *reinterpret_cast<v4f_any*>(g.c + i) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (i + e < count) {
      float* p = g.c + int64_t(row) * g.ldc + col;
      if (g.accumulate) *p = *p + v[e];
      else *p = g.bias ? lin_epi(v[e], g.bias[col], g.relu) : v[e];
    }
    if (++col == g.n) {
      col = 0;
      ++row;
    }
  }
}

__global__ __launch_bounds__(256) void fold_bf3(Bf3Fold a, Bf3Fold b) {
  const int block = int(blockIdx.x);
  if (block < a.blocks) fold_bf3_block(a.a, block, a.blocks_c);
  else fold_bf3_block(b.a, block - a.blocks, b.blocks_c);
}

// ------------------------------------------------------------------- host

using Bf3Big = Bf3Cfg<2, 4, 4, 2, 1, 1, false>;   // 256 x 256, 8 waves of 128 x 64
using Bf3Wide = Bf3Cfg<4, 2, 2, 2, 1, 1, true>;   // 256 x 128, 8 waves of 64 x 64
using Bf3Mid = Bf3Cfg<4, 2, 1, 2, 2, 4, true>;    // 128 x 128, 8 waves of 32 x 64, two a CU
using Bf3Flat = Bf3Cfg<1, 4, 2, 1, 2, 2, true>;   // 64 x 128, 4 waves of 64 x 32
using Bf3Small = Bf3Cfg<2, 2, 1, 1, 2, 2, true>;  // 64 x 64, 4 waves of 32 x 32

// kBf3Tiles is what these types are.
template <class C>
constexpr bool bf3_is(int cfg) {
  return kBf3Tiles[cfg].bm == C::BM && kBf3Tiles[cfg].bn == C::BN &&
         kBf3Tiles[cfg].threads == C::THREADS && kBf3Tiles[cfg].apart == C::APART;
}
static_assert(bf3_is<Bf3Big>(0) && bf3_is<Bf3Wide>(1) && bf3_is<Bf3Mid>(2) &&
              bf3_is<Bf3Flat>(3) && bf3_is<Bf3Small>(4));

Bf3Plan bf3_plan(Runtime* rt, const GemmArgs& g) {
  return lmp_hip::bf3_plan(rt->cu_count, int64_t(LMP_NOALLOC_SCRATCH_BYTES), g.m, g.n, g.k);
}

// Calls f with the configuration's type.
template <class F>
int with_bf3_cfg(int cfg, F&& f) {
  switch (cfg) {
    case 0: return f(Bf3Big{});
    case 1: return f(Bf3Wide{});
    case 2: return f(Bf3Mid{});
    case 3: return f(Bf3Flat{});
    default: return f(Bf3Small{});
  }
}

// The launch arguments of `g` under `plan`, without the partials' memory.
Bf3Args bf3_args(const GemmArgs& g, const Bf3Plan& plan) {
  Bf3Args a{};
  a.g = g;
  const Bf3Tile& t = kBf3Tiles[plan.cfg];
  a.g.tiles_m = (g.m + t.bm - 1) / t.bm;
  a.g.tiles_n = (g.n + t.bn - 1) / t.bn;
  const int steps = (g.k + kBf3K - 1) / kBf3K;
  a.steps_per_split = (steps + plan.splits - 1) / plan.splits;
  a.splits = (steps + a.steps_per_split - 1) / a.steps_per_split;
  a.cs_at = (int64_t(g.m) * g.n + 3) / 4 * 4;
  a.part_stride = a.cs_at + (g.colsum ? (int64_t(g.n) + 3) / 4 * 4 : 0);
  return a;
}

int bf3_take_partials(Bf3Args& a, const Workspace& ws) {
  if (a.splits == 1) return LMP_OK;
  return ws.take(size_t(a.splits) * size_t(a.part_stride) * sizeof(float), &a.part);
}

uint32_t bf3_workgroups(const Bf3Args& a) {
  return uint32_t(int64_t(a.g.tiles_m) * a.g.tiles_n * a.splits);
}

// The fold of one or two products; those without a split take no workgroup.
int launch_fold_bf3(Runtime* rt, const Bf3Args& a, const Bf3Args* b = nullptr) {
  auto fold = [](const Bf3Args& x) {
    Bf3Fold f{x, 0, 0};
    if (x.splits > 1) {
      f.blocks_c = int((int64_t(x.g.m) * x.g.n + 1023) / 1024);
      f.blocks = f.blocks_c + (x.g.colsum ? (x.g.n + 1023) / 1024 : 0);
    }
    return f;
  };
  const Bf3Fold fa = fold(a), fb = b ? fold(*b) : Bf3Fold{};
  if (fa.blocks + fb.blocks == 0) return LMP_OK;
  hipLaunchKernelGGL(fold_bf3, dim3(uint32_t(fa.blocks + fb.blocks)), dim3(256), 0, rt->stream,
                     fa, fb);
  LMP_LAUNCH_CHECK("fold_bf3");
  return LMP_OK;
}

template <bool TA, bool TB>
int launch_bf3_as(Runtime* rt, GemmArgs g, const Bf3Plan& plan, const Workspace& ws) {
  Bf3Args a = bf3_args(g, plan);
  if (const int rc = bf3_take_partials(a, ws); rc != LMP_OK) return rc;
  const int rc = with_bf3_cfg(plan.cfg, [&](auto cfg) {
    using C = decltype(cfg);
    hipLaunchKernelGGL((gemm_bf3<C::THREADS, C::MINB, C, TA, TB>), dim3(bf3_workgroups(a)),
                       dim3(C::THREADS), 0, rt->stream, a);
    LMP_LAUNCH_CHECK("gemm_bf3");
    return launch_fold_bf3(rt, a);
  });
  if (a.part) ws.give(a.part);  // stream-ordered: the fold reads it first
  return rc;
}

template <bool TA, bool TB>
int launch_bf3_planned(Runtime* rt, GemmArgs g, const Workspace& ws, bool* colsum_done) {
  if (TB) g.colsum = nullptr;  // the sums ride where B's rows run along n
  const Bf3Plan plan = bf3_plan(rt, g);
  if (plan.cfg < 0) return fail(LMP_ERR_UNSUPPORTED, "gemm: more tiles than a grid holds");
  if (g.colsum && colsum_done) *colsum_done = true;
  return launch_bf3_as<TA, TB>(rt, g, plan, ws);
}

// A weight gradient (A transposed, with its column sums) and an input gradient
// (B transposed) as one launch and, where either is split, one fold; false,
// with nothing launched, if their workgroups differ in size or are more than a
// grid holds.
bool launch_bf3_pair_planned(Runtime* rt, const GemmArgs& gw, const GemmArgs& gx, int* rc) {
  const Bf3Plan pw = bf3_plan(rt, gw), px = bf3_plan(rt, gx);
  if (pw.cfg < 0 || px.cfg < 0) return false;
  const int threads = kBf3Tiles[pw.cfg].threads;
  if (kBf3Tiles[px.cfg].threads != threads) return false;
  Bf3Args w = bf3_args(gw, pw), x = bf3_args(gx, px);
  if (!bf3_pair_fits(bf3_workgroups(w), bf3_workgroups(x), threads)) return false;
  const Workspace ws{};
  if ((*rc = bf3_take_partials(w, ws)) != LMP_OK) return true;
  if ((*rc = bf3_take_partials(x, ws)) != LMP_OK) {
    if (w.part) ws.give(w.part);
    return true;
  }
  *rc = with_bf3_cfg(pw.cfg, [&](auto cw) {
    return with_bf3_cfg(px.cfg, [&](auto cx) {
      using CW = decltype(cw);
      using CX = decltype(cx);
      if constexpr (CW::THREADS == CX::THREADS) {
        constexpr int kMinB = CW::MINB < CX::MINB ? CW::MINB : CX::MINB;
        hipLaunchKernelGGL((gemm_bf3_pair<CW::THREADS, kMinB, CW, CX>),
                           dim3(bf3_workgroups(w) + bf3_workgroups(x)), dim3(CW::THREADS), 0,
                           rt->stream, w, x);
        LMP_LAUNCH_CHECK("gemm_bf3_pair");
        return launch_fold_bf3(rt, w, &x);
      } else {
        return fail(LMP_ERR_RUNTIME, "linear_backward: workgroup sizes differ");
      }
    });
  });
  if (w.part) ws.give(w.part);  // stream-ordered: the fold reads them first
  if (x.part) ws.give(x.part);
  return true;
}

}  // namespace
}  // namespace lmp_hip
