// gfx950 kernels that bring a weight into the stored format and into the operand the GEMM kernels consume.
//   prepare_kernel  : reference operands (1-bit values, reordered 2-bit-index metadata) -> prepared operand
//   pack_kernel     : dense fp16, bf16 or fp32 weight -> the reference operands (2:4 magnitude mask, compression, one-bit values)
#include "onebit_device.h"
#include "onebit_launch.h"

namespace onebit {

// Position of a workgroup in a two-dimensional list that is walked in strips: `along` runs over [0, length), `across` over
// the strips' widths. Workgroup b runs on XCD b % 8, so each XCD is given a contiguous range of the list: strip after
// strip, inside a strip `along` slowest, its `width` workgroups side by side. The grid holds whole strips.
struct StripPosition {
  int along, across;
};
__device__ __forceinline__ StripPosition strip_position(int width, int length) {
  const int per = gridDim.x / 8, rem = gridDim.x % 8, xcd = blockIdx.x % 8;
  const int v = xcd * per + (xcd < rem ? xcd : rem) + blockIdx.x / 8;
  const int strip = v / (width * length), w = v % (width * length);
  return StripPosition{w / width, strip * width + w % width};
}

// =====================================================================================================
// 32 x 32 bit transpose across each half of a wavefront: on entry bit b of lane 32 h + r is element (r, b), on return
// element (b, r). Five exchange steps (xor 16, 8, 4, 2, 1), each one lane exchange, one rotate, one bit select; the
// lane-dependent rotate amounts and masks are built once per wavefront.
// =====================================================================================================
struct BitTranspose {
  uint32_t rotate[5], keep[5];
  __device__ __forceinline__ explicit BitTranspose(int lane) {
    constexpr uint32_t kLow[5] = {0x0000FFFFu, 0x00FF00FFu, 0x0F0F0F0Fu, 0x33333333u, 0x55555555u};
#pragma unroll
    for (int step = 0; step < 5; ++step) {
      const int d = 16 >> step;
      const bool upper = (lane & d) != 0;
      rotate[step] = upper ? d : 32 - d;                 // the partner's bits move down into the upper lane, up into the lower
      keep[step] = upper ? ~kLow[step] : kLow[step];     // bits that stay
    }
  }
  __device__ __forceinline__ uint32_t operator()(uint32_t x) const {
    auto exchange = [&](uint32_t y, int step) __attribute__((always_inline)) {
      const uint32_t moved = __builtin_amdgcn_alignbit(y, y, rotate[step]);
      return (x & keep[step]) | (moved & ~keep[step]);
    };
    x = exchange(__builtin_amdgcn_ds_swizzle(x, (16 << 10) | 0x1F), 0);
    x = exchange(__builtin_amdgcn_mov_dpp(x, 0x128, 0xF, 0xF, true), 1);  // rotate by 8 inside 16 lanes = xor 8
    x = exchange(__builtin_amdgcn_ds_swizzle(x, (4 << 10) | 0x1F), 2);
    x = exchange(__builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, true), 3);   // quad order 2 3 0 1 = xor 2
    x = exchange(__builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, true), 4);   // quad order 1 0 3 2 = xor 1
    return x;
  }
};

// =====================================================================================================
// prepare_kernel: one wavefront per 64 rows (two row blocks) and K chunk.
// Reads  a : bit (r, j) of the (m x k/2) column-major one-bit matrix = bit (r + j m) % 8 of byte (r + j m) / 8
//            (csrc/kernel_lib.cu:28,37; produced by onebit_sparse_mul/__init__.py:139-143), 1 = +1, 0 = -1
//        e : int16 metadata (m x k/16) in the reference's reordered layout or the CUTLASS one
//            (_semi_structured_conversions.py:21-48,173-177)
// Writes the block described in onebit_device.h. K is padded up to a multiple of 256 with +1 values on
// positions 0,1 of each group; the GEMM kernels multiply that padding by zero rows of B.
//
// Bound: memory (m k 3/16 bytes each way). The 64 rows' value bits of one compressed column are one aligned 8-byte
// word of `a`, and consecutive columns lie m / 8 bytes apart, so a 128-byte line of `a` serves sixteen row pairs: the
// workgroups of an XCD walk down K in strips of sixteen row pairs, four workgroups side by side, and its L2 fetches a
// line once. (Row pairs of one workgroup / workgroups of a strip, us inside a HIP graph at 4096 x 11008 and 28672 x 8192:
// 2 / 8 5.8, 23.8; 4 / 4 5.4, 21.8; 8 / 2 6.1, 21.9; without strips, K fastest, 8 pairs: 6.3, 25.6.)
// A lane loads the words of the columns whose bits its own sign words hold, in bit order, so a 32 x 32 bit transpose per
// sign word replaces 64 extract-and-insert instructions; in the reference's layout the metadata of a row and the row
// four below it share a dword. Against one wavefront per block that gathers its sign bits through LDS (us): 4096 x 4096
// 3.8 -> 3.0, 11008 x 4096 7.6 -> 5.4, 4096 x 11008 10.0 -> 5.4, 8192 x 8192 10.3 -> 7.4, 28672 x 8192 34.9 -> 21.8
// (88 MB at 4.0 TB/s; a copy of 2 GiB runs at 4.9).
// =====================================================================================================
constexpr int kPreparePairs = 4, kPrepareStrip = 4;  // row pairs per workgroup, workgroups side by side in a strip

template <bool REFERENCE_LAYOUT>
__global__ __launch_bounds__(64 * kPreparePairs) void prepare_kernel(const uint8_t* __restrict__ a,
                                                                     const uint16_t* __restrict__ e,
                                                                     uint8_t* __restrict__ prep, int m, int k,
                                                                     int kc_total, int layout) {
  const int lane = threadIdx.x & 63;
  const StripPosition at = strip_position(kPrepareStrip, kc_total);
  const int kc = at.along;
  const int pair = at.across * kPreparePairs + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (pair >= m / 64) return;  // m % 64 == 0: every row of a pair exists
  const int i = lane & 31, ga = lane >> 5;
  const int ncols = k / 16;

  // Sign words: bit b of word h of lane (row, ga) is kept value t of K step s = 4 h + (j / 4), with b = 15 - j (t even)
  // or 31 - j (t odd), j = 4 (s % 4) + t / 2; kept value t of step s is compressed column 8 (2 s + ga) + t of the chunk.
  // Lane (b, ga) loads the column of bit b: .x the rows of the first row block, .y those of the second.
  u32x2_t column[2];
  const int j = 15 - (i & 15);
  const int64_t col0 = (int64_t)kc * 128 + 16 * (j >> 2) + 8 * ga + 2 * (j & 3) + (i >> 4);
  const bool aligned = (reinterpret_cast<uintptr_t>(a) & 7) == 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t col = col0 + 64 * h;
    column[h] = u32x2_t{0xFFFFFFFFu, 0xFFFFFFFFu};  // padding past K: +1
    if (col < k / 2) {
      const uint8_t* src = a + (((int64_t)pair * 64 + col * m) >> 3);
      if (aligned) column[h] = *reinterpret_cast<const u32x2_t*>(src);
      else __builtin_memcpy(&column[h], src, 8);
    }
  }
  u32x4_t meta[2];
  if constexpr (REFERENCE_LAYOUT) {
    // dword of rows r and r + 4 (b2 of the row = the dword's half), metadata column 16 kc + 2 s + ga
    const uint32_t* src = reinterpret_cast<const uint32_t*>(e) + (size_t)kc * 8 * m + (size_t)pair * 64 +
                          ((((i >> 1) & 1) << 5) | (((i >> 3) & 3) << 2) | ((i & 1) << 1) | ga);
    const uint32_t half = ((i >> 2) & 1) ? 0x07060302u : 0x05040100u;  // high or low halves of two steps' dwords
    uint32_t raw[2][kStepsPerChunk];
#pragma unroll
    for (int s = 0; s < kStepsPerChunk; ++s)
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        raw[blk][s] = 0x44444444u;
        if (kc * 16 + 2 * s < ncols) raw[blk][s] = src[(size_t)s * m + 16 * blk];  // ncols is even
      }
#pragma unroll
    for (int blk = 0; blk < 2; ++blk)
#pragma unroll
      for (int q = 0; q < 4; ++q) meta[blk][q] = __builtin_amdgcn_perm(raw[blk][2 * q + 1], raw[blk][2 * q], half);
  } else {
    // In every layout the element of column c + 2 lies a fixed distance after that of column c.
    const int c0 = kc * 16 + ga;
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      const int64_t r = (int64_t)pair * 64 + 32 * blk + i;
      int64_t off = layout == 0 ? meta_offset_reference(r, c0, m) : layout == 1 ? meta_offset_cutlass(r, c0, m) : r * ncols + c0;
      const int64_t off_step = layout == 2 ? 2 : 2 * (int64_t)m;
#pragma unroll
      for (int q = 0; q < 4; ++q) meta[blk][q] = 0;
#pragma unroll
      for (int s = 0; s < kStepsPerChunk; ++s) {
        uint32_t mv = 0x4444u;
        if (c0 + 2 * s < ncols) mv = e[off];
        off += off_step;
        meta[blk][s >> 1] |= mv << (16 * (s & 1));
      }
    }
  }
  const BitTranspose transpose(lane);
#pragma unroll
  for (int blk = 0; blk < 2; ++blk) {
    uint8_t* block = prep + ((size_t)(2 * pair + blk) * kc_total + kc) * kBlockBytes;
    *reinterpret_cast<u32x4_t*>(block + lane * 16) = meta[blk];
    // a set bit of the sign words means -1
    *reinterpret_cast<u32x2_t*>(block + kSignOffset + lane * 8) =
        u32x2_t{~transpose(column[0][blk]), ~transpose(column[1][blk])};
  }
}

// =====================================================================================================
// pack_kernel: dense weight (m x k, row-major; fp16, bf16 or fp32) -> the reference's stored operands (a bits, e metadata).
// Fuses the steps of BinaryLinear_2_4.pack (onebit_sparse_mul/__init__.py:130-145): optional 2:4 magnitude
// pruning (mask_creator, _semi_structured_conversions.py:286-314; among equal magnitudes the lower index is
// pruned first), compression to kept values + nibbles (:126-159, including the fixed encodings of groups
// with fewer or more than two non-zeros), sign quantisation (value > 0 -> 1, __init__.py:22-23), transposed
// bit packing (__init__.py:25-34,142-143) and the metadata reorder (:21-48).
//
// One wavefront = 64 rows x 64 K. The rows' 128 (fp32: 256) bytes come in by asynchronous copies and are turned in LDS,
// after which lane r holds row r: sixteen groups of four. Everything that decides about a group is one bit
// per value or per pair of values (which of two magnitudes is smaller, zero or not, the sign), so these bits are shifted
// into slices of sixteen groups, two values per 32-bit register, and the rules are then evaluated once for all sixteen
// groups with bitwise instructions. Slice bit 4 g + c belongs to group g of metadata column c: the four nibbles of a column
// are then four bits apart, as in its word. About 32 vector instructions per group where comparing floats group by
// group took about 110.
// Bound: memory (2 m k bytes in, m k 3/16 out). The workgroups of an XCD walk in strips of sixteen row tiles, as in
// prepare_kernel, so that the eight-byte pieces of a line of `a` meet in its L2. Row tiles per workgroup / workgroups of a
// strip, us inside a HIP graph at 11008 x 4096: 2 / 8 20.2, 4 / 4 20.6, 8 / 2 21.9, 16 / 1 24.2. Against 64-row wavefronts
// that read their own row's line lane by lane and compared floats: 4096 x 4096 26.2 -> 10.1 us, 11008 x 4096 68.4 -> 20.6
// (98 MB: 4.8 TB/s, the rate of a 2 GiB copy), 28672 x 8192 316 -> 105. bf16 and fp32 weights, which took the tensor route
// before (a sort of every group, some fifty launches): 11008 x 4096 15.4 ms -> 22 us and 27.8 ms -> 34 us.
// =====================================================================================================
constexpr int kPackTiles = 4, kPackStrip = 4;  // row tiles (wavefronts) per workgroup, workgroups side by side in a strip

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t packed_sub(uint32_t x, uint32_t y) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2_t, x) - __builtin_bit_cast(u16x2_t, y));
}
__device__ __forceinline__ uint32_t packed_add(uint32_t x, uint32_t y) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(u16x2_t, x) + __builtin_bit_cast(u16x2_t, y));
}
__device__ __forceinline__ uint32_t packed_min(uint32_t x, uint32_t y) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, x), __builtin_bit_cast(u16x2_t, y)));
}
__device__ __forceinline__ uint32_t majority(uint32_t x, uint32_t y, uint32_t z) { return ((x ^ y) & (z ^ x)) ^ x; }

// Bits of the weight's type. bf16 and fp32 weights follow the unfused route, w * mask and then (fp32) a rounding to half
// precision: what the mask removes from an infinite or NaN weight is NaN, which is not zero, and NaN counts as the
// largest magnitude; fp32 values up to 2^-25 become zero. fp16 weights keep the rule that NaN outranks nothing.
template <int DTYPE>
struct PackType;
template <>
struct PackType<kPackF16> {
  typedef _Float16 type;
  static constexpr uint32_t kInfinity = 0x7C00, kLargestZero = 0, kMagnitude = 0x7FFF7FFFu;
};
template <>
struct PackType<kPackBF16> {
  typedef uint16_t type;
  static constexpr uint32_t kInfinity = 0x7F80, kLargestZero = 0, kMagnitude = 0x7FFF7FFFu;
};
template <>
struct PackType<kPackF32> {
  typedef float type;
  static constexpr uint32_t kInfinity = 0x7F800000u, kLargestZero = 0x33000000u, kMagnitude = 0x7FFFFFFFu;
};

template <int DTYPE>
__global__ __launch_bounds__(64 * kPackTiles) void pack_kernel(const typename PackType<DTYPE>::type* __restrict__ w,
                                                               uint8_t* __restrict__ a, uint16_t* __restrict__ e, int m,
                                                               int k, int prune, int layout, int k_tiles) {
  using Type = PackType<DTYPE>;
  constexpr int SIZE = sizeof(typename Type::type);
  constexpr int ROW_BYTES = 64 * SIZE, PIECES = ROW_BYTES / 16, ROWS_PER_COPY = 64 / PIECES;
  constexpr bool NAN_RANKS = DTYPE != kPackF16;
  __shared__ __attribute__((aligned(16))) char lds[kPackTiles * 64 * ROW_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const StripPosition at = strip_position(kPackStrip, k_tiles);
  const int tile = at.across * kPackTiles + wave;
  if (tile >= m / 64) return;  // m % 64 == 0: every row of a tile exists; wavefronts do not meet at barriers
  const int64_t row0 = (int64_t)tile * 64;
  const int ncols = k / 16, c_first = at.along * 4;
  const int c_count = ncols - c_first < 4 ? ncols - c_first : 4;  // the last tile may hold two columns only (k % 32 == 0)

  // ---- 64 rows into LDS, whole rows per copy; piece q (16 bytes) of row r goes to position q ^ (r % PIECES)
  char* const image = lds + wave * (64 * ROW_BYTES);
  {
    const char* src = reinterpret_cast<const char*>(w + (row0 + lane / PIECES) * k + 16 * c_first);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int piece = (lane % PIECES) ^ ((i * ROWS_PER_COPY + lane / PIECES) % PIECES);
      const int from = piece < SIZE * c_count ? piece : 0;  // past K: any valid address will do, the results are not stored
      lds_dma16(src + (size_t)i * ROWS_PER_COPY * SIZE * k + 16 * from, lds_offset_of(image) + i * 1024);
    }
  }
  wait_vmcnt<0>();
  uint32_t d[ROW_BYTES / 4];  // the row; group q (four values): two dwords of two values, or (fp32) four dwords
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(image + lane * ROW_BYTES + ((q ^ (lane % PIECES)) << 4));
    d[4 * q] = v.x; d[4 * q + 1] = v.y; d[4 * q + 2] = v.z; d[4 * q + 3] = v.w;
  }

  // ---- slices. less_ij: magnitude j < magnitude i (i < j), i.e. i outranks j; otherwise j outranks i (ties: the higher
  // index). Low half | high half of a register: 02|13, 03|12, 01|23 for pairs, 0|1 and 2|3 for single values.
  uint32_t less_02_13 = 0, less_03_12 = 0, less_01_23 = 0, nonzero_01 = 0, nonzero_23 = 0, nan_01 = 0, nan_23 = 0,
           minus_01 = 0, minus_23 = 0, huge_01 = 0, huge_23 = 0;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const int q = 4 * (t & 3) + (t >> 2);  // group t / 4 of column t % 4
    auto push = [](uint32_t& slice, uint32_t x) __attribute__((always_inline)) {  // bits 15 and 31 of x
      slice = (x & 0x80008000u) | ((slice >> 1) & 0x7FFF7FFFu);
    };
    if constexpr (SIZE == 2) {
      const uint32_t d0 = d[2 * q], d1 = d[2 * q + 1];
      uint32_t m0 = d0 & Type::kMagnitude, m1 = d1 & Type::kMagnitude;  // magnitudes order like their bits
      if constexpr (NAN_RANKS) m0 = packed_min(m0, (Type::kInfinity + 1) * 0x10001u), m1 = packed_min(m1, (Type::kInfinity + 1) * 0x10001u);
      push(less_02_13, packed_sub(m1, m0));
      push(less_03_12, packed_sub(__builtin_amdgcn_alignbit(m1, m1, 16), m0));
      push(less_01_23, packed_sub(__builtin_amdgcn_perm(m1, m0, 0x07060302u), __builtin_amdgcn_perm(m1, m0, 0x05040100u)));
      // magnitude > limit sets bit 15 of magnitude + (0x7FFF - limit)
      constexpr uint32_t kNonzero = 0x7FFFu * 0x10001u, kNan = (0x7FFFu - Type::kInfinity) * 0x10001u;
      push(nonzero_01, packed_add(m0, kNonzero));
      push(nonzero_23, packed_add(m1, kNonzero));
      push(nan_01, packed_add(m0, kNan));
      push(nan_23, packed_add(m1, kNan));
      if constexpr (NAN_RANKS) push(huge_01, packed_add(m0, kNan + 0x10001u)), push(huge_23, packed_add(m1, kNan + 0x10001u));
      push(minus_01, d0);
      push(minus_23, d1);
    } else {
      uint32_t mag[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mag[i] = d[4 * q + i] & Type::kMagnitude;
        mag[i] = mag[i] < Type::kInfinity + 1 ? mag[i] : Type::kInfinity + 1;  // every NaN alike
      }
      // bits 31 of two words to bits 15 and 31
      auto tops = [](uint32_t low, uint32_t high) __attribute__((always_inline)) {
        return __builtin_amdgcn_perm(high, low, 0x07060302u);
      };
      push(less_02_13, tops(mag[2] - mag[0], mag[3] - mag[1]));
      push(less_03_12, tops(mag[3] - mag[0], mag[2] - mag[1]));
      push(less_01_23, tops(mag[1] - mag[0], mag[3] - mag[2]));
      constexpr uint32_t kNonzero = 0x7FFFFFFFu - Type::kLargestZero, kNan = 0x7FFFFFFFu - Type::kInfinity;
      push(nonzero_01, tops(mag[0] + kNonzero, mag[1] + kNonzero));
      push(nonzero_23, tops(mag[2] + kNonzero, mag[3] + kNonzero));
      push(nan_01, tops(mag[0] + kNan, mag[1] + kNan));
      push(nan_23, tops(mag[2] + kNan, mag[3] + kNan));
      push(huge_01, tops(mag[0] + (kNan + 1), mag[1] + (kNan + 1)));
      push(huge_23, tops(mag[2] + (kNan + 1), mag[3] + (kNan + 1)));
      push(minus_01, tops(d[4 * q], d[4 * q + 1]));
      push(minus_23, tops(d[4 * q + 2], d[4 * q + 3]));
    }
  }

  // ---- the rules, on 16-bit slices (the upper halves of these registers hold other slices and are masked at the end)
  const uint32_t nan0 = nan_01, nan1 = nan_01 >> 16, nan2 = nan_23, nan3 = nan_23 >> 16;
  uint32_t keep0 = ~0u, keep1 = ~0u, keep2 = ~0u, keep3 = ~0u;
  if (prune) {
    // fp16: a comparison with NaN is false both ways
    auto comparable = [](uint32_t x, uint32_t y) __attribute__((always_inline)) { return NAN_RANKS ? ~0u : ~(x | y); };
    const uint32_t ok01 = comparable(nan0, nan1), ok02 = comparable(nan0, nan2), ok03 = comparable(nan0, nan3),
                   ok12 = comparable(nan1, nan2), ok13 = comparable(nan1, nan3), ok23 = comparable(nan2, nan3);
    const uint32_t l01 = less_01_23, l23 = less_01_23 >> 16, l02 = less_02_13, l13 = less_02_13 >> 16, l03 = less_03_12,
                   l12 = less_03_12 >> 16;
    // a value goes when two of the other three outrank it
    keep0 = ~majority(~l01 & ok01, ~l02 & ok02, ~l03 & ok03);
    keep1 = ~majority(l01 & ok01, ~l12 & ok12, ~l13 & ok13);
    keep2 = ~majority(l02 & ok02, l12 & ok12, ~l23 & ok23);
    keep3 = ~majority(l03 & ok03, l13 & ok13, l23 & ok23);
  }
  uint32_t p0 = keep0 & nonzero_01, p1 = keep1 & (nonzero_01 >> 16), p2 = keep2 & nonzero_23,
           p3 = keep3 & (nonzero_23 >> 16);
  const uint32_t plus0 = p0 & ~minus_01 & ~nan0, plus1 = p1 & ~(minus_01 >> 16) & ~nan1, plus2 = p2 & ~minus_23 & ~nan2,
                 plus3 = p3 & ~(minus_23 >> 16) & ~nan3;
  if (NAN_RANKS && prune) p0 |= huge_01, p1 |= huge_01 >> 16, p2 |= huge_23, p3 |= huge_23 >> 16;  // 0 * infinity
  // Bits of the nibble idx0 | idx1 << 2 for the pattern of non-zeros (p0 p1 p2 p3). With p0 and p1 it names 0 and 1; with
  // one of them, that one and 3 if p3, else 2; with neither, 2 and 3. (Which also gives the reference's fixed encodings
  // of groups with other than two non-zeros.)
  const uint32_t n0 = ~p0 & p1, n1 = ~(p0 | p1), n2 = ~(p0 ^ p1) | p3, n3 = ~(p0 & p1);
  // signs of the two kept values, one bit per group: the first in the low half, the second in the high half
  const uint32_t first = plus0 | (~p0 & (plus1 | (~p1 & plus2)));
  const uint32_t second = (~n3 & plus1) | (n3 & ((n2 & plus3) | (~n2 & plus2)));

  // ---- a: lane (half h, bit b) of the transposed slices holds rows 32 h ... 32 h + 31 of bit b, which is kept value
  // 2 g + b / 16 of column c (b % 16 = 4 g + c)
  const BitTranspose transpose(lane);
  const uint32_t rows = transpose((first & 0xFFFFu) | (second << 16));
  {
    const int b = lane & 31, c = b & 3;
    const int64_t column = 8 * (c_first + c) + 2 * ((b >> 2) & 3) + (b >> 4);
    if (c < c_count) *reinterpret_cast<uint32_t*>(a + ((row0 + 32 * (lane >> 5) + column * m) >> 3)) = rows;
  }

  // ---- e: the words of the four columns
  uint32_t word[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint32_t b0 = n0 >> c, b1 = c < 1 ? n1 << 1 : n1 >> (c - 1), b2 = c < 2 ? n2 << (2 - c) : n2 >> (c - 2),
                   b3 = c < 3 ? n3 << (3 - c) : n3;
    word[c] = (b0 & 0x1111u) | (b1 & 0x2222u) | (b2 & 0x4444u) | (b3 & 0x8888u);
  }
  if (layout == 0 && (reinterpret_cast<uintptr_t>(e) & 3) == 0) {
    // Rows r and r + 4 of one column share a dword, and the dwords of an even and the next odd column are neighbours: the
    // lane of row r stores the even column's, the lane of row r + 4 the odd column's; 256 consecutive bytes per pair.
    const bool upper = (lane >> 2) & 1;
    uint32_t* const dst = reinterpret_cast<uint32_t*>(e) + row0 +
                          ((((lane >> 1) & 1) << 5) | ((lane >> 3) << 2) | ((lane & 1) << 1) | ((lane >> 2) & 1));
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
      const uint32_t other = __builtin_amdgcn_ds_swizzle(upper ? word[c] : word[c + 1], (4 << 10) | 0x1F);
      const uint32_t pair = upper ? other | (word[c + 1] << 16) : word[c] | (other << 16);
      if (c < c_count) dst[(size_t)((c_first + c) >> 1) * m] = pair;
    }
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (c >= c_count) break;  // wave-uniform
      const int64_t r = row0 + lane;
      const int64_t off = layout == 0   ? meta_offset_reference(r, c_first + c, m)
                          : layout == 1 ? meta_offset_cutlass(r, c_first + c, m)
                                        : r * ncols + c_first + c;
      e[off] = (uint16_t)word[c];
    }
  }
}

hipError_t launch_prepare(const void* a, const void* e, void* prep, int m, int k, int layout, hipStream_t stream) {
  const int kc_total = (k + kChunkK - 1) / kChunkK;
  constexpr int kStripPairs = kPreparePairs * kPrepareStrip;
  const dim3 grid(kc_total * kPrepareStrip * ((m / 64 + kStripPairs - 1) / kStripPairs));
  // the dword form of the metadata loads needs e on a 4-byte boundary
  const auto kernel = layout == 0 && (reinterpret_cast<uintptr_t>(e) & 3) == 0 ? prepare_kernel<true> : prepare_kernel<false>;
  return launch_kernel(kernel, grid, dim3(64 * kPreparePairs), 0, stream, (const uint8_t*)a, (const uint16_t*)e, (uint8_t*)prep, m, k,
                       kc_total, layout);
}

template <int DTYPE>
static hipError_t launch_pack_type(const void* w, void* a, void* e, int m, int k, int prune, int layout, hipStream_t stream) {
  const int k_tiles = (k / 16 + 3) / 4;
  constexpr int kStripTiles = kPackTiles * kPackStrip;
  const dim3 grid(k_tiles * kPackStrip * ((m / 64 + kStripTiles - 1) / kStripTiles));
  return launch_kernel(pack_kernel<DTYPE>, grid, dim3(64 * kPackTiles), 0, stream, (const typename PackType<DTYPE>::type*)w, (uint8_t*)a,
                       (uint16_t*)e, m, k, prune, layout, k_tiles);
}

hipError_t launch_pack(const void* w, int dtype, void* a, void* e, int m, int k, int prune, int layout, hipStream_t stream) {
  switch (dtype) {
    case kPackF32: return launch_pack_type<kPackF32>(w, a, e, m, k, prune, layout, stream);
    case kPackF16: return launch_pack_type<kPackF16>(w, a, e, m, k, prune, layout, stream);
    case kPackBF16: return launch_pack_type<kPackBF16>(w, a, e, m, k, prune, layout, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace onebit
