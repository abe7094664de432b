// gfx950 kernels that bring a weight into the stored format and into the operand the GEMM kernels consume.
//   prepare_kernel  : reference operands (1-bit values, reordered 2-bit-index metadata) -> prepared operand
//   pack_kernel     : dense fp16 weight -> the reference operands (2:4 magnitude mask, compression, one-bit values)
#include "onebit_device.h"
#include "onebit_launch.h"

namespace onebit {

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
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous range of the list ordered row groups fastest
  const int per = gridDim.x / 8, rem = gridDim.x % 8, xcd = blockIdx.x % 8;
  const int v = xcd * per + (xcd < rem ? xcd : rem) + blockIdx.x / 8;
  const int strip = v / (kPrepareStrip * kc_total), w = v % (kPrepareStrip * kc_total);
  const int kc = w / kPrepareStrip;
  const int pair = (strip * kPrepareStrip + w % kPrepareStrip) * kPreparePairs + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
// pack_kernel: dense fp16 weight (m x k, row-major) -> the reference's stored operands (a bits, e metadata).
// Fuses the steps of BinaryLinear_2_4.pack (onebit_sparse_mul/__init__.py:130-145): optional 2:4 magnitude
// pruning (mask_creator, _semi_structured_conversions.py:286-314; among equal magnitudes the lower index is
// pruned first), compression to kept values + nibbles (:126-159, including the fixed encodings of groups
// with fewer or more than two non-zeros), sign quantisation (value > 0 -> 1, __init__.py:22-23), transposed
// bit packing (__init__.py:25-34,142-143) and the metadata reorder (:21-48).
// One wavefront = 64 consecutive rows x four metadata columns (64 dense K, one 128-byte line per row); the eight
// sign bits of a row and column are gathered across the wavefront with ballots, so every store of `a` is 8 bytes
// of 64 consecutive rows.
// =====================================================================================================
__device__ __constant__ uint8_t kNibbleOfPattern[16] = {0xE, 0x8, 0x9, 0x4, 0xE, 0x8, 0x9, 0x4,
                                                        0xE, 0xC, 0xD, 0x4, 0xE, 0xC, 0xD, 0x4};

__global__ __launch_bounds__(64) void pack_kernel(const _Float16* __restrict__ w, uint8_t* __restrict__ a,
                                                  uint16_t* __restrict__ e, int m, int k, int prune, int layout) {
  const int64_t r = (int64_t)blockIdx.y * 64 + threadIdx.x;  // m % 64 == 0: always a valid row
  const int ncols = k / 16;
  // four metadata columns (64 weights = 128 consecutive bytes of the lane's row) per wavefront: requests of whole
  // 128-byte lines; the last group of a row may hold two columns only (k % 32 == 0)
  const int c_first = blockIdx.x * 4;
  const int c_count = ncols - c_first < 4 ? ncols - c_first : 4;
  u32x4_t line[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (i < 2 * c_count) line[i] = reinterpret_cast<const u32x4_t*>(w + r * k + 16 * c_first)[i];
#pragma unroll
  for (int ci = 0; ci < 4; ++ci) {
    if (ci >= c_count) break;  // wave-uniform
    const int c = c_first + ci;                       // metadata column
    u32x4_t raw[2] = {line[2 * ci], line[2 * ci + 1]};
    _Float16 v[16];
    __builtin_memcpy(v, raw, 32);
    uint32_t word = 0, bits = 0;  // bits: bit t = kept value t of this metadata element is > 0
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float x[4], mag[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = (float)v[4 * g + i];
        mag[i] = x[i] < 0.f ? -x[i] : x[i];
      }
      int pattern = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bool keep = true;
        if (prune) {
          int beaten = 0;  // elements that outrank i: larger magnitude, or equal magnitude and higher index
#pragma unroll
          for (int j = 0; j < 4; ++j) beaten += (j != i) && (mag[j] > mag[i] || (mag[j] == mag[i] && j > i));
          keep = beaten < 2;
        }
        if (!keep) x[i] = 0.f;
        pattern |= (x[i] != 0.f) << i;
      }
      const int nib = kNibbleOfPattern[pattern];
      const int i0 = nib & 3, i1 = nib >> 2;
      word |= (uint32_t)nib << (4 * g);
      float k0 = x[0], k1 = x[0];
#pragma unroll
      for (int i = 1; i < 4; ++i) {
        if (i0 == i) k0 = x[i];
        if (i1 == i) k1 = x[i];
      }
      bits |= (uint32_t)(k0 > 0.f) << (2 * g);
      bits |= (uint32_t)(k1 > 0.f) << (2 * g + 1);
    }
    int64_t off;
    if (layout == 0) off = meta_offset_reference(r, c, m);
    else if (layout == 1) off = meta_offset_cutlass(r, c, m);
    else off = r * ncols + c;
    e[off] = (uint16_t)word;
    const int64_t row0 = (int64_t)blockIdx.y * 64;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const uint64_t mask = __ballot((bits >> t) & 1u);  // bit l = row row0 + l, compressed column 8c + t
      if (threadIdx.x == 0) {
        const int64_t pos = row0 + (int64_t)(8 * c + t) * m;  // multiple of 64
        *reinterpret_cast<uint64_t*>(a + (pos >> 3)) = mask;
      }
    }
  }
}

hipError_t launch_prepare(const void* a, const void* e, void* prep, int m, int k, int layout, hipStream_t stream) {
  const int kc_total = (k + kChunkK - 1) / kChunkK;
  constexpr int kStripPairs = kPreparePairs * kPrepareStrip;
  const dim3 grid(kc_total * kPrepareStrip * ((m / 64 + kStripPairs - 1) / kStripPairs));
  // the dword form of the metadata loads needs e on a 4-byte boundary
  const auto kernel = layout == 0 && (reinterpret_cast<uintptr_t>(e) & 3) == 0 ? prepare_kernel<true> : prepare_kernel<false>;
  hipLaunchKernelGGL(kernel, grid, dim3(64 * kPreparePairs), 0, stream, (const uint8_t*)a, (const uint16_t*)e,
                     (uint8_t*)prep, m, k, kc_total, layout);
  return hipGetLastError();
}

hipError_t launch_pack(const void* w, void* a, void* e, int m, int k, int prune, int layout, hipStream_t stream) {
  hipLaunchKernelGGL(pack_kernel, dim3((k / 16 + 3) / 4, m / 64), dim3(64), 0, stream, (const _Float16*)w, (uint8_t*)a,
                     (uint16_t*)e, m, k, prune, layout);
  return hipGetLastError();
}

}  // namespace onebit
