// gfx950 kernels that bring a weight into the stored format and into the operand the GEMM kernels consume.
//   prepare_kernel  : reference operands (1-bit values, reordered 2-bit-index metadata) -> prepared operand
//   pack_kernel     : dense fp16 weight -> the reference operands (2:4 magnitude mask, compression, one-bit values)
#include "onebit_device.h"
#include "onebit_launch.h"

namespace onebit {

// =====================================================================================================
// prepare_kernel: one wavefront per prepared block (rb, kc).
// Reads  a : bit (r, j) of the (m x k/2) column-major one-bit matrix = bit (r + j m) % 8 of byte (r + j m) / 8
//            (csrc/kernel_lib.cu:28,37; produced by onebit_sparse_mul/__init__.py:139-143), 1 = +1, 0 = -1
//        e : int16 metadata (m x k/16) in the reference's reordered layout or the CUTLASS one
//            (_semi_structured_conversions.py:21-48,173-177)
// Writes the block described in onebit_device.h. K is padded up to a multiple of 256 with +1 values on
// positions 0,1 of each group; the GEMM kernels multiply that padding by zero rows of B.
// =====================================================================================================
__global__ __launch_bounds__(64) void prepare_kernel(const uint8_t* __restrict__ a, const uint16_t* __restrict__ e,
                                                     uint8_t* __restrict__ prep, int m, int k, int kc_total,
                                                     int layout) {
  const int kc = blockIdx.x, rb = blockIdx.y, lane = threadIdx.x;
  const int i = lane & 31, ga = lane >> 5;
  const int64_t r = (int64_t)rb * kRowBlock + i;  // m % 32 == 0: every row of the block exists
  const int ncols = k / 16;
  // The value bits of the block's 32 rows for one compressed column are one aligned dword of `a` (bit position
  // 32 rb + j m, m % 32 == 0). The block spans 128 compressed columns: two dwords per lane, shared through LDS.
  __shared__ __attribute__((aligned(16))) uint32_t column_bits[128];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int local = lane + 64 * half;
    const int64_t j = (int64_t)kc * 128 + local;     // compressed column
    uint32_t word = 0xFFFFFFFFu;                      // padding past K: +1
    if (j < k / 2) {
      const uint8_t* src = a + (((int64_t)rb * kRowBlock + j * m) >> 3);
      if ((reinterpret_cast<uintptr_t>(a) & 3) == 0)
        word = *reinterpret_cast<const uint32_t*>(src);
      else
        word = (uint32_t)src[0] | ((uint32_t)src[1] << 8) | ((uint32_t)src[2] << 16) | ((uint32_t)src[3] << 24);
    }
    column_bits[local] = ~word;  // stored inverted: a set bit now means -1, which is what the sign words hold
  }
  __syncthreads();
  uint32_t meta[4] = {0, 0, 0, 0};
  uint32_t sign[2] = {0, 0};
  // metadata column of step s: c = 16 kc + 2 s + ga. In all three layouts the element of column c + 2 lies a fixed
  // distance after that of column c (one column pair = 2 m elements in the reordered layouts), so one offset is
  // computed and then advanced.
  const int c0 = kc * 16 + ga;
  int64_t off = layout == 0 ? meta_offset_reference(r, c0, m) : layout == 1 ? meta_offset_cutlass(r, c0, m) : r * ncols + c0;
  const int64_t off_step = layout == 2 ? 2 : 2 * (int64_t)m;
#pragma unroll
  for (int s = 0; s < kStepsPerChunk; ++s) {
    const int c = c0 + 2 * s;
    uint32_t mv = 0x4444u;
    if (c < ncols) mv = e[off];
    off += off_step;
    meta[s >> 1] |= mv << (16 * (s & 1));
    // kept value t of this step = compressed column 8 c + t = entry 8 (2 s + ga) + t of the block's 128; it goes to
    // bit 15 - j (t even) or 31 - j (t odd) of the step group's sign word, j = 4 (s % 4) + t / 2: one bit-field
    // extract and one shift-or per value
    const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(&column_bits[8 * (2 * s + ga)]);
    const u32x4_t hi = *reinterpret_cast<const u32x4_t*>(&column_bits[8 * (2 * s + ga) + 4]);
    const uint32_t w8[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int j = 4 * (s & 3) + (t >> 1);
      const int position = ((t & 1) ? 31 : 15) - j;
      sign[s >> 2] |= ((w8[t] >> i) & 1u) << position;
    }
  }
  uint8_t* block = prep + ((size_t)rb * kc_total + kc) * kBlockBytes;
  u32x4_t mvec = {meta[0], meta[1], meta[2], meta[3]};
  u32x2_t svec = {sign[0], sign[1]};
  *reinterpret_cast<u32x4_t*>(block + lane * 16) = mvec;
  *reinterpret_cast<u32x2_t*>(block + kSignOffset + lane * 8) = svec;
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
  const int rb_total = (m + kRowBlock - 1) / kRowBlock;
  dim3 grid(kc_total, rb_total);
  hipLaunchKernelGGL(prepare_kernel, grid, dim3(64), 0, stream, (const uint8_t*)a, (const uint16_t*)e, (uint8_t*)prep,
                     m, k, kc_total, layout);
  return hipGetLastError();
}

hipError_t launch_pack(const void* w, void* a, void* e, int m, int k, int prune, int layout, hipStream_t stream) {
  hipLaunchKernelGGL(pack_kernel, dim3((k / 16 + 3) / 4, m / 64), dim3(64), 0, stream, (const _Float16*)w, (uint8_t*)a,
                     (uint16_t*)e, m, k, prune, layout);
  return hipGetLastError();
}

}  // namespace onebit
