// Host-visible launch interface of the gfx950 kernels (internal to libonebitmul).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace onebit {

// A kernel's launch by the runtime's own entry: 2.28 us on the host, 2.42 with the launch syntax, which hands the geometry over in a call of
// its own, and 0.04 for asking for the error apart.
template <class... Parameters>
inline hipError_t launch_kernel(void (*kernel)(Parameters...), dim3 grid, dim3 threads, size_t lds, hipStream_t stream, Parameters... arguments) {
  void* pointers[] = {&arguments...};
  const hipError_t status = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, threads, pointers, lds, stream);
  if (status != hipSuccess) (void)hipGetLastError();  // reported here, not by the next call
  return status;
}

struct GemmArgs {
  const uint8_t* prep;   // prepared A operand
  const _Float16* b;     // K x N row-major fp16
  const void* c;         // M x N row-major source (read only when beta != 0)
  void* d;               // M x N row-major destination
  int m, n, k;
  int kc_total;          // 256-wide K chunks in the prepared operand
  float alpha, beta;
  int c_f16, d_f16;      // 1: fp16, 0: fp32
  int tiles_m, tiles_n;  // filled by the launcher
  int xcds;              // filled by the launcher: XCDs the workgroups are dealt over (workgroup b runs on XCD b % xcds)
  // K split over workgroups (grid.y = splits): split s multiplies the K chunks [s * chunks_per_split, +chunks_per_split)
  // and writes raw fp32 sums to split_ws + s * m * n; a second kernel adds the splits in order and applies the
  // epilogue. splits <= 1: one pass straight into d. split_ws: at least splits * m * n floats, 16-byte aligned.
  int splits;
  int chunks_per_split;
  float* split_ws;
  // B whose rows are not 16-byte aligned (n % 8 != 0, or a base address that is not): if b_pad is set (at least
  // k * round_up(n, 8) halves, 16-byte aligned), the launcher first copies B into it with rows padded to a multiple of 8
  // columns and the main kernel reads that; otherwise a B that may be read as a ragged one (read_as_ragged) is copied to
  // LDS from where it lies, and what is left takes the slower element-copy variant. ldb (elements between B rows) is filled
  // by the launcher.
  _Float16* b_pad;
  int ldb;
  // linear-layer form (launch_gemm_tokens) only: m values added to every token's row of y, may be null; its type (ElementType);
  // bf16 = 1: x is bf16, and so is a 16-bit y (d_f16 = 1)
  const void* bias;
  int bias_type;
  int bf16;
};

struct SkinnyArgs {
  const uint8_t* prep;
  const _Float16* b;
  const void* c;
  void* d;
  int m, n, k;
  int kc_total;
  float alpha, beta;
  int c_f16, d_f16;
  // token-major form (launch_skinny_tokens) only: b is x (n tokens x k), d is y (n tokens x m), alpha, beta and c are
  // not used, bias (m values, may be null, of type bias_type) is added to every token's row; bf16 = 1: x is bf16, and so is
  // a 16-bit y (d_f16 = 1)
  const void* bias;
  int bias_type;
  int bf16;
  // K split over workgroups (grid.y = splits), for few row groups over a long K: split s multiplies the K chunks
  // [s * chunks_per_split, +chunks_per_split) and writes raw fp32 sums to split_ws + s * m * n (laid out like the
  // result); a second kernel adds the splits in order and applies the epilogue. splits <= 1: one pass straight into d.
  int splits;
  int chunks_per_split;
  float* split_ws;
  // launch_skinny_tokens only: b is x in fp32, rounded to fp16 as it is read (bf16 = 0)
  int x_f32;
  // wide_kernel only: tokens (columns) a workgroup multiplies (at most 64); strips: the grid is walked in strips of two column
  // groups, on a device of eight XCDs; ldb: elements between B rows in the plain form, n rounded up to eight or n itself
  int tokens_per_group;
  int strips;
  int ldb;
};

// Several token-major products with the same token count in one launch of the split-K kernel (no K split over
// workgroups); first_block is filled by the launcher.
constexpr int kSkinnyMaxGroup = 16;
struct SkinnyGroupArgs {
  SkinnyArgs problem[kSkinnyMaxGroup];
  int first_block[kSkinnyMaxGroup + 1];
  int count;
};

// Whether the asynchronous copies can read a B of rows that are no whole 16-byte pieces where it lies. They take 16 bytes from any
// address; a piece that starts at an odd multiple of two bytes costs 3.8 times as much of a compute unit's load path as one on a
// 4-byte boundary (64 rows of 128 bytes, ldb = 64 | 66 | 68 | 65, one workgroup: 14.8 | 14.8 | 14.8 | 35.2 us). At least eight
// values a row, so that only the last row's last piece reaches past B.
inline bool read_as_ragged(const void* b, int n) { return n >= 8 && (reinterpret_cast<uintptr_t>(b) & 15) == 0; }

enum TileConfig { kTile512x128 = 0, kTile256x128 = 1, kTile128x128 = 2, kTile256x256 = 3, kTile256x128w = 4, kTile512x128t = 5, kTile128x128s = 6, kTile256x64 = 7, kTile256x256w8 = 8, kTile512x128w8 = 9, kTile256x128w8 = 10, kTile128x128w8 = 11, kTile64x128 = 12, kTile128x128k2 = 13, kTile64x128k2 = 14, kTile512x128m16 = 15, kTileAuto = -1 };

// Whether the main kernel's tile has a build that reads a ragged B: those that the plan chooses.
inline bool tile_reads_ragged(int tile) {
  switch (tile) {
    case kTile256x128w: case kTile128x128s: case kTile512x128w8: case kTile256x128w8: case kTile128x128w8: case kTile64x128:
    case kTile128x128k2: case kTile64x128k2: case kTile512x128m16: return true;
    default: return false;
  }
}

hipError_t launch_prepare(const void* a, const void* e, void* prep, int m, int k, int layout, hipStream_t stream);
hipError_t launch_gemm(GemmArgs args, int tile_config, hipStream_t stream);
// The linear layer's form of the main kernel: b is x (n tokens x k, token-major, 16-byte aligned), d is y (n tokens x
// m), y = x W^T + bias; c, alpha, beta and the padded copy of B are not used, splits / chunks_per_split / split_ws as in
// launch_gemm. Tiles 4, 6, 9, 10, 11, 12, 13, 14, 15.
hipError_t launch_gemm_tokens(GemmArgs args, int tile_config, hipStream_t stream);
// dense (m x k) -> one-bit values `a` and metadata `e`; prune != 0 applies the 2:4 magnitude mask first. dtype: the codes
// of the C ABI.
enum PackDtype { kPackF32 = 0, kPackF16 = 1, kPackBF16 = 2 };
hipError_t launch_pack(const void* w, int dtype, void* a, void* e, int m, int k, int prune, int layout, hipStream_t stream);

// Second pass of a K split: ordered sum of the partial results and the epilogue (bias and row_length for the
// token-major form, where element i of y takes bias[i % m]).
hipError_t launch_split_reduce(const float* ws, int splits, size_t total, const void* c, void* d, float alpha,
                                      float beta, int c_f16, int d_type, const void* bias, int bias_type, int row_length,
                                      hipStream_t stream);

// B with rows padded to a multiple of eight columns (dst: k * round_up(n, 8) halves).
hipError_t launch_pad_b(const _Float16* b, _Float16* dst, int k, int n, hipStream_t stream);

// Split-K kernel for n <= 64; rows_per_group (32, 64 or 128) = weight rows one workgroup covers (n > 32: at most 64).
constexpr int kSkinnyMaxN = 64;
hipError_t launch_skinny(SkinnyArgs args, int rows_per_group, hipStream_t stream);
// The linear layer's form of the same kernel: y[t][r] = sum_k W[r][k] x[t][k] + bias[r] for n <= kSkinnyTokens tokens, x and y
// token-major (x 16-byte aligned).
constexpr int kSkinnyTokens = 16;
hipError_t launch_skinny_tokens(SkinnyArgs args, int rows_per_group, hipStream_t stream);
// count <= kSkinnyMaxGroup problems of the same form, each with its own weight, x, bias, y, m and k, in one launch.
hipError_t launch_skinny_group(SkinnyGroupArgs group, int rows_per_group, hipStream_t stream);

// The linear layer's form whose images of x asynchronous copies bring to LDS (wide_kernel): any number of tokens, in
// groups of at most 64 per workgroup; row groups of 32, 64 or 128.
hipError_t launch_wide_tokens(SkinnyArgs args, int rows_per_group, hipStream_t stream);
// The plain form: B 16-byte aligned with ldb % 8 == 0, columns in groups of a multiple of eight, at most 64.
hipError_t launch_wide(SkinnyArgs args, int rows_per_group, hipStream_t stream);
hipError_t launch_wide_tokens_group(SkinnyGroupArgs group, int rows_per_group, hipStream_t stream);

}  // namespace onebit
