// Plain form of the main kernel and its helpers: pad_b_kernel (unaligned B rows), splitk_reduce_kernel (K split).
#include "onebit_gemm.h"

namespace onebit {

// =====================================================================================================
// pad_b_kernel: copies B (k x n, row stride n, any alignment) into rows of ldb = round_up(n, 8) halves, so that every row starts 16-byte aligned for the asynchronous copies of the main kernel.
// Bound: memory, 2 k n bytes each way (and a few us of launch and latency below about 10 MB). A workgroup takes `rows`
// whole rows, as many as fit its 1024 pieces, or 1024 pieces of one longer row, so that neighbouring lanes write
// neighbouring pieces across row ends; the four loads of a thread, 16 bytes at any alignment, come before its first store.
// Against two-byte loads, one piece per thread (us): 4096 x 1001 9.0 -> 7.0, 20864 x 707 18.3 -> 12.0, 12832 x 3241 41.7 -> 29.3.
// =====================================================================================================
constexpr int kPadPieces = 1024;

// rows > 1: reciprocal = 2^32 / (ldb / 8) + 1, with which the quotients below 2^11 that occur are exact
__global__ __launch_bounds__(256) void pad_b_kernel(const _Float16* __restrict__ b, _Float16* __restrict__ dst, int k,
                                                    int n, int ldb, int rows, uint32_t reciprocal) {
  const int row0 = blockIdx.x * rows, per_row = ldb / 8, piece0 = blockIdx.y * kPadPieces;
  const size_t last_start = (size_t)k * n - 8;  // k >= 32
  u32x4_t v[kPadPieces / 256];
#pragma unroll
  for (int i = 0; i < kPadPieces / 256; ++i) {
    const int local = threadIdx.x + 256 * i;
    const int r = rows > 1 ? (int)__umulhi(local, reciprocal) : 0, col = 8 * (piece0 + local - r * per_row);
    // a piece that reaches past the end of its row takes the next row's first values along: nothing is made of them, they
    // only meet columns that are never stored. Past the end of B it is moved back and shifted into place below.
    const size_t start = (size_t)(row0 + r) * n + col;
    v[i] = *reinterpret_cast<const u32x4_any_t*>(b + (start <= last_start ? start : last_start));
  }
#pragma unroll
  for (int i = 0; i < kPadPieces / 256; ++i) {
    const int local = threadIdx.x + 256 * i;
    const int r = rows > 1 ? (int)__umulhi(local, reciprocal) : 0, col = 8 * (piece0 + local - r * per_row);
    const int row = row0 + r;
    if (r >= rows || row >= k || col >= ldb) continue;
    const size_t start = (size_t)row * n + col;
    if (start > last_start) v[i] = drop_halves(v[i], (int)(start - last_start));
    *reinterpret_cast<u32x4_t*>(dst + (size_t)row * ldb + col) = v[i];
  }
}

// =====================================================================================================
// splitk_reduce_kernel: d = alpha * (sum over splits, in split order, of the fp32 partial sums) + beta * c.
// Elementwise over the m * n results; VEC = 4 when the element count and the alignment of c and d allow it.
// Linear-layer form: bias (row_length values, may be null) is added instead, element i taking bias[i % row_length].
// =====================================================================================================
template <int VEC>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ ws, int splits, size_t stride,
                                                            const void* __restrict__ c, void* __restrict__ d,
                                                            size_t total, float alpha, float beta, int c_f16,
                                                            int d_type, const void* __restrict__ bias, int bias_type,
                                                            int row_length) {
  const size_t first = ((size_t)blockIdx.x * 256 + threadIdx.x) * VEC;
  if (first >= total) return;
  float x[VEC];
#pragma unroll
  for (int j = 0; j < VEC; ++j) x[j] = 0.f;
  for (int s = 0; s < splits; ++s) {
    const float* src = ws + (size_t)s * stride + first;
    if (VEC == 4) {
      const float4 v = *reinterpret_cast<const float4*>(src);
      x[0] += v.x; x[1 % VEC] += v.y; x[2 % VEC] += v.z; x[3 % VEC] += v.w;
    } else {
      x[0] += src[0];
    }
  }
#pragma unroll
  for (int j = 0; j < VEC; ++j) {
    x[j] = alpha * x[j];
    if (beta != 0.f) {
      const float cv = c_f16 ? (float)reinterpret_cast<const _Float16*>(c)[first + j]
                             : reinterpret_cast<const float*>(c)[first + j];
      x[j] = x[j] + beta * cv;
    }
  }
  if (bias) {
    const size_t at = first % (size_t)row_length;  // row_length is a multiple of 4: a vector never wraps
#pragma unroll
    for (int j = 0; j < VEC; ++j) x[j] += load_element(bias, bias_type, at + j);
  }
  if (VEC == 4) {
    if (d_type == kF32)
      *reinterpret_cast<float4*>(reinterpret_cast<float*>(d) + first) = float4{x[0], x[1 % VEC], x[2 % VEC], x[3 % VEC]};
    else
      *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(d) + first) =
          d_type == kF16 ? u32x2_t{round_pair<false>(x[0], x[1 % VEC]), round_pair<false>(x[2 % VEC], x[3 % VEC])}
                         : u32x2_t{round_pair<true>(x[0], x[1 % VEC]), round_pair<true>(x[2 % VEC], x[3 % VEC])};
  } else {
    if (d_type == kF32) reinterpret_cast<float*>(d)[first] = x[0];
    else reinterpret_cast<uint16_t*>(d)[first] = d_type == kF16 ? round_one<false>(x[0]) : round_one<true>(x[0]);
  }
}

// Second pass of a K split: ordered sum of the partial results and the epilogue (bias and row_length for the
// token-major form, where element i of y takes bias[i % m]).
hipError_t launch_split_reduce(const float* ws, int splits, size_t total, const void* c, void* d, float alpha,
                                      float beta, int c_f16, int d_type, const void* bias, int bias_type, int row_length,
                                      hipStream_t stream) {
  const bool vec = total % 4 == 0 && (reinterpret_cast<uintptr_t>(d) & 15) == 0 &&
                   (beta == 0.f || (reinterpret_cast<uintptr_t>(c) & 15) == 0) && (!bias || row_length % 4 == 0);
  if (vec)
    return launch_kernel(splitk_reduce_kernel<4>, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, stream, ws, splits, total, c, d,
                         total, alpha, beta, c_f16, d_type, bias, bias_type, row_length);
  return launch_kernel(splitk_reduce_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, ws, splits, total, c, d, total,
                       alpha, beta, c_f16, d_type, bias, bias_type, row_length);
}

static hipError_t launch_gemm_pass(GemmArgs args, int tile_config, hipStream_t stream) {
  const bool aligned = (args.ldb % 8 == 0) && ((reinterpret_cast<uintptr_t>(args.b) & 15) == 0);
  if (!aligned) {
    if (read_as_ragged(args.b, args.ldb)) {
      switch (tile_config) {  // tile_reads_ragged
        case kTile256x128w: return launch_gemm_cfg<2, 2, 4, 2, true, false, 1, false, false, true>(args, stream);
        case kTile128x128s: return launch_gemm_cfg<2, 2, 2, 2, true, false, 1, false, false, true>(args, stream);
        case kTile512x128w8: return launch_gemm_cfg<4, 2, 4, 2, true, false, 1, false, false, true>(args, stream);
        case kTile256x128w8: return launch_gemm_cfg<4, 2, 2, 2, true, false, 1, false, false, true>(args, stream);
        case kTile128x128w8: return launch_gemm_cfg<2, 4, 2, 1, true, false, 1, false, false, true>(args, stream);
        case kTile64x128: return launch_gemm_cfg<2, 2, 1, 2, true, false, 1, false, false, true>(args, stream);
        case kTile128x128k2: return launch_gemm_cfg<2, 2, 2, 2, true, false, 2, false, false, true>(args, stream);
        case kTile64x128k2: return launch_gemm_cfg<2, 2, 1, 2, true, false, 2, false, false, true>(args, stream);
        case kTile512x128m16: return launch_gemm_cfg<4, 1, 4, 4, true, false, 1, true, false, true>(args, stream);
        default: break;
      }
    }
    return launch_gemm_cfg<4, 1, 1, 4, false>(args, stream);
  }
  switch (tile_config) {
    case kTile512x128: return launch_gemm_cfg<4, 1, 4, 4, true>(args, stream);
    case kTile256x128: return launch_gemm_cfg<4, 1, 2, 4, true>(args, stream);
    case kTile128x128: return launch_gemm_cfg<4, 1, 1, 4, true>(args, stream);
    case kTile256x256: return launch_gemm_cfg<2, 2, 4, 4, true>(args, stream);
    case kTile256x128w: return launch_gemm_cfg<2, 2, 4, 2, true>(args, stream);
    case kTile512x128t: return launch_gemm_cfg<2, 2, 8, 2, true>(args, stream);
    case kTile128x128s: return launch_gemm_cfg<2, 2, 2, 2, true>(args, stream);
    case kTile256x64: return launch_gemm_cfg<2, 2, 4, 1, true>(args, stream);
    case kTile256x256w8: return launch_gemm_cfg<2, 4, 4, 2, true>(args, stream);
    case kTile512x128w8: return launch_gemm_cfg<4, 2, 4, 2, true>(args, stream);
    case kTile256x128w8: return launch_gemm_cfg<4, 2, 2, 2, true>(args, stream);
    case kTile128x128w8: return launch_gemm_cfg<2, 4, 2, 1, true>(args, stream);
    case kTile64x128: return launch_gemm_cfg<2, 2, 1, 2, true>(args, stream);
    case kTile128x128k2: return launch_gemm_cfg<2, 2, 2, 2, true, false, 2>(args, stream);
    case kTile64x128k2: return launch_gemm_cfg<2, 2, 1, 2, true, false, 2>(args, stream);
    case kTile512x128m16: return launch_gemm_cfg<4, 1, 4, 4, true, false, 1, true>(args, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_pad_b(const _Float16* b, _Float16* dst, int k, int n, hipStream_t stream) {
  const int per_row = (n + 7) / 8, rows = per_row > 1 && per_row < kPadPieces ? kPadPieces / per_row : 1;
  return launch_kernel(pad_b_kernel, dim3((k + rows - 1) / rows, (per_row + kPadPieces - 1) / kPadPieces), dim3(256), 0, stream, b, dst, k, n,
                       8 * per_row, rows, (uint32_t)((uint64_t(1) << 32) / per_row + 1));
}

hipError_t launch_gemm(GemmArgs args, int tile_config, hipStream_t stream) {
  if (prepared_bytes(args.m, args.k) >= (size_t(1) << 32)) return hipErrorInvalidValue;  // 32-bit copy offsets
  args.ldb = args.n;
  const bool aligned = (args.n % 8 == 0) && ((reinterpret_cast<uintptr_t>(args.b) & 15) == 0);
  if (!aligned && args.b_pad) {
    if (hipError_t st = launch_pad_b(args.b, args.b_pad, args.k, args.n, stream); st != hipSuccess) return st;
    args.b = args.b_pad;
    args.ldb = (args.n + 7) / 8 * 8;
  }
  const int chunks = (args.k + kChunkK - 1) / kChunkK;
  if (args.splits <= 1) {
    args.splits = 1;
    args.chunks_per_split = chunks;
    return launch_gemm_pass(args, tile_config, stream);
  }
  if (args.chunks_per_split < 1 || (long)(args.splits - 1) * args.chunks_per_split >= chunks || !args.split_ws)
    return hipErrorInvalidValue;  // an empty split would address past the prepared operand
  // pass 1: raw fp32 partial sums per split; pass 2: ordered sum and epilogue
  GemmArgs pass = args;
  pass.alpha = 1.f;
  pass.beta = 0.f;
  pass.c = nullptr;
  pass.d = args.split_ws;
  pass.d_f16 = 0;
  if (hipError_t st = launch_gemm_pass(pass, tile_config, stream); st != hipSuccess) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, args.c, args.d, args.alpha, args.beta,
                             args.c_f16, args.d_f16, nullptr, 0, 1, stream);
}

}  // namespace onebit
