// Token-major form of the main kernel (the linear layer).
#include "onebit_gemm.h"

namespace onebit {

template <bool BF16>
static hipError_t launch_tokens_tile(const GemmArgs& a, int tile_config, hipStream_t stream) {
  switch (tile_config) {
    case kTile256x128w: return launch_gemm_cfg<2, 2, 4, 2, true, true, 1, false, BF16>(a, stream);
    case kTile128x128s: return launch_gemm_cfg<2, 2, 2, 2, true, true, 1, false, BF16>(a, stream);
    case kTile512x128w8: return launch_gemm_cfg<4, 2, 4, 2, true, true, 1, false, BF16>(a, stream);
    case kTile256x128w8: return launch_gemm_cfg<4, 2, 2, 2, true, true, 1, false, BF16>(a, stream);
    case kTile128x128w8: return launch_gemm_cfg<2, 4, 2, 1, true, true, 1, false, BF16>(a, stream);
    case kTile64x128: return launch_gemm_cfg<2, 2, 1, 2, true, true, 1, false, BF16>(a, stream);
    case kTile128x128k2: return launch_gemm_cfg<2, 2, 2, 2, true, true, 2, false, BF16>(a, stream);
    case kTile64x128k2: return launch_gemm_cfg<2, 2, 1, 2, true, true, 2, false, BF16>(a, stream);
    case kTile512x128m16: return launch_gemm_cfg<4, 1, 4, 4, true, true, 1, true, BF16>(a, stream);
    default: return hipErrorInvalidValue;  // the tiles the automatic choice uses
  }
}

hipError_t launch_gemm_tokens(GemmArgs args, int tile_config, hipStream_t stream) {
  if (prepared_bytes(args.m, args.k) >= (size_t(1) << 32)) return hipErrorInvalidValue;  // 32-bit copy offsets
  if ((reinterpret_cast<uintptr_t>(args.b) & 15) != 0 || (size_t)args.k * 256 * 2 >= (size_t(1) << 32))
    return hipErrorInvalidValue;  // 16-byte copies of x; 32-bit offsets inside a tile's token rows
  const int chunks = (args.k + kChunkK - 1) / kChunkK;
  args.ldb = args.k;
  args.alpha = 1.f;
  args.beta = 0.f;
  args.c = nullptr;
  auto pass = [&](GemmArgs a) {
    return a.bf16 ? launch_tokens_tile<true>(a, tile_config, stream) : launch_tokens_tile<false>(a, tile_config, stream);
  };
  if (args.splits <= 1) {
    args.splits = 1;
    args.chunks_per_split = chunks;
    return pass(args);
  }
  if (args.chunks_per_split < 1 || (long)(args.splits - 1) * args.chunks_per_split >= chunks || !args.split_ws)
    return hipErrorInvalidValue;  // an empty split would address past the prepared operand
  // pass 1: raw fp32 partial sums per split, token-major like y; pass 2: ordered sum and bias
  GemmArgs first = args;
  first.d = args.split_ws;
  first.d_f16 = 0;
  first.bias = nullptr;
  if (hipError_t st = pass(first); st != hipSuccess) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, nullptr, args.d, 1.f, 0.f, 0,
                             args.d_f16 && args.bf16 ? kBF16 : args.d_f16, args.bias, args.bias_type, args.m, stream);
}

}  // namespace onebit
