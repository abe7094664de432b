// Token-major form of the split-K kernel (the linear layer, up to sixteen tokens), one product or several per launch.
#include "onebit_skinny.h"

namespace onebit {

template <int NW, int R, bool BF16>
static hipError_t launch_skinny_tokens_type(const SkinnyArgs& args, hipStream_t stream) {
  return launch_skinny_token_loads<NW, R, BF16>(args, stream);
}

template <int NW, int R>
static hipError_t launch_skinny_tokens_cfg(const SkinnyArgs& args, hipStream_t stream) {
  if (args.x_f32) {  // one token per load instruction, eight at once
    switch (args.n) {
      case 1: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 1, 16>(args, stream);
      case 2: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 2, 16>(args, stream);
      case 3: case 4: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 4, 16>(args, stream);
      case 5: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 5, 16>(args, stream);
      case 6: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 6, 16>(args, stream);
      case 7: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 7, 16>(args, stream);
      case 8: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 8, 16>(args, stream);
      case 9: case 10: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 10, 16>(args, stream);
      case 11: case 12: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 12, 16>(args, stream);
      case 13: case 14: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 14, 16>(args, stream);
      default: return launch_skinny_mode<NW, R, kSkinnyBTokens32 + 16, 16>(args, stream);
    }
  }
  return args.bf16 ? launch_skinny_tokens_type<NW, R, true>(args, stream) : launch_skinny_tokens_type<NW, R, false>(args, stream);
}

hipError_t launch_skinny_tokens(SkinnyArgs args, int rows_per_group, hipStream_t stream) {
  if (args.n < 1 || args.n > kSkinnyTokens) return hipErrorInvalidValue;
  // 16-byte loads of x; lane offsets of up to 64 token rows must stay below the "outside" offset of the kernel
  if ((reinterpret_cast<uintptr_t>(args.b) & 15) != 0 || (size_t)args.k * 64 * (args.x_f32 ? 4 : 2) >= 0xFFFFFF00u || (args.x_f32 && args.bf16))
    return hipErrorInvalidValue;
  SkinnyArgs pass;
  if (hipError_t st = skinny_split_setup(args, pass); st != hipSuccess) return st;
  hipError_t st;
  switch (rows_per_group) {
    case 32: st = launch_skinny_tokens_cfg<16, 1>(pass, stream); break;
    case 64: st = launch_skinny_tokens_cfg<8, 2>(pass, stream); break;
    case 128: st = launch_skinny_tokens_cfg<8, 4>(pass, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (st != hipSuccess || args.splits <= 1) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, nullptr, args.d, 1.f, 0.f, 0,
                             args.d_f16 && args.bf16 ? kBF16 : args.d_f16, args.bias, args.bias_type, args.m, stream);
}

template <int NW, int R, int MODE, bool BF16, int MOST>
static hipError_t launch_skinny_group_most(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  const dim3 grid(blocks), threads(64 * NW);
  const auto l = group_launch<MOST>(g);
  return launch_kernel(skinny_group_kernel<NW, R, MODE, BF16, MOST>, grid, threads, 0, stream, l.first[1], l.first[2], l.first[3], g.count,
                       g.problem[0].n, l.shared, l.table);
}
template <int NW, int R, int MODE, bool BF16>
static hipError_t launch_skinny_group_mode(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  return g.count <= kGroupFew ? launch_skinny_group_most<NW, R, MODE, BF16, kGroupFew>(g, blocks, stream)
                              : launch_skinny_group_most<NW, R, MODE, BF16, kSkinnyMaxGroup>(g, blocks, stream);
}

template <int NW, int R, bool BF16>
static hipError_t launch_skinny_group_type(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  switch (token_loads(g.problem[0].n)) {
    case 1: return launch_skinny_group_mode<NW, R, kSkinnyBTokens + 1, BF16>(g, blocks, stream);
    case 2: return launch_skinny_group_mode<NW, R, kSkinnyBTokens + 2, BF16>(g, blocks, stream);
    case 4: return launch_skinny_group_mode<NW, R, kSkinnyBTokens + 4, BF16>(g, blocks, stream);
    case 6: return launch_skinny_group_mode<NW, R, kSkinnyBTokens + 6, BF16>(g, blocks, stream);
    default: return launch_skinny_group_mode<NW, R, kSkinnyBTokens + 8, BF16>(g, blocks, stream);
  }
}

template <int NW, int R>
static hipError_t launch_skinny_group_cfg(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  return g.problem[0].bf16 ? launch_skinny_group_type<NW, R, true>(g, blocks, stream)
                           : launch_skinny_group_type<NW, R, false>(g, blocks, stream);
}

hipError_t launch_skinny_group(SkinnyGroupArgs g, int rows_per_group, hipStream_t stream) {
  if (g.count < 1 || g.count > kSkinnyMaxGroup) return hipErrorInvalidValue;
  const int tokens = g.problem[0].n;
  if (tokens < 1 || tokens > kSkinnyTokens) return hipErrorInvalidValue;
  if (rows_per_group != 32 && rows_per_group != 64 && rows_per_group != 128) return hipErrorInvalidValue;
  int blocks = 0;
  for (int i = 0; i < g.count; ++i) {
    SkinnyArgs& p = g.problem[i];
    if (p.n != tokens || !same_group_types(p, g.problem[0]) || p.m <= 0 || p.k <= 0 || !p.prep || !p.b || !p.d) return hipErrorInvalidValue;
    // 16-byte loads of x; lane offsets of up to 64 token rows must stay below the "outside" offset of the kernel
    if ((reinterpret_cast<uintptr_t>(p.b) & 15) != 0 || (size_t)p.k * 64 * 2 >= 0xFFFFFF00u) return hipErrorInvalidValue;
    p.splits = 1;
    p.chunks_per_split = p.kc_total;
    p.split_ws = nullptr;
    g.first_block[i] = blocks;
    blocks += (p.m + rows_per_group - 1) / rows_per_group;
  }
  g.first_block[g.count] = blocks;
  switch (rows_per_group) {
    case 32: return launch_skinny_group_cfg<16, 1>(g, blocks, stream);
    case 64: return launch_skinny_group_cfg<8, 2>(g, blocks, stream);
    default: return launch_skinny_group_cfg<8, 4>(g, blocks, stream);
  }
}

}  // namespace onebit
