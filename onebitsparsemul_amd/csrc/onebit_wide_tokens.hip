// Token-major form of wide_kernel (the linear layer), one product or several per launch.
#include "onebit_wide.h"

namespace onebit {

// Several products that share the token count, workgroups numbered over their row groups as in skinny_group_kernel.
template <int R, int COPIES, bool BF16, bool PARTS, int MOST>
__global__ __launch_bounds__(64 * kWideWaves, 2) void wide_tokens_group_kernel(int first1, int first2, int first3, int count, int tokens,
                                                                               GroupShared shared, GroupTable<MOST> table) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  int block;
  const SkinnyArgs p = group_problem(first1, first2, first3, count, tokens, shared, table, block);
  wide_body<R, COPIES, true, BF16, PARTS, false>(p, block, 0, blockIdx.y * shared.tokens_per_group, smem);
}

template <int R, int COPIES, bool BF16>
static hipError_t launch_wide_one(const SkinnyArgs& args, int, hipStream_t stream) {
  return launch_wide_kernel<R, COPIES, true, BF16>(args, stream);
}
template <int R, int COPIES, bool BF16, bool PARTS, int MOST>
static hipError_t launch_wide_group(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  static std::atomic<bool> attr_done[64] = {};
  constexpr int lds = WideShape<R, COPIES>::LDS_BYTES;
  const auto kern = wide_tokens_group_kernel<R, COPIES, BF16, PARTS, MOST>;
  if (hipError_t st = wide_lds_limit(reinterpret_cast<const void*>(kern), lds, attr_done); st != hipSuccess) return st;
  const int n = g.problem[0].n, tokens = g.problem[0].tokens_per_group;
  const auto l = group_launch<MOST>(g);
  return launch_kernel(kern, dim3(blocks, (n + tokens - 1) / tokens), dim3(64 * kWideWaves), lds, stream, l.first[1], l.first[2], l.first[3],
                       g.count, n, l.shared, l.table);
}
template <int R, int COPIES, bool BF16>
static hipError_t launch_wide_one(const SkinnyGroupArgs& g, int blocks, hipStream_t stream) {
  bool parts = false;
  for (int i = 0; i < g.count; ++i) parts = parts || wide_has_parts(g.problem[i].kc_total);
  // us without a remainder, with parts | without: 8 x 2048 x 4096 with 17 tokens 7.56 | 7.30, 5 x 512 x 4096 with 48 5.17 | 4.97
  if (g.count > kGroupFew)
    return parts ? launch_wide_group<R, COPIES, BF16, true, kSkinnyMaxGroup>(g, blocks, stream)
                 : launch_wide_group<R, COPIES, BF16, false, kSkinnyMaxGroup>(g, blocks, stream);
  return parts ? launch_wide_group<R, COPIES, BF16, true, kGroupFew>(g, blocks, stream)
               : launch_wide_group<R, COPIES, BF16, false, kGroupFew>(g, blocks, stream);
}

// One instantiation per copy, not per pair of copies (a column tile of sixteen tokens): the eight tokens that an odd count leaves
// out need not be fetched (us with 24 | 32 tokens: 4096 x 11008 8.4 | 8.8, 11008 x 28672 26.8 | 28.8, 4096 x 8192 6.9 | 7.1).
template <int R, bool BF16, class Args>
static hipError_t launch_wide_copies(const Args& args, int tokens, int blocks, hipStream_t stream) {
  switch ((tokens + 7) / 8) {
    case 1: return launch_wide_one<R, 1, BF16>(args, blocks, stream);
    case 2: return launch_wide_one<R, 2, BF16>(args, blocks, stream);
    case 3: return launch_wide_one<R, 3, BF16>(args, blocks, stream);
    case 4: return launch_wide_one<R, 4, BF16>(args, blocks, stream);
    case 5: return launch_wide_one<R, 5, BF16>(args, blocks, stream);
    case 6: return launch_wide_one<R, 6, BF16>(args, blocks, stream);
    case 7: return launch_wide_one<R, 7, BF16>(args, blocks, stream);
    case 8: return launch_wide_one<R, 8, BF16>(args, blocks, stream);
    default: return hipErrorInvalidValue;
  }
}

template <class Args>
static hipError_t launch_wide_rows(const Args& args, int rows, int tokens, bool bf16, int blocks, hipStream_t stream) {
  switch (rows) {
    case 32: return bf16 ? launch_wide_copies<1, true>(args, tokens, blocks, stream) : launch_wide_copies<1, false>(args, tokens, blocks, stream);
    case 64: return bf16 ? launch_wide_copies<2, true>(args, tokens, blocks, stream) : launch_wide_copies<2, false>(args, tokens, blocks, stream);
    case 128: return bf16 ? launch_wide_copies<4, true>(args, tokens, blocks, stream) : launch_wide_copies<4, false>(args, tokens, blocks, stream);
    default: return hipErrorInvalidValue;
  }
}

// 16-byte copies of x; lane offsets inside 64 token rows of k values
static bool wide_operand_fits(const SkinnyArgs& p) {
  return (reinterpret_cast<uintptr_t>(p.b) & 15) == 0 && (size_t)p.k * kSkinnyMaxN * 2 < (size_t(1) << 32);
}

hipError_t launch_wide_tokens(SkinnyArgs args, int rows_per_group, hipStream_t stream) {
  const int tokens = args.tokens_per_group;
  if (args.n < 1 || tokens < 1 || tokens > kSkinnyMaxN || rows_per_group < 1 || !wide_operand_fits(args)) return hipErrorInvalidValue;
  SkinnyArgs pass;
  if (hipError_t st = skinny_split_setup(args, pass); st != hipSuccess) return st;
  const hipError_t st = launch_wide_rows(pass, rows_per_group, tokens, args.bf16, 0, stream);
  if (st != hipSuccess || args.splits <= 1) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, nullptr, args.d, 1.f, 0.f, 0,
                             args.d_f16 && args.bf16 ? kBF16 : args.d_f16, args.bias, args.bias_type, args.m, stream);
}

hipError_t launch_wide_tokens_group(SkinnyGroupArgs g, int rows_per_group, hipStream_t stream) {
  if (g.count < 1 || g.count > kSkinnyMaxGroup || rows_per_group < 1) return hipErrorInvalidValue;
  const int n = g.problem[0].n, tokens = g.problem[0].tokens_per_group;
  if (n < 1 || tokens < 1 || tokens > kSkinnyMaxN) return hipErrorInvalidValue;
  int blocks = 0;
  for (int i = 0; i < g.count; ++i) {
    SkinnyArgs& p = g.problem[i];
    if (p.n != n || p.tokens_per_group != tokens || !same_group_types(p, g.problem[0]) || p.m <= 0 || p.k <= 0 || !p.prep || !p.b || !p.d ||
        !wide_operand_fits(p))
      return hipErrorInvalidValue;
    p.splits = 1;
    p.chunks_per_split = p.kc_total;
    p.split_ws = nullptr;
    g.first_block[i] = blocks;
    blocks += (p.m + rows_per_group - 1) / rows_per_group;
  }
  g.first_block[g.count] = blocks;
  return launch_wide_rows(g, rows_per_group, tokens, g.problem[0].bf16, blocks, stream);
}

}  // namespace onebit
