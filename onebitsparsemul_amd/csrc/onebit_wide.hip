// Plain form of wide_kernel.
#include "onebit_wide.h"

namespace onebit {

template <int R, int COPIES>
static hipError_t launch_wide_plain(const SkinnyArgs& args, dim3 grid, hipStream_t stream) {
  static std::atomic<bool> attr_done[64] = {};
  return launch_wide<R, COPIES>(wide_kernel<R, COPIES, false, false>, attr_done, args, grid, stream);
}

template <int R>
static hipError_t launch_wide_columns(const SkinnyArgs& args, dim3 grid, hipStream_t stream) {
  switch ((args.tokens_per_group + 15) / 16) {
    case 1: return launch_wide_plain<R, 2>(args, grid, stream);
    case 2: return launch_wide_plain<R, 4>(args, grid, stream);
    case 3: return launch_wide_plain<R, 6>(args, grid, stream);
    case 4: return launch_wide_plain<R, 8>(args, grid, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_wide(SkinnyArgs args, int rows_per_group, hipStream_t stream) {
  const int columns = args.tokens_per_group;
  // 16-byte copies of B's rows, 32-bit offsets inside an image
  if (args.n < 1 || columns < 1 || columns > kSkinnyMaxN || columns % 8 != 0 || rows_per_group < 1 || args.ldb < args.n ||
      args.ldb % 8 != 0 || (reinterpret_cast<uintptr_t>(args.b) & 15) != 0 || (size_t)args.ldb * 128 >= (size_t(1) << 32))
    return hipErrorInvalidValue;
  SkinnyArgs pass;
  if (hipError_t st = skinny_split_setup(args, pass); st != hipSuccess) return st;
  const dim3 grid((args.m + rows_per_group - 1) / rows_per_group, args.splits, (args.n + columns - 1) / columns);
  hipError_t st;
  switch (rows_per_group) {
    case 32: st = launch_wide_columns<1>(pass, grid, stream); break;
    case 64: st = launch_wide_columns<2>(pass, grid, stream); break;
    case 128: st = launch_wide_columns<4>(pass, grid, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (st != hipSuccess || args.splits <= 1) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, args.c, args.d, args.alpha, args.beta,
                             args.c_f16, args.d_f16, nullptr, 0, 1, stream);
}

}  // namespace onebit
