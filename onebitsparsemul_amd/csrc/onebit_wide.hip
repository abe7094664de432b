// Plain form of wide_kernel.
#include "onebit_wide.h"

namespace onebit {

template <int R, bool RAGGED>
static hipError_t launch_wide_columns(const SkinnyArgs& args, hipStream_t stream) {
  switch ((args.tokens_per_group + 15) / 16) {
    case 1: return launch_wide_kernel<R, 2, false, false, RAGGED>(args, stream);
    case 2: return launch_wide_kernel<R, 4, false, false, RAGGED>(args, stream);
    case 3: return launch_wide_kernel<R, 6, false, false, RAGGED>(args, stream);
    case 4: return launch_wide_kernel<R, 8, false, false, RAGGED>(args, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_wide(SkinnyArgs args, int rows_per_group, hipStream_t stream) {
  const int columns = args.tokens_per_group;
  // 16-byte copies of B's rows, 32-bit offsets inside an image; rows of a ragged B where they lie, or of its padded copy
  const bool ragged = args.ldb % 8 != 0;
  if (args.n < 1 || columns < 1 || columns > kSkinnyMaxN || columns % 8 != 0 || rows_per_group < 1 || (ragged ? args.ldb != args.n || !read_as_ragged(args.b, args.n) : args.ldb != (args.n + 7) / 8 * 8 || (reinterpret_cast<uintptr_t>(args.b) & 15) != 0) || (size_t)args.ldb * 128 >= (size_t(1) << 32))
    return hipErrorInvalidValue;
  SkinnyArgs pass;
  if (hipError_t st = skinny_split_setup(args, pass); st != hipSuccess) return st;
  hipError_t st;
  switch (rows_per_group) {
    case 32: st = ragged ? launch_wide_columns<1, true>(pass, stream) : launch_wide_columns<1, false>(pass, stream); break;
    case 64: st = ragged ? launch_wide_columns<2, true>(pass, stream) : launch_wide_columns<2, false>(pass, stream); break;
    case 128: st = ragged ? launch_wide_columns<4, true>(pass, stream) : launch_wide_columns<4, false>(pass, stream); break;
    default: return hipErrorInvalidValue;
  }
  if (st != hipSuccess || args.splits <= 1) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, args.c, args.d, args.alpha, args.beta,
                             args.c_f16, args.d_f16, nullptr, 0, 1, stream);
}

}  // namespace onebit
