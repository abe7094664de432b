// Plain form of the split-K kernel.
#include "onebit_skinny.h"

namespace onebit {

template <int NW, int R>
static hipError_t launch_skinny_cfg(const SkinnyArgs& args, hipStream_t stream) {
  const bool aligned = (reinterpret_cast<uintptr_t>(args.b) & 15) == 0;
  // Beyond sixteen columns what wide_kernel leaves: B that is not read in 16-byte pieces in place, some products of 32 columns,
  // and more rows than give its grid two workgroups per compute unit (65536 on the whole GPU, where the main kernel takes 33
  // columns or more; 8192 on a partition of 32 compute units).
  if (args.n > 32) {  // 64-column images, two column fragments: at most two row blocks fit the registers
    constexpr int R64 = R > 2 ? 2 : R;
    if (args.n == 64 && aligned) return launch_skinny_mode<NW, R64, kSkinnyBFull, 64>(args, stream);
    return launch_skinny_mode<NW, R64, kSkinnyBAny, 64>(args, stream);
  }
  if (args.n > 16) {  // 32-column images
    if (args.n == 32 && aligned) return launch_skinny_mode<NW, R, kSkinnyBFull, 32>(args, stream);
    return launch_skinny_mode<NW, R, kSkinnyBAny, 32>(args, stream);
  }
  if (args.n == 16 && aligned) return launch_skinny_mode<NW, R, kSkinnyBFull, 16>(args, stream);
  // one column: B is a token-major x of one token and D is its y (same memory in both layouts)
  if (args.n == 1 && aligned && (size_t)args.k * 64 * 2 < 0xFFFFFF00u)
    return launch_skinny_mode<NW, R, kSkinnyBTokens, 16>(args, stream);
  if ((args.n == 2 || args.n == 4) && aligned && (size_t)args.k * args.n * 2 < 0xFFFFFF00u)
    return launch_skinny_mode<NW, R, kSkinnyBRun, 16>(args, stream);
  return launch_skinny_mode<NW, R, kSkinnyBAny, 16>(args, stream);
}

hipError_t launch_skinny(SkinnyArgs args, int rows_per_group, hipStream_t stream) {
  if (args.n < 1 || args.n > kSkinnyMaxN) return hipErrorInvalidValue;
  SkinnyArgs pass;
  if (hipError_t st = skinny_split_setup(args, pass); st != hipSuccess) return st;
  hipError_t st;
  switch (rows_per_group) {
    case 32: st = launch_skinny_cfg<16, 1>(pass, stream); break;  // sixteen wavefronts split K: small M
    case 64: st = launch_skinny_cfg<8, 2>(pass, stream); break;
    case 128: st = launch_skinny_cfg<8, 4>(pass, stream); break;  // n > 32: 64-row groups
    default: return hipErrorInvalidValue;
  }
  if (st != hipSuccess || args.splits <= 1) return st;
  return launch_split_reduce(args.split_ws, args.splits, (size_t)args.m * args.n, args.c, args.d, args.alpha, args.beta,
                             args.c_f16, args.d_f16, nullptr, 0, 1, stream);
}

}  // namespace onebit
