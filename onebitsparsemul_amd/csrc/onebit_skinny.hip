// Plain form of the split-K kernel.
#include "onebit_skinny.h"

namespace onebit {

template <int NW, int R>
static hipError_t launch_skinny_cfg(const SkinnyArgs& args, hipStream_t stream) {
  const bool aligned = (reinterpret_cast<uintptr_t>(args.b) & 15) == 0;
  // Beyond sixteen columns what wide_kernel leaves: B at an unaligned base, an odd n on few rows, some products of 32 columns,
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
  if (args.n == 1 && aligned && (size_t)args.k * 64 * 2 < 0xFFFFFF00u) return launch_skinny_mode<NW, R, kSkinnyBTokens + 1, 16>(args, stream);
  // Two to eight columns by fours of K positions (us inside HIP graphs, weights from HBM; before: two and four columns as one run of
  // pieces spread by element stores, the others as pieces at any alignment, of which those of odd rows cost 3.8 times the load path |
  // now): 4096 x 11008 with 2 / 3 / 4 / 5 / 6 / 7 / 8 9.1 | 5.1, 8.4 | 5.2, 6.9 | 5.3, 8.4 | 5.7, 6.9 | 5.7, 8.4 | 5.9, 6.7 | 6.4; 11008 x
  // 4096 with 2 / 5 / 8 6.2 | 4.9, 6.6 | 5.1, 5.7 | 5.4; 28672 x 8192 13.9 | 11.1, 14.6 | 12.4, 13.0 | 12.8; 512 x 512 with 3 2.94 | 2.36.
  // Eight columns are whole pieces at 16-byte boundaries, and as those faster where there are few chunks (2048 x 5120 3.98 | 4.24, 20480 x
  // 2048 5.41 | 5.66).
  const bool eight_as_pieces = R != 2 && args.chunks_per_split < (NW == 16 ? 32 : 16);
  if (aligned && (size_t)args.k * args.n * 2 < 0xFFFFFF00u)
    switch (args.n) {
      case 2: return launch_skinny_mode<NW, R, kSkinnyBColumns + 2, 16>(args, stream);
      case 3: return launch_skinny_mode<NW, R, kSkinnyBColumns + 3, 16>(args, stream);
      case 4: return launch_skinny_mode<NW, R, kSkinnyBColumns + 4, 16>(args, stream);
      case 5: return launch_skinny_mode<NW, R, kSkinnyBColumns + 5, 16>(args, stream);
      case 6: return launch_skinny_mode<NW, R, kSkinnyBColumns + 6, 16>(args, stream);
      case 7: return launch_skinny_mode<NW, R, kSkinnyBColumns + 7, 16>(args, stream);
      case 8: if (eight_as_pieces) break; else return launch_skinny_mode<NW, R, kSkinnyBColumns + 8, 16>(args, stream);
      default: break;
    }
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
