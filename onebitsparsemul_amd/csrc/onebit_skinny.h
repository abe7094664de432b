// The split-K kernel for N <= 64 (decode shapes) on gfx950, plain and token-major (see onebit_gemm.h), and the launch of one
// instantiation. onebit_skinny.hip and onebit_skinny_tokens.hip instantiate it.
#pragma once
#include "onebit_device.h"
#include "onebit_launch.h"
#include <climits>
#include <type_traits>

namespace onebit {

// =====================================================================================================
// skinny_kernel: N <= 64 (decode shapes). HBM-bound: every byte of the prepared operand is read once.
// Workgroup = NW wavefronts that share R row blocks (32 rows each) and split K among themselves: wavefront w
// takes the K chunks (of 256) w, w + NW, w + 2 NW, ... Each wavefront stages B rows in a private 8 KiB LDS region
// as a zero-padded fp16 image of NC columns (NC = 16: the 256 rows of a chunk; NC = 32: 128 rows, two images per
// chunk; NC = 64: 64 rows, four images, two column fragments), feeds them to SMFMAC through transpose reads (one fragment serves the R row blocks) and keeps a 32x32
// fp32 partial tile per row block (NC = 16: two 16x16 tiles, multiplied with v_smfmac_f32_16x16x64_f16, which has no
// idle columns at sixteen). The prepared operand and the next image are loaded into registers while the
// current one is multiplied. Wavefronts never wait for one another inside the K loop (LDS operations of one
// wavefront execute in order). The NW partial tiles of a row block are added through LDS in wavefront order
// (deterministic; the tiles take the place of the images, as many row blocks per round as fit the 8 KiB) and the
// epilogue is applied. grid = M / (32 R) workgroups; no global workspace, no atomics.
// =====================================================================================================
constexpr int kSkinnyRegion = 8192;  // bytes of one B image

// How B rows reach the image. kSkinnyBFull: n == NC, 16-byte aligned, whole images are consecutive memory. kSkinnyBAny: any
// n, any alignment: 16-byte pieces, ceil(n / 8) per row, loaded from wherever the row starts (gfx950 loads 16 bytes at any
// address). A piece that reaches past its row's end takes the next row's first elements along; they land in columns at or
// past n, whose results are never stored, so nothing has to be cleared or masked. It replaced element copies and two modes
// of checked pieces (us inside a HIP graph): 14016 x 14 x 7136 43.2 -> 9.2, 11008 x 15 x 4096 23.1 -> 8.5, 4096 x 33 x 4096
// 27.8 -> 12.1, 11008 x 63 x 4096 51.1 -> 14.5; n % 8 == 0: 11008 x 8 x 4096 5.8 -> 5.2, 28672 x 40 x 8192 40.8 -> 32.6.
// kSkinnyBTokens: the token-major form of the linear layer. B is x, n rows (tokens) of k consecutive values, and
// the result is written as y[token][weight row] (+ bias[weight row]). The image is then token-major too: row t holds
// the image's K range of token t in 16-byte pieces, piece p stored at position p ^ token_swizzle(t) so that lanes
// which read the same piece of consecutive tokens fall into different banks; a lane's SMFMAC operand is two plain
// 16-byte reads (K consecutive inside a piece), no transpose. Up to sixteen tokens; more go to wide_kernel.
// kSkinnyBTokens + l: l load instructions take an image, two tokens each. How many is known to the compiler, and none is in a branch,
// because its waits for an earlier load count only what is requested behind it on every path.
// kSkinnyBColumns + n: n = 2 ... 8 columns, B 16-byte aligned. Four rows of B are 8 n consecutive bytes that begin at a multiple of
// eight: each lane loads those of four K positions, n / 2 instructions per chunk, and stores them as n columns of four K values into
// an image that is token-major, read as such; the tiles' reduction turns them back.
// kSkinnyBTokens32: the token-major form on fp32 activations, rounded to fp16 (nearest even) on their way into the image. One load
// instruction takes a token's 256 K, whole lines, so there are as many as tokens. A conversion in front of the kernel costs a
// launch and an allocation (us per layer call, conversion in front -> here: 4096 x 4096 with 1 / 16 tokens 9.2 / 9.0 -> 4.8 / 4.9,
// 28672 x 8192 with 8 / 16 14.0 / 15.5 -> 11.8 / 14.8, 4096 x 11008 with 16 9.0 -> 8.7).
// kSkinnyBTokens32 + l: l load instructions take an image, the ninth and later ones in a second batch. No more than one past the last
// token: a surplus one costs its place in the load path (us inside HIP graphs, weights from HBM, each load in a branch of its own | eight
// and eight for nine tokens and more | this: 8192 x 8192 with 9 / 13 tokens 7.5 | 8.8 | 7.3, 8.4 | 9.0 | 8.5, 4096 x 11008 with 9 8.3 |
// 9.4 | 7.6, 4096 x 4096 with 9 / 16 5.0 | 5.4 | 4.5, 5.8 | 5.7 | 5.4, 28672 x 8192 with 10 15.5 | 16.0 | 14.4).
enum SkinnyBMode { kSkinnyBFull = 0, kSkinnyBAny = 1, kSkinnyBColumns = 16, kSkinnyBTokens = 32, kSkinnyBTokens32 = 48 };

// The body of the split-K kernel for workgroup (block_x, block_y) of problem p: block_x = row group, block_y = K split.
template <int NW, int R, int MODE, int NC, bool BF16 = false>
__device__ __forceinline__ void skinny_body(const SkinnyArgs& p, const int block_x, const int block_y) {
  constexpr int NT = 64 * NW;
  constexpr int IMG_ROWS = kSkinnyRegion / (NC * 2);   // B rows per image: 256, 128 or 64
  constexpr int SUB = kChunkK / IMG_ROWS;              // images per chunk: 1, 2 or 4
  constexpr int IMG_STEPS = kStepsPerChunk / SUB;      // 32-wide K steps per image: 8, 4 or 2
  constexpr int ROW_BYTES = NC * 2;
  constexpr int NF = NC <= 32 ? 1 : NC / 32;           // 32-column fragments per image row
  constexpr int TILE_BYTES = kRowBlock * NC * 4;       // one fp32 partial tile
  static_assert(NC == 16 || NC == 32 || NC == 64, "image width");
  static_assert(MODE == kSkinnyBFull || MODE == kSkinnyBAny || NC == 16, "the column and token modes are for 16 columns");
  // the partial tiles reuse the wavefront's image memory, RT row blocks per round of the final reduction
  constexpr int RT = R * TILE_BYTES <= kSkinnyRegion ? R : kSkinnyRegion / TILE_BYTES;
  static_assert(RT >= 1 && R % RT == 0, "the row blocks must divide into whole reduction rounds");
  constexpr bool X32 = MODE > kSkinnyBTokens32, TOKENS = MODE > kSkinnyBTokens;
  constexpr int COLUMNS = MODE > kSkinnyBColumns && !TOKENS ? MODE - kSkinnyBColumns : 0;
  static_assert(COLUMNS <= 8, "two to eight columns");
  constexpr bool TOKEN_IMAGE = TOKENS || COLUMNS > 0;
  static_assert(!X32 || !BF16, "fp32 activations are multiplied as fp16");
  // Sixteen columns fill half of the 32x32x32 SMFMAC's result tile; v_smfmac_f32_16x16x64_f16 has no idle half and
  // multiplies a row block's chunk in half the matrix-pipe time (eight instructions of four passes).
  constexpr bool M16 = NC == 16;
  constexpr int PPT = IMG_ROWS / 8;                    // token-major image: 16-byte pieces per token row
  constexpr int TPI = 64 / PPT;                        // ... and tokens covered by the 64 pieces of one wavefront load
  constexpr int TOKEN_ROW_BYTES = IMG_ROWS * 2;
  constexpr int LOADS32 = X32 ? MODE - kSkinnyBTokens32 : 0, SECOND_LOADS = LOADS32 > 8 ? LOADS32 - 8 : 0;
  constexpr int TOKEN_LOADS = X32 ? LOADS32 - SECOND_LOADS : TOKENS ? MODE - kSkinnyBTokens : 8;
  __shared__ __attribute__((aligned(16))) char bs[NW * kSkinnyRegion];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rb_total = p.m / kRowBlock;
  const int rb_first = block_x * R;
  char* region = bs + wave * kSkinnyRegion;
  // kernel arguments the lambdas use, as values (capturing the argument struct would move it to scratch memory)
  const _Float16* __restrict__ b_ptr = p.b;
  const uint8_t* __restrict__ prep = p.prep;
  const int n_cols = p.n, k_rows = p.k, kc_total = p.kc_total;

  // The streaming loads go through buffer descriptors: wave-uniform base and offset in scalar registers, lane
  // offsets in one vector register, no vector address arithmetic inside the K loop. One descriptor per row block
  // (its kc_total blocks are consecutive, under 4 GiB for any K the argument checks admit) and one for B.
  const uint32_t meta_off = (uint32_t)lane * 16u, sign_off = (uint32_t)kSignOffset + (uint32_t)lane * 8u;
  buffer_t a_buffer[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int rb = rb_first + r;
    if (rb >= rb_total) rb = rb_total - 1;  // never stored
    a_buffer[r] = make_buffer(prep + (size_t)rb * kc_total * kBlockBytes, (uint32_t)kc_total * kBlockBytes);
  }
  auto load_a = [&](int kc, AChunk (&a)[R]) __attribute__((always_inline)) {
    if (kc >= kc_total) kc = kc_total - 1;  // never multiplied
    const uint32_t block = (uint32_t)kc * kBlockBytes;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      a[r].meta = buffer_load16(a_buffer[r], meta_off, block);
      a[r].sign = buffer_load8(a_buffer[r], sign_off, block);
    }
  };
  // K split over workgroups (grid.y > 1): this workgroup multiplies the chunks [kc_begin, kc_end) and writes raw fp32
  // sums to its slice of the partial-sum buffer; a second kernel adds the slices in order and applies the epilogue.
  const int kc_begin = block_y * p.chunks_per_split;
  const int kc_end = kc_begin + p.chunks_per_split < kc_total ? kc_begin + p.chunks_per_split : kc_total;
  const int first = kc_begin + wave;  // this wavefront's first chunk
  // Short K (at most two chunks per wavefront, e.g. 11008 x 4096): everything the wavefront will read is requested
  // at once, so the kernel pays one memory latency instead of one per chunk.
  constexpr bool kShortPath = NW <= 8 && SUB == 1;
  const bool short_k = kShortPath && kc_end - kc_begin <= 2 * NW;
  // The prepared operand comes from HBM and is what the first SMFMAC waits for longest: the loop form issues its first
  // loads here, before the rest of the set-up (B descriptor, image offsets, fragment addresses), which then runs under
  // their latency (4096 x 4096 x 16: 4.87 -> 4.70 us). The short form keeps B first: loads return in order, and a B image
  // requested behind the weights would reach LDS only after them (11008 x 4096 x 1: 5.6 -> 6.3 us when tried).
  AChunk a_cur[R], a_next[R];
  if (!short_k) {
    load_a(first, a_cur);
    __builtin_amdgcn_sched_barrier(0);
  }
  const size_t b_bytes = (size_t)k_rows * n_cols * (X32 ? 4 : 2);
  const bool b_fits = b_bytes < (size_t(1) << 32);  // else every image takes the general path
  const buffer_t b_buffer = make_buffer(b_ptr, b_fits ? (uint32_t)b_bytes : 0u);
  auto rows_valid_of = [&](int k_base) __attribute__((always_inline)) {
    const int rows = k_rows - k_base;
    return rows < 0 ? 0 : (rows > IMG_ROWS ? IMG_ROWS : rows);
  };
  // pieces at any alignment: a load instruction covers any_rows whole rows, lane = (row, piece) of them
  // (sixteen-column images: one or two pieces, without the divisions, which cost a short K 0.15 us)
  const int any_pieces = (n_cols + 7) / 8, any_rows = NC == 16 ? 64 >> (any_pieces - 1) : 64 / any_pieces;
  const int any_row = NC == 16 ? lane >> (any_pieces - 1) : lane / any_pieces;
  const int any_piece = NC == 16 ? lane & (any_pieces - 1) : lane % any_pieces;
  const bool any_used = any_row < any_rows;
  const uint32_t any_load = (uint32_t)(any_row * n_cols + 8 * any_piece) * 2u, any_load_step = (uint32_t)(any_rows * n_cols) * 2u;
  const uint32_t any_store = (uint32_t)any_row * ROW_BYTES + 16u * any_piece;
  // Image t of this wavefront = B rows [k_base, k_base + IMG_ROWS) with k_base = (wave + NW (t / SUB)) * 256 +
  // (t % SUB) * IMG_ROWS. The image travels through registers, loaded while the previous image is multiplied.
  // token-major image: piece lane + 64 i = K values [8 p, 8 p + 8) of the image for token token_lane + TPI i
  const int piece_lane = lane % PPT, token_lane = lane / PPT;
  const uint32_t token_load_base = ((uint32_t)token_lane * (uint32_t)k_rows + 8u * piece_lane) * 2u;
  const uint32_t token_load_step = (uint32_t)TPI * (uint32_t)k_rows * 2u;
  const uint32_t token_store_base =
      (uint32_t)token_lane * TOKEN_ROW_BYTES + (uint32_t)((piece_lane ^ token_swizzle<TOKEN_ROW_BYTES>(token_lane)) << 4);
  // fp32 activations, up to eight tokens from first_token on. Load i: the image's K range of one token, four values per lane; K positions
  // at or past k: outside the descriptor, as below (the launcher checks that 64 * k * 4 stays well below 2^32). Tokens 8 to 15
  // are requested when the first eight have been stored: 64 registers of loads in flight do not fit beside the rest.
  auto load_b32 = [&](int k_base, int first_token, auto loads_tag, u32x4_t (&v)[8]) __attribute__((always_inline)) {
    const bool whole = k_base + IMG_ROWS <= k_rows;  // wave-uniform
    const bool inside = k_base + 4 * lane < k_rows;
#pragma unroll
    for (int i = 0; i < decltype(loads_tag)::value; ++i) {
      const uint32_t offset = meta_off + (uint32_t)(first_token + i) * (uint32_t)k_rows * 4u;
      // Sixteen wavefronts with six loads or more at a time: one per sixteen clocks, as many as the load path takes. All at once they
      // keep out the other wavefronts' (8192 x 8192 with 6 / 8 tokens 6.08 / 6.50 us with a branch around each, 6.32 / 6.77 at once, 5.98 /
      // 6.40 so; 2048 x 8192 with 8 5.63, 5.70, 5.42; one per 48 clocks 6.02)
      if (NW == 16 && LOADS32 >= 6 && LOADS32 <= 8 && i > 0) asm volatile("s_nop 15" ::: "memory");
      // tokens past the last: outside the descriptor, as in load_b
      v[i] = buffer_load16(b_buffer, whole ? offset : inside ? offset + (uint32_t)k_base * 4u : 0xFFFFFF00u, whole ? (uint32_t)k_base * 4u : 0u);
    }
  };
  auto store_b32 = [&](int first_token, auto loads_tag, const u32x4_t (&v)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < decltype(loads_tag)::value; ++i) {
      const float4v_t f = __builtin_bit_cast(float4v_t, v[i]);
      const int token = first_token + i;
      *reinterpret_cast<u32x2_t*>(region + token * TOKEN_ROW_BYTES + (((lane >> 1) ^ token_swizzle<TOKEN_ROW_BYTES>(token)) << 4) +
                                  (lane & 1) * 8) = u32x2_t{round_pair<false>(f[0], f[1]), round_pair<false>(f[2], f[3])};
    }
  };
  auto load_b = [&](int k_base, u32x4_t (&v)[8], bool spaced = false) __attribute__((always_inline)) {
    if constexpr (COLUMNS > 0) {
      // four K positions of a lane: all of them inside K or none (k % 32 == 0); those past its end are sent outside the
      // descriptor, which reads zeros (the launcher checks k n 2 < 2^32)
      const uint32_t image = (uint32_t)k_base * (COLUMNS * 2), at = (uint32_t)lane * (COLUMNS * 8);
      const bool whole = k_base + IMG_ROWS <= k_rows;  // wave-uniform
      const uint32_t lane_at = whole ? at : k_base + 4 * lane < k_rows ? at + image : 0xFFFFFF00u, image_at = whole ? image : 0u;
#pragma unroll
      for (int i = 0; i < COLUMNS / 2; ++i) v[i] = buffer_load16(b_buffer, lane_at + 16u * i, image_at);
      if constexpr (COLUMNS % 2 != 0) {
        const u32x2_t rest = buffer_load8(b_buffer, lane_at + 8u * (COLUMNS - 1), image_at);
        v[COLUMNS / 2].x = rest.x; v[COLUMNS / 2].y = rest.y;
      }
      return;
    }
    if (X32) {
      load_b32(k_base, 0, std::integral_constant<int, TOKEN_LOADS>{}, v);
      return;
    }
    if (TOKENS) {
      // offsets at or past n * k * 2 (tokens >= n) fall outside the descriptor and read as zero; K positions at or past k are sent
      // there too (the launcher checks that 64 * k * 2 stays well below 2^32). Where the image's whole K range exists, the lane
      // offsets do not change from image to image and a scalar offset is added, which the range check does not look at.
      const bool whole = k_base + IMG_ROWS <= k_rows;  // wave-uniform
      const bool inside = k_base + 8 * piece_lane < k_rows;
      const uint32_t lane_at = whole ? token_load_base : token_load_base + (uint32_t)k_base * 2u, image_at = whole ? (uint32_t)k_base * 2u : 0u;
#pragma unroll
      for (int i = 0; i < TOKEN_LOADS; ++i) {
        if (spaced && i > 0) asm volatile("s_nop 15" ::: "memory");
        v[i] = buffer_load16(b_buffer, whole || inside ? lane_at + i * token_load_step : 0xFFFFFF00u, image_at);
      }
      return;
    }
    if (MODE == kSkinnyBFull) {
      if (b_fits && k_base + IMG_ROWS <= k_rows) {
        // the whole image lies inside B (wave-uniform test): 8 KiB of consecutive memory, no per-piece checks
        const uint32_t image = (uint32_t)k_base * (NC * 2);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = buffer_load16(b_buffer, meta_off + 1024u * i, image);
        return;
      }
      const int rows_valid = rows_valid_of(k_base);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int q = lane + i * 64;
        const bool ok = q / (NC / 8) < rows_valid;
        v[i] = *reinterpret_cast<const u32x4_t*>(b_ptr + (ok ? (size_t)k_base * NC + (size_t)q * 8 : 0));
        if (!ok) v[i] = u32x4_t{0, 0, 0, 0};
      }
      return;
    }
    // (wave-uniform) rows from the image's first on, as far as they matter: none past the end of K
    const int rows_left = k_rows - k_base < IMG_ROWS + 8 ? k_rows - k_base : IMG_ROWS + 8;
    if (rows_left <= 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = u32x4_t{0, 0, 0, 0};
      return;
    }
    // lane offsets that do not change from image to image; lanes without a piece and pieces that would end past the rows
    // left (the last image's, k % 32 == 0: at least 32 rows) load the last whole piece instead
    const char* image = reinterpret_cast<const char*>(b_ptr + (size_t)k_base * n_cols);
    const uint32_t last = (uint32_t)(rows_left * n_cols - 8) * 2u;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i * any_rows < IMG_ROWS) {
        const uint32_t offset = any_load + i * any_load_step;
        v[i] = *reinterpret_cast<const u32x4_any_t*>(image + (offset < last ? offset : last));
      }
    // whole pieces: every piece of a row that exists ends inside it. Asked with sixteen wavefronts and sixteen-column images
    // only: a test at run time makes the others slower (us, with and without it: 19456 x 20 x 8672 24.9 | 19.6, 896 x 30 x 9152
    // 10.6 | 9.1; eight columns on 64-row groups 8 % in the median of long K)
    const bool whole_pieces = NC == 16 && NW == 16 && n_cols % 8 == 0;
    if (rows_left < IMG_ROWS + (whole_pieces ? 0 : 8)) {
      // last image: what was read from the last whole piece is shifted into place, rows at or past K are zeros
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i * any_rows < IMG_ROWS) {
          const uint32_t offset = any_load + i * any_load_step;
          if (offset > last) v[i] = whole_pieces ? u32x4_t{0, 0, 0, 0} : drop_halves(v[i], (int)(offset - last) / 2);
        }
    }
  };
  auto store_b = [&](int k_base, const u32x4_t (&v)[8]) __attribute__((always_inline)) {
    if (X32) {
      store_b32(0, std::integral_constant<int, TOKEN_LOADS>{}, v);
      if constexpr (SECOND_LOADS > 0) {
        u32x4_t w[8];
        load_b32(k_base, 8, std::integral_constant<int, SECOND_LOADS>{}, w);
        store_b32(8, std::integral_constant<int, SECOND_LOADS>{}, w);
      }
      return;
    }
    if (MODE == kSkinnyBAny) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i * any_rows < IMG_ROWS && any_used && any_row + i * any_rows < IMG_ROWS)
          *reinterpret_cast<u32x4_t*>(region + any_store + i * any_rows * ROW_BYTES) = v[i];
      return;
    }
    if constexpr (COLUMNS > 0) {
      auto value = [&](int row, int col) __attribute__((always_inline)) { return row * COLUMNS + col; };
      auto pair = [&](int low, int high) __attribute__((always_inline)) {  // halves `low` and `high` of the lane's 4 n as one word
        const uint32_t from_low = low & 1 ? 0x0302u : 0x0100u, from_high = high & 1 ? 0x07060000u : 0x05040000u;
        return __builtin_amdgcn_perm(v[high / 8][high / 2 % 4], v[low / 8][low / 2 % 4], from_low | from_high);
      };
#pragma unroll
      for (int c = 0; c < COLUMNS; ++c)
        *reinterpret_cast<u32x2_t*>(region + c * TOKEN_ROW_BYTES + (((lane >> 1) ^ token_swizzle<TOKEN_ROW_BYTES>(c)) << 4) + (lane & 1) * 8) =
            u32x2_t{pair(value(0, c), value(1, c)), pair(value(2, c), value(3, c))};
      return;
    }
    if (TOKENS) {
      // token = token_lane + TPI i with token_lane < TPI (a power of two): the two terms share no bits, so the swizzle of
      // piece i differs from that of piece 0 by a compile-time XOR
#pragma unroll
      for (int i = 0; i < TOKEN_LOADS; ++i)
        *reinterpret_cast<u32x4_t*>(region + (token_store_base ^ (uint32_t)(token_swizzle<TOKEN_ROW_BYTES>(TPI * i) << 4)) + i * 1024) = v[i];
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) *reinterpret_cast<u32x4_t*>(region + (lane + i * 64) * 16) = v[i];
  };

  float16_t acc[R][NF];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[r][f][v] = 0.f;
  float4v_t acc16[R][2];  // M16: rows 0-15 and 16-31 of the row block; register v of lane l = row 4 (l / 16) + v, column l % 16
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int h = 0; h < 2; ++h) acc16[r][h] = float4v_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t one = packed_one_in_vgpr<BF16>();
  const int i16 = lane & 15, gb = lane >> 5, g16 = lane >> 4;
  // (32x32x32 form, NC >= 32; sixteen-column images use the 16x16x64 form further down)
  const int chunk8 = (NC >= 32 ? ((lane & 31) >> 4) * 4 : 0) + (i16 & 3);  // 8-byte piece of the 32-column fragment
  const char* lane_ptr = region + (8 * gb + (i16 >> 2)) * ROW_BYTES + chunk8 * 8;

  // ---- 16x16x64 form (M16). The instruction's A lane (row l % 16, group g = l / 16) holds eight kept values and their
  // 16 index bits for 16 consecutive K positions, as a lane of the prepared block does for one K step: lane
  // (row, half ga) of the block, step s. Which K positions group g stands for is free as long as B agrees, so the
  // operands are built with one v_permlane16_swap per register pair instead of a gather: swapping the odd 16-lane
  // rows of metadata register 2 P with the even rows of register 2 P + 1 leaves in the first register, for
  // block rows 0-15, the groups (ga 0, steps 4 P + {0, 1}), (ga 0, steps 4 P + {2, 3}), (ga 1, steps 4 P + {0, 1}),
  // (ga 1, steps 4 P + {2, 3}) and in the second register the same for block rows 16-31; ABID picks the even or the
  // odd step of each pair. Instruction (P, abid) therefore covers K positions 128 P + 32 abid + [0, 32) and
  // 128 P + 32 abid + 64 + [0, 32) of the chunk: group g positions 128 P + 32 abid + 64 (g % 2) + 16 (g / 2) + [0, 16).
  // The sign words travel the same way (a register swapped with its own copy) and are shifted by 8 (g % 2) once, after
  // which the expansion uses compile-time shifts. B lane (column l % 16, group gb) holds instruction K rows
  // 8 gb + [0, 8) and 32 + 8 gb + [0, 8), i.e. chunk rows base + [0, 8) and base + 16 + [0, 8) with
  // base = 128 P + 32 abid + 64 (gb / 2) + 8 (gb % 2).
  struct A16 {
    uint32_t idx[2][2];   // [row half][P]
    uint32_t sign[2][2];
  };
  const uint32_t sign_shift16 = 8u * (g16 & 1);
  auto gather16 = [&](const AChunk& a) __attribute__((always_inline)) {
    A16 t;
#pragma unroll
    for (int P = 0; P < 2; ++P) {
      const auto m = __builtin_amdgcn_permlane16_swap(a.meta[2 * P], a.meta[2 * P + 1], false, false);
      const uint32_t w = P == 0 ? a.sign.x : a.sign.y;
      const auto sg = __builtin_amdgcn_permlane16_swap(w, w, false, false);
      t.idx[0][P] = m[0];
      t.idx[1][P] = m[1];
      t.sign[0][P] = sg[0] << sign_shift16;
      t.sign[1][P] = sg[1] << sign_shift16;
    }
    return t;
  };
  const char* lane_ptr16 = region + (64 * (g16 >> 1) + 8 * (g16 & 1) + (i16 >> 2)) * ROW_BYTES + (i16 & 3) * 8;
  const uint32_t token_read_base16 =
      (uint32_t)i16 * TOKEN_ROW_BYTES + (uint32_t)(((8 * (g16 >> 1) + (g16 & 1)) ^ token_swizzle<TOKEN_ROW_BYTES>(i16)) << 4);
  // B operand of instruction F = 2 P + abid
  auto frag16 = [&](int F) __attribute__((always_inline)) {
    u32x8_t raw;
    if (TOKEN_IMAGE) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t t = *reinterpret_cast<const u32x4_t*>(
            region + (token_read_base16 ^ (uint32_t)((16 * (F >> 1) + 4 * (F & 1) + 2 * h) << 4)));
        raw[4 * h] = t.x; raw[4 * h + 1] = t.y; raw[4 * h + 2] = t.z; raw[4 * h + 3] = t.w;
      }
      return __builtin_bit_cast(half16_t, raw);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row_const = 128 * (F >> 1) + 32 * (F & 1) + 4 * (q & 1) + 16 * (q >> 1);
      const u32x2_t t = lds_read_tr16(lane_ptr16 + row_const * ROW_BYTES);
      raw[2 * q] = t.x;
      raw[2 * q + 1] = t.y;
    }
    return __builtin_bit_cast(half16_t, raw);
  };
  auto compute16 = [&](const AChunk (&a)[R]) __attribute__((always_inline)) {
    // The compute unit serves the older half of the wavefronts first, when their loads are accepted and again when both of a
    // SIMD's have work; from its first chunk on the younger half goes first, so that the two end closer together (us, without ->
    // with, token-major form: 11008 x 4096 with 1 / 4 / 16 tokens 5.00 / 5.02 / 5.63 -> 4.87 / 4.88 / 5.56, 8192 x 8192 with 8
    // 5.92 -> 5.66; the plain form no different, 4096 x 4 x 11008 6.83 -> 6.93).
    if (TOKENS && wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
    half16_t bf[4];
#pragma unroll
    for (int F = 0; F < 4; ++F) bf[F] = frag16(F);
    A16 t[R];
#pragma unroll
    for (int r = 0; r < R; ++r) t[r] = gather16(a[r]);
#pragma unroll
    for (int F = 0; F < 4; ++F)
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          u32x4_t av;
#pragma unroll
          for (int q = 0; q < 4; ++q) av[q] = ((t[r].sign[h][F >> 1] << (4 * (F & 1) + q)) & 0x80008000u) | one;
          const half8_t a8 = __builtin_bit_cast(half8_t, av);
          acc16[r][h] = (F & 1) == 0 ? smfmac16<0, BF16>(a8, bf[F], acc16[r][h], t[r].idx[h][F >> 1])
                                     : smfmac16<1, BF16>(a8, bf[F], acc16[r][h], t[r].idx[h][F >> 1]);
        }
  };

  auto frag = [&](int image_step, int f) __attribute__((always_inline)) {
    u32x8_t raw;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int row_const = image_step * 32 + 4 * (q & 1) + 16 * (q >> 1);
      const u32x2_t t = lds_read_tr16(lane_ptr + row_const * ROW_BYTES + f * 64);
      raw[2 * q] = t.x;
      raw[2 * q + 1] = t.y;
    }
    return __builtin_bit_cast(half16_t, raw);
  };
  // the SMFMACs of image SUB_INDEX of a chunk: steps SUB_INDEX * IMG_STEPS ... + IMG_STEPS - 1
  auto compute = [&](const AChunk (&a)[R], auto sub_tag) __attribute__((always_inline)) {
    if constexpr (M16) {
      compute16(a);
      return;
    }
    constexpr int FIRST_STEP = decltype(sub_tag)::value * IMG_STEPS;
    // Fragments are read in groups of FG K steps (4 FG transpose reads per column fragment) into one of two register
    // sets: while the SMFMACs of a group run, the reads of the next group are already in flight, so only the first
    // group of an image waits for LDS. The scheduling barriers keep later groups' reads from being hoisted as well
    // (8 registers per fragment). Sixteen-wavefront workgroups have 128 registers per wavefront and no room for the
    // second set: they read each group when it is due.
    constexpr bool kAhead = NW <= 8;
    constexpr int FG = (R >= 4 || NF > 1) ? 2 : 4;
    constexpr int GROUPS = IMG_STEPS / FG;
    static_assert(IMG_STEPS % FG == 0 && GROUPS >= 1 && GROUPS <= 4, "whole groups of K steps per image");
    half16_t bfrag[kAhead ? 2 : 1][FG][NF];
    auto read_group = [&](int first_in_image, half16_t (&dst)[FG][NF]) __attribute__((always_inline)) {
#pragma unroll
      for (int st = 0; st < FG; ++st)
#pragma unroll
        for (int f = 0; f < NF; ++f) dst[st][f] = frag(first_in_image + st, f);
    };
    auto group = [&](auto index_tag) __attribute__((always_inline)) {
      constexpr int G = decltype(index_tag)::value;
      if constexpr (G < GROUPS) {
        constexpr int FIRST = FIRST_STEP + G * FG;  // step within the chunk
        constexpr int SET = kAhead ? (G & 1) : 0;
        if constexpr (!kAhead) read_group(G * FG, bfrag[0]);
        else if constexpr (G + 1 < GROUPS) read_group((G + 1) * FG, bfrag[SET ^ 1]);
        auto step = [&](auto offset_tag) __attribute__((always_inline)) {
          constexpr int OFFSET = decltype(offset_tag)::value;
          if constexpr (OFFSET < FG) {
            constexpr int STEP = FIRST + OFFSET;
#pragma unroll
            for (int r = 0; r < R; ++r) {
              const half8_t av = expand_signs<STEP>(a[r], one);
#pragma unroll
              for (int f = 0; f < NF; ++f)
                acc[r][f] = smfmac_step<STEP, false, BF16>(a[r], av, bfrag[SET][OFFSET][f], acc[r][f]);
            }
          }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        if constexpr (G + 1 < GROUPS) __builtin_amdgcn_sched_barrier(0);
      }
    };
    if constexpr (kAhead) read_group(0, bfrag[0]);
    group(std::integral_constant<int, 0>{});
    group(std::integral_constant<int, 1>{});
    group(std::integral_constant<int, 2>{});
    group(std::integral_constant<int, 3>{});
  };

  // The next image is requested while this one is multiplied. Sixteen wavefronts have 128 registers each: no room for an image
  // of 32 registers with wide columns, and with sixteen its requests crowd out the ones for the weights (4096 x 11008 with 16
  // tokens 8.45 -> 8.9 us).
  constexpr bool kFewLoads = (TOKENS && !X32 && TOKEN_LOADS <= 2) || COLUMNS > 0;
  constexpr bool kPrefetchB = NW <= 8 || kFewLoads;
  u32x4_t breg[8];
  char* const d_out = reinterpret_cast<char*>(p.d) + (size_t)block_y * p.m * p.n * (p.d_f16 ? 2 : 4);
  if (short_k) {
    u32x4_t breg2[8];
    load_b(first * kChunkK, breg);
    load_a(first, a_cur);
    // (pieces at any alignment: not when a K split leaves this wavefront one chunk, 512 x 20352 with three columns 9.9 -> 8.8 us)
    if (MODE != kSkinnyBAny || first + NW < kc_end) load_b((first + NW) * kChunkK, breg2);
    load_a(first + NW, a_next);
    if (first < kc_end) {
      store_b(first * kChunkK, breg);
      compute(a_cur, std::integral_constant<int, 0>{});
    }
    if (first + NW < kc_end) {
      store_b((first + NW) * kChunkK, breg2);
      compute(a_next, std::integral_constant<int, 0>{});
    }
  }
  // Two or three chunks for each of sixteen wavefronts: as in the short form, everything is requested at once. A wavefront without a
  // last chunk requests one too, which it does not multiply: past the weight's end the weight's last one and zeros of B, in a K split
  // the next split's. None stands in a branch, where the compiler could not count it (see kSkinnyBTokens); 17 chunks, 32 requested, are
  // faster so, too. us, one chunk after the other | this: 4096 x 11008 with 1 / 4 tokens 6.03 | 4.97, 6.22 | 5.22; 4096 x 4352 with 1 / 4 4.04 | 3.66,
  // 4.23 | 3.94; 33 chunks, 8192 x 8448 6.09 | 5.44, 6.08 | 5.55. Images of four loads are no faster for it, 2048 x 5120 with five tokens
  // 3.65 | 4.11.
  const bool at_once = NW == 16 && kFewLoads && kc_end - kc_begin > NW && kc_end - kc_begin <= 3 * NW;
  if constexpr (NW == 16 && kFewLoads) {
    auto rounds_at_once = [&](auto rounds_tag) __attribute__((always_inline)) {
      constexpr int ROUNDS = decltype(rounds_tag)::value;
      u32x4_t b[ROUNDS][8];
      AChunk a[ROUNDS - 1][R];
      load_b(first * kChunkK, b[0]);
#pragma unroll
      for (int i = 1; i < ROUNDS; ++i) {
        load_a(first + i * NW, a[i - 1]);
        load_b((first + i * NW) * kChunkK, b[i]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < ROUNDS; ++i) {
        if (i == ROUNDS - 1 && first + i * NW >= kc_end) break;  // wave-uniform
        store_b((first + i * NW) * kChunkK, b[i]);
        if (i == 0) compute(a_cur, std::integral_constant<int, 0>{});
        else compute(a[i - 1], std::integral_constant<int, 0>{});
      }
    };
    if (at_once) {
      if (kc_end - kc_begin > 2 * NW) rounds_at_once(std::integral_constant<int, 3>{});
      else rounds_at_once(std::integral_constant<int, 2>{});
    }
  }
  // (of sixteen wavefronts a short K leaves some without a chunk: no request for those)
  // Eight loads of tokens: the first image's one per sixteen clocks. All at once, behind the requests for the weights, they keep out the
  // other wavefronts' (us, a branch around each | at once | this: 10624 x 5024 with 16 tokens 6.69 | 6.91 | 6.63, 8256 x 4992 with 14 6.42 |
  // 6.64 | 6.37, 8768 x 8096 with 15 8.67 | 8.89 | 8.64, 4608 x 20320 with 15 10.7 | 10.9 | 10.6; the loop's spaced as well, no better)
  constexpr bool kSpaced = TOKENS && !X32 && TOKEN_LOADS == 8 && NW == 8;
  if (kPrefetchB && !short_k && !at_once && (NW <= 8 || first < kc_end)) load_b(first * kChunkK, breg, kSpaced);
  for (int kc = short_k || at_once ? kc_end : first; kc < kc_end; kc += NW) {
    const int k_base = kc * kChunkK;
    // this wavefront has another chunk after this one (wave-uniform): only then is the next chunk requested; a load
    // past the last chunk would be one more instruction for the memory pipeline, a third of them when a wavefront
    // has two or three chunks
    const bool more = kc + NW < kc_end;
    if (!kPrefetchB) load_b(k_base, breg);
    store_b(k_base, breg);  // after the previous image's fragment reads: LDS operations of a wavefront execute in order
    if (kPrefetchB && (SUB > 1 || more)) load_b(SUB > 1 ? k_base + IMG_ROWS : k_base + NW * kChunkK, breg);
    if (more) load_a(kc + NW, a_next);
    compute(a_cur, std::integral_constant<int, 0>{});
    // the chunk's further images (SUB - 1 of them)
    auto further = [&](auto sub_tag) __attribute__((always_inline)) {
      constexpr int S = decltype(sub_tag)::value;
      if constexpr (S < SUB) {
        const int image_base = k_base + S * IMG_ROWS;
        if (!kPrefetchB) {
          __builtin_amdgcn_sched_barrier(0);  // this image's loads stay behind the previous image's SMFMACs
          load_b(image_base, breg);
        }
        store_b(image_base, breg);
        if (kPrefetchB && (S + 1 < SUB || more)) load_b(S + 1 < SUB ? image_base + IMG_ROWS : k_base + NW * kChunkK, breg);
        compute(a_cur, sub_tag);
      }
    };
    further(std::integral_constant<int, 1>{});
    further(std::integral_constant<int, 2>{});
    further(std::integral_constant<int, 3>{});
#pragma unroll
    for (int r = 0; r < R; ++r) a_cur[r] = a_next[r];
  }

  smfmac_drain();
  // ---- add the NW partial tiles through LDS: region of wavefront w := its R tiles as [r][32 rows][NC cols] fp32
  constexpr int ROUND_ROWS = RT * kRowBlock;
  // token-major form: a thread's results of a round are one row of several tokens, its bias is requested in front of the barrier
  // (what a bias costs, us, loaded behind the sums | here: 11008 x 4096 with 4 tokens 0.25 | 0.08, with 16 0.38 | 0.07, 28672 x 8192 with
  // 16 0.50 | 0.02)
  static_assert(NT % ROUND_ROWS == 0, "a thread's row of a round");
  float row_bias[R / RT];
  if (TOKENS && p.bias)
#pragma unroll
    for (int round = 0; round < R / RT; ++round) {
      const int row = rb_first * kRowBlock + round * ROUND_ROWS + tid % ROUND_ROWS;
      row_bias[round] = load_element(p.bias, p.bias_type, row < p.m ? row : 0);
    }
#pragma unroll
  for (int round = 0; round < R / RT; ++round) {
    if (round > 0) __syncthreads();  // the previous round's tiles have been read
    {
      float* tile = reinterpret_cast<float*>(region);
      const int col = lane & 31;
      if (M16) {
#pragma unroll
        for (int rr = 0; rr < RT; ++rr)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int row = 16 * h + 4 * g16 + v;
              const float value = acc16[round * RT + rr][h][v];
              // token-major: [token][weight row of the round], the row index XOR-swizzled by the token so that neither
              // these stores (16 tokens, one row) nor the reads below (one token, consecutive rows) collide in a bank
              if (TOKEN_IMAGE) tile[i16 * ROUND_ROWS + ((rr * 32 + row) ^ i16)] = value;
              else tile[(rr * 32 + row) * NC + i16] = value;
            }
      } else if (col < NC) {
#pragma unroll
        for (int rr = 0; rr < RT; ++rr)
#pragma unroll
          for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              const int row = 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
              const float value = acc[round * RT + rr][f][v];
              tile[(rr * 32 + row) * NC + f * 32 + col] = value;
            }
      }
    }
    __syncthreads();
    const int round_row0 = rb_first * kRowBlock + round * ROUND_ROWS;
    if (TOKEN_IMAGE) {
      // (plain form: neighbouring threads take neighbouring results, and there are no others than its columns')
      for (int idx = tid; idx < ROUND_ROWS * (COLUMNS > 0 ? COLUMNS : NC); idx += NT) {
        const int local = COLUMNS > 0 ? idx / (COLUMNS + (COLUMNS == 0)) : idx % ROUND_ROWS;
        const int token = COLUMNS > 0 ? idx - local * COLUMNS : idx / ROUND_ROWS;
        const int pos = token * ROUND_ROWS + (local ^ (token & 31));
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += reinterpret_cast<const float*>(bs + w * kSkinnyRegion)[pos];
        const int row = round_row0 + local;
        if (token < p.n && row < p.m) {
          if (TOKENS && p.bias) sum += row_bias[round];
          const size_t o = COLUMNS > 0 ? (size_t)row * COLUMNS + token : (size_t)token * p.m + row;
          // a B of one column is a token-major x of one token and its result column is y: the launcher sends such calls
          // here with their alpha, beta and C (element o of C in both layouts); the linear layer passes 1, 0, null
          sum = p.alpha * sum;
          if (p.beta != 0.f)
            sum = sum + p.beta * (p.c_f16 ? (float)reinterpret_cast<const _Float16*>(p.c)[o] : reinterpret_cast<const float*>(p.c)[o]);
          if (p.d_f16) reinterpret_cast<uint16_t*>(d_out)[o] = round_one<BF16>(sum);
          else reinterpret_cast<float*>(d_out)[o] = sum;
        }
      }
    } else {
      for (int idx = tid; idx < ROUND_ROWS * NC; idx += NT) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += reinterpret_cast<const float*>(bs + w * kSkinnyRegion)[idx];
        const int col = idx % NC;
        const int row = round_row0 + idx / NC;
        if (col < p.n && row < p.m) {
          const size_t o = (size_t)row * p.n + col;
          float x = p.alpha * sum;
          if (p.beta != 0.f) {
            const float cv = p.c_f16 ? (float)reinterpret_cast<const _Float16*>(p.c)[o] : reinterpret_cast<const float*>(p.c)[o];
            x = x + p.beta * cv;
          }
          if (p.d_f16) reinterpret_cast<_Float16*>(d_out)[o] = (_Float16)x;
          else reinterpret_cast<float*>(d_out)[o] = x;
        }
      }
    }
  }
}

// A kernel's arguments as three vectors of fourteen dwords in all, which the hardware puts into scalar registers before a wavefront
// starts (the build asks for that); out of a struct they would have to be loaded, 0.2 us before the first address can be formed.
// Vectors, because the host pays for every argument of a launch. us inside a HIP graph, weights from HBM, struct -> this: 11008 x
// 4096 with 1 / 4 / 16 tokens 5.58 / 5.56 / 6.48 -> 5.10 / 5.10 / 6.27, 28672 x 8192 with one 13.2 -> 12.7, 11008 x 4 x 4096 6.25 ->
// 5.94. With flags, alpha and beta in a fourth vector that is loaded where the results are stored, the smallest calls were slower than
// with the struct: 512 x 2 x 512 2.93 | 3.09 | 2.87 as a struct | so | now, 512 x 4 x 512 2.84 | 2.86 | 2.78, 512 x 3 x 512 2.81 | 2.97 |
// 2.88.
enum ArgFlags : uint32_t { kArgD16 = 1, kArgC16 = 2, kArgBias = 4 };  // bits 3 and 4: type of the bias
struct LaunchArgs {
  u32x8_t operands;  // prep, b; n, k, m, chunks_per_split (chunks of 256 of an int K: 23 bits; what a kernel adds from bit 24 on)
  u32x4_t results;   // d, the bias (token-major form) or C: a call has one of them at most
  u32x2_t scale;     // alpha, beta
  uint32_t flags;
};
static LaunchArgs pack_args(const SkinnyArgs& a) {
  const uint64_t prep = (uint64_t)a.prep, b = (uint64_t)a.b, d = (uint64_t)a.d, extra = (uint64_t)(a.bias ? a.bias : a.c);
  return LaunchArgs{u32x8_t{(uint32_t)prep, (uint32_t)(prep >> 32), (uint32_t)b, (uint32_t)(b >> 32), (uint32_t)a.n, (uint32_t)a.k,
                            (uint32_t)a.m, (uint32_t)a.chunks_per_split},
                    u32x4_t{(uint32_t)d, (uint32_t)(d >> 32), (uint32_t)extra, (uint32_t)(extra >> 32)},
                    u32x2_t{__builtin_bit_cast(uint32_t, a.alpha), __builtin_bit_cast(uint32_t, a.beta)},
                    (a.d_f16 ? kArgD16 : 0) | (a.c_f16 ? kArgC16 : 0) | (a.bias ? kArgBias : 0) | (uint32_t)a.bias_type << 3};
}
__device__ __forceinline__ SkinnyArgs unpack_args(u32x8_t operands, u32x4_t results, u32x2_t scale, uint32_t flags) {
  auto pointer = [](uint32_t low, uint32_t high) __attribute__((always_inline)) { return (uint64_t)high << 32 | low; };
  SkinnyArgs p{};
  p.prep = reinterpret_cast<const uint8_t*>(pointer(operands[0], operands[1]));
  p.b = reinterpret_cast<const _Float16*>(pointer(operands[2], operands[3]));
  p.n = operands[4]; p.k = operands[5]; p.m = operands[6]; p.chunks_per_split = operands[7] & 0xFFFFFFu;
  p.kc_total = (p.k + kChunkK - 1) / kChunkK;
  p.d = reinterpret_cast<void*>(pointer(results[0], results[1]));
  p.c = reinterpret_cast<const void*>(pointer(results[2], results[3]));  // read where beta != 0 only: never with a bias
  p.bias = flags & kArgBias ? p.c : nullptr;
  p.d_f16 = flags & kArgD16; p.c_f16 = flags & kArgC16; p.bias_type = flags >> 3 & 3;
  // (values, not elements: the compiler casts the bits of a vector's first element where an element is named)
  p.alpha = __builtin_bit_cast(float, (uint32_t)scale[0]); p.beta = __builtin_bit_cast(float, (uint32_t)scale[1]);
  return p;
}

// operands[7]: ArgFlags from bit 24 on
template <int NW, int R, int MODE, int NC, bool BF16>
__global__ __launch_bounds__(64 * NW, NW == 16 ? 4 : 2) void skinny_kernel(u32x8_t operands, u32x4_t results, u32x2_t scale) {
  const SkinnyArgs p = unpack_args(operands, results, scale, operands[7] >> 24);
  skinny_body<NW, R, MODE, NC, BF16>(p, blockIdx.x, blockIdx.y);
}

// The same with its arguments as a struct: all of them loaded at the start, the compiler's schedule of the image's requests and
// stores another one. Pieces at any alignment are the faster for it with images of 32 and 64 columns, and with those of sixteen where
// a wavefront of a 128-row group has one or two chunks, or one of a 64-row group two, and more where the pieces of ten to fourteen
// columns start at whole words (us inside a HIP graph, weights from HBM, vectors | struct: 4096 x 33 x 4096 12.8 | 12.1, 1344 x 47 x 1376
// 6.6 | 6.2, 4096 x 18 x 4096 5.9 | 5.7, 832 x 18 x 6112 7.0 | 6.9; 24576 x 3 x 4096 10.6 | 9.8, 17408 x 8 x 2048 6.0 | 5.7, 9216 x 3 x
// 4096 7.4 | 7.2; 12672 x 12 x 6752 9.96 | 9.68, 13888 x 10 x 9952 13.65 | 13.16, 9344 x 14 x 24032 27.4 | 25.9). Elsewhere the vectors are
// (28672 x 8 x 8192 13.8 | 16.0, 18432 x 3 x 8192 14.4 | 16.0, 25280 x 11 x 4992 13.0 | 13.7; 64-row groups of one chunk: 8256 x 13 x 512
// 4.1 | 4.2, 10176 x 3 x 2048 4.7 | 4.8, of three and more 1 to 3 % where a piece may start at any half, none from the sixth on; 32-row
// groups: 2048 x 8 x 3456 3.75 | 3.87, 8192 x 3 x 8192 8.4 | 8.7).
template <int NW, int R, int MODE, int NC, bool BF16>
__global__ __launch_bounds__(64 * NW, NW == 16 ? 4 : 2) void skinny_struct_kernel(SkinnyArgs p) {
  skinny_body<NW, R, MODE, NC, BF16>(p, blockIdx.x, blockIdx.y);
}

// Grouped form: several independent products y_i = x_i W_i^T + bias_i that share the token count, in one launch. The
// workgroups are numbered over the concatenated row groups of the problems; a workgroup finds its problem by
// comparing its number with the problems' first workgroups (wave-uniform, a handful of scalar compares) and then runs
// the token-major body on that problem's arguments. Decode-sized products take a few microseconds each, of which the
// launch itself and the ramp of the memory pipeline are a large part: one launch for the q / k / v or gate / up
// projections of a layer pays them once.
// What decides about the problem comes in scalar registers, so that a workgroup of up to four problems waits for one load of 40
// bytes where it walked through a table of first workgroups and then read its problem (us inside a HIP graph, before -> now:
// 3 x 4096 x 4096 with eight tokens 6.18 -> 5.35, 4096 + 2 x 1024 4.57 -> 4.09, 2 x 11008 x 4096 with sixteen 9.02 -> 7.97).
struct GroupProblem {
  const uint8_t* prep;
  const _Float16* b;
  void* d;
  const void* bias;
  int m, k;
};
// Up to MOST problems. The host pays for the bytes of a launch's arguments (64 | 192 | 384 | 720 bytes: 2.5 | 3.0 | 3.4 | 3.5 us), so
// there are kernels for up to four, whose first workgroups are arguments of their own.
template <int MOST>
struct GroupTable {
  GroupProblem problem[MOST];
  int first_block[MOST];
};
constexpr int kGroupFew = 4;
template <>
struct GroupTable<kGroupFew> {
  GroupProblem problem[kGroupFew];
};
struct GroupShared {  // the same for all problems (same_group_types)
  int d_f16, bias_type, tokens_per_group;
};

// First workgroups of problems 1, 2 and 3 (INT_MAX where there is none), the number of problems, the token count; `problem`: of
// this workgroup, `block`: its number among that problem's.
template <int MOST>
__device__ __forceinline__ SkinnyArgs group_problem(int first1, int first2, int first3, int count, int tokens, const GroupShared& shared,
                                                    const GroupTable<MOST>& table, int& block) {
  block = blockIdx.x;
  int which = (block >= first1) + (block >= first2) + (block >= first3);
  int first = block >= first3 ? first3 : block >= first2 ? first2 : block >= first1 ? first1 : 0;
  if constexpr (MOST > kGroupFew)
    for (int i = kGroupFew; i < count; ++i)
      if (block >= table.first_block[i]) which = i, first = table.first_block[i];
  const GroupProblem& q = table.problem[which];
  SkinnyArgs p{};
  p.prep = q.prep; p.b = q.b; p.d = q.d; p.bias = q.bias;
  p.m = q.m; p.n = tokens; p.k = q.k;
  p.kc_total = p.chunks_per_split = (q.k + kChunkK - 1) / kChunkK;
  p.alpha = 1.f;
  p.d_f16 = shared.d_f16; p.bias_type = shared.bias_type; p.tokens_per_group = shared.tokens_per_group;
  block -= first;
  return p;
}

template <int NW, int R, int MODE, bool BF16, int MOST>
__global__ __launch_bounds__(64 * NW, NW == 16 ? 4 : 2) void skinny_group_kernel(int first1, int first2, int first3, int count,
                                                                                 int tokens, GroupShared shared, GroupTable<MOST> table) {
  int block;
  const SkinnyArgs p = group_problem(first1, first2, first3, count, tokens, shared, table, block);
  skinny_body<NW, R, MODE, 16, BF16>(p, block, 0);
}

static bool same_group_types(const SkinnyArgs& a, const SkinnyArgs& b) {
  return a.bf16 == b.bf16 && a.d_f16 == b.d_f16 && a.bias_type == b.bias_type;
}

// The arguments of a grouped launch from the launcher's (first_block filled in).
template <int MOST>
struct GroupLaunch {
  int first[4];
  GroupShared shared;
  GroupTable<MOST> table;
};
template <int MOST>
static GroupLaunch<MOST> group_launch(const SkinnyGroupArgs& g) {
  GroupLaunch<MOST> l{};
  for (int i = 0; i < 4; ++i) l.first[i] = i < g.count ? g.first_block[i] : INT_MAX;
  l.shared = GroupShared{g.problem[0].d_f16, g.problem[0].bias_type, g.problem[0].tokens_per_group};
  for (int i = 0; i < g.count; ++i) {
    const SkinnyArgs& p = g.problem[i];
    l.table.problem[i] = GroupProblem{p.prep, p.b, p.d, p.bias, p.m, p.k};
    if constexpr (MOST > kGroupFew) l.table.first_block[i] = g.first_block[i];
  }
  return l;
}

template <int NW, int R, int MODE, int NC, bool BF16 = false>
static hipError_t launch_skinny_mode(const SkinnyArgs& args, hipStream_t stream) {
  const dim3 grid((args.m / kRowBlock + R - 1) / R, args.splits), threads(64 * NW);
  constexpr bool kPieces = MODE == kSkinnyBAny;
  if constexpr (kPieces && (NC > 16 || NW <= 8)) {  // see skinny_struct_kernel
    const bool words = R == 2 && args.n >= 10 && args.n <= 14 && args.n % 2 == 0 && (reinterpret_cast<uintptr_t>(args.b) & 3) == 0;
    if (NC > 16 || (args.chunks_per_split > (R == 2 ? NW : 0) && (words || args.chunks_per_split <= 2 * NW)))
      return launch_kernel(skinny_struct_kernel<NW, R, MODE, NC, BF16>, grid, threads, 0, stream, args);
  }
  if constexpr (!kPieces || NC == 16) {
    LaunchArgs a = pack_args(args);
    a.operands[7] |= a.flags << 24;
    return launch_kernel(skinny_kernel<NW, R, MODE, NC, BF16>, grid, threads, 0, stream, a.operands, a.results, a.scale);
  }
  return hipErrorInvalidValue;  // not reached: wide images of pieces went the other way
}

// Load instructions per image of the token-major form on 16-bit activations, of those that there are kernels for. us inside HIP
// graphs, weights from HBM, eight conditional ones | this: 4096 x 11008 with 1 / 4 / 8 / 16 tokens 6.03 | 4.97, 6.22 | 5.22, 6.41 | 5.75,
// 7.26 | 7.08, 4096 x 4096 3.73 | 3.29, 3.79 | 3.37, 3.94 | 3.60, 4.33 | 4.08, 11008 x 4096 5.00 | 4.89, 5.05 | 4.60, 5.25 | 4.66, 5.87 |
// 5.58, 28672 x 8192 with 1 / 8 / 16 12.1 | 11.5, 12.5 | 12.3, 13.8 | 13.8; on fp32 activations 4096 x 4096 with 1 / 4 4.00 | 3.31, 4.12 |
// 3.58. More loads than tokens cost their place in the load path (8192 x 8192 with 9 tokens 6.16 with six, 6.68 with eight).
static int token_loads(int tokens) { return tokens <= 2 ? 1 : tokens <= 4 ? 2 : tokens <= 8 ? 4 : tokens <= 12 ? 6 : 8; }
template <int NW, int R, bool BF16>
static hipError_t launch_skinny_token_loads(const SkinnyArgs& args, hipStream_t stream) {
  switch (token_loads(args.n)) {
    case 1: return launch_skinny_mode<NW, R, kSkinnyBTokens + 1, 16, BF16>(args, stream);
    case 2: return launch_skinny_mode<NW, R, kSkinnyBTokens + 2, 16, BF16>(args, stream);
    case 4: return launch_skinny_mode<NW, R, kSkinnyBTokens + 4, 16, BF16>(args, stream);
    case 6: return launch_skinny_mode<NW, R, kSkinnyBTokens + 6, 16, BF16>(args, stream);
    default: return launch_skinny_mode<NW, R, kSkinnyBTokens + 8, 16, BF16>(args, stream);
  }
}

// Fills in the K split of a split-K kernel launch: splits <= 1 = one pass straight into d.
static hipError_t skinny_split_setup(SkinnyArgs& args, SkinnyArgs& first_pass) {
  if (args.splits <= 1) {
    args.splits = 1;
    args.chunks_per_split = args.kc_total;
    first_pass = args;
    return hipSuccess;
  }
  if (args.chunks_per_split < 1 || (long)(args.splits - 1) * args.chunks_per_split >= args.kc_total || !args.split_ws)
    return hipErrorInvalidValue;  // an empty split would only add zeros, but it is a planning error
  first_pass = args;  // raw fp32 partial sums per split, laid out like the result
  first_pass.alpha = 1.f;
  first_pass.beta = 0.f;
  first_pass.c = nullptr;
  first_pass.bias = nullptr;
  first_pass.d = args.split_ws;
  first_pass.d_f16 = 0;
  return hipSuccess;
}

}  // namespace onebit
