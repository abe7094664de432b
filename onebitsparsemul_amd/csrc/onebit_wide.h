// The split-K kernel whose images of B asynchronous copies bring to LDS, plain and token-major, and the launch of one
// instantiation. onebit_wide.hip and onebit_wide_tokens.hip instantiate it.
#pragma once
#include "onebit_skinny.h"

#include <atomic>

namespace onebit {

// =====================================================================================================
// wide_kernel: y[t][r] = sum_k W[r][k] x[t][k] + bias[r] (token-major form) and D = alpha A B + beta C (plain form) for 17
// tokens or columns and more, in groups of up to 64 per workgroup. The plain form differs in how an image lies in LDS
// and is read (see wide_body) and in the epilogue; below, x and token stand for B and column too.
// Workgroup = eight wavefronts that share R row blocks (32 rows each) and split K among themselves chunk by chunk, as in
// skinny_kernel. What differs is how x gets to the matrix cores: every wavefront keeps a ring of two images (64 K values of
// all tokens, 2 KB per sixteen) in LDS that asynchronous copies fill. No registers hold x on its way, so the tile can be
// 128 x 64 (R = 4), and with v_smfmac_f32_16x16x64 there are no idle columns at 16 or 48 tokens; one fragment read from LDS
// serves 2 R SMFMACs (R of the 32x32x32 ones that whole 32-column tiles take).
// Bound: no single resource. Stamps of every wavefront, launches back to back, weights from HBM (us after the first one's start,
// wavefronts 0-3 | 4-7):
//                                        28672 x 8192, 48 tokens   the same, 64   4096 x 11008, 500 tokens
//   first operand and image there        2.6 | 3.3                 2.8 | 3.4      2.0 | 2.9
//   first chunk multiplied               7.5 | 6.6                 8.3 | 7.1      6.9 | 6.3
//   last chunk (of 4, 4, 6 or 5)         17.5 | 14.5               19.7 | 16.6    24.7 | 19.5
//   all partial tiles in LDS             18.0                      20.5           25.9
//   tiles added, stored                  21.9                      24.6           28.0
// 2 to 3 us until the operands come; the first chunk, up to 1.7 us longer than a later one; a chunk of each of the eight wavefronts
// from then on 5400 to 5900 clocks of those that go first, 6900 to 7200 of the others, against 5000 to 5200 of a full pipeline that a
// compute unit's 64 bytes per clock set (76 KB of x and weights per 64 K at 64 tokens, 60 at 48); those that go first then wait 3 to 6
// us; and 2 to 4 us of reduction. SMFMACs fill 30 % (48 tokens) and 47 % (500) of the time.
// skinny_kernel's 64-row groups staged x through registers, 16 KB of LDS writes and reads per 64 x 64 weights; a 128-row group halves
// that. us inside a HIP graph under load, weights from HBM, skinny_kernel -> now: 28672 x 8192 with 24 / 48 / 64 tokens 16.6 / 33.4 /
// 35.9 -> 15.6 / 21.8 / 23.8; 11008 x 4096 8.0 / 11.0 / 11.7 -> 6.3 / 8.0 / 9.5; 4096 x 4096 5.7 / 8.4 / 8.7 -> 3.8 / 4.6 / 4.7; 1024 x
// 1024 with 56 5.0 -> 2.55. Up to sixteen tokens there is no gain (11008 x 4096 with 16: 6.4 -> 6.1, with 4: 5.5 -> 5.8; 28672 x 8192
// with 16: 13.5 -> 14.0): skinny_kernel keeps those.
// Beyond 64 tokens, and for products, the host's plan compares it with the kernel it would replace (onebit_capi.hip).
// =====================================================================================================
// Source of zeros for the copies of K positions at or past K.
static __device__ __attribute__((aligned(16))) uint32_t g_zero16_wide[4] = {0, 0, 0, 0};

constexpr int kWideWaves = 8;
constexpr int kWideImageK = 64;

template <int R, int COPIES>
struct WideShape {
  static constexpr int CT = (COPIES + 1) / 2;            // column tiles of sixteen tokens
  static constexpr int IMAGE_BYTES = 16 * CT * kWideImageK * 2;
  static constexpr int REGION = 2 * IMAGE_BYTES;         // ring of one wavefront; holds the sums of RT row blocks at the end
  static constexpr int RT = R < 2 ? R : 2;
  static constexpr int LDS_BYTES = kWideWaves * REGION;
};

// COPIES: 1 KiB copies per image, one per eight tokens. A workgroup multiplies up to 8 COPIES tokens from first_token on.
// TOKENS = false is the plain form, D = alpha A B + beta C, a column of B in the place of a token: B's rows start 16-byte
// aligned (ldb % 8 == 0, first_token % 8 == 0), an image is 64 of them as they lie, COPIES 16-byte pieces each, read through
// transpose reads; COPIES is even. RAGGED: n is no multiple of eight and the rows are read where they lie, 16 bytes from any
// address on (ldb = n): a piece that reaches past the end of its row takes values of the next one along, which only meet columns
// that are never stored; past the end of B it is moved back and shifted into place in LDS.
// PARTS: the chunks that are left after whole rounds of eight, up to four of them, are dealt over the wavefronts in parts
// of 64 or 128 K values, where otherwise some wavefronts have a chunk more and the others wait for them: 9 chunks are five
// images in a row instead of eight, 43 are 22 instead of 24.
template <int R, int COPIES, bool TOKENS, bool BF16, bool PARTS, bool RAGGED>
__device__ __forceinline__ void wide_body(const SkinnyArgs& p, const int block_x, const int block_y, const int first_token,
                                          char* const smem) {
  using Shape = WideShape<R, COPIES>;
  constexpr int NW = kWideWaves, CT = Shape::CT, RT = Shape::RT;
  // Whole 32-column tiles take the 32x32x32 SMFMAC: with two wavefronts per SIMD it runs at 35.8 clocks beside the four sign
  // expansions it needs at 64 columns (32 alone), the 16x16x64 one at 43.4 for the same work beside its two, and the prepared
  // operand is used as it is stored (us: 28672 x 8192 with 32 tokens 16.7 -> 16.1, 8192 x 8192 with 128 15.9 -> 15.2, 16384 x 16384
  // with 64 27.7 -> 26.9; where every compute unit is busy and power sets the clock about 1 % the other way).
  constexpr bool S32 = CT % 2 == 0;
  // a chunk of few column tiles is over before the next one's operand can come from HBM: it is requested a chunk earlier
  constexpr bool FAR = CT == 1 || (CT == 3 && R <= 2);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rb_total = p.m / kRowBlock, rb_first = block_x * R;
  char* const region = smem + wave * Shape::REGION;
  const uint32_t region_offset = lds_offset_of(smem) + wave * Shape::REGION;
  const int kc_total = p.kc_total, k_total = p.k;
  // plain form: eight columns fewer than the image holds where the group is an odd number of pieces wide. The next group
  // stores those eight, and D may be C: each element must be read and written once.
  const int group = TOKENS ? 8 * COPIES : p.tokens_per_group;
  const int tokens = p.n - first_token < group ? p.n - first_token : group;
  const int kc_begin = block_y * p.chunks_per_split;
  const int kc_end = kc_begin + p.chunks_per_split < kc_total ? kc_begin + p.chunks_per_split : kc_total;
  const int first = kc_begin + wave;

  const uint32_t meta_off = (uint32_t)lane * 16u, sign_off = (uint32_t)kSignOffset + (uint32_t)lane * 8u;
  buffer_t a_buffer[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int rb = rb_first + r;
    if (rb >= rb_total) rb = rb_total - 1;  // never stored
    a_buffer[r] = make_buffer(p.prep + (size_t)rb * kc_total * kBlockBytes, (uint32_t)kc_total * kBlockBytes);
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
  AChunk raw[R], next[R] = {};
  load_a(first, raw);
  __builtin_amdgcn_sched_barrier(0);

  // Plain form: piece q of row r lies at position q ^ row_swizzle(r), so that the 32 lanes of one transpose read (rows r ...
  // r + 3 and r + 8 ... r + 11, 32 bytes each) meet in no bank where the row stride would make them.
  constexpr int PIECES = 2 * CT;
  auto row_swizzle = [](int row) __attribute__((always_inline)) {
    return PIECES == 8 ? (((row >> 1) & 1) << 2) | (((row >> 3) & 1) << 1) : PIECES == 4 ? ((row >> 3) & 1) << 1 : 0;
  };
  // copy i of an image: tokens 8 i ... 8 i + 7, eight 16-byte pieces each; piece q of token t lies at position
  // q ^ token_swizzle(t). Tokens past the end: the last one again, their results are not stored.
  uint32_t copy_off[COPIES];
  const int piece0 = (lane & 7) ^ (lane >> 4);
#pragma unroll
  for (int i = 0; i < COPIES; ++i) {
    if constexpr (TOKENS) {
      int token = 8 * i + (lane >> 3);
      if (token >= tokens) token = tokens - 1;
      copy_off[i] = ((uint32_t)token * (uint32_t)k_total + 8u * (piece0 ^ (4 * (i & 1)))) * 2u;
    } else {
      const int row = (64 * i + lane) / PIECES;
      int col = 8 * (((64 * i + lane) % PIECES) ^ row_swizzle(row));
      if (first_token + col >= p.ldb) col = 0;  // columns past the row's end: the first ones again, never stored
      copy_off[i] = ((uint32_t)row * (uint32_t)p.ldb + col) * 2u;
    }
  }
  const size_t k_stride = TOKENS ? 2 : (size_t)p.ldb * 2;  // bytes from one K position to the next
  const char* const x_bytes = reinterpret_cast<const char*>(p.b + (TOKENS ? (size_t)first_token * k_total : (size_t)first_token));
  const char* const zeros = reinterpret_cast<const char*>(g_zero16_wide);
  // RAGGED: the last row's image takes the general path
  const int k_inside = RAGGED ? k_total - 1 : k_total;
  const char* const last_piece = reinterpret_cast<const char*>(p.b) + (size_t)k_total * p.ldb * 2 - 16;
  auto copy_image = [&](int k0, int slot) __attribute__((always_inline)) {
    const uint32_t dst = __builtin_amdgcn_readfirstlane(region_offset + slot * Shape::IMAGE_BYTES);
    if (k0 + kWideImageK <= k_inside) {  // wave-uniform
#pragma unroll
      for (int i = 0; i < COPIES; ++i) lds_dma16_base(x_bytes + k0 * k_stride, copy_off[i], dst + i * 1024);
    } else {
      // K positions at or past k come from a block of zeros
#pragma unroll
      for (int i = 0; i < COPIES; ++i) {
        uint32_t off = copy_off[i];
        asm volatile("" : "+v"(off));  // keeps the 64-bit addresses out of the registers of the other path
        const int k = k0 + (TOKENS ? 8 * (piece0 ^ (4 * (i & 1))) : (64 * i + lane) / PIECES);
        const char* from = x_bytes + k0 * k_stride + off;
        if (RAGGED && from > last_piece) from = last_piece;
        lds_dma16(k < k_total ? from : zeros, dst + i * 1024);
      }
    }
  };

  // RAGGED: the piece that was moved back, of the last row of B, if it is in this image
  auto mend_image = [&](int k0, int slot) __attribute__((always_inline)) {
    const int row = k_total - 1 - k0, piece = (p.n - 1 - first_token) >> 3;
    if (!RAGGED || row < 0 || row >= kWideImageK || piece >= PIECES) return;  // wave-uniform
    shift_piece(region + slot * Shape::IMAGE_BYTES + ((row * PIECES + (piece ^ row_swizzle(row))) << 4), first_token + 8 * piece + 8 - p.n, lane);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  const int i16 = lane & 15, g16 = lane >> 4;
  const uint32_t one = packed_one_in_vgpr<BF16>();
  float4v_t acc[S32 ? 1 : 2 * R][S32 ? 1 : CT];
  float16_t acc32[S32 ? R : 1][S32 ? CT / 2 : 1];
#pragma unroll
  for (int rt = 0; rt < (S32 ? 1 : 2 * R); ++rt)
#pragma unroll
    for (int ct = 0; ct < (S32 ? 1 : CT); ++ct) {
      acc[rt][ct] = float4v_t{0.f, 0.f, 0.f, 0.f};
      asm volatile("" : "+v"(acc[rt][ct]));
    }
#pragma unroll
  for (int r = 0; r < (S32 ? R : 1); ++r)
#pragma unroll
    for (int f = 0; f < (S32 ? CT / 2 : 1); ++f) {
#pragma unroll
      for (int v = 0; v < 16; ++v) acc32[r][f][v] = 0.f;
      asm volatile("" : "+v"(acc32[r][f]));
    }

  // Operands of one chunk. A lane of the prepared block (row l % 32, half ga) holds, per 32-wide step, what a lane of the
  // instruction (row l % 16, group g) holds for sixteen K positions. With the index halves of two stages' even steps in one
  // register and those of their odd steps in another, one v_permlane16_swap leaves the groups (even, ga 0), (odd, ga 0),
  // (even, ga 1), (odd, ga 1) of block rows 0-15 in the first and of rows 16-31 in the second; ABID picks the stage. Group g
  // thus covers K positions 32 (g % 2) + 16 (g / 2) + [0, 16) of the 64-wide stage.
  struct ATile {
    uint32_t idx[2][2], sign[2][2];  // [row half][stage pair]
  };
  ATile t[R];
  const uint32_t sign_shift = 4u * (g16 & 1);
  auto gather = [&](const AChunk (&a)[R]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const uint32_t even = __builtin_amdgcn_perm(a[r].meta[2 * q + 1], a[r].meta[2 * q], 0x05040100u);
        const uint32_t odd = __builtin_amdgcn_perm(a[r].meta[2 * q + 1], a[r].meta[2 * q], 0x07060302u);
        const auto m = __builtin_amdgcn_permlane16_swap(even, odd, false, false);
        const uint32_t w = q == 0 ? a[r].sign.x : a[r].sign.y;
        const auto sg = __builtin_amdgcn_permlane16_swap(w, w, false, false);
        t[r].idx[0][q] = m[0];
        t[r].idx[1][q] = m[1];
        t[r].sign[0][q] = sg[0] << sign_shift;
        t[r].sign[1][q] = sg[1] << sign_shift;
      }
  };
  // B operand of column tile ct: pieces 4 (g / 2) + g % 2 and that + 2 of token 16 ct + l % 16
  const uint32_t read_base = (uint32_t)i16 * 128u + (uint32_t)(((4 * (g16 >> 1) + (g16 & 1)) ^ token_swizzle(i16)) << 4);
  // plain form: K rows 32 (g / 2) + 8 (g % 2) + {0 ... 7, 16 ... 23} of column l % 16, four by a transpose read
  const int lane_row = 32 * (g16 >> 1) + 8 * (g16 & 1) + (i16 >> 2);
  uint32_t tile_off[CT];
  if constexpr (!TOKENS)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
      tile_off[ct] = lane_row * PIECES * 16 + (((2 * ct + ((i16 & 3) >> 1)) ^ row_swizzle(lane_row)) << 4) + (i16 & 1) * 8;
  half16_t frag[CT];
  // 32x32x32 form: frag[2 f + ks] = K step ks of the columns 32 f ... 32 f + 31
  const int gb = lane >> 5, col32 = lane & 31;
  const uint32_t read_base32 = (uint32_t)col32 * 128u + (uint32_t)((gb ^ token_swizzle(col32)) << 4);
  const int lane_row32 = 8 * gb + (i16 >> 2);
  const int c8 = (col32 >> 4) * 4 + (i16 & 3);
  auto read_image = [&](int slot) __attribute__((always_inline)) {
    if constexpr (S32) {
#pragma unroll
      for (int f = 0; f < CT / 2; ++f)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          u32x8_t raw_frag;
          if constexpr (TOKENS) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              const u32x4_t v = *reinterpret_cast<const u32x4_t*>(region + (read_base32 ^ ((4 * ks + 2 * h) << 4)) + slot * Shape::IMAGE_BYTES + f * 4096);
              raw_frag[4 * h] = v.x; raw_frag[4 * h + 1] = v.y; raw_frag[4 * h + 2] = v.z; raw_frag[4 * h + 3] = v.w;
            }
          } else {
            const int lc = 4 * f + (c8 >> 1);
            const uint32_t off = lane_row32 * PIECES * 16 + ((lc ^ row_swizzle(lane_row32)) << 4) + (c8 & 1) * 8;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const u32x2_t v = lds_read_tr16(region + slot * Shape::IMAGE_BYTES + off + (32 * ks + 4 * (q & 1) + 16 * (q >> 1)) * PIECES * 16);
              raw_frag[2 * q] = v.x; raw_frag[2 * q + 1] = v.y;
            }
          }
          frag[2 * f + ks] = __builtin_bit_cast(half16_t, raw_frag);
        }
      return;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
      u32x8_t raw_frag;
      if constexpr (!TOKENS) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2_t v = lds_read_tr16(region + slot * Shape::IMAGE_BYTES + tile_off[ct] + (4 * (q & 1) + 16 * (q >> 1)) * PIECES * 16);
          raw_frag[2 * q] = v.x; raw_frag[2 * q + 1] = v.y;
        }
      } else
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(region + (read_base ^ (h << 5)) + slot * Shape::IMAGE_BYTES + ct * 2048);
        raw_frag[4 * h] = v.x; raw_frag[4 * h + 1] = v.y; raw_frag[4 * h + 2] = v.z; raw_frag[4 * h + 3] = v.w;
      }
      frag[ct] = __builtin_bit_cast(half16_t, raw_frag);
    }
  };
  auto compute = [&](auto s_tag) __attribute__((always_inline)) {
    constexpr int S = decltype(s_tag)::value;
    if constexpr (S32) {
      half8_t av[2];
      av[0] = expand_signs<2 * S>(raw[0], one);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int i = ks * R + r;
          if (i + 1 < 2 * R) av[(i + 1) & 1] = (i + 1) / R == 0 ? expand_signs<2 * S>(raw[(i + 1) % R], one) : expand_signs<2 * S + 1>(raw[(i + 1) % R], one);
#pragma unroll
          for (int f = 0; f < CT / 2; ++f)
            acc32[r][f] = ks == 0 ? smfmac_step<2 * S, false, BF16>(raw[r], av[i & 1], frag[2 * f + ks], acc32[r][f])
                                  : smfmac_step<2 * S + 1, false, BF16>(raw[r], av[i & 1], frag[2 * f + ks], acc32[r][f]);
          __builtin_amdgcn_sched_barrier(0);
        }
      return;
    }
    // the signs of the next row tile are expanded in front of the SMFMACs of the current one; the fences keep the optimizer
    // from expanding all of them first, which takes more registers than there are
    auto expand = [&](int rt) __attribute__((always_inline)) {
      u32x4_t av;
#pragma unroll
      for (int q = 0; q < 4; ++q) av[q] = ((t[rt >> 1].sign[rt & 1][S / 2] << (8 * (S & 1) + q)) & 0x80008000u) | one;
      return __builtin_bit_cast(half8_t, av);
    };
    half8_t av[2];
    av[0] = expand(0);
#pragma unroll
    for (int rt = 0; rt < 2 * R; ++rt) {
      if (rt + 1 < 2 * R) av[(rt + 1) & 1] = expand(rt + 1);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        acc[rt][ct] = smfmac16<S & 1, BF16>(av[rt & 1], frag[ct], acc[rt][ct], t[rt >> 1].idx[rt & 1][S / 2]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Requests return in order, and a wait names how many younger ones may be outstanding. Per chunk a wavefront requests its
  // image 2, the prepared operand of its next chunk, image 3 and the first two images of the next chunk; before the loop the
  // operand of the first chunk and its first two images. Nothing is requested past the last chunk (wave-uniform branches).
  // FAR: the operand of the chunk after the next one at the end of a chunk, behind image 1 of the next, and before the loop that of the
  // second chunk, last. us, weights from HBM, otherwise -> this: 4096 x 11008 with 24 / 40 / 64 tokens 8.7 / 10.5 / 10.7 -> 8.5 / 10.3 /
  // 10.5 (as it was before the operand was requested inside the chunk), 7360 x 10880 with 77 16.4 -> 15.7, 11264 x 40 x 3072 8.1 -> 7.6;
  // four row blocks with three tiles, whose chunks take longer, and whole 32-column tiles are no faster for it.
  // A compute unit takes 64 bytes of requests per clock, so what stands in front of the first SMFMAC is what all wavefronts
  // request before it: the second chunk's operand, requested up front too, held that up by 48 KB (28672 x 8192 with 48 tokens:
  // the first SMFMAC of a workgroup 6000 to 8000 clocks after its start). And the older four wavefronts are served first all the
  // way, ending 5000 clocks before the younger ones, whose SIMDs then have one wavefront each; the younger ones go first from
  // here on. us, weights from HBM, both: 28672 x 8192 with 64 23.7 -> 22.9, 16384 x 16384 with 64 26.9 -> 25.6, 4096 x 4096 with
  // 32 3.93 -> 3.72, 2048 x 8192 with 256 10.4 -> 9.8.
  if (first < kc_end) {
    // parts: the remainder's chunks in halves, up to two of them in quarters
    static_assert((NW & (NW - 1)) == 0, "a round is a power of two");
    const int left = (kc_end - kc_begin) & (NW - 1);
    const int halvings = !PARTS || left > 4 || kc_end - kc_begin < NW ? 0 : left > 2 ? 1 : 2;
    const int whole_end = halvings ? kc_end - left : kc_end;
    const int part_kc = whole_end + (wave >> halvings), part_images = 4 >> halvings;
    const int part_image = (wave & ((1 << halvings) - 1)) * part_images;  // first image of the part, of four
    const bool has_part = PARTS && part_kc < kc_end;
    copy_image(first * kChunkK, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (S32) {
      // the compiler's wait for the operand counts its own loads only: image 1 goes behind it (4096 x 4096 with 128 tokens
      // 6.2 -> 6.0; in the other form the operand is first used further down and image 1 is better requested here)
#pragma unroll
      for (int r = 0; r < R; ++r) asm volatile("" : "+v"(raw[r].meta), "+v"(raw[r].sign));
      __builtin_amdgcn_sched_barrier(0);
    }
    copy_image(first * kChunkK + kWideImageK, 1);
    if (FAR && first + NW < whole_end) load_a(first + NW, next);
    else if (FAR && PARTS && has_part) load_a(part_kc, next);
    __builtin_amdgcn_sched_barrier(0);
    if (wave >= NW / 2) __builtin_amdgcn_s_setprio(1);
    if constexpr (!S32) gather(raw);
    int kc = first;
#pragma unroll 1
    do {
      const bool whole = kc + NW < whole_end, more = whole || has_part;  // what follows: a chunk, a part or nothing
      const int next_kc = !PARTS || whole ? kc + NW : part_kc;
      const int next_k0 = next_kc * kChunkK + (!PARTS || whole ? 0 : part_image * kWideImageK);
      auto stage = [&](auto s_tag) __attribute__((always_inline)) {
        constexpr int S = decltype(s_tag)::value;
        // all but the requests younger than image S
        if (more) wait_vmcnt<((FAR ? S < 2 : S == 1 || S == 2) ? COPIES + 2 * R : COPIES)>();
        else wait_vmcnt<(S < 3 ? COPIES : 0)>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (RAGGED) mend_image(kc * kChunkK + S * kWideImageK, S & 1);
        read_image(S & 1);
        if constexpr (S == (FAR ? 2 : 3)) {
          // the wait the compiler puts in front of the operand's first use counts its own loads only and so also waits for
          // every copy issued by then: here that is one image, which has had a stage's time
#pragma unroll
          for (int r = 0; r < R; ++r) asm volatile("" : "+v"(next[r].meta), "+v"(next[r].sign));
        }
        if (S < 2 || (S == 2 ? more : whole || (has_part && part_images > 1))) {
          wait_vmcnt_lgkm0<63>();  // the image is in registers: its place is free
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
          copy_image(S < 2 ? kc * kChunkK + (S + 2) * kWideImageK : next_k0 + (S - 2) * kWideImageK, S & 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        compute(s_tag);
        if constexpr (S == 0 && !FAR) {
          if (more) load_a(next_kc, next);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      stage(std::integral_constant<int, 0>{});
      stage(std::integral_constant<int, 1>{});
      stage(std::integral_constant<int, 2>{});
      stage(std::integral_constant<int, 3>{});
      if (PARTS && !whole && has_part) {  // the operand of the part's images to the front
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (part_image & 2) next[r].meta.x = next[r].meta.z, next[r].meta.y = next[r].meta.w, next[r].sign.x = next[r].sign.y;
          if (part_image & 1) next[r].meta.x = next[r].meta.y, next[r].sign.x <<= 8;
        }
      }
      if constexpr (S32) {
#pragma unroll
        for (int r = 0; r < R; ++r) raw[r] = next[r];
      } else {
        gather(next);
        if constexpr (FAR) {
          if (whole && kc + 2 * NW < whole_end) load_a(kc + 2 * NW, next);
          else if (PARTS && whole && has_part) load_a(part_kc, next);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      kc += NW;
    } while (kc < whole_end);
    if (PARTS && has_part) {
      if (part_images > 1) wait_vmcnt<COPIES>();
      else wait_vmcnt<0>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const int part_k0 = part_kc * kChunkK + part_image * kWideImageK;
      if constexpr (RAGGED) mend_image(part_k0, 0);
      read_image(0);
      compute(std::integral_constant<int, 0>{});
      if (part_images > 1) {
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (RAGGED) mend_image(part_k0 + kWideImageK, 1);
        read_image(1);
        compute(std::integral_constant<int, 1>{});
      }
    }
  }

  // ---- add the eight partial tiles, RT row blocks per round: a token's rows as 16-byte slots of four rows, slot s at
  // position s ^ (token % slots)
  constexpr int SLOTS = RT * 8;
  char* const y_out = reinterpret_cast<char*>(p.d) + (size_t)block_y * p.m * p.n * 4;  // a K split's slice: fp32 sums
  // A thread's results of a round are four rows of several tokens: their bias is requested once, in front of the reduction's barrier, which
  // hides its latency. The calls without one have a barrier and sums of their own: what selects or skips a bias, and whatever stands in
  // front of the barrier (a wait for the operands that a wavefront without a chunk has requested, too), is 2 to 5 % of a call of few
  // chunks. us, bias of each row loaded behind the sums | requested in front of one barrier for both | behind it, sums of their own | this:
  // with a bias 28672 x 8192 with 48 tokens 22.5 | 21.1 | 21.5 | 21.0, 11008 x 4096 with 64 10.2 | 9.6 | 9.8 | 9.7, 16384 x 1024 with 64 5.64 |
  // 5.35 | 5.22 | 5.07, 16704 x 1056 with 44 9.25 | 8.10 | 8.23 | 8.10; without 16384 x 1024 with 64 4.98 | 5.22 | 4.93 | 4.93, 11520 x
  // 1312 with 53 5.43 | 5.62 | 5.38 | 5.40, 1152 x 960 with 175 2.96 | 3.02 | 2.97 | 2.95, 18304 x 768 with 64 6.17 | 6.31 | 6.20 | 6.13.
  static_assert(64 * NW % SLOTS == 0, "a thread's rows of a round");
#pragma unroll
  for (int round = 0; round < R / RT; ++round) {
    if (round > 0) __syncthreads();
    if constexpr (S32) {
#pragma unroll
      for (int rr = 0; rr < RT; ++rr)
#pragma unroll
        for (int f = 0; f < CT / 2; ++f)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int token = 32 * f + col32, slot = 8 * rr + 2 * q + gb;
            const float16_t& a = acc32[round * RT + rr][f];
            *reinterpret_cast<float4v_t*>(region + (token * SLOTS + (slot ^ (token & (SLOTS - 1)))) * 16) =
                float4v_t{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
          }
    } else
#pragma unroll
    for (int rr = 0; rr < RT; ++rr)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const int token = 16 * ct + i16, slot = 8 * rr + 4 * h + g16;
          *reinterpret_cast<float4v_t*>(region + (token * SLOTS + (slot ^ (token & (SLOTS - 1)))) * 16) =
              acc[2 * (round * RT + rr) + h][ct];
        }
    auto finish = [&](auto bias_tag) __attribute__((always_inline)) {
      constexpr bool BIAS = decltype(bias_tag)::value;
      u32x4_t bias_raw = {};
      if constexpr (BIAS) {
        const int row = (rb_first + round * RT) * kRowBlock + 4 * (tid % SLOTS);
        bias_raw = load_four(p.bias, p.bias_type, row < p.m ? row : 0);
      }
      __syncthreads();
      for (int idx = tid; idx < SLOTS * 16 * CT; idx += 64 * NW) {
        const int slot = TOKENS ? idx % SLOTS : idx / (16 * CT), token = TOKENS ? idx / SLOTS : idx % (16 * CT);
        const int at = (token * SLOTS + (slot ^ (token & (SLOTS - 1)))) * 16;
        float4v_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += *reinterpret_cast<const float4v_t*>(smem + w * Shape::REGION + at);
        const int row = (rb_first + round * RT) * kRowBlock + 4 * slot;
        if (token >= tokens || row >= p.m) continue;
        if constexpr (!TOKENS) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const size_t o = (size_t)(row + e) * p.n + first_token + token;
            float x = p.alpha * sum[e];
            if (p.beta != 0.f)
              x = x + p.beta * (p.c_f16 ? (float)reinterpret_cast<const _Float16*>(p.c)[o] : reinterpret_cast<const float*>(p.c)[o]);
            if (p.d_f16) reinterpret_cast<_Float16*>(y_out)[o] = (_Float16)x;
            else reinterpret_cast<float*>(y_out)[o] = x;
          }
          continue;
        }
        if constexpr (BIAS) sum += values_of_four(bias_raw, p.bias_type);
        const size_t o = (size_t)(first_token + token) * p.m + row;
        if (p.d_f16)
          *reinterpret_cast<u32x2_any_t*>(y_out + o * 2) = u32x2_t{round_pair<BF16>(sum[0], sum[1]), round_pair<BF16>(sum[2], sum[3])};
        else
          *reinterpret_cast<u32x4_any_t*>(y_out + o * 4) = __builtin_bit_cast(u32x4_t, sum);
      }
    };
    if (!TOKENS || __builtin_expect(p.bias == nullptr, 1)) finish(std::false_type{});
    else finish(std::bool_constant<TOKENS>{});
  }
}

// Arguments as for skinny_kernel, but: operands[7] holds the columns per workgroup from bit 24 on; shape[0] ArgFlags and, from bit 5
// on, the column groups of a grid that is walked in strips (0: the grid has them as its third dimension), shape[1] 2^32 / (2 row
// groups) + 1. `scale`, which the token-major form does not use, is the only argument that is not in registers from the start.
// In strips of two column groups an XCD is given a contiguous range of the list (workgroup b runs on XCD b % 8, all eight are there:
// the launcher's condition), so that what its workgroups read of x and of the weight meets in its L2; where that pays is the host's
// rule (wide_in_strips).
template <int R, int COPIES, bool TOKENS, bool BF16, bool PARTS, bool RAGGED>
__global__ __launch_bounds__(64 * kWideWaves, 2) void wide_kernel(u32x8_t operands, u32x4_t results, u32x2_t shape, u32x2_t scale) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  SkinnyArgs p = unpack_args(operands, results, scale, shape[0]);
  p.tokens_per_group = operands[7] >> 24;
  p.ldb = RAGGED ? p.n : (p.n + 7) & ~7;  // the launcher's condition
  int x = blockIdx.x, group = blockIdx.z;
  if (const int groups = shape[0] >> 5; groups > 0) {
    const int row_groups = (p.m + 32 * R - 1) / (32 * R);
    const int total = row_groups * groups, per = total / 8, rem = total % 8, xcd = x % 8;
    const int v = xcd * per + (xcd < rem ? xcd : rem) + x / 8;
    int strip = (int)__umulhi((uint32_t)v, shape[1]), w = v - strip * 2 * row_groups;
    if (w < 0) --strip, w += 2 * row_groups;  // the reciprocal is rounded up
    const bool pair = 2 * (strip + 1) * row_groups <= total;
    x = pair ? w >> 1 : w;
    group = 2 * strip + (pair ? w & 1 : 0);
  }
  wide_body<R, COPIES, TOKENS, BF16, PARTS, RAGGED>(p, x, blockIdx.y, group * p.tokens_per_group, smem);
}

// The dynamic-LDS limit of a kernel, a per-device attribute; threads that race here set the same value.
static hipError_t wide_lds_limit(const void* kern, int lds, std::atomic<bool> (&attr_done)[64]) {
  if (lds <= 65536) return hipSuccess;
  int device = 0;
  if (hipError_t st = hipGetDevice(&device); st != hipSuccess) return st;
  if (device < 0 || device >= 64) return hipErrorInvalidDevice;
  if (attr_done[device].load(std::memory_order_acquire)) return hipSuccess;
  if (hipError_t st = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds); st != hipSuccess) return st;
  attr_done[device].store(true, std::memory_order_release);
  return hipSuccess;
}

// Whether a workgroup that multiplies `chunks` chunks deals a remainder in parts. us inside HIP graphs, weights from HBM, a chunk to a
// wavefront | parts: one or two chunks left of two rounds, layers 5760 x 2272 with 54 tokens 5.76 | 5.37, 2752 x 2368 with 62 5.26 | 4.73,
// 5568 x 2496 with 21 5.20 | 4.63, 10048 x 2464 with 43 8.42 | 7.74, 1472 x 2496 with 128 5.46 | 4.92; of more rounds 28672 x 8448 with
// 48 23.6 | 23.0, 6720 x 8352 with 17 9.45 | 8.89, 1280 x 10592 with 153 10.4 | 10.0; three or four chunks of up to five rounds 0.98 of the
// time in the mean of 111 calls (4096 x 11008 with 32 / 500 8.55 | 8.38, 30.8 | 30.6), of more 1.00 of 71 (three layers of 1536 x 15168 with
// 20 11.65 | 12.19, eight of 576 x 21120 with 22 17.1 | 17.7): a chunk to a wavefront. From five chunks on a part is a chunk, and below a round the calls wait for the host. The build
// of the kernel without parts is 1 to 4 % faster where there are none (4096 x 4096 with 48 5.2 | 5.4).
static bool wide_has_parts(int chunks) {
  const int left = chunks % kWideWaves;
  return chunks >= kWideWaves && left >= 1 && left <= (chunks < 6 * kWideWaves ? 4 : 2);
}

template <int R, int COPIES, bool TOKENS, bool BF16, bool PARTS, bool RAGGED>
static hipError_t launch_wide_parts(const SkinnyArgs& args, hipStream_t stream) {
  static std::atomic<bool> attr_done[64] = {};
  constexpr int lds = WideShape<R, COPIES>::LDS_BYTES;
  const auto kern = wide_kernel<R, COPIES, TOKENS, BF16, PARTS, RAGGED>;
  if (hipError_t st = wide_lds_limit(reinterpret_cast<const void*>(kern), lds, attr_done); st != hipSuccess) return st;
  const int rows = (args.m + 32 * R - 1) / (32 * R), groups = (args.n + args.tokens_per_group - 1) / args.tokens_per_group;
  LaunchArgs a = pack_args(args);
  a.operands[7] |= (uint32_t)args.tokens_per_group << 24;
  const u32x2_t shape = {a.flags | (args.strips ? (uint32_t)groups << 5 : 0u), (uint32_t)((uint64_t(1) << 32) / (2 * rows) + 1)};
  const dim3 grid = args.strips ? dim3(rows * groups, args.splits) : dim3(rows, args.splits, groups);
  return launch_kernel(kern, grid, dim3(64 * kWideWaves), lds, stream, a.operands, a.results, shape, a.scale);
}

template <int R, int COPIES, bool TOKENS, bool BF16, bool RAGGED = false>
static hipError_t launch_wide_kernel(const SkinnyArgs& args, hipStream_t stream) {
  if (wide_has_parts(args.chunks_per_split))  // of all splits but perhaps the last
    return launch_wide_parts<R, COPIES, TOKENS, BF16, true, RAGGED>(args, stream);
  return launch_wide_parts<R, COPIES, TOKENS, BF16, false, RAGGED>(args, stream);
}

}  // namespace onebit
