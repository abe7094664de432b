// The main SMFMAC kernel of the one-bit 2:4 sparse GEMM on gfx950, D = alpha * A * B + beta * C (B staged through LDS, A
// expanded in registers), in its plain form and in the token-major form of the linear layer, y = x W^T + bias with x and y
// stored token by token (the transposes of B and D), and the launch of one instantiation. onebit_gemm.hip and
// onebit_gemm_tokens.hip instantiate it. Replaces the CUTLASS specialisations of the reference (csrc/kernel.h:13-72,
// csrc/threadblock.h:62-233, csrc/warp.h:18-690) with code written for 64-wide wavefronts; nothing is translated from them.
#pragma once
#include "onebit_device.h"
#include "onebit_launch.h"
#include <atomic>
#include <type_traits>

namespace onebit {

// =====================================================================================================
// Main kernel.
// Workgroup = 4 or 8 wavefronts arranged WM x WN; each wavefront owns FM x FN accumulator tiles of 32 x 32.
// B is staged through LDS in stages of 64 K rows; the LDS image of a stage is row-major (N contiguous)
// with the 16-byte column chunks of row r XOR-swizzled so that the four rows a 16-lane group touches in
// one transpose read fall into different bank groups.
// =====================================================================================================
constexpr int kStageK = 64;
constexpr int kStages = 4;  // LDS ring; one prepared-operand chunk (256 K) = one trip around the ring

template <int BN>
__device__ __forceinline__ int chunk_swizzle(int row) {
  // 16-byte chunk index XOR; rows r..r+3 must land in four different 64-byte bank groups. Bit 3 of the row swaps the
  // 32-byte halves of a group: the 16x16x64 form's lanes 0-15 and 16-31 read 32 bytes each of rows r..r+3 and
  // r+8..r+11 in one pass (the 32x32x32 form reads whole 64-byte groups and does not notice).
  return (BN >= 128) ? (((row & 3) << 2) | (((row >> 3) & 1) << 1)) : (((row >> 1) & 1) << 2);
}

// KG = 2: two groups of WM x WN wavefronts cover the same tile; group g multiplies K step g of every 64-row stage,
// and the two partial tiles are added through LDS at the end (twice the wavefronts per SIMD for the same tile).
template <int WM, int WN, int FM, int FN, int KG = 1>
struct TileShape {
  static constexpr int BM = WM * FM * 32;
  static constexpr int BN = WN * FN * 32;
  static constexpr int CH = BN / 8;                       // 16-byte chunks per LDS row
  static constexpr int NW = WM * WN * KG;                 // wavefronts per workgroup
  static constexpr int NL = kStageK * CH / (64 * NW);     // chunk copies per thread per stage
  static constexpr int STAGE_BYTES = kStageK * BN * 2;
  static constexpr int LDS_B_BYTES = kStages * STAGE_BYTES;
  static constexpr int NA = ((BM / 32) * 1536 + 1024 * NW - 1) / (1024 * NW);  // 1 KiB A copies per wavefront per chunk
  static constexpr int LDS_BYTES = LDS_B_BYTES + NA * 1024 * NW;
  static_assert(NW == 4 || NW == 8, "four or eight wavefronts per workgroup");
  static_assert(kStageK * CH % (64 * NW) == 0, "the stage must divide into whole wavefront copies");
  static_assert(NL >= 1, "tile too narrow for the copy pattern");
  static_assert(KG == 1 || (KG == 2 && WM * FM <= 4), "the second group's partial tile must fit the stage ring");
};

// XCD-aware tile order. Workgroup b runs on XCD b % xcds (xcds = 8 on a whole MI355X; the launcher derives it from the
// device's compute-unit count, so a partitioned GPU keeps the property), so XCD x is given a contiguous range of a tile list
// that is ordered in blocks of GROUP_M row tiles x 4 column tiles (row tile fastest), blocks running down M inside
// a strip of 4 column tiles, strips running along N. GROUP_M x 4 = the workgroups resident on one XCD (64 for the
// four-wavefront tiles with two workgroups per CU; 32 for the tiles with one per CU), which then form one block: every B column
// panel it streams is shared by GROUP_M workgroups and every A row panel by 4 in that XCD's L2, and the whole
// range of one XCD covers few column strips, so B is fetched into few L2s.
// strip_reciprocal = 2^32 / (4 tiles_m) + 1. The other two quotients are of a divisor from 1 to 4 and below 4: no division in front of the
// first copy (measured at GemmResult).
constexpr int kStripTiles = 4;
template <int GROUP_M>
__device__ __forceinline__ void tile_of_block(int b, int tiles_m, int tiles_n, int xcds, uint32_t strip_reciprocal, int& tm, int& tn) {
  static_assert(GROUP_M == 8 || GROUP_M == 16, "a power of two");
  const int total = tiles_m * tiles_n;
  int per, rem, x, local;
  if (xcds == 8) {  // the usual case with constant divisors
    per = total >> 3, rem = total & 7, x = b & 7, local = b >> 3;
  } else {
    per = total / xcds, rem = total % xcds, x = b % xcds, local = b / xcds;
  }
  const int v = x * per + (x < rem ? x : rem) + local;
  int strip = (int)__umulhi((uint32_t)v, strip_reciprocal), w = v - strip * kStripTiles * tiles_m;
  if (w < 0) --strip, w += kStripTiles * tiles_m;  // the reciprocal is rounded up
  const int strip_w = (tiles_n - strip * kStripTiles) < kStripTiles ? (tiles_n - strip * kStripTiles) : kStripTiles;
  const uint32_t rows = (uint32_t)w / GROUP_M;  // of tiles, in units of a group's height
  const int group = strip_w == 4 ? rows >> 2 : strip_w == 3 ? rows / 3 : strip_w == 2 ? rows >> 1 : rows;
  const int group_h = (tiles_m - group * GROUP_M) < GROUP_M ? (tiles_m - group * GROUP_M) : GROUP_M;
  const int u = w - group * GROUP_M * strip_w;
  const int column = (u >= group_h) + (u >= 2 * group_h) + (u >= 3 * group_h);
  tm = group * GROUP_M + u - column * group_h;
  tn = strip * kStripTiles + column;
}

// One stage (64 K = two SMFMAC K steps) of a wavefront's FM x FN tile.
template <int FM, int FN, int BN, int STAGE_IN_CHUNK>
__device__ __forceinline__ void compute_stage(const char* stage_lds, const AChunk (&a)[FM], float16_t (&acc)[FM][FN],
                                              const int (&frag_off)[FN], int lane_row_off, uint32_t one) {
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    half16_t bv[FN];
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      u32x8_t raw;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row_const = ks * 32 + 4 * (q & 1) + 16 * (q >> 1);
        const u32x2_t t = lds_read_tr16(stage_lds + lane_row_off + row_const * (BN * 2) + frag_off[fn]);
        raw[2 * q] = t.x;
        raw[2 * q + 1] = t.y;
      }
      bv[fn] = __builtin_bit_cast(half16_t, raw);
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      half8_t av;
      if (ks == 0) av = expand_signs<2 * STAGE_IN_CHUNK>(a[fm], one);
      else av = expand_signs<2 * STAGE_IN_CHUNK + 1>(a[fm], one);
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        if (ks == 0) acc[fm][fn] = smfmac_step<2 * STAGE_IN_CHUNK, false>(a[fm], av, bv[fn], acc[fm][fn]);
        else acc[fm][fn] = smfmac_step<2 * STAGE_IN_CHUNK + 1, false>(a[fm], av, bv[fn], acc[fm][fn]);
      }
    }
  }
}

// ---- building blocks of the asynchronous-copy main loop ----------------------------------------------
// Token-major stage image (linear-layer form): row t = the stage's 64 K values of token t (128 bytes, eight 16-byte
// pieces, piece p stored at position p ^ token_swizzle(t)). The operand of K step ks is pieces 4 ks + gb and 4 ks + 2 + gb of
// the lane's token: two plain 16-byte reads at the precomputed lane offsets piece_off[2 ks + h].
// One packed register (kept values 2p, 2p+1 of K step STEP) of expand_signs. The empty volatile statement keeps the two
// instructions where they are written: the optimizer otherwise sinks them past the stage's barrier to the block of their
// first use.
template <int STEP>
__device__ __forceinline__ uint32_t expand_sign_register(const AChunk& a, uint32_t packed_one, int p) {
  const uint32_t w = STEP < 4 ? a.sign.x : a.sign.y;
  uint32_t v = ((w << (4 * (STEP % 4) + p)) & 0x80008000u) | packed_one;
  asm volatile("" : "+v"(v));
  return v;
}

// One piece of the B fragments of a K step: piece r of the row-major image is transpose read q = r % 4 of fragment
// r / 4, piece r of the token-major image is 16-byte read h = r % 2 of fragment r / 2.
template <int BN>
__device__ __forceinline__ void load_b_piece(const char* stage_lds, int ks, int r, u32x8_t* bv, const int* frag_off,
                                             int lane_row_off) {
  const int fn = r >> 2, q = r & 3;
  const int row_const = ks * 32 + 4 * (q & 1) + 16 * (q >> 1);
  const u32x2_t t = lds_read_tr16(stage_lds + lane_row_off + row_const * (BN * 2) + frag_off[fn]);
  bv[fn][2 * q] = t.x;
  bv[fn][2 * q + 1] = t.y;
}

__device__ __forceinline__ void load_b_piece_tokens(const char* wave_lds, int ks, int r, u32x8_t* bv,
                                                    const int* piece_off) {
  const int fn = r >> 1, h = r & 1;
  const u32x4_t t = *reinterpret_cast<const u32x4_t*>(wave_lds + piece_off[2 * ks + h] + fn * (32 * kStageK * 2));
  bv[fn][4 * h] = t.x; bv[fn][4 * h + 1] = t.y; bv[fn][4 * h + 2] = t.z; bv[fn][4 * h + 3] = t.w;
}

// The SMFMACs of one K step with the fetch work for the next step placed between them by hand: fetch(slot) runs right
// behind SMFMAC number `slot`, and scheduling fences keep it there (the compiler would otherwise keep the
// inline-assembly SMFMACs of the one-wavefront-per-SIMD tiles in one block, and order the rest as it likes).
template <int STEP, bool PINNED, bool BF16, int FM, int FN, class Fetch>
__device__ __forceinline__ void mfma_frags_fused(const AChunk (&a)[FM], const u32x4_t (&av)[FM], const u32x8_t (&bv)[FN],
                                                 float16_t (&acc)[FM][FN], Fetch&& fetch) {
#pragma unroll
  for (int fm = 0; fm < FM; ++fm)
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      __builtin_amdgcn_s_setprio(1);  // the wavefront that is about to issue an SMFMAC wins the arbitration on its SIMD
      const half8_t a8 = __builtin_bit_cast(half8_t, av[fm]);
      const half16_t b16 = __builtin_bit_cast(half16_t, bv[fn]);
      acc[fm][fn] = fm == 0 && fn == 0 ? smfmac_step<STEP, PINNED, BF16, true>(a[fm], a8, b16, acc[fm][fn])
                                       : smfmac_step<STEP, PINNED, BF16>(a[fm], a8, b16, acc[fm][fn]);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(fm * FN + fn);
      __builtin_amdgcn_sched_barrier(0);
    }
}

// us inside HIP graphs, arguments as one struct and three divisions by run-time values in front of the first copy | this: 512^3 5.12 |
// 4.78, 1024^3 7.11 | 6.47, 2048^3 15.2 | 14.8, 11008 x 256 x 4096 20.8 | 20.0, 640 x 816 x 576 7.64 | 7.08, 4096^3 62.6 | 61.6; large
// products within 1 %.
// A launch's arguments: eight dwords of operands (prep, b; m, n, k, ldb), four of the grid (tiles_m, tiles_n, reciprocal of a strip,
// chunks_per_split with the XCDs from bit 24 on) and what the epilogue takes.
struct GemmResult {
  void* d;
  const void* c;
  const void* bias;
  float alpha, beta;
  int c_f16, d_f16, bias_type;
};

// Source of zeros for the asynchronous copies of B rows at or past K.
static __device__ __attribute__((aligned(16))) uint32_t g_zero16[4] = {0, 0, 0, 0};

// TOKENS (with DMA only): the linear-layer form. p.b is x (p.n tokens x p.k, token-major), p.d is y (p.n tokens x
// p.m), the epilogue is y = acc + bias; a tile column is a token.
// RAGGED (plain form with DMA): n is no multiple of eight and the rows of B are copied from where they lie (ldb = n). A piece that
// reaches past the end of its row takes values of the next one along, which only meet columns that are never stored; past the
// end of B it is moved back and shifted into place in LDS (mend_stage). An instantiation of its own: the tests for that row made
// a product of few chunks slower (2048 x 512 x 512 5.25 -> 5.64 us).
template <int WM, int WN, int FM, int FN, bool DMA, bool TOKENS = false, int KG = 1, bool M16 = false, bool BF16 = false, bool RAGGED = false>
__global__ __launch_bounds__(64 * WM * WN * KG, (FM * FN <= 8 ? 2 : 1)) void gemm_kernel(u32x8_t operands, u32x4_t tiles, GemmResult result) {
  static_assert(!M16 || (DMA && KG == 1 && WN == 1 && FM == 4 && FN == 4), "the 16x16x64 form exists for the 512x128 four-wavefront tile");
  static_assert(TOKENS || !BF16, "bf16 activations exist for the token-major form");
  static_assert(DMA || !TOKENS, "the token-major form uses the asynchronous copies");
  static_assert(!RAGGED || (DMA && !TOKENS), "rows that lie anywhere are the plain form's");
  static_assert(DMA || KG == 1, "the two-group form uses the asynchronous copies");
  using TS = TileShape<WM, WN, FM, FN, KG>;
  constexpr int BM = TS::BM, BN = TS::BN, CH = TS::CH, NL = TS::NL, NW = TS::NW;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  // What the first copies need is in scalar registers when a wavefront starts (see LaunchArgs); the rest is loaded under them.
  GemmArgs p{};
  p.prep = reinterpret_cast<const uint8_t*>((uint64_t)operands[1] << 32 | operands[0]);
  p.b = reinterpret_cast<const _Float16*>((uint64_t)operands[3] << 32 | operands[2]);
  p.m = operands[4]; p.n = operands[5]; p.k = operands[6]; p.ldb = operands[7];
  p.kc_total = (p.k + kChunkK - 1) / kChunkK;
  p.tiles_m = tiles[0]; p.tiles_n = tiles[1]; p.chunks_per_split = tiles[3] & 0xFFFFFFu; p.xcds = tiles[3] >> 24;
  p.d = result.d; p.c = result.c; p.alpha = result.alpha; p.beta = result.beta; p.c_f16 = result.c_f16; p.d_f16 = result.d_f16;
  p.bias = result.bias; p.bias_type = result.bias_type;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, kept in a scalar register
  const int kg = KG == 2 ? wave / (WM * WN) : 0;   // K group of this wavefront
  const int wave_in_group = KG == 2 ? wave % (WM * WN) : wave;
  const int wm = wave_in_group / WN, wn = wave_in_group % WN;
  int tile_m, tile_n;
  // one workgroup per compute unit (eight wavefronts, or four that use all the registers): 32 resident on an XCD
  tile_of_block<(NW == 8 || FM * FN > 8 ? 8 : 16)>(blockIdx.x, p.tiles_m, p.tiles_n, p.xcds, tiles[2], tile_m, tile_n);
  const int row0 = tile_m * BM + wm * FM * 32;  // first row of this wavefront
  const int n0 = tile_n * BN;                   // first column of the workgroup
  const int col0 = n0 + wn * FN * 32;           // first column of this wavefront

  // ---- A operand addressing (prepared blocks) ----
  const int rb_total = p.m / kRowBlock;
  const uint8_t* a_block[FM];
#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
    int rb = row0 / kRowBlock + fm;
    if (rb >= rb_total) rb = rb_total - 1;  // rows past M: compute on valid data, never stored
    a_block[fm] = p.prep + (size_t)rb * p.kc_total * kBlockBytes;
  }

  // ---- B fragment addressing inside a stage ----
  const int i16 = lane & 15;
  const int gb = lane >> 5;
  const int c8 = ((lane & 31) >> 4) * 4 + (i16 & 3);  // 8-byte chunk inside the 32-column fragment
  const int lane_row = 8 * gb + (i16 >> 2);           // + compile-time row constants
  const int lane_row_off = lane_row * (BN * 2);
  int frag_off[FN];
#pragma unroll
  for (int fn = 0; fn < FN; ++fn) {
    const int lc = 4 * (wn * FN + fn) + (c8 >> 1);
    frag_off[fn] = ((lc ^ chunk_swizzle<BN>(lane_row)) << 4) + (c8 & 1) * 8;
  }

  int piece_off[4];  // token-major image: byte offsets of the lane's four pieces of a stage (see load_b_frags_tokens)
  {
    const int token = lane & 31;
    const int base = token * (kStageK * 2) + ((gb ^ token_swizzle(token)) << 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) piece_off[j] = base ^ ((4 * (j >> 1) + 2 * (j & 1)) << 4);
  }
  const char* const wave_image = smem + wn * FN * (32 * kStageK * 2);  // first token row of this wavefront in stage 0

  const uint32_t one = packed_one_in_vgpr<BF16>();
  // 32x32x32 form: FM x FN tiles of 32 x 32; 16x16x64 form: 2 FM x 2 FN tiles of 16 x 16 (the other array has one element)
  float16_t acc[M16 ? 1 : FM][M16 ? 1 : FN];
  float4v_t acc16[M16 ? 2 * FM : 1][M16 ? 2 * FN : 1];
#pragma unroll
  for (int fm = 0; fm < (M16 ? 1 : FM); ++fm)
#pragma unroll
    for (int fn = 0; fn < (M16 ? 1 : FN); ++fn)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[fm][fn][v] = 0.f;
#pragma unroll
  for (int rt = 0; rt < (M16 ? 2 * FM : 1); ++rt)
#pragma unroll
    for (int ct = 0; ct < (M16 ? 2 * FN : 1); ++ct) acc16[rt][ct] = float4v_t{0.f, 0.f, 0.f, 0.f};

  const int stages_total = (p.k + kStageK - 1) / kStageK;
  const int chunks = (stages_total + kStages - 1) / kStages;
  // K split over workgroups: this one multiplies chunks [chunk_begin, chunk_end) and writes to its own slice of d
  const int chunk_begin = blockIdx.y * p.chunks_per_split;  // the launcher makes every split non-empty
  const int chunk_end = chunk_begin + p.chunks_per_split < chunks ? chunk_begin + p.chunks_per_split : chunks;
  char* const d_out = reinterpret_cast<char*>(p.d) + (size_t)blockIdx.y * p.m * p.n * (p.d_f16 ? 2 : 4);
  // Two K groups: with an even number of row fragments each group finishes half of them (it hands the other half of
  // its sums to the other group); otherwise the second group hands everything to the first and stores nothing.
  constexpr bool kSplitEpilogue = KG == 2 && FM % 2 == 0;
  const int row_limit = (kg == 0 || kSplitEpilogue) ? p.m : 0;
  auto finishes = [&](int fm) __attribute__((always_inline)) { return !kSplitEpilogue || (fm >= FM / 2) == (kg == 1); };

  if constexpr (DMA) {
    // ---- asynchronous copy pattern for B: NL 16-byte copies per thread per stage ----
    // copy i of wavefront w fills LDS slots [(NW i + w) * 64, +64) of the stage; slot = (row, physical chunk).
    // Global address = wave-uniform base of the stage + per-lane byte offset.
    uint32_t b_off[NL];
    int copy_row[NL];  // first K row of the stage that copy i carries
    uint32_t lds_dst[NL];
    const uint32_t smem_base = lds_offset_of(smem);
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int slot = (NW * i + wave) * 64 + lane;
      if constexpr (TOKENS) {
        // slot = (token of the tile, physical piece): fetches K values [8 lc, 8 lc + 8) of the stage for that token
        int token = slot / 8;
        const int lc = (slot % 8) ^ token_swizzle(token);
        if (n0 + token >= p.n) token = 0;  // tokens past the end: any valid address will do, the results are not stored
        b_off[i] = (uint32_t)(token * p.k + 8 * lc) * 2u;  // the launcher checks that BN * k * 2 fits 32 bits
        copy_row[i] = 8 * lc;
      } else {
        const int row = slot / CH, pc = slot % CH;
        const int lc = pc ^ chunk_swizzle<BN>(row);
        int col = 8 * lc;
        if (n0 + col >= p.ldb) col = 0;  // columns past the row: any valid address will do, the results are not stored
        b_off[i] = (uint32_t)(row * p.ldb + col) * 2u;
        copy_row[i] = row;
      }
      lds_dst[i] = smem_base + (NW * i + wave) * 1024;
    }
    const int k_inside = RAGGED ? p.k - 1 : p.k;  // RAGGED: the stage of B's last row takes the general form of the copies
    const char* const last_piece = reinterpret_cast<const char*>(p.b) + (size_t)p.k * p.ldb * 2 - 16;
    // the piece of stage `stage` that was moved back, if there is one and this wavefront copied it
    auto mend_stage = [&](int stage) __attribute__((always_inline)) {
      const int row = (p.k - 1) % kStageK, piece = (p.n - 1 - n0) / 8, slot = row * CH + (piece ^ chunk_swizzle<BN>(row));
      if (!RAGGED || stage != (p.k - 1) / kStageK || piece >= CH || slot / 64 % NW != wave) return;  // wave-uniform
      shift_piece(smem + (stage % kStages) * TS::STAGE_BYTES + slot * 16, n0 + 8 * piece + 8 - p.n, lane);
      wait_vmcnt_lgkm0<63>();
      asm volatile("" ::: "memory");
    };
    const size_t stage_stride = TOKENS ? (size_t)kStageK * 2 : (size_t)kStageK * p.ldb * 2;
    const char* b_stage = reinterpret_cast<const char*>(p.b) + (TOKENS ? (size_t)n0 * p.k * 2 : (size_t)n0 * 2) +
                          (size_t)chunk_begin * kStages * stage_stride;  // advances one stage per copy
    const char* zeros = reinterpret_cast<const char*>(g_zero16);
    int next_k0 = chunk_begin * kChunkK;  // first K row of the next stage to copy
    // Rows at or past K are copied from a block of zeros, so stages past the end of K (the ring always runs
    // whole chunks of four stages) and the padding of the prepared operand contribute nothing, and the
    // number of copies in flight, which the vmcnt waits rely on, is the same in every iteration.
    auto issue_b = [&](int ring) {
      if (next_k0 + kStageK <= k_inside) {  // wave-uniform: a full stage
#pragma unroll
        for (int i = 0; i < NL; ++i) lds_dma16_base(b_stage, b_off[i], lds_dst[i] + ring * TS::STAGE_BYTES);
      } else {
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          uint32_t off = b_off[i];
          asm volatile("" : "+v"(off));  // keeps the 64-bit addresses out of the registers of the other path
          const char* src = b_stage + off;
          if (RAGGED && src > last_piece) src = last_piece;
          if (next_k0 + copy_row[i] >= p.k) src = zeros;
          lds_dma16(src, lds_dst[i] + ring * TS::STAGE_BYTES);
        }
      }
      b_stage += stage_stride;
      next_k0 += kStageK;
    };
    // the same for a stage that the caller knows to lie inside K: no branch, so that the K loop's body stays one block
    auto issue_b_full = [&](int ring) {
#pragma unroll
      for (int i = 0; i < NL; ++i) lds_dma16_base(b_stage, b_off[i], lds_dst[i] + ring * TS::STAGE_BYTES);
      b_stage += stage_stride;
      next_k0 += kStageK;
    };

    // ---- asynchronous copy pattern for A: the workgroup's BM/32 prepared blocks of one K chunk ----
    // LDS image = the blocks back to back; NA copies of 1 KiB per wavefront (the tail past the last block
    // re-copies the first block into padding so that every wavefront issues the same number of requests).
    constexpr int NA = TS::NA;
    char* a_lds = smem + TS::LDS_B_BYTES;
    uint32_t a_off[NA];
    uint32_t a_dst[NA];
    {
      const int rb0 = tile_m * (BM / kRowBlock);
#pragma unroll
      for (int j = 0; j < NA; ++j) {
        const int byte = (NW * j + wave) * 1024 + lane * 16;
        int blk = byte / kBlockBytes, off = byte % kBlockBytes;
        if (blk >= BM / kRowBlock) blk = 0;
        int rb = rb0 + blk;
        if (rb >= rb_total) rb = rb_total - 1;
        a_off[j] = (uint32_t)((size_t)rb * p.kc_total * kBlockBytes + off);  // the launcher checks it fits 32 bits
        a_dst[j] = smem_base + TS::LDS_B_BYTES + (NW * j + wave) * 1024;
      }
    }
    const char* a_chunk = reinterpret_cast<const char*>(p.prep) + (size_t)chunk_begin * kBlockBytes;  // advances one K chunk per copy
    int next_chunk = chunk_begin;
    auto advance_a = [&]() {
      if (next_chunk + 1 < chunks) a_chunk += kBlockBytes;  // past the last chunk the last one is copied again
      ++next_chunk;
    };
    auto issue_a = [&]() {
#pragma unroll
      for (int j = 0; j < NA; ++j) lds_dma16_base(a_chunk, a_off[j], a_dst[j]);
      advance_a();
    };
    const char* a_frag_lds[FM];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) a_frag_lds[fm] = a_lds + (wm * FM + fm) * kBlockBytes;

    // ---- the K loop ------------------------------------------------------------------------------------
    // Software pipeline over a ring of four 64-row stages of B (and one K chunk of A) in LDS. The SMFMACs of one K step
    // run while the B fragments and the expanded signs of the next step this wavefront multiplies are fetched; one
    // workgroup barrier per stage publishes the next stage and frees the ring slot of the one whose reads have all been
    // issued, into which the stage four ahead is then copied.
    // Request order: A(0) B(0) B(1) B(2) B(3) | chunk c: stage 0: A(c+1) B(4c+4)  stage 1: B(4c+5)
    //                                                     stage 2: B(4c+6)        stage 3: B(4c+7)
    // The order of the instructions inside each K-step region is written out and fenced: behind SMFMAC number `slot` of
    // the step comes that slot's share of the fetch work (fragment reads in the first half of the slots, the two
    // instructions per sign register spread evenly, the copies one by one), so that the two wavefronts of a SIMD, which
    // leave every barrier in lock-step, alternate on the matrix pipe instead of both fetching first; left to itself the
    // optimizer sinks the sign expansion past the barrier to the block of its first use.
    constexpr bool PINNED = FM * FN > 8;
    constexpr int SLOTS = FM * FN;
    constexpr int PIECES = TOKENS ? 2 * FN : 4 * FN;
    constexpr int PPS = (2 * PIECES + SLOTS - 1) / SLOTS > 1 ? (2 * PIECES + SLOTS - 1) / SLOTS : 1;  // pieces per slot
    auto read_piece = [&](int ring_slot, int ks, int r, u32x8_t* bv) __attribute__((always_inline)) {
      if constexpr (TOKENS) load_b_piece_tokens(wave_image + ring_slot * TS::STAGE_BYTES, ks, r, bv, piece_off);
      else load_b_piece<BN>(smem + ring_slot * TS::STAGE_BYTES, ks, r, bv, frag_off, lane_row_off);
    };
// the fetch work behind SMFMAC `slot`: pieces of the fragments of (RING, KS) into BV, registers of step FILL_STEP of A_SRC into AV
#define ONEBIT_FETCH_SLOT(RING, KS, BV, FILL_STEP, A_SRC, AV)                                                      \
          _Pragma("unroll") for (int r = 0; r < PIECES; ++r)                                                        \
            if (r / PPS == slot) read_piece((RING), (KS), r, BV);                                                   \
          _Pragma("unroll") for (int g = 0; g < 4 * FM; ++g)                                                        \
            if (g * FN / 4 == slot) AV[g / 4][g % 4] = expand_sign_register<(FILL_STEP)>(A_SRC[g / 4], one, g % 4);
// the copies of stage S + 4 (and of the next chunk of A) behind SMFMAC `slot`: one by one when the stage is known to lie
// inside K (A first, same request order), else all behind the first SMFMAC through the general, branching form.
// The copies are spread evenly over the region's slots: the wavefronts of a workgroup leave the barrier together, a
// compute unit's address path takes one 16-byte-per-lane copy instruction per 16 clocks, and copies issued back to back
// by every wavefront at once queue up there and hold the issuing wavefronts.
#define ONEBIT_COPY_SLOT(S, ISSUE_A)                                                                               \
          if constexpr (FULL) {                                                                                    \
            constexpr int COPIES = ((ISSUE_A) ? NA : 0) + NL, CPS = (COPIES + SLOTS - 1) / SLOTS;                  \
            constexpr int SPREAD = COPIES <= SLOTS ? SLOTS / COPIES : 1;  /* slots from one copy to the next */    \
            _Pragma("unroll") for (int c = 0; c < COPIES; ++c)                                                     \
              if ((c / CPS) * SPREAD == slot) {                                                                    \
                const int i = c - ((ISSUE_A) ? NA : 0);                                                            \
                if (i < 0) lds_dma16_base(a_chunk, a_off[c], a_dst[c]);                                            \
                else lds_dma16_base(b_stage, b_off[i], lds_dst[i] + (S) * TS::STAGE_BYTES);                        \
              }                                                                                                    \
            if (slot == ((COPIES - 1) / CPS) * SPREAD) {                                                           \
              if (ISSUE_A) advance_a();                                                                            \
              b_stage += stage_stride;                                                                             \
              next_k0 += kStageK;                                                                                  \
            }                                                                                                      \
            __builtin_amdgcn_sched_barrier(0);                                                                     \
          } else if (slot == 0) {                                                                                  \
            if (ISSUE_A) issue_a();                                                                                \
            issue_b(S);                                                                                            \
            __builtin_amdgcn_sched_barrier(0);                                                                     \
          }
    // chunk kc copies the stages of chunk kc + 1: they are whole while (kc + 2) * 256 <= K
    const int full_end = k_inside / kChunkK - 1 < chunk_end ? k_inside / kChunkK - 1 : chunk_end;

    if constexpr (M16) {
      // ---- 16x16x64 form of the K loop (one wavefront per SIMD, wave tile 128 x 128 = 8 x 8 tiles of 16 x 16) ----
      // One SMFMAC covers a whole 64-row stage. A-operand lane (row l % 16, group l / 16) holds the kept values of K
      // positions [16 g, 16 g + 16) of the stage, i.e. what lane row + 32 (g % 2) of the prepared block holds for K step
      // 2 S + g / 2; B-operand lane (column l % 16, group g) holds K rows 8 g ... 8 g + 7 of both 32-row halves.
      // First half of a stage (before the barrier): row tiles 0-3 against all column tiles, the signs of the next row
      // tile and of row tiles 4-7 expanded between the SMFMACs. Second half: column tile by column tile against row
      // tiles 4-7; a column tile's fragment registers are free after its four SMFMACs and take the next stage's
      // fragment, which the barrier has just published.
      constexpr int RT = 2 * FM, CT = 2 * FN;
      const int g16 = lane >> 4, c16 = lane & 15;
      const int brow = 8 * g16 + (c16 >> 2);  // + 0, 4, 32, 36
      const int brow_off = brow * (BN * 2);
      int ct_off[CT];
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
        ct_off[ct] = (((2 * (wn * CT + ct) + ((c16 & 3) >> 1)) ^ chunk_swizzle<BN>(brow)) << 4) + (c16 & 1) * 8;
      // Token-major image (linear-layer form): the operand of token 16 ct + c16 is pieces g16 and 4 + g16 of its row, two plain
      // 16-byte reads (q = 0, 1); the swizzle of a token row depends on c16 alone, so the column tile is an immediate offset.
      const int token_piece = c16 * (kStageK * 2) + ((g16 ^ token_swizzle(c16)) << 4);
      auto read_b16 = [&](int ring_slot, int ct, int q, u32x8_t* bv) __attribute__((always_inline)) {
        if constexpr (TOKENS) {
          if (q < 2) {
            const u32x4_t t = *reinterpret_cast<const u32x4_t*>(smem + ring_slot * TS::STAGE_BYTES + ct * (16 * kStageK * 2) +
                                                                 (token_piece ^ (q << 6)));
            bv[ct][4 * q] = t.x; bv[ct][4 * q + 1] = t.y; bv[ct][4 * q + 2] = t.z; bv[ct][4 * q + 3] = t.w;
          }
          return;
        }
        const int row_const = 4 * (q & 1) + 32 * (q >> 1);
        const u32x2_t t = lds_read_tr16(smem + ring_slot * TS::STAGE_BYTES + brow_off + row_const * (BN * 2) + ct_off[ct]);
        bv[ct][2 * q] = t.x;
        bv[ct][2 * q + 1] = t.y;
      };
      // per row tile: metadata of stages 0,1 and 2,3 (16 bits each, chosen by ABID), sign words of stages 0,1 and 2,3
      struct ATile { uint32_t idx01, idx23, w01, w23; };
      const uint32_t half_select = (g16 >> 1) ? 0x07060302u : 0x05040100u;
      const int sign_shift = 4 * (g16 >> 1);
      // A row tile's operands of one chunk in two steps, so that the LDS latency of the first lies under SMFMACs: the
      // holder lane's 24 bytes as they are, then the selection of this lane's 16 index bits per stage and the shift
      // of its sign words.
      struct ARaw { u32x4_t meta; u32x2_t sign; };
      auto load_a_raw = [&](int rt) __attribute__((always_inline)) {
        const char* block = a_frag_lds[rt >> 1];
        const int holder = c16 + 16 * (rt & 1) + 32 * (g16 & 1);
        ARaw r;
        r.meta = *reinterpret_cast<const u32x4_t*>(block + holder * 16);
        r.sign = *reinterpret_cast<const u32x2_t*>(block + kSignOffset + holder * 8);
        return r;
      };
      auto finish_a = [&](const ARaw& r) __attribute__((always_inline)) {
        ATile t;
        t.idx01 = __builtin_amdgcn_perm(r.meta.y, r.meta.x, half_select);
        t.idx23 = __builtin_amdgcn_perm(r.meta.w, r.meta.z, half_select);
        t.w01 = r.sign.x << sign_shift;
        t.w23 = r.sign.y << sign_shift;
        return t;
      };
      auto gather_a = [&](int rt) __attribute__((always_inline)) { return finish_a(load_a_raw(rt)); };
      // register p (kept values 2p, 2p+1) of the expanded signs of stage S
      auto expand16 = [&](const ATile& t, int S, int p_) __attribute__((always_inline)) {
        const uint32_t w = S < 2 ? t.w01 : t.w23;
        uint32_t v = ((w << (8 * (S & 1) + p_)) & 0x80008000u) | one;
        asm volatile("" : "+v"(v));
        return v;
      };
      auto mma16 = [&](float4v_t& c, const u32x4_t& av, const u32x8_t& bv, const ATile& t, int S) __attribute__((always_inline)) {
        const uint32_t idx = S < 2 ? t.idx01 : t.idx23;
        const half8_t a8 = __builtin_bit_cast(half8_t, av);
        const half16_t b16 = __builtin_bit_cast(half16_t, bv);
        // accumulators tied to accumulation registers, as in smfmac_step
        if constexpr (BF16) {
          if ((S & 1) == 0) asm("v_smfmac_f32_16x16x64_bf16 %0, %1, %2, %3" : "+a"(c) : "v"(a8), "v"(b16), "v"(idx));
          else asm("v_smfmac_f32_16x16x64_bf16 %0, %1, %2, %3 abid:1" : "+a"(c) : "v"(a8), "v"(b16), "v"(idx));
        } else if ((S & 1) == 0) asm("v_smfmac_f32_16x16x64_f16 %0, %1, %2, %3" : "+a"(c) : "v"(a8), "v"(b16), "v"(idx));
        else asm("v_smfmac_f32_16x16x64_f16 %0, %1, %2, %3 abid:1" : "+a"(c) : "v"(a8), "v"(b16), "v"(idx));
      };

      // wait states behind what a loop copies between registers, see smfmac_step
      auto settle16 = [&](u32x4_t& av, u32x8_t& bv, const ATile& t) __attribute__((always_inline)) {
        asm volatile("s_nop 1" : "+v"(av), "+v"(bv) : "v"(t.idx01));
      };

      issue_a();
#pragma unroll
      for (int s = 0; s < kStages; ++s) issue_b(s);
      ATile a_cur[RT];
      u32x8_t bv[CT];
      u32x4_t av_roll[2], av_hi[RT / 2];
      wait_vmcnt<3 * NL>();  // A(0) and B(0) have landed
      if constexpr (RAGGED) mend_stage(chunk_begin * kStages);
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) a_cur[rt] = gather_a(rt);
#pragma unroll
      for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int q = 0; q < 4; ++q) read_b16(0, ct, q, bv);
#pragma unroll
      for (int p_ = 0; p_ < 4; ++p_) av_roll[0][p_] = expand16(a_cur[0], 0, p_);

      auto chunk_body = [&](auto full_tag, int kc) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_tag)::value;
        constexpr int SLOTS = RT / 2 * CT;  // SMFMACs per half stage (shadows the 32x32x32 form's count for the copy macro)
        auto stage = [&](auto s_tag, auto wait_tag, auto issue_a_tag) __attribute__((always_inline)) {
          constexpr int S = decltype(s_tag)::value;
          constexpr int WAITCNT = decltype(wait_tag)::value;
          constexpr bool ISSUE_A = decltype(issue_a_tag)::value;
          // first half: row tiles 0-3
#pragma unroll
          for (int rt = 0; rt < RT / 2; ++rt)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
              if (S == 0 && rt == 0 && ct == 0) settle16(av_roll[0], bv[0], a_cur[0]);
              mma16(acc16[rt][ct], av_roll[rt & 1], bv[ct], a_cur[rt], S);
              __builtin_amdgcn_sched_barrier(0);
              // this slot's share of the eight registers to expand: the next row tile's four, then row tile 4 + rt's four
#pragma unroll
              for (int e = ct * 8 / CT; e < (ct + 1) * 8 / CT; ++e) {
                if (e < 4) {
                  if (rt + 1 < RT / 2) av_roll[(rt + 1) & 1][e] = expand16(a_cur[rt + 1], S, e);
                } else {
                  av_hi[rt][e - 4] = expand16(a_cur[RT / 2 + rt], S, e - 4);
                }
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          wait_vmcnt_lgkm0<WAITCNT>();  // copies of stage S+1 landed
          if constexpr (RAGGED && !FULL) mend_stage(kc * kStages + S + 1);
          __builtin_amdgcn_s_barrier();
          // Last stage of a chunk: the next chunk of A is readable after this stage's barrier. Row tiles 0-3 are done
          // with this chunk: their holder lanes' bytes are requested right here and turned into operands behind the
          // SMFMACs of column tile 1, by when they have arrived; row tiles 4-7 are multiplied to the end of the stage:
          // requested behind column tile 5, turned into operands after the last SMFMAC.
          constexpr bool LAST = S == kStages - 1;
          ARaw a_raw[RT / 2];
          if constexpr (LAST) {
#pragma unroll
            for (int rt = 0; rt < RT / 2; ++rt) a_raw[rt] = load_a_raw(rt);
            __builtin_amdgcn_sched_barrier(0);
          }
          // second half: column tile by column tile against row tiles 4-7
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int rl = 0; rl < RT / 2; ++rl) {
              const int slot = ct * (RT / 2) + rl;
              mma16(acc16[RT / 2 + rl][ct], av_hi[rl], bv[ct], a_cur[RT / 2 + rl], S);
              __builtin_amdgcn_sched_barrier(0);
              ONEBIT_COPY_SLOT(S, ISSUE_A)
              // the fragment of column tile ct - 1 for the next stage, one read behind each of this tile's SMFMACs
              if (ct >= 1) read_b16((S + 1) % kStages, ct - 1, rl, bv);
              if constexpr (LAST) {
                if (ct == 1) a_cur[rl] = finish_a(a_raw[rl]);
                if (ct == CT - 3) a_raw[rl] = load_a_raw(RT / 2 + rl);
              }
              // signs of row tile 0 of the next stage
              if (ct == CT - 1) av_roll[0][rl] = expand16(a_cur[0], (S + 1) % kStages, rl);
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
          for (int q = 0; q < 4; ++q) read_b16((S + 1) % kStages, CT - 1, q, bv);
          if constexpr (LAST) {
#pragma unroll
            for (int rl = 0; rl < RT / 2; ++rl) a_cur[RT / 2 + rl] = finish_a(a_raw[rl]);
          }
        };
        using std::integral_constant;
        stage(integral_constant<int, 0>{}, integral_constant<int, 2 * NL>{}, std::true_type{});        // waits for B(4c+1)
        stage(integral_constant<int, 1>{}, integral_constant<int, 2 * NL + NA>{}, std::false_type{});  // B(4c+2)
        stage(integral_constant<int, 2>{}, integral_constant<int, 2 * NL + NA>{}, std::false_type{});  // B(4c+3)
        stage(integral_constant<int, 3>{}, integral_constant<int, 2 * NL>{}, std::false_type{});       // B(4c+4)
      };
      int kc = chunk_begin;
      for (; kc < full_end; ++kc) chunk_body(std::true_type{}, kc);
      for (; kc < chunk_end; ++kc) chunk_body(std::false_type{}, kc);
      wait_vmcnt<0>();  // drain the copies issued past the end before the LDS is released
    } else if constexpr (KG == 1) {
      // The barrier sits in the middle of each stage s: it publishes stage s+1 (read right after it) and frees the ring
      // slot of stage s (all of its reads were issued in the first half).
      issue_a();
#pragma unroll
      for (int s = 0; s < kStages; ++s) issue_b(s);

      AChunk a_cur[FM], a_next[FM];
      u32x8_t bv0[FN], bv1[FN];
      u32x4_t av0[FM], av1[FM];
      wait_vmcnt<3 * NL>();  // A(0) and B(0) have landed
      if constexpr (RAGGED) mend_stage(chunk_begin * kStages);
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) a_cur[fm] = load_a_chunk_lds(a_frag_lds[fm], lane);
#pragma unroll
      for (int r = 0; r < PIECES; ++r) read_piece(0, 0, r, bv0);
#pragma unroll
      for (int g = 0; g < 4 * FM; ++g) av0[g / 4][g % 4] = expand_sign_register<0>(a_cur[g / 4], one, g % 4);

#define ONEBIT_FUSED_STAGE(S, WAITCNT, ISSUE_A)                                                                  \
      {                                                                                                            \
        mfma_frags_fused<2 * (S), PINNED, BF16>(a_cur, av0, bv0, acc, [&](int slot) __attribute__((always_inline)) {     \
          ONEBIT_FETCH_SLOT((S), 1, bv1, 2 * (S) + 1, a_cur, av1)                                                  \
        });                                                                                                        \
        wait_vmcnt_lgkm0<(WAITCNT)>(); /* copies of stage S+1 landed; this wavefront's reads of stage S returned */ \
        if constexpr (RAGGED && !FULL) mend_stage(kc * kStages + (S) + 1);                                                   \
        __builtin_amdgcn_s_barrier();                                                                              \
        if constexpr ((S) == kStages - 1) {                                                                        \
          /* the next chunk of A is readable after this stage's barrier */                                         \
          _Pragma("unroll") for (int fm = 0; fm < FM; ++fm) a_next[fm] = load_a_chunk_lds(a_frag_lds[fm], lane);   \
          __builtin_amdgcn_sched_barrier(0);                                                                       \
        }                                                                                                          \
        mfma_frags_fused<2 * (S) + 1, PINNED, BF16>(a_cur, av1, bv1, acc, [&](int slot) __attribute__((always_inline)) { \
          ONEBIT_COPY_SLOT(S, ISSUE_A)                                                                             \
          if constexpr ((S) < kStages - 1) {                                                                       \
            ONEBIT_FETCH_SLOT((S) + 1, 0, bv0, 2 * (S) + 2, a_cur, av0)                                            \
          } else {                                                                                                 \
            ONEBIT_FETCH_SLOT(0, 0, bv0, 0, a_next, av0)                                                           \
          }                                                                                                        \
        });                                                                                                        \
        if constexpr ((S) == kStages - 1) {                                                                        \
          _Pragma("unroll") for (int fm = 0; fm < FM; ++fm) a_cur[fm] = a_next[fm];                                \
        }                                                                                                          \
      }

      auto chunk_body = [&](auto full_tag, int kc) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_tag)::value;  // the four stages copied during this chunk lie inside K
        ONEBIT_FUSED_STAGE(0, 2 * NL, true)        // waits for B(4c+1); newer requests: B(4c+2), B(4c+3)
        ONEBIT_FUSED_STAGE(1, 2 * NL + NA, false)  // waits for B(4c+2); newer: B(4c+3), A(c+1), B(4c+4)
        ONEBIT_FUSED_STAGE(2, 2 * NL + NA, false)  // waits for B(4c+3); newer: A(c+1), B(4c+4), B(4c+5)
        ONEBIT_FUSED_STAGE(3, 2 * NL, false)       // waits for B(4c+4), which is newer than A(c+1)
      };
      int kc = chunk_begin;
      for (; kc < full_end; ++kc) chunk_body(std::true_type{}, kc);
      for (; kc < chunk_end; ++kc) chunk_body(std::false_type{}, kc);
#undef ONEBIT_FUSED_STAGE
      wait_vmcnt<0>();  // drain the copies issued past the end before the LDS is released
    } else {
      // Two K groups: this wavefront multiplies K step KGV of every stage. One barrier per stage: before it the
      // wavefront waits for its fragments of stage S (read during stage S - 1) and for the copies of stage S + 1; after
      // it the ring slot of stage S is free for stage S + 4 and stage S + 1 is readable. Same request order and wait
      // counts as the one-group pipeline.
      auto run = [&](auto group_tag) __attribute__((always_inline)) {
        constexpr int KGV = decltype(group_tag)::value;
        issue_a();
#pragma unroll
        for (int s = 0; s < kStages; ++s) issue_b(s);
        AChunk a_cur[FM], a_next[FM];
        u32x8_t bv_even[FN], bv_odd[FN];
        u32x4_t av_even[FM], av_odd[FM];
        wait_vmcnt<3 * NL>();  // A(0) and B(0) have landed
      if constexpr (RAGGED) mend_stage(chunk_begin * kStages);
        __builtin_amdgcn_s_barrier();
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) a_cur[fm] = load_a_chunk_lds(a_frag_lds[fm], lane);
#pragma unroll
        for (int r = 0; r < PIECES; ++r) read_piece(0, KGV, r, bv_even);
#pragma unroll
        for (int g = 0; g < 4 * FM; ++g) av_even[g / 4][g % 4] = expand_sign_register<KGV>(a_cur[g / 4], one, g % 4);
#define ONEBIT_GROUP_STAGE(S, WAITCNT, ISSUE_A, BV, AV, BV_NEXT, AV_NEXT)                                         \
        {                                                                                                        \
          wait_vmcnt_lgkm0<(WAITCNT)>();                                                                         \
          if constexpr (RAGGED && !FULL) mend_stage(kc * kStages + (S) + 1);                                               \
          __builtin_amdgcn_s_barrier();                                                                          \
          if constexpr ((S) == kStages - 1) {                                                                    \
            _Pragma("unroll") for (int fm = 0; fm < FM; ++fm) a_next[fm] = load_a_chunk_lds(a_frag_lds[fm], lane); \
            __builtin_amdgcn_sched_barrier(0);                                                                   \
          }                                                                                                      \
          mfma_frags_fused<2 * (S) + KGV, false, BF16>(a_cur, AV, BV, acc, [&](int slot) __attribute__((always_inline)) { \
            ONEBIT_COPY_SLOT(S, ISSUE_A)                                                                         \
            if constexpr ((S) < kStages - 1) {                                                                   \
              ONEBIT_FETCH_SLOT((S) + 1, KGV, BV_NEXT, 2 * ((S) + 1) + KGV, a_cur, AV_NEXT)                      \
            } else {                                                                                             \
              ONEBIT_FETCH_SLOT(0, KGV, BV_NEXT, KGV, a_next, AV_NEXT)                                           \
            }                                                                                                    \
          });                                                                                                    \
          if constexpr ((S) == kStages - 1) {                                                                    \
            _Pragma("unroll") for (int fm = 0; fm < FM; ++fm) a_cur[fm] = a_next[fm];                            \
          }                                                                                                      \
        }
        auto chunk_body = [&](auto full_tag, int kc) __attribute__((always_inline)) {
          constexpr bool FULL = decltype(full_tag)::value;
          ONEBIT_GROUP_STAGE(0, 2 * NL, true, bv_even, av_even, bv_odd, av_odd)
          ONEBIT_GROUP_STAGE(1, 2 * NL + NA, false, bv_odd, av_odd, bv_even, av_even)
          ONEBIT_GROUP_STAGE(2, 2 * NL + NA, false, bv_even, av_even, bv_odd, av_odd)
          ONEBIT_GROUP_STAGE(3, 2 * NL, false, bv_odd, av_odd, bv_even, av_even)
        };
        int kc = chunk_begin;
        for (; kc < full_end; ++kc) chunk_body(std::true_type{}, kc);
        for (; kc < chunk_end; ++kc) chunk_body(std::false_type{}, kc);
#undef ONEBIT_GROUP_STAGE
        wait_vmcnt<0>();  // drain the copies issued past the end before the LDS is released
      };
      if (kg == 0) run(std::integral_constant<int, 0>{});
      else run(std::integral_constant<int, 1>{});
#undef ONEBIT_FETCH_SLOT
#undef ONEBIT_COPY_SLOT
      smfmac_drain();
      __syncthreads();  // the stage ring is free
      if constexpr (kSplitEpilogue) {
        // each group keeps half of the row fragments and passes its sums for the other half through the ring, lane for
        // lane: group 0 finishes fragments [0, FM / 2), group 1 the rest
        constexpr int HALF = FM / 2, PER_WAVE = HALF * FN * 16 * 64;
        float* const given = reinterpret_cast<float*>(smem) + (size_t)wave * PER_WAVE + lane;
        const float* const taken =
            reinterpret_cast<const float*>(smem) + (size_t)(wave_in_group + (1 - kg) * WM * WN) * PER_WAVE + lane;
#pragma unroll
        for (int fm = 0; fm < HALF; ++fm)
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              if (kg == 0) given[((fm * FN + fn) * 16 + v) * 64] = acc[HALF + fm][fn][v];
              else given[((fm * FN + fn) * 16 + v) * 64] = acc[fm][fn][v];
            }
        __syncthreads();
#pragma unroll
        for (int fm = 0; fm < HALF; ++fm)
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
              if (kg == 0) acc[fm][fn][v] += taken[((fm * FN + fn) * 16 + v) * 64];
              else acc[HALF + fm][fn][v] += taken[((fm * FN + fn) * 16 + v) * 64];
            }
      } else {
        // the second group's partial tile goes to the first, lane for lane
        float* const handover = reinterpret_cast<float*>(smem) + (size_t)wave_in_group * (FM * FN * 16 * 64) + lane;
        if (kg == 1) {
#pragma unroll
          for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn)
#pragma unroll
              for (int v = 0; v < 16; ++v) handover[((fm * FN + fn) * 16 + v) * 64] = acc[fm][fn][v];
        }
        __syncthreads();
        if (kg == 0) {
#pragma unroll
          for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn)
#pragma unroll
              for (int v = 0; v < 16; ++v) acc[fm][fn][v] += handover[((fm * FN + fn) * 16 + v) * 64];
        }
      }
      __syncthreads();  // the epilogue's scratch overlaps the handover area
    }
  } else {
    // ---- generic path: any N, any K % 32 == 0, any alignment. One stage at a time, element copies. ----
    for (int kc = chunk_begin; kc < chunk_end; ++kc) {
      AChunk a_cur[FM];
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) a_cur[fm] = load_a_chunk(a_block[fm] + (size_t)kc * kBlockBytes, lane);
      auto fill = [&](int stage) {
        const int k0 = (kc * kStages + stage) * kStageK;
        __syncthreads();
        for (int idx = tid; idx < kStageK * BN; idx += 64 * NW) {
          const int row = idx / BN, col = idx % BN;
          _Float16 v = (_Float16)0.f;
          if (k0 + row < p.k && n0 + col < p.n) v = p.b[(size_t)(k0 + row) * p.n + n0 + col];
          const int lc = (col >> 3) ^ chunk_swizzle<BN>(row);
          *reinterpret_cast<_Float16*>(smem + row * (BN * 2) + (lc << 4) + (col & 7) * 2) = v;
        }
        __syncthreads();
      };
      if (kc * kStages + 0 < stages_total) { fill(0); compute_stage<FM, FN, BN, 0>(smem, a_cur, acc, frag_off, lane_row_off, one); }
      if (kc * kStages + 1 < stages_total) { fill(1); compute_stage<FM, FN, BN, 1>(smem, a_cur, acc, frag_off, lane_row_off, one); }
      if (kc * kStages + 2 < stages_total) { fill(2); compute_stage<FM, FN, BN, 2>(smem, a_cur, acc, frag_off, lane_row_off, one); }
      if (kc * kStages + 3 < stages_total) { fill(3); compute_stage<FM, FN, BN, 3>(smem, a_cur, acc, frag_off, lane_row_off, one); }
    }
  }

  smfmac_drain();
  if constexpr (TOKENS) {
    // ---- epilogue of the linear-layer form: y[token][row] = acc + bias[row], fp16 (RNE) or fp32 ----
    const int token_lane = lane & 31;
    // the four bias values from a row on that is a multiple of four, any four where the row is past the end (never stored);
    // p.bias is not null
    auto bias_vector = [&](int row, float* out) __attribute__((always_inline)) {
      const size_t at = row < p.m ? row : 0;
      if (p.bias_type != kF32) {
        const u32x2_t words = *reinterpret_cast<const u32x2_any_t*>(reinterpret_cast<const uint16_t*>(p.bias) + at);
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          const float2v_t v = unpack_pair(words[e / 2], p.bias_type);
          out[e] = v.x; out[e + 1] = v.y;
        }
      } else {
        const u32x4_t v = *reinterpret_cast<const u32x4_any_t*>(reinterpret_cast<const float*>(p.bias) + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = __builtin_bit_cast(float, (uint32_t)v[e]);
      }
    };
    // A tile's sums out of the accumulation registers, here: left to itself the compiler moves all 256 in front of the branches
    // between the forms below, where they do not fit (44 registers spilled).
    auto take_sums = [&](const float4v_t& sums) __attribute__((always_inline)) {
      float4v_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float x;
        asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x) : "a"((float)sums[e]));
        v[e] = x;
      }
      return v;
    };
    // Each wavefront turns its tile through a private LDS scratch, after which every lane stores 16 bytes of one token's
    // row of y.
    __syncthreads();  // every wavefront is done with the stage ring, which becomes the scratch
    constexpr int WCOLS = FN * 32;
    char* const scratch = smem + wave * (WCOLS * 128);
    const int g16 = lane >> 4, c16 = lane & 15;
    if (p.d_f16) {
      // 16-bit result: the bias is added and the sum rounded in the accumulator layout, where four registers of a lane are
      // four consecutive rows of its token, 8 bytes of y. A turn takes as many tokens as the scratch holds with all of the
      // wavefront's rows, up to 256 bytes of a token, so that the stores write whole lines of y; one 32-row block at a time
      // they wrote halves of lines, of sixteen tokens per instruction. us, that -> this (fp16 | bf16; the 16x16x64 tile went
      // through the scratch as floats before, and spilled): 8192 x 8192 with 8192 tokens 438 -> 423 | 424 -> 406, 11008 x 4096
      // with 4096 172 -> 164 | 166 -> 154, 4096 x 4096 with 4096 62.1 -> 57.6 | 59.6 -> 55.3; fewer tiles than compute units
      // 35.2 -> 34.9 (2048 tokens).
      constexpr int FRAGS = kSplitEpilogue ? FM / 2 : FM;  // of the rows that this wavefront finishes
      constexpr int PIECES = 4 * FRAGS;                    // 16-byte pieces of a token's rows
      constexpr int TURN = FRAGS > 2 ? 2 * WCOLS / FRAGS : WCOLS;
      static_assert(TURN * PIECES <= WCOLS * 8 && WCOLS % TURN == 0 && TURN % (M16 ? 16 : 32) == 0, "tokens per turn");
      // byte offset of the 8-byte slot `slot` (four rows) of the turn's token t; lanes of sixteen consecutive tokens that
      // write one slot, or read one token, meet in no bank
      auto slot_at = [&](int t, int slot) __attribute__((always_inline)) {
        return t * (PIECES * 16) + ((((slot >> 1) ^ ((t * PIECES >> 4) & (PIECES - 1))) << 4) | ((slot & 1) << 3));
      };
      auto turns = [&](auto bias_tag) __attribute__((always_inline)) {
        constexpr bool BIAS = decltype(bias_tag)::value;
        constexpr int GROUPS = M16 ? 2 : 4;  // of four rows, per 32-row block and lane
        // 32x32x32 form: registers 4 q ... 4 q + 3 are rows 8 q + 4 (lane / 32) on; 16x16x64 form: the registers of tile
        // (2 fm + q, ct) are rows 16 q + 4 (lane / 16) on of token 16 ct + lane % 16
        auto slot_of = [&](int q) __attribute__((always_inline)) { return M16 ? 4 * q + g16 : 2 * q + gb; };
        float bias[BIAS ? FM * GROUPS : 1][4];
        if constexpr (BIAS) {
#pragma unroll
          for (int i = 0; i < FM * GROUPS; ++i)
            if (finishes(i / GROUPS)) bias_vector(row0 + i / GROUPS * 32 + 4 * slot_of(i % GROUPS), bias[i]);
        }
        const int lane_piece = lane % PIECES, lane_token = lane / PIECES;
        const int row = row0 + (kSplitEpilogue ? kg * FRAGS * 32 : 0) + 8 * lane_piece;
        const int tokens = row < row_limit ? p.n : 0;
        int token = col0 + lane_token;
        _Float16* y = reinterpret_cast<_Float16*>(d_out) + (size_t)token * p.m + row;
        const size_t step = (size_t)(64 / PIECES) * p.m;
#pragma unroll
        for (int first = 0; first < WCOLS; first += TURN) {
#pragma unroll
          for (int fm = 0; fm < FM; ++fm) {
            if (!finishes(fm)) continue;  // the other K group stores this fragment
#pragma unroll
            for (int q = 0; q < GROUPS; ++q) {
              const int slot = slot_of(q);
              auto put = [&](int t, float x0, float x1, float x2, float x3) __attribute__((always_inline)) {
                if constexpr (BIAS) {
                  const float* const b4 = bias[fm * GROUPS + q];
                  x0 += b4[0]; x1 += b4[1]; x2 += b4[2]; x3 += b4[3];
                }
                *reinterpret_cast<u32x2_t*>(scratch + slot_at(t, 8 * (fm % FRAGS) + slot)) =
                    u32x2_t{round_pair<BF16>(x0, x1), round_pair<BF16>(x2, x3)};
              };
              if constexpr (M16) {
#pragma unroll
                for (int ct = first / 16; ct < (first + TURN) / 16; ++ct) {
                  const float4v_t v = take_sums(acc16[2 * fm + q][ct]);
                  put(ct * 16 - first + c16, v[0], v[1], v[2], v[3]);
                }
              } else {
#pragma unroll
                for (int fn = first / 32; fn < (first + TURN) / 32; ++fn)
                  put(fn * 32 - first + token_lane, acc[fm][fn][4 * q], acc[fm][fn][4 * q + 1], acc[fm][fn][4 * q + 2],
                      acc[fm][fn][4 * q + 3]);
              }
            }
          }
#pragma unroll
          for (int it = 0; it < TURN * PIECES / 64; ++it) {
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(scratch + slot_at(it * (64 / PIECES) + lane_token, 2 * lane_piece));
            if (token < tokens) *reinterpret_cast<u32x4_any_t*>(y) = v;
            token += 64 / PIECES;
            y += step;
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (p.bias) turns(std::true_type{});
      else turns(std::false_type{});
      return;
    }
    // fp32 result, one 32-row block at a time: [token][32 rows], a lane's four registers of one group one 16-byte slot (slot
    // s = rows 4 s ... 4 s + 3, stored at position s ^ (token % 8) against bank conflicts).
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      if (!finishes(fm)) continue;  // the other K group stores this fragment
      if constexpr (M16) {
        // slot 4 rh + lane / 16 of token 16 ct + lane % 16
#pragma unroll
        for (int rh = 0; rh < 2; ++rh)
#pragma unroll
          for (int ct = 0; ct < 2 * FN; ++ct) {
            const float4v_t v4 = take_sums(acc16[2 * fm + rh][ct]);
            *reinterpret_cast<float4*>(scratch + (ct * 16 + c16) * 128 + (((4 * rh + g16) ^ token_swizzle(c16)) << 4)) =
                float4{v4[0], v4[1], v4[2], v4[3]};
          }
      } else {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<float4*>(scratch + (fn * 32 + token_lane) * 128 + (((2 * q + gb) ^ token_swizzle(token_lane)) << 4)) =
                float4{acc[fm][fn][4 * q], acc[fm][fn][4 * q + 1], acc[fm][fn][4 * q + 2], acc[fm][fn][4 * q + 3]};
      }
      const int j = lane % 8, row = row0 + fm * 32 + 4 * j;
      float bias4[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias) bias_vector(row, bias4);
#pragma unroll
      for (int it = 0; it < WCOLS * 8 / 64; ++it) {
        const int t = it * 8 + lane / 8, token = col0 + t;
        const float4 v4 = *reinterpret_cast<const float4*>(scratch + t * 128 + ((j ^ token_swizzle(t)) << 4));
        if (token < p.n && row < row_limit)
          *reinterpret_cast<u32x4_any_t*>(reinterpret_cast<float*>(d_out) + (size_t)token * p.m + row) =
              __builtin_bit_cast(u32x4_t, float4{v4.x + bias4[0], v4.y + bias4[1], v4.z + bias4[2], v4.w + bias4[3]});
      }
    }
    return;
  }
  // ---- epilogue: D = alpha * acc + beta * C (csrc/kernel.h:27-31), fp16 (RNE) or fp32 output ----
  if constexpr (DMA) {
    // Coalesced form: each wavefront turns one 32-row block of its tile at a time through a private LDS
    // scratch (fp32, row-major) so that every lane then handles 16 bytes of one output row: C is read and D
    // written in full 128-byte segments instead of 64-byte (fp16) pieces per accumulator register.
    __syncthreads();  // every wavefront is done with the stage ring, which becomes the scratch
    constexpr int WCOLS = FN * 32;                   // columns of the wavefront's tile
    float* scratch = reinterpret_cast<float*>(smem) + wave * (32 * WCOLS);
    const int col_lane = lane & 31, row_lane = 4 * (lane >> 5);
    // Column swizzle of the scratch against bank conflicts, the same for rows of floats and for row pairs of packed
    // halves: line L keeps its 16-byte slots swapped in pairs when L is odd (two consecutive lines are read by one
    // group of sixteen lanes: they then touch different banks), and, with lines of 256 bytes or more, its two halves of
    // 128 bytes swapped when bit 2 (rows) or bit 1 (row pairs) of L is set (the upper half-wavefront writes the line
    // that many below the lower half's).
    constexpr int kHalfSwap = WCOLS >= 64 ? 32 : 0;
    // The accumulators of 32-row block fm into the scratch. 32x32x32 form: register v of fragment fn is row
    // 8 (v / 4) + 4 (lane / 32) + v % 4, column 32 fn + lane % 32; 16x16x64 form: register v of tile (2 fm + rh, ct) is
    // row 16 rh + 4 (lane / 16) + v, column 16 ct + lane % 16. In both, bit 2 of the row is one bit of the lane
    // (the writer's own half swap) and bit 0 of the row is bit 0 of v.
    const int g16 = lane >> 4, c16 = lane & 15;
    const int half_write = (M16 ? (g16 & 1) : (lane >> 5)) * kHalfSwap;
    auto store_rows = [&](int fm) __attribute__((always_inline)) {
      if constexpr (M16) {
#pragma unroll
        for (int rh = 0; rh < 2; ++rh)
#pragma unroll
          for (int ct = 0; ct < 2 * FN; ++ct)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              scratch[(16 * rh + 4 * g16 + v) * WCOLS + ((ct * 16 + c16) ^ half_write ^ ((v & 1) << 2))] =
                  acc16[2 * fm + rh][ct][v];
      } else {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            scratch[(8 * (v / 4) + row_lane + (v % 4)) * WCOLS + ((fn * 32 + col_lane) ^ half_write ^ ((v & 1) << 2))] =
                acc[fm][fn][v];
      }
    };
    auto read_swizzle = [&](int line, int half_bit) __attribute__((always_inline)) {
      return ((line & 1) << 2) ^ (((line >> half_bit) & 1) * kHalfSwap);
    };
    // Rows of C and D may start at any element (n is any number). Whole pieces of 8 halves or 4 floats are moved as
    // vectors at any alignment; what is left of the rows behind their last whole piece, element by element from the
    // scratch: sum_at(r, c) is the alpha-scaled sum of row r, column c of the block.
    auto cut_rows = [&](int row_base, int piece, auto&& sum_at) __attribute__((always_inline)) {
      const int tail = p.n - p.n % piece;
      if (tail == p.n || tail < col0 || tail >= col0 + WCOLS) return;  // wave-uniform
#pragma unroll 1
      for (int i = lane; i < 32 * 8; i += 64) {
        const int r = i >> 3, row = row_base + r, col = tail + (i & 7);
        if (row < row_limit && col < p.n) {
          const size_t o = (size_t)row * p.n + col;
          float x = sum_at(r, col - col0);
          if (p.beta != 0.f)
            x = x + p.beta * (p.c_f16 ? (float)reinterpret_cast<const _Float16*>(p.c)[o] : reinterpret_cast<const float*>(p.c)[o]);
          if (p.d_f16) reinterpret_cast<_Float16*>(d_out)[o] = (_Float16)x;
          else reinterpret_cast<float*>(d_out)[o] = x;
        }
      }
    };
    // The pieces of C that a lane will need for one 32-row block are requested together, before the block's sums
    // travel through the scratch, so that one memory latency per block is paid instead of one per piece.
    const bool use_c = p.beta != 0.f;
    if (p.d_f16 && !use_c && WCOLS >= 8) {
      // fp16 result without C: alpha * sum is rounded in the accumulator layout, where registers v and v + 1 (v even)
      // of a lane are rows r and r + 1 of one column; the two halves go through the scratch as one word (a quarter of
      // the LDS traffic of the fp32 form). A lane then reads eight such words (columns c .. c + 7 of a row pair),
      // separates low and high halves and stores 16 bytes of row r and 16 bytes of row r + 1.
      uint32_t* const words = reinterpret_cast<uint32_t*>(scratch);  // [16 row pairs][WCOLS]
      constexpr int PER_PAIR = WCOLS / 8;            // 8-column pieces per row pair
      constexpr int TASKS = 16 * PER_PAIR;           // (row pair, piece) per 32-row block
      constexpr int ITERS = (TASKS + 63) / 64;
      // alpha == 1 is tested once per wavefront, not per value: two copies of the loop
      auto packed_turn = [&](auto scale_tag) __attribute__((always_inline)) {
      constexpr bool SCALE = decltype(scale_tag)::value;
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) {
        if (!finishes(fm)) continue;  // the other K group stores this fragment
        const int row_base = row0 + fm * 32;
        auto pack = [&](float x0, float x1) __attribute__((always_inline)) {  // one packed conversion per register pair
          if constexpr (SCALE) return round_pair<false>(p.alpha * x0, p.alpha * x1);
          else return round_pair<false>(x0, x1);
        };
        if constexpr (M16) {
          // registers (0, 1) and (2, 3) of a tile: rows 16 rh + 4 (lane / 16) + 2 h and the next, row pair
          // 8 rh + 2 (lane / 16) + h
#pragma unroll
          for (int rh = 0; rh < 2; ++rh)
#pragma unroll
            for (int ct = 0; ct < 2 * FN; ++ct)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                words[(8 * rh + 2 * g16 + h) * WCOLS + ((ct * 16 + c16) ^ half_write ^ (h << 2))] =
                    pack(acc16[2 * fm + rh][ct][2 * h], acc16[2 * fm + rh][ct][2 * h + 1]);
        } else {
#pragma unroll
          for (int fn = 0; fn < FN; ++fn)
#pragma unroll
            for (int q = 0; q < 8; ++q)
              // rows 8 (q / 2) + 4 (lane / 32) + 2 (q % 2) and the next: row pair 4 (q / 2) + 2 (lane / 32) + q % 2
              words[(4 * (q / 2) + (row_lane >> 1) + (q & 1)) * WCOLS + ((fn * 32 + col_lane) ^ half_write ^ ((q & 1) << 2))] =
                  pack(acc[fm][fn][2 * q], acc[fm][fn][2 * q + 1]);
        }
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
          const int task = it * 64 + lane;
          if (TASKS % 64 != 0 && task >= TASKS) break;
          const int pair = task / PER_PAIR, c8 = (task % PER_PAIR) * 8;
          const int sw = read_swizzle(pair, 1);
          const u32x4_t lo = *reinterpret_cast<const u32x4_t*>(words + pair * WCOLS + (c8 ^ sw));
          const u32x4_t hi = *reinterpret_cast<const u32x4_t*>(words + pair * WCOLS + ((c8 + 4) ^ sw));
          const uint32_t d[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
          u32x4_t even_row, odd_row;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            even_row[j] = __builtin_amdgcn_perm(d[2 * j + 1], d[2 * j], 0x05040100u);  // low halves
            odd_row[j] = __builtin_amdgcn_perm(d[2 * j + 1], d[2 * j], 0x07060302u);   // high halves
          }
          const int row = row_base + 2 * pair, col = col0 + c8;
          if (col + 8 <= p.n) {
            _Float16* const out = reinterpret_cast<_Float16*>(d_out) + (size_t)row * p.n + col;
            if (row < row_limit) *reinterpret_cast<u32x4_any_t*>(out) = even_row;
            if (row + 1 < row_limit) *reinterpret_cast<u32x4_any_t*>(out + p.n) = odd_row;
          }
        }
        cut_rows(row_base, 8, [&](int r, int c) {  // already scaled and rounded: the low half of a word is the even row
          const uint32_t word = words[(r >> 1) * WCOLS + (c ^ read_swizzle(r >> 1, 1))];
          return (float)__builtin_bit_cast(_Float16, (uint16_t)(r & 1 ? word >> 16 : word));
        });
      }
      };
      if (p.alpha != 1.f) packed_turn(std::true_type{});
      else packed_turn(std::false_type{});
      return;
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      if (!finishes(fm)) continue;  // the other K group stores this fragment
      const int row_base = row0 + fm * 32;
      if (p.d_f16) {
        constexpr int PER_ROW = WCOLS / 8;           // 16-byte pieces (8 halves) per row
        constexpr int ITERS = 32 * PER_ROW / 64;
        uint32_t c_raw[ITERS][8];                    // fp16 C: one 16-byte load per piece (words 0-3); fp32 C: two
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
          const int piece = it * 64 + lane;
          const int row = row_base + piece / PER_ROW, col = col0 + (piece % PER_ROW) * 8;
          u32x4_t lo = u32x4_t{0, 0, 0, 0}, hi = u32x4_t{0, 0, 0, 0};
          if (use_c && row < row_limit && col + 8 <= p.n) {
            const size_t o = (size_t)row * p.n + col;
            if (p.c_f16) {
              lo = *reinterpret_cast<const u32x4_any_t*>(reinterpret_cast<const _Float16*>(p.c) + o);
            } else {
              lo = *reinterpret_cast<const u32x4_any_t*>(reinterpret_cast<const float*>(p.c) + o);
              hi = *reinterpret_cast<const u32x4_any_t*>(reinterpret_cast<const float*>(p.c) + o + 4);
            }
          }
          c_raw[it][0] = lo.x; c_raw[it][1] = lo.y; c_raw[it][2] = lo.z; c_raw[it][3] = lo.w;
          c_raw[it][4] = hi.x; c_raw[it][5] = hi.y; c_raw[it][6] = hi.z; c_raw[it][7] = hi.w;
        }
        store_rows(fm);
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
          const int piece = it * 64 + lane;
          const int r = piece / PER_ROW, c8 = (piece % PER_ROW) * 8;
          const int row = row_base + r, col = col0 + c8;
          const int sw = read_swizzle(r, 2);
          const float4 lo = *reinterpret_cast<const float4*>(scratch + r * WCOLS + (c8 ^ sw));
          const float4 hi = *reinterpret_cast<const float4*>(scratch + r * WCOLS + ((c8 + 4) ^ sw));
          float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
          if (row < row_limit && col + 8 <= p.n) {
            const size_t o = (size_t)row * p.n + col;
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] = p.alpha * x[j];
            if (use_c) {
              if (p.c_f16) {
                const half8_t cv =
                    __builtin_bit_cast(half8_t, u32x4_t{c_raw[it][0], c_raw[it][1], c_raw[it][2], c_raw[it][3]});
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = x[j] + p.beta * (float)cv[j];
              } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = x[j] + p.beta * __builtin_bit_cast(float, c_raw[it][j]);
              }
            }
            half8_t out;
#pragma unroll
            for (int j = 0; j < 8; ++j) out[j] = (_Float16)x[j];
            *reinterpret_cast<u32x4_any_t*>(reinterpret_cast<_Float16*>(d_out) + o) = __builtin_bit_cast(u32x4_t, out);
          }
        }
        cut_rows(row_base, 8, [&](int r, int c) { return p.alpha * scratch[r * WCOLS + (c ^ read_swizzle(r, 2))]; });
      } else {
        constexpr int PER_ROW = WCOLS / 4;           // 16-byte pieces (4 floats) per row
        constexpr int ITERS = 32 * PER_ROW / 64;
        uint32_t c_raw[ITERS][4];                    // fp32 C: one 16-byte load per piece; fp16 C: one 8-byte load
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
          const int piece = it * 64 + lane;
          const int row = row_base + piece / PER_ROW, col = col0 + (piece % PER_ROW) * 4;
          u32x4_t lo = u32x4_t{0, 0, 0, 0};
          if (use_c && row < row_limit && col + 4 <= p.n) {
            const size_t o = (size_t)row * p.n + col;
            if (p.c_f16) {
              const u32x2_t t = *reinterpret_cast<const u32x2_any_t*>(reinterpret_cast<const _Float16*>(p.c) + o);
              lo.x = t.x; lo.y = t.y;
            } else {
              lo = *reinterpret_cast<const u32x4_any_t*>(reinterpret_cast<const float*>(p.c) + o);
            }
          }
          c_raw[it][0] = lo.x; c_raw[it][1] = lo.y; c_raw[it][2] = lo.z; c_raw[it][3] = lo.w;
        }
        store_rows(fm);
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
          const int piece = it * 64 + lane;
          const int r = piece / PER_ROW, c4 = (piece % PER_ROW) * 4;
          const int row = row_base + r, col = col0 + c4;
          const float4 a4 = *reinterpret_cast<const float4*>(scratch + r * WCOLS + (c4 ^ read_swizzle(r, 2)));
          float x[4] = {a4.x, a4.y, a4.z, a4.w};
          if (row < row_limit && col + 4 <= p.n) {
            const size_t o = (size_t)row * p.n + col;
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = p.alpha * x[j];
            if (use_c) {
              if (p.c_f16) {
                const half4_t cv = __builtin_bit_cast(half4_t, u32x2_t{c_raw[it][0], c_raw[it][1]});
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = x[j] + p.beta * (float)cv[j];
              } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = x[j] + p.beta * __builtin_bit_cast(float, c_raw[it][j]);
              }
            }
            *reinterpret_cast<u32x4_any_t*>(reinterpret_cast<float*>(d_out) + o) =
                __builtin_bit_cast(u32x4_t, float4{x[0], x[1], x[2], x[3]});
          }
        }
        cut_rows(row_base, 4, [&](int r, int c) { return p.alpha * scratch[r * WCOLS + (c ^ read_swizzle(r, 2))]; });
      }
    }
    return;
  }
  // Direct form (generic variant): one element per accumulator register.
  auto finish_element = [&](int row, int col, float sum) __attribute__((always_inline)) {
    if (row < row_limit && col < p.n) {
      const size_t o = (size_t)row * p.n + col;
      float x = p.alpha * sum;
      if (p.beta != 0.f) {
        const float cv = p.c_f16 ? (float)reinterpret_cast<const _Float16*>(p.c)[o]
                                 : reinterpret_cast<const float*>(p.c)[o];
        x = x + p.beta * cv;
      }
      if (p.d_f16) reinterpret_cast<_Float16*>(d_out)[o] = (_Float16)x;
      else reinterpret_cast<float*>(d_out)[o] = x;
    }
  };
  const int col_lane = lane & 31;
  const int row_lane = 4 * (lane >> 5);
#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
    if (!finishes(fm)) continue;  // the other K group stores this fragment
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      const int col = col0 + fn * 32 + col_lane;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        finish_element(row0 + fm * 32 + 8 * (v / 4) + row_lane + (v % 4), col, acc[fm][fn][v]);
      }
    }
  }
}

template <int WM, int WN, int FM, int FN, bool DMA, bool TOKENS = false, int KG = 1, bool M16 = false, bool BF16 = false, bool RAGGED = false>
static hipError_t launch_gemm_cfg(GemmArgs args, hipStream_t stream) {
  using TS = TileShape<WM, WN, FM, FN, KG>;
  args.tiles_m = (args.m + TS::BM - 1) / TS::BM;
  args.tiles_n = (args.n + TS::BN - 1) / TS::BN;
  const int lds = DMA ? TS::LDS_BYTES : TS::STAGE_BYTES;
  auto kern = gemm_kernel<WM, WN, FM, FN, DMA, TOKENS, KG, M16, BF16, RAGGED>;
  // the dynamic-LDS limit is a per-device attribute of the kernel; threads that race here set the same value
  static std::atomic<bool> attr_done[64] = {};
  int device = 0;
  if (hipError_t st = hipGetDevice(&device); st != hipSuccess) return st;
  if (device < 0 || device >= 64) return hipErrorInvalidDevice;
  if (!attr_done[device].load(std::memory_order_acquire)) {
    hipError_t st = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (st != hipSuccess) return st;
    attr_done[device].store(true, std::memory_order_release);
  }
  // XCDs of the device as the tile order sees them: gfx950 has 32 compute units per XCD, a whole MI355X eight of them;
  // a partition of the GPU shows fewer compute units and is served by as many XCDs
  static std::atomic<int> xcds_of[64] = {};
  int xcds = xcds_of[device].load(std::memory_order_relaxed);
  if (xcds <= 0) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus <= 0) cus = 256;
    xcds = cus / 32 < 1 ? 1 : (cus / 32 > 8 ? 8 : cus / 32);
    xcds_of[device].store(xcds, std::memory_order_relaxed);
  }
  args.xcds = xcds;
  const uint64_t prep = (uint64_t)args.prep, b = (uint64_t)args.b;
  const u32x8_t operands = {(uint32_t)prep, (uint32_t)(prep >> 32), (uint32_t)b, (uint32_t)(b >> 32), (uint32_t)args.m, (uint32_t)args.n,
                            (uint32_t)args.k, (uint32_t)args.ldb};
  const u32x4_t tiles = {(uint32_t)args.tiles_m, (uint32_t)args.tiles_n,
                         (uint32_t)((uint64_t(1) << 32) / ((uint64_t)kStripTiles * args.tiles_m) + 1),
                         (uint32_t)args.chunks_per_split | (uint32_t)args.xcds << 24};  // (chunks of 256 of an int K: 23 bits)
  const GemmResult result{args.d, args.c, args.bias, args.alpha, args.beta, args.c_f16, args.d_f16, args.bias_type};
  return launch_kernel(kern, dim3(args.tiles_m * args.tiles_n, args.splits), dim3(64 * TS::NW), lds, stream, operands, tiles, result);
}

}  // namespace onebit
