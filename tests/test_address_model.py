"""Host-side model of every global address the kernels form, checked against the buffers the C ABI hands them.

The kernels' addresses depend on shapes, launch plan and pointers only, never on operand contents, so their index
arithmetic can be restated on the CPU (numpy, one array element per lane) and every access asserted to lie inside its
operand: the prepared weight, B (or its padded copy), C / D, the K-split partial sums. The model restates the index
arithmetic of onebitsparsemul_amd/csrc/: prepare_kernel and pack_kernel, skinny_kernel with its five B staging modes, wide_kernel
in both forms (its walk over the grid, a remainder in parts, the requests a wait names, both SMFMACs' reads of an image), gemm_kernel's
asynchronous copy pattern, epilogue ranges and the turns of both epilogues through LDS, splitk_reduce_kernel, pad_b_kernel. Where a load
deliberately reaches past a row (pieces at any alignment, rows read where they lie, padded copy) the elements that arrive are tracked
too. The route of a call comes from the library itself (onebit_sparse_describe_call, host-only); that the build which the library
launches is the one modelled here is checked in test_kernel_builds.py. It covers the benchmark configurations and the long-K shapes
with 33 to 64 columns (8192 x 28672 with n = 40, 48, 64). No GPU is touched.
"""
import numpy as np
import pytest

from onebitsparsemul_amd import _native

BLOCK, SIGN_OFF, CHUNK_K, ROW_BLOCK, STAGE_K, STAGES = 1536, 1024, 256, 32, 64, 4
LANE = np.arange(64, dtype=np.int64)

# TileConfig code -> (WM, WN, FM, FN, KG), as in launch_gemm_pass
TILES = {0: (4, 1, 4, 4, 1), 1: (4, 1, 2, 4, 1), 2: (4, 1, 1, 4, 1), 3: (2, 2, 4, 4, 1), 4: (2, 2, 4, 2, 1),
         5: (2, 2, 8, 2, 1), 6: (2, 2, 2, 2, 1), 7: (2, 2, 4, 1, 1), 8: (2, 4, 4, 2, 1), 9: (4, 2, 4, 2, 1),
         10: (4, 2, 2, 2, 1), 11: (2, 4, 2, 1, 1), 12: (2, 2, 1, 2, 1), 13: (2, 2, 2, 2, 2), 14: (2, 2, 1, 2, 2),
         15: (4, 1, 4, 4, 1)}  # 15: tile 0's geometry on the 16x16x64 SMFMAC (same copies, same result region)


def prepared_bytes(m, k):
    return ((m + 31) // 32) * ((k + 255) // 256) * BLOCK


def inside(offsets, width, size, what):
    offsets = np.asarray(offsets, dtype=np.int64)
    assert offsets.size == 0 or (offsets.min() >= 0 and offsets.max() + width <= size), \
        f"{what}: [{offsets.min()}, {offsets.max() + width}) outside a buffer of {size} bytes"


def meta_offset_reference(r, c, m):
    b0, b1, b2, b345 = r & 1, (r >> 1) & 1, (r >> 2) & 1, (r >> 3) & 7
    return (c >> 1) * 2 * m + (r >> 6) * 128 + ((b1 << 6) | (b345 << 3) | (b0 << 2) | ((c & 1) << 1) | b2)


# ---------------------------------------------------------------------------------------------------------------
def strip_positions(grid, width, length):
    """(along, across) of every workgroup of a grid that is walked in strips (strip_position)"""
    block = np.arange(grid, dtype=np.int64)
    per, rem, xcd = grid // 8, grid % 8, block % 8
    v = xcd * per + np.minimum(xcd, rem) + block // 8
    strip, w = v // (width * length), v % (width * length)
    return w // width, strip * width + w % width


def check_strips(grid, width, length, groups):
    """every (along, group) once; the workgroups past the last group return"""
    along, across = strip_positions(grid, width, length)
    used = across < groups
    assert along.min() >= 0 and along.max() < length and across.min() >= 0
    cells = along[used] * groups + across[used]
    assert np.array_equal(np.sort(cells), np.arange(length * groups))


def check_prepare(m, k):
    kc_total, pairs, ncols = (k + 255) // 256, m // 64, k // 16
    a_bytes, e_bytes = m * k // 16, m * ncols * 2
    strips = (pairs + 15) // 16
    check_strips(kc_total * 4 * strips, 4, kc_total, (pairs + 3) // 4)  # four wavefronts (row pairs) per workgroup
    i, ga = LANE & 31, LANE >> 5
    for kc in sorted({0, kc_total // 2, kc_total - 1}):
        for pair in sorted({0, pairs // 2, pairs - 1}):
            # value bits: eight bytes, the 64 rows of one compressed column
            j = 15 - (i & 15)
            col0 = kc * 128 + 16 * (j >> 2) + 8 * ga + 2 * (j & 3) + (i >> 4)
            for h in (0, 1):
                # bit i of sign word h: kept value t of step s, which is compressed column 8 (2 s + ga) + t of the chunk
                t, s = 2 * (j & 3) + (i >> 4), 4 * h + (j >> 2)
                col = col0 + 64 * h
                assert np.array_equal(col, kc * 128 + 8 * (2 * s + ga) + t)
                assert np.array_equal(i, np.where(t % 2 == 0, 15, 31) - (4 * (s % 4) + t // 2))
                ok = col < k // 2
                at = pair * 64 + col[ok] * m
                assert (at % 64 == 0).all()
                inside(at >> 3, 8, a_bytes, "prepare: value bits")
            # metadata, reference layout: dwords of rows r and r + 4
            src = kc * 8 * m + pair * 64 + ((((i >> 1) & 1) << 5) | (((i >> 3) & 3) << 2) | ((i & 1) << 1) | ga)
            for s in range(8):
                if kc * 16 + 2 * s >= ncols:
                    continue
                for blk in (0, 1):
                    dword = src + s * m + 16 * blk
                    inside(dword * 4, 4, e_bytes, "prepare: metadata")
                    row = pair * 64 + 32 * blk + i
                    assert np.array_equal(2 * dword + ((i >> 2) & 1), meta_offset_reference(row, kc * 16 + 2 * s + ga, m))
            # metadata, general form: the running offset is the closed form
            for blk in (0, 1):
                r, c0 = pair * 64 + 32 * blk + i, kc * 16 + ga
                off = meta_offset_reference(r, c0, m)
                for s in range(8):
                    ok = c0 + 2 * s < ncols
                    assert np.array_equal(off[ok], meta_offset_reference(r[ok], (c0 + 2 * s)[ok], m))
                    inside(off[ok] * 2, 2, e_bytes, "prepare: metadata (general form)")
                    off = off + 2 * m
                block = ((2 * pair + blk) * kc_total + kc) * BLOCK
                inside(block + LANE * 16, 16, prepared_bytes(m, k), "prepare: block metadata")
                inside(block + SIGN_OFF + LANE * 8, 8, prepared_bytes(m, k), "prepare: block signs")


def check_pack(m, k, size):
    """pack_kernel on values of `size` bytes: rows into LDS and back, value bits and metadata out"""
    row_bytes, pieces = 64 * size, 4 * size
    rows_per_copy = 64 // pieces
    k_tiles, tiles, ncols = (k // 16 + 3) // 4, m // 64, k // 16
    check_strips(k_tiles * 4 * ((tiles + 15) // 16), 4, k_tiles, (tiles + 3) // 4)
    a_bytes, e_bytes = m * k // 16, m * ncols * 2
    for along in sorted({0, k_tiles // 2, k_tiles - 1}):
        c_first = along * 4
        c_count = min(ncols - c_first, 4)
        for tile in sorted({0, tiles // 2, tiles - 1}):
            row0 = tile * 64
            # copies: LDS piece position -> (row, piece) it holds
            image = {}
            for copy in range(pieces):
                row = copy * rows_per_copy + LANE // pieces
                piece = (LANE % pieces) ^ (row % pieces)
                used = np.where(piece < size * c_count, piece, 0)
                inside(((row0 + row) * k + 16 * c_first) * size + 16 * used, 16, m * k * size, "pack: weights")
                for lane in range(64):
                    image[copy * 64 + lane] = (row[lane], piece[lane])
            assert len(image) == 64 * pieces
            for q in range(pieces):
                at = LANE * row_bytes + ((q ^ (LANE % pieces)) << 4)
                assert (at % 16 == 0).all()
                assert all(image[at[lane] // 16] == (lane, q) for lane in range(64))
            # value bits: lane (h, b) stores the 32 rows of half h of kept value 2 g + b / 16 of column c, b % 16 = 4 g + c
            b, half = LANE & 31, LANE >> 5
            c = b & 3
            column = 8 * (c_first + c) + 2 * ((b >> 2) & 3) + (b >> 4)
            ok = c < c_count
            bit = row0 + 32 * half + column * m
            assert (bit % 32 == 0).all() and len(set(bit[ok])) == ok.sum()
            inside(bit[ok] >> 3, 4, a_bytes, "pack: value bits")
            # metadata, dword form: the lane of row r the even column of rows r and r + 4, that of row r + 4 the odd one
            upper = (LANE >> 2) & 1
            dst = row0 + ((((LANE >> 1) & 1) << 5) | ((LANE >> 3) << 2) | ((LANE & 1) << 1) | upper)
            for c in range(0, c_count, 2):
                dword = dst + ((c_first + c) >> 1) * m
                inside(dword * 4, 4, e_bytes, "pack: metadata")
                low_row = row0 + (LANE & ~4)
                assert np.array_equal(2 * dword, meta_offset_reference(low_row, c_first + c + upper, m))
                assert np.array_equal(2 * dword + 1, meta_offset_reference(low_row + 4, c_first + c + upper, m))
            for c in range(c_count):
                inside(meta_offset_reference(row0 + LANE, c_first + c, m) * 2, 2, e_bytes, "pack: metadata (general form)")


# ---------------------------------------------------------------------------------------------------------------
def token_loads(n, x32=False):
    """load instructions per image of the token-major form: of two tokens each on 16-bit activations, of one on fp32"""
    if x32:
        return n if n <= 2 or 5 <= n <= 8 else n + n % 2
    return 1 if n <= 2 else 2 if n <= 4 else 4 if n <= 8 else 6 if n <= 12 else 8


def skinny_variant(n, rows, chunks, b_aligned=True, tokens=False, x32=False):
    """(wavefronts, row blocks, image columns, mode, loads per image where the build names them); chunks: of a K split"""
    nw, r = {32: (16, 1), 64: (8, 2), 128: (8, 4)}[rows]
    nc = 64 if n > 32 else 32 if n > 16 else 16
    if nc == 64:
        r = min(r, 2)
    if tokens:
        assert n <= 16
        return nw, r, nc, "tokens32" if x32 else "tokens", token_loads(n, x32)
    if n == nc and b_aligned:
        return nw, r, nc, "full", 8
    if n == 1 and b_aligned:
        return nw, r, nc, "tokens", 1   # a k x 1 B is a token-major x of one token
    if 2 <= n <= 8 and b_aligned and not (n == 8 and r != 2 and chunks < (32 if nw == 16 else 16)):
        return nw, r, nc, "columns", (n + 1) // 2   # four K positions per lane
    return nw, r, nc, "any", 8          # 16-byte pieces wherever the rows start


def drop_halves(values, count):
    """the eight values from number `count` on, zeros (-1) behind them"""
    return [values[count + j] if count + j < 8 else -1 for j in range(8)]


def check_any_image(n, k, nc, k_base):
    """One image of the pieces at any alignment: every load inside B, and in the image every element below column n is the
    element of B it stands for, or zero at or past K. An element of B is tracked by its number."""
    img_rows, pieces = 8192 // (nc * 2), (n + 7) // 8
    any_rows = 64 >> (pieces - 1) if nc == 16 else 64 // pieces
    any_row = LANE >> (pieces - 1) if nc == 16 else LANE // pieces
    any_piece = LANE & (pieces - 1) if nc == 16 else LANE % pieces
    assert np.array_equal(any_row, LANE // pieces) and any_rows == 64 // pieces and np.array_equal(any_piece, LANE % pieces)
    rows_left = min(k - k_base, img_rows + 8)
    image = np.full((img_rows, nc), -2, dtype=np.int64)  # -2: what LDS held before
    if rows_left <= 0:
        return
    last = (rows_left * n - 8) * 2
    for i in range(8):
        if i * any_rows >= img_rows:
            continue
        offset = (any_row * n + 8 * any_piece) * 2 + i * any_rows * n * 2
        assert offset.max() < (1 << 32)
        at = np.minimum(offset, last)
        inside(k_base * n * 2 + at, 16, k * n * 2, "split-K kernel: B pieces")
        for lane in range(64):
            values = [k_base * n + at[lane] // 2 + j for j in range(8)]
            if rows_left < img_rows + (0 if n % 8 == 0 else 8) and offset[lane] > last:
                values = [-1] * 8 if n % 8 == 0 else drop_halves(values, (offset[lane] - last) // 2)
            row = any_row[lane] + i * any_rows
            if any_row[lane] < any_rows and row < img_rows:
                image[row, 8 * any_piece[lane]:8 * any_piece[lane] + 8] = values
    row, col = np.arange(img_rows)[:, None], np.arange(n)[None, :]
    assert np.array_equal(image[:, :n], np.where(k_base + row < k, (k_base + row) * n + col, -1))


def token_image_16(n, k, k_base):
    """The token-major image of 16-bit activations: byte offset of each eight values -> (token, first K), from the stores of the
    pieces."""
    image = {}
    for i in range(8):
        for lane in range(64):
            piece, token = lane % 32, lane // 32 + 2 * i
            swizzle = (lane // 32) & 15
            at = ((lane // 32) * 512 + ((piece ^ swizzle) << 4) ^ (((2 * i) & 15) << 4)) + i * 1024
            assert at not in image
            image[at] = (token, k_base + 8 * piece)
    return image


def check_tokens32_image(n, k, k_base):
    """One image of fp32 activations: every load inside x and what it brings where the 16-bit form has it (a token's K in pieces of
    eight, a piece as two halves). The loads of a token past the last one fall outside the descriptor."""
    size, image = n * k * 4, token_image_16(n, k, k_base)
    whole, seen = k_base + CHUNK_K <= k, set()
    loads = token_loads(n, x32=True)
    assert n <= loads <= n + 1
    for token in range(loads):
        offset = LANE * 16 + token * k * 4
        if whole:
            lane_off, scalar_off = offset, k_base * 4
        else:
            lane_off, scalar_off = np.where(k_base + 4 * LANE < k, offset + k_base * 4, 0xFFFFFF00), 0
        accessed = lane_off + 16 <= size  # the descriptor's range check looks at the lane offset alone
        assert lane_off.max() < (1 << 32) and np.array_equal(accessed, (lane_off != 0xFFFFFF00) & (token < n))
        inside(lane_off[accessed] + scalar_off, 16, size, "split-K kernel: fp32 x rows")
        assert np.array_equal((lane_off + scalar_off)[accessed] // 4, (token * k + k_base + 4 * LANE)[accessed])
        at = token * 512 + (((LANE >> 1) ^ (token & 15)) << 4) + (LANE & 1) * 8
        for lane in range(64):
            assert image[at[lane] // 16 * 16] == (token, k_base + 8 * (lane >> 1)) and at[lane] not in seen
            seen.add(at[lane])
    assert len(seen) == 64 * loads and max(seen) + 8 <= 8192


def check_columns_image(n, k, k_base):
    """One image of two to eight columns: a lane loads the 4 n values of four K positions and stores them as n columns of four K values,
    where the token-major reads look for them. An element of B is tracked by its number, zeros as -1."""
    size, image = k * n * 2, token_image_16(n, k, k_base)
    base, at = k_base * n * 2, LANE * n * 8
    if k_base + CHUNK_K <= k:
        lane_at, image_at = at, base
    else:
        lane_at, image_at = np.where(k_base + 4 * LANE < k, at + base, 0xFFFFFF00), 0
    halves = np.full((64, 32), -2, dtype=np.int64)  # the lane's v[i]: eight values each
    loads = [(16 * i, 16) for i in range(n // 2)] + ([(8 * (n - 1), 8)] if n % 2 else [])
    for i, (start, width) in enumerate(loads):
        offset = lane_at + start
        assert offset.max() + width <= (1 << 32)
        accessed = offset + width <= size  # the descriptor's range check looks at the lane offset alone
        assert np.array_equal(accessed, lane_at != 0xFFFFFF00)
        inside(offset[accessed] + image_at, width, size, "split-K kernel: fours of K positions")
        assert (offset[accessed] % 8 == 0).all()
        for j in range(width // 2):
            halves[:, 8 * i + j] = np.where(accessed, (offset + image_at) // 2 + j, -1)
    seen = set()
    for c in range(n):
        where = c * 512 + (((LANE >> 1) ^ (c & 15)) << 4) + (LANE & 1) * 8
        for lane in range(64):
            assert image[where[lane] // 16 * 16] == (c, k_base + 8 * (lane >> 1)) and where[lane] not in seen
            seen.add(where[lane])
        for j in range(4):  # half j of the lane's eight bytes: K position 4 lane + j
            row = k_base + 4 * LANE + j
            assert np.array_equal(halves[:, j * n + c], np.where(row < k, row * n + c, -1))
    assert len(seen) == 64 * n and max(seen) + 8 <= 8192


def check_skinny(m, n, k, rows, tokens=False, b_aligned=True, d_size=2, splits=1, x32=False):
    kc_total, rb_total = (k + 255) // 256, m // 32
    cps = (kc_total + splits - 1) // splits if splits > 1 else kc_total
    nw, R, nc, mode, loads = skinny_variant(n, rows, cps, b_aligned, tokens, x32)
    img_rows = 8192 // (nc * 2)
    sub = CHUNK_K // img_rows
    prep_size, b_size = prepared_bytes(m, k), k * n * (4 if x32 else 2)
    grid = (rb_total + R - 1) // R
    few_loads = mode == "columns" or (mode == "tokens" and loads <= 2)
    prefetch_b = nw <= 8 or few_loads
    images = set()
    splits = (kc_total + cps - 1) // cps
    assert (splits - 1) * cps < kc_total  # the launcher's check: no empty split
    b_fits = b_size < (1 << 32)
    if mode in ("tokens", "tokens32"):
        assert k * 64 * (4 if x32 else 2) < 0xFFFFFF00  # the launcher's check
    if mode == "columns":
        assert k * n * 2 < 0xFFFFFF00   # the launcher's check
    for wg, split in [(g, sp) for g in sorted({0, 1, grid // 2, grid - 1} & set(range(grid)))
                      for sp in sorted({0, splits // 2, splits - 1})]:
        rb_first = wg * R
        kc_begin = split * cps
        kc_end = min(kc_begin + cps, kc_total)
        short_k = nw <= 8 and sub == 1 and kc_end - kc_begin <= 2 * nw
        at_once = nw == 16 and few_loads and nw < kc_end - kc_begin <= 3 * nw
        rounds = 3 if kc_end - kc_begin > 2 * nw else 2  # of a wavefront that requests everything at once
        for wave in range(nw):
            first = kc_begin + wave
            # --- prepared operand through one descriptor per row block
            chunks = []
            if short_k:
                chunks += [first, first + nw]
            elif at_once:
                chunks += [first + i * nw for i in range(rounds)]
                # multiplied: all but the last where there is none left for this wavefront
                multiplied = chunks[:-1] if chunks[-1] >= kc_end else chunks
                assert multiplied == list(range(first, kc_end, nw))
            else:
                chunks.append(first)   # requested before the loop (clamped to the last chunk when past it)
                kc = first
                while kc < kc_end:
                    if kc + nw < kc_end:
                        chunks.append(kc + nw)
                    kc += nw
            for r in range(R):
                rb = min(rb_first + r, rb_total - 1)
                base, size = rb * kc_total * BLOCK, kc_total * BLOCK
                assert size < (1 << 32)
                for kc in chunks:
                    block = min(kc, kc_total - 1) * BLOCK
                    for off, width in ((LANE * 16, 16), (SIGN_OFF + LANE * 8, 8)):
                        inside(block + off, width, size, "split-K kernel: prepared block inside its descriptor")
                        inside(base + block + off, width, prep_size, "split-K kernel: prepared operand")
            # --- B images
            k_bases = []
            if short_k:
                k_bases.append(first * CHUNK_K)
                if mode != "any" or first + nw < kc_end:
                    k_bases.append((first + nw) * CHUNK_K)
            elif at_once:
                k_bases += [kc * CHUNK_K for kc in chunks]
            else:
                kc = first
                if prefetch_b and (nw <= 8 or first < kc_end):
                    k_bases.append(first * CHUNK_K)
                while kc < kc_end:
                    for s in range(sub):
                        k_bases.append(kc * CHUNK_K + s * img_rows)
                    if prefetch_b and kc + nw < kc_end:
                        k_bases.append(kc * CHUNK_K + nw * CHUNK_K)  # the next chunk's first image
                    kc += nw
            for k_base in k_bases:
                rows_valid = min(max(k - k_base, 0), img_rows)
                if mode == "tokens32":
                    if k_base not in images:
                        images.add(k_base)
                        if len(images) <= 4 or k - k_base < 2 * CHUNK_K:
                            check_tokens32_image(n, k, k_base)
                    continue
                if mode == "tokens":
                    # raw buffer loads: the descriptor (n * k * 2 bytes) checks the lane offset alone and returns zero
                    # without an access when it is out of range; the scalar offset is added afterwards
                    ppt = img_rows // 8
                    tpi = 64 // ppt
                    piece_lane, token_lane = LANE % ppt, LANE // ppt
                    assert n <= tpi * loads
                    for i in range(loads):
                        if k_base + img_rows <= k:
                            lane_off = (token_lane * k + 8 * piece_lane) * 2 + i * tpi * k * 2
                            scalar_off = k_base * 2
                        else:
                            ins = k_base + 8 * piece_lane < k
                            lane_off = np.where(ins, (token_lane * k + 8 * piece_lane) * 2 + k_base * 2 + i * tpi * k * 2,
                                                0xFFFFFF00)
                            scalar_off = 0
                        assert lane_off.max() < (1 << 32)
                        accessed = lane_off + 16 <= b_size
                        assert np.array_equal(accessed, (token_lane + tpi * i < n) & (lane_off != 0xFFFFFF00))
                        inside(lane_off[accessed] + scalar_off, 16, b_size, "split-K kernel: x rows")
                    continue
                if mode == "columns":
                    if k_base not in images:
                        images.add(k_base)
                        if len(images) <= 4 or k - k_base < 2 * CHUNK_K:
                            check_columns_image(n, k, k_base)
                    continue
                if mode == "full":
                    if b_fits and k_base + img_rows <= k:
                        inside(k_base * nc * 2 + LANE[None, :] * 16 + 1024 * np.arange(8)[:, None], 16, b_size,
                               "split-K kernel: whole B image")
                    else:
                        q = LANE[None, :] + 64 * np.arange(8)[:, None]
                        ok = (q // (nc // 8)) < rows_valid
                        inside((k_base * nc + q[ok] * 8) * 2, 16, b_size, "split-K kernel: B image pieces")
                elif k_base not in images:  # (the same for every row group)
                    images.add(k_base)
                    if len(images) <= 24 or k - k_base < 2 * CHUNK_K:
                        check_any_image(n, k, nc, k_base)
        # --- result: rows of the workgroup's row blocks, columns below n
        rows_out = np.arange(rb_first * 32, min((rb_first + R) * 32, m))
        cols = np.arange(n)
        elem = 4 if splits > 1 else d_size          # a split writes fp32 partial sums to its slice of the workspace
        slice0 = split * m * n * elem if splits > 1 else 0
        total = splits * m * n * elem
        if mode in ("tokens", "tokens32"):  # (one column: the same element in both layouts)
            inside(slice0 + (cols[None, :] * m + rows_out[:, None]) * elem, elem, total, "split-K kernel: y")
        else:
            inside(slice0 + (rows_out[:, None] * n + cols[None, :]) * elem, elem, total, "split-K kernel: D")
    if splits > 1:
        check_reduce(m, n, splits, d_size)


WIDE_WAVES, WIDE_IMAGE_K = 8, 64


def row_swizzle(row, pieces):
    return ((((row >> 1) & 1) << 2) | (((row >> 3) & 1) << 1)) if pieces == 8 else ((row >> 3) & 1) << 1 if pieces == 4 else 0 * row


def wide_copies(tokens_form, copies, tokens, k, ldb, first_column):
    """per copy: lane offsets in bytes, K position inside the image and column of the piece a lane brings"""
    out = []
    for i in range(copies):
        if tokens_form:
            token = np.minimum(8 * i + (LANE >> 3), tokens - 1)
            piece = (LANE & 7) ^ (LANE >> 4) ^ (4 * (i & 1))
            out.append(((token * k + 8 * piece) * 2, 8 * piece, 8 * i + (LANE >> 3)))
        else:
            slot = 64 * i + LANE
            row = slot // copies  # `copies` pieces per row
            col = 8 * ((slot % copies) ^ row_swizzle(row, copies))
            used = np.where(first_column + col >= ldb, 0, col)
            out.append(((row * ldb + used) * 2, row, col))
    return out


def wide_strip_walk(row_groups, groups):
    """(row group, column group) of every workgroup of a grid that is walked in strips of two column groups, in the kernel's
    arithmetic: 32-bit reciprocal, eight XCDs"""
    total = row_groups * groups
    reciprocal = ((1 << 32) // (2 * row_groups) + 1) & 0xFFFFFFFF
    x = np.arange(total, dtype=np.int64)
    per, rem, xcd = total // 8, total % 8, x % 8
    v = xcd * per + np.minimum(xcd, rem) + x // 8
    strip = (v * reciprocal) >> 32
    w = v - strip * 2 * row_groups
    strip, w = np.where(w < 0, strip - 1, strip), np.where(w < 0, w + 2 * row_groups, w)
    pair = 2 * (strip + 1) * row_groups <= total
    return np.where(pair, w >> 1, w), 2 * strip + np.where(pair, w & 1, 0)


def check_wide_strips(row_groups, groups):
    """every (row group, column group) once"""
    rows, cols = wide_strip_walk(row_groups, groups)
    assert rows.min() >= 0 and rows.max() < row_groups and cols.min() >= 0 and cols.max() < groups
    assert len(set(rows * groups + cols)) == row_groups * groups


def wide_has_parts(chunks):
    """whether the launcher takes the build that deals a remainder in parts"""
    left = chunks % WIDE_WAVES
    return chunks >= WIDE_WAVES and 1 <= left <= (4 if chunks < 6 * WIDE_WAVES else 2)


def wide_deal(kc_begin, kc_end, wave, parts):
    """(whole chunks, part) of a wavefront: part = (chunk, first image, images) or None"""
    left = (kc_end - kc_begin) & (WIDE_WAVES - 1)
    halvings = 0 if not parts or left > 4 or kc_end - kc_begin < WIDE_WAVES else 1 if left > 2 else 2
    whole_end = kc_end - left if halvings else kc_end
    chunk, images = whole_end + (wave >> halvings), 4 >> halvings
    part = (chunk, (wave & ((1 << halvings) - 1)) * images, images) if parts and chunk < kc_end else None
    return list(range(kc_begin + wave, whole_end, WIDE_WAVES)), part


def wide_requests(chunks, part, copies, R, far):
    """The requests of a wavefront in order, and at each stage's wait how many of the youngest may be outstanding. Returns the prepared
    operands and images in the order of their requests; asserts that a wait leaves nothing outstanding that the stage reads and does not
    wait for anything younger than its image, and that what is multiplied as image S of an operand is that image's."""
    issued, operands, images = [], [], []

    def image(chunk, stage):
        images.append(chunk * 4 + stage)
        issued.extend([("image", chunk, stage)] * copies)

    def operand(chunk):
        operands.append(chunk)
        issued.extend([("operand", chunk, 0)] * (2 * R))  # metadata and signs of each row block

    def wait(allowed, chunk, stage):
        done = issued[:len(issued) - allowed]
        assert done.count(("image", chunk, stage)) == copies and done[-1] == ("image", chunk, stage), (chunk, stage)
        return done

    if not chunks:
        return [], []
    operand(chunks[0])
    image(chunks[0], 0)
    image(chunks[0], 1)
    if far and len(chunks) > 1:
        operand(chunks[1])
    elif far and part:
        operand(part[0])
    for at, kc in enumerate(chunks):
        whole = at + 1 < len(chunks)
        more = whole or part is not None
        next_kc = chunks[at + 1] if whole else part[0] if part else None
        next_first = 0 if whole else part[1] if part else None
        for stage in range(4):
            if more:
                allowed = copies + 2 * R if (stage < 2 if far else stage in (1, 2)) else copies
            else:
                allowed = copies if stage < 3 else 0
            done = wait(allowed, kc, stage)
            if more and stage == (2 if far else 3):
                # the next operand's first use: it has arrived, and the compiler's wait for it covers one image more
                assert done.count(("operand", next_kc, 0)) == 2 * R and allowed == copies
            if stage < 2:
                image(kc, stage + 2)
            elif more if stage == 2 else whole or (part is not None and part[2] > 1):
                image(next_kc, next_first + stage - 2)
            if stage == 0 and more and not far:
                operand(next_kc)
        if far and at + 2 < len(chunks):
            operand(chunks[at + 2])
        elif far and whole and part:
            operand(part[0])
    if part:
        chunk, first, count = part
        # the operand's words, moved to the front: image S is multiplied with metadata word S and sign word S / 2 shifted by 8 (S % 2)
        meta, sign = [0, 1, 2, 3], [(0, 0), (1, 0)]
        if first & 2:
            meta[0], meta[1], sign[0] = meta[2], meta[3], sign[1]
        if first & 1:
            meta[0], sign[0] = meta[1], (sign[0][0], sign[0][1] + 8)
        wait(copies if count > 1 else 0, chunk, first)
        for stage in range(count):
            assert meta[stage] == first + stage
            assert (sign[0][0], sign[0][1] + 8 * stage) == ((first + stage) // 2, 8 * ((first + stage) % 2))
        if count > 1:
            wait(0, chunk, first + 1)
    return operands, images


def check_moved_piece(moved, row, col, start, n, k):
    """The pieces of a ragged B that would reach past its end (start: byte where they would begin, of values that are used): of the last
    row the last one alone, which holds behind the shift the values that it stands for."""
    assert moved.sum() <= 1
    for j in np.flatnonzero(moved):
        shift = (start[j] - (k * n * 2 - 16)) // 2
        assert row[j] == k - 1 and col[j] // 8 == (n - 1) // 8 and shift == col[j] + 8 - n and 0 < shift < 8
        values = drop_halves([k * n - 8 + e for e in range(8)], shift)
        assert all(values[e] == row[j] * n + col[j] + e for e in range(n - col[j]))


def check_wide(m, n, k, rows, columns, splits, tokens=False, pad_b=False, d_size=2):
    """wide_kernel, either form: the launcher's checks, the walk over the grid, the prepared operand, the copies of x or B into the ring
    of two images (K tail, last column group, a ragged B where it lies), the fragment reads of an image, the results"""
    R = rows // 32
    ldb = k if tokens else (n + 7) // 8 * 8 if pad_b else n
    copies = (columns + 7) // 8 if tokens else 2 * ((columns + 15) // 16)
    ct_count = (copies + 1) // 2
    pieces = 2 * ct_count
    image_bytes = 16 * ct_count * WIDE_IMAGE_K * 2
    lds = WIDE_WAVES * 2 * image_bytes
    assert 1 <= columns <= 64 and columns % 8 == 0 and lds <= 160 * 1024
    ragged = not tokens and ldb % 8 != 0  # rows that start anywhere, copied from where they lie
    assert (k * 64 * 2 if tokens else ldb * 128) < (1 << 32) and (tokens or (ldb == n >= 8 if ragged else ldb >= n))
    # the reduction's tiles take the place of the ring: min(R, 2) row blocks of 32 rows, sixteen columns per tile, fp32
    assert min(R, 2) * 32 * 16 * ct_count * 4 <= 2 * image_bytes
    kc_total, rb_total = (k + 255) // 256, m // 32
    prep_size, b_size = prepared_bytes(m, k), (n * k if tokens else k * ldb) * 2
    cps = (kc_total + splits - 1) // splits if splits > 1 else kc_total
    splits = (kc_total + cps - 1) // cps
    assert (splits - 1) * cps < kc_total
    grid, col_groups = (rb_total + R - 1) // R, (n + columns - 1) // columns
    # ---- an image: every piece of it copied once, a lane's reads find the K positions and columns it multiplies
    image = {}
    for i, (_, k_at, col) in enumerate(wide_copies(tokens, copies, 8 * copies, k, max(ldb, 8 * copies), 0)):
        for lane in range(64):
            where = i * 64 + lane
            assert where * 16 + 16 <= image_bytes and where not in image
            image[where] = (k_at[lane], col[lane])  # eight K positions of a token, or eight columns of a K position
    check_wide_strips(grid, col_groups)
    i16, g16 = LANE & 15, LANE >> 4
    # whole 32-column tiles: the 32x32x32 SMFMAC, whose lane (column l % 32, half l / 32) holds K positions 8 half ... + 7 and
    # 16 + 8 half ... + 7 of each 32-wide step
    half, col32 = LANE >> 5, LANE & 31
    for f in range(ct_count // 2 if ct_count % 2 == 0 else 0):
        for ks in range(2):
            if tokens:
                base = col32 * 128 + ((half ^ ((col32 >> 1) & 7)) << 4)
                for h in range(2):
                    at = (base ^ ((4 * ks + 2 * h) << 4)) + f * 4096
                    for lane in range(64):
                        assert at[lane] % 16 == 0 and at[lane] + 16 <= image_bytes
                        if 32 * f + col32[lane] < 8 * copies:
                            assert image[at[lane] // 16] == (32 * ks + 16 * h + 8 * half[lane], 32 * f + col32[lane])
            else:
                row0 = 8 * half + (i16 >> 2)
                c8 = (col32 >> 4) * 4 + (i16 & 3)
                tile = row0 * pieces * 16 + (((4 * f + (c8 >> 1)) ^ row_swizzle(row0, pieces)) << 4) + (c8 & 1) * 8
                for q in range(4):
                    step = 32 * ks + 4 * (q & 1) + 16 * (q >> 1)
                    at = tile + step * pieces * 16
                    for lane in range(64):  # four columns of a K position per lane of the transpose read
                        assert at[lane] + 8 <= image_bytes and at[lane] % 16 == 8 * (c8[lane] & 1)
                        assert image[at[lane] // 16] == (row0[lane] + step, 32 * f + 8 * (c8[lane] >> 1))
    for ct in range(ct_count if ct_count % 2 else 0):
        if tokens:
            base = i16 * 128 + (((4 * (g16 >> 1) + (g16 & 1)) ^ ((i16 >> 1) & 7)) << 4)
            for h in range(2):
                at = (base ^ (h << 5)) + ct * 2048
                for lane in range(64):
                    token, want_k = 16 * ct + i16[lane], 32 * (g16[lane] >> 1) + 8 * (g16[lane] & 1) + 16 * h
                    assert at[lane] % 16 == 0 and at[lane] + 16 <= image_bytes
                    if token < 8 * copies:  # an odd copy count leaves the last eight tokens of a tile unwritten: never stored
                        assert image[at[lane] // 16] == (want_k, token)
        else:
            lane_row = 32 * (g16 >> 1) + 8 * (g16 & 1) + (i16 >> 2)
            tile = lane_row * pieces * 16 + (((2 * ct + ((i16 & 3) >> 1)) ^ row_swizzle(lane_row, pieces)) << 4) + (i16 & 1) * 8
            for q in range(4):
                step = 4 * (q & 1) + 16 * (q >> 1)
                at = tile + step * pieces * 16
                for lane in range(64):  # four columns of a K position per lane of the transpose read
                    assert at[lane] + 8 <= image_bytes
                    assert image[at[lane] // 16] == (lane_row[lane] + step, 16 * ct + 8 * ((i16[lane] & 3) >> 1))
    # ---- addresses
    for group in sorted({0, col_groups // 2, col_groups - 1}):
        first_column = group * columns
        here = min(n - first_column, 8 * copies if tokens else columns)
        assert here >= 1
        base0 = first_column * (k if tokens else 1) * 2
        plan = wide_copies(tokens, copies, here, k, ldb, first_column)
        for lane_off, _, _ in plan:
            assert lane_off.max() < (1 << 32)
        for split in sorted({0, splits // 2, splits - 1}):
            kc_begin = split * cps
            kc_end = min(kc_begin + cps, kc_total)
            dealt = []
            for wave in range(WIDE_WAVES):
                mine, part = wide_deal(kc_begin, kc_end, wave, wide_has_parts(cps))
                chunks, images = wide_requests(mine, part, copies, R, far=ct_count == 1 or (ct_count == 3 and R <= 2))
                # every image of its chunks once, in order, and of its part
                assert images == [c * 4 + s for c in mine for s in range(4)] + (
                    [part[0] * 4 + part[1] + s for s in range(part[2])] if part else [])
                assert chunks == mine + ([part[0]] if part else [])
                dealt += images
                chunks = chunks or [kc_begin + wave]  # requested, clamped, by a wavefront without a chunk
                for kc in chunks:
                    for wg in sorted({0, grid // 2, grid - 1}):
                        for r in range(R):
                            rb = min(wg * R + r, rb_total - 1)
                            block = min(kc, kc_total - 1) * BLOCK
                            for off, width in ((LANE * 16, 16), (SIGN_OFF + LANE * 8, 8)):
                                inside(block + off, width, kc_total * BLOCK, "wide_kernel: prepared block inside its descriptor")
                                inside(rb * kc_total * BLOCK + block + off, width, prep_size, "wide_kernel: prepared operand")
                for at in images:
                    k0 = at * WIDE_IMAGE_K
                    for i, (lane_off, k_at, col) in enumerate(plan):
                        real = k0 + k_at < k  # the others are copied from the block of zeros
                        assert real.all() or k0 + WIDE_IMAGE_K > k
                        start = base0 + k0 * (2 if tokens else ldb * 2) + lane_off
                        if ragged and k0 + WIDE_IMAGE_K > k - 1:  # the general path moves pieces past the end of B back
                            moved = real & (start > b_size - 16) & (first_column + col < n)
                            check_moved_piece(moved, k0 + k_at, first_column + col, start, n, k)
                            # mend_image: the one place in the image that is shifted
                            row, piece = k - 1 - k0, (n - 1 - first_column) // 8
                            if 0 <= row < WIDE_IMAGE_K and piece < pieces:
                                slot = row * pieces + (piece ^ int(row_swizzle(np.int64(row), pieces)))
                                assert np.array_equal(moved, 64 * i + LANE == slot)
                            else:
                                assert not moved.any()
                            start = np.minimum(start, b_size - 16)
                        inside(start[real], 16, b_size, "wide_kernel: copies")
            assert sorted(dealt) == list(range(4 * kc_begin, 4 * kc_end))
        # ---- results of the group: rows below m, this group's columns and no other's
        cols = first_column + np.arange(here)
        assert cols.max() < n and (group == col_groups - 1 or here == columns)
        elem = 4 if splits > 1 else d_size
        for wg in sorted({0, grid // 2, grid - 1}):
            out_rows = np.arange(wg * R * 32, min((wg + 1) * R * 32, m))
            for split in {0, splits - 1}:
                at = cols[None, :] * m + out_rows[:, None] if tokens else out_rows[:, None] * n + cols[None, :]
                inside((split * m * n * (splits > 1) + at) * elem, elem, splits * m * n * elem, "wide_kernel: results")
    if splits > 1:
        check_reduce(m, n, splits, d_size)
    if pad_b:
        check_pad_b(n, k)


def check_pad_b(n, k):
    """pad_b_kernel: every load inside B, every piece of the copy written once with the elements it stands for"""
    per_row = (n + 7) // 8
    ldb, rows = 8 * per_row, 1024 // per_row if 1 < per_row < 1024 else 1
    reciprocal = ((1 << 32) // per_row + 1) & 0xFFFFFFFF
    last_start, local = k * n - 8, np.arange(1024, dtype=np.int64)
    if rows > 1:
        assert np.array_equal((local * reciprocal) >> 32, local // per_row)
    grid_x, grid_y = (k + rows - 1) // rows, (per_row + 1023) // 1024
    written = 0
    for x in sorted({0, 1, grid_x // 2, grid_x - 2, grid_x - 1} & set(range(grid_x))):
        for y in range(grid_y):
            r = (local * reciprocal) >> 32 if rows > 1 else 0 * local
            col, row = 8 * (y * 1024 + local - r * per_row), x * rows + r
            start = row * n + col
            at = np.minimum(start, last_start)
            inside(at * 2, 16, k * n * 2, "pad_b: source")
            stored = (r < rows) & (row < k) & (col < ldb)
            written += stored.sum()
            inside((row[stored] * ldb + col[stored]) * 2, 16, k * ldb * 2, "pad_b: destination")
            assert len(set(row[stored] * ldb + col[stored])) == stored.sum()
            for j in np.flatnonzero(stored)[[0, -1]] if stored.any() else ():
                values = [at[j] + e for e in range(8)]
                if start[j] > last_start:
                    values = drop_halves(values, start[j] - last_start) if start[j] - last_start < 8 else [-1] * 8
                assert all(values[e] == row[j] * n + col[j] + e for e in range(min(8, n - col[j])))
            wide = (start > last_start) & stored  # each of the shifted pieces
            for j in np.flatnonzero(wide):
                values = drop_halves([at[j] + e for e in range(8)], min(8, start[j] - last_start))
                assert all(values[e] == row[j] * n + col[j] + e for e in range(min(8, n - col[j])))
    if grid_x <= 5:
        assert written == k * per_row


def check_reduce(m, n, splits, d_size):
    """splitk_reduce_kernel: one thread per 4 (or 1) results"""
    total = m * n
    vec = 4 if total % 4 == 0 else 1
    first = (np.arange((total // vec + 255) // 256 * 256, dtype=np.int64)) * vec
    first = first[first < total]
    for s in (0, splits - 1):
        inside((s * total + first) * 4, 4 * vec, splits * total * 4, "reduce: partial sums")
    inside(first * d_size, d_size * vec, total * d_size, "reduce: result")


# ---------------------------------------------------------------------------------------------------------------
def tile_of_block(b, tiles_m, tiles_n, group_m, xcds=8):
    """in the kernel's arithmetic: a 32-bit reciprocal in the place of the division by a strip's tiles"""
    total = tiles_m * tiles_n
    per, rem = total // xcds, total % xcds
    x, local = b % xcds, b // xcds
    v = x * per + min(x, rem) + local
    reciprocal = ((1 << 32) // (4 * tiles_m) + 1) & 0xFFFFFFFF
    strip = (v * reciprocal) >> 32
    w = v - strip * 4 * tiles_m
    if w < 0:
        strip, w = strip - 1, w + 4 * tiles_m
    strip_w = min(tiles_n - strip * 4, 4)
    rows = w // group_m
    group = {4: rows >> 2, 3: rows // 3, 2: rows >> 1, 1: rows}[strip_w]
    group_h = min(tiles_m - group * group_m, group_m)
    u = w - group * group_m * strip_w
    column = (u >= group_h) + (u >= 2 * group_h) + (u >= 3 * group_h)
    return group * group_m + u - column * group_h, strip * 4 + column


RAGGED_TILES = (4, 6, 9, 10, 11, 12, 13, 14, 15)  # with a build that copies a ragged B from where it lies


def check_gemm(m, n, k, tile, splits, pad_b, tokens=False, b_aligned=True, d_size=2):
    WM, WN, FM, FN, KG = TILES[tile]
    whole_rows = tokens or pad_b or (n % 8 == 0 and b_aligned)
    ragged = not whole_rows and b_aligned and n >= 8 and tile in RAGGED_TILES
    aligned = whole_rows or ragged
    if not aligned:
        WM, WN, FM, FN, KG = 4, 1, 1, 4, 1  # the element-copy variant
    BM, BN, NW = WM * FM * 32, WN * FN * 32, WM * WN * KG
    CH = BN // 8
    NL = STAGE_K * CH // (64 * NW)
    NA = ((BM // 32) * BLOCK + 1024 * NW - 1) // (1024 * NW)
    tiles_m, tiles_n = (m + BM - 1) // BM, (n + BN - 1) // BN
    chunks_total = (k + 255) // 256
    prep_size = prepared_bytes(m, k)
    assert prep_size < (1 << 32)  # 32-bit copy offsets (the C ABI refuses larger weights)
    cps = (chunks_total + splits - 1) // splits
    splits = (chunks_total + cps - 1) // cps
    assert (splits - 1) * cps < chunks_total  # the launcher's check: no empty split
    ldb = k if tokens else ((n + 7) // 8 * 8 if pad_b else n)
    b_size = (n * k if tokens else k * ldb) * 2
    if tokens:
        assert k * 256 * 2 < (1 << 32)
    # the workgroup -> tile mapping is a bijection
    # (for every XCD count the launcher can derive: 8 on a whole GPU, fewer on a partition)
    for xcds in (8, 4, 2, 1):
        seen = {tile_of_block(b, tiles_m, tiles_n, 8 if NW == 8 or FM * FN > 8 else 16, xcds) for b in range(tiles_m * tiles_n)}
        assert seen == {(tm, tn) for tm in range(tiles_m) for tn in range(tiles_n)}
    rb_total = m // 32
    corner_tiles = {(0, 0), (tiles_m - 1, 0), (0, tiles_n - 1), (tiles_m - 1, tiles_n - 1), (tiles_m // 2, tiles_n // 2)}
    for split in sorted({0, splits - 1, splits // 2}):
        chunk_begin = split * cps
        chunk_end = min(chunk_begin + cps, chunks_total)
        for tile_m, tile_n in corner_tiles:
            n0 = tile_n * BN
            if aligned:
                k_inside = k - 1 if ragged else k
                # a chunk of the loop copies the next one's stages; where those lie inside K it has no test for the last row
                full_end = min(k_inside // CHUNK_K - 1, chunk_end)
                mended = {chunk_begin * STAGES} | {kc * STAGES + s + 1 for kc in range(max(full_end, chunk_begin), chunk_end) for s in range(STAGES)}
                last_stage = (k - 1) // STAGE_K
                if ragged and chunk_begin * STAGES <= last_stage < chunk_end * STAGES:
                    assert last_stage in mended
                found = []
                for wave in range(NW):
                    for i in range(NL):
                        slot = (NW * i + wave) * 64 + LANE
                        if tokens:
                            token = slot // 8
                            sw = np.where(True, (token >> 1) & 7, 0)
                            lc = (slot % 8) ^ sw
                            token = np.where(n0 + token >= n, 0, token)
                            b_off = (token * k + 8 * lc) * 2
                            copy_row = 8 * lc
                            stage_stride, stage0 = STAGE_K * 2, n0 * k * 2
                        else:
                            row, pc = slot // CH, slot % CH
                            sw = (((row & 3) << 2) | (((row >> 3) & 1) << 1)) if BN >= 128 else (((row >> 1) & 1) << 2)
                            lc = pc ^ sw
                            col = np.where(n0 + 8 * lc >= ldb, 0, 8 * lc)
                            b_off = (row * ldb + col) * 2
                            copy_row = row
                            stage_stride, stage0 = STAGE_K * ldb * 2, n0 * 2
                        assert b_off.max() < (1 << 32)
                        # stages copied: the first four of the split's range, then four more per chunk of the loop
                        for stage in range(chunk_begin * STAGES, chunk_end * STAGES + STAGES):
                            next_k0 = stage * STAGE_K
                            base = stage0 + stage * stage_stride
                            if next_k0 + STAGE_K <= k_inside:
                                inside(base + b_off, 16, b_size, "main kernel: B stage copy")
                            else:
                                assert full_end <= chunk_begin or stage // STAGES > full_end
                                real = next_k0 + copy_row < k  # the other lanes copy from the block of zeros
                                start = base + b_off
                                if ragged:  # pieces past the end of B are moved back
                                    moved = real & (start > b_size - 16) & (n0 + 8 * lc < n)
                                    check_moved_piece(moved, next_k0 + copy_row, n0 + 8 * lc, start, n, k)
                                    found += [(stage, slot[j], wave) for j in np.flatnonzero(moved)]
                                    start = np.minimum(start, b_size - 16)
                                inside(start[real], 16, b_size, "main kernel: B stage copy (K tail)")
                    rb0 = tile_m * (BM // 32)
                    for j in range(NA):
                        byte = (NW * j + wave) * 1024 + LANE * 16
                        blk, off = byte // BLOCK, byte % BLOCK
                        blk = np.where(blk >= BM // 32, 0, blk)
                        rb = np.minimum(rb0 + blk, rb_total - 1)
                        a_off = rb * chunks_total * BLOCK + off
                        # the chunk pointer advances while next_chunk + 1 < chunks: it never passes the last chunk
                        for chunk in range(chunk_begin, min(chunk_end + 1, chunks_total)):
                            inside(chunk * BLOCK + a_off, 16, prep_size, "main kernel: prepared block copy")
                if ragged:  # mend_stage: the one place that is shifted, in the stage of the last row, by the wavefront that copied it
                    row, piece = (k - 1) % STAGE_K, (n - 1 - n0) // 8
                    sw = (((row & 3) << 2) | (((row >> 3) & 1) << 1)) if BN >= 128 else (((row >> 1) & 1) << 2)
                    copied = chunk_begin * STAGES <= last_stage < (chunk_end + 1) * STAGES
                    place = row * CH + (piece ^ sw)
                    assert found == ([(last_stage, place, place // 64 % NW)] if piece < CH and copied else [])
            else:
                rows_k = np.arange(k)
                cols = n0 + np.arange(BN)
                cols = cols[cols < n]
                inside((rows_k[:, None] * n + cols[None, :]) * 2, 2, k * n * 2, "main kernel: B elements")
                for fm in range(FM):
                    for wm in range(WM):
                        rb = min((tile_m * BM + wm * FM * 32) // 32 + fm, rb_total - 1)
                        for chunk in range(chunk_begin, chunk_end):
                            base = rb * chunks_total * BLOCK + chunk * BLOCK
                            inside(base + LANE * 16, 16, prep_size, "main kernel: prepared block (direct)")
                            inside(base + SIGN_OFF + LANE * 8, 8, prep_size, "main kernel: prepared signs (direct)")
            # result range of the tile: rows below m, columns below n, in this split's slice when K is split
            rows_out = np.arange(tile_m * BM, min((tile_m + 1) * BM, m))
            cols_out = np.arange(n0, min(n0 + BN, n))
            elem = 4 if splits > 1 else d_size
            slice0 = split * m * n * elem if splits > 1 else 0
            total = (splits if splits > 1 else 1) * m * n * elem
            if tokens:
                inside(slice0 + (cols_out[None, :] * m + rows_out[:, None]) * elem, elem, total, "main kernel: y")
                rows_tile = tile_m * BM + 4 * np.arange(BM // 4)  # the bias: four values, of row 0 past the end
                for size in (2, 4):
                    inside(np.where(rows_tile < m, rows_tile, 0) * size, 4 * size, m * size, "main kernel: bias")
            else:
                inside(slice0 + (rows_out[:, None] * n + cols_out[None, :]) * elem, elem, total, "main kernel: D")
    if splits > 1:
        check_reduce(m, n, splits, d_size)
    if pad_b:
        check_pad_b(n, k)


def check_call(m, n, k, tokens=False, b_aligned=True):
    plan = _native.describe_launch(m, n, k, b_aligned=b_aligned or tokens, tokens=tokens)
    if plan["kernel"] == "skinny_kernel":
        check_skinny(m, n, k, plan["rows"], tokens=tokens, b_aligned=b_aligned, splits=plan["splits"])
        if tokens:
            check_skinny(m, n, k, plan["rows"], tokens=True, splits=plan["splits"], x32=True)
    elif plan["kernel"] == "wide_kernel":
        check_wide(m, n, k, plan["rows"], plan["columns"], plan["splits"], tokens=tokens, pad_b=plan["pad_b"])
    else:
        check_gemm(m, n, k, plan["tile"], plan["splits"], plan["pad_b"] and not tokens, tokens=tokens, b_aligned=b_aligned)
    return plan


@pytest.fixture()
def hooks():
    def reset():
        _native.set_tile_config(-1)
        _native.set_skinny_enabled(True)
        _native.set_skinny_rows(-1)
        _native.set_split_k(-1)
        _native.set_pad_b(True)
    reset()
    yield
    reset()


@pytest.mark.parametrize("m,k", [(64, 32), (512, 512), (8192, 8192), (11008, 4096), (4096, 11008), (8192, 28672), (25600, 25600)])
def test_prepare_kernel_addresses(m, k):
    check_prepare(m, k)


@pytest.mark.parametrize("m,k", [(64, 32), (64, 64), (512, 512), (192, 1056), (11008, 4096), (28672, 8192)])
@pytest.mark.parametrize("size", [2, 4])
def test_pack_kernel_addresses(m, k, size):
    check_pack(m, k, size)


@pytest.mark.parametrize("k", [32, 96, 256, 288, 512])
def test_pieces_at_any_alignment(k):
    """every column count of the images; K that ends inside an image, at its end and before it"""
    for n in range(1, 65):
        nc = 64 if n > 32 else 32 if n > 16 else 16
        for k_base in range(0, 512, 8192 // (nc * 2)):
            check_any_image(n, k, nc, k_base)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 63, 66, 99, 119, 1001, 8185, 8200])
@pytest.mark.parametrize("k", [32, 96, 992])
def test_padded_copy_addresses(n, k):
    check_pad_b(n, k)


@pytest.mark.parametrize("n", [17, 24, 34, 40, 56, 65, 66, 72, 104, 257])
@pytest.mark.parametrize("m,k", [(64, 32), (192, 1056), (64, 2336), (128, 2848), (320, 4640), (1024, 8192)])
def test_wide_kernel_addresses(n, m, k):
    """every width of the column groups the plan can choose, each row group, K splits, remainders with and without parts; B in place,
    a ragged one too, and through its padded copy"""
    for rows in (32, 64, 128):
        for columns in {8 * ((min(n, 16 * width) + 7) // 8) for width in (1, 2, 3, 4)}:
            for splits in (1, 3):
                splits = min(splits, (k + 255) // 256)
                check_wide(m, n, k, rows, columns, splits, tokens=True)
                check_wide(m, n, k, rows, columns, splits)
                if n % 8:
                    check_wide(m, n, k, rows, columns, splits, pad_b=True)


@pytest.mark.parametrize("n", [40, 48, 64])
@pytest.mark.parametrize("rows", [32, 64, -1])
def test_long_k_wide_skinny_shapes(hooks, n, rows):
    """8192 x 28672 with 33 to 64 columns: wide_kernel and the 64-column images of skinny_kernel with 32- and 64-row
    workgroups, and the main kernel with the K split its plan chooses, plain and token-major."""
    m, k = 8192, 28672
    if rows < 0:
        _native.set_skinny_enabled(False)
        for tokens in (False, True):
            assert check_call(m, n, k, tokens=tokens)["kernel"] == "gemm_kernel"
        return
    _native.set_skinny_rows(rows)
    for tokens in (False, True):
        assert check_call(m, n, k, tokens=tokens)["kernel"] == "wide_kernel"
    _native.set_tile_config(0)  # a forced tile keeps products out of wide_kernel
    assert check_call(m, n, k)["kernel"] == "skinny_kernel"


@pytest.mark.parametrize("m,n,k", [(512, 512, 512), (1024, 1024, 1024), (2048, 2048, 2048), (4096, 4096, 4096), (8192, 8192, 8192),
                                   (11008, 1, 4096), (11008, 4, 4096), (11008, 16, 4096), (4096, 1, 11008),
                                   (4096, 4, 11008), (4096, 16, 11008), (4096, 2048, 4096), (16384, 16384, 16384),
                                   (25600, 25600, 25600)])
def test_benchmark_configurations(hooks, m, n, k):
    check_call(m, n, k)
    if n >= 16:
        check_call(m, n, k, tokens=True)


@pytest.mark.parametrize("m,n,k,b_aligned", [(64, 1, 32, True), (192, 5, 800, True), (320, 8, 4128, True), (128, 13, 12320, True),
                                             (320, 17, 4128, True), (1088, 31, 2208, True), (64, 33, 32, True),
                                             (1088, 63, 2208, True), (2048, 32, 20480, True), (4096, 16, 16384, True),
                                             (576, 200, 352, True), (640, 1001, 160, True), (4096, 1001, 4096, True),
                                             (256, 264, 512, False), (1024, 203, 4128, True), (128, 1000, 4128, True),
                                             (4096, 50, 4096, True), (4096, 49, 4096, True), (11008, 1001, 4096, True),
                                             (4096, 1002, 4096, True), (512, 555, 1856, True), (28672, 40, 512, True), (20480, 64, 1024, True), (4096, 384, 11008, True),
                                             (64, 72, 64, False), (2112, 1032, 64, True), (4096, 16, 16384, True),
                                             (2048, 33, 28672, True), (11008, 32, 28672, True), (192, 5, 12320, True),
                                             (320, 2, 4128, True), (320, 4, 4128, True), (2240, 1, 8224, True),
                                             (192, 4, 800, False), (192, 2, 12320, True)])
def test_ragged_and_split_shapes(hooks, m, n, k, b_aligned):
    for rows in (-1, 32, 64, 128):
        _native.set_skinny_rows(rows)
        for tile in (-1, 0):  # 0: a forced tile keeps products out of wide_kernel
            _native.set_tile_config(tile)
            check_call(m, n, k, b_aligned=b_aligned)
        _native.set_tile_config(-1)
    _native.set_skinny_rows(-1)
    check_call(m, n, k, tokens=True)
    for splits in (2, 3, 16):  # the split-K kernel's own K split over workgroups (n <= 64), forced
        _native.set_split_k(splits)
        for rows in (32, 64, 128):
            _native.set_skinny_rows(rows)
            check_call(m, n, k, b_aligned=b_aligned)
            check_call(m, n, k, tokens=True)
    _native.set_skinny_rows(-1)
    _native.set_skinny_enabled(False)
    for splits in (-1, 1, 3, 16):
        _native.set_split_k(splits)
        check_call(m, n, k, b_aligned=b_aligned)
        check_call(m, n, k, tokens=True)


@pytest.mark.parametrize("tile", sorted(TILES))
def test_every_tile_configuration(hooks, tile):
    _native.set_tile_config(tile)
    _native.set_skinny_enabled(False)
    for m, n, k in ((1024, 512, 1024), (576, 264, 192), (2112, 1032, 64), (8192, 8192, 8192)):
        check_call(m, n, k)
        if tile in (4, 6, 9, 10, 11, 12, 13, 14, 15):
            check_call(m, n, k, tokens=True)


@pytest.mark.parametrize("tile", RAGGED_TILES)
@pytest.mark.parametrize("k", [32, 64, 256, 288, 544, 1056, 2272])
def test_main_kernel_on_rows_that_lie_anywhere(tile, k):
    for n in (9, 65, 66, 127, 130, 1001):
        for splits in (1, 2, 3):
            check_gemm(576, n, k, tile, min(splits, (k + 255) // 256), False)


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("k", [256, 2048, 4128, 8192, 11008, 12288, 12320])
def test_few_columns_and_tokens(rows, k):
    """one chunk per wavefront, two and three (requested at once on sixteen of them) and more, the last of them without a last one"""
    for splits in (1, 2):
        splits = min(splits, (k + 255) // 256)
        for n in range(1, 17):
            check_skinny(192, n, k, rows, splits=splits)
            check_skinny(192, n, k, rows, tokens=True, splits=splits)


def test_the_model_catches_an_out_of_range_access():
    """the checker itself: a prepared operand one block too small, or B one row too short, must be flagged"""
    with pytest.raises(AssertionError):
        inside(np.array([0, prepared_bytes(64, 256) - 8]), 16, prepared_bytes(64, 256), "probe")
    real = prepared_bytes

    def short(m, k):
        return real(m, k) - BLOCK
    globals()["prepared_bytes"] = short
    try:
        with pytest.raises(AssertionError):
            check_skinny(1024, 16, 4096, 64)
        with pytest.raises(AssertionError):
            check_wide(1024, 48, 4096, 64, 48, 1)
        with pytest.raises(AssertionError):
            check_gemm(1024, 512, 1024, 9, 1, False)
    finally:
        globals()["prepared_bytes"] = real


# ---- the epilogue's turn through the LDS scratch (gemm_kernel, coalesced form) ------------------------------------
# Restates the index arithmetic of the two forms: fp32 rows [32][WCOLS] and packed fp16 row pairs [16][WCOLS], both with
# the column swizzle (16-byte slots swapped in pairs on odd lines, 128-byte halves swapped when bit 2 of the row / bit 1
# of the row pair is set and a line has at least 64 columns).

def _half_swap(wcols):
    return 32 if wcols >= 64 else 0


def _scratch_rows_model(fn_count):
    """(writes, reads) of the fp32 form for one 32-row block: dicts word -> (row, column) written / read."""
    wcols = fn_count * 32
    writes, reads = {}, {}
    for lane in range(64):
        col_lane, row_lane = lane & 31, 4 * (lane >> 5)
        half_write = (lane >> 5) * _half_swap(wcols)
        for fn in range(fn_count):
            for v in range(16):
                row = 8 * (v // 4) + row_lane + v % 4
                word = row * wcols + ((fn * 32 + col_lane) ^ half_write ^ ((v & 1) << 2))
                assert word not in writes
                writes[word] = (row, fn * 32 + col_lane)
    per_row = wcols // 8
    for it in range(32 * per_row // 64):
        for lane in range(64):
            piece = it * 64 + lane
            r, c8 = piece // per_row, (piece % per_row) * 8
            sw = ((r & 1) << 2) ^ (((r >> 2) & 1) * _half_swap(wcols))
            for part, base in ((0, c8), (1, c8 + 4)):
                for j in range(4):
                    reads[r * wcols + (base ^ sw) + j] = (r, base + j)
    return wcols, writes, reads


def _scratch_pairs_model(fn_count):
    """the packed form: word -> (row pair, column)."""
    wcols = fn_count * 32
    writes, reads = {}, {}
    for lane in range(64):
        col_lane, row_lane = lane & 31, 4 * (lane >> 5)
        half_write = (lane >> 5) * _half_swap(wcols)
        for fn in range(fn_count):
            for q in range(8):
                pair = 4 * (q // 2) + (row_lane >> 1) + (q & 1)
                rows = 8 * (q // 2) + row_lane + 2 * (q % 2)   # registers 2q, 2q + 1 of the accumulator layout
                assert rows == 2 * pair
                word = pair * wcols + ((fn * 32 + col_lane) ^ half_write ^ ((q & 1) << 2))
                assert word not in writes
                writes[word] = (pair, fn * 32 + col_lane)
    per_pair = wcols // 8
    tasks = 16 * per_pair
    for it in range((tasks + 63) // 64):
        for lane in range(64):
            task = it * 64 + lane
            if task >= tasks:
                continue
            pair, c8 = task // per_pair, (task % per_pair) * 8
            sw = ((pair & 1) << 2) ^ (((pair >> 1) & 1) * _half_swap(wcols))
            for base in (c8, c8 + 4):
                for j in range(4):
                    reads[pair * wcols + (base ^ sw) + j] = (pair, base + j)
    return wcols, writes, reads


@pytest.mark.parametrize("fn_count", [1, 2, 4])
@pytest.mark.parametrize("model,lines", [(_scratch_rows_model, 32), (_scratch_pairs_model, 16)])
def test_epilogue_scratch_is_written_once_and_read_back_where_it_was_written(model, lines, fn_count):
    wcols, writes, reads = model(fn_count)
    assert sorted(writes) == list(range(lines * wcols))          # every word of the wavefront's scratch, once, in range
    assert reads == writes                                       # a reader finds (line, column) where the writer put it


def test_epilogue_scratch_swizzle_avoids_bank_conflicts():
    # The tiles the planner uses have 64-column wavefront tiles. 64 banks of 4 bytes. A 4-byte store instruction: the 32
    # lanes of each half-wavefront touch 32 different banks and the two halves touch different ones. A 16-byte read: the
    # 16 lanes served together (two lines) touch 64 different banks.
    wcols = 64
    for v in range(16):
        banks = []
        for lane in range(64):
            row = 8 * (v // 4) + 4 * (lane >> 5) + v % 4
            word = row * wcols + ((lane & 31) ^ ((lane >> 5) * 32) ^ ((v & 1) << 2))
            banks.append(word % 64)
        assert len(set(banks)) == 64
    per_row = wcols // 8
    for group in range(4):
        banks = []
        for lane in range(16 * group, 16 * group + 16):
            r, c8 = lane // per_row, (lane % per_row) * 8
            sw = ((r & 1) << 2) ^ (((r >> 2) & 1) * 32)
            banks += [(r * wcols + (c8 ^ sw) + j) % 64 for j in range(4)]
        assert len(set(banks)) == 64


# ---- the turns of the token-major epilogue through the LDS scratch ------------------------------------------------
TOKEN_TILES = (4, 6, 9, 10, 11, 12, 13, 14, 15)


@pytest.mark.parametrize("tile", TOKEN_TILES)
def test_token_epilogue_16_bit_turns(tile):
    """Every four rows of every token that a wavefront finishes are written once, inside its scratch, and read back as what they are; all
    of them are stored; sixteen lanes meet in no bank."""
    _, _, FM, FN, KG = TILES[tile]
    m16 = tile == 15
    wcols, split = FN * 32, KG == 2 and FM % 2 == 0
    frags = FM // 2 if split else FM
    pieces, turn = 4 * frags, 2 * wcols // frags if frags > 2 else wcols
    groups = 2 if m16 else 4
    assert turn * pieces <= wcols * 8 and wcols % turn == 0 and turn % (16 if m16 else 32) == 0

    def slot_at(t, slot):
        return t * (pieces * 16) + ((((slot >> 1) ^ ((t * pieces >> 4) & (pieces - 1))) << 4) | ((slot & 1) << 3))

    for kg in range(2 if split else 1):
        stored = set()
        for first in range(0, wcols, turn):
            scratch = {}
            for fm in range(FM):
                if split and (fm >= FM // 2) != (kg == 1):
                    continue
                for q in range(groups):
                    tiles = range(first // 16, (first + turn) // 16) if m16 else range(first // 32, (first + turn) // 32)
                    for part in tiles:
                        at = []
                        for lane in range(64):
                            if m16:  # registers of tile (2 fm + q, ct): rows 16 q + 4 (lane / 16) on of token 16 ct + lane % 16
                                slot, row, t = 4 * q + (lane >> 4), 16 * q + 4 * (lane >> 4), part * 16 - first + (lane & 15)
                            else:    # registers 4 q ... 4 q + 3: rows 8 q + 4 (lane / 32) on of token 32 fn + lane % 32
                                slot, row, t = 2 * q + (lane >> 5), 8 * q + 4 * (lane >> 5), part * 32 - first + (lane & 31)
                            where = slot_at(t, 8 * (fm % frags) + slot)
                            assert where not in scratch and where + 8 <= wcols * 128
                            scratch[where] = ((fm % frags) * 32 + row, first + t)
                            at.append(where)
                        for sixteen in range(0, 64, 16):
                            banks = [b % 64 for w in at[sixteen:sixteen + 16] for b in (w // 4, w // 4 + 1)]
                            assert len(set(banks)) == 32
            for it in range(turn * pieces // 64):
                at = []
                for lane in range(64):
                    piece, t = lane % pieces, it * (64 // pieces) + lane // pieces
                    where = slot_at(t, 2 * piece)
                    assert where % 16 == 0
                    assert scratch[where] == (8 * piece, first + t) and scratch[where + 8] == (8 * piece + 4, first + t)
                    stored.add((8 * piece, first + t))
                    at.append(where)
                for sixteen in range(0, 64, 16):
                    assert len({(w // 4 + j) % 64 for w in at[sixteen:sixteen + 16] for j in range(4)}) == 64
        assert stored == {(8 * piece, t) for piece in range(pieces) for t in range(wcols)}


@pytest.mark.parametrize("tile", TOKEN_TILES)
def test_token_epilogue_fp32_turns(tile):
    _, _, FM, FN, _ = TILES[tile]
    wcols, scratch = FN * 32, {}
    for lane in range(64):
        if tile == 15:
            parts = [(ct * 16 + (lane & 15), 4 * rh + (lane >> 4), lane & 15) for rh in range(2) for ct in range(2 * FN)]
        else:
            parts = [(fn * 32 + (lane & 31), 2 * q + (lane >> 5), lane & 31) for fn in range(FN) for q in range(4)]
        for token, slot, low in parts:  # slot s: rows 4 s ... 4 s + 3 of the 32-row block
            where = token * 128 + ((slot ^ ((low >> 1) & 7)) << 4)
            assert where not in scratch and where + 16 <= wcols * 128
            scratch[where] = (4 * slot, token)
    read = set()
    for it in range(wcols * 8 // 64):
        for lane in range(64):
            j, t = lane % 8, it * 8 + lane // 8
            assert scratch[t * 128 + ((j ^ ((t >> 1) & 7)) << 4)] == (4 * j, t)
            read.add((4 * j, t))
    assert len(read) == 8 * wcols == len(scratch)


@pytest.mark.parametrize("row_groups", [1, 2, 3, 7, 8, 11, 15, 31, 32, 53, 131, 1000])
def test_strips_reach_every_workgroup_once(row_groups):
    """odd and even numbers of column groups, fewer workgroups than XCDs, numbers that eight does not divide"""
    for groups in (1, 2, 3, 4, 5, 8, 9, 19, 63):
        check_wide_strips(row_groups, groups)


@pytest.mark.parametrize("chunks", [1, 2, 3, 7])
@pytest.mark.parametrize("R", [1, 2, 4])
def test_waits_of_wide_kernel_name_the_requests_behind_an_image(chunks, R):
    for copies in range(1, 9):
        for far in (False, True):
            for part in (None, (8 * chunks, 0, 1), (8 * chunks, 1, 1), (8 * chunks, 2, 1), (8 * chunks, 3, 1), (8 * chunks, 0, 2),
                         (8 * chunks + 1, 2, 2)):
                wide_requests(list(range(0, 8 * chunks, 8)), part, copies, R, far)


@pytest.mark.parametrize("m,k", [(64, 32), (192, 1056), (320, 4640), (1024, 8192), (128, 16416)])
def test_fp32_activations_addresses(m, k):
    for n in (1, 7, 8, 9, 16):
        for rows in (32, 64, 128):
            for splits in (1, 3):
                check_skinny(m, n, k, rows, tokens=True, splits=min(splits, (k + 255) // 256), x32=True, d_size=4)


# ---------------------------------------------------------------------------------------------------------------
# the split-K kernel's 16x16x64 form: which K positions of a chunk each lane group of an instruction multiplies, on
# the A side (prepared block lanes after v_permlane16_swap) and on the B side (rows of the image a lane reads)
# ---------------------------------------------------------------------------------------------------------------
def _permlane16_swap(x, y):
    """v_permlane16_swap x, y: the odd 16-lane rows of x trade places with the even rows of y"""
    x, y = x.copy(), y.copy()
    for row in (0, 2):
        lo, hi = slice(16 * row, 16 * row + 16), slice(16 * (row + 1), 16 * (row + 2))
        x[hi], y[lo] = y[lo].copy(), x[hi].copy()
    return x, y


def test_split_k_16x16x64_operands_agree_on_k():
    lane = np.arange(64)
    # lane of the prepared block: row lane % 32, half ga = lane // 32 of each 32-wide K step; metadata register d
    # holds steps 2 d (low half word, ABID 0) and 2 d + 1 (high, ABID 1); the value tracked here is (lane, register)
    src = {d: lane * 8 + d for d in range(4)}
    for P in range(2):
        first, second = _permlane16_swap(src[2 * P], src[2 * P + 1])
        for half, reg in enumerate((first, second)):          # operands of block rows 0-15 and 16-31
            src_lane, src_reg = reg // 8, reg % 8
            assert np.array_equal(src_lane % 32, 16 * half + lane % 16)  # every lane group holds its own row l % 16
            ga = src_lane // 32
            for abid in range(2):
                step = 2 * src_reg + abid
                a_first_k = 32 * step + 16 * ga            # the lane's 16 consecutive K positions of the chunk
                # the instruction pairs A group g, position j with B group (16 g + j) % 32 // 8, slot
                # 8 ((16 g + j) // 32) + (16 g + j) % 8; a B lane of group gb reads image rows
                # base + {0..7} (slots 0-7) and base + 16 + {0..7} (slots 8-15)
                for g in range(4):
                    first_k = a_first_k[16 * g]
                    assert (a_first_k[16 * g:16 * g + 16] == first_k).all()
                    for j in range(16):
                        ik = 16 * g + j
                        gb, slot = (ik % 32) // 8, 8 * (ik // 32) + ik % 8
                        base = 128 * P + 32 * abid + 64 * (gb >> 1) + 8 * (gb & 1)
                        assert base + slot % 8 + 16 * (slot // 8) == first_k + j
                # sign bits: register q of step s uses shift 4 (s % 4) + q of the lane's word for steps 4 P ... 4 P + 3;
                # the kernel shifts by 8 (g % 2) once and then by 4 abid + q
                g_of_lane = lane // 16
                assert np.array_equal(4 * (step % 4), 8 * (g_of_lane % 2) + 4 * abid)
                assert (step // 4 == P).all()
    # the sign words travel like the metadata: a register swapped with its own copy puts the word of block lane
    # (row, ga) in lane groups g = 2 ga and 2 ga + 1 of the half that holds the row
    first, second = _permlane16_swap(lane.copy(), lane.copy())
    for half, reg in enumerate((first, second)):
        assert np.array_equal(reg % 32, 16 * half + lane % 16)
        assert np.array_equal(reg // 32, lane // 32)
