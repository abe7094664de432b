"""Products whose number of columns is no multiple of eight: the asynchronous copies read the rows of B where they lie, a
piece at the end of a row takes values of the next one along, and the last row's last piece is moved back inside B and shifted into
place in LDS. Integer operands: bit-exact. B ends where its memory ends."""
import numpy as np
import pytest
import torch

from onebitsparsemul_amd import _native, dequant_desparse_tile, synthetic


def pieces_of_b(m, n, k, width):
    """(row, first column of the group, piece of the group, start, after the shift) of each 16-byte copy as the kernels form it, in values"""
    last = k * n - 8
    for first in range(0, n, width):
        for row in (0, 1, k - 2, k - 1):
            for piece in range(width // 8):
                col = 8 * piece if first + 8 * piece < n else 0
                start = row * n + first + col
                yield row, first, piece, min(start, last), max(0, start - last)


@pytest.mark.parametrize("n", [8, 9, 10, 18, 30, 63, 66, 102, 130, 1001, 1002])
@pytest.mark.parametrize("k", [32, 96, 320])
def test_copies_stay_inside_b_and_bring_every_value_that_is_used(n, k):
    for width in (16, 32, 48, 64, 128):
        for row, first, piece, start, shift in pieces_of_b(64, n, k, width):
            assert 0 <= start and start + 8 <= k * n
            columns = [c for c in range(first + 8 * piece, min(first + 8 * piece + 8, first + width)) if c < n]
            if columns:  # the kernels shift by what the last row's last piece lacks, and no other piece
                lacks = first + 8 * piece + 8 - n if row == k - 1 and piece == (n - 1 - first) // 8 else 0
                assert shift == max(0, lacks)
                assert [start + shift + i for i in range(len(columns))] == [row * n + c for c in columns]


def test_which_calls_read_b_where_it_lies():
    def plan(m, n, k, **kw):
        return _native.describe_launch(m, n, k, **kw)
    assert plan(4096, 1002, 4096)["pad_b"] is False and plan(4096, 1001, 4096)["pad_b"] is True
    assert plan(4096, 1002, 4096, b_aligned=False)["pad_b"] is True
    assert plan(4096, 100, 4096)["kernel"] == "wide_kernel" and plan(4096, 100, 4096)["pad_b"] is False
    assert all(plan(4096, n, 4096)["kernel"] == "wide_kernel" for n in (49, 50))
    assert plan(11008, 1001, 4096)["pad_b"] is False and plan(11008, 1001, 4096, b_aligned=False)["pad_b"] is True
    split = plan(512, 258, 16384)
    assert split["splits"] > 1 and split["pad_b"] is True


# an odd n on either side of the lines by chunks, of the 256 x 128, the 128 x 128 tile in two K groups and the 64 x 128 one
@pytest.mark.parametrize("m,n,k,tile,padded", [(21312, 969, 3872, 4, True), (21312, 969, 3840, 4, False), (26112, 85, 1536, 13, True),
                                               (26112, 85, 1280, 13, False), (9728, 333, 1696, 13, False), (12480, 73, 1600, 12, True),
                                               (12480, 83, 1120, 12, False), (6272, 225, 1568, 12, False)])
def test_odd_counts_are_copied_where_that_is_faster(m, n, k, tile, padded):
    """us through the copy | in place: 21312 x 3872 with 969 columns 96.4 | 100.3, 26112 x 1536 with 85 14.1 | 14.9, 12480 x 1600 with 73
    12.5 | 13.7"""
    plan = _native.describe_launch(m, n, k)
    assert (plan["tile"], plan["pad_b"]) == (tile, padded)


@pytest.mark.parametrize("m,n,k,wide", [(1600, 22, 320, False), (8192, 30, 1024, False), (8256, 30, 1024, True), (8192, 30, 1056, True),
                                        (8192, 34, 1024, True), (4160, 35, 8192, False), (2368, 17, 8192, False), (5376, 45, 8096, False),
                                        (4096, 35, 7936, True), (4096, 35, 8224, True), (4096, 35, 8192, True), (4096, 49, 8192, True), (4096, 36, 8192, True)])
def test_up_to_64_columns_go_where_they_are_faster(m, n, k, wide):
    """us, skinny_kernel | wide_kernel in place: 1600 x 320 with 22 columns and a C 3.8 | 4.2, 4160 x 8192 with 35 14.3 | 18.7, 2368 x 8192
    with 17 9.4 | 11.5, 5376 x 8096 with 45 15.4 | 18.9"""
    assert (_native.describe_launch(m, n, k)["kernel"] == "wide_kernel") == wide


@pytest.fixture
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


def check(m, n, k, seed, prepared, dense):
    """pad_b off: every tile and column group in place, not only where the plan has it so"""
    _native.set_pad_b(False)
    b = synthetic.make_b(k, n, seed=seed, kind="int")
    c = torch.from_numpy(np.random.default_rng(seed).integers(-8, 9, (m, n))).to(torch.float32)
    at_the_end = torch.full((k * n + 64,), float("nan"), dtype=torch.float16, device="cuda")[64:].view(k, n)  # 128-byte aligned
    at_the_end.copy_(b)
    for out in (torch.float16, torch.float32):
        d = torch.full((m + 1, n), 7.0, dtype=out, device="cuda")
        _native.matmul_prepared(prepared, at_the_end, d[:m], m, n, k, c=c.cuda(), alpha=0.5, beta=2.0)
        assert torch.equal(d[:m].cpu(), (0.5 * (dense @ b.double()) + 2.0 * c.double()).to(out)), (n, out)
        assert bool((d[m] == 7).all())


# K whose last row is the last of a stage of 64, its middle, and its 32nd; one stage, a chunk, more than a chunk behind whole ones
@pytest.mark.gpu
@pytest.mark.parametrize("k", [32, 64, 256, 288, 320, 544, 1024])
@pytest.mark.parametrize("tile,m", [(9, 576), (10, 320), (4, 320), (6, 192), (11, 192), (12, 128), (13, 192), (14, 128), (15, 576)])
def test_main_kernel(hooks, tile, m, k):
    _native.set_tile_config(tile)
    _native.set_skinny_enabled(False)
    a, meta = synthetic.make_weight(m, k, seed=tile + k)
    prepared = _native.prepare(a.cuda(), meta.cuda(), m, k)
    dense = dequant_desparse_tile(a, meta).double()
    for n in (65, 66, 71, 126, 130, 131, 132, 257, 258):
        for splits in (1, 2) if k >= 544 else (1,):
            _native.set_split_k(splits)
            check(m, n, k, n + k, prepared, dense)


@pytest.mark.gpu
@pytest.mark.parametrize("k", [32, 64, 320, 1056, 2048, 2336, 2560])
@pytest.mark.parametrize("rows", [32, 64, 128])
def test_wide_kernel(hooks, rows, k):
    _native.set_skinny_rows(rows)
    weights = {}
    for m in (2112, 576, 8256):
        a, meta = synthetic.make_weight(m, k, seed=rows + k)
        weights[m] = _native.prepare(a.cuda(), meta.cuda(), m, k), dequant_desparse_tile(a, meta).double()
    for n in (17, 18, 20, 22, 23, 26, 34, 39, 42, 46, 50, 57, 58, 62, 63, 66, 98, 114, 127):
        # rows from which on wide_kernel multiplies these columns; beyond 64 few rows, and not on the shortest K
        m = 576 if n > 64 else 8256 if n % 2 == 0 and n <= 32 and k <= 1024 else 2112
        for splits in (1, 2) if k >= 1056 else (1,):
            if n > 64 and k < splits * (1024 if rows == 128 else 256):
                continue
            _native.set_split_k(splits)
            _native.set_pad_b(False)
            plan = _native.describe_launch(m, n, k)
            assert (plan["kernel"], plan["rows"], plan["pad_b"]) == ("wide_kernel", rows, False), (m, n, splits)
            check(m, n, k, n + k, *weights[m])
