"""Products whose number of columns is no multiple of the 16-byte vectors: rows of C and D start at any element, the last
piece of a row is cut short, the last one of C lies at the end of its memory. Integer operands: bit-exact."""
import numpy as np
import pytest
import torch

import oracle
from onebitsparsemul_amd import _native, synthetic

pytestmark = pytest.mark.gpu


def guarded(values, shift):
    """A copy of `values` on the GPU, `shift` elements into a buffer that ends with it exactly; the buffer too."""
    flat = torch.full((values.numel() + shift,), 7.0, dtype=values.dtype, device="cuda")
    flat[shift:] = values.reshape(-1).cuda()
    return flat[shift:].view(values.shape), flat


@pytest.mark.parametrize("tile,m,k", [(9, 576, 288), (10, 320, 544), (4, 320, 288), (6, 192, 288), (13, 192, 544), (14, 128, 544),
                                      (15, 576, 288)])
@pytest.mark.parametrize("n", [65, 127, 131, 257])
def test_main_kernel_ragged_rows(tile, m, k, n):
    _native.set_tile_config(tile)
    _native.set_skinny_enabled(False)
    try:
        a, meta = synthetic.make_weight(m, k, seed=tile + n)
        prepared = _native.prepare(a.cuda(), meta.cuda(), m, k)
        b = synthetic.make_b(k, n, seed=n, kind="int")
        c = torch.from_numpy(np.random.default_rng(n).integers(-8, 9, (m, n))).to(torch.float32)
        for c_type, out, shift in ((None, torch.float16, 1), (torch.float16, torch.float16, 3), (torch.float32, torch.float16, 0),
                                   (torch.float16, torch.float32, 1), (torch.float32, torch.float32, 3), (None, torch.float32, 0)):
            c_gpu = None if c_type is None else guarded(c.to(c_type), shift)[0]
            d, flat = guarded(torch.zeros((m, n), dtype=out), shift)
            _native.matmul_prepared(prepared, guarded(b, shift)[0], d, m, n, k, c=c_gpu, alpha=0.5 if c_type else 1.0,
                                    beta=0.0 if c_type is None else 2.0)
            torch.cuda.synchronize()
            want = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k,
                                           c=None if c_type is None else c.numpy(), alpha=0.5 if c_type else 1.0,
                                           beta=0.0 if c_type is None else 2.0,
                                           d_dtype=oracle.F16 if out == torch.float16 else oracle.F32)
            assert np.array_equal(d.cpu().numpy(), want), (c_type, out, shift)
            assert bool((flat[:shift] == 7.0).all())
    finally:
        _native.set_tile_config(-1)
        _native.set_skinny_enabled(True)


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 3, 4, 7, 8, 9, 15, 17, 24, 25, 33, 40, 49, 63])
def test_split_k_kernel_any_columns(rows, n):
    """B rows that start at any element: every count of 16-byte pieces per row, the end of B inside a piece, K tails that leave
    the last image with 32 rows or end it exactly."""
    _native.set_skinny_rows(rows)
    try:
        for m, k, shift in ((192, 256, 1), (64, 2592, 0), (320, 4128, 3), (128, 512, 2)):
            a, meta = synthetic.make_weight(m, k, seed=n + k)
            prepared = _native.prepare(a.cuda(), meta.cuda(), m, k)
            b = synthetic.make_b(k, n, seed=n, kind="int")
            d = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
            _native.matmul_prepared(prepared, guarded(b, shift)[0], d, m, n, k)
            torch.cuda.synchronize()
            want = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k)
            assert np.array_equal(d.cpu().numpy(), want), (m, k, shift)
    finally:
        _native.set_skinny_rows(-1)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 7, 9])
@pytest.mark.parametrize("k", [28672, 65536])
def test_padded_copy_of_rows_shorter_than_a_piece(n, k):
    """Several of B's last rows end within one 16-byte piece of its end (or all of them, n < 8)."""
    m = 64
    a, meta = synthetic.make_weight(m, k, seed=n)
    b = synthetic.make_b(k, n, seed=n, kind="int")
    _native.set_skinny_enabled(False)
    try:
        d = torch.empty((m, n), dtype=torch.float32, device="cuda")
        _native.matmul_prepared(_native.prepare(a.cuda(), meta.cuda(), m, k), b.cuda(), d, m, n, k)
    finally:
        _native.set_skinny_enabled(True)
    ref = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k, d_dtype=oracle.F32)
    assert np.array_equal(d.cpu().numpy(), ref)
