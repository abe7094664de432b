"""wide_kernel on grids that are walked in strips of two column groups and on grids that are not, against the oracle on small
integers (exact in fp32): odd and even numbers of column groups, numbers of workgroups that eight does and does not divide, few of them,
K split over workgroups, a padded copy of B."""
import numpy as np
import pytest
import torch

import oracle
from onebitsparsemul_amd import _native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _defaults():
    yield
    _native.set_skinny_rows(-1)
    _native.set_split_k(-1)


def _operands(m, k, columns, seed):
    a, meta = synthetic.make_weight(m, k, seed=seed)
    return a, meta, _native.prepare(a.cuda(), meta.cuda(), m, k), synthetic.make_b(k, columns, seed=seed + 1, kind="int")


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("m,k,n", [(64, 28672, 72), (320, 8192, 248), (960, 6528, 136), (1984, 2784, 66), (704, 2144, 100), (448, 4640, 480)])
def test_layers(rows, m, k, n):
    _native.set_skinny_rows(rows)
    a, meta, prep, b = _operands(m, k, n, m + k)
    want = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k, d_dtype=oracle.F32).T
    for y_type in (torch.float32, torch.float16):
        y = torch.full((n, m), float("nan"), dtype=y_type, device="cuda")
        _native.linear_prepared(prep, b.T.contiguous().cuda(), y, m, k)
        assert torch.equal(y.cpu(), torch.from_numpy(np.ascontiguousarray(want)).to(y_type)), y_type


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("m,k,n", [(64, 28672, 72), (320, 8192, 248), (960, 6528, 88), (1984, 2784, 65), (704, 2144, 346), (448, 4640, 600)])
@pytest.mark.parametrize("splits", [1, 3])
def test_products(rows, m, k, n, splits):
    _native.set_skinny_rows(rows)
    _native.set_split_k(splits)
    a, meta, prep, b = _operands(m, k, n, m + n)
    c = torch.from_numpy(np.random.default_rng(n).integers(-8, 9, (m, n))).to(torch.float16)
    d = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda")
    _native.matmul_prepared(prep, b.cuda(), d, m, n, k, c=c.cuda(), alpha=0.5, beta=2.0)
    want = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k, c=c.float().numpy(), alpha=0.5, beta=2.0,
                                   d_dtype=oracle.F32)
    assert np.array_equal(d.cpu().numpy(), want)
