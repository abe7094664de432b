"""The split-K kernel's two argument forms, on either side of the lines between them (eight and sixteen chunks of K per split, ten to
fourteen columns in whole words or not), with all that a call can pass: C of either type, alpha, beta, results of either type, K split or
not. Integer operands:
bit-exact."""
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


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 10, 13, 14, 16, 18, 32, 41, 64])
def test_every_argument_reaches_the_kernel(rows, n):
    _native.set_skinny_rows(rows)
    for m, k, splits in ((192, 2048, 1), (192, 2080, 1), (192, 4096, 1), (192, 4128, 1), (64, 8192, 2), (64, 8224, 2)):
        _native.set_split_k(splits)
        a, meta = synthetic.make_weight(m, k, seed=n + k)
        prepared = _native.prepare(a.cuda(), meta.cuda(), m, k)
        b = synthetic.make_b(k, n, seed=n, kind="int")
        c = torch.from_numpy(np.random.default_rng(n).integers(-8, 9, (m, n))).to(torch.float32)
        for c_type, out in ((None, torch.float16), (torch.float16, torch.float32), (torch.float32, torch.float16), (None, torch.float32)):
            # one element beyond a 16-byte boundary: the pieces of every column count
            for shift in (0, 1):
                flat = torch.zeros(k * n + shift, dtype=torch.float16, device="cuda")
                flat[shift:] = b.reshape(-1).cuda()
                d = torch.full((m, n), float("nan"), dtype=out, device="cuda")
                scale = dict(alpha=0.5, beta=2.0) if c_type else dict(alpha=1.0, beta=0.0)
                _native.matmul_prepared(prepared, flat[shift:].view(k, n), d, m, n, k,
                                        c=None if c_type is None else c.to(c_type).cuda(), **scale)
                torch.cuda.synchronize()
                want = oracle.reference_matmul(a.numpy(), b.numpy(), meta.numpy(), m, n, k, c=None if c_type is None else c.numpy(),
                                               d_dtype=oracle.F16 if out == torch.float16 else oracle.F32, **scale)
                assert np.array_equal(d.cpu().numpy(), want), (k, splits, c_type, out, shift)
