"""Token-major form of the main kernel: its results and biases at any alignment, through every tile that has the form, against
the oracle on small integers (sums below 2^24 are exact in fp32; the one rounding to the result's type is torch's)."""
import numpy as np
import pytest
import torch

import oracle
from onebitsparsemul_amd import _native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _defaults():
    yield
    _native.set_tile_config(-1)
    _native.set_skinny_enabled(True)


@pytest.mark.parametrize("tile", [4, 6, 9, 10, 11, 12, 13, 14, 15])
@pytest.mark.parametrize("tokens,m,k", [(1, 64, 256), (129, 576, 544), (131, 704, 800)])
def test_results_and_biases_off_16_byte_boundaries(tile, tokens, m, k):
    _native.set_tile_config(tile)
    _native.set_skinny_enabled(False)
    a, meta = synthetic.make_weight(m, k, seed=m + tokens)
    x = synthetic.make_b(tokens, k, seed=tokens, kind="int")
    sums = oracle.host_gemm(oracle.decompress_operands(a.numpy(), meta.numpy(), m, k),
                            np.ascontiguousarray(x.numpy().astype(np.float32).T), d_dtype=oracle.F32, acc="f32").T
    prep = _native.prepare(a.cuda(), meta.cuda(), m, k)
    values = synthetic.make_b(1, m + 1, seed=tokens + 1, kind="int").reshape(m + 1)
    for x_type, y_type in ((torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)):
        for bias_type in (None, torch.float16, torch.bfloat16, torch.float32):
            bias = None if bias_type is None else values.to(bias_type).cuda()[1:]
            store = torch.full((tokens * m + 2,), float("nan"), dtype=y_type, device="cuda")
            y = store[1:-1].view(tokens, m)
            _native.linear_prepared(prep, x.to(x_type).cuda(), y, m, k, bias=bias)
            torch.cuda.synchronize()
            want = torch.from_numpy(sums + (0 if bias is None else values[1:].float().numpy()[None, :])).to(y_type)
            assert torch.equal(y.cpu(), want), (y_type, bias_type)
            assert bool(store[0].isnan()) and bool(store[-1].isnan()), (y_type, bias_type)  # nothing beside y is written
