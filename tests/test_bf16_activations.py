"""The token-major form on bf16 activations: multiplied as they are, fp32 accumulation, one rounding to bf16. Integer
activations (exact in bf16) make every sum exact in fp32, so fp32 results equal the oracle's bit for bit and bf16 results
equal its fp32 result rounded once."""
import numpy as np
import pytest
import torch

import oracle
import onebitsparsemul_amd as ob
from onebitsparsemul_amd import _native, synthetic

pytestmark = pytest.mark.gpu


def expected(a, meta, x, bias, m, k):
    tokens = x.shape[0]
    want = oracle.reference_matmul(a.numpy(), x.T.contiguous().numpy(), meta.numpy(), m, tokens, k, d_dtype=oracle.F32)
    return torch.from_numpy(want.T.copy()) + (0 if bias is None else bias.float())


def check(m, k, tokens, seed, bias_type=torch.bfloat16):
    a, meta = synthetic.make_weight(m, k, seed=seed)
    prepared = _native.prepare(a.cuda(), meta.cuda(), m, k)
    x = synthetic.make_b(tokens, k, seed=seed, kind="int")
    bias = None if bias_type is None else torch.from_numpy(np.random.default_rng(seed).integers(-8, 9, m)).to(bias_type)
    want = expected(a, meta, x, bias, m, k)
    for out in (torch.bfloat16, torch.float32):
        y = torch.full((tokens, m), float("nan"), dtype=out, device="cuda")
        _native.linear_prepared(prepared, x.bfloat16().cuda(), y, m, k, bias=None if bias is None else bias.cuda())
        torch.cuda.synchronize()
        assert torch.equal(y.cpu(), want.to(out)), (m, k, tokens, out)


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("tokens", [1, 16, 17, 33, 64])
def test_split_k_kernel(rows, tokens):
    _native.set_skinny_rows(rows)
    try:
        check(320, 288, tokens, seed=tokens, bias_type=torch.float32)
        check(192, 4128, tokens, seed=tokens)
    finally:
        _native.set_skinny_rows(-1)


@pytest.mark.parametrize("tile,m", [(4, 320), (6, 192), (9, 576), (10, 320), (11, 192), (12, 128), (13, 192), (14, 128), (15, 576)])
@pytest.mark.parametrize("splits", [1, 2])
def test_main_kernel_tiles(tile, m, splits):
    _native.set_tile_config(tile)
    _native.set_skinny_enabled(False)
    _native.set_split_k(splits)
    try:
        check(m, 544, 65, seed=tile)
        check(m, 800, 130, seed=tile, bias_type=None)
    finally:
        _native.set_tile_config(-1)
        _native.set_skinny_enabled(True)
        _native.set_split_k(-1)


@pytest.mark.parametrize("tokens", [3, 70])
def test_layer_and_group_with_bf16_bias(tokens):
    k, sizes = 288, (192, 64)
    layers, wants = [], []
    x = synthetic.make_b(tokens, k, seed=5, kind="int")
    for i, m in enumerate(sizes):
        a, meta = synthetic.make_weight(m, k, seed=i)
        layer = ob.BinaryLinear_2_4(k, m).cuda()
        layer.load_state_dict({"packed_binary_sparse": a, "meta": meta})
        layer.bias = torch.arange(m).remainder(17).bfloat16().cuda()
        layers.append(layer)
        wants.append(expected(a, meta, x, layer.bias.cpu(), m, k).bfloat16())
    x = x.bfloat16().cuda()
    ys = ob.forward_grouped(layers, x)
    for layer, want, y in zip(layers, wants, ys):
        assert y.dtype == torch.bfloat16 and torch.equal(y.cpu(), want)
        assert torch.equal(layer(x).cpu(), want)
