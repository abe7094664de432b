"""fp32 activations of up to sixteen tokens, rounded to fp16 by the kernel that reads them: bit for bit the result of converting
them first (same kernel, same order of the sums)."""
import pytest
import torch

from onebitsparsemul_amd import BinaryLinear_2_4, _native, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _defaults():
    yield
    _native.set_skinny_rows(-1)
    _native.set_skinny_enabled(True)


def _activations(tokens, k, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn((tokens, k), generator=g)
    # ties between two fp16 values, subnormal results, the largest values that still round down and the first that overflow
    x.view(-1)[::7] = torch.tensor([1 + 2.0**-11, 1 + 3 * 2.0**-11, 2.0**-25, 2.0**-24 * 1.5, 65519.99, -65504.0, 3e-39]).repeat(
        (x.numel() // 49) + 1)[: x.view(-1)[::7].numel()]
    return x


def _f32(prep, x, bias, y, m, k):
    code = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
    return _native.lib().onebit_sparse_linear_prepared_f32(
        prep.data_ptr(), x.data_ptr(), bias.data_ptr() if bias is not None else None, y.data_ptr(), x.shape[0], m, k,
        code[bias.dtype] if bias is not None else 1, code[y.dtype], torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("rows", [32, 64, 128])
@pytest.mark.parametrize("tokens", [1, 2, 7, 8, 9, 15, 16])
@pytest.mark.parametrize("m,k", [(64, 32), (192, 1056), (256, 4096), (448, 8480), (128, 16416)])
def test_equals_the_converted_call(rows, tokens, m, k):
    _native.set_skinny_rows(rows)
    a, meta = synthetic.make_weight(m, k, seed=m + k)
    prep = _native.prepare(a.cuda(), meta.cuda(), m, k)
    x = _activations(tokens, k, tokens).cuda()
    bias = synthetic.make_b(1, m, seed=3).reshape(m).cuda()
    for y_dtype, b in ((torch.float32, None), (torch.float16, bias)):
        want, got = (torch.full((tokens, m), float("nan"), dtype=y_dtype, device="cuda") for _ in range(2))
        _native.linear_prepared(prep, x.half(), want, m, k, bias=b)
        assert _f32(prep, x, b, got, m, k) == 0
        torch.cuda.synchronize()
        assert torch.equal(got, want)


def test_infinity_and_nan_stay_in_their_token():
    m, k, tokens = 128, 512, 5
    a, meta = synthetic.make_weight(m, k, seed=9)
    prep = _native.prepare(a.cuda(), meta.cuda(), m, k)
    x = _activations(tokens, k, 1)
    x[1, 3], x[3, 200], x[3, 201] = float("nan"), float("inf"), 1e30
    x = x.cuda()
    want, got = (torch.zeros((tokens, m), dtype=torch.float32, device="cuda") for _ in range(2))
    _native.linear_prepared(prep, x.half(), want, m, k)
    assert _f32(prep, x, None, got, m, k) == 0
    assert torch.equal(torch.nan_to_num(got, nan=7.0), torch.nan_to_num(want, nan=7.0))
    assert bool(torch.isfinite(got[[0, 2, 4]]).all())


def test_refusals_and_the_layer():
    m, k = 128, 512
    a, meta = synthetic.make_weight(m, k, seed=4)
    prep = _native.prepare(a.cuda(), meta.cuda(), m, k)
    y = torch.zeros((17, m), dtype=torch.float32, device="cuda")
    assert _f32(prep, torch.zeros((17, k), device="cuda"), None, y, m, k) != 0   # more tokens than the kernel takes
    storage = torch.randn(4 * k + 1, device="cuda")
    assert _f32(prep, storage[1:].view(4, k), None, y[:4], m, k) != 0             # not 16-byte aligned
    layer = BinaryLinear_2_4(k, m).cuda()
    layer.load_state_dict({"packed_binary_sparse": a.cuda(), "meta": meta.cuda()})
    x = storage[1:].view(4, k)
    for view in (x, x.clone(), x.clone().T.contiguous().T, torch.cat([x] * 5)):   # unaligned, aligned, strided, more tokens
        want = torch.empty((view.shape[0], m), dtype=torch.float32, device="cuda")
        _native.linear_prepared(prep, view.half().contiguous(), want, m, k)
        got = layer(view)
        assert got.dtype == torch.float32 and torch.equal(got, want)
    _native.set_skinny_enabled(False)  # the kernel that reads fp32 is off: the layer converts, for the main kernel
    want = torch.empty((4, m), dtype=torch.float32, device="cuda")
    _native.linear_prepared(prep, x.half().contiguous(), want, m, k)
    assert torch.equal(layer(x.clone()), want)
