"""Calls of more than 64 columns or tokens that wide_kernel takes because its workgroups have a compute unit each, or because it splits
K less: the plan on either side of that line, and the product where rows, columns, K ranges and chunks end raggedly."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, dequant_desparse_tile, synthetic


# layers and products, workgroups of 64 and 128 rows, groups of 32, 48 and 64 columns, the main kernel with and without a K split
CALLS = [(True, 3520, 206, 1248), (True, 1216, 1077, 3808), (True, 704, 985, 7456), (False, 1088, 416, 672), (False, 1856, 471, 2400),
         (False, 2560, 440, 5376)]
SPLIT_CALLS = [(True, 576, 484, 10848), (False, 704, 280, 15360)]


def groups(plan, m, n):
    return -(-m // plan["rows"]) * -(-n // plan["columns"])


@pytest.mark.parametrize("tokens,m,n,k", CALLS)
def test_one_round_of_workgroups(tokens, m, n, k):
    plan = _native.describe_launch(m, n, k, tokens=tokens)
    assert plan["kernel"] == "wide_kernel" and plan["splits"] == 1 and groups(plan, m, n) <= 256


@pytest.mark.parametrize("tokens,m,n,k", [(True, 5568, 334, 5376), (True, 14784, 91, 1408), (True, 1792, 1250, 7328), (False, 768, 616, 8192)])
def test_more_rounds_and_split_products_stay_on_the_main_kernel(tokens, m, n, k):
    assert _native.describe_launch(m, n, k, tokens=tokens)["kernel"] == "gemm_kernel"


# long K, the main kernel in splits of it: on either side of the lines by chunks, tile and rows of a group
@pytest.mark.parametrize("m,n,k,wide", [(2048, 846, 27552, False), (3776, 496, 26336, False), (2240, 679, 16224, False),
                                        (1280, 295, 22304, False), (2048, 1001, 15648, True), (3328, 465, 17440, True),
                                        (3712, 228, 17984, True), (960, 329, 17696, True)])
def test_long_k_of_layers(m, n, k, wide):
    """us on the main kernel | on wide_kernel: 61.6 | 70.2, 61.9 | 67.0, 39.7 | 42.5, 24.4 | 26.4; the others are 0.85 to 0.88 of the time"""
    plan = _native.describe_launch(m, n, k, tokens=True)
    assert (plan["kernel"] == "wide_kernel") == wide and (wide or plan["splits"] > 1)


@pytest.mark.parametrize("tokens,m,n,k", SPLIT_CALLS)
def test_split_plans(tokens, m, n, k):
    plan = _native.describe_launch(m, n, k, tokens=tokens)
    assert plan["kernel"] == "wide_kernel" and plan["splits"] >= 3


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,m,n,k", CALLS + SPLIT_CALLS)
def test_products_equal_the_dense_ones(tokens, m, n, k):
    """Activations are small integers and +-0.5: every partial sum is exact in fp32 and in any order."""
    a, meta = synthetic.make_weight(m, k, 3, device="cuda")
    weight, dense = PreparedWeight(a, meta), dequant_desparse_tile(a.cpu(), meta.cpu()).float()
    x = torch.randint(-4, 5, (n, k), generator=torch.Generator().manual_seed(k)) / 2
    want = x @ dense.T
    if tokens:
        y = torch.full((n, m), 7.0, device="cuda")
        _native.linear_prepared(weight.buffer, x.half().cuda(), y, m, k)
        assert torch.equal(y.cpu(), want)
    else:
        d = weight.matmul(x.half().T.contiguous().cuda(), out_dtype=torch.float32)
        assert torch.equal(d.cpu(), want.T)
