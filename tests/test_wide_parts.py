"""wide_kernel where whole rounds of eight chunks leave one to four: they are dealt over the wavefronts in parts of 64 or 128 K
values. Activations are small integers and +-0.5, so every partial sum is exact in fp32 and in any order."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, dequant_desparse_tile, synthetic
from test_address_model import wide_deal, wide_has_parts


@pytest.mark.parametrize("kc_begin", [0, 13])
def test_every_image_goes_to_one_wavefront(kc_begin):
    """in both builds, for every number of chunks that either may be launched with"""
    for chunks in range(1, 60):
        for parts in (False, True):
            dealt = []
            for wave in range(8):
                mine, part = wide_deal(kc_begin, kc_begin + chunks, wave, parts)
                dealt.append([4 * kc + s for kc in mine for s in range(4)] + ([4 * part[0] + part[1] + s for s in range(part[2])] if part else []))
            assert sorted(i for images in dealt for i in images) == list(range(4 * kc_begin, 4 * (kc_begin + chunks)))
            if parts and wide_has_parts(chunks):
                assert max(len(images) for images in dealt) == chunks // 8 * 4 + (1 if chunks % 8 <= 2 else 2)


@pytest.fixture
def hooks():
    lib = _native.lib()
    yield lib
    lib.onebit_sparse_set_skinny_rows(-1)
    lib.onebit_sparse_set_split_k(-1)


# 9, 10, 11, 12 and 13 chunks, 17 of two rounds; K that ends inside an image of a part, behind its first value and at its end
@pytest.mark.gpu
@pytest.mark.parametrize("k", [2080, 2304, 2336, 2560, 2784, 2976, 3072, 3200, 4128])
@pytest.mark.parametrize("rows", [32, 64, 128])
def test_parts_equal_the_dense_product(hooks, rows, k):
    m = 192
    a, meta = synthetic.make_weight(m, k, 3, device="cuda")
    weight, dense = PreparedWeight(a, meta), dequant_desparse_tile(a.cpu(), meta.cpu()).double()
    hooks.onebit_sparse_set_skinny_rows(rows)
    g = torch.Generator().manual_seed(k)
    for i, n in enumerate((17, 24, 32, 40, 48, 64, 72)):
        dtype = (torch.float16, torch.bfloat16)[i % 2]
        x = torch.randint(-4, 5, (n, k), generator=g) / 2
        want = x.double() @ dense.T
        for splits in (1, 2):
            hooks.onebit_sparse_set_split_k(splits)
            y = torch.full((n, m), 7.0, device="cuda")
            _native.linear_prepared(weight.buffer, x.to("cuda", dtype), y, m, k)
            assert torch.equal(y.cpu(), want.float()), (n, splits)
            if n % 8 == 0:
                d = weight.matmul(x.half().T.contiguous().cuda(), out_dtype=torch.float32)
                assert torch.equal(d.cpu(), want.T.float()), (n, splits)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [17, 64])
def test_grouped_products_of_which_one_has_parts(tokens):
    problems, singles = [], []
    for i, (m, k) in enumerate(((192, 1056), (64, 2304), (448, 3584))):
        a, meta = synthetic.make_weight(m, k, i, device="cuda")
        buffer = PreparedWeight(a, meta).buffer
        x = torch.randint(-4, 5, (tokens, k), generator=torch.Generator().manual_seed(i)).half().cuda()
        y, single = torch.zeros(tokens, m, device="cuda").half(), torch.zeros(tokens, m, device="cuda").half()
        _native.linear_prepared(buffer, x, single, m, k)
        problems.append((buffer, x, y, m, k, None))
        singles.append(single)
    _native.linear_prepared_grouped(problems)
    for problem, single in zip(problems, singles):
        assert torch.equal(problem[2], single)
