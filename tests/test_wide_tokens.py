"""The linear layer with 17 to 64 tokens: every row group and copy count, ends of K inside an image, row groups that reach past
M, K splits. Activations are small integers and +-0.5, so every partial sum is exact in fp32 and in any order: results must equal
the dense product."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, dequant_desparse_tile, synthetic

pytestmark = pytest.mark.gpu


def _dense(a, meta):
    return dequant_desparse_tile(a.cpu(), meta.cpu()).double()


@pytest.fixture
def hooks():
    lib = _native.lib()
    yield lib
    lib.onebit_sparse_set_skinny_rows(-1)
    lib.onebit_sparse_set_split_k(-1)


@pytest.mark.parametrize("m,k", [(64, 32), (192, 96), (448, 1056), (320, 2336), (192, 4640)])
@pytest.mark.parametrize("rows", [-1, 32, 64, 128])
def test_every_copy_count_equals_the_dense_product(hooks, m, k, rows):
    a, meta = synthetic.make_weight(m, k, 3, device="cuda")
    weight, dense = PreparedWeight(a, meta), _dense(a, meta)
    hooks.onebit_sparse_set_skinny_rows(rows)
    g = torch.Generator().manual_seed(m + k)
    for i, tokens in enumerate((17, 24, 25, 32, 33, 40, 41, 48, 49, 56, 57, 64)):
        dtype = (torch.float16, torch.bfloat16)[i % 2]
        x = torch.randint(-4, 5, (tokens, k), generator=g) / 2
        bias = torch.randint(-4, 5, (m,), generator=g).float()
        want = (x.double() @ dense.T + bias).float()
        for splits in (1, 2, 3):
            hooks.onebit_sparse_set_split_k(splits)
            y = torch.full((tokens, m), 7.0, device="cuda")
            _native.linear_prepared(weight.buffer, x.to("cuda", dtype), y, m, k, bias=bias.cuda())
            assert torch.equal(y.cpu(), want), (tokens, splits)
        got = weight.linear(x.to("cuda", dtype), bias=bias.cuda(), out_dtype=dtype)
        assert torch.equal(got.cpu(), want.to(dtype)), tokens


@pytest.mark.parametrize("tokens", [17, 31, 48, 64])
def test_grouped_equals_single(tokens):
    problems, singles = [], []
    for i, (m, k) in enumerate(((192, 1056), (64, 4640), (448, 1056))):
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


def test_values_behind_the_last_token_do_not_matter():
    """x and y are slices of larger buffers: infinities behind x are not read into results, and y's neighbours stay."""
    m, k, tokens = 192, 352, 19
    a, meta = synthetic.make_weight(m, k, 9, device="cuda")
    x = torch.full((tokens + 8, k), float("inf"), device="cuda", dtype=torch.float16)
    x[:tokens] = torch.randint(-4, 5, (tokens, k), device="cuda").half()
    y = torch.full((tokens + 1, m), 7.0, device="cuda")
    _native.linear_prepared(PreparedWeight(a, meta).buffer, x[:tokens], y[:tokens], m, k)
    assert torch.equal(y[:tokens].cpu().double(), x[:tokens].cpu().double() @ _dense(a, meta).T)
    assert bool((y[tokens] == 7).all())


@pytest.mark.parametrize("m,k,tokens", [(64, 32, 65), (192, 1056, 100), (448, 96, 257), (1024, 512, 129), (512, 4640, 70)])
def test_more_tokens_than_one_workgroup_takes(m, k, tokens):
    a, meta = synthetic.make_weight(m, k, 4, device="cuda")
    x = torch.randint(-4, 5, (tokens, k), generator=torch.Generator().manual_seed(tokens)) / 2
    want = (x.double() @ _dense(a, meta).T).float()
    for dtype in (torch.float16, torch.bfloat16):
        y = torch.full((tokens + 1, m), 7.0, device="cuda")
        _native.linear_prepared(PreparedWeight(a, meta).buffer, x.to("cuda", dtype), y[:tokens], m, k)
        assert torch.equal(y[:tokens].cpu(), want) and bool((y[tokens] == 7).all())
