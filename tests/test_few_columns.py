"""skinny_kernel with two to eight columns, read by fours of K positions, and with one to sixteen tokens by the number of load
instructions that take them: every count, K that ends inside an image, wavefronts with one, two and three chunks (requested at once on
sixteen wavefronts) and more, the last of them without a last one. Operands are small integers and halves, so sums are exact in any order."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, dequant_desparse_tile, synthetic
from test_address_model import check_columns_image

KS = [32, 256, 288, 2080, 4128, 8224, 11008, 12288, 12320]  # 1, 1, 2, 9, 17, 33, 43, 48 and 49 chunks


@pytest.mark.parametrize("n", range(2, 9))
def test_fours_of_k_positions(n):
    """the loads of a lane stay inside B and what it stores is found by the reads as the columns of its four K positions; K that ends inside
    an image, at its end and before it"""
    for k in (32, 96, 256, 288, 512):
        for k_base in range(0, k + 512, 256):
            check_columns_image(n, k, k_base)


@pytest.fixture
def hooks():
    lib = _native.lib()
    yield lib
    lib.onebit_sparse_set_skinny_rows(-1)
    lib.onebit_sparse_set_split_k(-1)


def weight_of(m, k):
    a, meta = synthetic.make_weight(m, k, 3, device="cuda")
    return PreparedWeight(a, meta), dequant_desparse_tile(a.cpu(), meta.cpu()).double()


@pytest.mark.gpu
@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("rows", [32, 64, 128])
def test_columns_equal_the_dense_product(hooks, rows, k):
    m = 192
    weight, dense = weight_of(m, k)
    hooks.onebit_sparse_set_skinny_rows(rows)
    g = torch.Generator().manual_seed(k)
    for n in range(1, 10):
        b = torch.randint(-4, 5, (k, n), generator=g).half()
        c = torch.randint(-4, 5, (m, n), generator=g).to((torch.float16, torch.float32)[n % 2])
        at_the_end = torch.full((k * n + 64,), float("nan"), dtype=torch.float16, device="cuda")[64:].view(k, n)
        at_the_end.copy_(b)
        product = dense @ b.double()
        for splits in (1, 2):
            hooks.onebit_sparse_set_split_k(splits)
            d = torch.full((m + 1, n), 7.0, device="cuda")
            weight.matmul(at_the_end, out=d[:m], c=c.cuda(), alpha=0.5, beta=2.0)
            assert torch.equal(d[:m].cpu(), (0.5 * product + 2.0 * c.double()).float()), (n, splits)
            assert bool((d[m] == 7).all())
        assert torch.equal(weight.matmul(at_the_end).cpu(), product.half()), n


@pytest.mark.gpu
@pytest.mark.parametrize("k", KS)
@pytest.mark.parametrize("rows", [32, 64, 128])
def test_tokens_equal_the_dense_product(hooks, rows, k):
    m = 192
    weight, dense = weight_of(m, k)
    hooks.onebit_sparse_set_skinny_rows(rows)
    g = torch.Generator().manual_seed(k)
    for tokens in range(1, 17):
        x = torch.randint(-4, 5, (tokens, k), generator=g) / 2
        want = (x.double() @ dense.T).float()
        for dtype in (torch.float16, torch.bfloat16, torch.float32):
            y = torch.full((tokens + 1, m), 7.0, device="cuda")
            if dtype == torch.float32:
                rc = _native.lib().onebit_sparse_linear_prepared_f32(weight.buffer.data_ptr(), x.cuda().data_ptr(), None, y.data_ptr(),
                                                                     tokens, m, k, 0, 0, torch.cuda.current_stream().cuda_stream)
                assert rc == 0, _native.last_error()
            else:
                _native.linear_prepared(weight.buffer, x.to("cuda", dtype), y[:tokens], m, k)
            torch.cuda.synchronize()
            assert torch.equal(y[:tokens].cpu(), want) and bool((y[tokens] == 7).all()), (tokens, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 3, 6, 10, 16])
def test_grouped_equals_single(tokens):
    problems, singles = [], []
    for i, (m, k) in enumerate(((192, 1056), (64, 8224), (448, 12320))):
        weight = weight_of(m, k)[0]
        x = torch.randint(-4, 5, (tokens, k), generator=torch.Generator().manual_seed(i)).half().cuda()
        y, single = torch.zeros(tokens, m, device="cuda").half(), torch.zeros(tokens, m, device="cuda").half()
        _native.linear_prepared(weight.buffer, x, single, m, k)
        problems.append((weight.buffer, x, y, m, k, None))
        singles.append(single)
    _native.linear_prepared_grouped(problems)
    for problem, single in zip(problems, singles):
        assert torch.equal(problem[2], single)
