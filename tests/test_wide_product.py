"""Products of 17 columns or more on few weight rows: column groups and their remainders, ends of K inside an image, row groups
past M, padded copies of B, alpha, beta and C of either type, K splits. Integer operands: results must equal the dense product."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, dequant_desparse_tile, synthetic

pytestmark = pytest.mark.gpu


@pytest.fixture
def hooks():
    lib = _native.lib()
    yield lib
    lib.onebit_sparse_set_skinny_rows(-1)
    lib.onebit_sparse_set_split_k(-1)


@pytest.mark.parametrize("m,k", [(64, 32), (192, 1056), (448, 96), (320, 4640)])
@pytest.mark.parametrize("rows", [-1, 32, 64, 128])
def test_columns_equal_the_dense_product(hooks, m, k, rows):
    a, meta = synthetic.make_weight(m, k, 3, device="cuda")
    weight, dense = PreparedWeight(a, meta), dequant_desparse_tile(a.cpu(), meta.cpu()).double()
    g = torch.Generator().manual_seed(m + k)
    hooks.onebit_sparse_set_skinny_rows(rows)
    for i, n in enumerate((24, 32, 40, 48, 56, 64, 65, 72, 99, 104, 136, 200, 257)):
        b = torch.randint(-4, 5, (k, n), generator=g).half()
        c = torch.randint(-4, 5, (m, n), generator=g).to((torch.float16, torch.float32)[i % 2])
        for splits in (-1, 2, 3):
            hooks.onebit_sparse_set_split_k(splits)
            d = torch.full((m + 1, n), 7.0, device="cuda")
            weight.matmul(b.cuda(), out=d[:m], c=c.cuda(), alpha=0.5, beta=2.0)
            assert torch.equal(d[:m].cpu(), (0.5 * (dense @ b.double()) + 2.0 * c.double()).float()), (n, splits)
            assert bool((d[m] == 7).all())
        assert torch.equal(weight.matmul(b.cuda()).cpu(), (dense @ b.double()).half())


@pytest.mark.parametrize("n", [72, 104, 200])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_result_over_c(n, dtype):
    """D may be C. Column groups of an odd number of 16-byte pieces (40 of 72 columns) do not reach into the next group, which
    would add C twice there."""
    m, k = 1024, 2048
    a, meta = synthetic.make_weight(m, k, 5, device="cuda")
    weight, dense = PreparedWeight(a, meta), dequant_desparse_tile(a.cpu(), meta.cpu()).double()
    g = torch.Generator().manual_seed(n)
    b = torch.randint(-1, 2, (k, n), generator=g).half()
    c = torch.randint(-4, 5, (m, n), generator=g).to(dtype)
    d = c.cuda()
    weight.matmul(b.cuda(), out=d, c=d, alpha=1.0, beta=1.0)
    assert torch.equal(d.cpu(), (dense @ b.double() + c.double()).to(dtype))


def test_small_unaligned_b_leaves_the_buffer_of_a_captured_graph():
    """The padded copy of B (576 x 119, the larger in values) is the smaller in bytes: the second call must not replace the
    buffer that the graph reads. Both start at an odd value, where a copy is made whatever kernel reads it."""
    assert _native.describe_launch(256, 119, 576, b_aligned=False, compute_units=None)["pad_b"]
    stream = torch.cuda.Stream()
    weights = {k: synthetic.make_weight(256, k, k, device="cuda") for k in (576, 992)}
    prepared = {k: PreparedWeight(*w) for k, w in weights.items()}
    dense = {k: dequant_desparse_tile(w[0].cpu(), w[1].cpu()).double() for k, w in weights.items()}
    g = torch.Generator().manual_seed(1)
    large, small = (torch.randint(-4, 5, shape, generator=g).half() for shape in ((576, 119), (992, 66)))
    large_gpu, small_gpu = (torch.empty(b.numel() + 1, dtype=b.dtype, device="cuda")[1:].view(b.shape).copy_(b) for b in (large, small))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        prepared[576].matmul(large_gpu)
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            d = prepared[576].matmul(large_gpu)
        for _ in range(3):
            got = prepared[992].matmul(small_gpu)
            d.zero_()
            graph.replay()
            stream.synchronize()
            assert torch.equal(got.cpu(), (dense[992] @ small.double()).half())
            assert torch.equal(d.cpu(), (dense[576] @ large.double()).half())
