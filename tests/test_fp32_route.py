"""Which fp32 activations of a layer the kernel reads itself, and which are converted in front of it."""
import pytest
import torch

from onebitsparsemul_amd import BinaryLinear_2_4, _native, synthetic


@pytest.fixture(autouse=True)
def _defaults():
    yield
    _native.set_skinny_rows(-1)
    _native.set_skinny_enabled(True)


def _layer(m, k):
    a, meta = synthetic.make_weight(m, k, seed=m + k)
    layer = BinaryLinear_2_4(k, m).cuda()
    layer.load_state_dict({"packed_binary_sparse": a.cuda(), "meta": meta.cuda()})
    return layer


def test_few_tokens_through_the_kernel_that_is_on():
    def reads(*size):
        return _native.lib().onebit_sparse_linear_reads_f32(*size, None)
    assert reads(1, 4096, 4096) == 1 and reads(16, 4096, 4096) == 1 and reads(17, 4096, 4096) == 0
    assert reads(0, 4096, 4096) == 0 and reads(4, 100, 4096) == 0
    _native.set_skinny_enabled(False)
    assert reads(1, 4096, 4096) == 0


@pytest.mark.parametrize("tokens,m,k,faster", [
    (16, 4096, 9568, 1), (16, 4096, 12192, 0), (9, 8192, 12256, 1), (9, 8192, 15616, 0),  # one round of workgroups
    (8, 4096, 28672, 1), (16, 4096, 28672, 1), (16, 8192, 28672, 0), (16, 11008, 28672, 0),  # K in four, in two, not split
    (8, 7168, 18720, 1), (8, 7168, 18752, 0), (5, 11008, 28672, 1),                      # up to eight tokens
    (16, 32768, 4096, 1), (16, 32768 + 64, 4096, 0), (16, 49152, 2048, 1), (8, 49152, 8192, 1), (8, 131072, 8192, 0),  # more rounds
])
def test_where_reading_fp32_is_faster(tokens, m, k, faster):
    assert _native.lib().onebit_sparse_linear_reads_f32(tokens, m, k, None) == faster


@pytest.mark.gpu
def test_the_layer_converts_where_that_is_faster():
    for m, k, allocations in ((11008, 28672, 2), (4096, 11008, 1)):  # the converted copy and the result, or the result
        layer, x = _layer(m, k), torch.randn(16, k, device="cuda")
        layer(x)
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        y = layer(x)
        assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == allocations
        want = torch.empty_like(y)
        _native.linear_prepared(layer._prepared.buffer, x.half(), want, m, k)
        assert torch.equal(y, want)


@pytest.mark.gpu
def test_captured_where_the_host_decides_outside_a_graph():
    """converted in a graph, read as fp32 outside of one: the same results on every replay"""
    m, k = 4096, 11008
    layer, x = _layer(m, k), torch.randn(16, k, device="cuda")
    want = layer(x)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        layer(x)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = layer(x)
    for _ in range(4):
        x.neg_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, layer(x))
    assert torch.equal(y, want)


@pytest.mark.gpu
def test_a_failed_call_is_not_made_again():
    """A refused call raises where it was refused: no conversion, no second attempt whose success or error would stand for it."""
    layer = _layer(128, 512)
    x = torch.randn(4, 512, device="cuda")
    layer(x)
    _native.set_skinny_rows(96)  # no such row group: the launch is refused on the host
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    with pytest.raises(RuntimeError):
        layer(x)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == 1  # the result, no converted copy of x


class _Elsewhere(torch.Tensor):
    """fp32 values that arrive with the conversion, none in the tensor's own memory"""

    @staticmethod
    def __new__(cls, values):
        self = torch.Tensor._make_wrapper_subclass(cls, values.shape, dtype=torch.float32, device=values.device)
        self.values = values
        return self

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        assert func in (torch.ops.aten.to.dtype, torch.ops.aten._to_copy.default), func
        return args[0].values.to(args[1] if len(args) > 1 else kwargs["dtype"])


@pytest.mark.gpu
@pytest.mark.parametrize("tokens", [1, 16])
def test_values_that_are_not_what_lies_in_memory(tokens):
    layer = _layer(128, 512)
    x = torch.randn(tokens, 512, device="cuda")
    assert torch.equal(layer(torch._neg_view(x)), layer(-x))
    assert torch.equal(layer(_Elsewhere(x)), layer(x))
