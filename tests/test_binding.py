"""Arguments of the package's calls through the compiled binding."""
import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, synthetic


def test_no_out_dtype_is_a_type_error_of_no_call():
    """torch's default type stands in for None, as in torch.empty; what is refused here is the operand on the CPU."""
    weight = PreparedWeight.__new__(PreparedWeight)
    weight.m, weight.k, weight.buffer = 64, 32, torch.zeros(2 * 1536, dtype=torch.uint8)
    with pytest.raises(ValueError, match="must live on the GPU"):
        weight.matmul(torch.zeros(32, 4).half(), out_dtype=None)


@pytest.mark.gpu
def test_result_type_of_no_out_dtype():
    a, meta = synthetic.make_weight(64, 32, 1, device="cuda")
    weight, b = PreparedWeight(a, meta), synthetic.make_b(32, 4, 2, kind="int", device="cuda")
    d = weight.matmul(b, out_dtype=None)
    assert d.dtype == torch.get_default_dtype() and torch.equal(d, weight.matmul(b, out_dtype=d.dtype))
