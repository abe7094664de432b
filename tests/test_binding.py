"""Arguments and threads of the package's calls through the compiled binding."""
import threading
import time

import pytest
import torch

from onebitsparsemul_amd import PreparedWeight, _native, synthetic


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


@pytest.mark.gpu
def test_other_threads_run_while_a_call_waits_for_the_device():
    """A call whose buffer has to grow frees the old one after a device synchronization, and this one has some tenths of a second
    of queued work to wait for. The interpreter lock is not held meanwhile."""
    weights = {m: PreparedWeight(*synthetic.make_weight(m, 28672, m, device="cuda")) for m in (512, 2048)}
    b = synthetic.make_b(28672, 16, 3, device="cuda")
    large = torch.randn(8192, 8192, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    _native.release_buffers()
    with torch.cuda.stream(stream):
        weights[512].matmul(b)  # the buffer that has to grow
        for _ in range(60):
            large @ large
    took, gap = [], 0.0

    def grow():
        begin = time.perf_counter()
        with torch.cuda.stream(stream):
            weights[2048].matmul(b)
        took.append(time.perf_counter() - begin)

    thread = threading.Thread(target=grow)
    last = time.perf_counter()
    thread.start()
    while thread.is_alive():
        time.sleep(0.001)
        now = time.perf_counter()
        gap, last = max(gap, now - last), now
    thread.join()
    torch.cuda.synchronize()
    assert took[0] > 0.1, f"the call waited for {took[0]:.3f} s only"
    assert gap < took[0] / 2, f"nothing ran for {gap:.3f} of {took[0]:.3f} s"
