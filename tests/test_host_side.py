"""The host side of the C ABI (csrc/onebit_capi.hip) without a GPU: the library's object is linked against tests/host/device_stub.cpp,
which stands in for the HIP runtime and the kernels, and called from Python threads. ctypes releases the interpreter lock, so the
threads really meet inside the library."""
import ctypes
import os
import random
import subprocess
import threading

import pytest

from onebitsparsemul_amd import build as native_build

HERE = os.path.dirname(os.path.abspath(__file__))
vp, i32, f32 = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
KERNELS = ("gemm_kernel", "skinny_kernel", "wide_kernel")


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("host")
    obj, out = str(folder / "device_stub.o"), str(folder / "libhost.so")
    subprocess.run([os.path.join(os.path.dirname(native_build.HIPCC), "..", "llvm", "bin", "clang++"), "-O1", "-std=c++17", "-fPIC",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", native_build.CSRC, "-I", native_build.INCLUDE, "-c",
                    os.path.join(HERE, "host", "device_stub.cpp"), "-o", obj], check=True)
    # -Bsymbolic: the stand-ins, not the HIP runtime that torch has loaded
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", out, obj, "-Wl,-u,onebit_sparse_prepare", native_build.STATIC_LIB,
                    "-lpthread"], check=True)
    lib = ctypes.CDLL(out)
    lib.onebit_sparse_last_error.restype = ctypes.c_char_p
    lib.stub_violation.restype = ctypes.c_char_p
    lib.stub_allocated_bytes.restype = ctypes.c_size_t
    lib.onebit_sparse_matmul_prepared.argtypes = [vp, vp, vp, vp, i32, i32, i32, f32, f32, i32, i32, vp]
    lib.onebit_sparse_matmul_prepared_static.argtypes = lib.onebit_sparse_matmul_prepared.argtypes
    lib.onebit_sparse_linear_prepared.argtypes = [vp, vp, vp, vp, i32, i32, i32, i32, i32, vp]
    lib.onebit_sparse_describe_call.argtypes = [i32] * 6 + [ctypes.POINTER(i32)]
    lib.onebit_sparse_matmul_ex.argtypes = [vp, vp, vp, vp, vp, i32, i32, i32, f32, f32, i32, i32, i32, vp]
    return lib


@pytest.fixture
def fresh(host):
    host.onebit_sparse_release_buffers()
    host.stub_set(0, 0)
    host.stub_reset()
    yield host
    host.stub_set(0, 0)
    host.onebit_sparse_set_weight_cache(0)


def product(lib, m, n, k, b=0x2000):  # addresses that nobody reads
    return lib.onebit_sparse_matmul_prepared(0x1000, b, None, 0x3000, m, n, k, 1.0, 0.0, 0, 1, None)


def layer(lib, m, tokens, k):
    return lib.onebit_sparse_linear_prepared(0x1000, 0x2000, None, 0x3000, tokens, m, k, 1, 1, None)


def one_call(lib, m, n, k, a=0x4000):
    return lib.onebit_sparse_matmul_ex(a, 0x2000, None, 0x3000, 0x5000, m, n, k, 1.0, 0.0, 0, 0, 0, None)


def last_launch(lib):
    out = (i32 * 5)()
    lib.stub_last_launch(out)
    return dict(kernel=KERNELS[out[0]], rows_or_tile=out[1], splits=out[2], padded=bool(out[3]), columns=out[4])


def in_threads(*bodies):
    failed = []

    def run(body):
        try:
            body()
        except BaseException as err:  # noqa: BLE001  (re-raised below)
            failed.append(err)

    threads = [threading.Thread(target=run, args=(body,)) for body in bodies]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if failed:
        raise failed[0]


# (call, m, columns or tokens, k) that split K over workgroups: through skinny_kernel, wide_kernel and the main kernel
SPLIT_CALLS = [(product, 2048, 16, 28672), (product, 2048, 40, 28672), (product, 4096, 256, 11008), (layer, 4096, 16, 16384),
               (layer, 2048, 48, 28672), (layer, 2048, 128, 28672), (layer, 512, 96, 28672), (layer, 8192, 520, 28672)]


@pytest.mark.parametrize("call,m,n,k", SPLIT_CALLS)
def test_threads_on_one_stream_do_not_meet_in_a_buffer(fresh, call, m, n, k):
    """Two threads submit split products of growing size to one stream. Each call's two kernels (partial sums, then their sum) are
    enqueued before another call's, and no call's buffer is replaced between its look-up and its launch."""
    assert call(fresh, m, n, k) == 0 and last_launch(fresh)["splits"] > 1
    fresh.onebit_sparse_release_buffers()
    fresh.stub_set(2000, 0)

    def body(offset):
        for i in range(6):
            rows = m // 2 // 64 * 64 + 64 * (2 * i + offset)  # every call needs a larger buffer than the one before
            assert call(fresh, rows, n, k) == 0, fresh.onebit_sparse_last_error()

    in_threads(lambda: body(0), lambda: body(1))
    assert fresh.stub_violations() == 0, fresh.stub_violation().decode()


def test_cached_weight_is_not_evicted_between_look_up_and_launch(fresh):
    """A cache of one entry and two threads with a weight each: every call evicts the other thread's copy."""
    assert fresh.onebit_sparse_set_weight_cache(1) == 0
    fresh.stub_set(2000, 0)

    def body(a):
        for _ in range(6):
            assert one_call(fresh, 512, 16, 512, a=a) == 0, fresh.onebit_sparse_last_error()

    in_threads(lambda: body(0x4000), lambda: body(0x6000))
    assert fresh.stub_violations() == 0, fresh.stub_violation().decode()


@pytest.mark.parametrize("call,m,k", [(layer, 2048, 28672), (layer, 512, 28672), (layer, 1024, 20480), (product, 2048, 28672),
                                      (product, 512, 16384)])
def test_fewer_columns_never_replace_the_partial_sum_buffer(fresh, call, m, k):
    """From 64 columns or tokens down, the range where the split does not depend on them but through wide_kernel's own plan: a
    graph captured with more columns keeps its buffer, and a call with fewer can be captured after it without a warm-up."""
    assert call(fresh, m, 64, k) == 0 and last_launch(fresh)["splits"] > 1
    fresh.stub_set(0, 1)
    for n in range(63, 16, -1):
        assert call(fresh, m, n, k) == 0, (n, fresh.onebit_sparse_last_error())


def test_small_unaligned_b_never_replaces_the_padded_copy_of_another(fresh):
    """The copy of 992 x 66 values is the larger in bytes than that of 576 x 119: made into the same buffer, and captured after it
    without a warm-up."""
    assert product(fresh, 256, 119, 576, b=0x2002) == 0 and last_launch(fresh)["padded"]
    before = fresh.stub_allocated_bytes()
    fresh.stub_set(0, 1)
    assert product(fresh, 256, 66, 992, b=0x2002) == 0 and last_launch(fresh)["padded"]
    assert fresh.stub_allocated_bytes() == before


@pytest.mark.parametrize("call,m,n,k", [(layer, 896, 704, 24256), (layer, 1088, 1758, 13888), (layer, 704, 1920, 14816),
                                        (layer, 640, 676, 17536), (layer, 1088, 1694, 5696), (layer, 1344, 969, 9216),
                                        (layer, 2496, 197, 19648), (product, 20864, 152, 7616), (product, 768, 616, 8192),
                                        (layer, 49152, 33, 1024), (layer, 131072, 64, 1024), (layer, 131072, 56, 2048),
                                        (layer, 45056, 64, 4096), (layer, 45056, 48, 3616), (layer, 45056, 48, 4128)])
def test_calls_that_the_main_kernel_multiplies_faster(fresh, call, m, n, k):
    """Few rows that read a large x, shapes where the two kernels' models are near each other, very many rows of short K: 3 to
    90 % slower through wide_kernel."""
    assert call(fresh, m, n, k) == 0
    assert last_launch(fresh)["kernel"] == "gemm_kernel"


@pytest.mark.parametrize("call,m,n,k", [(layer, 4096, 500, 11008), (layer, 5312, 278, 18944), (layer, 1024, 256, 4096),
                                        (layer, 4096, 128, 4096), (product, 4096, 256, 4096), (layer, 131072, 48, 4096),
                                        (layer, 65536, 64, 8192), (layer, 40960, 64, 512), (layer, 41024, 64, 7936),
                                        (layer, 41024, 56, 8160), (layer, 3648, 181, 992), (layer, 2176, 184, 512),
                                        (layer, 2304, 536, 5024)])
def test_calls_that_wide_kernel_multiplies_faster(fresh, call, m, n, k):
    assert call(fresh, m, n, k) == 0
    assert last_launch(fresh)["kernel"] == "wide_kernel"


@pytest.mark.parametrize("m,n,k", [(1024, 128, 2048), (4096, 96, 4096), (2048, 160, 4096), (5120, 128, 8192), (4096, 24, 8192)])
def test_product_is_not_split_because_the_plan_it_replaces_is(fresh, m, n, k):
    """Slower by up to a half when split in two only because the main kernel's or skinny_kernel's plan would split."""
    fresh.stub_set(0, 1)
    assert product(fresh, m, n, k) == 0, fresh.onebit_sparse_last_error()
    assert last_launch(fresh)["kernel"] == "wide_kernel" and last_launch(fresh)["splits"] == 1


@pytest.mark.parametrize("m,k,kernel", [(20480, 4096, "skinny_kernel"), (28672, 5536, "skinny_kernel"), (2048, 1056, "skinny_kernel"),
                                        (11008, 28672, "skinny_kernel"), (4096, 11008, "skinny_kernel"), (5120, 8192, "skinny_kernel"),
                                        (2048, 11008, "wide_kernel"),
                                        (4096, 4096, "wide_kernel"), (40960, 4096, "wide_kernel"), (11008, 1056, "wide_kernel"),
                                        (8192, 992, "skinny_kernel"), (8256, 992, "wide_kernel"), (9920, 992, "wide_kernel")])
def test_kernel_of_32_columns(fresh, m, k, kernel):
    assert product(fresh, m, 32, k) == 0
    assert last_launch(fresh)["kernel"] == kernel


@pytest.mark.parametrize("call,m,n,rows", [(product, 18688, 3, 128), (product, 16448, 12, 128), (product, 16384, 3, 64),
                                           (product, 18688, 4, 128), (product, 18688, 1, 128), (layer, 18688, 3, 128)])
def test_pieces_at_any_alignment_in_one_round(fresh, call, m, n, rows):
    """64-row groups of that mode beyond one per compute unit took up to 22 % longer than the element copies before them. The other
    modes' are no slower in one round either (18688 x 1280, 64- | 128-row groups: four columns 5.3 | 5.3 us, one 6.6 | 5.4, a layer of
    three tokens 6.5 | 5.3)."""
    assert call(fresh, m, n, 1280) == 0
    assert last_launch(fresh)["rows_or_tile"] == rows


@pytest.mark.parametrize("call,m,n,k,split", [(layer, 11008, 32, 28672, True), (layer, 14336, 24, 24576, True),
                                              (product, 14336, 24, 28672, True), (layer, 11008, 17, 20480, False),
                                              (layer, 11008, 24, 11008, False), (layer, 5120, 17, 13824, True),
                                              (product, 2048, 32, 9600, True), (product, 2048, 32, 8192, True),
                                              (product, 4096, 64, 9600, True), (product, 2048, 24, 9600, True),
                                              (product, 8192, 64, 8192, False), (layer, 4096, 24, 11008, False)])
def test_long_k_stays_split(fresh, call, m, n, k, split):
    """Unsplit on wide_kernel slower, by up to 15 %, than the split plan of skinny_kernel that it replaces, or not."""
    assert call(fresh, m, n, k) == 0
    launch = last_launch(fresh)
    assert (launch["kernel"], launch["splits"] > 1) == ("wide_kernel", split)


def test_description_is_what_is_launched(fresh):
    """onebit_sparse_describe_call against the launch of the call itself: both forms, ragged and unaligned B, the hooks."""
    rng = random.Random(1)
    hooks = (fresh.onebit_sparse_set_tile_config, fresh.onebit_sparse_set_skinny_rows, fresh.onebit_sparse_set_split_k)
    plan, seen = (i32 * 5)(), set()
    try:
        for _ in range(3000):
            m, k = 64 * int(2 ** rng.uniform(0, 10)), 32 * int(2 ** rng.uniform(0, 9.8))
            n, tokens, aligned = int(2 ** rng.uniform(0, 11)), rng.random() < 0.5, rng.random() < 0.8
            if rng.random() < 0.5:
                n = (n + 7) // 8 * 8
            settings = (rng.choice((-1, -1, -1, 4, 9)), rng.choice((-1, -1, 32, 64, 128)), rng.choice((-1, -1, -1, 1, 2, 7)))
            for hook, value in zip(hooks, settings):
                hook(value)
            assert fresh.onebit_sparse_describe_call(tokens, m, n, k, aligned, 256, plan) == 0
            if tokens:
                rc = layer(fresh, m, n, k)
            elif k * n < 65536:  # described as the non-allocating entry point reads it
                rc = fresh.onebit_sparse_matmul_prepared_static(0x1000, 0x2000 if aligned else 0x2002, None, 0x3000, m, n, k, 1.0, 0.0,
                                                                0, 1, None)
            else:
                rc = product(fresh, m, n, k, b=0x2000 if aligned else 0x2002)
            if rc != 0 and not tokens and k * n < 65536:
                assert b"static workspace" in fresh.onebit_sparse_last_error()
                continue
            assert rc == 0, fresh.onebit_sparse_last_error()
            got = last_launch(fresh)
            described = dict(kernel=KERNELS[plan[0]], rows_or_tile=plan[1], splits=plan[2], padded=bool(plan[3]),
                             columns=plan[4])
            assert got == described, (m, n, k, tokens, aligned, settings)
            seen.add((got["kernel"], got["splits"] > 1, got["padded"], tokens))
    finally:
        for hook in hooks:
            hook(-1)
    assert len(seen) >= 11, seen
    assert fresh.stub_violations() == 0, fresh.stub_violation().decode()


@pytest.mark.parametrize("call,m,n,k,strips", [
    (layer, 1024, 488, 4096, 0), (layer, 1024, 489, 4096, 1),    # sixteen row groups: from 4 MB of x on
    (layer, 1984, 123, 2784, 1), (layer, 1984, 66, 1792, 0),     # 31 row groups: from 1.5 MB of x and weight on
    (product, 1984, 184, 5536, 1), (product, 704, 48, 2976, 0), (product, 2688, 296, 2848, 0),
    (product, 4096, 256, 4096, 0), (product, 2048, 256, 8192, 1), (product, 1024, 64, 4096, 0),
    (layer, 4096, 64, 11008, 0), (layer, 28672, 48, 8192, 0),    # up to 64 tokens, one column group
])
def test_where_the_grid_is_walked_in_strips(fresh, call, m, n, k, strips):
    assert call(fresh, m, n, k) == 0
    assert last_launch(fresh)["kernel"] == "wide_kernel" and fresh.stub_last_strips() == strips


@pytest.mark.parametrize("tokens,m,k,outside,captured", [(16, 4096, 9568, 1, 1), (16, 4096, 9600, 1, 0), (13, 4096, 11008, 1, 0),
                                                         (16, 4096, 12192, 0, 0), (9, 8192, 15584, 1, 0), (9, 8192, 15616, 0, 0)])
def test_fp32_activations_in_and_outside_a_graph(fresh, tokens, m, k, outside, captured):
    """where the kernel's time does not cover the host's for a conversion in front of it, a captured call converts and another does not"""
    assert fresh.onebit_sparse_linear_reads_f32(tokens, m, k, None) == outside
    fresh.stub_set(0, 1)
    assert fresh.onebit_sparse_linear_reads_f32(tokens, m, k, None) == captured


def test_a_refused_question_does_not_fail_the_call_after_it(fresh):
    """On the default stream the HIP runtime refuses to say whether it is captured while another stream is: no error of the layer's."""
    fresh.stub_set(0, -1)
    assert fresh.onebit_sparse_linear_reads_f32(13, 4096, 11008, None) == 0
    assert layer(fresh, 4096, 13, 11008) == 0
