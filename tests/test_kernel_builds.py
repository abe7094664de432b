"""Which build of a kernel a call launches, without a GPU: the library is linked against tests/host/launch_stub.cpp, which stands in for
the HIP runtime and records the kernels' names."""
import ctypes
import os
import random
import re
import subprocess

import pytest

from onebitsparsemul_amd import _native
from onebitsparsemul_amd import build as native_build
from test_address_model import RAGGED_TILES, TILES, skinny_variant, wide_has_parts

HERE = os.path.dirname(os.path.abspath(__file__))
vp, i32, f32 = ctypes.c_void_p, ctypes.c_int, ctypes.c_float


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    folder = tmp_path_factory.mktemp("host")
    obj, out = str(folder / "launch_stub.o"), str(folder / "libhost.so")
    subprocess.run([os.path.join(os.path.dirname(native_build.HIPCC), "..", "llvm", "bin", "clang++"), "-O1", "-std=c++17", "-fPIC",
                    "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-c", os.path.join(HERE, "host", "launch_stub.cpp"), "-o", obj],
                   check=True)
    # -Bsymbolic: the stand-ins, not the HIP runtime that torch has loaded
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", out, obj, "-Wl,-u,onebit_sparse_prepare", native_build.STATIC_LIB,
                    "-lpthread"], check=True)
    lib = ctypes.CDLL(out)
    lib.stub_launched.restype = ctypes.c_char_p
    lib.onebit_sparse_last_error.restype = ctypes.c_char_p
    lib.onebit_sparse_linear_prepared_f32.argtypes = [vp, vp, vp, vp, i32, i32, i32, i32, i32, vp]
    lib.onebit_sparse_linear_prepared_typed.argtypes = [vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, vp]
    lib.onebit_sparse_matmul_prepared.argtypes = [vp, vp, vp, vp, i32, i32, i32, f32, f32, i32, i32, vp]
    lib.onebit_sparse_linear_prepared_grouped.argtypes = [ctypes.POINTER(_native.LinearProblem), i32, i32, i32, i32, vp]
    return lib


def launched(lib, call, *args):
    """[(kernel, template arguments)] of a call's launches"""
    lib.stub_reset()
    assert call(*args) == 0, lib.onebit_sparse_last_error()
    # (a name with _Float16 among its parameters stays mangled)
    found = [re.search(r"(\w+)<([^>]*)>\(", name) or re.match(r"_ZN6onebit\d+([a-z_]+)(E)", name)
             for name in lib.stub_launched().decode().splitlines()]
    return [(m[1], m[2].split(", ")) for m in found]


@pytest.mark.parametrize("rows", [32, 64, 128])
def test_fp32_activations_take_no_more_than_one_surplus_load(host, rows):
    """One load instruction per token and image: a surplus one costs its place in the load path (8192 x 8192 with nine tokens 7.3 us, 8.8
    with sixteen loads)."""
    host.onebit_sparse_set_skinny_rows(rows)
    try:
        for tokens in range(1, 17):
            (kernel, arguments), = launched(host, host.onebit_sparse_linear_prepared_f32, 0x1000, 0x2000, None, 0x3000, tokens, 8192, 8192, 1,
                                            0, None)
            loads = int(arguments[2]) - 48  # kSkinnyBTokens32
            assert kernel == "skinny_kernel" and tokens <= loads <= tokens + 1, (tokens, loads)
    finally:
        host.onebit_sparse_set_skinny_rows(-1)


@pytest.mark.parametrize("count", [1, 2, 4, 5, 16])
@pytest.mark.parametrize("k,parts", [(4096, False), (5120, True), (4096 + 1792, False),  # 16, 20 and 23 chunks of 256
                                     (11776, False), (11008, True), (12800, True), (13056, False)])  # 46, 43, 50 and 51
def test_groups_take_the_build_with_parts_where_a_remainder_is_dealt_in_parts(host, count, k, parts):
    """The build with parts is 1 to 4 % slower where there are none."""
    problems = (_native.LinearProblem * count)(*[_native.LinearProblem(0x1000, 0x2000, None, 0x3000, 512, k)] * count)
    for tokens in (17, 64):
        (kernel, arguments), = launched(host, host.onebit_sparse_linear_prepared_grouped, problems, count, tokens, 1, 1, None)
        if kernel == "wide_kernel":  # R, COPIES, TOKENS, BF16, PARTS, RAGGED
            assert arguments[4] == str(parts).lower()
        else:                        # R, COPIES, BF16, PARTS, MOST
            assert kernel == "wide_tokens_group_kernel" and arguments[3] == str(parts).lower()
            assert int(arguments[4]) == (4 if count <= 4 else 16)


@pytest.mark.parametrize("tile", [-1, *range(16)])
@pytest.mark.parametrize("n,k", [(1002, 4096), (1001, 4096), (102, 512), (12, 4096), (9, 512)])
def test_no_ragged_product_takes_the_element_copies(host, tile, n, k):
    """A tile, forced by the hook too, that has no build for rows that lie anywhere reads the padded copy: more than ten times faster."""
    host.onebit_sparse_set_tile_config(tile)
    host.onebit_sparse_set_skinny_enabled(0)
    try:
        kernels = launched(host, host.onebit_sparse_matmul_prepared, 0x1000, 0x2000, None, 0x3000, 4096, n, k, 1.0, 0.0, 0, 1, None)
    finally:
        host.onebit_sparse_set_tile_config(-1)
        host.onebit_sparse_set_skinny_enabled(1)
    gemm = [arguments for kernel, arguments in kernels if kernel == "gemm_kernel"]  # WM, WN, FM, FN, DMA, TOKENS, KG, M16, BF16, RAGGED
    padded = kernels[0][0] == "pad_b_kernel"
    assert len(gemm) == 1 and gemm[0][4] == "true" and (gemm[0][9] == "false") == padded


def as_modelled(m, n, k, tokens, b_aligned):
    """(kernel, template arguments) of the product that the address model checks for a call"""
    plan = _native.describe_launch(m, n, k, b_aligned=b_aligned, tokens=tokens)
    chunks = (k + 255) // 256
    chunks = (chunks + plan["splits"] - 1) // plan["splits"]
    flag = {True: "true", False: "false"}
    if plan["kernel"] == "skinny_kernel":
        nw, r, nc, mode, loads = skinny_variant(n, plan["rows"], chunks, b_aligned, tokens)
        number = {"full": 0, "any": 1, "columns": 16 + n, "tokens": 32 + loads}[mode]
        return plan, "skinny", [str(nw), str(r), str(number), str(nc), "false"]
    padded = plan["pad_b"] and not tokens
    if plan["kernel"] == "wide_kernel":
        copies = (plan["columns"] + 7) // 8 if tokens else 2 * ((plan["columns"] + 15) // 16)
        ragged = not tokens and not padded and n % 8 != 0
        return plan, "wide_kernel", [str(plan["rows"] // 32), str(copies), flag[tokens], "false", flag[wide_has_parts(chunks)], flag[ragged]]
    WM, WN, FM, FN, KG = TILES[plan["tile"]]
    ragged = not tokens and not padded and n % 8 != 0
    assert not ragged or plan["tile"] in RAGGED_TILES
    return plan, "gemm_kernel", [str(WM), str(WN), str(FM), str(FN), "true", flag[tokens], str(KG), flag[plan["tile"] == 15], "false", flag[ragged]]


@pytest.mark.parametrize("tokens", [False, True])
@pytest.mark.parametrize("few", [False, True])
def test_the_address_model_describes_the_builds_that_are_launched(host, tokens, few):
    rng = random.Random(few + 2 * tokens)
    seen = set()
    for _ in range(1500):
        m, k = 64 * round(2 ** rng.uniform(0, 9)), 32 * round(2 ** rng.uniform(0, 9.8))
        n = rng.randint(1, 16) if few else round(2 ** rng.uniform(4.05, 11))
        b_aligned = tokens or rng.random() < 0.9
        plan, kernel, arguments = as_modelled(m, n, k, tokens, b_aligned)
        if not b_aligned and kernel == "gemm_kernel" and not plan["pad_b"]:
            continue  # a small copy, made where its buffer can be had: not in the plan
        b = 0x2000 if b_aligned else 0x2002
        if tokens:
            kernels = launched(host, host.onebit_sparse_linear_prepared_typed, 0x1000, b, None, 0x3000, n, m, k, 1, 1, 1, None)
        else:
            kernels = launched(host, host.onebit_sparse_matmul_prepared, 0x1000, b, None, 0x3000, m, n, k, 1.0, 0.0, 0, 1, None)
        products = [(name, found) for name, found in kernels if name not in ("pad_b_kernel", "splitk_reduce_kernel")]
        if kernel == "skinny":
            kernel = "skinny_struct_kernel" if products[0][0] == "skinny_struct_kernel" else "skinny_kernel"
        assert products == [(kernel, arguments)], (m, n, k, b_aligned, plan)
        assert [name for name, _ in kernels].count("splitk_reduce_kernel") == (plan["splits"] > 1)
        assert [name for name, _ in kernels].count("pad_b_kernel") == (plan.get("pad_b", False) and not tokens)
        seen.add((kernel, *arguments))
    assert len(seen) >= (10 if few else 30)
