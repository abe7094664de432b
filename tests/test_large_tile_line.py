"""Where the 512 x 128 tile runs on four wavefronts (code 15) and where on eight (code 9), both forms (CPU: the host-only
description of a call)."""
import ctypes

import pytest

from onebitsparsemul_amd import _native


def _tile(token_major, m, n, k):
    plan = (ctypes.c_int * 5)()
    assert _native.lib().onebit_sparse_describe_call(token_major, m, n, k, 1, 256, plan) == 0
    assert plan[0] == 0 and plan[2] == 1  # the main kernel, K not split
    return plan[1]


@pytest.mark.parametrize("token_major", [0, 1])
@pytest.mark.parametrize("m,n,k,tile", [
    (8192, 1536, 10752 + 32, 15),  # 192 tiles, three quarters of a round, 43 chunks of K, the last of them an eighth
    (8192, 1536, 10752, 9),        # 42 chunks
    (11008, 1024, 11008, 9),       # 176 tiles
    (8192, 1792, 4096, 15),        # 224 tiles: 0.875 of a round, any K
])
def test_four_or_eight_wavefronts(token_major, m, n, k, tile):
    assert _tile(token_major, m, n, k) == tile
