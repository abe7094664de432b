"""The main kernel's tile order without divisions: the reciprocal of a strip and the comparisons give the quotients."""
import random

import pytest

from test_address_model import tile_of_block


def by_division(v, tiles_m, tiles_n, group_m):
    strip = v // (tiles_m * 4)
    strip_w = min(tiles_n - strip * 4, 4)
    w = v - strip * 4 * tiles_m
    group = w // (group_m * strip_w)
    group_h = min(tiles_m - group * group_m, group_m)
    u = w - group * group_m * strip_w
    return group * group_m + u % group_h, strip * 4 + u // group_h


def as_in_the_kernel(v, tiles_m, tiles_n, group_m):
    return tile_of_block(v, tiles_m, tiles_n, group_m, xcds=1)  # (one XCD: workgroup v is place v of the list)


@pytest.mark.parametrize("group_m", [8, 16])
def test_every_tile_as_by_division(group_m):
    rng = random.Random(group_m)
    sizes = [(1, 1), (1, 9), (9, 1), (8, 4), (16, 4), (17, 5), (43, 7), (25, 100)]
    sizes += [(rng.randint(1, 120), rng.randint(1, 60)) for _ in range(20)]
    for tiles_m, tiles_n in sizes:
        for v in range(tiles_m * tiles_n):
            assert as_in_the_kernel(v, tiles_m, tiles_n, group_m) == by_division(v, tiles_m, tiles_n, group_m)
    for tiles_m, tiles_n in ((400000, 5000), (3, 700000000), (1 << 20, 2000)):
        last = tiles_m * tiles_n - 1
        for v in [0, last] + [rng.randint(0, last) for _ in range(2000)]:
            assert as_in_the_kernel(v, tiles_m, tiles_n, group_m) == by_division(v, tiles_m, tiles_n, group_m)
