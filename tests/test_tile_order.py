"""Which block a workgroup takes (et_amd/csrc/tile_order.h), as the host compiler builds it, against Python's integers."""
import ctypes as C
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "et_amd", "csrc")
SOURCE = r"""
#include "tile_order.h"
extern "C" void rest(int n, int d, int *out) {
    const et::QuotRem v = et::quot_rem(n, d, et::magic_of(d));
    out[0] = v.q;
    out[1] = v.r;
}
extern "C" void rest_small(int n, int d, int *out) {
    const et::QuotRem v = et::quot_rem_small(n, d, et::magic_of(d));
    out[0] = v.q;
    out[1] = v.r;
}
extern "C" void walk(int outer, int inner, int group, const int *vid, int n, int *out) {
    const et::GroupWalk w = et::group_walk(outer, inner, group);
    for (int i = 0; i < n; i++)
        et::group_walk_at(w, vid[i], out[2 * i], out[2 * i + 1]);
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_order")
    (d / "order.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "order.so"), str(d / "order.cpp")])
    return C.CDLL(str(d / "order.so"))


def blocks(order, outer, inner, group, vids):
    out = (C.c_int * (2 * len(vids)))()
    order.walk(outer, inner, group, (C.c_int * len(vids))(*vids), len(vids), out)
    return list(zip(out[::2], out[1::2]))


def test_quotient_and_rest(order):
    r, out = random.Random(5), (C.c_int * 2)()
    divisors = [1, 2, 3, 5, 7, 11, 12, 16, 96, 641, 65535, 65536, 65537, 6700417, 2 ** 30, 2 ** 31 - 1]
    divisors += [r.randrange(1, 2 ** r.randrange(1, 32)) for _ in range(300)]
    for d in divisors:
        top = (2 ** 31 - 1) // d
        for q in {0, 1, 2, top // 2, top, r.randrange(top + 1)}:
            for n in (q * d - 1, q * d, q * d + 1, q * d + d - 1):
                if 0 <= n < 2 ** 31:
                    order.rest(n, d, out)
                    assert tuple(out) == divmod(n, d), (n, d)


@pytest.mark.parametrize("group", [1, 2, 4, 8, 16])
def test_grouped_walk_takes_every_block_once(order, group):
    for outer, inner in ((16, 1), (17, 3), (31, 12), (48, 7), (66, 9)):
        got = blocks(order, outer, inner, group, range(outer * inner))
        want = [(o, i) for g in range(0, outer, group) for i in range(inner) for o in range(g, min(g + group, outer))]
        assert got == want


@pytest.mark.parametrize("outer,inner,group", [
    (2048, 501, 16),      # 65536 rows x 32016 outputs in 32 x 64: blocks times blocks of a group beyond 32 bits
    (1000, 4099, 16),
    (50000, 167, 8),
])
def test_grouped_walk_of_many_blocks(order, outer, inner, group):
    """a sample of blocks around every group's edges: in range, and the block that the walk has there"""
    div, total = group * inner, outer * inner
    assert total * div >= 2 ** 31
    vids = sorted({v for g in range(0, outer // group + 1, 5) for e in (g * div, g * div + div // 2)
                   for v in range(e - 20, e + 20) if 0 <= v < total} | set(range(total - 50, total)))
    for v, got in zip(vids, blocks(order, outer, inner, group, vids)):
        g, k = divmod(v, div)
        n = min(group, outer - g * group)
        assert got == (g * group + k % n, k // n), v


def test_quotient_of_few_linears(order):
    """the form without the correction, for up to four linears' column groups: the product stays below 2^32"""
    out = (C.c_int * 2)()
    for d in (1, 2, 3, 7, 33, 390, 4095, 4096, 16383):
        for n in {0, 1, d - 1, d, d + 1, 2 * d - 1, 2 * d, 3 * d - 1, 3 * d, 4 * d - 1}:
            assert 4 * d * d < 2 ** 32
            order.rest_small(n, d, out)
            assert tuple(out) == divmod(n, d), (n, d)
