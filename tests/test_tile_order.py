"""Which block a workgroup takes (et_amd/csrc/tile_order.h), as the host compiler builds it, against Python's integers."""
import ctypes as C
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "et_amd", "csrc")
SOURCE = r"""
#include "tile_order.h"
extern "C" int rest(int n, int d, int *out) {
    const et::QuotRem v = et::quot_rem(n, d, et::magic_of(d));
    out[0] = v.q;
    out[1] = v.r;
    return et::quotients_fit((int64_t)n + 1, d);
}
extern "C" int fit(int64_t blocks, int64_t div) { return et::quotients_fit(blocks, div); }
extern "C" int walk(int outer, int inner, int group, const int *vid, int n, int *out) {
    et::GroupWalk w;
    if (!et::group_walk(w, outer, inner, group))
        return 0;
    for (int i = 0; i < n; i++)
        et::group_walk_at(w, vid[i], out[2 * i], out[2 * i + 1]);
    return w.group;
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile_order")
    (d / "order.cpp").write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "order.so"), str(d / "order.cpp")])
    lib = C.CDLL(str(d / "order.so"))
    lib.fit.argtypes = [C.c_int64, C.c_int64]
    return lib


def blocks(order, outer, inner, group, vids):
    out = (C.c_int * (2 * len(vids)))()
    return order.walk(outer, inner, group, (C.c_int * len(vids))(*vids), len(vids), out), list(zip(out[::2], out[1::2]))


def test_quotient_and_rest(order):
    """exact for every number of a launch whose quotients fit"""
    r, out = random.Random(5), (C.c_int * 2)()
    divisors = [1, 2, 3, 5, 7, 11, 12, 16, 96, 641, 65535, 65536, 65537, 6700417, 2 ** 30, 2 ** 31 - 1]
    divisors += [r.randrange(1, 2 ** r.randrange(1, 32)) for _ in range(300)]
    for d in divisors:
        top = min(2 ** 31 - 2, (2 ** 32 - 1) // d - 1) // d
        for q in {0, 1, 2, top // 2, top, r.randrange(top + 1)}:
            for n in (q * d - 1, q * d, q * d + 1, q * d + d - 1):
                if 0 <= n < 2 ** 31 - 1 and (n + 1) * d < 2 ** 32:
                    assert order.rest(n, d, out) == 1 and tuple(out) == divmod(n, d), (n, d)


def test_quotients_that_do_not_fit(order):
    out = (C.c_int * 2)()
    assert order.fit(2048 * 501, 8 * 501) == 1 and order.fit(2048 * 501, 16 * 501) == 0
    assert order.fit(2 ** 31 - 1, 2) == 1 and order.fit(2 ** 31, 1) == 0 and order.fit(2 ** 40, 2 ** 40) == 0
    assert order.fit(65536, 65535) == 1 and order.fit(65536, 65536) == 0

    def rest(n, d):
        order.rest(n, d, out)
        return tuple(out)

    # (what the condition is for: at the ends of groups the quotient is one too large)
    assert any(rest(n, 16 * 501) != divmod(n, 16 * 501) for n in range(16 * 501 - 1, 2048 * 501, 16 * 501))


@pytest.mark.parametrize("group", [1, 2, 4, 8, 16])
def test_grouped_walk_takes_every_block_once(order, group):
    for outer, inner in ((16, 1), (17, 3), (31, 12), (48, 7), (66, 9)):
        taken, got = blocks(order, outer, inner, group, range(outer * inner))
        want = [(o, i) for g in range(0, outer, group) for i in range(inner) for o in range(g, min(g + group, outer))]
        assert taken == group and got == want


@pytest.mark.parametrize("outer,inner,group,taken", [
    (2048, 501, 16, 8),      # 65536 rows x 32016 outputs in 32 x 64: groups of sixteen are beyond 32 bits
    (1000, 2003, 16, 1),
    (50000, 143, 8, 4),
    (1024, 2048, 16, 0),     # not even single tiles
])
def test_grouped_walk_of_many_blocks(order, outer, inner, group, taken):
    """a sample of blocks around every group's edges: in range, and the block that the walk has there"""
    div, total = max(taken, 1) * inner, outer * inner
    assert taken * 2 > group or total * 2 * div >= 2 ** 32
    vids = sorted({v for g in range(0, outer // max(taken, 1) + 1, 5) for e in (g * div, g * div + div // 2)
                   for v in range(e - 20, e + 20) if 0 <= v < total} | set(range(total - 50, total)))
    got_taken, got = blocks(order, outer, inner, group, vids)
    assert got_taken == taken
    if taken:
        for v, place in zip(vids, got):
            g, k = divmod(v, div)
            n = min(taken, outer - g * taken)
            assert place == (g * taken + k % n, k // n), v
