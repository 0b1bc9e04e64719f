"""The program that keeps the linear forms' times and fits (CPU part): its terms are the library's."""
import ctypes as C
import os
import re
import sys
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "et_amd", "bench"))

import linear_forms as lf  # noqa: E402
from et_amd import lib  # noqa: E402


def library_estimate(line, **keys):
    L, n = lib(), len(line["outputs"])
    K = line["inputs"]
    tiles = [int((K // 16) * (v // 16) * (1.0 - line["sparsity"])) for v in line["outputs"]]
    t, g = C.c_double(), C.c_double()
    try:
        for k, v in keys.items():
            assert L.et_tuning_set(k.encode(), v[0]) == 0
        assert L.et_tile_plan_estimate(K, (C.c_int * n)(*line["outputs"]), (C.c_int * n)(*tiles), n, line["rows"],
                                       line["gelu"], C.byref(t), C.byref(g)) == 0
    finally:
        for k, v in keys.items():
            L.et_tuning_set(k.encode(), v[1])
    return t.value


def panel_costs():
    src = open(os.path.join(ROOT, "et_amd", "csrc", "tile_linear.hip")).read()
    return {name: [float(v) for v in re.search(key + r" = \{([^}]*)\}", src).group(1).split(",")]
            for name, key in (("32 rows", "tl_cost32"), ("64 rows", "tl_cost64"), ("64 rows, 12 waves", "tl_cost64x12"))}


@pytest.mark.parametrize("rows", [37, 700, 9000])
@pytest.mark.parametrize("K,Ns,gelu", lf.PANEL)
def test_panel_terms_add_up_to_the_estimate(K, Ns, gelu, rows):
    costs, cus = panel_costs(), max(lib().et_device_cu_count(), 1)
    for k, (height, waves, nb) in enumerate(lf.FORMS):
        if height * (K + 16) * 2 + waves * height * (16 * nb + 8) * 2 > 160 * 1024:
            continue
        per = lf.up(max(Ns) // 16, waves * nb) * len(Ns)
        for d in {1, per if per <= 16 else 1}:
            line = dict(inputs=K, outputs=Ns, gelu=gelu, sparsity=0.8, rows=rows, form=f"panel{k}", d=d)
            name, terms = lf.features(line, cus)
            want = library_estimate(line, tile_form=(k, -1), tile_ipw=(d, 0))
            assert len(terms) == len(lf.TERMS[name])
            assert sum(c * v for c, v in zip(costs[name], terms)) == pytest.approx(want, rel=1e-9)


@pytest.mark.parametrize("rows", [37, 700, 9000])
@pytest.mark.parametrize("K,Ns,gelu", lf.CHUNKS)
def test_chunk_terms_follow_the_estimate(K, Ns, gelu, rows):
    """the constants stand in the library's formulas: the terms have to span the same differences"""
    cus = max(lib().et_device_cu_count(), 1)
    for form, keys, const in (
            ("chunk", dict(tile_chunked=(0, -1), tile_splitk_rows=(0, -1)),
             (1.367, 0.9615, 0.0867, 0.4349, 0.01745, 0.6037, 0.0673)),
            ("fetch1", dict(tile_chunked=(1, -1), tile_splitk_rows=(0, -1)),
             (1.775, 1.997, 0.378, 0.233, 0.0397, 0.0140, 0.00429, 0.0980)),
            ("fetch4", dict(tile_chunked=(4, -1), tile_splitk_rows=(0, -1)),
             (1.775, 1.997, 0.378, 0.233, 0.0397, 0.0140, 0.00429, 0.0980)),
            ("rows", dict(tile_splitk_rows=(1 << 20, -1)), (1.75, 0.0514, 0.4525, 43.3e-5, 1.093e-2, 1.4, 0.0825))):
        line = dict(inputs=K, outputs=Ns, gelu=gelu, sparsity=0.5, rows=rows, form=form, d=0)
        name, terms = lf.features(line, cus)
        assert len(terms) == len(lf.TERMS[name]) == len(const)
        assert sum(c * v for c, v in zip(const, terms)) == pytest.approx(library_estimate(line, **keys), rel=1e-6), form


@pytest.mark.parametrize("rows", [37, 700, 9000])
@pytest.mark.parametrize("K,Ns,gelu", lf.CHUNKS)
def test_tall_panel_terms_follow_the_estimate(K, Ns, gelu, rows):
    cus = max(lib().et_device_cu_count(), 1)
    split, whole = (1.468, 2.068, 1.277, 0, 0, 0.0512, 0.00231, 0.0332), (1.094, 2.931, 0.4926, 0.2443, 0.0840, 0.0414, 0, 0.0736)
    for form in (5, 6, 7, 8):
        line = dict(inputs=K, outputs=Ns, gelu=gelu, sparsity=0.5, rows=rows, form=f"tall{form}", d=0)
        name, terms = lf.features(line, cus)
        assert len(terms) == len(lf.TERMS[name])
        const = split if form == 6 else whole
        assert 1.15 * sum(c * v for c, v in zip(const, terms)) == pytest.approx(
            library_estimate(line, tile_chunked=(form, -1), tile_splitk_rows=(0, -1)), rel=1e-6), form


def test_dense_choice_is_kept_by_its_sizes():
    """More shapes than the table of kept choices has entries, in two orders and from two threads, neighbours that differ in
    one thing among them: always the least block."""
    L = lib()
    shapes = [(K, Ns, gelu, rows) for K, Ns, gelu in ((768, (768,), 0), (768, (3072,), 1), (1024, (1024,) * 3, 0), *lf.CHUNKS)
              for rows in (16, 37, 61, 104, 250, 345, 700, 1300, 2048, 5000, 9000, 16384)]
    one_thing = [(768, (3072,), 0, 2048), (768, (3072,), 1, 2048),                             # GELU
                 (768, (768,), 0, 2048), (768, (768, 768), 0, 2048), (768, (768,) * 3, 0, 2048),  # linears
                 (768, (768, 3072), 0, 2048), (768, (768, 768), 0, 2048),                      # the second one's width
                 (768, (768, 768, 3072), 0, 2048), (768, (768,) * 3, 0, 2048),                 # the third one's
                 (3072, (768,) * 3, 0, 2048), (3072, (768,) * 3, 0, 1024)]                     # inputs, rows
    shapes += one_thing * 2
    assert len(shapes) > 64

    def dense_us(K, Ns, gelu, rows):
        n, t, g = len(Ns), C.c_double(), C.c_double()
        assert L.et_tile_plan_estimate(K, (C.c_int * n)(*Ns), (C.c_int * n)(*[(K // 16) * (v // 16) for v in Ns]), n, rows,
                                       gelu, C.byref(t), C.byref(g)) == 0
        return g.value

    def block_us(form):
        assert L.et_tuning_set(b"dense_form", form) == 0
        return [dense_us(*s) for s in shapes]

    try:
        want = [min(v) for v in zip(*(block_us(f) for f in range(11)))]
    finally:
        L.et_tuning_set(b"dense_form", -1)
    assert all(a != b for a, b in zip(want[-len(one_thing):], want[-len(one_thing) + 1:]))
    assert [dense_us(*s) for s in shapes] == want
    got = []
    other = threading.Thread(target=lambda: got.extend(dense_us(*s) for s in reversed(shapes)))
    other.start()
    assert [dense_us(*s) for s in reversed(shapes)] == want[::-1]
    other.join()
    assert got == want[::-1]


def test_line_of_full_plans_is_the_librarys():
    """the program's line between tile kernels and dense product, among others where input and result beyond 48 MB decide"""
    L, beyond = lib(), 0
    for K, Ns, gelu in ((256, (1024,), 1), (512, (512,), 0), (768, (768,), 0), (768, (3072,), 1), (768, (768,) * 3, 0), (640, (640,) * 3, 0), (512, (1024,), 0), *lf.CHUNKS):
        for rows in [16, 100, 1000, 3000, *range(4000, 40000, 311)]:
            n, t, g = len(Ns), C.c_double(), C.c_double()
            assert L.et_tile_plan_estimate(K, (C.c_int * n)(*Ns), (C.c_int * n)(*[(K // 16) * (v // 16) for v in Ns]), n, rows,
                                           gelu, C.byref(t), C.byref(g)) == 0
            takes = lf.takes_dense(K, Ns, rows, t.value, g.value)
            beyond += takes != (lf.DENSE_LAUNCH + g.value < t.value)
            assert L.et_tile_plan_prefers_dense(K, (C.c_int * n)(*Ns), n, rows, gelu) == takes, (K, Ns, rows)
    if L.et_device_cu_count() in (0, 256):  # (without a device the estimates count one compute unit)
        assert beyond > 0


def test_prefers_dense_follows_its_key_and_the_plans_that_have_a_dense_form():
    L, one = lib(), lambda *v: (C.c_int * len(v))(*v)
    sizes = (768, one(768), 1, 16, 0)
    try:
        assert L.et_tuning_set(b"plan_dense", 2) == 0
        assert L.et_tile_plan_prefers_dense(*sizes) == 1
        assert L.et_tile_plan_prefers_dense(784, one(768), 1, 16, 0) == 0  # K not a multiple of 32: no row-major W
        assert L.et_tile_plan_prefers_dense(768, one(768, 768, 768, 768), 4, 16, 0) == 0
        assert L.et_tile_plan_prefers_dense(768, one(760), 1, 16, 0) == 0 and L.et_tile_plan_prefers_dense(768, None, 1, 16, 0) == 0
        assert L.et_tile_plan_prefers_dense(768, one(768), 1, 0, 0) == 0
        assert L.et_tuning_set(b"plan_dense", 0) == 0
        assert L.et_tile_plan_prefers_dense(*sizes) == 0
    finally:
        L.et_tuning_set(b"plan_dense", 1)


def test_times_are_read_back(tmp_path):
    p = tmp_path / "times.txt"
    p.write_text("A heading.\n\n768 768+768 1 0.8 100 panel3 2 7.25 6.90\n768 768+768 1 0.8 100 auto 0 7.10 6.90\n")
    a, b = lf.read(p)
    assert a["outputs"] == (768, 768) and a["form"] == "panel3" and a["d"] == 2 and a["us"] == 7.25 and a["est"] == 6.9
    assert lf.shape_of(a) == lf.shape_of(b)
