"""The forms of a planned linear: their times, the library's estimates of them, and the fit behind the estimates.

A planned linear runs as one of several kernels and shapes of work item, chosen by estimated time (tile_linear.hip,
tile_rows.hip, dense_gemm.hip; et_tile_plan_estimate gives the estimate).  This program keeps what such a choice rests on:

  python3 et_amd/bench/linear_forms.py measure TIMES     times every form over a seeded sample of linears (GPU)
  python3 et_amd/bench/linear_forms.py report TIMES      how far the estimates and the choices are from the times
  python3 et_amd/bench/linear_forms.py fit TIMES         non-negative least squares for each kernel's cost terms

TIMES has a line per launch: inputs, outputs (of joined linears), GELU, sparsity, rows, form, items per workgroup, measured
microseconds, estimated microseconds.  The form "auto" is the library's own choice.  After a change to one of the kernels:
measure, fit, carry the figures over, measure again and look at the choices in the report.
"""
import ctypes as C
import os
import random
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, ROOT)

PANEL = ((512, (512,), 0), (512, (2048,), 1), (768, (768,), 0), (768, (768, 768, 768), 0), (768, (3072,), 1),
         (1024, (1024, 1024, 1024), 0), (1024, (4096,), 1))
CHUNKS = ((2048, (512,), 0), (3072, (768,), 0), (4096, (1024,), 0))
SPARSITIES = (0.0, 0.5, 0.8, 0.9)
FORMS = ((32, 8, 1), (32, 8, 2), (32, 8, 3), (64, 12, 2), (64, 8, 3), (64, 8, 2), (64, 8, 1))  # rows, waves, block-rows
DENSE_LAUNCH = 3.5  # us that the library adds to the dense product's estimate when it is weighed against the tile kernels
LAUNCH = 3.0        # ... of which so many are the launch, which the dense product's estimate leaves out
TILES_BEYOND_MB, TILES_BEYOND = 48.0, 1.1  # the tile kernels' share of their estimate where input and result are larger
TERMS = {  # kernel -> its cost terms, in the order of features()
    "32 rows": "launch traffic traffic_over round item item_nb item_stream panel out gelu mfma result wg".split(),
    "64 rows": "launch traffic traffic_over round item item_nb item_stream panel out gelu mfma result wg".split(),
    "64 rows, 12 waves": "launch traffic traffic_over round item item_nb item_stream panel out gelu mfma result wg".split(),
    "chunk by chunk": "launch round*chunk round*nb*pairs cu*chunk cu*nb*pairs cu*nb traffic".split(),
    "fetching waves": "launch round round*chunk round*nb*chunk round*nb*pairs round*fill*nb*pairs round*group*pairs traffic".split(),
    "48 rows": "launch round round*chunk round*nb*chunk round*nb*pairs round*fill*nb*pairs round*group*pairs traffic".split(),
    "48 rows, two waves a block-row": "launch round round*chunk round*nb*chunk round*nb*pairs round*fill*nb*pairs round*group*pairs traffic".split(),
    "whole rows": "launch traffic round round*K round*group*pairs round*nb round*fill".split(),
}


# ---- the terms' values for one launch -------------------------------------------------------------------------------
def order(x, w, panels, groups, most):
    return x <= most and min(groups, 8) * x + w < x + min(panels, 8) * w


def traffic(x, w, panels, groups, most):
    return min(groups, 8) * x + w if order(x, w, panels, groups, most) else x + min(panels, 8) * w


def up(a, b):
    return -(-a // b)


def rows_shape(M, K, nbr, nlin, pairs, cus):
    best, shape = 1e30, None
    for s in range(5):
        for b in range(1, (4 if s == 0 else 1) + 1):
            br = 16 >> s
            wgs = up(M, 16) * up(nbr, br * b) * nlin
            lat = 1.2 + b * (0.3 + 0.35 * (pairs / (1 << s)) / 8) + (0.3 if s else 0.0)
            t = up(wgs, cus) * (lat + (32.0 * K + 1024.0 * br * b * pairs) / 130e3)
            if t < best * 0.999:
                best, shape = t, (b, s)
    return shape


def features(line, cus=256):
    """(kernel, values of its terms); None for a dense form"""
    K, Ns, gelu, M, form, d = (line[k] for k in ("inputs", "outputs", "gelu", "rows", "form", "d"))
    nlin, nbr = len(Ns), max(Ns) // 16
    tiles = [int((K // 16) * (n // 16) * (1.0 - line["sparsity"])) for n in Ns]
    pairs = sum(0.5 * t / (n // 16) for t, n in zip(tiles, Ns)) / nlin
    w, x = sum(512e-6 * t for t in tiles), 2e-6 * M * K
    if form.startswith("panel"):
        height, waves, nb = FORMS[int(form[5:])]
        lds = height * (K + (0 if K & 31 else 16)) * 2 + waves * height * (16 * nb + 8) * 2
        panels, per_panel = up(M, height), up(nbr, waves * nb) * nlin
        groups = per_panel // d
        nwg = panels * groups
        on_cu = up(nwg, cus)
        rounds = up(on_cu, 2 if height == 32 and 2 * lds <= 160 * 1024 else 1)
        mb = traffic(x, w, panels, groups, 1.75)
        G = min(waves * nb, nbr)
        return ("32 rows" if height == 32 else "64 rows" if waves == 8 else "64 rows, 12 waves",
                [1, mb, max(0.0, mb - 12.0), rounds, rounds * d, rounds * d * nb, rounds * d * nb * pairs, on_cu * height * K,
                 on_cu * d * G * height, on_cu * d * G * height * gelu, on_cu * d * G * height * pairs, M * sum(Ns), nwg])
    nchunk = up(K, 768)
    if form == "chunk":
        panels = up(M, 32)
        nb = next((n for n in (3, 2, 1) if panels * up(nbr, 8 * n) * nlin >= 512), 1)
        ncg = up(nbr, 8 * nb) * nlin
        rounds, on_cu = up(panels * ncg, 2 * cus), up(panels * ncg, cus)
        return "chunk by chunk", [1, rounds * nchunk, rounds * nb * pairs, on_cu * nchunk, on_cu * nb * pairs, on_cu * nb,
                                  traffic(x, w, panels, ncg, 1.75)]
    if form.startswith("fetch"):
        nb, panels = int(form[5:]), up(M, 32)
        ncg = up(nbr, 12 * nb) * nlin
        rounds, fill = up(panels * ncg, cus), min(1.0, panels * ncg / cus)
        return "fetching waves", [1, rounds, rounds * nchunk, rounds * nb * nchunk, rounds * nb * pairs,
                                  rounds * fill * nb * pairs, rounds * min(12 * nb, nbr) * pairs,
                                  traffic(x, w, panels, ncg, 1.75)]
    if form.startswith("tall"):
        group = {5: 12, 6: 6, 7: 24, 8: 36}[int(form[4:])]
        panels, nb = up(M, 48), group / 12
        ncg = up(nbr, group) * nlin
        rounds, fill = up(panels * ncg, cus), min(1.0, panels * ncg / cus)
        return "48 rows, two waves a block-row" if group == 6 else "48 rows", [
            1, rounds, rounds * nchunk, rounds * nb * nchunk, rounds * nb * pairs, rounds * fill * nb * pairs,
            rounds * min(group, nbr) * pairs, traffic(x, w, panels, ncg, 1.75)]
    if form == "rows":
        b, s = rows_shape(M, K, nbr, nlin, pairs, cus)
        group, panels = (16 >> s) * b, up(M, 16)
        ncg = up(nbr, group) * nlin
        rounds, fill = up(panels * ncg, cus), min(1.0, panels * ncg / cus)
        return "whole rows", [1, traffic(x, w, panels, ncg, 2.5), rounds, rounds * K, rounds * group * pairs, rounds * b,
                              rounds * fill]
    return None


# ---- measuring ------------------------------------------------------------------------------------------------------
def measure(path):
    import numpy as np
    import torch
    from et_amd import formats, lib
    from et_amd.encoder import Linear_tile, run_multi
    L, rng = lib(), random.Random(20)
    most = 16384

    def keys(**values):
        for k, v in values.items():
            assert L.et_tuning_set(k.encode(), v) == 0, k

    def automatic():
        keys(tile_form=-1, tile_ipw=0, tile_chunked=-1, tile_splitk_rows=-1, plan_dense=1, dense_form=-1)

    def linear(K, N, gelu, sparsity):
        rp, ro = formats.gen_sparse_tile_mat(N, K, sparsity, rng.randrange(1 << 30))
        data = np.random.default_rng(N + K).standard_normal(ro.size * 256, np.float32).astype(np.float16)
        return Linear_tile(K, N, most, ro.size, data, rp, ro, np.zeros(N, np.float16), bool(gelu))

    side = torch.cuda.Stream()

    def us(run, runs=20):
        """a launch among `runs` of a graph, the fastest of four replays"""
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            run()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            for _ in range(runs):
                run()
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3 / runs)
        return min(times[1:])

    def estimate(K, Ns, lts, M, gelu, dense):
        n = len(Ns)
        t, g = C.c_double(), C.c_double()
        arr = C.c_int * n
        assert L.et_tile_plan_estimate(K, arr(*Ns), arr(*[int((K // 16) * (v // 16) * (1.0 - lts[0].sparsity)) for v in Ns]), n, M,
                                       gelu, C.byref(t), C.byref(g)) == 0
        return g.value if dense else t.value

    spin = torch.empty(1 << 26, device="cuda")
    with open(path, "w") as f:
        for K, Ns, gelu in PANEL + CHUNKS:
            for sparsity in SPARSITIES:
                lts = [linear(K, N, gelu, sparsity) for N in Ns]
                for lt in lts:
                    lt.sparsity = sparsity
                x = torch.randn((most, K), device="cuda").to(torch.float16)
                outs = [torch.empty((most, N), dtype=torch.float16, device="cuda") for N in Ns]
                for i in range(8):
                    M = int(37 * (most / 37) ** ((i + rng.random()) / 8))
                    ys = [o[:M] for o in outs]
                    run = (lambda: run_multi(lts, x[:M], ys)) if len(lts) > 1 else (lambda: lts[0].run(x[:M], out=ys[0]))
                    for _ in range(50):
                        spin.add_(1.0)  # (clocks)

                    def line(form, d, dense=False):
                        t = us(run)
                        f.write(f"{K} {'+'.join(map(str, Ns))} {gelu} {sparsity} {M} {form} {d} {t:.2f} "
                                f"{estimate(K, Ns, lts, M, gelu, dense):.2f}\n")

                    keys(plan_dense=0)
                    line("auto", 0)
                    if K <= 1024:
                        for k, (height, waves, nb) in enumerate(FORMS):
                            if height * (K + 16) * 2 + waves * height * (16 * nb + 8) * 2 > 160 * 1024:
                                continue
                            per = up(max(Ns) // 16, waves * nb) * len(Ns)
                            ds = [d for d in range(1, min(per, 16) + 1) if per % d == 0]
                            for d in sorted(rng.sample(ds, min(2, len(ds)))):
                                keys(tile_form=k, tile_ipw=d)
                                line(f"panel{k}", d)
                        keys(tile_form=-1, tile_ipw=0)
                    else:
                        for nb in range(5):
                            keys(tile_chunked=nb, tile_splitk_rows=0)
                            line(f"fetch{nb}" if nb else "chunk", 0)
                        for form in range(5, 9):
                            keys(tile_chunked=form, tile_splitk_rows=0)
                            line(f"tall{form}", 0)
                        keys(tile_chunked=-1, tile_splitk_rows=most)
                        line("rows", 0)
                        keys(tile_splitk_rows=-1)
                    if sparsity == 0.0:
                        keys(plan_dense=1)
                        line("auto+dense", 0)
                        keys(plan_dense=2)
                        for k in range(11):
                            keys(dense_form=k)
                            line(f"dense{k}", 0, dense=True)
                    automatic()
                print(K, Ns, sparsity, flush=True)
                f.flush()


# ---- reading --------------------------------------------------------------------------------------------------------
def read(path):
    out = []
    for text in open(path):
        p = text.split()
        if len(p) != 9 or not p[0].isdigit():
            continue  # (a heading)
        out.append(dict(inputs=int(p[0]), outputs=tuple(map(int, p[1].split("+"))), gelu=int(p[2]), sparsity=float(p[3]),
                        rows=int(p[4]), form=p[5], d=int(p[6]), us=float(p[7]), est=float(p[8])))
    return out


def shape_of(line):
    return tuple(line[k] for k in ("inputs", "outputs", "gelu", "sparsity", "rows"))


def report(lines):
    kernels = {}
    for l in lines:
        if l["form"].startswith("auto"):
            continue
        dense = l["form"].startswith("dense")
        kernel = "dense product" if dense else features(l)[0]
        kernels.setdefault(kernel, []).append(abs((l["est"] + LAUNCH * dense) / l["us"] - 1))
    chosen = {}  # the block of least estimated time: the one that runs, and that the tile kernels are weighed against
    for l in lines:
        if l["form"].startswith("dense") and l["est"] < chosen.get(shape_of(l), dict(est=1e30))["est"]:
            chosen[shape_of(l)] = l
    if chosen:
        kernels["dense, chosen block"] = [abs((l["est"] + LAUNCH) / l["us"] - 1) for l in chosen.values()]
    for kernel, err in kernels.items():
        err.sort()
        print(f"{kernel:20s} {len(err):5d} launches, estimates off by {100 * sum(err) / len(err):.1f} % in the mean, "
              f"{100 * err[len(err) * 9 // 10]:.0f} % for one in ten")
    for choice in ("auto", "auto+dense"):
        behind, worst = [], []
        for shape in {shape_of(l) for l in lines if l["form"] == choice}:
            mine = [l for l in lines if shape_of(l) == shape]
            got = next(l["us"] for l in mine if l["form"] == choice)
            best = min(l["us"] for l in mine if choice == "auto+dense" or not l["form"].startswith(("dense", "auto+")))
            behind.append(got / best - 1)
            worst.append((got / best - 1, got, best, shape))
        if behind:
            worst.sort(reverse=True)
            print(f"{choice}: {len(behind)} linears, {100 * sum(behind) / len(behind):.1f} % behind the fastest form measured "
                  f"in the mean; furthest: " + "; ".join(f"{s} {g:.1f} against {b:.1f} us" for _, g, b, s in worst[:3]))
    blocks = {}
    for l in lines:
        if l["form"].startswith("dense"):
            blocks.setdefault(shape_of(l), []).append(l)
    if blocks:
        behind = sorted((min(ls, key=lambda l: l["est"])["us"] / min(l["us"] for l in ls) - 1, shape) for shape, ls in blocks.items())
        print(f"dense blocks: {len(behind)} full plans, {100 * sum(b for b, _ in behind) / len(behind):.1f} % behind the fastest "
              f"block in the mean; furthest: " + "; ".join(f"{s} {100 * b:.0f} %" for b, s in behind[:-4:-1]))
    both = {}
    for l in lines:
        if l["form"] == "auto+dense":
            both.setdefault(shape_of(l), {"of": (l["inputs"], l["outputs"], l["rows"])})["est_tiles"] = l["est"]
    for l in lines:
        if shape_of(l) in both:
            b = both[shape_of(l)]
            if l["form"] == "auto":
                b["tiles"] = l["us"]
            elif l["form"].startswith("dense"):
                if l["est"] < b.get("est_dense", 1e30):
                    b["est_dense"], b["dense"] = l["est"], l["us"]
    for extra in (DENSE_LAUNCH - 0.3, DENSE_LAUNCH, DENSE_LAUNCH + 0.3):
        lost = [(b["dense"] if takes_dense(*b["of"], b["est_tiles"], b["est_dense"], extra) else b["tiles"]) / min(b["dense"], b["tiles"]) - 1
                for b in both.values() if "est_dense" in b]
        if lost:
            print(f"full plans, {extra:.1f} us on top of the dense product's estimate: {100 * sum(lost) / len(lost):.1f} % behind the "
                  f"faster of the two, {100 * max(lost):.0f} % at most")


def takes_dense(K, Ns, rows, est_tiles, est_dense, extra=DENSE_LAUNCH):
    """the library's line for full plans (et_tile_plan_prefers_dense)"""
    mb = 2e-6 * rows * (K + sum(Ns))
    return extra + est_dense < est_tiles * (TILES_BEYOND if mb > TILES_BEYOND_MB else 1.0)


def fit(lines):
    import numpy as np
    from scipy.optimize import nnls
    kernels = {}
    for l in lines:
        f = None if l["form"].startswith("auto") else features(l)
        if f:
            kernels.setdefault(f[0], []).append((f[1], l["us"]))
    for kernel, data in kernels.items():
        t = np.array([u for _, u in data])
        A = np.array([v for v, _ in data], dtype=np.float64) / t[:, None]
        scale = np.maximum(A.max(0), 1e-30)
        c = nnls(A / scale, np.ones(len(t)))[0] / scale
        err = np.abs(A @ c - 1)
        print(f"{kernel}: {len(t)} launches, off by {100 * err.mean():.1f} % in the mean")
        print("   " + ", ".join(f"{n} {v:.3g}" for n, v in zip(TERMS[kernel], c)))


if __name__ == "__main__":
    if len(sys.argv) != 3 or sys.argv[1] not in ("measure", "report", "fit"):
        sys.exit(__doc__)
    if sys.argv[1] == "measure":
        measure(sys.argv[2])
    else:
        {"report": report, "fit": fit}[sys.argv[1]](read(sys.argv[2]))
