"""The work that performance is judged on: encoder layers, layer stacks and single operators as a program that
uses this library runs them, through the public Python entry points.

A case is a dict of plain values; `kind` says which entry point it goes through:

  layer      Encoder_tile.run: one layer of tile-pruned linears over a padded batch
  prune      Encoder_prune.run: the same with a row-pruned value projection and pruned attention
  attnaware  Encoder_attnaware.run: query / key / output / feed-forward linears row-pruned
  stack      Encoder_stack.run: several Encoder_length layers over a batch of sequences of different lengths
  linear     Linear_tile.run: one planned tile-pruned linear
  launcher   kernels.tile_spmm_add_bias: one tile-pruned linear on the caller's own tile_mat arrays
  layernorm  kernels.skip_layernorm, in place

Weights are N(0, 0.02) in fp16 on a seeded random tile pattern, activations N(0, 1), LayerNorm scales around one."""
import math
import random

import numpy as np
import torch

from et_amd import formats, kernels
from et_amd.encoder import (Encoder_attnaware, Encoder_length, Encoder_prune, Encoder_stack, Encoder_tile, Linear_row,
                            Linear_tile)

WIDTHS = {512: (8, 2048), 768: (12, 3072), 1024: (16, 4096)}  # model width -> heads, feed-forward width
MASKS = ("none", "zeros", "padding", "dense")
SPARSITIES = (0.0, 0.5, 0.8, 0.8, 0.9)
LINEARS = ((768, 768), (768, 3072), (3072, 768), (1024, 1024), (1024, 4096), (4096, 1024))  # inputs, outputs
MOST_ROWS = 16384


def listed():
    return [
        # one sentence through an unpruned layer: the latency of an interactive request, all launches and round trips
        dict(name="layer dense 1x128", kind="layer", d=768, seq=128, batch=1, sparsity=0.0, mask="zeros", natural=False),
        # a short sentence of odd length through a pruned layer: the smallest layer call
        dict(name="layer 80% 1x37", kind="layer", d=768, seq=37, batch=1, sparsity=0.8, mask="none", natural=False),
        # the benchmark's layer: a full server batch
        dict(name="layer 80% 16x512", kind="layer", d=768, seq=512, batch=16, sparsity=0.8, mask="zeros", natural=False),
        # a small batch with a padding mask, moderately pruned, textbook softmax
        dict(name="layer 50% 4x384 padded", kind="layer", d=768, seq=384, batch=4, sparsity=0.5, mask="padding", natural=True),
        # the wider model of the tests, ragged sequence length
        dict(name="layer 80% 8x250 d1024", kind="layer", d=1024, seq=250, batch=8, sparsity=0.8, mask="none", natural=True),
        # the reference's pruned wiring: value projection keeps 230 of 768 rows
        dict(name="prune 16x512", kind="prune", d=768, seq=512, batch=16, sparsity=0.8, rows_pruned=0.7, mask="zeros"),
        # attention-aware pruning through the whole layer
        dict(name="attnaware 32x256", kind="attnaware", d=768, seq=256, batch=32, rows_pruned=0.7, mask="zeros"),
        # a 12-layer model over a large batch of sequences of 32 to 512 rows
        dict(name="stack 12x 64x512", kind="stack", d=768, seq=512, batch=64, layers=12, sparsity=0.8, shortest=32),
        # the same model answering a handful of requests
        dict(name="stack 12x 6x100", kind="stack", d=768, seq=100, batch=6, layers=12, sparsity=0.8, shortest=9),
        # one feed-forward linear of a user who builds a layer of their own
        dict(name="linear 4096 768-3072", kind="linear", rows=4096, inputs=768, outputs=3072, sparsity=0.8, gelu=True),
        # the reference's launcher on the caller's arrays, ragged row count, inputs beyond one panel
        dict(name="launcher 1000 3072-768", kind="launcher", rows=1000, inputs=3072, outputs=768, sparsity=0.8, gelu=False),
        # skip connection + LayerNorm on its own, operands beyond the last-level cache
        dict(name="layernorm 131072x768", kind="layernorm", rows=131072, d=768),
    ]


def _between(rng, lo, hi):
    """an integer, its logarithm uniform"""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random):
    kind = rng.choice(("layer", "layer", "layer", "layer", "prune", "attnaware", "stack", "stack", "linear", "linear",
                       "launcher", "layernorm"))
    d = rng.choice((512, 768, 768, 768, 1024))
    rows = _between(rng, 16, MOST_ROWS)
    seq = min(rows, _between(rng, 16, 1024))
    batch = max(1, rows // seq)
    if kind == "layer":
        return dict(kind=kind, d=d, seq=seq, batch=batch, sparsity=rng.choice(SPARSITIES), mask=rng.choice(MASKS),
                    natural=rng.random() < 0.5)
    if kind == "prune":
        return dict(kind=kind, d=768, seq=seq, batch=batch, sparsity=rng.choice(SPARSITIES[1:]),
                    rows_pruned=rng.choice((0.5, 0.7, 0.8)), mask=rng.choice(MASKS))
    if kind == "attnaware":
        return dict(kind=kind, d=768, seq=seq, batch=batch, rows_pruned=rng.choice((0.5, 0.7, 0.8)),
                    mask=rng.choice(MASKS))
    if kind == "stack":
        seq, batch = _between(rng, 32, 512), _between(rng, 1, 64)
        return dict(kind=kind, d=768, seq=seq, batch=batch, layers=rng.choice((4, 6, 12)), sparsity=rng.choice((0.5, 0.8, 0.9)),
                    shortest=max(1, seq // rng.randint(2, 16)))
    if kind == "layernorm":
        return dict(kind=kind, rows=_between(rng, 16, 131072), d=d)
    inputs, outputs = rng.choice(LINEARS)
    return dict(kind=kind, rows=rows if kind == "linear" else min(rows, 4096), inputs=inputs, outputs=outputs,
                sparsity=rng.choice(SPARSITIES if kind == "linear" else SPARSITIES[1:]), gelu=outputs > inputs)


class _Inputs:
    """Seeded values, drawn on the GPU (a model's worth of weights takes milliseconds there)."""

    def __init__(self, seed):
        self.seed = seed & 0x7FFFFFFF
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(self.seed)
        self.count = 0

    def device(self, *shape, std=1.0):
        return (torch.randn(shape, generator=self.gen, device="cuda") * std).to(torch.float16)

    def host(self, *shape, std=0.02):
        return self.device(*shape, std=std).cpu().numpy()

    def next_seed(self):
        self.count += 1
        return self.seed * 64 + self.count

    def tile_mat(self, inputs, outputs, sparsity):
        row_ptr, row_offset = formats.gen_sparse_tile_mat(outputs, inputs, sparsity, self.next_seed())
        return row_ptr, row_offset, self.host(row_offset.size * 256), self.host(outputs)

    def linear(self, inputs, outputs, rows, sparsity, gelu=False):
        row_ptr, row_offset, data, bias = self.tile_mat(inputs, outputs, sparsity)
        return Linear_tile(inputs, outputs, rows, row_offset.size, data, row_ptr, row_offset, bias, gelu)

    def row_linear(self, inputs, outputs, rows, row_id, heads, gelu=False):
        return Linear_row(inputs, outputs, rows, self.host(row_id.size, inputs), row_id, row_id.size,
                          self.host(row_id.size), heads, is_gelu=gelu)

    def kept_rows(self, n, pruned):
        return formats.gen_sparse_row_mat(n, pruned, self.next_seed())

    def layernorm(self, d):
        return [(1 + self.host(d, std=0.1)).astype(np.float16), self.host(d, std=0.1)] * 2

    def mask(self, kind, seq):
        if kind == "none":
            return None
        m = np.zeros((seq, seq), np.float16)
        if kind == "padding":  # the last eighth of the keys is padding
            m[:, seq - max(1, seq // 8):] = -30000.0
        elif kind == "dense":  # an additive bias per pair of positions
            m[:] = self.host(seq, seq, std=0.5)
        return m


def _workspace(cls, d, seq, heads, batch):
    return torch.empty(cls.buffer_size(d, seq, heads, batch) // 2, dtype=torch.float16, device="cuda")


def _tile_linears(g, d, dff, rows, sparsity):
    return [g.linear(d, d, rows, sparsity) for _ in range(4)] + [g.linear(d, dff, rows, sparsity, True),
                                                                 g.linear(dff, d, rows, sparsity)]


def _lengths(case, seed):
    r = np.random.default_rng(seed)
    return r.integers(case["shortest"], case["seq"] + 1, size=case["batch"]).astype(np.int32)


def prepare(case, seed):
    g, kind = _Inputs(seed), case["kind"]
    if kind == "layernorm":
        rows, d = case["rows"], case["d"]
        gamma, beta = (torch.from_numpy(a).cuda() for a in g.layernorm(d)[:2])
        return dict(kind=kind, x=g.device(rows, d), skip=g.device(rows, d), gamma=gamma, beta=beta)
    if kind in ("linear", "launcher"):
        rows, inputs, outputs = case["rows"], case["inputs"], case["outputs"]
        x = g.device(rows, inputs)
        out = torch.empty((rows, outputs), dtype=torch.float16, device="cuda")
        if kind == "linear":
            return dict(kind=kind, x=x, out=out, op=g.linear(inputs, outputs, rows, case["sparsity"], case["gelu"]))
        arrays = [torch.from_numpy(a).cuda() for a in g.tile_mat(inputs, outputs, case["sparsity"])]
        return dict(kind=kind, x=x, out=out, arrays=arrays, outputs=outputs, gelu=case["gelu"])

    d, seq, batch = case["d"], case["seq"], case["batch"]
    heads, dff = WIDTHS[d]
    rows = seq * batch
    x = g.device(rows, d)
    out = torch.empty_like(x)
    if kind == "stack":
        # (the layers run one after the other: they share one workspace)
        work = _workspace(Encoder_length, d, seq, heads, batch)
        layers = [Encoder_length(d, seq, heads, work, *_tile_linears(g, d, dff, rows, case["sparsity"]), *g.layernorm(d),
                                 None, batch) for _ in range(case["layers"])]
        op = Encoder_stack(layers, d, seq, batch)
        op.set_seq_lens(_lengths(case, 1))  # (of the case, not of the seed: work() counts their rows)
        return dict(kind=kind, op=op, x=x, out=out, work=work)
    mask = g.mask(case["mask"], seq)
    if kind == "layer":
        work = _workspace(Encoder_tile, d, seq, heads, batch)
        op = Encoder_tile(d, seq, heads, work, *_tile_linears(g, d, dff, rows, case["sparsity"]), *g.layernorm(d), mask, batch)
        if case["natural"]:
            op.set_log2_scale(kernels.LOG2E)
    elif kind == "prune":
        work = _workspace(Encoder_prune, d, seq, heads, batch)
        lin = _tile_linears(g, d, dff, rows, case["sparsity"])
        lin[2] = g.row_linear(d, d, rows, g.kept_rows(d, case["rows_pruned"]), heads)
        op = Encoder_prune(d, seq, heads, work, *lin, *g.layernorm(d), mask, batch)
    else:
        work = _workspace(Encoder_attnaware, d, seq, heads, batch)
        qk = formats.gen_head_balanced_rows(heads, d // heads, 32, g.next_seed())
        o_id, m1_id, m2_id = (g.kept_rows(n, case["rows_pruned"]) for n in (d, dff, d))
        hidden = (m1_id.size + 15) // 16 * 16
        lin = [g.row_linear(d, d, rows, qk, heads), g.row_linear(d, d, rows, qk, heads), g.linear(d, d, rows, 0.0),
               g.row_linear(d, d, rows, o_id, heads), g.row_linear(d, dff, rows, m1_id, heads, True),
               g.row_linear(hidden, d, rows, m2_id, heads)]
        op = Encoder_attnaware(d, seq, heads, work, *lin, *g.layernorm(d), mask, batch)
    return dict(kind=kind, op=op, x=x, out=out, work=work)


def run(state):
    kind = state["kind"]
    if kind == "layernorm":
        return kernels.skip_layernorm(state["x"], state["skip"], state["gamma"], state["beta"])
    if kind == "linear":
        return state["op"].run(state["x"], out=state["out"])
    if kind == "launcher":
        row_ptr, row_offset, data, bias = state["arrays"]
        return kernels.tile_spmm_add_bias(state["x"], row_ptr, row_offset, data, bias, state["outputs"], gelu=state["gelu"],
                                          out=state["out"])
    return state["op"].run(state["out"], state["x"])


def _tiles(inputs, outputs, sparsity):
    return int((inputs // 16) * (outputs // 16) * (1.0 - sparsity))


def work(case):
    kind = case["kind"]
    if kind == "layernorm":
        n = case["rows"] * case["d"]
        return {"bytes": 6 * n + 4 * case["d"], "flops": 0}
    if kind in ("linear", "launcher"):
        rows, inputs, outputs = case["rows"], case["inputs"], case["outputs"]
        nt = _tiles(inputs, outputs, case["sparsity"])
        return {"bytes": 2 * rows * (inputs + outputs) + 516 * nt + 2 * outputs, "flops": 512 * nt * rows}
    d, seq, batch = case["d"], case["seq"], case["batch"]
    dff = WIDTHS[d][1]
    lens = _lengths(case, 1).astype(np.int64) if kind == "stack" else np.full(batch, seq, np.int64)
    rows, pairs = int(lens.sum()), int((lens * lens).sum())
    mask = 2 * seq * seq if case.get("mask", "none") in ("padding", "dense") else 0
    if kind in ("layer", "stack"):
        nt = 4 * _tiles(d, d, case["sparsity"]) + 2 * _tiles(d, dff, case["sparsity"])
        n = case.get("layers", 1)
        act = 4 * rows * d if kind == "layer" else 2 * rows * d + 2 * batch * seq * d
        return {"bytes": act + n * 516 * nt + mask, "flops": n * (512 * nt * rows + 4 * pairs * d)}
    keep = 1.0 - case["rows_pruned"]
    if kind == "prune":
        nt = 3 * _tiles(d, d, case["sparsity"]) + 2 * _tiles(d, dff, case["sparsity"])
        kept = int(d * keep)
        return {"bytes": 4 * rows * d + 516 * nt + 2 * kept * d + mask,
                "flops": 512 * nt * rows + 2 * rows * d * kept + 2 * pairs * (d + kept)}
    o, m1 = int(d * keep), int(dff * keep)
    weights = d * d // 2 * 2 + d * d + o * d + m1 * d + o * m1  # query and key keep half of their rows
    return {"bytes": 4 * rows * d + 2 * weights + mask, "flops": 2 * rows * weights + 3 * pairs * d}


def tolerance(case):
    # fp16 operands and results, fp32 sums: a result is within half a unit in the last place (2^-11) of the exact
    # sum of what it was given; the intermediate activations of a layer are rounded the same way, so another order
    # of summation moves some of them by a unit, and a stack adds the layers up
    return {"rel": {"layer": 2e-3, "prune": 2e-3, "attnaware": 2e-3, "stack": 5e-3}.get(case["kind"], 1e-3)}
