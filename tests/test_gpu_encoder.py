"""Encoder layers (the reference's Encoder_* objects) against the CPU oracle."""
import math

import numpy as np
import pytest
import torch

import oracle.et_oracle as orc
from helpers import rng, randn_h, make_tile_linear, check_close

pytestmark = pytest.mark.gpu
LOG2E = math.log2(math.e)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def make_layer(r, d, dff, sp, seed, std=0.02, bias_std=0.02):
    shapes = [(d, d)] * 4 + [(dff, d), (d, dff)]
    lins = [make_tile_linear(r, n, k, sp, seed=seed + j, std=std, bias_std=bias_std) for j, (n, k) in enumerate(shapes)]
    ln = [randn_h(r, (d,), 0.1) + np.float16(1), randn_h(r, (d,), 0.1), randn_h(r, (d,), 0.1) + np.float16(1), randn_h(r, (d,), 0.1)]
    return lins, ln


def build_linears(lins, rows):
    from et_amd.encoder import Linear_tile
    return [Linear_tile(l["K"], l["N"], rows, l["row_offset"].size, l["data"], l["row_ptr"], l["row_offset"], l["bias"], j == 4)
            for j, l in enumerate(lins)]


def workspace(cls, d, S, H, B):
    return torch.empty(cls.buffer_size(d, S, H, B) // 2, dtype=torch.float16, device="cuda")


@pytest.mark.parametrize("S,B,sp,ls,use_mask", [
    (128, 1, 0.0, 1.0, True),       # config 1: dense single sequence
    (128, 2, 0.8, LOG2E, False),
    (512, 2, 0.8, 1.0, True),       # config 3 shape, batch cut to 2
])
def test_encoder_tile_layer(S, B, sp, ls, use_mask):
    from et_amd.encoder import Encoder_tile
    r = rng(500 + S + B)
    d, H, dff = 768, 12, 3072
    lins, ln = make_layer(r, d, dff, sp, seed=900)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5) if use_mask else None
    want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, ls)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    enc.set_log2_scale(ls)
    xd = dev(x)
    out = torch.empty_like(xd)
    got = host(enc.run(out, xd))
    check_close(got, want, what="Encoder_tile")
    # out may alias in (test/tile_test.cu:41 calls run(in, in))
    got2 = host(enc.run(xd, xd))
    assert np.array_equal(got2, got)


def test_encoder_tile_layer_config3_full_size():
    """The benchmark's layer at its size (batch 16 x seq 512, 80 % tiles, zero additive mask, the default
    workload): sequences do not interact, so the oracle runs two of them as a batch of their own and the
    full launch must agree on their rows; in place gives the same bits."""
    from et_amd.encoder import Encoder_tile
    r = rng(560)
    d, H, dff, S, B = 768, 12, 3072, 512, 16
    lins, ln = make_layer(r, d, dff, 0.8, seed=905)
    x = randn_h(r, (B * S, d))
    mask = np.zeros((S, S), np.float16)
    sample = [3, 15]
    rows = np.concatenate([np.arange(b * S, (b + 1) * S) for b in sample])
    want = orc.encoder_tile_layer(x[rows], lins, ln, mask, S, H, len(sample), None, 1.0)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    xd = dev(x)
    got = host(enc.run(torch.empty_like(xd), xd))
    check_close(got[rows], want, what="Encoder_tile, config 3 full size")
    assert np.array_equal(host(enc.run(xd, xd)), got)


@pytest.mark.parametrize("mode", [2, 3])
def test_encoder_tile_layer_with_the_paired_tail(mode):
    """an Encoder_tile sized and built while the paired layer tail is switched on runs its tail through
    et_tile_plan_run_tail_ws with the exchange area behind its workspace units: the oracle's layer, the same bits
    on a second run, and close to the default encoder's output (fp32 summation order differs)"""
    from et_amd import lib
    from et_amd.encoder import Encoder_tile
    r = rng(577)
    d, H, dff, S, B = 768, 12, 3072, 128, 10
    lins, ln = make_layer(r, d, dff, 0.8, seed=911)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.3)
    want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0)
    xd = dev(x)
    plain = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    base = host(plain.run(torch.empty_like(xd), xd))
    lib().et_tuning_set(b"tile_tail_pair", mode)
    try:
        assert Encoder_tile.buffer_size(d, S, H, B) > 5 * B * S * d * 2
        enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
        got = host(enc.run(torch.empty_like(xd), xd))
        again = host(enc.run(torch.empty_like(xd), xd))
    finally:
        lib().et_tuning_set(b"tile_tail_pair", 0)
    check_close(got, want, what=f"Encoder_tile with the paired tail (mode {mode})")
    assert np.array_equal(got, again)
    assert np.abs(got.astype(np.float32) - base.astype(np.float32)).max() <= 3e-2
    assert (got != base).mean() < 0.05
    assert (got != base).any()          # (it did take the other kernel: the fp32 sums are added in another order)


@pytest.mark.parametrize("kind", ["padding", "dense"])
def test_encoder_tile_layer_config3_full_size_with_a_mask(kind):
    """the same layer at the same size with masks that the attention launch has to read: a padding mask over the
    last 64 keys (whole key tiles that end early, the form the benchmark's latency_us_padding_mask times) and a
    dense random additive mask (every tile read and added); two sequences from across the batch against the
    oracle"""
    from et_amd.encoder import Encoder_tile
    r = rng(561)
    d, H, dff, S, B = 768, 12, 3072, 512, 16
    lins, ln = make_layer(r, d, dff, 0.8, seed=906)
    x = randn_h(r, (B * S, d))
    if kind == "padding":
        mask = np.zeros((S, S), np.float16)
        mask[:, S - 64:] = -30000.0
    else:
        mask = randn_h(r, (S, S), 0.5)
    sample = [0, 11]
    rows = np.concatenate([np.arange(b * S, (b + 1) * S) for b in sample])
    want = orc.encoder_tile_layer(x[rows], lins, ln, mask, S, H, len(sample), None, 1.0)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    xd = dev(x)
    got = host(enc.run(torch.empty_like(xd), xd))
    check_close(got[rows], want, what=f"Encoder_tile, config 3 full size, {kind} mask")


@pytest.mark.parametrize("d,H,dff,S,B,sp", [
    (1024, 16, 4096, 128, 8, 0.8),    # BERT-large widths: K = 1024 in one chunk, 4096 in six
    (1024, 16, 4096, 64, 1, 0.5),     # ... and on few rows
    (512, 8, 2048, 96, 40, 0.7),      # 3840 rows of 512: the one-launch tail on another width
    (384, 12, 1536, 50, 3, 0.6),      # head_dim 32
    (1024, 8, 2048, 80, 2, 0.8),      # head_dim 128
])
def test_encoder_tile_layer_other_widths(d, H, dff, S, B, sp):
    from et_amd.encoder import Encoder_tile
    r = rng(540 + d + S)
    lins, ln = make_layer(r, d, dff, sp, seed=905, std=0.03)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5)
    want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    xd = dev(x)
    got = host(enc.run(torch.empty_like(xd), xd))
    check_close(got, want, what=f"Encoder_tile, d_model {d}")
    assert np.array_equal(host(enc.run(xd, xd)), got)


@pytest.mark.parametrize("S,B", [(128, 2), (200, 3)])
def test_encoder_tile_layer_fused_tail_forced(S, B):
    """the one-launch layer tail (normally used for more row panels) inside Encoder_tile, forced on small shapes"""
    from et_amd import lib
    from et_amd.encoder import Encoder_tile
    r = rng(620 + S)
    d, H, dff = 768, 12, 3072
    lins, ln = make_layer(r, d, dff, 0.8, seed=940)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5)
    want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    xd = dev(x)
    stepwise = host(enc.run(torch.empty_like(xd), xd))
    try:
        lib().et_tuning_set(b"tile_ln_min_panels", 1)
        fused = host(enc.run(torch.empty_like(xd), xd))
        inplace = host(enc.run(xd, xd))
    finally:
        lib().et_tuning_set(b"tile_ln_min_panels", 0)
    check_close(fused, want, what="Encoder_tile, fused tail")
    check_close(stepwise, want, what="Encoder_tile, step by step")
    assert np.abs(fused.astype(np.float32) - stepwise.astype(np.float32)).max() <= 2e-2
    assert np.array_equal(inplace, fused)


def test_encoder_tile_layer_vs_torch_fp32_layer():
    """Independent of the oracle: a textbook post-LN transformer layer written with torch ops in fp32 on the CPU
    (dense weights with the pruned tiles zeroed, softmax base e, tanh GELU, LayerNorm eps 1e-6)."""
    import torch.nn.functional as F
    from et_amd.encoder import Encoder_tile
    r = rng(77)
    d, H, dff, S, B = 768, 12, 3072, 128, 2
    hd = d // H
    lins, ln = make_layer(r, d, dff, 0.8, seed=960, std=0.03, bias_std=0.05)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5)

    def dense(l):
        W = np.zeros((l["N"], l["K"]), np.float32)
        rp, ro, data = l["row_ptr"], l["row_offset"], l["data"].reshape(-1, 16, 16)
        for bn in range(l["N"] // 16):
            for i in range(rp[bn], rp[bn + 1]):
                W[bn * 16:(bn + 1) * 16, ro[i]:ro[i] + 16] = data[i]
        return torch.from_numpy(W), torch.from_numpy(l["bias"].astype(np.float32))

    (Wq, bq), (Wk, bk), (Wv, bv), (Wo, bo), (W1, b1), (W2, b2) = [dense(l) for l in lins]
    g1, be1, g2, be2 = [torch.from_numpy(t.astype(np.float32)) for t in ln]
    xt = torch.from_numpy(x.astype(np.float32))
    q, k, v = F.linear(xt, Wq, bq), F.linear(xt, Wk, bk), F.linear(xt, Wv, bv)
    heads = lambda t: t.view(B, S, H, hd).transpose(1, 2)
    # the reference scales by half(sqrt(1/head_dim)) (kernels/attention.cu:126)
    scale = float(np.float16(math.sqrt(1.0 / hd)))
    p = torch.softmax(heads(q) @ heads(k).transpose(-1, -2) * scale + torch.from_numpy(mask.astype(np.float32)), -1)
    attn = (p @ heads(v)).transpose(1, 2).reshape(B * S, d)
    mid = F.layer_norm(F.linear(attn, Wo, bo) + xt, (d,), g1, be1, eps=1e-6)
    y = F.layer_norm(F.linear(F.gelu(F.linear(mid, W1, b1), approximate="tanh"), W2, b2) + mid, (d,), g2, be2, eps=1e-6)
    enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    enc.set_log2_scale(LOG2E)  # textbook softmax instead of the reference's base 2
    xd = dev(x)
    got = host(enc.run(torch.empty_like(xd), xd))
    # half storage between the steps against fp32 throughout
    check_close(got, y.numpy(), max_abs=3e-2, mean_rel=3e-3, what="Encoder_tile vs torch fp32 layer")


def test_encoder_prune_layer():
    prune_case(768, 12, 3072, 128, 2)


@pytest.mark.parametrize("S,B", [(37, 1), (128, 2), (300, 7)])
def test_encoder_prune_layer_1024_wide(S, B):
    """V's plan has two column chunks there, Q's and K's one"""
    prune_case(1024, 16, 4096, S, B)


def prune_case(d, H, dff, S, B):
    from et_amd.encoder import Encoder_prune, Linear_row
    r = rng(600)
    lins, ln = make_layer(r, d, dff, 0.8, seed=910)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5)
    v_id = orc.gen_sparse_row_mat(d, 0.7, seed=5)              # 230 surviving V rows
    Wv, bv = randn_h(r, (v_id.size, d), 0.02), randn_h(r, (v_id.size,), 0.02)
    # oracle: step by step (encoder/encoder.cu:65-92)
    tl = lambda j, inp, g=False: orc.tile_linear(inp, lins[j]["row_ptr"], lins[j]["row_offset"], lins[j]["data"], lins[j]["bias"], lins[j]["N"], gelu=g)
    q, k = tl(0, x), tl(1, x)
    vc = orc.row_linear(x, Wv, bv)
    z = orc.prune_attention(q, k, vc, None, v_id, orc.head_ptr(v_id, H, d // H), mask, S, d, H, B)
    h1 = orc.skip_layernorm(tl(3, z), x, ln[0], ln[1])
    want = orc.skip_layernorm(tl(5, tl(4, h1, True)), h1, ln[2], ln[3])
    L = build_linears(lins, B * S)
    L[2] = Linear_row(d, d, B * S, Wv, v_id, v_id.size, bv, H)
    assert d != 768 or (L[2].nrow == 240 and L[2].row_id_size == 230)
    enc = Encoder_prune(d, S, H, workspace(Encoder_prune, d, S, H, B), *L, *ln, mask, B)
    xd = dev(x)
    got = host(enc.run(torch.empty_like(xd), xd))
    check_close(got, want, what="Encoder_prune")


@pytest.mark.parametrize("balanced", [True, False])
def test_encoder_attnaware_layer_config4_wiring(balanced):
    """Attention-aware pruning through the layer: Q/K keep 32 of 64 columns per head (same set), O/FFN1/FFN2 row-pruned at 70 %.
    Oracle = its own ops chained step by step; invariant = the same layer with DENSE linears whose pruned
    rows are zero (and, for FFN2, the dropped hidden units' columns).  balanced = False moves 12 kept
    columns from head 0 to head 1 (20 and 44 columns): the ragged pruned-attention kernel instead of the
    narrow-head one."""
    attnaware_case(S=64, B=2, balanced=balanced, sample=[0, 1])


def test_encoder_attnaware_layer_config4_full_size():
    """the same layer at the benchmark's size (batch 32 x seq 256).  Sequences do not interact, so the
    oracle runs three of them as a batch of their own and the full launch must agree on their rows."""
    attnaware_case(S=256, B=32, balanced=True, sample=[0, 17, 31])


@pytest.mark.parametrize("S,B,balanced,sample", [(37, 1, True, [0]), (64, 2, False, [0, 1]), (250, 8, True, [5])])
def test_encoder_attnaware_layer_1024_wide(S, B, balanced, sample):
    """Q's and K's plans have two column chunks there, V's one"""
    attnaware_case(S, B, balanced, sample, d=1024, H=16, dff=4096)


def attnaware_case(S, B, balanced, sample, d=768, H=12, dff=3072):
    from et_amd.encoder import Encoder_attnaware, Linear_row, Linear_tile
    r = rng(650)
    hd = d // H
    x_all = randn_h(r, (B * S, d))
    rows = np.concatenate([np.arange(b * S, (b + 1) * S) for b in sample])
    x, Bfull, B = x_all[rows], B, len(sample)   # the oracle's batch: the sampled sequences
    T = B * S
    mask = randn_h(r, (S, S), 0.5)
    ln = [randn_h(r, (d,), 0.2) + np.float16(1), randn_h(r, (d,), 0.2), randn_h(r, (d,), 0.2) + np.float16(1), randn_h(r, (d,), 0.2)]
    W = {k: randn_h(r, shp, 0.03) for k, shp in dict(q=(d, d), k=(d, d), v=(d, d), o=(d, d), m1=(dff, d), m2=(d, dff)).items()}
    bsz = {k: randn_h(r, (W[k].shape[0],), 0.05) for k in W}
    qk_id = orc.gen_head_balanced_rows(H, hd, 32, seed=11)       # 384 kept Q/K columns, 32 per head
    if not balanced:
        spare = np.setdiff1d(np.arange(hd, 2 * hd), qk_id)[:12]  # unused columns of head 1
        qk_id = np.sort(np.concatenate([qk_id[12:], spare])).astype(np.int32)
        assert np.array_equal(orc.head_ptr(qk_id, H, hd)[:3], [0, 20, 64])
    o_id = orc.gen_sparse_row_mat(d, 0.7, seed=12)               # 230 rows
    m1_id = orc.gen_sparse_row_mat(dff, 0.7, seed=13)            # 921 rows
    m2_id = orc.gen_sparse_row_mat(d, 0.7, seed=14)              # 230 rows
    pad16 = lambda n: (n + 15) // 16 * 16
    # FFN2 sees the compact hidden: gather its input columns to the kept hidden units, pad to FFN1's padded width
    W2c = np.zeros((m2_id.size, pad16(m1_id.size)), np.float16)
    W2c[:, :m1_id.size] = W["m2"][m2_id][:, m1_id]

    # ---- oracle, step by step
    qc, kc = orc.row_linear(x, W["q"][qk_id], bsz["q"][qk_id]), orc.row_linear(x, W["k"][qk_id], bsz["k"][qk_id])
    vfull = (x.astype(np.float32) @ W["v"].astype(np.float32).T + bsz["v"].astype(np.float32)).astype(np.float16)
    z = orc.prune_attention(qc, kc, vfull, orc.head_ptr(qk_id, H, hd), None, None, mask, S, d, H, B)
    def scatter(c, ids):
        out = np.zeros((T, d), np.float16)
        out[:, ids] = c[:, :ids.size]
        return out
    h1 = orc.skip_layernorm(scatter(orc.row_linear(z, W["o"][o_id], bsz["o"][o_id]), o_id), x, ln[0], ln[1])
    hid = orc.gelu(orc.row_linear(h1, W["m1"][m1_id], bsz["m1"][m1_id]))
    hid_p = np.zeros((T, pad16(m1_id.size)), np.float16)
    hid_p[:, :m1_id.size] = hid
    want = orc.skip_layernorm(scatter(orc.row_linear(hid_p, W2c, bsz["m2"][m2_id]), m2_id), h1, ln[2], ln[3])

    # ---- invariant: dense linears with the pruned rows zeroed give the same layer (fp64)
    def zero_rows(w, b, ids):
        wz, bz = np.zeros_like(w, np.float64), np.zeros_like(b, np.float64)
        wz[ids], bz[ids] = w[ids], b[ids]
        return wz, bz
    x64 = x.astype(np.float64)
    lin = lambda inp, wb: (inp @ wb[0].T + wb[1]).astype(np.float16)
    qd, kd = lin(x64, zero_rows(W["q"], bsz["q"], qk_id)), lin(x64, zero_rows(W["k"], bsz["k"], qk_id))
    zd = orc.otf_attention(qd, kd, vfull, mask, S, H, B, None, 1.0, f64=True)
    h1d = orc.skip_layernorm(lin(zd.astype(np.float64), zero_rows(W["o"], bsz["o"], o_id)), x, ln[0], ln[1], f64=True)
    hidd = orc.gelu(lin(h1d.astype(np.float64), zero_rows(W["m1"], bsz["m1"], m1_id)))
    hidd[:, np.setdiff1d(np.arange(dff), m1_id)] = 0               # gelu(0) = 0 anyway
    outd = orc.skip_layernorm(lin(hidd.astype(np.float64), zero_rows(W["m2"], bsz["m2"], m2_id)), h1d, ln[2], ln[3], f64=True)
    check_close(want, outd, what="config-4 oracle vs dense-with-zeroed-rows")

    # ---- the class
    vt = dict(N=d, K=d)
    vt["row_ptr"], vt["row_offset"] = orc.gen_sparse_tile_mat(d, d, 0.0, seed=1)
    vt["data"] = orc.tile_pack(W["v"], vt["row_ptr"], vt["row_offset"])
    B, T = Bfull, Bfull * S                     # the device runs the whole batch
    Lq = Linear_row(d, d, T, W["q"][qk_id], qk_id, qk_id.size, bsz["q"][qk_id], H)
    Lk = Linear_row(d, d, T, W["k"][qk_id], qk_id, qk_id.size, bsz["k"][qk_id], H)
    Lv = Linear_tile(d, d, T, vt["row_offset"].size, vt["data"], vt["row_ptr"], vt["row_offset"], bsz["v"], False)
    Lo = Linear_row(d, d, T, W["o"][o_id], o_id, o_id.size, bsz["o"][o_id], H)
    L1 = Linear_row(d, dff, T, W["m1"][m1_id], m1_id, m1_id.size, bsz["m1"][m1_id], H, is_gelu=True)
    L2 = Linear_row(pad16(m1_id.size), d, T, W2c, m2_id, m2_id.size, bsz["m2"][m2_id], H)
    assert (Lq.nrow, Lo.nrow, L1.nrow, L2.nrow) == ((384, 240, 928, 240) if d == 768 else (512, 320, 1232, 320))
    enc = Encoder_attnaware(d, S, H, workspace(Encoder_attnaware, d, S, H, B), Lq, Lk, Lv, Lo, L1, L2, *ln, mask, B)
    xd = dev(x_all)
    got = host(enc.run(torch.empty_like(xd), xd))[rows]
    check_close(got, want, what="Encoder_attnaware")
    check_close(got, outd, what="Encoder_attnaware vs dense-with-zeroed-rows")


@pytest.mark.parametrize("M,K,n,size,alias", [
    (1, 64, 5, 64, False),              # one row, one block-row
    (15, 768, 230, 768, True),          # the last block-row padded; out over the skip rows
    (17, 624, 154, 768, False),         # an odd number of tiles in a list; rows of X narrower than the result
    (1025, 1024, 384, 1024, False),     # three block-rows a wave, two pieces a lane
    (4097, 928, 230, 768, True),        # 32 rows a workgroup, the last one with one
    (4130, 512, 130, 512, False),       # one piece a lane
    (8200, 768, 377, 768, False),       # 64 rows a workgroup
    (40, 1104, 100, 768, False),        # two column chunks: the two launches
    (40, 768, 385, 768, False),         # too wide: the two launches
])
def test_row_linear_scatter_layernorm(M, K, n, size, alias):
    """row-pruned linear + expansion + skip + LayerNorm against the oracle's steps"""
    import ctypes as C
    from et_amd import lib
    from et_amd._lib import check
    r = rng(2500 + M + K)
    N = (n + 15) // 16 * 16
    W = np.zeros((N, K), np.float16)
    W[:n] = randn_h(r, (n, K), 0.04)
    bias = np.zeros(N, np.float16)
    bias[:n] = randn_h(r, (n,), 0.1)
    col = np.sort(r.permutation(size)[:n]).astype(np.int32)
    X, skip = randn_h(r, (M, K)), randn_h(r, (M, size))
    gamma, beta = randn_h(r, (size,), 0.2) + np.float16(1), randn_h(r, (size,), 0.2)
    rows = np.unique(np.concatenate([np.arange(min(M, 40)), np.arange(max(M - 40, 0), M)]))
    y = np.zeros((rows.size, size), np.float16)
    y[:, col] = orc.row_linear(X[rows], W, bias)[:, :n]
    want = orc.skip_layernorm(y, skip[rows], gamma, beta)
    rp = (np.arange(N // 16 + 1) * (K // 16)).astype(np.int32)
    ro = np.tile(np.arange(K // 16) * 16, N // 16).astype(np.int32)
    data = orc.tile_pack(W, rp, ro)
    L, p = lib(), C.c_void_p()
    check(L.et_tile_plan_create(C.byref(p), K, N, ro.size, data.ctypes.data, rp.ctypes.data, ro.ctypes.data, bias.ctypes.data))
    try:
        Xd, sd, gd, bd, cd = dev(X), dev(skip), dev(gamma), dev(beta), dev(col)
        out = sd if alias else torch.empty_like(sd)
        compact = torch.empty((M, N), dtype=torch.float16, device="cuda")
        check(L.et_tile_plan_run_scatter_ln(p, out.data_ptr(), Xd.data_ptr(), compact.data_ptr(), cd.data_ptr(), n, sd.data_ptr(),
                                            gd.data_ptr(), bd.data_ptr(), size, M, torch.cuda.current_stream().cuda_stream))
        check_close(host(out)[rows], want, what="row linear + LayerNorm")
    finally:
        L.et_tile_plan_destroy(p)


@pytest.mark.parametrize("M,K,n,size,alias", [
    (1, 64, 3, 8, True),                # one piece in all
    (17, 64, 20, 264, False),           # a piece behind the first 32 lanes
    (31, 128, 40, 520, True),           # ... and behind two whole pieces; the last pair of rows has one
    (33, 64, 50, 776, False),           # four pieces a lane, the last one lane's
    (4104, 96, 30, 1016, True),         # 32 rows a workgroup, two pairs a wave
])
def test_row_linear_scatter_layernorm_rows_in_pairs(M, K, n, size, alias):
    """two rows of a wave at once, 32 lanes each: widths that leave lanes without a piece"""
    test_row_linear_scatter_layernorm(M, K, n, size, alias)


def test_encoder_length_paths():
    from et_amd.encoder import Encoder_length
    r = rng(700)
    d, H, dff, S, B = 768, 12, 3072, 256, 3
    lins, ln = make_layer(r, d, dff, 0.8, seed=920)
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5)
    enc = Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    xd = dev(x)
    want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0)
    got = host(enc.run(torch.empty_like(xd), xd))
    check_close(got, want, what="Encoder_length, on-the-fly")
    enc.set_shared_qk(True)       # the reference's own route: scores through memory (encoder/encoder.cu:126-137)
    got_s = host(enc.run(torch.empty_like(xd), xd))
    check_close(got_s, want, what="Encoder_length, shared QK")
    enc.set_shared_qk(False)
    lens = np.array([256, 40, 131], np.int32)
    enc.set_seq_lens(lens)
    want_l = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, lens, 1.0)
    got_l = host(enc.run(torch.empty_like(xd), xd))
    for b in range(B):   # valid positions equal the padded run; padding rows are zero
        sl = slice(b * S, b * S + lens[b])
        check_close(got_l[sl], want_l[sl], what=f"Encoder_length packed, seq {b}")
        assert (got_l[b * S + lens[b]:(b + 1) * S] == 0).all()
    got_alias = host(enc.run(xd, xd))
    assert np.array_equal(got_alias, got_l)
    # lengths outside [0, seq_len] are refused by the C++ class before anything is uploaded (the Python
    # class has its own check in front, so the C entry point is called directly)
    import ctypes as C
    from et_amd import lib
    for bad in ([256, 257, 1], [5, -1, 3]):
        arr = (C.c_int * B)(*bad)
        assert lib().et_encoder_set_seq_lens(enc._h, C.cast(arr, C.c_void_p)) < 0
        assert b"seq_len" in lib().et_last_error()
    got_after = host(enc.run(torch.empty_like(xd), dev(x)))     # the refused calls changed nothing
    assert np.array_equal(got_after, got_l)


def test_encoder_stack_variable_length():
    from et_amd.encoder import Encoder_length, Encoder_stack
    r = rng(800)
    d, H, dff, S, B, NL = 256, 4, 1024, 128, 4, 3
    layers, params = [], []
    for i in range(NL):
        lins, ln = make_layer(r, d, dff, 0.5, seed=930 + 10 * i, std=0.05)
        params.append((lins, ln))
        layers.append(Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, None, B))
    x = randn_h(r, (B * S, d))
    lens = np.array([128, 9, 77, 50], np.int32)
    stack = Encoder_stack(layers, d, S, B)
    stack.set_seq_lens(lens)
    xd = dev(x)
    got = host(stack.run(torch.empty_like(xd), xd))
    cur = x
    for lins, ln in params:
        cur = orc.encoder_tile_layer(cur, lins, ln, None, S, H, B, lens, 1.0)
    for b in range(B):
        sl = slice(b * S, b * S + lens[b])
        check_close(got[sl], cur[sl], what=f"stack seq {b}")
        assert (got[b * S + lens[b]:(b + 1) * S] == 0).all()
    stack.set_seq_lens(None)    # full-length batch through the same stack
    got_full = host(stack.run(torch.empty_like(xd), xd))
    cur = x
    for lins, ln in params:
        cur = orc.encoder_tile_layer(cur, lins, ln, None, S, H, B, None, 1.0)
    check_close(got_full, cur, what="stack full length")


def test_encoder_stack_config5_full_size():
    """The benchmark's stack at its size: 12 BERT-base layers, 80 % tile-pruned, batch 64, lengths drawn from
    32..512 and padded to 512.  Sequences do not interact, so the oracle runs three of them (the shortest,
    a middle one, the longest) one at a time through the 12 layers; the packed run must agree on their
    valid rows and leave their padding rows zero, and the padded run on the shortest one's 512 rows.
    Tolerance for TWELVE layers: max-abs 4e-2, mean-rel 3e-3 (one layer's is 2e-2 / 1e-3)."""
    from et_amd.encoder import Encoder_length, Encoder_stack
    r = rng(810)
    d, H, dff, S, B, NL = 768, 12, 3072, 512, 64, 12
    lens = r.integers(32, 513, size=B).astype(np.int32)
    layers, params = [], []
    for i in range(NL):
        lins, ln = make_layer(r, d, dff, 0.8, seed=1000 + 10 * i)
        params.append((lins, ln))
        layers.append(Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, None, B))
    x = randn_h(r, (B * S, d))
    stack = Encoder_stack(layers, d, S, B)
    stack.set_seq_lens(lens)
    xd = dev(x)
    got = host(stack.run(torch.empty_like(xd), xd))
    order = np.argsort(lens, kind="stable")
    def oracle_seq(b, n):
        cur = x[b * S:(b + 1) * S]
        for lins, ln in params:
            cur = orc.encoder_tile_layer(cur, lins, ln, None, S, H, 1, None if n == S else np.array([n], np.int32), 1.0)
        return cur
    for b in (order[0], order[B // 2], order[-1]):
        want = oracle_seq(b, lens[b])
        check_close(got[b * S:b * S + lens[b]], want[:lens[b]], max_abs=4e-2, mean_rel=3e-3, what=f"packed stack, seq {b} ({lens[b]} rows)")
    for b in range(B):
        assert (got[b * S + lens[b]:(b + 1) * S] == 0).all()
    stack.set_seq_lens(None)
    got_full = host(stack.run(torch.empty_like(xd), xd))
    b = order[0]
    check_close(got_full[b * S:(b + 1) * S], oracle_seq(b, S), max_abs=4e-2, mean_rel=3e-3, what="padded stack")


def test_encoder_runs_inside_a_captured_hip_graph():
    """run() allocates nothing, never synchronises and issues only kernel launches on the caller's
    stream, so a caller can capture it in a HIP graph: every replay equals the eager result."""
    from et_amd.encoder import Encoder_length, Encoder_stack, Encoder_tile
    r = rng(810)
    d, H, dff, S, B, NL = 256, 4, 1024, 128, 4, 2
    lens = np.array([128, 9, 77, 50], np.int32)
    layers = []
    for i in range(NL):
        lins, ln = make_layer(r, d, dff, 0.5, seed=960 + 10 * i, std=0.05)
        layers.append(Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, None, B))
    stack = Encoder_stack(layers, d, S, B)
    stack.set_seq_lens(lens)
    lins, ln = make_layer(r, d, dff, 0.8, seed=990, std=0.05)
    mask = randn_h(r, (S, S), 0.5)
    tile = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *build_linears(lins, B * S), *ln, mask, B)
    inputs = [dev(randn_h(r, (B * S, d))) for _ in range(3)]
    for name, run in (("stack, packed rows", stack.run), ("Encoder_tile", tile.run)):
        eager = [host(run(torch.empty_like(x), x)) for x in inputs]
        x_static, out_static = torch.empty_like(inputs[0]), torch.empty_like(inputs[0])
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):   # warm-up on the capture stream
            x_static.copy_(inputs[0])
            run(out_static, x_static)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            run(out_static, x_static)
        for k in (1, 2, 0, 2):          # eager work and synchronisations between the replays
            x_static.copy_(inputs[k])
            out_static.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(host(out_static), eager[k]), f"{name}: replay with input {k}"
            again = host(run(torch.empty_like(inputs[k]), inputs[k]))
            assert np.array_equal(again, eager[k])
        del graph


@pytest.mark.parametrize("program", ["tile_test", "prune_test", "length_test"])
def test_cpp_caller_of_the_reference_classes(tmp_path, program):
    """et_amd/examples/*.cpp are the reference's test/tile_test.cu, prune_test.cu and length_test.cu on this
    library's headers (plain C++, no HIP headers, linked with -let_amd).  Each one's output equals the same
    layer built through the Python binding, bit for bit, and the oracle within tolerance."""
    import os
    import subprocess
    from et_amd import formats
    from et_amd.encoder import Encoder_length, Encoder_prune, Encoder_tile, Linear_row
    exe = os.path.join(os.path.dirname(os.path.abspath(formats.__file__)), "examples", program)
    assert os.path.exists(exe), "built by et_amd.build (build_examples)"
    S, B, sp = 128, 2, 0.8
    d, H, dff = 768, 12, 3072
    out_path = str(tmp_path / "out.bin")
    res = subprocess.run([exe, out_path, str(S), str(B), str(sp)], capture_output=True, text=True, timeout=110)
    assert res.returncode == 0, res.stderr
    got = np.fromfile(out_path, dtype=np.float16).reshape(-1, d)
    # the same layer here: seeds 1..6, surviving weights 0.01, biases 0.1, gamma 1, beta 0, zero mask
    shapes = [(d, d)] * 4 + [(dff, d), (d, dff)]
    lins = []
    for seed, (N, Kd) in enumerate(shapes, start=1):
        rp, ro = formats.gen_sparse_tile_mat(N, Kd, sp, seed)
        lins.append(dict(N=N, K=Kd, row_ptr=rp, row_offset=ro, data=np.full(ro.size * 256, 0.01, np.float16),
                         bias=np.full(N, 0.1, np.float16)))
    s, vals = 12345, np.empty(B * S * d, np.float32)
    for i in range(vals.size):          # the programs' 64-bit LCG
        s = (s * 6364136223846793005 + 1442695040888963407) & 0xFFFFFFFFFFFFFFFF
        vals[i] = np.float32(s >> 40) * np.float32(1.0 / 8388608.0) - np.float32(1.0)
    x = vals.astype(np.float16).reshape(B * S, d)
    ln = [np.ones(d, np.float16), np.zeros(d, np.float16)] * 2
    mask = np.zeros((S, S), np.float16)
    xd = dev(x)
    L = build_linears(lins, B * S)
    if program == "tile_test":
        enc = Encoder_tile(d, S, H, workspace(Encoder_tile, d, S, H, B), *L, *ln, mask, B)
        same = host(enc.run(torch.empty_like(xd), xd))
        want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0)
    elif program == "prune_test":
        v_id = formats.gen_sparse_row_mat(d, sp, 3)
        Wv, bv = np.full((v_id.size, d), 0.01, np.float16), np.full(v_id.size, 0.1, np.float16)
        L[2] = Linear_row(d, d, B * S, Wv, v_id, v_id.size, bv, H)
        enc = Encoder_prune(d, S, H, workspace(Encoder_prune, d, S, H, B), *L, *ln, mask, B)
        same = host(enc.run(torch.empty_like(xd), xd))
        tl = lambda j, inp, g=False: orc.tile_linear(inp, lins[j]["row_ptr"], lins[j]["row_offset"],
                                                     lins[j]["data"], lins[j]["bias"], lins[j]["N"], gelu=g)
        z = orc.prune_attention(tl(0, x), tl(1, x), orc.row_linear(x, Wv, bv), None, v_id,
                                orc.head_ptr(v_id, H, d // H), mask, S, d, H, B)
        h1 = orc.skip_layernorm(tl(3, z), x, ln[0], ln[1])
        want = orc.skip_layernorm(tl(5, tl(4, h1, True)), h1, ln[2], ln[3])
    else:
        enc = Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *L, *ln, mask, B)
        full = host(enc.run(torch.empty_like(xd), xd))
        lens = np.array([max(S - 7 * b, 1) for b in range(B)], np.int32)
        enc.set_seq_lens(lens)
        same = np.concatenate([full, host(enc.run(torch.empty_like(xd), xd))])
        want = np.concatenate([orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, None, 1.0),
                               orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, lens, 1.0)])
        for b in range(B):              # padding rows of the packed run are zero on the device
            want[B * S + b * S + lens[b]:B * S + (b + 1) * S] = 0
    assert got.shape == same.shape and np.array_equal(got, same)
    check_close(got, want, what="C++ caller " + program)


@pytest.mark.parametrize("d,H,dff,S,B,sp,lens,use_mask", [
    (768, 12, 3072, 1, 1, 0.8, None, False),           # one row
    (768, 12, 3072, 16, 1, 0.8, None, True),           # one whole panel
    (768, 12, 3072, 17, 3, 0.5, None, True),           # panels that hold rows of two sequences
    (768, 12, 3072, 96, 1, 0.9, None, False),          # the most rows
    (1024, 16, 4096, 24, 2, 0.8, [24, 0], False),      # six chunks of the hidden width; an empty sequence
    (64, 2, 128, 3, 30, 0.6, [3, 1, 2] * 10, True),    # head width 32, many sequences per panel
    (512, 8, 2048, 40, 2, 0.0, [7, 33], False),        # dense
])
def test_layer_in_one_launch(request, d, H, dff, S, B, sp, lens, use_mask):
    """few rows: the whole layer as one launch (padded, and packed where lengths are given) against the oracle and
    against the separate launches; runs repeat bit for bit, also from a captured graph between eager runs"""
    from et_amd import lib
    from et_amd.encoder import Encoder_length
    # (dense weights would have 80 rows run as separate launches)
    request.addfinalizer(lambda: lib().et_tuning_set(b"layer_flow_rows", -1))
    lib().et_tuning_set(b"layer_flow_rows", 96)
    r = rng(1300 + d + S * B)
    lins, ln = make_layer(r, d, dff, sp, seed=1400 + S, std=0.03, bias_std=0.05)
    mask = randn_h(r, (S, S), 0.5) if use_mask else None
    work = workspace(Encoder_length, d, S, H, B).fill_(7.0)
    enc = Encoder_length(d, S, H, work, *build_linears(lins, B * S), *ln, mask, B)
    xs = [randn_h(r, (B * S, d)) for _ in range(3)]
    for use in ([None, np.array(lens, np.int32)] if lens else [None]):
        enc.set_seq_lens(use)
        valid = np.concatenate([np.arange(b * S, b * S + (S if use is None else use[b])) for b in range(B)])
        got = [host(enc.run(torch.empty_like(dev(x)), dev(x))) for x in xs]
        for x, g in zip(xs, got):
            want = orc.encoder_tile_layer(x, lins, ln, mask, S, H, B, use, 1.0)
            check_close(g[valid], want[valid], what="layer in one launch")
            assert (np.delete(g, valid, 0) == 0).all()
        if use is None:                 # (it is that form: the separate launches write the workspace)
            assert (host(work) == 7.0).all()
        try:
            lib().et_tuning_set(b"layer_flow_rows", 0)
            steps = host(enc.run(torch.empty_like(dev(xs[0])), dev(xs[0])))
        finally:
            lib().et_tuning_set(b"layer_flow_rows", 96)
        assert (host(work) != 7.0).any()
        assert np.abs(steps.astype(np.float32) - got[0].astype(np.float32)).max() <= 2e-2
        x_static, out_static = torch.empty_like(dev(xs[0])), torch.empty_like(dev(xs[0]))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            enc.run(out_static, x_static)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            enc.run(out_static, x_static)
        for k in (1, 0, 2, 0):
            x_static.copy_(dev(xs[k]))
            out_static.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(host(out_static), got[k])
            assert np.array_equal(host(enc.run(torch.empty_like(x_static), dev(xs[k]))), got[k])
        del graph


@pytest.mark.parametrize("d,H,dff,S,B,sp,lens,use_mask", [
    (768, 12, 3072, 10, 9, 0.8, None, True),           # a head's projections and attention as a unit; more units than CUs
    (768, 12, 3072, 33, 2, 0.9, [33, 1], False),       # ... a CU for every unit; one row behind two panels
    (512, 8, 2048, 16, 5, 0.9, [16, 0, 7, 16, 0], True),  # empty sequences have no unit when packed
    (256, 4, 1024, 96, 1, 0.0, None, False),           # dense lists short enough for a wave
])
def test_layer_in_one_launch_heads_as_units(request, d, H, dff, S, B, sp, lens, use_mask):
    test_layer_in_one_launch(request, d, H, dff, S, B, sp, lens, use_mask)


@pytest.mark.parametrize("d,H,dff,S,B,one_launch", [
    (512, 8, 2048, 128, 1, True),      # 216 units
    (512, 8, 2048, 75, 2, False),      # 276: beyond the line
    (768, 12, 3072, 96, 1, True),      # 246
    (768, 12, 3072, 112, 1, False),    # 285
])
def test_layer_in_one_launch_by_its_units(d, H, dff, S, B, one_launch):
    """either side of the line, against the oracle; the separate launches write the workspace, the one launch does not"""
    from et_amd import lib
    from et_amd.encoder import Encoder_tile
    if lib().et_device_cu_count() != 256:
        pytest.skip("the line is one unit per compute unit of 256")
    r = rng(1700 + d + S)
    lins, ln = make_layer(r, d, dff, 0.8, seed=1800 + S, std=0.03, bias_std=0.05)
    work = workspace(Encoder_tile, d, S, H, B).fill_(7.0)
    enc = Encoder_tile(d, S, H, work, *build_linears(lins, B * S), *ln, None, B)
    x = randn_h(r, (B * S, d))
    got = host(enc.run(torch.empty_like(dev(x)), dev(x)))
    assert (host(work) == 7.0).all() == one_launch
    check_close(got, orc.encoder_tile_layer(x, lins, ln, None, S, H, B, None, 1.0), what="layer by its units")


@pytest.mark.parametrize("d,S,B,sp,lens,use_mask,ls", [
    (64, 1, 1, 0.5, None, False, 1.0),                      # one row, one head
    (768, 16, 3, 0.8, None, True, 1.0),                     # whole panels; mask rows of whole loads
    (768, 37, 2, 0.8, [37, 5], True, LOG2E),                # odd panels and mask rows; padding rows
    (768, 64, 9, 0.8, None, False, 1.0),                    # the sequences of an XCD in turn, one of them over
    (512, 65, 2, 0.5, [65, 0], False, LOG2E),               # one row in the last panel; an empty sequence
    (768, 128, 2, 0.8, [128, 97], True, 1.0),               # the most rows: five panels of eight in the ring
    (1024, 113, 3, 0.9, [96, 113, 48], False, LOG2E),       # three panels in the ring, refilled
    (320, 50, 2, 0.0, None, True, 1.0),                     # dense lists of ten pairs
])
def test_projections_and_attention_of_a_head_in_one_launch(d, S, B, sp, lens, use_mask, ls):
    """et_qkv_attention on a padded batch, with lengths and packed, against the oracle's linears and attention"""
    import ctypes as C
    from et_amd import lib
    from et_amd._lib import check
    r = rng(2100 + d + S + B)
    H = d // 64
    lins = [make_tile_linear(r, d, d, sp, seed=2200 + S + j, std=0.04, bias_std=0.05) for j in range(3)]
    x = randn_h(r, (B * S, d))
    mask = randn_h(r, (S, S), 0.5) if use_mask else None
    q, k, v = (orc.tile_linear(x, l["row_ptr"], l["row_offset"], l["data"], l["bias"], d) for l in lins)
    L = lib()
    plans = []
    try:
        for l in lins:
            plans.append(C.c_void_p())
            check(L.et_tile_plan_create(C.byref(plans[-1]), d, d, l["row_offset"].size, l["data"].ctypes.data,
                                        l["row_ptr"].ctypes.data, l["row_offset"].ctypes.data, l["bias"].ctypes.data))
        md = dev(mask) if use_mask else None
        mp = md.data_ptr() if use_mask else None
        for n in ([None, np.array(lens, np.int32)] if lens else [None]):
            want = orc.otf_attention(q, k, v, mask, S, H, B, n, ls)
            nd = None if n is None else dev(n)
            out = torch.full((B * S, d), 9.0, dtype=torch.float16, device="cuda")
            check(L.et_qkv_attention(out.data_ptr(), dev(x).data_ptr(), *plans, mp, None if n is None else nd.data_ptr(), None,
                                     S, S, d, H, B, ls, torch.cuda.current_stream().cuda_stream))
            got = host(out)
            valid = np.concatenate([np.arange(b * S, b * S + (S if n is None else n[b])) for b in range(B)])
            check_close(got[valid], want[valid], max_abs=5e-3, mean_rel=1e-3, what="projections and attention")
            assert (np.delete(got, valid, 0) == 0).all()
            if n is not None:
                cu = dev(np.concatenate([[0], np.cumsum(n)]).astype(np.int32))
                xp = dev(x[valid])
                out = torch.full_like(xp, 9.0)
                check(L.et_qkv_attention(out.data_ptr(), xp.data_ptr(), *plans, mp, None, cu.data_ptr(), int(n.max()), S, d, H,
                                         B, ls, torch.cuda.current_stream().cuda_stream))
                assert np.array_equal(host(out), got[valid])
    finally:
        for p in plans:
            L.et_tile_plan_destroy(p)


def test_projections_and_attention_refuse_what_they_do_not_take():
    import ctypes as C
    from et_amd import lib
    from et_amd._lib import check
    L, r = lib(), rng(2300)
    mats = {n: make_tile_linear(r, n, n, 0.5, seed=n) for n in (128, 1536)}
    mats["dense"] = make_tile_linear(r, 768, 768, 0.0, seed=3)  # lists beyond a wave's registers
    plans = {}
    try:
        for n, l in mats.items():
            plans[n] = C.c_void_p()
            check(L.et_tile_plan_create(C.byref(plans[n]), l["K"], l["N"], l["row_offset"].size, l["data"].ctypes.data,
                                        l["row_ptr"].ctypes.data, l["row_offset"].ctypes.data, l["bias"].ctypes.data))
        x = torch.zeros((129, 1536), dtype=torch.float16, device="cuda")

        def run(name, d, H, most, S, cu=None):
            p = plans[name]
            return L.et_qkv_attention(x.data_ptr(), x.data_ptr(), p, p, p, None, None, cu, most, S, d, H, 1, 1.0, None)
        for args in ((128, 128, 4, 32, 32), (128, 128, 2, 129, 129), (1536, 1536, 24, 32, 32), ("dense", 768, 12, 32, 32),
                     (128, 128, 2, 16, 32), (128, 128, 2, 0, 0)):
            assert run(*args) < 0, args
    finally:
        for p in plans.values():
            L.et_tile_plan_destroy(p)


@pytest.mark.parametrize("S,B,off", [(32, 2, 8), (16, 3, 24), (48, 2, 56), (37, 2, 64)])
def test_layer_in_one_launch_workspace_alignment(S, B, off):
    """a workspace `off` halves behind a 256-byte boundary, several sequences that end on a panel: the rows handed over
    inside the launch lie in lines of their own, not in the workspace, which stays as it was"""
    from et_amd import lib
    from et_amd.encoder import Encoder_length
    r = rng(1500 + S + off)
    d, H, dff = 256, 4, 1024
    lins, ln = make_layer(r, d, dff, 0.5, seed=1600 + S, std=0.03, bias_std=0.05)
    x = randn_h(r, (B * S, d))
    whole = torch.full((Encoder_length.buffer_size(d, S, H, B) // 2 + 128,), 7.0, dtype=torch.float16, device="cuda")
    assert whole.data_ptr() % 256 == 0
    enc = Encoder_length(d, S, H, whole[off:], *build_linears(lins, B * S), *ln, None, B)
    want = orc.encoder_tile_layer(x, lins, ln, None, S, H, B, None, 1.0)
    first = host(enc.run(torch.empty_like(dev(x)), dev(x)))
    check_close(first, want, what=f"layer in one launch, workspace at +{2 * off} bytes")
    for _ in range(20):
        assert np.array_equal(host(enc.run(torch.empty_like(dev(x)), dev(x))), first)
    assert (host(whole) == 7.0).all()
    try:
        lib().et_tuning_set(b"layer_flow_rows", 0)
        steps = host(enc.run(torch.empty_like(dev(x)), dev(x)))
    finally:
        lib().et_tuning_set(b"layer_flow_rows", -1)
    check_close(steps, want, what="separate launches")
    assert (host(whole) != 7.0).any()


@pytest.mark.parametrize("S,B,lens", [(37, 1, None), (48, 2, None), (24, 4, [24, 3, 17, 9])])
def test_layer_in_one_launch_after_a_wait_that_gave_up(S, B, lens):
    """waits that give up at once (poll limit 0): the launch ends, the next call reports it once, and every run from then
    on is right, eager and replayed - also after two such launches in a row"""
    from et_amd import EtError, lib
    from et_amd.encoder import Encoder_length
    r = rng(1700 + S)
    d, H, dff = 768, 12, 3072
    lins, ln = make_layer(r, d, dff, 0.8, seed=1800 + S, std=0.03, bias_std=0.05)
    x = dev(randn_h(r, (B * S, d)))
    enc = Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, None, B)
    enc.set_seq_lens(None if lens is None else np.array(lens, np.int32))
    run = lambda: host(enc.run(torch.empty_like(x), x))
    good = run()
    out = torch.empty_like(x)
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        enc.run(out, x)
    try:
        for launches in (1, 2, 1):
            lib().et_tuning_set(b"tile_wait_spin", 0)
            for _ in range(launches):
                print("zero-poll launch", flush=True)
                run()
                if lib().et_wait_status_take() == 0:
                    pytest.skip("no wait was ever in vain")
            lib().et_wait_status_raise_for_test()
            lib().et_tuning_set(b"tile_wait_spin", -1)
            with pytest.raises(EtError) as e:
                run()
            assert "gave up a bounded wait" in str(e.value)
            for _ in range(5):
                assert np.array_equal(run(), good)
                out.zero_()
                graph.replay()
                assert np.array_equal(host(out), good)
            assert lib().et_wait_status_take() == 0
    finally:
        lib().et_tuning_set(b"tile_wait_spin", -1)
        lib().et_wait_status_take()
    del graph


@pytest.mark.parametrize("sp", [0.5, 0.85])
def test_layer_in_one_launch_infinite_activation_without_a_tile(sp):
    """an infinite activation in a tile column that Q, K and V have no tile in stays with its own row (the skip
    connection): the other rows are what they are with a finite one"""
    from et_amd.encoder import Encoder_length
    r = rng(2000)
    d, H, dff, S, B = 768, 12, 3072, 24, 2
    lins, ln = make_layer(r, d, dff, sp, seed=2100, std=0.03, bias_std=0.05)
    for l in lins[:3]:
        keep = l["row_offset"] != 0
        rows = np.repeat(np.arange(d // 16), np.diff(l["row_ptr"]))[keep]
        l["row_ptr"] = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=d // 16))]).astype(np.int32)
        l["data"] = l["data"].reshape(-1, 256)[keep].copy()
        l["row_offset"] = l["row_offset"][keep].copy()
    x = randn_h(r, (B * S, d))
    xi = x.copy()
    xi[5, 3] = np.inf
    enc = Encoder_length(d, S, H, workspace(Encoder_length, d, S, H, B), *build_linears(lins, B * S), *ln, None, B)
    fin, inf = (host(enc.run(torch.empty_like(dev(v)), dev(v))) for v in (x, xi))
    check_close(fin, orc.encoder_tile_layer(x, lins, ln, None, S, H, B, None, 1.0), what="finite")
    others = np.arange(B * S) != 5
    assert np.array_equal(inf[others], fin[others]) and not np.isfinite(inf[5]).any()


def test_layer_flow_refuses_what_it_has_no_room_for():
    """row offsets beyond the object's capacity, and a packed run without any, are errors in front of the launch"""
    import ctypes as C
    from et_amd import lib
    from et_amd._lib import EtError, check
    L, d, H, dff, S, B = lib(), 64, 2, 128, 10, 3
    lins, ln = make_layer(rng(2200), d, dff, 0.5, seed=2300)
    p = lambda a: np.ascontiguousarray(a).ctypes.data_as(C.c_void_p)
    ip = lambda a: np.ascontiguousarray(a, np.int32).ctypes.data_as(C.POINTER(C.c_int))
    plans = []
    flow = C.c_void_p()
    try:
        for l in lins:
            plans.append(C.c_void_p())
            check(L.et_tile_plan_create(C.byref(plans[-1]), l["K"], l["N"], l["row_offset"].size, p(l["data"]), ip(l["row_ptr"]),
                                        ip(l["row_offset"]), p(l["bias"])))
        check(L.et_layer_flow_create(C.byref(flow), *plans, S, H, B))
        assert flow.value
        x = dev(np.zeros((7, B * S, d), np.float16))
        vec = dev(np.ones(d, np.float16))
        cu = dev(np.array([0, 10, 12, 30], np.int32))
        ptr = lambda t: C.c_void_p(t.data_ptr())
        cup = C.cast(cu.data_ptr(), C.POINTER(C.c_int))
        run = lambda: check(L.et_layer_flow_run(flow, *[ptr(x[i]) for i in range(6)], None, None, cup, *[ptr(vec)] * 4, 1.0, None))
        with pytest.raises(EtError):
            run()
        for bad in ([0, 10, 20, 31], [0, 11, 12, 13], [1, 2, 3, 4], [0, 5, 4, 9]):
            with pytest.raises(EtError):
                check(L.et_layer_flow_set_packed(flow, ip(bad)))
            with pytest.raises(EtError):
                run()
        check(L.et_layer_flow_set_packed(flow, ip([0, 10, 12, 22])))
    finally:
        L.et_layer_flow_destroy(flow)
        for q in plans:
            L.et_tile_plan_destroy(q)
