"""The matrix-core kernels of the grouped layer on inputs at the ends of f32:
subnormal products of scales, infinities, NaN, values that overflow, rows of
zeros and equal logits. The references are the dot4 kernels and, for the
routing of over 64 seqs, calls of fewer; NaN results compare as NaN."""
import numpy as np
import pytest
import torch

import ft_hip
import moe_synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def same(a, b):
    """The same bits, any NaN equal to any other."""
    na, nb = np.isnan(a), np.isnan(b)
    return np.array_equal(na, nb) and np.array_equal(a.view(np.uint32)[~na], b.view(np.uint32)[~nb])


def bank_of(gemv, hidden, inter, E):
    gu_b, _, eb = moe_synth.expert_geometry(moe_synth.Shape("t", hidden, inter, E, 1, 1, 81), ft_hip.LAYOUT_Q4R)
    src = torch.empty(E * eb, dtype=torch.uint8, device=DEV)
    for e in range(E):
        gemv.gen_q4_rows(9000 + e, 0, 2 * inter, hidden, moe_synth.gen_scale(0.02), src[e * eb:e * eb + gu_b])
        gemv.gen_q4_rows(9500 + e, 0, hidden, inter, moe_synth.gen_scale(0.02), src[e * eb + gu_b:(e + 1) * eb])
    bank = torch.empty(E * gemv.fused_expert_bytes(hidden, inter), dtype=torch.uint8, device=DEV)
    gemv.pack_experts_fused(src, ft_hip.LAYOUT_Q4R, eb, bank, E, hidden, inter)
    return bank


def layer(gemv, x, w, bias, bank, inter, E, K, record=True):
    B, hidden = x.shape
    ws = torch.empty(gemv.moe_layer_grouped_workspace_bytes(B, hidden, inter, E, K), dtype=torch.uint8, device=DEV)
    out = torch.zeros_like(x)
    ids = torch.zeros(B * K, dtype=torch.int32, device=DEV)
    wts = torch.zeros(B * K, dtype=torch.float32, device=DEV)
    gu = torch.zeros((B * K, 2 * inter), dtype=torch.float32, device=DEV) if record else None
    act = torch.zeros((B * K, inter // 32, 40), dtype=torch.uint8, device=DEV) if record else None
    gemv.moe_layer_grouped(x, out, B, hidden, inter, E, K, w, bias, None, bank, ids, wts, ws, gu, act)
    torch.cuda.synchronize()
    return [None if t is None else t.cpu().numpy() for t in (out, ids, wts, gu, act)]


def tokens(kind, B, hidden, rng):
    x = rng.standard_normal((B, hidden)).astype(np.float32)
    x[:, 32:64] = 0.0  # a block whose output is the experts' sum alone
    if kind == "products below 2^-126":      # d4 * d8 of the gate|up rows
        x *= np.float32(1e-34)
    elif kind == "act products below 2^-126":  # of the down rows: act values of about 1e-34
        x *= np.float32(1e-17)
    elif kind == "subnormal":
        x *= np.float32(1e-39)
    elif kind == "special":
        x[0, 100], x[1, 5], x[2, 2000] = np.inf, -np.inf, np.nan
        x[3] = np.clip(x[3], -3, 3) * np.float32(1e38)   # the gate|up sums overflow, then GELU * up
        x[4] = 0.0
        x[5] = -0.0
        x[6, 700] = np.float32(3e38)
        x[7] *= np.float32(1e19)   # act values overflow
    return x


# (31 act blocks: an act block per wave; 3: a slice per wave)
@pytest.mark.parametrize("hidden,inter,E,B", [(2816, 96, 8, 20), (2816, 992, 40, 64), (4096, 96, 8, 20), (4096, 992, 60, 64)])
@pytest.mark.parametrize("kind", ["products below 2^-126", "act products below 2^-126", "subnormal", "special"])
def test_token_tiles_at_the_ends_of_f32(gemv, hidden, inter, E, B, kind):
    bank = bank_of(gemv, hidden, inter, E)
    rng = np.random.default_rng(hidden + inter)
    x = torch.from_numpy(tokens(kind, B, hidden, rng)).to(DEV)
    w = torch.zeros((E, hidden), dtype=torch.float32, device=DEV)
    bias = torch.from_numpy(rng.standard_normal(E).astype(np.float32)).to(DEV)  # with w = 0, the same experts for all
    K = 2
    got = {}
    try:
        for name, m in (("mfma", 1), ("dot4", 10**6)):
            gemv.set_grouped_mfma_min(m)
            got[name] = layer(gemv, x, w, bias, bank, inter, E, K)
    finally:
        gemv.set_grouped_mfma_min(0)
    a, b = got["mfma"], got["dot4"]
    assert np.array_equal(a[1], b[1]) and same(a[2], b[2])
    assert same(a[3], b[3]), "gate|up sums"
    if kind.startswith("products"):
        assert np.any(a[3] != 0)
    assert same(a[4][..., :4].copy().view(np.float32), b[4][..., :4].copy().view(np.float32)), "act d"
    assert np.array_equal(a[4][..., 4:], b[4][..., 4:]), "act quants"
    assert np.array_equal(np.isnan(a[0]), np.isnan(b[0]))


@pytest.mark.parametrize("hidden,inter,E,K,B", [(2816, 96, 20, 1, 64), (4096, 992, 40, 4, 24)])
@pytest.mark.parametrize("kind", ["act products below 2^-126", "special"])
def test_down_sums_at_the_ends_of_f32(gemv, hidden, inter, E, K, B, kind):
    """Where the automatic choice keeps the dot4 kernels' down order, also here."""
    bank = bank_of(gemv, hidden, inter, E)
    rng = np.random.default_rng(hidden + inter + 1)
    x = torch.from_numpy(tokens(kind, B, hidden, rng)).to(DEV)
    w = torch.zeros((E, hidden), dtype=torch.float32, device=DEV)
    bias = torch.from_numpy(rng.standard_normal(E).astype(np.float32)).to(DEV)
    got = []
    try:
        for m in (0, 10**6):
            gemv.set_grouped_mfma_min(m)
            got.append(layer(gemv, x, w, bias, bank, inter, E, K, record=False)[0])
    finally:
        gemv.set_grouped_mfma_min(0)
    assert same(got[0], got[1])
    if kind.startswith("act"):
        assert np.any(got[0][:, 32:64] != 0) and np.all(np.abs(got[0][:, 32:64]) < 1e-30)


@pytest.mark.parametrize("hidden,E,K", [(2816, 128, 8), (4096, 32, 4)])
@pytest.mark.parametrize("kind", ["subnormal", "special", "equal logits"])
@pytest.mark.parametrize("norm", [False, True])
def test_routing_of_many_seqs_at_the_ends_of_f32(gemv, hidden, E, K, kind, norm):
    B, inter = 70, 32
    bank = bank_of(gemv, hidden, inter, E)
    rng = np.random.default_rng(hidden + E)
    x = torch.from_numpy(tokens(kind, B, hidden, rng)).to(DEV)
    W = (rng.standard_normal((E, hidden)) * 0.02).astype(np.float32)
    if kind == "equal logits":
        W[:] = W[0]
    elif kind == "special":
        W[3, 9], W[5] = np.inf, 0.0
    w = torch.from_numpy(W).to(DEV)
    try:
        gemv.set_input_norm(norm)
        ids, wts = layer(gemv, x, w, None, bank, inter, E, K, record=False)[1:3]
        ids, wts = ids.reshape(B, K), wts.reshape(B, K)
        for t0 in range(0, B, 35):
            i, v = layer(gemv, x[t0:t0 + 35].contiguous(), w, None, bank, inter, E, K, record=False)[1:3]
            assert np.array_equal(i.reshape(-1, K), ids[t0:t0 + 35])
            assert same(v.reshape(-1, K), wts[t0:t0 + 35])
        if kind == "equal logits":
            assert np.array_equal(ids, np.tile(np.arange(K), (B, 1)))
    finally:
        gemv.set_input_norm(0)
