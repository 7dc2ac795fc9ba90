"""The launches of small layers at the edges of their forms: the gate|up of
q4r rows of at least 32 blocks with two lanes on each of a row's chains (six
rounds of eight blocks at once) while pairs share no weights, the GEMV and down
launches that load a row of up to 32 blocks before the activations, the combine
over a pair list in rounds of 256 pairs, and the dot4 layer with a workgroup
row per pair (fewer pairs than experts)."""
import numpy as np
import pytest
import torch

import ft_hip
import test_gpu_grouped_tiles as tiles
import test_gpu_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hidden", [32, 160, 256, 992, 1024, 1056, 1504, 1536, 1568, 2816, 3104])
def test_gate_up_two_lanes_per_chain_same_bits(gemv, orc, hidden):
    """q4_0 rows have one lane per chain: the same chains in the same order, so
    the act blocks of the two layouts are the same bytes."""
    inter, n_exp, n = 64, 3, 4
    x = np.random.default_rng(hidden).standard_normal((2, hidden)).astype(np.float32)
    q8 = ops.dev(np.concatenate([ops.q8_from_oracle(orc, r) for r in x]))
    slots = ops.dev(np.array([2, 0, 1, 2], np.int32))
    got = []
    for layout in (ft_hip.LAYOUT_Q4_0, ft_hip.LAYOUT_Q4R):
        bank = ops.make_bank(orc, n_exp, 2 * inter, hidden, hidden, layout)
        out = torch.zeros(n * (inter // 32) * 40, dtype=torch.uint8, device=DEV)
        gemv.gemv_gate_up_act(ops.dev(bank.ravel()), bank.shape[1], slots, n, 2, q8, hidden, inter, out, layout=layout)
        got.append(ops.host(out))
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("layout", [ft_hip.LAYOUT_Q4_0, ft_hip.LAYOUT_Q4R])
@pytest.mark.parametrize("k,n_rows", [(64, 1), (992, 33), (1024, 31), (1056, 33), (256, 33), (288, 33), (512, 33),
                                      (544, 33), (768, 33), (800, 33), (1280, 33), (1312, 33), (1792, 33), (1824, 33)])
def test_gemv_rows_of_about_32_blocks(gemv, orc, layout, k, n_rows):
    ops.test_block_dots_and_gemv(gemv, orc, layout, k, n_rows)


@pytest.mark.parametrize("layout", [ft_hip.LAYOUT_Q4_0, ft_hip.LAYOUT_Q4R])
@pytest.mark.parametrize("top_k,hidden,inter", [(2, 128, 32), (4, 640, 992), (2, 256, 1024), (2, 256, 1056)])
def test_layer_down_rows_of_about_32_blocks(gemv, orc, layout, top_k, hidden, inter):
    ops.test_moe_layer_small_shapes(gemv, orc, layout, top_k, 24, hidden, inter)


@pytest.mark.parametrize("n_pairs,n_seqs,hidden", [(1, 2, 32), (9, 1, 300), (255, 3, 257), (256, 2, 256), (257, 1, 64),
                                                   (700, 5, 512)])
def test_reduce_pairs_rounds_bit_exact(gemv, orc, n_pairs, n_seqs, hidden):
    """Pair lists that end inside, at and past a round, in any order, the last
    sequence without a pair."""
    rng = np.random.default_rng(n_pairs)
    y = rng.standard_normal((n_pairs, hidden)).astype(np.float32)
    w = rng.random(n_pairs).astype(np.float32)
    seq_of = rng.integers(0, max(1, n_seqs - 1), n_pairs).astype(np.int32)
    out0 = rng.standard_normal((n_seqs, hidden)).astype(np.float32)
    out = ops.dev(out0)
    gemv.reduce_pairs_weighted(ops.dev(y), ops.dev(w), ops.dev(seq_of), out, hidden, n_pairs, n_seqs)
    out = ops.host(out)
    for s in range(n_seqs):
        ps = np.nonzero(seq_of == s)[0]
        exp = orc.combine(y[ps], w[ps], out0[s]) if len(ps) else out0[s]
        assert np.array_equal(out[s].view(np.uint32), exp.view(np.uint32)), s


@pytest.mark.parametrize("counts", [[0] * 60 + [17, 2, 1, 0],      # experts of several pairs: the first takes them
                                    [1] * 63 + [0],                # one pair fewer than experts
                                    [0] * 32 + [2] * 32])          # as many: a workgroup row per expert
@pytest.mark.parametrize("hidden", [2816, 4096])
def test_dot4_row_per_pair_matches_tiles(gemv, hidden, counts):
    tiles.test_token_tiles_match_dot4(gemv, hidden, 96, counts, True)


@pytest.mark.parametrize("layout", [ft_hip.LAYOUT_Q4_0, ft_hip.LAYOUT_Q4R])
@pytest.mark.parametrize("hidden,inter,n_experts,top_k,n", [(1024, 512, 8, 4, 16),   # many pairs per expert
                                                            (2816, 704, 24, 8, 3),
                                                            (3072, 768, 40, 4, 5),
                                                            (2048, 8192, 8, 2, 6)])      # long rows, read more than once
def test_layer_of_many_tokens_same_bits_as_one_by_one(gemv, layout, hidden, inter, n_experts, top_k, n):
    """A layer's forms go by the pairs and workgroups of the call: each token of
    a batch has the bits of a call of its own."""
    m = ops.moe_synth.SyntheticMoE(gemv, ops.moe_synth.Shape("small", hidden, inter, n_experts, top_k, 1, 9), n_layers=1,
                                   layout=layout)
    x = torch.stack([m.hidden(t) for t in range(n)])

    def layer(part):
        b = len(part)
        ids = torch.zeros(b * top_k, dtype=torch.int32, device=DEV)
        wts = torch.zeros(b * top_k, dtype=torch.float32, device=DEV)
        out = torch.zeros_like(part)
        m.layer(0, part, out, ids, wts, m.workspace(b), n_seqs=b)
        return ops.host(out).view(np.uint32), ops.host(ids), ops.host(wts)

    out, ids, wts = layer(x)
    for t in range(n):
        o, i, w = layer(x[t:t + 1].contiguous())
        assert np.array_equal(o[0], out[t])
        assert np.array_equal(i, ids[t * top_k:(t + 1) * top_k]) and np.array_equal(w, wts[t * top_k:(t + 1) * top_k])
