"""The order in which the DiT path's input layers take their sums.

A sum's order decides its last bits, which the fp16 layers behind it carry on, so it is one and the
same for every launch form: one chain of fp32 additions over the convolutions' taps in order.
"""

from __future__ import annotations

import pytest
import torch

from tests.gpu_helpers import make_estimator, random_packed, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("rows", [45, 300, 700, 1100], ids=str)
def test_position_conv_sums_its_taps_in_one_chain(fcv, rows):
    """Tap 0 gives 2^25, where fp32 steps by 4; taps 16 to 30 give 1 each, a quarter per matrix
    instruction.  One chain drops every quarter; sums of later taps that start from zero keep them
    and add 16.  The bias takes 2^25 off again, so the rest shows in the second convolution (the
    identity on even channel groups) and in the LayerNorm of the result."""
    dims = fcv.synthetic.DiTDims(depth=1)
    sd = {n: torch.zeros(s) for n, s in fcv.synthetic.state_dict_shapes(dims)}
    pre = "input_embed."
    sd[pre + "proj.bias"] += 16.0
    w1 = sd[pre + "conv_pos_embed.conv1.0.weight"]   # [channel][input of the group][tap]
    w1[:, :, 0] = 2.0 ** 15
    w1[:, :, 16:] = 2.0 ** -10
    sd[pre + "conv_pos_embed.conv1.0.bias"] -= 2.0 ** 25
    cpg = w1.shape[1]
    w2 = sd[pre + "conv_pos_embed.conv2.0.weight"]
    for c in range(dims.dim):
        if c // cpg % 2 == 0:
            w2[c, c % cpg, -1] = 1.0
    sd["proj_out.weight"][:, :cpg] = 0.5
    sd["proj_out.bias"] += 3.0
    est = make_estimator(fcv, sd, depth=1)
    say(f"[conv chain] {rows}")
    x, mu, cond, spks, t = random_packed([rows], seed=5, t=0.4)
    v = est.forward_packed(x, mu, cond, spks, t, [rows]).cpu()
    full = v[w1.shape[2] - 1:]  # rows that every tap reaches
    assert torch.equal(full, torch.full_like(full, 3.0)), float((full - 3.0).abs().max())


def _one_chain_frontend(fcv, lookahead):
    """Front-end whose first convolution sums 2^25 (tap 0), then 3 from each later tap, less 2^25;
    the second is the identity on its last tap; every embedding is 1 in all 80 features."""
    dims = fcv.synthetic.FlowDims(vocab=4, channels=128, lookahead=lookahead)
    sd = {k: torch.zeros_like(v) for k, v in fcv.synthetic.random_flow_state_dict(dims).items()}
    sd["input_embedding.weight"] += 1.0
    w1 = sd["pre_lookahead_layer.conv1.weight"]
    w1[:, 0, 0] = 2.0 ** 25
    w1[:, :, 1:] = 3.0 / 80
    sd["pre_lookahead_layer.conv1.bias"] -= 2.0 ** 25
    sd["pre_lookahead_layer.conv2.weight"][:, :80, 2] = torch.eye(80)
    fe = fcv.FlowFrontEnd(vocab_size=4, channels=128, pre_lookahead_len=lookahead, device="cuda:0")
    fe.load_reference_state_dict(sd)
    fe.finalize_weights()
    return fe


@pytest.mark.parametrize("tokens", [50, 800])
@pytest.mark.parametrize("lookahead", [1, 3, 7])
def test_token_features_sum_their_taps_in_one_chain(fcv, lookahead, tokens):
    """2^25 steps by 4 in fp32, so one chain drops what the later taps add, some 0.15 at a time; a sum
    that starts from zero at a later tap keeps its 3."""
    fe = _one_chain_frontend(fcv, lookahead)
    say(f"[token feature chain] lookahead {lookahead}, {tokens} tokens")
    mu, _ = fe.token_features([[1] * tokens])
    assert torch.equal(mu.cpu(), torch.ones(2 * tokens, 80))


def test_speaker_projection_sums_in_one_chain(fcv):
    """64 equal elements of norm 8: 2^25 from the first product, 1 from each of the others, which one
    chain drops."""
    dims = fcv.synthetic.FlowDims(vocab=4, channels=128)
    sd = {k: torch.zeros_like(v) for k, v in fcv.synthetic.random_flow_state_dict(dims).items()}
    sd["spk_embed_affine_layer.weight"][:, 0] = 2.0 ** 28
    sd["spk_embed_affine_layer.weight"][:, 1:64] = 8.0
    sd["spk_embed_affine_layer.bias"] -= 2.0 ** 25
    fe = fcv.FlowFrontEnd(vocab_size=4, channels=128, device="cuda:0")
    fe.load_reference_state_dict(sd)
    fe.finalize_weights()
    x = torch.zeros(3, 192)
    x[:, :64] = 1.0
    say("[speaker chain]")
    assert torch.equal(fe.speaker(x).cpu(), torch.zeros(3, 80))
