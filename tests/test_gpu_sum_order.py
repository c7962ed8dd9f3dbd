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
