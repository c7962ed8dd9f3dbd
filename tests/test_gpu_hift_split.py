"""The vocoder's split-f16 convolutions (two f16 halves per fp32 operand, hift_split.hip) against
the fp32 matrix-core convolutions, which a handle without packed weights runs: every tile, tap
window and document boundary, activations far outside the f16 range, and non-finite input.

Bound: an operand's halves hold 22 bits (2^-22 per product) and both kernels accumulate K <= 8192
terms in fp32, so one convolution differs by about 1e-6; the vocoder's waveform carries the
difference of some 80 convolutions (2e-5 measured on either side against 64 bits, so 1e-4, the bar
of the oracle comparison, with the two errors added).
"""

from __future__ import annotations

import pytest
import torch

from tests.gpu_helpers import rel_l2, say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _pair(fcv, monkeypatch, gain=1.0, dims=None):
    """(vocoder with split weights, vocoder on the fp32 kernels), the same seeded weights; `gain`
    scales conv_pre and the source convolutions, and with them every later activation, while the
    last convolution's gain undoes it."""
    dims = dims or fcv.synthetic.HiFTDims()
    sd = fcv.synthetic.random_hift_state_dict(dims, seed=91)
    g = ".parametrizations.weight.original0"
    for name in sd:
        if name.startswith("conv_pre") or name.startswith("source_downs"):
            sd[name] = sd[name] * (gain if not name.endswith("original1") else 1.0)
        if name.endswith("alpha"):
            sd[name] = sd[name] / gain
        if name.endswith("bias") and (name.startswith("ups") or "resblocks" in name):
            sd[name] = sd[name] * gain
    sd["conv_post" + g] = sd["conv_post" + g] / gain
    buf = fcv.synthetic.random_hift_buffers(dims, max_samples=480 * 140, seed=92)
    out = []
    for split in (True, False):
        v = fcv.HiFTVocoder(dims, device="cuda:0", buffers=buf)
        v.load_reference_state_dict(sd)
        if not split:
            monkeypatch.setattr(v._lib, "fcv_hift_packed_bytes", lambda h: 0)
        v.finalize_weights()
        assert (v._packed is not None) == split
        out.append(v)
    monkeypatch.undo()
    return out


# frames per request: single rows of a tile, documents shorter than a tap window, tile edges
# (8, 40 and 120 rows a frame in the three stages against 32- and 64-row tiles), many documents
@pytest.mark.parametrize("frames", [[1], [3, 1, 2, 1], [8, 9], [16, 40, 1, 33], [131], [2] * 70],
                         ids=lambda f: f"{len(f)}x{max(f)}")
@pytest.mark.parametrize("tile", ["32", "64"])
def test_split_matches_fp32(fcv, monkeypatch, frames, tile):
    split, fp32 = _pair(fcv, monkeypatch)
    g = torch.Generator().manual_seed(93)
    mels = [torch.randn(80, n, generator=g).cuda() for n in frames]
    say(f"[split] {frames} tile {tile}")
    monkeypatch.setenv("FCV_HIFT_TILE", tile)
    got = split.inference_batched(mels, graph=False)
    ref = fp32.inference_batched(mels, graph=False)
    err = rel_l2(torch.cat([a.reshape(-1) for a in got]), torch.cat([a.reshape(-1) for a in ref]))
    say(f"[split] rel_l2 {err:.2e}")
    assert err <= 1e-4


@pytest.mark.parametrize("gain", [2.0 ** 24, 2.0 ** -40], ids=["large", "small"])
def test_split_holds_the_fp32_range(fcv, monkeypatch, gain):
    """Activations of 10^7 and 10^-12, past what f16 holds: the operands' scales keep them."""
    split, fp32 = _pair(fcv, monkeypatch, gain)
    g = torch.Generator().manual_seed(94)
    mels = [torch.randn(80, n, generator=g).cuda() for n in (20, 7)]
    got, ref = split.inference_batched(mels), fp32.inference_batched(mels)
    for a, b in zip(got, ref):
        assert torch.isfinite(b).all() and float(b.std()) > 1e-4
        err = rel_l2(a, b)
        say(f"[split] gain {gain:.1e} rel_l2 {err:.2e}")
        assert err <= 1e-4


@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_frame_stays_causal(fcv, monkeypatch, value):
    """A non-finite Mel frame changes nothing before its convolutions' right context reaches it
    (4 frames), and nothing of the other documents, as on the fp32 kernels."""
    split, _ = _pair(fcv, monkeypatch)
    g = torch.Generator().manual_seed(95)
    mels = [torch.randn(80, n, generator=g).cuda() for n in (30, 12)]
    bad = [mels[0].clone(), mels[1]]
    bad[0][:, 20] = value
    ref, got = split.inference_batched(mels), split.inference_batched(bad)
    keep = (20 - 4 - 1) * 480
    assert torch.isfinite(ref[0]).all()
    assert torch.equal(got[0][:, :keep], ref[0][:, :keep])
    assert torch.equal(got[1], ref[1])


def test_concurrent_groups_repeat_bit_for_bit(fcv, monkeypatch):
    """Two request groups sharing the GPU: forty passes give the same bits (a window overwritten
    while another wave still reads it shows only under such load)."""
    split, _ = _pair(fcv, monkeypatch)
    g = torch.Generator().manual_seed(96)
    mels = [torch.randn(80, n, generator=g).cuda() for n in (139, 120, 131)]
    ref = split.inference_batched(mels)
    for _ in range(40):
        got = split.inference_batched(mels)
        assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.mark.parametrize("channels", [slice(0, 80), slice(7, 8)], ids=["frame", "channel"])
@pytest.mark.parametrize("loud", [1e6, 1e10, 1e20])
def test_loud_frame_costs_the_others_no_precision(fcv, monkeypatch, loud, channels):
    """One frame of large finite values: the audio before its right context reaches it (4 frames) is
    bit for bit what it is without that frame, and the audio past the convolutions' reach (some 20
    frames) matches the fp32 kernels as ever."""
    split, fp32 = _pair(fcv, monkeypatch)
    g = torch.Generator().manual_seed(97)
    mel = torch.randn(80, 90, generator=g).cuda()
    bad = mel.clone()
    bad[channels, 20] *= loud
    say(f"[split] one frame times {loud:.0e}")
    quiet, = split.inference_batched([mel])
    got, = split.inference_batched([bad])
    ref, = fp32.inference_batched([bad])
    before, after = (20 - 4 - 1) * 480, (20 + 35) * 480
    assert torch.equal(got[:, :before], quiet[:, :before])
    assert torch.isfinite(ref).all() and float(ref[:, after:].std()) > 1e-4
    for part in (slice(0, before), slice(after, None)):
        err = rel_l2(got[:, part], ref[:, part])
        say(f"[split] rel_l2 {err:.2e}")
        assert err <= 1e-4


def test_output_before_a_change_stays_bit_for_bit(fcv, monkeypatch):
    """A frame's audio depends on the frames its convolutions read, on none after them: what follows,
    and how long the request is, leaves it bit for bit (a session re-vocodes its prefix)."""
    split, _ = _pair(fcv, monkeypatch)
    g = torch.Generator().manual_seed(98)
    mel = torch.randn(80, 60, generator=g).cuda()
    other = mel.clone()
    other[:, 41:] *= 3.0
    say("[split] prefix")
    a, = split.inference_batched([mel])
    b, = split.inference_batched([other])
    c, = split.inference_batched([mel[:, :50]], [False])
    keep = (41 - 4 - 1) * 480
    assert torch.equal(a[:, :keep], b[:, :keep]) and torch.equal(a[:, :keep], c[:, :keep])


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("packed", [True, False], ids=["split", "fp32"])
def test_resblocks_one_by_one_give_the_same_bits(fcv, monkeypatch, packed, graph):
    """A workspace too small for a stage's resblocks to run together takes them one after another
    (running sum, then the mean in the last one's epilogue), as every capacity past the limit does:
    final and non-final documents, one of them of a single row, and replays of a captured call."""
    voc = _pair(fcv, monkeypatch)[0 if packed else 1]
    g = torch.Generator().manual_seed(99)
    mels = [torch.randn(80, n, generator=g).cuda() for n in (33, 1, 24, 70)]
    fin = [True, True, False, False]
    say(f"[split] resblocks one by one, packed {packed}, graph {graph}")
    run = lambda: voc.inference_batched(mels, fin, concurrency=1, graph=graph)
    ref = [run() for _ in range(3)][-1]
    need = voc._lib.fcv_hift_workspace_bytes_capacity
    monkeypatch.setattr(voc._lib, "fcv_hift_workspace_bytes_capacity",
                        lambda h, f, d: need(h, f, d) // 2)
    voc._lanes[0][1] = None
    for _ in range(3):
        got = run()
        assert all(torch.equal(a, b) for a, b in zip(got, ref))


def test_packed_weights_take_the_place_of_the_fp32_ones(fcv):
    """After the packing only the weights that some kernel reads in fp32 stay on the card."""
    dims = fcv.synthetic.HiFTDims()
    v = fcv.HiFTVocoder(dims, device="cuda:0",
                        buffers=fcv.synthetic.random_hift_buffers(dims, max_samples=4800, seed=92))
    v.load_reference_state_dict(fcv.synthetic.random_hift_state_dict(dims, seed=91))
    before = torch.cuda.memory_allocated()
    v.finalize_weights()
    held = torch.cuda.memory_allocated() - before
    packed = v._packed.numel()
    say(f"[split] {packed >> 20} MB packed, {held >> 20} MB held")
    assert len(v._keep) == 321 - 76
    assert held < 1.5 * packed
