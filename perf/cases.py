"""Performance cases of the Token2Wav path, through its public entry points.

A case is one call that a serving program makes: the flow front-end, one DiT block, one estimator
forward, a packed CFG solve, tokens to Mel, or the vocoder.  Request sizes are texts of
comma-separated frame (or token) counts, so a case is a dict of plain values.

The model shapes are the CosyVoice3 ones (``DiTDims``, ``FlowDims``, ``HiFTDims``).  Weights are
seeded and fixed (a program serves one model); inputs come from the case and the seed.  DiT
weights are fp16 values, the dtype the path serves them in; peaked attention (q/k deviation 0.06)
and raised gates make every block count, as trained weights do.
"""

from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

REPO = Path(__file__).resolve().parent.parent
PKG = "faster_cosyvoice_amd"
DEV = "cuda:0"
CFG_RATE = 0.7
CHUNK = 50      # frames of the chunk-causal mask
LOOKAHEAD = 3   # tokens of right context of a non-final streaming chunk
RATIO = 2       # Mel frames per speech token
NOISE_SECONDS = 300


def _fcv():
    if PKG not in sys.modules:
        d = REPO / "faster-cosyvoice_amd"
        spec = importlib.util.spec_from_file_location(PKG, d / "__init__.py",
                                                      submodule_search_locations=[str(d)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[PKG] = mod
        spec.loader.exec_module(mod)
    return sys.modules[PKG]


# ---- the cases ---------------------------------------------------------------------------------

RAGGED8 = "1291,992,816,531,477,205,157,123"  # 8 offline requests of 1.2 to 26 s of audio
SINGLE = "550"

# 32 sessions of a packed streaming step: a prompt and prefix of 150-400 frames plus a hop
STREAM32 = ("362,339,348,277,217,186,378,201,354,431,258,297,307,329,461,311,"
            "306,247,442,280,324,391,268,215,479,233,337,404,292,366,415,250")

# 64 offline requests, log-normal around 800 frames (16 s), clipped to [64, 3000]
LOGNORMAL64 = ("863,739,1177,851,580,994,1741,1413,524,375,551,821,203,701,381,516,"
               "577,663,1023,1496,739,1818,535,986,1387,853,1193,1397,539,1833,327,654,"
               "598,910,1029,1130,426,696,2046,3000,419,1031,272,1127,759,908,660,1290,"
               "1157,851,1049,1093,462,698,652,64,641,1271,1667,903,555,340,2417,880")


def listed() -> list[dict]:
    return [
        # a session's first streaming chunk: prompt tokens + hop + lookahead into mu/cond/spks
        dict(name="frontend_first_chunk", op="frontend", lengths="93", final=False),
        # the front-end of an offline batch
        dict(name="frontend_batch8", op="frontend", lengths="646,496,408,265,239,103,79,62",
             final=True),
        # one DiT block (with its input and output layers) at the smallest offline request
        dict(name="block_300", op="forward", depth=1, lengths="300", cfg=False,
             streaming=False, padded=False),
        # one DiT block over a packed streaming step, chunk-causal mask
        dict(name="block_stream32", op="forward", depth=1, lengths=STREAM32, cfg=True,
             streaming=True, padded=False),
        # one estimator call for one request: the latency of a step
        dict(name="forward_single550", op="forward", depth=22, lengths=SINGLE, cfg=True,
             streaming=False, padded=False),
        # the padded drop-in estimator call on an offline batch
        dict(name="forward_padded8", op="forward", depth=22, lengths=RAGGED8, cfg=True,
             streaming=False, padded=True),
        # one estimator call on a full server's batch: the largest packed layout
        dict(name="forward_lognormal64", op="forward", depth=22, lengths=LOGNORMAL64, cfg=True,
             streaming=False, padded=False),
        # tokens to Mel of one session's streaming chunk (time to first audio)
        dict(name="flow_stream_chunk", op="flow", lengths="93", streaming=True),
        # the 10-step CFG solve of an offline batch, the headline workload
        dict(name="solve_ragged8", op="solve", lengths=RAGGED8, streaming=False),
        # the 10-step chunk-causal solve of 32 packed sessions
        dict(name="solve_stream32", op="solve", lengths=STREAM32, streaming=True),
        # vocoding one session's streaming chunk
        dict(name="vocoder_chunk68", op="vocoder", lengths="68", final=False, source=False),
        # vocoding an offline batch
        dict(name="vocoder_batch8", op="vocoder", lengths="903,680,512,398,286,119,94,73",
             final=True, source=False),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, most: int, lo: int, hi: int, total: int) -> str:
    """Up to ``most`` sizes in [lo, hi], their sum at most ``total``; batches of like and of
    unlike requests both occur."""
    n = _log_int(rng, 1, most)
    top = max(lo, min(hi, total // n))
    a = _log_int(rng, lo, top)
    b = _log_int(rng, a, top)
    return ",".join(str(rng.randint(a, b)) for _ in range(n))


def draw(rng) -> dict:
    op = rng.choice(("frontend", "forward", "forward", "flow", "solve", "vocoder", "vocoder"))
    if op == "frontend":
        return dict(op=op, lengths=_sizes(rng, 32, 8, 1500, 8000), final=rng.random() < 0.5)
    if op == "forward":
        depth = rng.choice((1, 22))
        cfg = depth == 22 or rng.random() < 0.5
        return dict(op=op, depth=depth, cfg=cfg, streaming=rng.random() < 0.5,
                    lengths=_sizes(rng, 64, 40, 3000, 50000), padded=rng.random() < 0.3)
    if op == "flow":
        return dict(op=op, lengths=_sizes(rng, 16, 20, 700, 2500), streaming=rng.random() < 0.6)
    if op == "solve":
        return dict(op=op, lengths=_sizes(rng, 32, 60, 1500, 8000), streaming=rng.random() < 0.5)
    return dict(op=op, lengths=_sizes(rng, 16, 24, 1500, 6000), final=rng.random() < 0.5,
                source=rng.random() < 0.3)


def _lengths(case) -> list[int]:
    return [int(v) for v in case["lengths"].split(",")]


# ---- seeded weights ----------------------------------------------------------------------------

_CACHE: dict = {}


def _once(key, make):
    if key not in _CACHE:
        _CACHE[key] = make()
    return _CACHE[key]


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device=DEV) * std


def _dit_weights(depth: int) -> dict[str, torch.Tensor]:
    """DiT state dict on the GPU: fp32 tensors that hold fp16 values."""
    def make():
        g, out = _gen(100 + depth), {}
        for name, shape in _fcv().synthetic.state_dict_shapes(
                _fcv().synthetic.DiTDims(depth=depth)):
            std = 0.06 if name.endswith(("to_q.weight", "to_k.weight")) else 0.02
            w = _randn(g, *shape, std=std)
            if name.startswith("transformer_blocks") and name.endswith("attn_norm.linear.bias"):
                w.view(6, -1)[[2, 5]] += 0.2
            out[name] = w.half().float()
        return out
    return _once(("dit_w", depth), make)


def _flow_weights() -> dict[str, torch.Tensor]:
    def make():
        g, out = _gen(7), {}
        fan = {"input_embedding": 1, "spk_embed_affine_layer": 192,
               "pre_lookahead_layer.conv1": 320, "pre_lookahead_layer.conv2": 3072}
        for name, shape in _fcv().synthetic.flow_state_dict_shapes():
            out[name] = _randn(g, *shape, std=fan[name.rsplit(".", 1)[0]] ** -0.5)
        return out
    return _once("flow_w", make)


def _hift_dims():
    return _fcv().synthetic.HiFTDims()


def _hift_weights() -> dict[str, torch.Tensor]:
    """Vocoder state dict with O(1) activations; F0 around 150 Hz, partly unvoiced."""
    def make():
        g, out = _gen(11), {}
        for name, shape in _fcv().synthetic.hift_state_dict_shapes(_hift_dims()):
            if name.endswith("original0"):
                w = 1.0 + _randn(g, *shape, std=0.1)
                if name.startswith("conv_post"):
                    w *= 0.3
            elif name.endswith("alpha"):
                w = 0.5 + torch.rand(*shape, generator=g, device=DEV)
            elif name.endswith("original1"):
                w = _randn(g, *shape)
            elif name.startswith("source_downs") and name.endswith("weight"):
                w = _randn(g, *shape, std=(shape[1] * shape[2]) ** -0.5)
            else:
                w = _randn(g, *shape, std=0.1)
            out[name] = w
        out["f0_predictor.classifier.weight"] *= 400.0
        out["f0_predictor.classifier.bias"].fill_(150.0)
        return out
    return _once("hift_w", make)


def _hift_buffers() -> dict[str, torch.Tensor]:
    def make():
        g, H = _gen(13), _hift_dims().nb_harmonics + 1
        rand_ini = torch.rand(1, H, generator=g, device=DEV)
        rand_ini[:, 0] = 0
        return {"rand_ini": rand_ini,
                "sine_waves": torch.rand(1, NOISE_SECONDS * 24000, H, generator=g, device=DEV)}
    return _once("hift_b", make)


def _rand_noise() -> torch.Tensor:
    """The decoder's fixed noise prefix, on the host as the program's model holds it."""
    return _once("noise", lambda: _randn(_gen(17), 1, 80, 50 * NOISE_SECONDS).cpu())


# ---- the program's models ----------------------------------------------------------------------


def _estimator(depth: int):
    return _once(("est", depth), lambda: _fcv().DiTEstimator.from_state_dict(
        dict(_dit_weights(depth)), device=DEV, depth=depth, static_chunk_size=CHUNK))


def _flow():
    def make():
        fe = _fcv().FlowFrontEnd(device=DEV)
        fe.load_reference_state_dict(_flow_weights())
        fe.finalize_weights()
        return fe
    return _once("flow", make)


def _vocoder():
    def make():
        voc = _fcv().HiFTVocoder(_hift_dims(), device=DEV, buffers=_hift_buffers())
        voc.load_reference_state_dict(_hift_weights())
        voc.finalize_weights()
        return voc
    return _once("voc", make)


# ---- inputs ------------------------------------------------------------------------------------


def _prompt_frames(mel: int) -> int:
    return int(0.35 * mel)


def _inputs(case: dict, seed: int) -> dict:
    """The case's inputs on the GPU, from the case and the seed alone."""
    g, op, lengths = _gen(seed), case["op"], _lengths(case)
    if op in ("frontend", "flow"):
        final = case["final"] if op == "frontend" else not case["streaming"]
        ids = torch.randint(0, 6561, (sum(lengths),), generator=g, device=DEV)
        mels = [RATIO * (n - (0 if final else LOOKAHEAD)) for n in lengths]
        prompts = [_randn(g, 1, _prompt_frames(m), 80) for m in mels]
        return dict(ids=ids.to(torch.int32), final=final, mels=mels, prompts=prompts,
                    xvec=_randn(g, len(lengths), 192),
                    noise=_randn(g, len(lengths), 80, max(mels)))
    if op == "vocoder":
        # log-Mel like input: smooth over time, O(1)
        def mel(n):
            x = _randn(g, 80, n + 8)
            return sum(x[:, k:k + n] for k in range(8)) / math.sqrt(8.0)
        return dict(mels=[mel(n) for n in lengths])
    rows, n = sum(lengths), len(lengths)
    noise, mu, prompt = (_randn(g, rows, 80) for _ in range(3))
    spks = _randn(g, n, 80)
    cond, off = torch.zeros(rows, 80, device=DEV), 0
    for m in lengths:
        cond[off:off + _prompt_frames(m)] = prompt[off:off + _prompt_frames(m)]
        off += m
    if op == "solve":
        return dict(x=noise, mu=mu, cond=cond, spks=spks, docs=lengths)
    t = torch.rand(1, generator=g, device=DEV)
    if case["cfg"]:  # the solver's stack: the unconditional half reads zero mu/cond/spks
        z = torch.zeros_like
        return dict(x=torch.cat([noise, noise]), mu=torch.cat([mu, z(mu)]),
                    cond=torch.cat([cond, z(cond)]), spks=torch.cat([spks, z(spks)]), t=t,
                    docs=lengths + lengths)
    return dict(x=noise, mu=mu, cond=cond, spks=spks, t=t, docs=lengths)


def _pad(rows: torch.Tensor, docs: list[int]) -> torch.Tensor:
    out, off = rows.new_zeros(len(docs), rows.shape[1], max(docs)), 0
    for d, n in enumerate(docs):
        out[d, :, :n] = rows[off:off + n].T
        off += n
    return out


def prepare(case: dict, seed: int) -> dict:
    s = _inputs(case, seed)
    op, lengths = case["op"], _lengths(case)
    s["case"] = case
    if op in ("frontend", "flow"):
        s["fe"] = _flow()
        if op == "flow":
            # the language model's tokens reach the flow as lists on the host
            ids, off, s["tokens"] = s["ids"].tolist(), 0, []
            for n in lengths:
                s["tokens"].append(ids[off:off + n])
                off += n
            if not hasattr(s["fe"], "decoder"):
                s["fe"].decoder = _fcv().CFMDecoder(_estimator(22), CFG_RATE,
                                                    rand_noise=_rand_noise())
    elif op == "vocoder":
        s["voc"] = _vocoder()
    elif op == "solve":
        s["est"] = _estimator(22)
    else:
        s["est"] = _estimator(case["depth"])
        if case["padded"]:
            docs = s["docs"]
            s["mask"] = _pad(torch.ones(sum(docs), 1, device=DEV), docs)
            for k in ("x", "mu", "cond"):
                s[k] = _pad(s[k], docs)
            s["t"] = s["t"].repeat(len(docs))
    return s


def run(s: dict):
    case = s["case"]
    op = case["op"]
    if op == "frontend":
        lengths = _lengths(case)
        mu, mels = s["fe"].token_features_device(s["ids"], lengths, [s["final"]] * len(lengths))
        spks = s["fe"].speaker(s["xvec"])
        cond, _ = s["fe"].prompt_condition(s["prompts"], mels)
        return {"mu": mu, "spks": spks, "cond": cond}
    if op == "flow":
        if case["streaming"]:
            return _fcv().flow_inference_batched_streaming(
                s["fe"], s["tokens"], s["prompts"], s["xvec"], [False] * len(s["tokens"]))
        return _fcv().flow_inference_batched(s["fe"], s["tokens"], s["prompts"], s["xvec"],
                                             noise=s["noise"])
    if op == "solve":
        return _fcv().solve_euler_packed(s["est"], s["x"], s["mu"], s["cond"], s["spks"],
                                         s["docs"], n_steps=10, cfg_rate=CFG_RATE,
                                         streaming=case["streaming"])
    if op == "vocoder":
        return s["voc"].inference_batched(s["mels"], [case["final"]] * len(s["mels"]),
                                          return_source=case["source"])
    if case["padded"]:
        return s["est"](s["x"], s["mask"], s["mu"], s["t"], s["spks"], s["cond"],
                        streaming=case["streaming"])
    return s["est"].forward_packed(s["x"], s["mu"], s["cond"], s["spks"], s["t"], s["docs"],
                                   streaming=case["streaming"])


# ---- what a pass cannot do without -------------------------------------------------------------


def _dit_work(docs: list[int], streaming: bool, depth: int, steps: int) -> dict:
    rows = sum(docs)
    pairs = 0
    for n in docs:
        q = np.arange(n)
        pairs += int(np.minimum((q // CHUNK + 1) * CHUNK, n).sum()) if streaming else n * n
    row = 2 * (320 * 1024 + 2 * 31 * 64 * 1024 + depth * 8 * 1024 * 1024 + 1024 * 80)
    weights = 2 * (320 * 1024 + 2 * 31 * 64 * 1024 + depth * 14 * 1024 * 1024 + 2 * 1024 * 1024
                   + 1024 * 80 + 1024 * 1280)
    return {"bytes": weights + steps * 4 * 80 * 4 * rows,
            "flops": steps * (row * rows + 4.0 * 1024 * pairs * depth)}


def work(case: dict) -> dict:
    op, lengths = case["op"], _lengths(case)
    front = {"bytes": 0, "flops": 0}
    if op in ("frontend", "flow"):
        final = case["final"] if op == "frontend" else not case["streaming"]
        tok = [n - (0 if final else LOOKAHEAD) for n in lengths]
        macs = 4 * 80 * 1024 + 3 * 1024 * 80
        front = {"bytes": 4 * macs + sum(tok) * (4 + 320 + RATIO * 320 * 3),
                 "flops": 2.0 * macs * sum(tok)}
        if op == "frontend":
            return front
        d = _dit_work([RATIO * n for n in tok] * 2, case["streaming"], 22, 10)
        return {k: front[k] + d[k] for k in d}
    if op == "vocoder":
        dims = _hift_dims()
        frames = sum(lengths)
        macs = sum(_fcv().synthetic.hift_macs_per_frame(dims).values())
        params = sum(math.prod(s) for _, s in _fcv().synthetic.hift_state_dict_shapes(dims))
        scale = dims.upsample_scale
        return {"bytes": 4 * params + frames * 4 * (80 + scale * (1 + dims.nb_harmonics + 1
                                                                  + int(case["source"]))),
                "flops": 2.0 * macs * frames}
    if op == "solve":
        return _dit_work(lengths * 2, case["streaming"], 22, 10)
    return _dit_work(lengths * (2 if case["cfg"] else 1), case["streaming"], case["depth"], 1)


def tolerance(case: dict):
    """About four times the error against ``exact`` measured on an MI355X (fp16 operands in the
    DiT, fp32 elsewhere): front-end 3e-7, vocoder 2.4e-5 (4.3e-5 on longer requests), one block
    3.8e-4, 22 blocks 1.1e-3, 10 steps 5e-4."""
    op = case["op"]
    if op == "frontend":
        return {"rel": 1.2e-6, "max": 5e-5}
    if op == "vocoder":
        return {"rel": 1.5e-4, "max": 1e-2}
    if op == "forward":
        return {"rel": 1.5e-3 if case["depth"] == 1 else 4.5e-3, "max": 0.1}
    return {"rel": 2e-3, "max": 0.1}


# ---- the same results in 64 bits ---------------------------------------------------------------

F64 = torch.float64


def _mish(x):
    return x * torch.tanh(torch.nn.functional.softplus(x, threshold=700.0))


class _Dit64:
    """Packed DiT forward in fp64 (AdaLN-Zero blocks, RoPE on flat columns 0..63, full or
    chunk-causal attention inside each document)."""

    def __init__(self, depth: int, docs: list[int], streaming: bool):
        self.w, self.depth, self.docs, self.streaming = _dit_weights(depth), depth, docs, streaming
        self.pos = torch.cat([torch.arange(n, device=DEV) for n in docs])
        inv = 1.0 / (10000.0 ** (torch.arange(0, 64, 2, dtype=torch.float32, device=DEV) / 64))
        ang = (self.pos.float()[:, None] * inv[None]).double()
        self.cos, self.sin = ang.cos(), ang.sin()

    def lin(self, x, name):
        return torch.addmm(self.w[name + ".bias"].double(), x, self.w[name + ".weight"].double().T)

    def conv(self, x, name):
        w = self.w[name + ".weight"].double()  # [1024, 64, 31]
        taps = w.shape[2]
        wg = w.view(16, 64, 64, taps)
        acc = self.w[name + ".bias"].double().expand(x.shape[0], -1).clone()
        for j in range(taps):
            back = taps - 1 - j
            src = torch.roll(x, back, 0)
            src = torch.where((self.pos >= back)[:, None], src, 0.0)
            part = torch.bmm(src.view(-1, 16, 64).transpose(0, 1).contiguous(),
                             wg[..., j].transpose(1, 2).contiguous())
            acc += part.transpose(0, 1).reshape(x.shape[0], -1)
        return _mish(acc)

    def rope(self, x):
        a, b = x[:, 0:64:2].clone(), x[:, 1:64:2].clone()
        x[:, 0:64:2] = a * self.cos - b * self.sin
        x[:, 1:64:2] = b * self.cos + a * self.sin
        return x

    def attend(self, q, k, v):
        out, off = torch.empty_like(q), 0
        for n in self.docs:
            split = lambda a: a[off:off + n].view(n, 16, 64).transpose(0, 1).contiguous()
            qd, kd, vd = split(q), split(k), split(v)
            for a in range(0, n, 1024):
                b = min(a + 1024, n)
                s = torch.bmm(qd[:, a:b].contiguous(), kd.transpose(1, 2).contiguous()) / 8.0
                if self.streaming:
                    limit = (torch.arange(a, b, device=DEV) // CHUNK + 1) * CHUNK
                    hide = torch.arange(n, device=DEV)[None] >= limit[:, None]
                    s.masked_fill_(hide[None], -math.inf)
                o = torch.bmm(torch.softmax(s, -1), vd)
                out[off + a:off + b] = o.transpose(0, 1).reshape(b - a, 1024)
            off += n
        return out

    def norm(self, x, scale, shift):
        x = torch.nn.functional.layer_norm(x, (1024,), eps=1e-6)
        return x * (1 + scale) + shift

    def __call__(self, x, mu, cond, spks, t: float):
        freqs = torch.exp(torch.arange(128, dtype=F64, device=DEV) * -(math.log(10000) / 127))
        arg = 1000.0 * t * freqs
        emb = torch.cat([arg.sin(), arg.cos()])[None]
        emb = self.lin(torch.nn.functional.silu(self.lin(emb, "time_embed.time_mlp.0")),
                       "time_embed.time_mlp.2")
        emb = torch.nn.functional.silu(emb)
        spk = torch.cat([spks[d:d + 1].expand(n, -1) for d, n in enumerate(self.docs)])
        h = self.lin(torch.cat([x, cond, mu, spk], 1), "input_embed.proj")
        pre = "input_embed.conv_pos_embed.conv"
        h = self.conv(self.conv(h, pre + "1.0"), pre + "2.0") + h
        for i in range(self.depth):
            p = f"transformer_blocks.{i}."
            sh1, sc1, g1, sh2, sc2, g2 = self.lin(emb, p + "attn_norm.linear").chunk(6, 1)
            a = self.norm(h, sc1, sh1)
            o = self.attend(self.rope(self.lin(a, p + "attn.to_q")),
                            self.rope(self.lin(a, p + "attn.to_k")), self.lin(a, p + "attn.to_v"))
            h = h + g1 * self.lin(o, p + "attn.to_out.0")
            a = self.lin(self.norm(h, sc2, sh2), p + "ff.ff.0.0")
            a = torch.nn.functional.gelu(a, approximate="tanh")
            h = h + g2 * self.lin(a, p + "ff.ff.2")
        scale, shift = self.lin(emb, "norm_out.linear").chunk(2, 1)
        return self.lin(self.norm(h, scale, shift), "proj_out")


def _solve64(x, mu, cond, spks, lengths, streaming):
    net = _Dit64(22, lengths + lengths, streaming)
    span = 1 - torch.cos(torch.linspace(0, 1, 11, dtype=torch.float32) * 0.5 * torch.pi)
    z = torch.zeros_like
    mu, cond, spks = (torch.cat([a, z(a)]) for a in (mu, cond, spks))
    rows, time, dt = x.shape[0], span[0], span[1] - span[0]
    for step in range(1, 11):
        v = net(torch.cat([x, x]), mu, cond, spks, float(time))
        x = x + float(dt) * ((1.0 + CFG_RATE) * v[:rows] - CFG_RATE * v[rows:])
        time = time + dt
        if step < 10:
            dt = span[step + 1] - time
    return x


def _front64(s: dict, lengths: list[int]):
    w = {k: v.double() for k, v in _flow_weights().items()}
    w1, b1 = w["pre_lookahead_layer.conv1.weight"], w["pre_lookahead_layer.conv1.bias"]
    w2, b2 = w["pre_lookahead_layer.conv2.weight"], w["pre_lookahead_layer.conv2.bias"]
    mu, off = [], 0
    for n in lengths:
        e = w["input_embedding.weight"][s["ids"][off:off + n].long()]
        off += n
        m = n if s["final"] else n - LOOKAHEAD
        right = torch.cat([e, e.new_zeros(LOOKAHEAD, 80)])
        c = b1 + sum(right[j:j + m] @ w1[:, :, j].T for j in range(4))
        c = torch.nn.functional.leaky_relu(c)
        left = torch.cat([c.new_zeros(2, c.shape[1]), c])
        y = b2 + sum(left[j:j + m] @ w2[:, :, j].T for j in range(3)) + e[:m]
        mu.append(y.repeat_interleave(RATIO, 0))
    spks = torch.nn.functional.linear(torch.nn.functional.normalize(s["xvec"].double(), dim=1),
                                      w["spk_embed_affine_layer.weight"],
                                      w["spk_embed_affine_layer.bias"])
    cond, off = torch.zeros(sum(s["mels"]), 80, dtype=F64, device=DEV), 0
    for p, m in zip(s["prompts"], s["mels"]):
        cond[off:off + p.shape[1]] = p[0].double()
        off += m
    return torch.cat(mu), spks, cond


class _Hift64:
    """The vocoder in fp64.  The source's frame phases follow their definition: fp32 increments
    from the fp64 F0 rounded to fp32, prefix sums rounded to fp32."""

    def __init__(self):
        self.d, self.w = _hift_dims(), {}
        for k, v in _hift_weights().items():
            v = v.double()
            if k.endswith("original0"):
                d = _hift_weights()[k[:-1] + "1"].double()
                self.w[k.split(".parametrizations")[0] + ".weight"] = \
                    d * (v / d.flatten(1).norm(dim=1).view(-1, 1, 1))
            elif not k.endswith("original1"):
                self.w[k] = v

    def conv(self, x, name, dilation=1, stride=1):
        """Valid convolution of ``x`` [C, T] as one product per tap."""
        w = self.w[name + ".weight"]
        k = w.shape[2]
        n = (x.shape[1] - dilation * (k - 1) - 1) // stride + 1
        y = self.w[name + ".bias"][:, None].expand(-1, n).clone()
        for j in range(k):
            y += w[:, :, j] @ x[:, j * dilation:j * dilation + (n - 1) * stride + 1:stride]
        return y

    def causal(self, x, name, dilation=1):
        k = self.w[name + ".weight"].shape[2]
        return self.conv(torch.nn.functional.pad(x, (dilation * (k - 1), 0)), name, dilation)

    def look(self, x, name, final):
        """Right-hand context: zeros at the end of a request, the chunk's last frames else."""
        pad = self.w[name + ".weight"].shape[2] - 1
        return self.conv(torch.nn.functional.pad(x, (0, pad)) if final else x, name)

    def snake(self, x, name):
        a = self.w[name + ".alpha"][:, None]
        return x + (1.0 / (a + 1e-9)) * torch.sin(x * a) ** 2

    def resblock(self, x, name, dils):
        for j, d in enumerate(dils):
            t = self.causal(self.snake(x, f"{name}.activations1.{j}"), f"{name}.convs1.{j}", d)
            t = self.causal(self.snake(t, f"{name}.activations2.{j}"), f"{name}.convs2.{j}")
            x = x + t
        return x

    def f0(self, mel, final):
        elu = torch.nn.functional.elu
        x = elu(self.look(mel.double(), "f0_predictor.condnet.0", final))
        for i in (2, 4, 6, 8):
            x = elu(self.causal(x, f"f0_predictor.condnet.{i}"))
        y = (self.w["f0_predictor.classifier.weight"] @ x
             + self.w["f0_predictor.classifier.bias"][:, None])
        return y[0].abs()

    def source(self, f0):
        d, H, buf = self.d, self.d.nb_harmonics + 1, _hift_buffers()
        scale, T = d.upsample_scale, f0.shape[0]
        # the frame-rate phase on the host, in the fp32 order that defines it
        f = f0.float().cpu()
        up = f.repeat_interleave(scale)[:, None]
        rad = ((up * torch.arange(1, H + 1, dtype=torch.float32)) / d.sampling_rate) % 1
        rad[0] = rad[0] + buf["rand_ini"][0].cpu()
        rad = torch.nn.functional.interpolate(rad.T[None], scale_factor=1 / scale, mode="linear")
        phase = torch.cumsum(rad[0].T, 0) * 2 * np.pi * scale
        phase = phase.to(DEV).double().repeat_interleave(scale, 0)
        uv = (up > d.nsf_voiced_threshold).to(DEV).double()
        noise = (uv * d.nsf_sigma + (1 - uv) * d.nsf_alpha / 3) * \
            buf["sine_waves"][0, :T * scale].double()
        waves = torch.sin(phase) * d.nsf_alpha * uv + noise
        return torch.tanh(waves @ self.w["m_source.l_linear.weight"][0]
                          + self.w["m_source.l_linear.bias"])

    def window(self):
        n = self.d.n_fft
        k = torch.arange(n, dtype=F64, device=DEV)
        return 0.5 - 0.5 * torch.cos(2 * np.pi * k / n)

    def dft(self):
        n = self.d.n_fft
        k = torch.arange(n, dtype=F64, device=DEV)
        a = 2 * np.pi * k[:n // 2 + 1, None] * k[None] / n
        return a.cos(), a.sin()

    def stft(self, s):
        d = self.d
        x = torch.nn.functional.pad(s[None, None], (d.n_fft // 2, d.n_fft // 2), mode="reflect")
        fr = x[0, 0].unfold(0, d.n_fft, d.hop_len) * self.window()
        c, i = self.dft()
        return torch.cat([c @ fr.T, -(i @ fr.T)])

    def istft(self, mag, ph):
        d, n = self.d, self.d.n_fft
        mag = mag.clamp(max=1e2)
        re, im = mag * torch.cos(ph), mag * torch.sin(ph)
        c, i = self.dft()
        two = torch.full((n // 2 + 1, 1), 2.0, dtype=F64, device=DEV)
        two[0] = two[-1] = 1.0
        fr = (c.T @ (two * re) - i.T @ (two * im)) / n * self.window()[:, None]
        T = fr.shape[1]
        y = torch.zeros(n + d.hop_len * (T - 1), dtype=F64, device=DEV)
        e = torch.zeros_like(y)
        for k in range(n):
            at = slice(k, k + d.hop_len * (T - 1) + 1, d.hop_len)
            y[at] += fr[k]
            e[at] += self.window()[k] ** 2
        cut = slice(n // 2, y.shape[0] - n // 2)
        return y[cut] / e[cut]

    def __call__(self, mel, final):
        d, F = self.d, torch.nn.functional
        s = self.source(self.f0(mel, final))
        spec = self.stft(s)
        x = mel.double() if final else mel.double()[:, :-3]
        x = self.look(x, "conv_pre", final)
        if not final:
            spec = spec[:, :-int(np.prod(d.upsample_rates)) * d.conv_pre_look_right]
        K = len(d.resblock_kernel_sizes)
        for i, rate in enumerate(d.upsample_rates):
            x = F.leaky_relu(x, d.lrelu_slope).repeat_interleave(rate, 1)
            x = self.causal(x, f"ups.{i}")
            if i == len(d.upsample_rates) - 1:
                x = torch.cat([x[:, 1:2], x], 1)
            k, stride = d.source_down(i)
            name = f"source_downs.{i}"
            si = self.conv(F.pad(spec, (stride - 1, 0)), name, 1, stride)
            x = x + self.resblock(si, f"source_resblocks.{i}", d.source_resblock_dilation_sizes[i])
            x = sum(self.resblock(x, f"resblocks.{i * K + j}", d.resblock_dilation_sizes[j])
                    for j in range(K)) / K
        x = self.causal(F.leaky_relu(x), "conv_post")
        half = d.n_fft // 2 + 1
        y = self.istft(torch.exp(x[:half]), torch.sin(x[half:]))
        if not final:
            y = y[:-int(np.prod(d.upsample_rates)) * d.hop_len]
        return y.clamp(-d.audio_limit, d.audio_limit)[None], s.view(1, 1, -1)


@torch.no_grad()
def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    op, lengths = case["op"], _lengths(case)
    if op == "vocoder":
        voc = _Hift64()
        both = [voc(m, case["final"]) for m in s["mels"]]
        speech = [a for a, _ in both]
        return (speech, [b for _, b in both]) if case["source"] else speech
    if op in ("frontend", "flow"):
        mu, spks, cond = _front64(s, lengths)
        if op == "frontend":
            return {"mu": mu, "spks": spks, "cond": cond}
        if case["streaming"]:
            noise = _rand_noise().to(DEV).double()[0]
            x = torch.cat([noise[:, :m].T for m in s["mels"]])
        else:
            x = torch.cat([s["noise"][b, :, :m].double().T for b, m in enumerate(s["mels"])])
        x = _solve64(x, mu, cond, spks, s["mels"], case["streaming"])
        out, off = [], 0
        for m, p in zip(s["mels"], s["prompts"]):
            out.append(x[off + p.shape[1]:off + m].T[None])
            off += m
        return out
    x, mu, cond, spks = (s[k].double() for k in ("x", "mu", "cond", "spks"))
    if op == "solve":
        return _solve64(x, mu, cond, spks, lengths, case["streaming"])
    net = _Dit64(case["depth"], s["docs"], case["streaming"])
    v = net(x, mu, cond, spks, float(s["t"][0]))
    return _pad(v, s["docs"]) if case["padded"] else v
