"""The work a user of the verify path has it do, as measurable cases.

Five kinds of call, each through the package's public entry points:

* ``linear``: one quantized projection of a decoder layer (the patched
  ``QuantizedLinear`` call), from one decode row over the verify rows of one
  request and of a batch to a prompt chunk, in the weight formats that MLX
  packs come in (4 bits in groups of 64; 4 or 8 bits in groups of 32/64/128);
* ``attention``: the ragged GQA attention of the verify rows over a padded
  KV cache (``ragged_sdpa``);
* ``experts``: the routed experts of one sparse block (``SwitchGLU`` with the
  sorted-rows patch), from a few verify rows to a prompt chunk;
* ``accept``: the accept/reject of one or more requests' drafts over the full
  vocabulary (``spec_accept``), with a top-k bound or by nucleus alone;
* ``step``: a whole captured verify step (embedding, decoder layers, lm_head,
  accept/reject), which returns its logits (a committed token of such a step
  turns on the last bits of two nearly equal probabilities; the tokens are
  compared where the accept step has its logits given).
"""

from __future__ import annotations

import math

import numpy as np
import torch

DEV = "cuda"

# (N, K) of the projections of the 27B-shaped dense decoder and the 125B-class
# MoE decoder: gate/up, down, q|k|v, o, one K/V projection; q|k|v, o, shared
# expert up and down.
SHAPES = [(17408, 5120), (5120, 17408), (7168, 5120), (5120, 5120), (1024, 5120),
          (5120, 4096), (4096, 4096), (1536, 4096), (4096, 1536)]


def listed():
    return [
        # One decode row through a K/V projection: the smallest call.
        dict(name="linear_one_row", kind="linear", m=1, n=1024, k=5120, bits=4, group=64),
        # The depth-3 verify rows of one request through gate/up: the ordinary call.
        dict(name="linear_verify", kind="linear", m=4, n=17408, k=5120, bits=4, group=64),
        # A continuous batch (16 requests of mixed depths) through down.
        dict(name="linear_batch", kind="linear", m=45, n=5120, k=17408, bits=4, group=64),
        # A prompt chunk through gate/up.
        dict(name="linear_prompt", kind="linear", m=512, n=17408, k=5120, bits=4, group=64),
        # The verify rows through a layer that a mixed pack keeps at 8 bits.
        dict(name="linear_8bit", kind="linear", m=4, n=17408, k=5120, bits=8, group=64),
        # One request, depth 3, at 4k context.
        dict(name="attention_one", kind="attention", b=1, rows=4, hq=40, hkv=8, ctx=4096, spread=0.0),
        # Eight requests of very different lengths up to 32k.
        dict(name="attention_ragged", kind="attention", b=8, rows=4, hq=40, hkv=8, ctx=32768, spread=1.0),
        # Sparse block of the 125B-class decoder: four requests' verify rows.
        dict(name="experts_verify", kind="experts", t=16, e=256, top=8, h=4096, f=1536),
        # The same block on a prompt chunk.
        dict(name="experts_prompt", kind="experts", t=512, e=256, top=8, h=4096, f=1536),
        # Accept/reject of one request's three drafts at the default sampler.
        dict(name="accept_top_k", kind="accept", b=1, depth=3, v=151936, top_k=20, top_p=0.95, temp=0.6),
        # Four requests sampled by nucleus alone (no top-k bound).
        dict(name="accept_nucleus", kind="accept", b=4, depth=3, v=151936, top_k=0, top_p=0.95, temp=0.6),
        # Two 27B-shaped layers, the lm_head and the accept step in one captured step.
        dict(name="step_dense", kind="step", layers=2, b=1, depth=3, ctx=4096, v=151936),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "attention", "experts", "accept", "step"])
    if kind == "linear":
        n, k = rng.choice(SHAPES)
        if rng.random() < 0.3:
            n -= rng.randrange(1, 32)   # a head or router width that is no multiple of a tile
        bits, group = rng.choice([(4, 64)] * 4 + [(4, 128), (4, 32), (8, 64), (8, 128), (8, 32)])
        m = _log(rng, 1, 512 if (bits, group) in ((4, 64), (4, 128)) else 64)
        return dict(kind=kind, m=m, n=n, k=k, bits=bits, group=group)
    if kind == "attention":
        hq, hkv = rng.choice([(40, 8), (32, 4)])
        return dict(kind=kind, b=rng.randint(1, 8), rows=rng.randint(1, 4), hq=hq, hkv=hkv,
                    ctx=_log(rng, 256, 32768), spread=round(rng.random(), 3))
    if kind == "experts":
        h, f = rng.choice([(4096, 1536), (2048, 768), (2048, 1536)])
        return dict(kind=kind, t=_log(rng, 1, 512), e=rng.choice([64, 128, 256]), top=rng.choice([4, 8]), h=h, f=f)
    if kind == "accept":
        return dict(kind=kind, b=rng.randint(1, 4), depth=rng.randint(1, 4), v=_log(rng, 8192, 151936),
                    top_k=rng.choice([20, 20, 40, 64, 0, 0]), top_p=rng.choice([0.95, 0.9, 0.8]),
                    temp=rng.choice([0.6, 0.8, 1.0]))
    return dict(kind=kind, layers=rng.randint(1, 2), b=rng.randint(1, 4), depth=rng.randint(1, 4),
                ctx=_log(rng, 512, 8192), v=_log(rng, 8192, 151936))


# -- inputs ---------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _triple(gen, n, k, bits, group, lead=()):
    """A random affine pack: uniform fields, centered groups with unit gain
    (an rms-1 input gives rms-1 outputs), bf16 scales and biases."""
    w = torch.randint(-2 ** 31, 2 ** 31 - 1, lead + (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=gen)
    top = (1 << bits) - 1
    std = 1.0 / math.sqrt(k * (top + 1) ** 2 / 12.0)
    s = (std * (0.5 + torch.rand(lead + (n, k // group), device=DEV, generator=gen))).to(torch.bfloat16)
    z = 0.5 * top + 0.05 * top * torch.randn(s.shape, device=DEV, generator=gen)
    return w, s, (-z * s.float()).to(torch.bfloat16)


def _dequant(w, s, b, bits):
    """float64 [N, K] of one pack."""
    n = w.shape[0]
    per = 32 // bits
    shift = torch.arange(per, device=w.device, dtype=torch.int32) * bits
    q = ((w.unsqueeze(-1) >> shift) & ((1 << bits) - 1)).reshape(n, s.shape[1], -1)
    return (q.double() * s.double().unsqueeze(-1) + b.double().unsqueeze(-1)).reshape(n, -1)


def _rows(gen, m, k):
    """Hidden rows as a decoder hands them on: rms ~1 with a few large channels."""
    x = torch.randn((m, k), device=DEV, generator=gen)
    x *= torch.exp(0.5 * torch.randn((1, k), device=DEV, generator=gen))
    return x.to(torch.bfloat16)


def _linear_inputs(c, seed):
    gen = _gen(seed)
    return _triple(gen, c["n"], c["k"], c["bits"], c["group"]), _rows(gen, c["m"], c["k"])


def _lengths(c, gen):
    """Context lengths: the longest is ctx, the others spread below it."""
    u = torch.rand(c["b"], device=DEV, generator=gen).cpu().numpy()
    lens = np.maximum(c["rows"] + 1, (c["ctx"] * (1.0 - 0.97 * c["spread"] * u)).astype(np.int64))
    lens[0] = c["ctx"]
    return lens


def _attention_inputs(c, seed):
    gen = _gen(seed)
    lens = _lengths(c, gen)
    cap = -(-c["ctx"] // 256) * 256
    q = torch.randn((c["b"], c["hq"], c["rows"], 128), device=DEV, generator=gen).to(torch.bfloat16)
    k, v = (torch.randn((c["b"], c["hkv"], cap, 128), device=DEV, generator=gen).to(torch.bfloat16) for _ in range(2))
    start = torch.tensor(lens - c["rows"], dtype=torch.int32, device=DEV)
    return q, k, v, start, lens


def _experts_inputs(c, seed):
    gen = _gen(seed)
    gate, up = (_triple(gen, c["f"], c["h"], 4, 64, (c["e"],)) for _ in range(2))
    down = _triple(gen, c["h"], c["f"], 4, 64, (c["e"],))
    x = _rows(gen, c["t"], c["h"])
    # Zipf-skewed routing: top experts of (popularity + per-token Gumbel noise).
    rank = torch.randperm(c["e"], generator=gen, device=DEV).float() + 1.0
    noise = -torch.log(-torch.log(torch.rand((c["t"], c["e"]), device=DEV, generator=gen).clamp(1e-9, 1 - 1e-6)))
    ids = torch.topk(noise - 1.1 * torch.log(rank), c["top"], dim=1).indices.to(torch.int32).contiguous()
    return gate, up, down, x, ids


def _logit_rows(gen, shape):
    """Logit rows of a language model: a wide body and, row by row more or
    less pronounced, a head of likely tokens."""
    x = 2.0 * torch.randn(shape, device=DEV, generator=gen)
    lead = x.reshape(-1, shape[-1])
    for r in range(lead.shape[0]):
        at = torch.randperm(shape[-1], device=DEV, generator=gen)[:48]
        top = 6.0 + 12.0 * torch.rand((), device=DEV, generator=gen)
        lead[r, at] += top * torch.rand(48, device=DEV, generator=gen)
    return x


def _accept_inputs(c, seed):
    gen = _gen(seed)
    b, d, v = c["b"], c["depth"], c["v"]
    target = _logit_rows(gen, (b, d + 1, v))
    draft = (target[:, :d] + 0.5 * torch.randn((b, d, v), device=DEV, generator=gen)).contiguous()
    law = torch.softmax(draft.reshape(b * d, v) / c["temp"], dim=-1)
    ids = torch.multinomial(law, 1, generator=gen).reshape(b, d).to(torch.int32)
    u = torch.rand((b, d + 1), dtype=torch.float64, device=DEV, generator=gen)
    return target, draft, ids, u


def _step_shape(c):
    return dict(layers=c["layers"], hidden=5120, ffn=17408, n_heads=40, n_kv_heads=8, head_dim=128, vocab=c["v"])


def _step_inputs(c, seed):
    gen = _gen(seed)
    s = _step_shape(c)
    h, f, d = s["hidden"], s["ffn"], s["head_dim"]
    heads = s["n_heads"] + 2 * s["n_kv_heads"]
    norm = lambda: (1.0 + 0.1 * torch.randn(h, device=DEV, generator=gen)).to(torch.bfloat16)  # noqa: E731
    cap = -(-(c["ctx"]) // 256) * 256
    w = dict(embed=_triple(gen, s["vocab"], h, 4, 64), head=_triple(gen, s["vocab"], h, 4, 64), norm=norm(), layers=[])
    w["embed"] = (w["embed"][0], (w["embed"][1].float() * math.sqrt(h)).to(torch.bfloat16),
                  (w["embed"][2].float() * math.sqrt(h)).to(torch.bfloat16))   # embedding rows of rms ~1
    for _ in range(s["layers"]):
        w["layers"].append(dict(
            norm1=norm(), qkv=_triple(gen, heads * d, h, 4, 64), o=_triple(gen, h, s["n_heads"] * d, 4, 64),
            norm2=norm(), gate=_triple(gen, f, h, 4, 64), up=_triple(gen, f, h, 4, 64), down=_triple(gen, h, f, 4, 64),
            k=torch.randn((c["b"], s["n_kv_heads"], cap, d), device=DEV, generator=gen).to(torch.bfloat16),
            v=torch.randn((c["b"], s["n_kv_heads"], cap, d), device=DEV, generator=gen).to(torch.bfloat16)))
    rows = c["depth"] + 1
    tokens = torch.randint(0, s["vocab"], (c["b"], rows), device=DEV, dtype=torch.int32, generator=gen)
    lens = np.maximum(rows + 1, (c["ctx"] * (1.0 - 0.5 * np.arange(c["b"]) / c["b"])).astype(np.int64))
    start = torch.tensor(lens - rows, dtype=torch.int32, device=DEV)
    draft = 3.0 * torch.randn((c["b"], c["depth"], s["vocab"]), device=DEV, generator=gen)
    u = torch.rand((c["b"], rows), dtype=torch.float64, device=DEV, generator=gen)
    return w, cap, tokens, start, draft, u


# -- the calls --------------------------------------------------------------------

def prepare(case, seed):
    from mtplx_amd import moe_sorted_gather as moe
    from mtplx_amd.nax_verify import install_nax_qlinear_patch
    from mtplx_amd.quant import QuantizedLinear
    from mtplx_amd.sampling import SamplerConfig

    kind = case["kind"]
    if kind == "linear":
        install_nax_qlinear_patch()
        (w, s, b), x = _linear_inputs(case, seed)
        return kind, QuantizedLinear(w, s, b, group_size=case["group"], bits=case["bits"]), x
    if kind == "attention":
        q, k, v, start, _ = _attention_inputs(case, seed)
        return kind, q, k, v, start
    if kind == "experts":
        moe.install_switch_glu_rows()
        gate, up, down, x, ids = _experts_inputs(case, seed)
        return kind, moe.SwitchGLU(*(moe.QuantizedSwitchLinear(*t) for t in (gate, up, down))), x, ids
    if kind == "accept":
        return (kind, *_accept_inputs(case, seed), SamplerConfig(case["temp"], case["top_p"], case["top_k"]))
    from mtplx_amd.verify_step import CapturedVerifyStep, DecoderConfig, Layer, VerifyModel, kv_to_blocks

    w, cap, tokens, start, draft, u = _step_inputs(case, seed)
    lin = lambda t: QuantizedLinear(*t)  # noqa: E731
    model = VerifyModel.from_weights(
        DecoderConfig(**_step_shape(case)), lin(w["embed"]),
        [Layer(in_norm=y["norm1"], qkv=lin(y["qkv"]), o=lin(y["o"]), post_norm=y["norm2"], gate=lin(y["gate"]),
               up=lin(y["up"]), down=lin(y["down"])) for y in w["layers"]], w["norm"], lin(w["head"]), device=DEV)
    model.allocate_cache(case["b"], cap, fill_random=False)
    for i, y in enumerate(w["layers"]):
        model.k_cache[i].copy_(kv_to_blocks(y["k"], "k"))
        model.v_cache[i].copy_(kv_to_blocks(y["v"], "v"))
    return kind, CapturedVerifyStep(model, tokens, start, draft, u, SamplerConfig(0.6, 0.95, 20))


def run(state):
    kind = state[0]
    if kind == "linear":
        _, module, x = state
        return module(x)
    if kind == "attention":
        from mtplx_amd.ragged_attention import ragged_sdpa

        _, q, k, v, start = state
        return ragged_sdpa(q, k, v, start)
    if kind == "experts":
        _, block, x, ids = state
        return block(x, ids)
    if kind == "accept":
        from mtplx_amd.sampling import spec_accept

        _, target, draft, ids, u, config = state
        r = spec_accept(target, draft, ids, u, config)
        return dict(tokens=r.tokens, accepted=r.n_accepted, probs=r.accept_probs, status=r.status)
    step = state[1]
    step.replay()
    return dict(logits=step.logits)


# -- what a pass cannot do without, and how far correct outputs may differ ---------

def _pack_bytes(n, k, bits, group):
    return n * k * bits // 8 + 2 * n * (k // group) * 2


def work(case):
    c = case
    if c["kind"] == "linear":
        return dict(bytes=_pack_bytes(c["n"], c["k"], c["bits"], c["group"]) + 2 * c["m"] * (c["n"] + c["k"]),
                    flops=2 * c["m"] * c["n"] * c["k"])
    if c["kind"] == "attention":
        keys = c["b"] * c["ctx"] * (1.0 - 0.97 * c["spread"] * 0.5 * (c["b"] - 1) / c["b"])   # expected
        return dict(bytes=int(keys * c["hkv"] * 512 + 4 * c["b"] * c["hq"] * c["rows"] * 128),
                    flops=int(4 * keys * c["hq"] * c["rows"] * 128))
    if c["kind"] == "experts":
        # Distinct experts that the skewed routing reaches, in expectation.
        p = 1.0 / np.arange(1, c["e"] + 1) ** 1.1
        p /= p.sum()
        used = float(np.sum(1.0 - (1.0 - np.minimum(1.0, c["top"] * p)) ** c["t"]))
        one = 2 * _pack_bytes(c["f"], c["h"], 4, 64) + _pack_bytes(c["h"], c["f"], 4, 64)
        r = c["t"] * c["top"]
        return dict(bytes=int(used * one + 2 * c["t"] * c["h"] + 2 * r * c["h"] + 4 * r), flops=6 * r * c["h"] * c["f"])
    if c["kind"] == "accept":
        n = c["b"] * (2 * c["depth"] + 1) * c["v"]
        return dict(bytes=4 * n, flops=4 * n)
    s, rows = _step_shape(c), c["b"] * (c["depth"] + 1)
    h, f = s["hidden"], s["ffn"]
    mats = s["layers"] * (7168 * h + h * h + 3 * f * h) + s["vocab"] * h
    keys = sum(c["ctx"] * (1.0 - 0.5 * i / c["b"]) for i in range(c["b"]))
    return dict(bytes=int(mats * 0.5625 + s["layers"] * keys * 8 * 512 + 4 * rows * s["vocab"] * 2
                          + 4 * c["b"] * c["depth"] * s["vocab"]),
                flops=int(2 * rows * mats + 4 * s["layers"] * keys * 40 * (c["depth"] + 1) * 128))


def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 6e-3}     # bf16 outputs of fp32 sums: 1.7e-3 from 64 bits
    if kind == "attention":
        return {"rel": 8e-3}     # bf16 probabilities and outputs: 2.2e-3
    if kind == "experts":
        return {"rel": 1.5e-2}   # bf16 gate, up, activation and outputs in a chain: 3.9e-3
    if kind == "accept":
        return {"rel": 1e-9, "differ": 0.0}   # fp64 laws; whole ids
    return {"rel": 2.5e-2}       # bf16 between all stages of two layers and the head: 6.2e-3


# -- the same in 64 bits ------------------------------------------------------------

def _sparse_law(row, c):
    """(ids ascending, probabilities) of a logit row: temperature softmax over
    the whole vocabulary, the top_k largest (ties to the lower id), the
    nucleus whose mass before each token is below top_p, renormalised."""
    p = np.exp((row - row.max()) / c["temp"])
    p /= p.sum()
    order = np.lexsort((np.arange(p.size), -p))
    if 0 < c["top_k"] < p.size:
        order = order[:c["top_k"]]
    before = np.concatenate([[0.0], np.cumsum(p[order])[:-1]])
    if 0.0 < c["top_p"] < 1.0:
        order = order[before < c["top_p"]]
    ids = np.sort(order)
    return ids, p[ids] / p[ids].sum()


def _exact_accept(c, seed):
    target, draft, ids, u = (t.cpu().numpy().astype(np.float64) for t in _accept_inputs(c, seed))
    probs = np.full((c["b"], c["depth"]), -1.0)
    for b in range(c["b"]):
        for d in range(c["depth"]):
            tok = int(ids[b, d])
            (pi, pv), (qi, qv) = _sparse_law(target[b, d], c), _sparse_law(draft[b, d], c)
            p, q = pv[pi == tok].sum(), qv[qi == tok].sum()
            probs[b, d] = (1.0 if p > 0 else 0.0) if q <= 0 else min(1.0, p / q)
            if u[b, d] > probs[b, d]:
                break
    return dict(tokens=None, accepted=None, probs=probs, status=None)


def _attend(q, k, v, start):
    """q [Hq, L, D] against k/v [Hkv, cap, D]: row i sees keys <= start + i."""
    hq, n, d = q.shape
    end = int(start) + n
    rep = hq // k.shape[0]
    out = torch.empty_like(q)
    mask = torch.arange(end, device=q.device)[None] > int(start) + torch.arange(n, device=q.device)[:, None]
    for h in range(hq):
        kk, vv = k[h // rep, :end].double(), v[h // rep, :end].double()
        s = ((q[h] @ kk.T) / math.sqrt(d)).masked_fill(mask, float("-inf"))
        out[h] = torch.softmax(s, dim=-1) @ vv
    return out


def _exact_step(c, seed):
    w, _, tokens, start, _, _ = _step_inputs(c, seed)
    b, n = tokens.shape
    mm = lambda x, t: x @ _dequant(*t, 4).T  # noqa: E731

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g.double()

    def rope(x, pos):
        ang = pos.double()[:, None] * 1.0e6 ** (-torch.arange(64, device=DEV).double() / 64.0)
        cs, sn = torch.cos(ang), torch.sin(ang)
        a, e = x[..., :64], x[..., 64:]
        return torch.cat([a * cs - e * sn, a * sn + e * cs], -1)

    at = tokens.reshape(-1).long()
    h = _dequant(w["embed"][0][at], w["embed"][1][at], w["embed"][2][at], 4)
    for y in w["layers"]:
        qkv = mm(norm(h, y["norm1"]), y["qkv"]).reshape(b, n, 56, 128)
        out = []
        for i in range(b):
            s0 = int(start[i])
            pos = s0 + torch.arange(n, device=DEV)
            heads = qkv[i].transpose(0, 1)
            kk, vv = y["k"][i].double(), y["v"][i].double()
            kk[:, s0:s0 + n], vv[:, s0:s0 + n] = rope(heads[40:48], pos), heads[48:]
            out.append(_attend(rope(heads[:40], pos), kk, vv, s0).transpose(0, 1).reshape(n, 5120))
        h = h + mm(torch.cat(out), y["o"])
        x = norm(h, y["norm2"])
        h = h + mm(torch.nn.functional.silu(mm(x, y["gate"])) * mm(x, y["up"]), y["down"])
    return dict(logits=mm(norm(h, w["norm"]), w["head"]))


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        t, x = _linear_inputs(case, seed)
        return x.double() @ _dequant(*t, case["bits"]).T
    if kind == "attention":
        q, k, v, start, _ = _attention_inputs(case, seed)
        return torch.stack([_attend(q[i].double(), k[i], v[i], start[i]) for i in range(case["b"])])
    if kind == "experts":
        gate, up, down, x, ids = _experts_inputs(case, seed)
        out = torch.zeros((case["t"], case["top"], case["h"]), dtype=torch.float64, device=DEV)
        for e in ids.unique().tolist():
            tok, slot = (ids == e).nonzero(as_tuple=True)
            g, p, d = (_dequant(*(t[e] for t in m), 4) for m in (gate, up, down))
            r = x[tok].double()
            out[tok, slot] = (torch.nn.functional.silu(r @ g.T) * (r @ p.T)) @ d.T
        return out
    return _exact_accept(case, seed) if kind == "accept" else _exact_step(case, seed)
