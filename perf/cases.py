"""The work that a user of this framework has it do, as cases to be timed and compared.

Three paths, each through the entry point that a program calls:

* ``denoise``: ``OpenPi0Inference.sample_actions`` from a prefix K/V cache (priming it, the Euler
  loop over the action expert, the random draws).  Batch, prefix length, number of Euler steps and
  ragged prompts vary.  ``sample_actions_with_velocities`` where a case is a block of the expert
  (few layers): the same launch, which also returns every step's velocity.
* ``prefill``: ``PrefixLM.build_prefix_cache`` from prefix embeddings to the K/V cache of every
  layer.  Cases hold one or two whole decoder layers and the last layer's K/V.
* ``vision``: ``VisionTower.embed_image`` from pixels to projected image embeddings.

``predict`` is the three in a row, from camera images and a tokenized prompt to actions.

All three run in bf16 with fp32 norms, softmax, accumulation and heads; there is no other data type.
A program loads one engine per model and keeps it: engines, their weights (random, of the
architecture's shapes) and their contexts are held here per geometry, and ``prepare`` makes new
inputs for them.  A context of a new signature is created, and run once on zeros, in ``prepare``.
"""

from __future__ import annotations

import math
import os
import sys
from dataclasses import replace

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pi05-infer_amd"))

from pi05_infer import prefix as P05  # noqa: E402
from pi05_infer import synthetic as S05  # noqa: E402
from pi05_infer import vision as V05  # noqa: E402
from pi05_infer.engine import OpenPi0InferConfig, OpenPi0Inference  # noqa: E402

BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
HORIZON, ACT, VOCAB = 50, 32, 257152
MLP, WID, HEADS, HD = 4096, 1024, 8, 256  # action expert
PMLP, PWID = 16384, 2048  # prefix language model
VMLP, VWID, VHEADS, PATCHES = 4304, 1152, 16, 256  # vision tower
EXPERT_LAYER = (HEADS * HD + 2 * HD) * WID + WID * HEADS * HD + 3 * MLP * WID
PREFIX_KV = 2 * HD * PWID
PREFIX_LAYER = (HEADS * HD) * PWID + PREFIX_KV + PWID * HEADS * HD + 3 * PMLP * PWID
VISION_LAYER = 4 * VWID * VWID + 2 * VWID * VMLP
PADS = ("none", "tail")


def listed():
    return [
        # the smallest call: a block of two expert layers over a short prefix, three Euler steps; what
        # counts is the launch, the priming and the hand-offs between phases
        {"name": "denoise_block", "kind": "denoise", "depth": 2, "steps": 3, "batch": 1, "prefix": 64, "pad": "none"},
        # the headline: one robot, three views and a 200-token prompt, 10 steps through all 18 layers
        {"name": "denoise_one", "kind": "denoise", "depth": 18, "steps": 10, "batch": 1, "prefix": 968, "pad": "none"},
        # three environments whose prompts differ in length, an odd prefix; a few layers
        {"name": "denoise_ragged3", "kind": "denoise", "depth": 4, "steps": 3, "batch": 3, "prefix": 301, "pad": "tail"},
        # eight environments served together, the whole loop
        {"name": "denoise_batch8", "kind": "denoise", "depth": 18, "steps": 10, "batch": 8, "prefix": 968, "pad": "tail"},
        # the longest prefix (several frames of views): attention counts
        {"name": "denoise_long", "kind": "denoise", "depth": 18, "steps": 10, "batch": 1, "prefix": 3272, "pad": "none"},
        # one decoder layer over one view and a short prompt, odd length: latency
        {"name": "prefill_short", "kind": "prefill", "depth": 2, "batch": 1, "prefix": 313, "pad": "none"},
        # two decoder layers over the headline's prefix
        {"name": "prefill_one", "kind": "prefill", "depth": 3, "batch": 1, "prefix": 968, "pad": "none"},
        # four environments with two views each, prompts padded to 200 tokens
        {"name": "prefill_batch4", "kind": "prefill", "depth": 3, "batch": 4, "prefix": 712, "pad": "tail"},
        # one camera
        {"name": "vision_one", "kind": "vision", "depth": 6, "batch": 1},
        # three cameras of one robot
        {"name": "vision_three", "kind": "vision", "depth": 6, "batch": 3},
        # three cameras of eight environments
        {"name": "vision_batch24", "kind": "vision", "depth": 6, "batch": 24},
        # a whole predict: three views and a 200-token prompt (partly padding) to actions
        {"name": "predict", "kind": "predict", "views": 3, "tokens": 200, "batch": 1, "steps": 10},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("denoise", "denoise", "prefill", "vision"))
    if kind == "denoise":
        batch = _log(rng, 1, 8)
        # the largest listed batch and the longest listed prefix do not come together
        plen = _log(rng, 17, max(64, min(3272, 8 * 968 // batch)))
        return {"kind": kind, "depth": rng.randint(2, 18), "steps": rng.randint(2, 10), "batch": batch, "prefix": plen, "pad": rng.choice(PADS)}
    if kind == "prefill":
        batch = _log(rng, 1, 4)
        return {"kind": kind, "depth": rng.randint(2, 3), "batch": batch, "prefix": _log(rng, 48, 2848 // batch if batch > 2 else 1200), "pad": rng.choice(PADS)}
    return {"kind": kind, "depth": rng.randint(2, 6), "batch": _log(rng, 1, 24)}


# ---------------------------------------------------------------------------------------------
# engines and inputs
# ---------------------------------------------------------------------------------------------
_weights: dict = {}
_engines: dict = {}
_warm: set = set()


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _expert_weights():
    """All 18 layers; a shallower expert uses the first ones and the same heads."""
    if "expert" not in _weights:
        gen = torch.Generator(device=_device()).manual_seed(11)
        w = {}
        for name, shape, is_bf in S05.parameter_specs(S05.ExpertGeometry()):
            w[name] = (torch.randn(*shape, generator=gen, device=_device()) * 0.02).to(BF if is_bf else F32)
        _weights["expert"] = w
    return _weights["expert"]


def _prefix_weights(depth):
    if ("prefix", depth) not in _weights:
        g = replace(P05.PrefixGeometry(), depth=depth)
        _weights["prefix", depth] = P05.make_weights(g, seed=12, device=_device(), with_embedding=depth == 18)
    return _weights["prefix", depth]


def _vision_weights(depth):
    if ("vision", depth) not in _weights:
        _weights["vision", depth] = V05.make_weights(replace(V05.VisionGeometry(), depth=depth), seed=13, device=_device())
    return _weights["vision", depth]


def _expert_engine(depth, steps):
    key = ("expert", depth, steps)
    if key not in _engines:
        g = replace(S05.ExpertGeometry(), depth=depth)
        m = OpenPi0Inference(OpenPi0InferConfig(num_steps=steps), g)
        m.to(_device())
        w = _expert_weights()
        m.load_state_dict({n: w[n] for n in m.expected_parameters()})
        _engines[key] = m.eval()
    return _engines[key]


def _prefix_engine(depth):
    if ("prefix", depth) not in _engines:
        m = P05.PrefixLM(replace(P05.PrefixGeometry(), depth=depth))
        m.to(_device())
        m.load_state_dict(_prefix_weights(depth))
        _engines["prefix", depth] = m
    return _engines["prefix", depth]


def _vision_engine(depth):
    if ("vision", depth) not in _engines:
        m = V05.VisionTower(replace(V05.VisionGeometry(), depth=depth))
        m.to(_device())
        m.load_state_dict(_vision_weights(depth))
        _engines["vision", depth] = m
    return _engines["vision", depth]


def _predict_engine(steps):
    key = ("predict", steps)
    if key not in _engines:
        m = OpenPi0Inference(OpenPi0InferConfig(num_steps=steps))
        m.to(_device())
        m.load_state_dict(_expert_weights())
        m.attach_prefix_lm(_prefix_engine(18))
        m.attach_vision_tower(_vision_engine(27))
        _engines[key] = m.eval()
    return _engines[key]


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _pad_mask(gen, batch, plen, pad):
    """Valid tokens: all, or (``tail``) prompts of different lengths padded at the end, up to a
    fifth of the prefix."""
    if pad == "none":
        return torch.ones(batch, plen, dtype=torch.bool, device=_device())
    cut = torch.randint(0, plen // 5 + 1, (batch, 1), generator=gen, device=_device())
    return torch.arange(plen, device=_device())[None, :] < plen - cut


def _inputs(case, seed):
    gen, dev, b = _gen(seed), _device(), case["batch"]

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    if case["kind"] == "denoise":
        n, d = case["prefix"], case["depth"]
        pad = _pad_mask(gen, b, n, case["pad"])
        return {"prefix_k": randn(b, d, n, HD).to(BF), "prefix_v": randn(b, d, n, HD).to(BF), "prefix_pad_masks": pad, "noise": randn(b, HORIZON, ACT)}
    if case["kind"] == "prefill":
        pad = _pad_mask(gen, b, case["prefix"], case["pad"])
        return {"embs": randn(b, case["prefix"], PWID).to(BF), "pad": pad}
    if case["kind"] == "vision":
        return {"pixels": torch.rand(b, 3, 224, 224, generator=gen, device=dev) * 2 - 1}
    t = case["tokens"]
    used = torch.randint(t // 4, t + 1, (b, 1), generator=gen, device=dev)
    return {
        "images": [torch.rand(b, 3, 224, 224, generator=gen, device=dev) * 2 - 1 for _ in range(case["views"])],
        "image_masks": [torch.ones(b, dtype=torch.bool, device=dev) for _ in range(case["views"])],
        "tokenized_prompt": torch.randint(0, VOCAB, (b, t), generator=gen, device=dev, dtype=torch.int32),
        "tokenized_prompt_mask": torch.arange(t, device=dev)[None, :] < used,
        "noise": randn(b, HORIZON, ACT),
    }


def _engine(case):
    if case["kind"] == "denoise":
        return _expert_engine(case["depth"], case["steps"])
    if case["kind"] == "prefill":
        return _prefix_engine(case["depth"])
    if case["kind"] == "vision":
        return _vision_engine(case["depth"])
    return _predict_engine(case["steps"])


def _call(case, engine, x):
    if case["kind"] == "denoise":
        obs = {k: x[k] for k in ("prefix_k", "prefix_v", "prefix_pad_masks")}
        if case["depth"] <= 4:
            actions, vel = engine.sample_actions_with_velocities(obs, x["noise"])
            return {"actions": actions, "velocities": vel}
        return engine.sample_actions(obs, x["noise"])
    if case["kind"] == "prefill":
        _, _, kv = engine.build_prefix_cache(x["embs"], x["pad"])
        return {"k": [k for k, _ in kv], "v": [v for _, v in kv]}
    if case["kind"] == "vision":
        return engine.embed_image(x["pixels"])
    return engine.sample_actions({k: v for k, v in x.items() if k != "noise"}, x["noise"])


def prepare(case, seed):
    case = {k: v for k, v in case.items() if k != "name"}
    engine = _engine(case)
    x = _inputs(case, seed)
    key = tuple(sorted((k, v) for k, v in case.items() if k != "pad"))
    if key not in _warm:
        zeros = {k: [torch.zeros_like(t) for t in v] if isinstance(v, list) else torch.zeros_like(v) for k, v in x.items()}
        for k, v in x.items():
            if "mask" in k or k == "pad":
                zeros[k] = [torch.ones_like(t) for t in v] if isinstance(v, list) else torch.ones_like(v)
        _call(case, engine, zeros)
        _warm.add(key)
    return case, engine, x


def run(state):
    return _call(*state)


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------
def _denoise_work(depth, steps, batch, plen):
    """Every Euler step needs the step before it, and the weights (35 MB a layer) and the prefix K/V
    are far larger than what the chip keeps next to its units: both are read once per step.  The
    modulation table row and the action tokens likewise."""
    rows = batch * HORIZON
    keys = plen + HORIZON
    nbytes = depth * EXPERT_LAYER * 2 + depth * batch * keys * HD * 2 * 2 + (2 * depth + 1) * 3 * WID * 4 + 2 * rows * ACT * 4
    flops = 2 * rows * (depth * EXPERT_LAYER + 2 * ACT * WID) + 4 * depth * rows * HEADS * HD * keys
    return steps * nbytes, steps * flops


def _prefill_work(depth, batch, plen):
    rows, full = batch * plen, depth - 1
    nbytes = (full * PREFIX_LAYER + PREFIX_KV) * 2 + rows * PWID * 2 + depth * rows * HD * 2 * 2
    flops = 2 * rows * (full * PREFIX_LAYER + PREFIX_KV) + full * 4 * batch * HEADS * plen * plen * HD
    return nbytes, flops


def _vision_work(depth, images):
    rows, pix = images * PATCHES, 3 * 14 * 14
    nbytes = depth * VISION_LAYER * 2 + VWID * pix * 4 + VWID * PWID * 2 + PATCHES * VWID * 4 + images * 3 * 224 * 224 * 4 + rows * PWID * 2
    flops = 2 * rows * (depth * VISION_LAYER + VWID * pix + VWID * PWID) + depth * 4 * images * PATCHES * PATCHES * VWID
    return nbytes, flops


def work(case):
    if case["kind"] == "denoise":
        parts = [_denoise_work(case["depth"], case["steps"], case["batch"], case["prefix"])]
    elif case["kind"] == "prefill":
        parts = [_prefill_work(case["depth"], case["batch"], case["prefix"])]
    elif case["kind"] == "vision":
        parts = [_vision_work(case["depth"], case["batch"])]
    else:
        b = case["batch"]
        plen = case["views"] * PATCHES + case["tokens"]
        parts = [_vision_work(27, case["views"] * b), _prefill_work(18, b, plen), _denoise_work(18, case["steps"], b, plen)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """About four times what two correct implementations differ by (bf16 between layers, fp32 sums in
    another order, another choice of GEMM algorithm included)."""
    if case["kind"] == "vision":
        return {"rel": 0.02, "max": 0.2}
    if case["kind"] == "prefill":
        return {"rel": 0.02, "max": 0.2}
    # velocities pass through every layer once; the actions are the noise less a small multiple of them
    return {"rel": 0.02, "max": 0.2} if case["kind"] == "denoise" and case["depth"] <= 4 else {"rel": 0.01, "max": 0.1}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, without rounding between the layers
# ---------------------------------------------------------------------------------------------
def _rms(x, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope(x, pos):
    """x [B, T, H, D], pos [B, T]: rotate the half-split pairs."""
    half = x.shape[-1] // 2
    freq = 10000.0 ** (-torch.arange(half, dtype=F64, device=x.device) / half)
    ang = pos.to(F64)[:, :, None, None] * freq
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * ang.cos() - hi * ang.sin(), hi * ang.cos() + lo * ang.sin()], dim=-1)


def _mqa(q, k, v, valid):
    """q [B, T, H, D]; k, v [B, S, D]; valid [B, S]."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()[:, None]) / math.sqrt(q.shape[-1])
    s = s.masked_fill(~valid[:, None, None, :], -math.inf)
    return torch.matmul(torch.softmax(s, dim=-1), v[:, None]).flatten(2)


def _exact_denoise(depth, steps, ks, vs, pad, noise):
    w = _expert_weights()

    def p(name):
        return w[name].to(F64)

    def linear(x, name):
        return x @ p(name + ".weight").T + p(name + ".bias")

    dev, b, plen = noise.device, noise.shape[0], pad.shape[1]
    pos = pad.sum(1, keepdim=True) + torch.arange(HORIZON, device=dev)
    valid = torch.cat([pad, torch.ones(b, HORIZON, dtype=torch.bool, device=dev)], dim=1)
    x, vel, dt = noise.to(F64), [], 1.0 / steps
    base = "paligemma_with_expert.gemma_expert.model."
    for s in range(steps):
        t = 1.0 - s * dt
        period = 4e-3 * (4.0 / 4e-3) ** torch.linspace(0, 1, WID // 2, dtype=F64, device=dev)
        ang = t * 2 * math.pi / period
        silu = torch.nn.functional.silu
        cond = silu(linear(silu(linear(torch.cat([ang.sin(), ang.cos()]), "time_mlp_in")), "time_mlp_out"))
        h = linear(x, "action_in_proj")
        for i in range(depth):
            n = f"{base}layers.{i}."
            scale, shift, gate = linear(cond, n + "input_layernorm.dense").chunk(3)
            y = _rms(h) * (1 + scale) + shift
            q = _rope((y @ p(n + "self_attn.q_proj.weight").T).view(b, HORIZON, HEADS, HD), pos)
            k = _rope((y @ p(n + "self_attn.k_proj.weight").T).view(b, HORIZON, 1, HD), pos)[:, :, 0]
            v = y @ p(n + "self_attn.v_proj.weight").T
            o = _mqa(q, torch.cat([ks[i].to(F64), k], dim=1), torch.cat([vs[i].to(F64), v], dim=1), valid)
            h = h + (o @ p(n + "self_attn.o_proj.weight").T) * gate
            scale, shift, gate = linear(cond, n + "post_attention_layernorm.dense").chunk(3)
            y = _rms(h) * (1 + scale) + shift
            y = _gelu(y @ p(n + "mlp.gate_proj.weight").T) * (y @ p(n + "mlp.up_proj.weight").T)
            h = h + (y @ p(n + "mlp.down_proj.weight").T) * gate
        scale, shift, _ = linear(cond, base + "norm.dense").chunk(3)
        v = linear(_rms(h) * (1 + scale) + shift, "action_out_proj")
        vel.append(v)
        x = x - v * dt
    return x, torch.stack(vel)


def _exact_prefill(depth, embs, pad):
    w = _prefix_weights(depth)
    b, plen, _ = embs.shape
    pos = pad.long().cumsum(1) - 1
    h, ks, vs = embs.to(F64), [], []
    for i in range(depth):
        n = f"paligemma_with_expert.paligemma.model.language_model.layers.{i}."

        def mm(x, name):
            return x @ w[n + name + ".weight"].to(F64).T

        y = _rms(h) * (1 + w[n + "input_layernorm.weight"].to(F64))
        k = _rope(mm(y, "self_attn.k_proj").view(b, plen, 1, HD), pos)[:, :, 0]
        v = mm(y, "self_attn.v_proj")
        ks.append(k)
        vs.append(v)
        if i == depth - 1:
            break
        q = _rope(mm(y, "self_attn.q_proj").view(b, plen, HEADS, HD), pos)
        o = torch.cat([_mqa(q[j : j + 1], k[j : j + 1], v[j : j + 1], pad[j : j + 1]) for j in range(b)])
        h = h + mm(o, "self_attn.o_proj")
        y = _rms(h) * (1 + w[n + "post_attention_layernorm.weight"].to(F64))
        h = h + mm(_gelu(mm(y, "mlp.gate_proj")) * mm(y, "mlp.up_proj"), "mlp.down_proj")
    return ks, vs


def _exact_vision(depth, pixels):
    w = _vision_weights(depth)
    base = "paligemma_with_expert.paligemma.model.vision_tower.vision_model."
    n = pixels.shape[0]

    def lin(x, name):
        return x @ w[name + ".weight"].to(F64).T + w[name + ".bias"].to(F64)

    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w[name + ".weight"].to(F64) + w[name + ".bias"].to(F64)

    def heads(x):
        return x.view(n, PATCHES, VHEADS, VWID // VHEADS).transpose(1, 2).contiguous()

    e = base + "embeddings."
    x = pixels.to(F64).reshape(n, 3, 16, 14, 16, 14).permute(0, 2, 4, 1, 3, 5).reshape(n, PATCHES, -1)
    h = x @ w[e + "patch_embedding.weight"].to(F64).reshape(VWID, -1).T + w[e + "patch_embedding.bias"].to(F64)
    h = h + w[e + "position_embedding.weight"].to(F64)
    for i in range(depth):
        m = f"{base}encoder.layers.{i}."
        y = norm(h, m + "layer_norm1")
        q, k, v = (heads(lin(y, m + f"self_attn.{c}_proj")) for c in "qkv")
        s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(VWID // VHEADS)
        o = torch.matmul(torch.softmax(s, dim=-1), v).transpose(1, 2).reshape(n, PATCHES, VWID)
        h = h + lin(o, m + "self_attn.out_proj")
        h = h + lin(_gelu(lin(norm(h, m + "layer_norm2"), m + "mlp.fc1")), m + "mlp.fc2")
    return lin(norm(h, base + "post_layernorm"), "paligemma_with_expert.paligemma.model.multi_modal_projector.linear")


@torch.no_grad()
def exact(case, seed):
    x = _inputs(case, seed)
    if case["kind"] == "denoise":
        layers = range(case["depth"])
        ks, vs = ([x[n][:, i] for i in layers] for n in ("prefix_k", "prefix_v"))
        actions, vel = _exact_denoise(case["depth"], case["steps"], ks, vs, x["prefix_pad_masks"], x["noise"])
        return {"actions": actions, "velocities": vel} if case["depth"] <= 4 else {"actions": actions}
    if case["kind"] == "prefill":
        ks, vs = _exact_prefill(case["depth"], x["embs"], x["pad"])
        return {"k": [k[:, None] for k in ks], "v": [v[:, None] for v in vs]}
    if case["kind"] == "vision":
        return _exact_vision(case["depth"], x["pixels"])
    table = _prefix_weights(18)["paligemma_with_expert.paligemma.model.language_model.embed_tokens.weight"]
    imgs = [_exact_vision(27, im) for im in x["images"]]
    embs = torch.cat(imgs + [table[x["tokenized_prompt"].long()].to(F64) * math.sqrt(PWID)], dim=1)
    pad = torch.cat([m[:, None].expand(-1, PATCHES) for m in x["image_masks"]] + [x["tokenized_prompt_mask"]], dim=1)
    ks, vs = _exact_prefill(18, embs, pad)
    return {"actions": _exact_denoise(18, case["steps"], ks, vs, pad, x["noise"])[0]}
