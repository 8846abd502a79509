"""Measured workloads of tjev_amd on one MI355X: what its users run through its public entry points.

Listed cases, by what they stand for:
- serving: one-token decode steps of one row and of a full batch; a short single-row prompt at
  the operator's default chunk, a long single-row prompt at the 9B layer's heads, and a batch of
  prompts continued from an earlier piece;
- training: the 0.8B and 9B layer shapes, one packed row of short sequences (varlen), ragged
  packed rows with a trained conv at the default chunk, a small fp32 layer, the v2 operator and
  the 4B block with merged LoRA, each forward and backward.

``draw`` gives further cases of the same ranges: 1 to 128 decode rows, 1 to 16384 tokens per
row, 1 to 8 rows, equal and grouped heads of 64 or 128, chunks 64 and 128, the precisions and
activation types in use, one, packed or cut segments. Sizes are the repository's benchmark and
test shapes or generic; weights and activations follow the benchmark's distributions.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import tjev_amd
from tjev_amd.serve import gdn_decode_step, gdn_prefill
from tjev_amd.v2 import chunk_gated_delta_rule_v2

TAPS = 4
RANK = 64
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, batch, length, hk, h, dim, chunk, dtype="bf16", precision="high", segments="one", conv_grad=False,
          hidden=0, fresh=True):
    c = dict(kind=kind, batch=batch, length=length, hk=hk, h=h, dim=dim, chunk=chunk, dtype=dtype, precision=precision,
             segments=segments, conv_grad=conv_grad, hidden=hidden, fresh=fresh)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one interactive request's step: 16 heads of state, launch-bound
        _case("decode_1row", "decode", 1, 1, 16, 16, 128, 64, fresh=False),
        # a full decode batch of the 0.8B layer (bench.py --config decode)
        _case("decode_64rows", "decode", 64, 1, 16, 16, 128, 64, fresh=False),
        # a chat-length prompt through gdn_prefill's defaults (chunk 64)
        _case("prefill_short", "prefill", 1, 333, 16, 16, 128, 64),
        # one long prompt at the 9B layer's grouped heads: few chains, many chunks
        _case("prefill_long_9B", "prefill", 1, 8192, 16, 32, 128, 128),
        # a batch of prompts resumed from their first piece's state and conv history
        _case("prefill_resume", "prefill", 4, 1500, 16, 16, 128, 128, fresh=False),
        # a training step of the 0.8B layer (bench.py's headline workload)
        _case("train_0.8B", "train", 4, 4096, 16, 16, 128, 128),
        # a training step of the 9B layer (bench.py --config 9B)
        _case("train_9B", "train", 2, 8192, 16, 32, 128, 128),
        # sequence packing: one row of sequences of about 300 tokens (bench.py --config varlen)
        _case("train_varlen", "train", 1, 16384, 16, 16, 128, 128, segments="geometric"),
        # a small packed batch at the operator's default chunk, ragged length, trained conv
        _case("train_ragged", "train", 2, 1777, 16, 32, 128, 64, segments="cuts", conv_grad=True),
        # the small fp32 configuration (full-precision runs and parity checks)
        _case("train_tiny_fp32", "train", 1, 512, 4, 4, 64, 64, dtype="fp32", precision="highest"),
        # the pre-gated operator in training (bench.py --config v2, fewer rows)
        _case("v2_train", "v2", 2, 2048, 16, 16, 128, 128),
        # the whole 4B layer with merged LoRA, one row (bench.py --config 4B-block, shorter)
        _case("block_4B", "block", 1, 2048, 16, 32, 128, 128, hidden=2560),
    ]


def _spread(rng, lo, hi):
    """An integer in [lo, hi], uniform over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "train", "train", "train", "train", "v2",
                       "block"])
    hk, h = rng.choice([(16, 16), (16, 16), (16, 32), (8, 16)])
    if kind == "decode":
        return _case(None, "decode", _spread(rng, 1, 128), 1, hk, h, 128, 64, fresh=False)
    dim = 128 if rng.random() < 0.85 else 64
    chunk = rng.choice([64, 128, 128])
    if kind == "prefill":
        batch = _spread(rng, 1, 8)
        return _case(None, "prefill", batch, _spread(rng, 1, 16384 // batch), hk, h, dim, chunk,
                     precision="mixed" if rng.random() < 0.15 else "high", fresh=rng.random() < 0.6)
    if kind == "block":
        return _case(None, "block", 1, _spread(rng, 128, 4096), 16, 32, 128, 128, hidden=2560,
                     segments=rng.choice(["one", "cuts"]))
    batch = _spread(rng, 1, 4)
    length = _spread(rng, 64, 16384 // batch)
    if kind == "v2":
        return _case(None, "v2", batch, max(64, length // 2), hk, h, dim, chunk, segments=rng.choice(["one", "geometric"]))
    if rng.random() < 0.15:
        return _case(None, "train", 1, _spread(rng, 64, 1024), 4, 4, 64, 64, dtype="fp32", precision="highest",
                     segments=rng.choice(["one", "cuts"]))
    return _case(None, "train", batch, length, hk, h, dim, chunk, precision="mixed" if rng.random() < 0.15 else "high",
                 segments=rng.choice(["one", "one", "geometric", "cuts"]), conv_grad=rng.random() < 0.3)


# --------------------------------------------------------------------------- inputs
def _segments(case, seed):
    """Segment ids [B, T] int32: one per row, packed sequences (lengths ~ Geometric(mean 300)
    clipped to [16, 4096]), or four random cuts with a padded tail."""
    batch, length = case["batch"], case["length"]
    rng = np.random.default_rng(seed)
    out = np.ones((batch, length), np.int32)
    for row in out:
        if case["segments"] == "geometric":
            pos, sid = 0, 1
            while pos < length:
                n = int(np.clip(rng.geometric(1.0 / 300), 16, 4096))
                row[pos:pos + n] = sid
                pos, sid = pos + n, sid + 1
        elif case["segments"] == "cuts" and length >= 8:
            cuts = np.sort(rng.choice(np.arange(1, length), 4, replace=False))
            row[:] = np.searchsorted(cuts, np.arange(length), side="right") + 1
            row[length - length // 16:] = 0
    return torch.from_numpy(out).cuda()


def _inputs(case, seed):
    """The path's tensors on the GPU, made from the seed: the benchmark's distributions."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = DTYPES[case["dtype"]]
    b, t, hk, h, d = case["batch"], case["length"], case["hk"], case["h"], case["dim"]
    width = 2 * hk * d + h * d

    def rn(*shape, dtype=torch.float32, std=1.0):
        return (torch.randn(shape, generator=gen, device="cuda") * std).to(dtype)

    s = {"a_log": torch.rand(h, generator=gen, device="cuda") * math.log(16.0), "dt_bias": rn(h)}
    if case["kind"] == "block":
        s["x"] = rn(b, t, case["hidden"], dtype=dt)
        s["dy"] = rn(b, t, case["hidden"], dtype=dt)
        s["seg"] = _segments(case, seed)
        return s
    if case["kind"] == "v2":  # q and k as the model passes them: l2-normalised, q scaled by D^-1/2
        s["q"] = (torch.nn.functional.normalize(rn(b, t, hk, d), dim=-1) * d ** -0.5).to(dt)
        s["k"] = torch.nn.functional.normalize(rn(b, t, hk, d), dim=-1).to(dt)
        s["v"] = rn(b, t, h, d, dtype=dt)
        s["g"] = -torch.exp(s["a_log"]) * torch.nn.functional.softplus(rn(b, t, h) + s["dt_bias"])
        s["beta"] = torch.sigmoid(rn(b, t, h))
        s["dy"] = rn(b, t, h, d, dtype=dt)
        s["seg"] = _segments(case, seed)
        return s
    lead = (b,) if case["kind"] == "decode" else (b, t)
    s["qkv"], s["a"], s["b"] = rn(*lead, width, dtype=dt), rn(*lead, h, dtype=dt), rn(*lead, h, dtype=dt)
    s["conv"] = rn(TAPS, width, std=0.5)
    if case["kind"] != "decode":
        s["seg"] = _segments(case, seed)
    if case["kind"] == "train":
        s["gate"], s["dy"] = rn(b, t, h, d, dtype=dt), rn(b, t, h, d, dtype=dt)
        s["norm"] = torch.ones(d, device="cuda")
    if case["kind"] in ("decode", "prefill") and not case["fresh"]:
        s["state"] = rn(b, h, d, d, std=0.05)
        s["hist"] = rn(b, TAPS - 1, width, dtype=dt)
    return s


def _shape(case):
    return dict(key_heads=case["hk"], key_dim=case["dim"], value_heads=case["h"], value_dim=case["dim"])


def _block(case, seed):
    return tjev_amd.GatedDeltaNetBlock(hidden=case["hidden"], rank=RANK, dtype=DTYPES[case["dtype"]], seed=int(seed) % 997,
                                       chunk=case["chunk"], precision=case["precision"], taps=TAPS, **_shape(case))


def _leaf_names(case):
    """The tensors a training step differentiates."""
    if case["kind"] == "v2":
        return ["q", "k", "v", "g", "beta"]
    return ["qkv", "a", "b", "a_log", "dt_bias", "gate"] + (["conv"] if case["conv_grad"] else [])


def prepare(case, seed):
    s = _inputs(case, seed)
    if case["kind"] == "block":
        s["block"] = _block(case, seed)
        s["x"].requires_grad_(True)
        s["leaves"] = [s["x"], *s["block"].parameters()]
    elif case["kind"] in ("train", "v2"):
        s["leaves"] = [s[n].requires_grad_(True) for n in _leaf_names(case)]
    return dict(s, case=dict(case))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":  # the serving loop's step: the recurrent state is updated in place
        out, hist, st = gdn_decode_step(state["qkv"], state["a"], state["b"], state["a_log"], state["dt_bias"], state["conv"],
                                        state["hist"], state["state"], inplace=True, **_shape(case))
        return {"out": out, "hist": hist, "state": st}
    if kind == "prefill":
        out, st, hist = gdn_prefill(state["qkv"], state["a"], state["b"], state["a_log"], state["dt_bias"], state["conv"],
                                    state["seg"], chunk=case["chunk"], precision=case["precision"],
                                    initial_state=state.get("state"), initial_conv=state.get("hist"), **_shape(case))
        return {"out": out, "hist": hist, "state": st}
    if kind == "train":
        out = tjev_amd.gdn_megakernel_normed(
            state["qkv"], state["a"], state["b"], state["a_log"], state["dt_bias"], state["conv"], state["seg"], state["gate"],
            state["norm"], chunk=case["chunk"], precision=case["precision"], **_shape(case))
    elif kind == "v2":
        out = chunk_gated_delta_rule_v2(state["q"], state["k"], state["v"], state["g"], state["beta"], state["seg"],
                                        chunk=case["chunk"], precision=case["precision"])
    else:
        out = state["block"](state["x"], state["seg"])
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, state["leaves"], state["dy"]))}


# --------------------------------------------------------------------------- work and tolerance
def work(case):
    """Each input read once and each output written once; the dense contractions of the chunked
    rule once each (one token: the recurrence's three matrix-vector products), nothing rebuilt."""
    b, t, hk, h, d = case["batch"], case["length"], case["hk"], case["h"], case["dim"]
    e = 2 if case["dtype"] == "bf16" else 4
    c, width, n = min(case["chunk"], max(1, t)), 2 * hk * d + h * d, b * t
    state, hist = b * h * d * d * 4, b * (TAPS - 1) * width * e
    if case["kind"] == "decode":
        return {"bytes": 2 * state + 2 * hist + n * ((width + 2 * h + h * d) * e) + TAPS * width * 4, "flops": 6.0 * n * h * d * d}
    core = n * h * (10.0 * c * d + c * c / 3 + 6 * d * d)  # per token: 5 C x C products, the inverse, 3 with the state
    back = n * h * (20.0 * c * d + 12 * d * d)  # per token: 10 C x C products, 6 with the state or its gradient
    if case["kind"] == "prefill":
        io = n * ((width + 2 * h + h * d) * e + 4) + state + hist + (0 if case["fresh"] else state + hist)
        return {"bytes": io, "flops": core}
    if case["kind"] == "v2":
        return {"bytes": n * (2 * (2 * hk * d + h * d) * e + 2 * h * d * e + 2 * 2 * h * 4 + 4), "flops": core + back}
    if case["kind"] == "train":
        return {"bytes": n * (2 * (width + 2 * h + 2 * h * d) * e + 4) + TAPS * width * 4 * (2 if case["conv_grad"] else 1),
                "flops": core + back}
    hid, outs = case["hidden"], [width, h * d, h, h]
    weights = sum(hid * o for o in outs) + h * d * hid
    adapters = sum(RANK * (hid + o) for o in outs) + RANK * (h * d + hid)
    # x W' and dy W'^T; the merge; the adapters' four thin products
    flops = 2 * 2.0 * n * weights + 2.0 * RANK * weights + 4 * 2.0 * n * adapters + core + back
    return {"bytes": n * 4 * hid * e + weights * e + adapters * 8, "flops": flops}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 2e-5}
    return {"rel": 2e-2 if case["kind"] == "block" or case["precision"] == "mixed" else 1e-2}


# --------------------------------------------------------------------------- the same in 64 bits
class _Stored(torch.autograd.Function):
    """x as the layer stores it between its stages (rounded to bf16), the gradient passed on."""

    @staticmethod
    def forward(ctx, x):
        return x.to(torch.bfloat16).to(x.dtype)

    @staticmethod
    def backward(ctx, d):
        return d


class _Inverse(torch.autograd.Function):
    """(I + L)^-1 of strictly lower triangular L [..., C, C], by doubling blocks."""

    @staticmethod
    def forward(ctx, low):
        c = low.shape[-1]
        inv = torch.eye(c, dtype=low.dtype, device=low.device).expand_as(low).clone()
        s = 1
        while s < c:
            i = torch.arange(c, device=low.device)
            off = ((i[:, None] // (2 * s) == i[None] // (2 * s)) & (i[:, None] // s % 2 == 1) & (i[None] // s % 2 == 0))
            inv = inv - inv @ (low * off) @ inv
            s *= 2
        ctx.save_for_backward(inv)
        return inv

    @staticmethod
    def backward(ctx, d):
        (inv,) = ctx.saved_tensors
        t = inv.transpose(-1, -2).contiguous()
        return -(t @ d.contiguous() @ t)


def _rule64(q, k, v, g, beta, seg, s0=None, c=64):
    """The chunked gated delta rule in fp64: q, k [B,T,H,D] (repeated to the value heads),
    v [B,T,H,D], g, beta [B,T,H] -> out [B,T,H,D] and the state after the last token."""
    b, t, h, d = v.shape
    n = -(-t // c)
    pad = n * c - t

    def chunks(x):
        x = torch.nn.functional.pad(x, (0, 0) * (x.dim() - 2) + (0, pad))
        return x.reshape(b, n, c, h, -1).permute(0, 3, 1, 2, 4).contiguous()

    q, k, v, beta = chunks(q), chunks(k), chunks(v), chunks(beta)
    gam = torch.cumsum(chunks(g)[..., 0], -1)
    seg = torch.nn.functional.pad(seg.long(), (0, pad)) if not pad else torch.cat([seg.long(), seg[:, -1:].long().expand(b, pad)], 1)
    first = seg[:, :1] if s0 is not None else torch.full_like(seg[:, :1], -2)
    before = torch.cat([first, seg[:, c - 1::c][:, :-1]], 1)[:, None, :, None]
    seg = seg.reshape(b, 1, n, c)
    mask = (seg[..., :, None] == seg[..., None, :]) & torch.ones(c, c, dtype=torch.bool, device=q.device).tril()
    decay = torch.exp((gam[..., :, None] - gam[..., None, :]).masked_fill(~mask, -math.inf))
    kt = k.transpose(-1, -2).contiguous()
    inv = _Inverse.apply((beta * (k @ kt) * decay).tril(-1))
    grow = (torch.exp(gam) * (seg == before))[..., None]
    last = gam[..., -1:]
    kws = (torch.exp(last - gam) * (seg == seg[..., -1:]))[..., None]
    carry = (torch.exp(last) * (seg[..., -1:] == before))[..., None]
    w, u = inv @ (k * beta * grow), inv @ (v * beta)
    qk, qg, kw = (q @ kt) * decay, q * grow, (k * kws).transpose(-1, -2).contiguous()
    s = torch.zeros(b, h, d, d, dtype=q.dtype, device=q.device) if s0 is None else s0
    outs = []
    for i in range(n):
        vn = u[:, :, i] - w[:, :, i] @ s
        outs.append(qk[:, :, i] @ vn + qg[:, :, i] @ s)
        s = carry[:, :, i] * s + kw[:, :, i] @ vn
    return torch.stack(outs, 2).permute(0, 2, 3, 1, 4).reshape(b, n * c, h, d)[:, :t], s


def _l2norm64(x):
    sq = (x * x).sum(-1, keepdim=True)
    zero = sq == 0
    return torch.where(zero, torch.zeros_like(x), x * torch.rsqrt(torch.where(zero, torch.ones_like(sq), sq) + 1e-6))


def _mega64(case, qkv, a, b, a_log, dt_bias, conv, seg, s0=None, hist=None):
    """Conv, SiLU, l2norm, gates and the rule in fp64."""
    bt, t, hk, h, d = case["batch"], qkv.shape[1], case["hk"], case["h"], case["dim"]
    seg = seg.long()
    front = torch.zeros(bt, TAPS - 1, qkv.shape[-1], dtype=qkv.dtype, device=qkv.device) if hist is None else hist
    fseg = torch.full((bt, TAPS - 1), -1, device=seg.device) if hist is None else seg[:, :1].expand(bt, TAPS - 1)
    xp, sp = torch.cat([front, qkv], 1), torch.cat([fseg, seg], 1)
    z = 0
    for lag in range(TAPS):
        at = TAPS - 1 - lag
        z = z + (xp[:, at:at + t] * (sp[:, at:at + t] == seg)[..., None]) * conv[TAPS - 1 - lag]
    act = z * torch.sigmoid(z) * (seg > 0)[..., None]
    q, k, v = act.split([hk * d, hk * d, h * d], -1)
    q = _l2norm64(q.reshape(bt, t, hk, d)).repeat_interleave(h // hk, 2) * d ** -0.5
    k = _l2norm64(k.reshape(bt, t, hk, d)).repeat_interleave(h // hk, 2)
    g = -torch.exp(a_log) * torch.nn.functional.softplus(a + dt_bias)
    return _rule64(q, k, v.reshape(bt, t, h, d), g, torch.sigmoid(b), seg, s0)


def _norm64(x, gate, weight, seg):
    y = weight * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * gate * torch.sigmoid(gate)
    return y * (seg > 0)[..., None, None]


def exact(case, seed):
    kind = case["kind"]
    s = {n: x.double() if x.is_floating_point() else x for n, x in _inputs(case, seed).items()}
    if kind in ("decode", "prefill"):
        with torch.no_grad():
            qkv, a, b = (x[:, None] if kind == "decode" else x for x in (s["qkv"], s["a"], s["b"]))
            seg = s.get("seg", torch.ones(case["batch"], 1, dtype=torch.int32, device="cuda"))
            out, st = _mega64(case, qkv, a, b, s["a_log"], s["dt_bias"], s["conv"], seg, s.get("state"), s.get("hist"))
            rows = qkv if "hist" not in s else torch.cat([s["hist"], qkv], 1)
            hist = torch.nn.functional.pad(rows, (0, 0, TAPS - 1, 0))[:, -(TAPS - 1):]
            return {"out": out[:, 0] if kind == "decode" else out, "hist": hist, "state": st}
    if kind == "block":  # the layer's bf16 tensors (merged weights, projections, core output) as stored
        blk, h, d, st = _block(case, seed), case["h"], case["dim"], _Stored.apply
        ps, leaves = [], [s["x"].requires_grad_(True)]
        for p in blk.projections():
            la, lb = (w.detach().double().requires_grad_(True) for w in (p.lora_a, p.lora_b))
            leaves += [la, lb]
            ps.append(st(p.weight.double() + p.scale * (st(la) @ st(lb))))
        x = s["x"] * (s["seg"] > 0)[..., None]
        qkv, z, b, a = (st(x @ w) for w in ps[:4])
        out, _ = _mega64(case, qkv, a, b, blk.a_log.double(), blk.dt_bias.double(), blk.conv.double(), s["seg"])
        out = st(_norm64(st(out), z.reshape(out.shape), blk.norm_weight.double(), s["seg"]))
        out = out.reshape(*x.shape[:2], h * d) @ ps[4]
    else:
        leaves = [s[n].requires_grad_(True) for n in _leaf_names(case)]
        if kind == "v2":
            rep = case["h"] // case["hk"]
            out, _ = _rule64(s["q"].repeat_interleave(rep, 2), s["k"].repeat_interleave(rep, 2), s["v"], s["g"], s["beta"],
                             s["seg"])
        else:
            out, _ = _mega64(case, s["qkv"], s["a"], s["b"], s["a_log"], s["dt_bias"], s["conv"], s["seg"])
            out = _norm64(out, s["gate"], s["norm"], s["seg"])
    return {"out": out.detach(), "grads": list(torch.autograd.grad(out, leaves, s["dy"]))}
