"""The work a user has this framework do, as measurable cases.

Every case is one call of a public operator of `flash_spacetime_amd`, forward
alone (`"mode": "fwd"`: inference, validation) or forward and backward
(`"mode": "step"`: training), in one of the three layouts the operators take:

* `padded`: q, k, v `[B, H, L, D]` with `[B]` lengths
  (`flash_spacetime_attention`);
* `packed`: `[T, H, D]` with `cu_seqlens` (`flash_spacetime_attention_varlen`);
* `qkv`: one projection's output `[B, L, 3, H, D]`
  (`flash_spacetime_attention_qkv`).

A case is a dict of plain values:

    layout, mode, dtype ("bf16" / "f32"), heads, dim, channels,
    batch (events), length (the padded length, or the longest event),
    lens: how the events' lengths are spread over the batch --
      "full"       every event has `length` tokens,
      "uniform"    evenly over 16 .. length,
      "lognormal"  the quantiles of lognormal(5, 1) clipped to 1 .. length,
                   one event in 100 of length 1,
      "6000,137"   the lengths themselves (batch of them),
    attn, act: whether the pair bias enters the logits / the values,
    qk: factor on q and k (30 gives logits of order 1e4).

The multiset of lengths belongs to the case, so its work does not depend on
the seed; the seed draws every value and the order of the events.
"""

from __future__ import annotations

import math
import statistics
from typing import Dict, List, Optional, Tuple

import torch

TIME_SCALE = 18.0


def _case(name, layout, mode, dtype, batch, length, heads, dim, channels, lens, attn=True, act=True, qk=1.0):
    case = {"layout": layout, "mode": mode, "dtype": dtype, "batch": batch, "length": length, "heads": heads,
            "dim": dim, "channels": channels, "lens": lens, "attn": attn, "act": act, "qk": qk}
    if name:
        case["name"] = name
    return case


def listed() -> List[Dict]:
    return [
        # One event through one attention layer, as an event-by-event
        # reconstruction calls it: the smallest call, all latency.
        _case("one_event_fwd", "padded", "fwd", "bf16", 1, 187, 12, 32, 16, "full"),
        # A handful of short events in float32, forward and backward: a
        # debugging or fine-tuning step (B=4, L=64, H=2 of the CPU plumbing
        # configuration).
        _case("tiny_step_f32", "padded", "step", "f32", 4, 64, 2, 32, 16, "full"),
        # An online inference batch of packed events with ragged lengths.
        _case("serve_packed_fwd", "packed", "fwd", "bf16", 48, 768, 12, 32, 16, "lognormal"),
        # A training micro-batch at the 192-pulse cap with C = D = 32, through
        # the model's fused projection (SpacetimeAttention's layout).
        _case("qkv_step", "qkv", "step", "bf16", 64, 192, 12, 32, 32, "uniform"),
        # The headline configuration's forward (validation over a batch).
        _case("padded_fwd", "padded", "fwd", "bf16", 256, 768, 12, 32, 16, "uniform"),
        # The headline training step.
        _case("padded_step", "padded", "step", "bf16", 256, 768, 12, 32, 16, "uniform"),
        # The uncapped training step on packed events.
        _case("packed_step", "packed", "step", "bf16", 4096, 3000, 12, 32, 16, "lognormal"),
        # Few very long packed events beside a short one, many heads.
        _case("uncapped_step", "packed", "step", "bf16", 3, 6000, 16, 48, 48, "6000,137,1503"),
        # Wide heads, long events, peaked logits.
        _case("long_step", "padded", "step", "bf16", 8, 4096, 8, 64, 64, "full", qk=30.0),
        # The headline shape in float32 (a smaller batch), forward and backward.
        _case("padded_step_f32", "padded", "step", "f32", 32, 768, 12, 32, 16, "uniform"),
        # Wide heads and long events in float32.
        _case("long_step_f32", "padded", "step", "f32", 4, 4096, 8, 64, 64, "full"),
    ]


def _pair_flops(case) -> float:
    """Operations per valid (query, key, head): forward, or forward and backward."""
    d, c = case["dim"], case["channels"]
    return 4 * (d + c) + (10 * d + 8 * c if case["mode"] == "step" else 0)


def _logint(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> Dict:
    largest = max(work(c)["flops"] for c in listed())
    while True:
        layout = rng.choice(["padded", "padded", "packed", "packed", "qkv"])
        mode = rng.choice(["fwd", "step", "step"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        heads = rng.choice([1, 2, 4, 6, 8, 8, 12, 12, 12, 16])
        dim, channels = rng.choice([(32, 16), (32, 16), (32, 32), (16, 16), (48, 48), (64, 64), (64, 16)])
        length = _logint(rng, 24, 3000)
        batch = _logint(rng, 1, 1024)
        lens = rng.choice(["full", "uniform", "uniform"] if layout != "packed" else ["uniform", "lognormal"])
        attn, act = rng.choice([(True, True)] * 4 + [(True, False), (False, True)])
        case = _case("", layout, mode, dtype, batch, length, heads, dim, channels, lens, attn, act)
        tokens = batch * length
        if tokens <= 250_000 and work(case)["flops"] * (4 if dtype == "f32" else 1) <= 0.5 * largest:
            return case


def lengths(case) -> List[int]:
    """The events' lengths (the order is drawn with the inputs)."""
    b, top, lens = case["batch"], case["length"], case["lens"]
    if lens == "full":
        return [top] * b
    if lens == "uniform":
        lo = min(16, top)
        return [lo + int((top + 1 - lo) * (i + 0.5) / b) for i in range(b)]
    if lens == "lognormal":
        normal = statistics.NormalDist(5.0, 1.0)
        out = [max(1, min(top, int(round(math.exp(normal.inv_cdf((i + 0.5) / b)))))) for i in range(b)]
        for i in range(-(-b // 100)):
            out[i] = 1
        return out
    return [int(x) for x in lens.split(",")]


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _inputs(case, seed: int) -> Dict[str, torch.Tensor]:
    """Operands on the GPU. Features are what the model feeds the layer after
    its standardisation (about N(0, 1), where part of the pairs reach the
    angle's clip and part do not) with one column the operator ignores."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    host = torch.Generator().manual_seed(seed)
    h, d, c, dt = case["heads"], case["dim"], case["channels"], _dtype(case)
    lens = torch.tensor(lengths(case), dtype=torch.int32)
    lens = lens[torch.randperm(len(lens), generator=host)]
    total = int(lens.sum())
    lead = (total,) if case["layout"] == "packed" else (case["batch"], case["length"])

    def rn(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    x: Dict[str, torch.Tensor] = {}
    if case["layout"] == "qkv":
        qkv = rn(*lead, 3, h, d)
        qkv[:, :, :2] *= case["qk"]
        x["qkv"] = qkv.to(dt)
        do_shape = (*lead, h, d)
    else:
        do_shape = (total, h, d) if case["layout"] == "packed" else (case["batch"], h, case["length"], d)
        x["q"] = (rn(*do_shape) * case["qk"]).to(dt)
        x["k"] = (rn(*do_shape) * case["qk"]).to(dt)
        x["v"] = rn(*do_shape).to(dt)
    x["feats"] = rn(*lead, 5)
    x["w"] = rn(d, c) / c ** 0.5
    x["b"] = rn(d) * 0.02
    if case["mode"] == "step":
        x["do"] = rn(*do_shape).to(dt)
    if case["layout"] == "packed":
        cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
        cu[1:] = torch.cumsum(lens, 0)
        x["cu"] = cu.to(dev)
    else:
        x["lens"] = lens.to(dev)
    return x


def prepare(case, seed: int) -> Dict:
    x = _inputs(case, seed)
    state = {"case": case, "x": x}
    if case["mode"] == "step":
        for name in ("q", "k", "v", "qkv", "w", "b"):
            if name in x:
                x[name].requires_grad_(True)
    return state


def run(state):
    """One forward, or one forward and backward: the output and the gradients
    of q, k, v (or qkv), W and b."""
    from flash_spacetime_amd import (
        flash_spacetime_attention,
        flash_spacetime_attention_qkv,
        flash_spacetime_attention_varlen,
    )

    case, x = state["case"], state["x"]
    flags = (case["attn"], case["act"])
    if case["layout"] == "packed":
        leaves = [x["q"], x["k"], x["v"], x["w"], x["b"]]
        out = flash_spacetime_attention_varlen(x["q"], x["k"], x["v"], x["feats"], x["w"], x["b"], x["cu"], None,
                                               *flags)
    elif case["layout"] == "qkv":
        leaves = [x["qkv"], x["w"], x["b"]]
        out = flash_spacetime_attention_qkv(x["qkv"], x["feats"], x["w"], x["b"], x["lens"], None, *flags)
    else:
        leaves = [x["q"], x["k"], x["v"], x["w"], x["b"]]
        out = flash_spacetime_attention(x["q"], x["k"], x["v"], x["feats"], x["w"], x["b"], x["lens"], None, *flags)
    if case["mode"] == "fwd":
        return [out]
    return [out.detach(), *torch.autograd.grad(out, leaves, x["do"])]


def work(case) -> Dict[str, float]:
    """Each valid row read once, every row of the outputs written once (padding
    rows are zeros the operator writes), and the algorithm's products over the
    valid pairs."""
    lens = lengths(case)
    h, d, c = case["heads"], case["dim"], case["channels"]
    esz = 2 if case["dtype"] == "bf16" else 4
    valid = sum(lens)
    rows = valid if case["layout"] == "packed" else case["batch"] * case["length"]
    pairs = float(sum(n * n for n in lens))
    small = 4 * (d * c + d)
    nbytes = valid * (3 * h * d * esz + 16) + rows * h * d * esz + small
    if case["mode"] == "step":
        nbytes += valid * h * d * esz + 3 * rows * h * d * esz + small
    return {"bytes": float(nbytes), "flops": pairs * h * _pair_flops(case)}


def tolerance(case) -> Dict[str, float]:
    """About four times the largest distance from the 64-bit result seen over
    the outputs. bf16: 4e-3 (2e-2 where logits of order 1e4 are formed from
    bf16 operands). float32: 1e-5 to 4e-5, growing with the channels and the
    length (the hardware's sine and cosine)."""
    if case["dtype"] == "bf16":
        return {"rel": 3e-2 if case["qk"] > 1 else 1.5e-2}
    return {"rel": 1.6e-4}


# ---------------------------------------------------------------------------
# The same results in 64 bits: the operator's definition, row block by row
# block, with its gradients written out.
# ---------------------------------------------------------------------------


def _frequencies(c: int, dev) -> torch.Tensor:
    """The spec's float32 ladder exp(-i ln(1e4) / (C/2)), correctly rounded."""
    i = torch.arange(c // 2, dtype=torch.float64, device=dev)
    return torch.exp(-i * (math.log(1e4) / (c / 2))).to(torch.float32).double()


def _event(q, k, v, pos, w, b, do, attn, act, freq) -> Tuple[torch.Tensor, ...]:
    """Output and gradients of one event; q, k, v, do are `[H, n, D]` float64."""
    h, n, d = q.shape
    c = w.shape[1]
    scale = d ** -0.5
    qt = q * scale
    out = torch.empty_like(q)
    grads = None
    if do is not None:
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        dw, db = torch.zeros_like(w), torch.zeros_like(b)
    block = max(16, min(n, int(4e8 / (n * max(c, h)))))
    for r0 in range(0, n, block):
        r1 = min(n, r0 + block)
        diff = pos[r0:r1, None, :] - pos[None, :, :]
        interval = diff[..., :3].pow(2).sum(-1) - (diff[..., 3] * TIME_SCALE).pow(2)
        x = 1024.0 * (torch.sign(interval) * interval.abs().sqrt()).clamp(-4.0, 4.0)
        theta = x[..., None] * freq
        e = torch.cat((theta.sin(), theta.cos()), -1)  # [rows, n, C]
        del diff, interval, x, theta
        qi = qt[:, r0:r1]
        s = qi @ k.transpose(1, 2)
        if attn:
            u = (qi @ w).transpose(0, 1).contiguous()  # [rows, H, C]
            s = s + (torch.bmm(u, e.transpose(1, 2).contiguous()).transpose(0, 1) + (qi @ b)[..., None])
        p = s.softmax(-1)
        del s
        o = p @ v
        pt = p.transpose(0, 1).contiguous()  # [rows, H, n]
        g = torch.bmm(pt, e).transpose(0, 1)  # [H, rows, C]
        if act:
            o = o + g @ w.t() + b
        out[:, r0:r1] = o
        if do is None:
            continue
        di = do[:, r0:r1]
        dp = di @ v.transpose(1, 2)
        if act:
            wt = (di @ w).transpose(0, 1).contiguous()
            dp = dp + torch.bmm(wt, e.transpose(1, 2).contiguous()).transpose(0, 1)
            db += di.sum((0, 1))
            dw += torch.einsum("hid,hic->dc", di, g)
        dp -= (p * dp).sum(-1, keepdim=True)
        ds = p * dp
        del dp
        dqt = ds @ k
        if attn:
            hh = torch.bmm(ds.transpose(0, 1).contiguous(), e).transpose(0, 1)
            dqt = dqt + hh @ w.t()
            dw += torch.einsum("hid,hic->dc", qi, hh)
        dq[:, r0:r1] = dqt * scale
        dk += ds.transpose(1, 2).contiguous() @ qi
        dv += p.transpose(1, 2).contiguous() @ di
    if do is not None:
        grads = (dq, dk, dv, dw, db)
    return out, grads


def exact(case, seed: int) -> Optional[List[torch.Tensor]]:
    x = _inputs(case, seed)
    dev = x["w"].device
    layout, step = case["layout"], case["mode"] == "step"
    h, d = case["heads"], case["dim"]
    w, b = x["w"].double(), x["b"].double()
    freq = _frequencies(case["channels"], dev)
    # Heads-last views [.., H, D] of every operand, events as row ranges.
    if layout == "qkv":
        q, k, v = (x["qkv"][:, :, i] for i in range(3))
        do = x.get("do")
    elif layout == "padded":
        q, k, v = (x[t].transpose(1, 2) for t in "qkv")
        do = x["do"].transpose(1, 2) if step else None
    else:
        q, k, v, do = x["q"], x["k"], x["v"], x.get("do")
    out = torch.zeros(q.shape, dtype=torch.float64, device=dev)
    dq, dk, dv = (torch.zeros_like(out) for _ in range(3)) if step else (None, None, None)
    dw, db = torch.zeros_like(w), torch.zeros_like(b)
    if layout == "packed":
        cu = x["cu"].tolist()
        spans = [slice(a, z) for a, z in zip(cu[:-1], cu[1:])]
    else:
        spans = [(i, slice(0, n)) for i, n in enumerate(x["lens"].tolist())]
    for at in spans:
        rows = lambda t: t[at].transpose(0, 1).double()  # noqa: E731  [H, n, D]
        if q[at].shape[0] == 0:
            continue
        o, grads = _event(rows(q), rows(k), rows(v), x["feats"][at][..., :4].double(), w, b,
                          rows(do) if step else None, case["attn"], case["act"], freq)
        out[at] = o.transpose(0, 1)
        if step:
            for full, part in zip((dq, dk, dv), grads):
                full[at] = part.transpose(0, 1)
            dw += grads[3]
            db += grads[4]
    if layout == "padded":
        out = out.transpose(1, 2)
    if not step:
        return [out]
    if layout == "qkv":
        return [out, torch.stack((dq, dk, dv), 2), dw, db]
    if layout == "padded":
        dq, dk, dv = (t.transpose(1, 2) for t in (dq, dk, dv))
    return [out, dq, dk, dv, dw, db]
