"""GPU tests of the operators' native host path (csrc/fst_host.cpp).

The host extension takes the forms of a call it knows and leaves every other
to the Python path. Each form below, taken or not, must give the results of
the Python path bit for bit (the same kernels run on the same operands):
layouts and strides of q, k, v and of the upstream gradient, dtypes of
lengths, features, weight and bias, absent bias, head groups, both dtypes.
What the Python path refuses stays refused with its exception.
"""

import ctypes

import pytest
import torch

from flash_spacetime_amd import _lib

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from flash_spacetime_amd import (
        backward, flash_spacetime_attention, flash_spacetime_attention_qkv, flash_spacetime_attention_varlen, forward,
        flash_spacetime_backward, flash_spacetime_forward, tune,
    )

DEV = "cuda"
B, L, D, C = 3, 37, 32, 16
LENS = [37, 16, 1]


def _draw(*shape, dtype=torch.bfloat16, seed=0):
    gen = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=gen).to(DEV, dtype)


# name -> dict of changes to the plain padded bf16 call
FORMS = {
    "plain": {},
    "float32": {"dtype": torch.float32},
    "token_major": {"layout": "token_major"},
    "one_head_token_major": {"layout": "token_major", "heads": 1},
    "sliced": {"layout": "sliced"},          # strides of a larger tensor
    "mixed": {"layout": "mixed"},            # q token-major, k and v dense
    "int64_lengths": {"lens": torch.int64},
    "int16_lengths": {"lens": torch.int16},
    "cpu_lengths": {"lens_dev": "cpu"},
    "four_features": {"feats": 4},
    "float64_features": {"feats_dtype": torch.float64},
    "strided_features": {"feats_strided": True},
    "bf16_weight": {"w_dtype": torch.bfloat16},
    "transposed_weight": {"w_t": True},
    "no_bias": {"bias": False},
    "no_act": {"flags": (True, False)},
    "no_attn": {"flags": (False, True)},
    "scale": {"scale": 0.3},
    "head_groups": {"heads": 17},
    "expanded_grad": {"grad": "expanded"},
    "token_major_grad": {"grad": "token_major"},
    "packed": {"layout": "packed"},
    "packed_strided": {"layout": "packed_strided"},
    "packed_int64": {"layout": "packed", "lens": torch.int64},
    "qkv": {"layout": "qkv"},
    "qkv_packed": {"layout": "qkv_packed"},
    "qkv_float32": {"layout": "qkv", "dtype": torch.float32},
    "qkv_expanded_grad": {"layout": "qkv", "grad": "expanded"},
}


def _run(form):
    o = {"dtype": torch.bfloat16, "heads": 4, "layout": "dense", "lens": torch.int32, "lens_dev": DEV, "feats": 5,
         "feats_dtype": torch.float32, "w_dtype": torch.float32, "bias": True, "flags": (True, True), "scale": None,
         "grad": "dense", "feats_strided": False, "w_t": False, **FORMS[form]}
    h, dt, lay, t = o["heads"], o["dtype"], o["layout"], sum(LENS)
    packed = lay in ("packed", "packed_strided", "qkv_packed")
    lead = (t,) if packed else (B, L)
    if lay in ("qkv", "qkv_packed"):
        ops = [_draw(*lead, 3, h, D, dtype=dt)]
    elif lay == "packed":
        ops = [_draw(t, h, D, dtype=dt, seed=i) for i in range(3)]
    elif lay == "packed_strided":
        ops = [_draw(t, h, D + 16, dtype=dt, seed=i)[..., :D] for i in range(3)]
    elif lay == "token_major":
        ops = [_draw(B, L, h, D, dtype=dt, seed=i).transpose(1, 2) for i in range(3)]
    elif lay == "mixed":
        ops = [_draw(B, L, h, D, dtype=dt).transpose(1, 2)] + [_draw(B, h, L, D, dtype=dt, seed=i) for i in (1, 2)]
    elif lay == "sliced":
        ops = [_draw(B, h, L + 3, D, dtype=dt, seed=i)[:, :, 1:L + 1] for i in range(3)]
    else:
        ops = [_draw(B, h, L, D, dtype=dt, seed=i) for i in range(3)]
    feats = _draw(*lead, o["feats"] + (3 if o["feats_strided"] else 0), dtype=o["feats_dtype"])
    feats = feats[..., 2:2 + o["feats"]] if o["feats_strided"] else feats
    w = (_draw(C, D, dtype=o["w_dtype"]).t() if o["w_t"] else _draw(D, C, dtype=o["w_dtype"])) / 4
    b = _draw(D, dtype=o["w_dtype"]) * 0.02 if o["bias"] else None
    lens = torch.tensor(LENS)
    if packed:
        lens = torch.cat([torch.zeros(1, dtype=lens.dtype), lens.cumsum(0)])
    lens = lens.to(o["lens_dev"], o["lens"])
    leaves = [x.detach().requires_grad_(True) for x in ops + [w] + ([b] if b is not None else [])]
    xs, wl, bl = leaves[:len(ops)], leaves[len(ops)], leaves[len(ops) + 1] if b is not None else None
    if lay == "qkv":
        out = flash_spacetime_attention_qkv(xs[0], feats, wl, bl, lens, o["scale"], *o["flags"])
    elif lay == "qkv_packed":
        out = flash_spacetime_attention_qkv(xs[0], feats, wl, bl, None, o["scale"], *o["flags"], cu_seqlens=lens)
    elif packed:
        out = flash_spacetime_attention_varlen(*xs, feats, wl, bl, lens, o["scale"], *o["flags"])
    else:
        out = flash_spacetime_attention(*xs, feats, wl, bl, lens, o["scale"], *o["flags"])
    g = _draw(*out.shape, dtype=dt, seed=9)
    if o["grad"] == "expanded":
        g = _draw(D, dtype=dt, seed=9).expand(out.shape)
    elif o["grad"] == "token_major":
        g = _draw(B, L, h, D, dtype=dt, seed=9).transpose(1, 2)
    grads = torch.autograd.grad(out, leaves, g, allow_unused=True)
    res = [out.detach(), *grads]
    if lay == "dense":
        kw = dict(scale=o["scale"], use_attn_bias=o["flags"][0], use_activation_bias=o["flags"][1])
        fo, lse = flash_spacetime_forward(*[x.detach() for x in xs], feats, w, b, lens, **kw)
        res += [fo, lse, *flash_spacetime_backward(*[x.detach() for x in xs], feats, w, b, lens, lse, g, **kw)]
    torch.cuda.synchronize()
    return res


@pytest.mark.parametrize("form", FORMS)
def test_native_path_equals_the_python_path(form, monkeypatch):
    got = _run(form)
    monkeypatch.setattr(forward, "_native_forward", lambda *a, **k: None)
    monkeypatch.setattr(backward, "_native_backward", lambda *a, **k: None)
    want = _run(form)
    assert len(got) == len(want)
    for i, (a, e) in enumerate(zip(got, want)):
        assert (a is None) == (e is None), i
        if a is not None:
            assert a.dtype == e.dtype and a.shape == e.shape and a.stride() == e.stride(), i
            assert torch.equal(a, e), i


@pytest.mark.parametrize("layout", ["dense", "token_major", "packed"])
def test_gradient_of_another_dtype(layout):
    """A float32 upstream gradient of bf16 operands (autograd casts it before it
    gets here) is converted, and the forward's output handed on, as the Python
    path does."""
    lead = (sum(LENS), 4) if layout == "packed" else (B, 4, L)
    q, k, v = (_draw(*lead, D, seed=i) for i in range(3))
    g = _draw(*lead, D, dtype=torch.float32, seed=9)
    if layout == "token_major":
        q, k, v = (_draw(B, L, 4, D, seed=i).transpose(1, 2) for i in range(3))
    lens = torch.tensor([0, 37, 53, 54] if layout == "packed" else LENS, device=DEV)
    feats = _draw(*((sum(LENS),) if layout == "packed" else (B, L)), 5, dtype=torch.float32)
    w, b = _draw(D, C, dtype=torch.float32) / 4, _draw(D, dtype=torch.float32) * 0.02
    out, lse, qc, kc, vc, pos4, w32, b32, len32, dims, scale = forward._native_forward(
        q, k, v, feats, w, b, lens, None, True, True, layout == "packed")
    args = (dims, qc, kc, vc, pos4, w32, b32, len32, lse, g, scale)
    got = backward._native_backward(*args, out)
    want = backward._run_backward(*args, forward.vec_shape(dims), out=out)
    same = backward._native_backward(*args[:9], g.bfloat16(), scale, out)
    for a, e, s in zip(got, want, same):
        assert a.dtype == e.dtype and a.stride() == e.stride()
        assert torch.equal(a, e) and torch.equal(a, s)


def test_the_usual_forms_take_the_native_path(monkeypatch):
    """The forms a model gives run natively, in both directions."""
    calls = []
    nf, nb = forward._native_forward, backward._native_backward
    monkeypatch.setattr(forward, "_native_forward", lambda *a, **k: (lambda r: (calls.append(r is not None), r)[1])(nf(*a, **k)))
    monkeypatch.setattr(backward, "_native_backward", lambda *a, **k: (lambda r: (calls.append(r is not None), r)[1])(nb(*a, **k)))
    for form in ("plain", "float32", "token_major", "int64_lengths", "no_bias", "packed", "qkv", "qkv_packed"):
        calls.clear()
        _run(form)
        assert calls and all(calls), form
    with tune.fixed_plan(1 << 8):  # a plan of the caller's is the Python path's
        calls.clear()
        _run("packed")
        assert calls and not any(calls)


def test_operators_run_without_the_extension(monkeypatch):
    want = {form: _run(form) for form in ("plain", "packed", "qkv")}
    monkeypatch.setattr(_lib, "_HOST", False)  # as _lib.host leaves it for an unusable extension
    for form, res in want.items():
        assert all(torch.equal(a, e) for a, e in zip(_run(form), res)), form


def test_refused_calls_stay_refused():
    q, k, v = (_draw(B, 4, L, D, seed=i) for i in range(3))
    feats, w, b = _draw(B, L, 5, dtype=torch.float32), _draw(D, C, dtype=torch.float32), None
    lens = torch.tensor(LENS, device=DEV)
    bad = [
        ((q, k, v, feats, _draw(D, 24, dtype=torch.float32), b, lens), "supports C"),
        ((q, k[:, :, :5], v, feats, w, b, lens), "same shape"),
        ((q, k.float(), v, feats, w, b, lens), "one dtype"),
        ((q, k, v, feats[..., :3], w, b, lens), "4 columns"),
        ((q, k, v, feats, w, _draw(5, dtype=torch.float32), lens), "bias must be"),
        ((q, k, v, feats, w, b, lens.float()), "integer"),
        ((q, k, v, feats, w, b, lens[:2]), "seqlens must be"),
        ((q.double(), k.double(), v.double(), feats, w, b, lens), "bfloat16 or float32"),
        ((q, k, v, feats, w, b, lens, float("inf")), "finite"),
    ]
    for args, what in bad:
        with pytest.raises(ValueError, match=what):
            flash_spacetime_attention(*args)
    with pytest.raises(ValueError, match="require grad"):
        flash_spacetime_attention(q, k, v, feats.clone().requires_grad_(True), w, b, lens)
    with pytest.raises(RuntimeError, match="GPU"):
        flash_spacetime_attention(q.cpu(), k, v, feats, w, b, lens)
    with pytest.raises((AttributeError, TypeError, ValueError)):
        flash_spacetime_attention_varlen(_draw(sum(LENS), 3, 4, D), None, None, _draw(sum(LENS), 5, dtype=torch.float32),
                                         w, b, torch.tensor([0, 54], device=DEV, dtype=torch.int32))


# The library's entry points replaced by host functions that return a status
# (nothing is launched): what the operators make of it.
_ENTRY = ("fst_supported", "fst_forward_workspace_bytes", "fst_forward", "fst_backward_workspace_bytes",
          "fst_backward", "fst_last_error")


def _bind(**stubs):
    lib = _lib.load()
    _lib.host().bind_library(*(ctypes.cast(stubs.get(n, getattr(lib, n)), ctypes.c_void_p).value for n in _ENTRY))


def _returning(name, status, calls):
    res, args = _lib.SIGNATURES[name]

    def entry(*_):
        calls.append(name)
        return status

    return ctypes.CFUNCTYPE(res, *args)(entry)


@pytest.mark.parametrize("name", ["fst_forward", "fst_backward"])
@pytest.mark.parametrize("status", [_lib.FST_ELAUNCH, _lib.FST_EWORKSPACE, _lib.FST_EUNSUPPORTED, _lib.FST_EINVAL])
def test_failed_calls_raise_and_refused_ones_take_the_python_path(name, status):
    """A launch error is reported, not hidden by a second run of the call; a
    call the library refuses is left to the Python path (which here runs it)."""
    calls, want = [], _run("packed")
    stub = _returning(name, status, calls)
    try:
        _bind(**{name: stub})
        if status in (_lib.FST_ELAUNCH, _lib.FST_EWORKSPACE):
            with pytest.raises(RuntimeError, match="flash_spacetime_" + name[4:]):
                _run("packed")
        else:
            assert all(torch.equal(a, e) for a, e in zip(_run("packed"), want))
    finally:
        _bind()
    assert calls == [name]
    assert all(torch.equal(a, e) for a, e in zip(_run("packed"), want))
