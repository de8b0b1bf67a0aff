"""GPU tests of the phases of a call run one by one.

After a call of all phases at once on a workspace, the later phases run on it
again by themselves must give the same bits, in the forward and the backward,
for calls of up to 64 events (which leave the work list unwritten) and more,
padded and packed, with the dW / db sums in the cols kernel's launch and in
launches of their own. The workspaces start as zeros, which a kernel that
read an unwritten list would take for a list of no work.

Up to 64 events of few tiles the kernels form the work list themselves; with
empty events appended past 64 the work-list kernel writes it. The events' rows must be the
same bits either way, and so must dW and db (an empty event adds zeros after
the others' partial sums). Malformed packed offsets must be refused alike.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from flash_spacetime_amd import _lib
    from flash_spacetime_amd.forward import _Prepared

DEV = "cuda"
LENS64 = [((11 * i) % 40) * (i % 6 != 2) for i in range(64)]
# (dtype, heads, dim, channels, lengths, packed)
CASES = [
    (torch.bfloat16, 8, 64, 64, [49, 16, 0, 1], False),
    (torch.bfloat16, 12, 32, 16, [33, 0, 17], True),
    (torch.bfloat16, 3, 16, 16, LENS64, False),
    (torch.bfloat16, 2, 16, 16, LENS64 + [5], True),       # 65 events: a written list
    (torch.bfloat16, 2, 16, 16, [300] * 60, False),        # too many tiles: a written list, dW / db in launches of their own
    (torch.bfloat16, 4, 16, 16, [700, 40, 0, 655, 16] * 3, False),  # padding-only tiles of many lengths
    (torch.bfloat16, 2, 16, 16, [1000] + LENS64[1:], True),
    (torch.float32, 12, 32, 16, [40, 0, 7], False),
    (torch.float32, 4, 16, 32, LENS64, True),
]
NAMES = ["out", "lse", "rowsum", "dq", "dk", "dv", "dW", "db"]


class Call:
    """One call's operands, outputs and workspaces; `empty` empty events follow
    the lengths given."""

    def __init__(self, dtype, heads, dim, chans, lens, packed, empty=0, cu=None):
        gen = torch.Generator().manual_seed(len(lens) + dim)
        n, total, top = len(lens), sum(lens), max(max(lens), 1)
        lead = (total, heads) if packed else (n, heads, top)

        def rn(*shape, dt=torch.float32):
            x = torch.randn(*shape, generator=gen)
            if empty and not packed:
                x = torch.cat([x, torch.ones(empty, *shape[1:])])
            return x.to(DEV, dt)

        q, k, v, self.do = (rn(*lead, dim, dt=dtype) for _ in range(4))
        feats = rn(total, 4) if packed else rn(n, top, 4)
        w = torch.randn(dim, chans, generator=gen).to(DEV) / chans ** 0.5
        b = torch.randn(dim, generator=gen).to(DEV) * 0.02
        seq = torch.tensor(lens + [0] * empty, dtype=torch.int32)
        offsets = torch.zeros(len(seq) + 1, dtype=torch.int32)
        offsets[1:] = torch.cumsum(seq, 0)
        if cu is not None:
            offsets = torch.tensor(cu + cu[-1:] * empty, dtype=torch.int32)
        self.prep = _Prepared(q, k, v, feats, w, b, None if packed else seq.to(DEV), None, True, True,
                              offsets.to(DEV) if packed else None)
        self.dims = self.prep.dims()
        lib = _lib.load()
        self.fws = torch.zeros(lib.fst_forward_workspace_bytes(*self.dims), device=DEV, dtype=torch.uint8)
        self.bws = torch.zeros(lib.fst_backward_workspace_bytes(*self.dims), device=DEV, dtype=torch.uint8)
        self.n, self.packed = n, packed
        self.lse = torch.zeros(self.prep.vec_shape(), device=DEV)
        self.out, self.dq, self.dk, self.dv = (torch.zeros_like(self.prep.q) for _ in range(4))
        self.rowsum, self.dw, self.db = torch.zeros_like(self.lse), torch.zeros_like(w), torch.zeros_like(b)

    def outputs(self):
        return [self.out, self.lse, self.rowsum, self.dq, self.dk, self.dv, self.dw, self.db]

    def forward(self, phases):
        p, P = self.prep, _lib.ptr
        _lib.check(_lib.load().fst_forward_phases(
            phases, *self.dims, P(p.q), P(p.k), P(p.v), P(p.pos4), P(p.weight), P(p.bias), P(p.lens), p.scale,
            P(self.out), P(self.lse), P(self.fws), self.fws.numel(), torch.cuda.current_stream().cuda_stream), "forward")

    def backward(self, phases):
        p, P = self.prep, _lib.ptr
        _lib.check(_lib.load().fst_backward_phases(
            phases, *self.dims, P(p.q), P(p.k), P(p.v), P(p.pos4), P(p.weight), P(p.bias), P(p.lens), P(self.lse),
            P(self.do), P(self.out), p.scale, P(self.dq), P(self.dk), P(self.dv), P(self.dw), P(self.db),
            P(self.rowsum), P(self.bws), self.bws.numel(), torch.cuda.current_stream().cuda_stream), "backward")


@pytest.mark.parametrize("case", range(len(CASES)))
def test_later_phases_after_a_whole_call(case):
    print(CASES[case][:4], len(CASES[case][4]), "packed" if CASES[case][5] else "padded", flush=True)
    call = Call(*CASES[case])
    call.forward(_lib.FST_FWD_ALL)
    call.backward(_lib.FST_BWD_ALL)
    want = [x.clone() for x in call.outputs()]
    for x in call.outputs():
        x.fill_(float("nan"))
    call.forward(_lib.FST_PHASE_FWD)
    for phase in (_lib.FST_PHASE_BWD_ROWS, _lib.FST_PHASE_BWD_COLS, _lib.FST_PHASE_REDUCE):
        call.backward(phase)
    torch.cuda.synchronize()
    for name, a, e in zip(NAMES, call.outputs(), want):
        assert torch.isfinite(e).all(), name
        assert torch.equal(a, e), name


@pytest.mark.parametrize("case", [i for i, c in enumerate(CASES) if len(c[4]) <= 64])
def test_list_formed_by_the_waves_equals_the_written_one(case):
    print(CASES[case][:4], len(CASES[case][4]), "packed" if CASES[case][5] else "padded", flush=True)
    few, many = Call(*CASES[case]), Call(*CASES[case], empty=65 - len(CASES[case][4]))
    for call in (few, many):
        call.forward(_lib.FST_FWD_ALL)
        call.backward(_lib.FST_BWD_ALL)
    torch.cuda.synchronize()
    for name, a, e in zip(NAMES, few.outputs(), many.outputs()):
        if not few.packed and name not in ("dW", "db"):
            assert (e[few.n:] == 0).all(), name
            e = e[:few.n]
        assert torch.equal(a, e), name


@pytest.mark.parametrize("cu", [[0, 20, 10, 50], [5, 20, 30, 50], [0, 20, 30, 60], [0, -3, 30, 50]],
                         ids=["decreasing", "start", "past-the-end", "negative"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_malformed_offsets_with_and_without_a_written_list(cu, dtype):
    args = (dtype, 4, 32, 16, [20, 10, 20], True)
    few, many = Call(*args, cu=cu), Call(*args, empty=62, cu=cu)
    for call in (few, many):
        call.forward(_lib.FST_FWD_ALL)
        call.backward(_lib.FST_BWD_ALL)
    torch.cuda.synchronize()
    for name, a, e in zip(NAMES, few.outputs(), many.outputs()):
        assert torch.equal(a.isnan(), e.isnan()), name
        assert torch.equal(a.nan_to_num(), e.nan_to_num()), name
        if name in ("out", "dW", "db"):
            assert a.isnan().any(), name
