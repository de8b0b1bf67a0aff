"""GPU tests of calls of few events, which run without a work-list kernel.

A whole forward or backward call of at most 64 events (and few tiles) has every
workgroup form the lists it needs (event order, tile counts, sanitised
offsets) and, for at most 1024 tiles, sums dW / db in the cols kernel's launch; the same
phases issued one by one form the same lists (else read them) and
reduce in the same order in launches of their own. Both must give the same
bits: around the 64-event line (63, 64, 65), with empty and one-token events,
padded and packed, both dtypes, and with malformed packed offsets (NaN from
both). test_phase_order_gpu.py compares the lists the workgroups form with
those the work-list kernel writes. Each width of
the reduction's workgroups (up to 4, 8 and 16 runs of 64 tiles), and the calls
past it (more runs, or more workgroups than CUs), are checked the same way.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from flash_spacetime_amd import _lib
    from flash_spacetime_amd.forward import _Prepared

DEV = "cuda"
# (dtype, heads, dim, channels, lengths, packed); padded to the longest.
LENS64 = [((7 * i) % 50) * (i % 5 != 3) for i in range(64)]
CASES = [
    (torch.bfloat16, 12, 32, 16, [187], False),
    (torch.bfloat16, 3, 16, 16, LENS64, False),
    (torch.bfloat16, 3, 16, 16, LENS64[:63], True),
    (torch.bfloat16, 4, 32, 32, LENS64, True),
    (torch.bfloat16, 4, 32, 16, LENS64 + [33], True),     # 65 events: the work-list kernel either way
    (torch.bfloat16, 8, 32, 16, [0, 16, 1, 17, 33, 0, 48, 2, 15], False),
    (torch.bfloat16, 8, 48, 48, [1, 0, 40], True),
    (torch.bfloat16, 2, 16, 16, [300] * 60, False),       # more than 1024 tiles
    (torch.bfloat16, 4, 16, 32, [200] * 20 + [1], False),  # 261 tiles: 5 runs
    (torch.bfloat16, 2, 48, 16, [250] * 32, True),         # 512 tiles: 8 runs
    (torch.bfloat16, 2, 16, 48, [190, 0, 200] * 15, False),  # 375 tiles: 6 runs
    (torch.bfloat16, 2, 64, 48, [256] * 64, False),        # 1024 tiles: 16 runs, 200 workgroups
    (torch.bfloat16, 2, 64, 64, [256] * 33, True),         # 9 runs, too many workgroups
    (torch.float32, 2, 16, 32, [250] * 40, False),
    (torch.float32, 8, 64, 64, [33] * 5, True),
    (torch.float32, 4, 16, 16, [0, 31, 1, 17], False),
    (torch.float32, 8, 32, 16, LENS64, True),
    (torch.float32, 12, 32, 16, [64, 0, 5], False),
]


def _call(whole, dtype, heads, dim, chans, lens, packed, cu=None):
    gen = torch.Generator().manual_seed(len(lens) + dim)
    rn = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    total, top = sum(lens), max(max(lens), 1)
    lead = (total, heads) if packed else (len(lens), heads, top)
    q, k, v, do = (rn(*lead, dim).to(DEV, dtype) for _ in range(4))
    feats = rn(total, 4) if packed else rn(len(lens), top, 4)
    w, b = (rn(dim, chans) / chans ** 0.5).to(DEV), (rn(dim) * 0.02).to(DEV)
    off = torch.zeros(len(lens) + 1, dtype=torch.int32)
    off[1:] = torch.cumsum(torch.tensor(lens), 0)
    if cu is not None:
        off = torch.tensor(cu, dtype=torch.int32)
    seq = torch.tensor(lens, dtype=torch.int32)
    prep = _Prepared(q, k, v, feats.to(DEV), w, b, None if packed else seq.to(DEV), None, True, True,
                     off.to(DEV) if packed else None)
    lib, dims, P = _lib.load(), prep.dims(), _lib.ptr
    out, lse = torch.zeros_like(prep.q), torch.zeros(prep.vec_shape(), device=DEV)
    rowsum = torch.zeros_like(lse)
    dq, dk, dv = (torch.zeros_like(prep.q) for _ in range(3))
    dw, db = torch.zeros(dim, chans, device=DEV), torch.zeros(dim, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    fb, bb = lib.fst_forward_workspace_bytes(*dims), lib.fst_backward_workspace_bytes(*dims)
    fws, bws = (torch.full((n,), 0x5a, device=DEV, dtype=torch.uint8) for n in (fb, bb))
    one = (_lib.FST_FWD_ALL,) if whole else (_lib.FST_PHASE_WORKLIST, _lib.FST_PHASE_FWD)
    for ph in one:
        _lib.check(lib.fst_forward_phases(ph, *dims, P(prep.q), P(prep.k), P(prep.v), P(prep.pos4), P(prep.weight),
                                          P(prep.bias), P(prep.lens), prep.scale, P(out), P(lse), P(fws), fb,
                                          stream), "forward")
    two = (_lib.FST_BWD_ALL,) if whole else (_lib.FST_PHASE_WORKLIST, _lib.FST_PHASE_BWD_ROWS,
                                             _lib.FST_PHASE_BWD_COLS, _lib.FST_PHASE_REDUCE)
    for ph in two:
        _lib.check(lib.fst_backward_phases(ph, *dims, P(prep.q), P(prep.k), P(prep.v), P(prep.pos4), P(prep.weight),
                                           P(prep.bias), P(prep.lens), P(lse), P(do), P(out), prep.scale, P(dq),
                                           P(dk), P(dv), P(dw), P(db), P(rowsum), P(bws), bb, stream), "backward")
    torch.cuda.synchronize()
    return [out, lse, rowsum, dq, dk, dv, dw, db]


NAMES = ["out", "lse", "rowsum", "dq", "dk", "dv", "dW", "db"]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_whole_call_equals_its_phases(case):
    print(CASES[case][:4], len(CASES[case][4]), "packed" if CASES[case][5] else "padded", flush=True)
    for name, a, b in zip(NAMES, _call(True, *CASES[case]), _call(False, *CASES[case])):
        assert torch.isfinite(a).all(), name
        assert torch.equal(a, b), name


@pytest.mark.parametrize("cu", [[0, 20, 10, 50], [5, 20, 30, 50], [0, 20, 30, 60], [0, -3, 30, 50]],
                         ids=["decreasing", "start", "past-the-end", "negative"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
def test_malformed_offsets_without_a_work_list(cu, dtype):
    """The same rows are refused with NaN, and the same rows left unwritten."""
    args = (dtype, 4, 32, 16, [20, 10, 20], True, cu)
    for name, a, b in zip(NAMES, _call(True, *args), _call(False, *args)):
        assert torch.equal(a.isnan(), b.isnan()), name
        assert torch.equal(a.nan_to_num(), b.nan_to_num()), name
        if name in ("out", "dW", "db"):
            assert a.isnan().any(), name
