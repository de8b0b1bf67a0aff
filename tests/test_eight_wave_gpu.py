"""GPU tests of the bf16 forward's and cols kernel's eight-wave instances.

Where the library's static choice runs eight waves (heavy lane states at 16
padded heads, wide heads at 8, and the cols kernel's 12 heads padded to 16;
without the bias on the logits the forward only in grids of up to 256
workgroups),
every row and key is computed with the arithmetic of the four-wave instances
that the occupancy plan bits name: out, lse, dq, dk, dv must agree bit for
bit, dW and db to the rounding of their float32 partial sums, and all with
the float64 oracle to the bf16 tolerance of the parity tests. Lengths sit at
the edges of the 16-row tiles and chunks; heads leave padded slots.
"""

import pytest
import torch

import oracle
from tests._cases import rel_err

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from flash_spacetime_amd import _lib, tune
    from tests.test_plans_gpu import BF, TOL, _inputs, _oracle, _run, _same

# (heads, dim, channels, lengths, packed, bias flags)
SHAPES = [
    (16, 48, 48, [33, 16, 1], True, (True, True)),
    (13, 64, 64, [47, 17], False, (True, True)),    # three padded heads
    (16, 64, 32, [31, 32], False, (True, False)),   # flags read at run time
    (14, 48, 16, [18, 15], True, (False, True)),    # cols kernel only
    (16, 32, 16, [49, 2], False, (True, True)),     # forward only, two workgroups per CU
    (12, 48, 48, [35, 16], False, (True, True)),    # cols kernel, 12 heads padded to 16
    (9, 48, 64, [20, 1], True, (True, True)),
    (8, 64, 16, [33, 15], True, (True, True)),      # cols kernel, four waves per SIMD
    (5, 48, 32, [17, 48], False, (False, False)),
    (11, 48, 64, [18, 33], True, (True, False)),    # cols kernel, one bias: 12 heads on four waves
    (13, 48, 48, [33, 15], False, (False, True)),   # forward: few tiles, eight waves
    (16, 64, 32, [17, 1] * 100, True, (False, True)),  # more than 256 workgroups, four waves
    (14, 64, 48, [9] * 260, False, (False, False)),
]


@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_eight_waves_match_four_and_the_oracle(case):
    heads, dim, chans, lens, packed, flags = SHAPES[case]
    print(f"H={heads} D={dim} C={chans} lens={lens} packed={packed} flags={flags}", flush=True)
    args = _inputs(BF, heads, dim, chans, lens, packed, 300 + case)
    tune.set_autotune(False)
    got = _run(args, flags, True)
    with tune.fixed_plan(_lib.FST_PLAN_FWD_OCC2 | _lib.FST_PLAN_COLS_OCC2):
        four = _run(args, flags, True)
    assert _same(got, four)
    ref = _oracle(args, flags, packed)
    out = got[0]
    if not packed:
        out = out * oracle.valid_row_mask(len(lens), max(lens), torch.tensor(lens))[:, None, :, None].to(out.device)
    for name, a, e in zip(["out", "dq", "dk", "dv", "dW", "db"], [out] + list(got[3]), [ref[0]] + ref[1]):
        if e is None or (name == "dW" and not any(flags)) or (name == "db" and not flags[1]):
            continue
        err = rel_err(a, e)
        assert err <= TOL[BF], f"{name} relative error {err:.3e}"


@pytest.mark.parametrize("packed", [True, False], ids=["packed", "heads_first"])
@pytest.mark.parametrize("flags", [(True, True), (False, True), (False, False)])
def test_rows_of_twelve_heads_padded_or_split_unevenly(packed, flags):
    """D = 48, C = 64: the rows kernel pads to 16 heads where a token's heads are
    adjacent and a bias is on, else splits 12 unevenly: the bits of the plan
    that names the padded one either way."""
    args = _inputs(BF, 10, 48, 64, [35, 16, 1], packed, 350)
    tune.set_autotune(False)
    got = _run(args, flags, True)
    with tune.fixed_plan(_lib.FST_PLAN_ROWS_W8):
        assert _same(got, _run(args, flags, True))
