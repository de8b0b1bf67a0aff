"""GPU tests of the float32 kernels' uneven eight-wave split of 12 heads.

Nine to twelve float32 heads run eight waves (two heads on four of them, one
on the others). Every row and key is computed with the arithmetic of the
four-wave tiles that the tile-height plan bits name, at the same key chunk:
out, lse, dq, dk, dv must agree bit for bit, dW and db to the rounding of
their partial sums, and all with the float64 oracle at the float32 tolerance
of the parity tests. Head counts leave padded heads on either kind of wave;
lengths sit at the edges of tiles and chunks. The passes over the keys are
those of four waves, so the four-wave plan of the backward, with no pass bit,
gives the static choice's bits at every width.
"""

import pytest
import torch

import oracle
from tests._cases import rel_err

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from flash_spacetime_amd import _lib, tune
    from tests.test_plans_gpu import F32, TOL, _inputs, _oracle, _run, _same

# (heads, dim, channels, lengths, packed, bias flags, keys per forward chunk and
# passes of the rows kernel in the static choice)
SHAPES = [
    (12, 32, 16, [33, 16, 1], False, (True, True), 16, 1),
    (12, 32, 32, [31, 64], True, (True, True), 32, 1),
    (9, 16, 16, [17, 15], False, (True, False), 16, 1),     # three padded heads
    (11, 48, 48, [32, 18], True, (True, True), 32, 2),
    (10, 16, 64, [47, 2], False, (False, True), 16, 2),     # no room for 32 keys
    (12, 64, 16, [20, 33], True, (True, True), 16, 1),      # four-wave cols kernel
    (12, 64, 48, [35, 1], False, (True, True), 32, 2),      # four-wave rows kernel
    (12, 64, 32, [16, 49], False, (False, False), 32, 2),
]


@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_uneven_split_matches_four_waves_and_the_oracle(case):
    heads, dim, chans, lens, packed, flags, keys, passes = SHAPES[case]
    print(f"H={heads} D={dim} C={chans} lens={lens} packed={packed} flags={flags}", flush=True)
    args = _inputs(F32, heads, dim, chans, lens, packed, 400 + case)
    tune.set_autotune(False)
    got = _run(args, flags)
    plan = (_lib.FST_PLAN_FWD_T16 | (_lib.FST_PLAN_FWD_KC16 if keys == 16 else _lib.FST_PLAN_FWD_KC32)
            | _lib.FST_PLAN_BWD_T16 | _lib.FST_PLAN_BWD_KC16
            | (_lib.FST_PLAN_BWD_PASS1 if passes == 1 else _lib.FST_PLAN_BWD_PASS2))
    with tune.fixed_plan(plan):
        assert _same(got, _run(args, flags))
    ref = _oracle(args, flags, packed)
    out = got[0]
    if not packed:
        out = out * oracle.valid_row_mask(len(lens), max(lens), torch.tensor(lens))[:, None, :, None].to(out.device)
    for name, a, e in zip(["out", "dq", "dk", "dv", "dW", "db"], [out] + list(got[3]), [ref[0]] + ref[1]):
        if e is None or (name == "dW" and not any(flags)) or (name == "db" and not flags[1]):
            continue
        err = rel_err(a, e)
        assert err <= TOL[F32], f"{name} relative error {err:.3e}"


@pytest.mark.parametrize("dim, chans", [(16, 64), (32, 16), (32, 48), (32, 64), (48, 16), (48, 32), (48, 48), (48, 64),
                                        (64, 32)])
def test_four_wave_backward_without_a_pass_bit_gives_the_same_bits(dim, chans):
    print(f"D={dim} C={chans}", flush=True)
    args, flags = _inputs(F32, 12, dim, chans, [130, 57], True, 500 + dim + chans), (True, True)
    tune.set_autotune(False)
    got = _run(args, flags)
    with tune.fixed_plan(_lib.FST_PLAN_BWD_T16):
        assert _same(got, _run(args, flags))
