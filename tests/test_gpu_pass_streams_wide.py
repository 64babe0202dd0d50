"""Which stream a matrix-core pass runs on: a fused one of 600 columns or more
moves to the plan's non-blocking stream as the plain one does, a narrower one and
a split-K one stay. Either must be ordered with the null stream's work before and
after it, with no synchronisation in between, and give the bits of a pass alone."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("i2", [596, 600])
@pytest.mark.parametrize("precision,kind", [(S.PREC_FP32, S.PASS_FUSED), (S.PREC_FP64_MFMA, S.PASS_FUSED),
                                            (S.PREC_FP32, S.PASS_SPLITK)])
def test_pass_streams_wide(device, i2, precision, kind):
    import torch
    blocks, nrhs = 32, 2
    j2 = 2 * blocks
    print(f"[pass streams wide] i2={i2} precision={precision} kind={kind}", flush=True)
    case = synth.make_case(i2, j2, 79, metric="latlon", lat_max=60.0, h_land=50.0)
    s = synth.make_rhs(case.mask, 80, nrhs)
    with S.SevpPlan(case.coefs, synth.reference_ie(j2, blocks), form=S.FORM_FULL_PERIODIC, nrhs_max=nrhs,
                    precision=precision) as plan:
        plan.set_pass(kind)
        plan.build_influence()
        want = torch.from_numpy(np.ascontiguousarray(
            plan.solve(s, np.zeros((i2 + 2, j2 + 2, nrhs), order="F")).transpose(2, 1, 0))).to(device)
        assert torch.isfinite(want).all()
        s_d = torch.from_numpy(np.ascontiguousarray(s.transpose(2, 1, 0))).to(device)
        x_d = torch.empty((nrhs, j2 + 2, i2 + 2), dtype=torch.float64, device=device)
        s2 = torch.empty_like(s_d)
        got = []
        for _ in range(3):  # the null stream before, between and after
            x_d.zero_()
            s2.copy_(s_d)
            plan.solve_dev(s2, x_d)
            got.append(x_d.clone())
            s2.fill_(float("nan"))
        torch.cuda.synchronize()
        assert all(torch.equal(g, want) for g in got)
