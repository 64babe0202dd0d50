"""One fused pass, with no refinement to repair it, against the plain FP64 pass:
from a first guess that is not zero, over blocks of one to four rows, at the
widths where the load groups, the pick of them and the bringing near of the next
matrices change.

Tolerances come from the operator itself: d is how far the plain pass moves when
only its influence matrices are rounded to FP32.  An FP32 pass also rounds its
error rows and sums (of at most 193 terms a wavefront, 14 units rounding as a
random walk): 32 d.  An FP64 pass makes the same errors in units of 2^-53 instead
of 2^-24, and so does the plain one: 64 d 2^-29.  Passes that differ only in the
row tiles of a workgroup add the same terms in the same order: the same bits."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth

pytestmark = pytest.mark.gpu

MIXED = [2, 3, 1, 2, 4, 2]  # heights
WIDTHS = [16, 20, 256, 260, 384, 388, 448, 452, 512, 516, 640, 644, 768, 772, 800, 804, 832, 836, 896,
          900, 1536, 1540]
CASES = [(i2, MIXED, periodic) for i2 in WIDTHS for periodic in (True, False)]
# FP64 matrices of a pass below and above what the last-level cache keeps
CASES += [(1440, [2] * 5, True), (1440, [2] * 6, True)]


@pytest.mark.parametrize("i2,heights,periodic", CASES)
def test_fused_one_pass(oracle, device, i2, heights, periodic):
    import torch
    ie = (1 + np.cumsum(heights)).astype(np.int32)
    j2, nrhs = int(ie[-1]) - 1, 17
    case = synth.make_case(i2, j2, 700 + i2, metric="latlon", lat_max=60.0, h_land=50.0)
    s = synth.make_rhs(case.mask, 701 + i2, nrhs)
    x0 = np.asfortranarray(np.random.default_rng(i2).standard_normal((i2 + 2, j2 + 2, nrhs)))
    s_d = torch.from_numpy(np.ascontiguousarray(s.transpose(2, 1, 0))).to(device)
    x0_d = torch.from_numpy(np.ascontiguousarray(x0.transpose(2, 1, 0))).to(device)
    with S.SevpPlan(case.coefs, ie, nrhs_max=nrhs, periodic=periodic,
                    form=S.FORM_FULL_PERIODIC if periodic else S.FORM_FULL) as plan:
        plan.build_influence()
        plain = x0_d.clone()
        plan.solve_dev(s_d, plain)
        rinv, rinv1 = [np.asfortranarray(m.astype(np.float32).astype(np.float64)) for m in plan.get_influence()]
        d = 0.0
        for r in (0, nrhs - 1):
            xr = np.asfortranarray(x0[:, :, r])
            (oracle.rep1 if periodic else oracle.rep)(case.coefs, rinv, rinv1, s[:, :, r], xr, ie)
            d = max(d, float(np.abs(xr.T - plain[r].cpu().numpy()).max()))
        for precision, tol in ((S.PREC_FP32, 32.0 * d), (S.PREC_FP64_MFMA, 64.0 * d * 2.0 ** -29)):
            plan.set_precision(precision)
            for waves in (8, 16):
                last = None
                for rows in (1, 2):
                    print(f"[fused one pass] i2={i2} heights={heights} periodic={periodic} "
                          f"precision={precision} waves={waves} rows={rows}", flush=True)
                    plan.set_tuning(S.PASS_FUSED, waves, 1, rows)
                    x = x0_d.clone()
                    plan.solve_dev(s_d, x)
                    torch.cuda.synchronize()
                    far = float((x - plain).abs().max())
                    print(f"[fused one pass] off by {far:.2e} of {tol:.2e}", flush=True)
                    assert far <= tol
                    assert last is None or torch.equal(x, last)
                    last = x
