"""The fused pass at the widths where a wavefront's share of the product's
chunks passes from one load group to the next (a quarter, half, the whole of
it, and the loop over several), for 8 and 16 wavefronts and one or two row
tiles, and right-hand-side counts around a row tile.  A refined solve reaches
the residual bound, which a separate kernel measures, only with right passes."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-10  # the refinement contract


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("i2", [16, 20, 256, 260, 384, 388, 512, 516, 768, 772, 1536, 1540])
def test_fused_groups(device, i2, periodic):
    import torch
    j2 = 8
    case = synth.make_case(i2, j2, 500 + i2, metric="latlon", lat_max=60.0, h_land=50.0)
    ie = synth.reference_ie(j2, 4)
    for nrhs in (1, 17):
        s = synth.make_rhs(case.mask, 501 + i2, nrhs)
        s_d = torch.from_numpy(np.ascontiguousarray(s.transpose(2, 1, 0))).to(device)
        with S.SevpPlan(case.coefs, ie, nrhs_max=nrhs, periodic=periodic,
                        form=S.FORM_FULL_PERIODIC if periodic else S.FORM_FULL) as plan:
            plan.build_influence()
            for precision in (S.PREC_FP32, S.PREC_FP64_MFMA):
                plan.set_precision(precision)
                for waves in (8, 16):
                    for rows in (1, 2):
                        print(f"[fused groups] i2={i2} periodic={periodic} nrhs={nrhs} "
                              f"precision={precision} waves={waves} rows={rows}", flush=True)
                        plan.set_tuning(S.PASS_FUSED, waves, 1, rows)
                        x_d = torch.zeros((nrhs, j2 + 2, i2 + 2), dtype=torch.float64, device=device)
                        rel, st, ok = plan.solve_refined_dev(s_d, x_d, tol=TOL, max_iter=8)
                        torch.cuda.synchronize()
                        assert ok and np.max(rel) <= TOL
