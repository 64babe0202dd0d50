"""The plain FP64 products at the edges of their tiles and dispatch: sums
shorter than a group, around a 64-term chunk and odd (4-byte DMAs), column
counts off the tile, and the right-hand-side counts and widths at which the
kernel changes.  One REP1 pass must equal the oracle's bit for bit."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth
from tests.conftest import fields_equal

pytestmark = pytest.mark.gpu

CASES = [(i2, nrhs) for i2 in (5, 17, 63, 64, 65, 128, 130) for nrhs in (1, 2, 3, 8, 9, 17)]
# one workgroup per CU is passed by 1, 2 and 4 computing wavefronts
CASES += [(400, 64), (401, 64), (520, 64), (521, 64), (1040, 64), (1041, 64), (720, 1), (721, 5)]


@pytest.mark.parametrize("i2,nrhs", CASES)
def test_plain_products(oracle, device, i2, nrhs):
    j2 = 6
    print(f"[plain products] i2={i2} nrhs={nrhs}", flush=True)
    case = synth.make_case(i2, j2, 900 + i2, metric="latlon", lat_max=60.0, h_land=50.0)
    ie = synth.reference_ie(j2, 3)
    s = synth.make_rhs(case.mask, 901 + i2, nrhs)
    x0 = np.asfortranarray(np.random.default_rng(i2).standard_normal((i2 + 2, j2 + 2, nrhs)))
    with S.SevpPlan(case.coefs, ie, form=S.FORM_FULL_PERIODIC, nrhs_max=nrhs) as plan:
        plan.build_influence()
        rinv, rinv1 = plan.get_influence()
        x = plan.solve(s, x0.copy(order="F"))
    for r in sorted({0, nrhs // 2, nrhs - 1}):
        xo = np.asfortranarray(x0[:, :, r])
        oracle.rep1(case.coefs, rinv, rinv1, s[:, :, r], xo, ie)
        assert fields_equal(x[:, :, r], xo), r
