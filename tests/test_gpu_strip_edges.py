"""The strip kernels at the edges of their layout: strip widths around the
halves a closure's column is split into and the products it takes four at a
time (2..32), around the 32- and 64-lane kernels and the width-specialised
ones, and marches whose record counts end on, before and after a chunk.  One
REPBIR call must equal the oracle's bit for bit."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth
from tests.conftest import all_finite, fields_equal

pytestmark = pytest.mark.gpu

WIDTHS = [2, 3, 5, 8, 9, 15, 16, 17, 23, 24, 25, 29, 30, 31, 32, 33, 47, 63, 64]
# a forward march has IE(NBLK) - 1 records, a backward one IE(NBLK) - 1 + NBLK;
# chunks are of 24 (32 lanes) or 16
CASES = [(w, list(range(3, 25, 2)) + [25]) for w in WIDTHS]
CASES += [(w, ie) for w in (24, 40) for ie in (
    [3], [2, 3], [17], [4, 18], [25], [26], list(range(3, 34, 2)), list(range(4, 49, 3)) + [49],
    list(range(5, 64, 6)))]


@pytest.mark.parametrize("m2,ie", CASES)
def test_repbir_edges(oracle, device, m2, ie):
    from oracle.oracle import P, _ci
    print(f"[strip edges] m2={m2} ie={ie}", flush=True)
    i2, off, j2, nblk = 80, 6, ie[-1] - 1, len(ie)
    case = synth.make_case(i2, j2, 300 + m2, metric="latlon", lat_max=60.0, h_land=50.0)
    ie = np.asarray(ie, np.int32)
    h = np.zeros((i2 + 2, j2 + 2), order="F")
    rv = np.zeros((m2, m2, nblk), order="F")
    rv1 = np.zeros((m2, m2, nblk), order="F")
    oracle.lib().orc_pre(*[P(c, off) for c in case.coefs], P(rv), P(rv1), P(h), P(ie), _ci(i2),
                         _ci(m2 + 2), _ci(m2), _ci(nblk))
    s = synth.make_rhs(case.mask, 301 + m2, 1)[:, :, 0]
    src = np.asfortranarray(s[off:off + m2, :])
    x0 = np.asfortranarray(np.random.default_rng(m2).standard_normal((i2 + 2, j2 + 2)))
    d0, d1 = np.zeros((m2, nblk), order="F"), np.zeros(m2)
    xg = x0.copy(order="F")
    S.repbir(*case.coefs, rv, rv1[:, :, :max(nblk - 1, 1)].copy(order="F"), d0, d1, d1, src, h, xg, ie,
             i2 + 2, i2, m2 + 2, m2, nblk, coef_off=off, x_off=off)
    xo = x0.copy(order="F")
    oracle.repbir_call([(c, off) for c in case.coefs], rv, rv1, d0.copy(order="F"), d1.copy(),
                       d1.copy(), src, h.copy(order="F"), (xo, off), ie, i2 + 2, i2, m2 + 2, m2, nblk)
    assert all_finite(xo)
    assert fields_equal(xg, xo)
