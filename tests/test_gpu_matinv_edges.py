"""The blocked MATINV at the edges of its panels and tiles: orders around
multiples of 32 and 64, odd ones (columns at 8-byte boundaries), a last panel
of one row, and a zero pivot inside and at the start of a panel (counted, its
infinities and NaN where the reference's elimination puts them)."""
import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from tests.conftest import fields_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,zero", [(95, None), (97, None), (127, None), (128, None), (129, None),
                                    (161, None), (193, None), (97, 40), (130, 96), (130, 128)])
def test_matinv_edges(oracle, device, n, zero):
    import torch
    print(f"[matinv edges] n={n} zero={zero}", flush=True)
    b = np.asfortranarray(np.random.default_rng(n).standard_normal((n, n)) + 0.5 * n * np.eye(n))
    if zero is not None:
        b[zero, :] = 0.0
        b[:, zero] = 0.0
    with np.errstate(all="ignore"):
        bo, zo = oracle.matinv(b)
    bd = torch.from_numpy(np.ascontiguousarray(b.T)).to(device)
    zp = torch.full((1,), -1, dtype=torch.int32, device=device)
    S.matinv_dev_noalloc(bd, n, zp)
    torch.cuda.synchronize()
    assert int(zp.item()) == zo == (0 if zero is None else 1)
    assert fields_equal(np.asfortranarray(bd.cpu().numpy().T), bo)
