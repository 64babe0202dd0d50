"""Which stream a full-width pass runs on: the plan's (a blocking one, so a
long pass moves to a non-blocking stream between two events), a caller's
non-blocking stream, and one that is being captured.  Each must be ordered
with the null stream's work before and after it, with no synchronisation in
between, and give the same bits; 31 and 32 blocks lie either side of the
rule's edge."""
import ctypes

import numpy as np
import pytest

from musoc_solver_amd import sevp as S
from musoc_solver_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("blocks", [31, 32])
@pytest.mark.parametrize("precision", [S.PREC_FP64, S.PREC_FP32])
def test_pass_streams(device, blocks, precision):
    import torch
    i2, j2, nrhs = 64, 2 * blocks, 3
    print(f"[pass streams] blocks={blocks} precision={precision}", flush=True)
    case = synth.make_case(i2, j2, 77, metric="latlon", lat_max=60.0, h_land=50.0)
    ie = synth.reference_ie(j2, blocks)
    s = synth.make_rhs(case.mask, 78, nrhs)
    with S.SevpPlan(case.coefs, ie, form=S.FORM_FULL_PERIODIC, nrhs_max=nrhs, precision=precision) as plan:
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

        def call(st):
            assert S.lib().sevp_solve_dev(plan._h, ctypes.c_void_p(s_d.data_ptr()),
                                          ctypes.c_void_p(x_d.data_ptr()), nrhs,
                                          ctypes.c_void_p(st.cuda_stream)) == 0

        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            x_d.zero_()
            call(side)
        torch.cuda.synchronize()
        assert torch.equal(x_d, want)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call(torch.cuda.current_stream())
        for _ in range(3):
            x_d.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(x_d, want)
