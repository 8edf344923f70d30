"""The rows per wavefront that the elastic kernels choose by themselves, against fixed ones.

A chunk's height decides which wavefronts form a cell and which of them stores it, not the
arithmetic of a cell: the sums over shots keep their order, so the bars are the rounding bars of
tests/test_gpu_elastic.py for two forms of one step (1e-12 / 1e-5 for traces and misfit, 1e-11 /
1e-4 for gradients).
"""
import pytest

from test_gpu_elastic import T, make_case, rel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# wavefronts on both sides of the rule's lines: a grid of a few rows, one shot (1 row), a grid
# whose columns end one past a strip, several shots (2 rows), a wide one (4 and 8 rows)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("NX,NY,nshots", [(17, 18, 1), (120, 111, 2), (200, 119, 5), (260, 470, 5)])
def test_chosen_rows_match_fixed_rows(orc, ads, cuda, NX, NY, nshots, dtype):
    p, models, srcs, rcvs, nstep = make_case(orc, ads, NX=NX, NY=NY, NSTEP=24, npml=6, nshots=min(nshots, 2),
                                             seed=5)
    srcs, rcvs = [srcs[s % 2] if s < len(srcs) else srcs[0] for s in range(nshots)], [rcvs[0]] * nshots
    mt = [T(m, dtype) for m in models]
    out = []
    for fixed in (True, False):
        plan = ads.ElasticPlan(p, srcs, rcvs, dtype=dtype)
        if fixed:
            plan.set_forward_kernels(1, 8)
            plan.set_adjoint_kernels(2, 8, 4)
        srcv = plan.pack_srcv([s.srcv for s in srcs])
        obs = plan.forward(*[m * f for m, f in zip(mt, (1.02, 0.97, 1.04))], srcv, 7).clone()
        L, g, t = plan.gradient(*mt, srcv, obs, 7, want_traces=True)
        out.append((obs.cpu(), float(L), t.clone().cpu(), [x.clone().cpu() for x in g]))
    (o0, L0, t0, g0), (o1, L1, t1, g1) = out
    bar_t, bar_g = (1e-12, 1e-11) if dtype == torch.float64 else (1e-5, 1e-4)
    assert rel(o1, o0) <= bar_t and rel(t1, t0) <= bar_t and abs(L1 - L0) <= bar_t * abs(L0)
    for a, b in zip(g1, g0):
        assert rel(a, b) <= bar_g
