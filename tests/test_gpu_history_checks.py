"""What the full-history entry points ask of a plan, and of the arrays they are given."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def acoustic_plan(ads, kernel, nstep):
    p = ads.AcousticPropagatorParams(NX=24, NY=20, NSTEP=max(nstep), DELTAX=10.0, DELTAY=10.0, DELTAT=1e-3,
                                     NPOINTS_PML=5, vp_ref=2000.0, PropagatorKernel=kernel)
    w = [1e3 * np.sin(0.3 * np.arange(n)) for n in nstep]
    srcs = [ads.AcousticSource([8 + 3 * s], [4], v[:, None]) for s, v in enumerate(w)]
    plan = ads.AcousticPlan(p, srcs, [ads.AcousticReceiver([5], [5])] * len(nstep), dtype=torch.float64, nstep=nstep)
    c = torch.linspace(1800.0, 2300.0, 26 * 22, dtype=torch.float64, device="cuda").reshape(26, 22)
    return plan, c, plan.pack_srcv([s.srcv for s in srcs])


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("nstep", [[31, 20], [20, 31, 31]])
def test_acoustic_history_refuses_short_records(ads, cuda, kernel, nstep):
    """A history holds NSTEP levels of every shot: a plan with a shorter record is refused on the host,
    whichever shot it is, before anything is written."""
    plan, c, srcv = acoustic_plan(ads, kernel, nstep)
    with pytest.raises(Exception, match="nstep == NSTEP"):
        plan.forward_history(c, srcv)
    u = torch.zeros((len(nstep), 32, 26, 22), dtype=torch.float64, device="cuda")
    with pytest.raises(Exception, match="nstep == NSTEP"):
        plan.backward_history(c, srcv, u, torch.ones_like(u))


@pytest.mark.parametrize("kernel", [0, 1])
def test_acoustic_history_with_one_auxiliary_array(ads, cuda, kernel):
    """phi_hist and psi_hist may each be null: whichever is given is filled as when both are."""
    import ctypes as C
    plan, c, srcv = acoustic_plan(ads, kernel, [31, 31])
    ref = plan.forward_history(c, srcv)
    assert all(float(t.abs().max()) > 0.0 for t in ref)
    sc = torch.empty(plan.lib.ads_acoustic_plan_history_scratch_size(plan.h), dtype=torch.uint8, device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for given in ((True, False), (False, True), (False, False)):
        out = [torch.full_like(ref[0], 7.0)] + [torch.full_like(ref[0], 7.0) if g else None for g in given]
        rc = plan.lib.ads_acoustic_plan_forward_history(
            plan.h, *[None if t is None else C.c_void_p(t.data_ptr()) for t in (c, srcv, *out, sc)], st)
        assert rc == 0
        for a, b in zip(out, ref):
            assert a is None or torch.equal(a, b), given


@pytest.mark.parametrize("nstep", [[24, 15], [15, 24, 24]])
def test_elastic_history_refuses_short_records(ads, cuda, nstep):
    """As the acoustic calls: the history and the pullback of a dense cotangent."""
    p = ads.ElasticPropagatorParams(NX=24, NY=20, NSTEP=max(nstep), DELTAX=10.0, DELTAY=10.0, DELTAT=1e-3,
                                    NPOINTS_PML=5, vp_ref=2500.0, f0=8.0)
    srcs = [ads.ElasticSource([8, 8], [6, 6], [2, 3], np.ones((n, 2))) for n in nstep]
    plan = ads.ElasticPlan(p, srcs, [ads.ElasticReceiver([5], [5], [0])] * len(nstep), dtype=torch.float64, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    m = [torch.full((26, 22), v, dtype=torch.float64, device="cuda") for v in (2000.0, 4e9, 4e9)]
    with pytest.raises(Exception, match="nstep == NSTEP"):
        plan.forward_history(*m, srcv)
    with pytest.raises(Exception, match="nstep == NSTEP"):
        plan.backward_dense(*m, srcv, torch.ones((len(nstep), 5, 25, 26, 22), dtype=torch.float64, device="cuda"), 8)
