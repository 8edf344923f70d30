"""Fields that are not finite: phi and psi stay 0 where no PML profile acts, whatever u holds there, so the
multi-level tiles step an overflowed run as single levels do."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def same(a, b):
    return bool(((a == b) | (torch.isnan(a) & torch.isnan(b))).all())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("NX,NY,si,sj,hy", [(30, 62, 12, 40, 9.0), (90, 110, 80, 13, 9.0), (90, 110, 45, 55, 10.0),
                                           (90, 110, 84, 104, 10.0)])
def test_infinite_source(ads, cuda, kernel, dtype, NX, NY, si, sj, hy):
    """An infinite source sample, near the PML, away from it and in a corner whose two profiles are equal on the
    diagonal."""
    npml, n = 8, 26
    p = ads.AcousticPropagatorParams(NX=NX, NY=NY, NSTEP=n, DELTAX=10.0, DELTAY=hy, DELTAT=1e-3,
                                     NPOINTS_PML=npml, vp_ref=2000.0, PropagatorKernel=kernel)
    w = np.sin(0.4 * np.arange(n))
    w[9] = np.inf
    ii, jj = np.meshgrid(np.arange(1, NX + 3), np.arange(1, NY + 3), indexing="ij")
    src, rcv = ads.AcousticSource([si], [sj], w[:, None]), ads.AcousticReceiver(ii.reshape(-1), jj.reshape(-1))
    plan = ads.AcousticPlan(p, [src], [rcv], dtype=dtype)
    c = torch.linspace(1800.0, 2300.0, (NX + 2) * (NY + 2), dtype=dtype, device="cuda").reshape(NX + 2, NY + 2)
    srcv = plan.pack_srcv([w[:, None]])
    plan.set_blocking(1)
    one = plan.forward(c, srcv, 100).clone()
    plan.set_blocking(2)
    tr = plan.forward(c, srcv, 100)
    assert not torch.isfinite(tr).all()
    assert same(tr, one)
    u, phi, psi = plan.forward_history(c, srcv)
    assert same(u.reshape(-1), one)
    q = ads.compute_PML_Params_(p)
    pml = (np.asarray(q.Σx).reshape(NX + 2, NY + 2) != 0) | (np.asarray(q.Σy).reshape(NX + 2, NY + 2) != 0)
    out = torch.as_tensor(~pml, device="cuda")
    out[0] = out[-1] = out[:, 0] = out[:, -1] = True
    assert (phi[0][:, out] == 0).all() and (psi[0][:, out] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kernel", [0, 1])
def test_infinite_last_sample(ads, cuda, kernel, dtype):
    """The last level's source sample reaches the source cell of the last level alone, which no receiver there reads and
    no dL/dC term uses unless the cell touches the PML: an infinite one leaves the gradient as it is."""
    p = ads.AcousticPropagatorParams(NX=30, NY=62, NSTEP=40, DELTAX=10.0, DELTAY=10.0, DELTAT=1e-3, NPOINTS_PML=8,
                                     vp_ref=2000.0, PropagatorKernel=kernel)
    c = torch.linspace(1800.0, 2300.0, 32 * 64, dtype=dtype, device="cuda").reshape(32, 64)
    out = []
    for last in (0.0, np.inf):
        w = 1e3 * np.sin(0.4 * np.arange(40))
        w[-1] = last
        plan = ads.AcousticPlan(p, [ads.AcousticSource([16], [30], w[:, None])],
                                [ads.AcousticReceiver(np.arange(2, 32), np.full(30, 12))], dtype=dtype)
        srcv = plan.pack_srcv([w[:, None]])
        obs = torch.ones(plan.trace_elems, dtype=dtype, device="cuda")
        out.append(plan.gradient(c, srcv, obs, 9)[1].clone())
    assert torch.isfinite(out[0]).all() and float(out[0].abs().max()) > 0.0
    assert torch.equal(out[1], out[0])
