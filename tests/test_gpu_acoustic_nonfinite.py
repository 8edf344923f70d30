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
