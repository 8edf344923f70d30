"""The multi-level tile kernels of the acoustic plan at the sizes where tiles, halos and point lists
change: against single-level stepping (bit for bit) and the FP64 oracle (1e-12 traces, 1e-10 gradients,
the bounds of the other FP64 acoustic tests)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ALL = (True, True, True, True)
# (NX, NY, npml, PML sides): one tile; one row / column beyond a tile; several plain tiles inside PML
# bands with remainders; no PML (ring cells only); a PML on some sides, its tiles next to plain ones
GRIDS = [(14, 9, 3, ALL), (30, 62, 4, ALL), (31, 63, 5, ALL), (171, 203, 6, ALL), (118, 131, 8, (False,) * 4),
         (149, 97, 7, (True, False, False, True))]


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def case(ads, orc, grid, kernel, nsteps):
    """Three shots: one source; a line of receivers along x with duplicated sources and receivers on a tile
    edge; a line of receivers along y, a source on the ring and a shorter record."""
    NX, NY, npml, use = grid
    rng = np.random.default_rng(NX + 7 * NY)
    p = ads.AcousticPropagatorParams(NX=NX, NY=NY, NSTEP=nsteps, DELTAX=10.0, DELTAY=9.0, DELTAT=1e-3,
                                     NPOINTS_PML=npml, vp_ref=2000.0, PropagatorKernel=kernel)
    p.USE_PML_XMIN, p.USE_PML_XMAX, p.USE_PML_YMIN, p.USE_PML_YMAX = use
    c = 1800.0 + 700.0 * rng.random((NX + 2, NY + 2))
    n = [nsteps, nsteps, nsteps - 5]
    w = [orc.ricker(k, 4.0, 8.0 + s, 1e6) for s, k in enumerate(n)]
    mi, mj = NX // 2 + 1, NY // 2 + 1
    srcs = [ads.AcousticSource([mi], [mj], w[0][:, None]),
            ads.AcousticSource([mi, mi, 2], [mj, mj, NY], np.stack([w[1], -0.5 * w[1], w[1]], 1)),
            ads.AcousticSource([1, NX], [3, 2], np.stack([w[2], 0.7 * w[2]], 1))]
    x, y = np.arange(1, NX + 3), np.arange(1, NY + 3)
    rcvs = [ads.AcousticReceiver([mi, mi], [2, mj]),
            ads.AcousticReceiver(np.r_[x, mi, mi], np.r_[np.full(len(x), 3), mj, mj]),
            ads.AcousticReceiver(np.r_[np.full(len(y), 4), NX + 1], np.r_[y, NY])]
    return p, c, srcs, rcvs, n, use


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("grid", range(len(GRIDS)))
def test_tiles_against_single_levels_and_oracle(orc, ads, cuda, kernel, grid):
    p, c, srcs, rcvs, n, use = case(ads, orc, GRIDS[grid], kernel, 33)
    k = 0 if kernel == 0 else 1
    Sx, Sy = orc.acoustic_pml(p.NX, p.NY, 10.0, 9.0, p.NPOINTS_PML, p.Rcoef, p.vp_ref, use=use)
    tr_ref, g_ref, obs = [], 0.0, []
    for s in range(3):
        args = (k, p.NX, p.NY, n[s], p.DELTAT, 10.0, 9.0, Sx, Sy)
        src = (srcs[s].srci, srcs[s].srcj, srcs[s].srcv)
        u, _, _ = orc.acoustic_forward(*args, c ** 2, *src)
        tr_ref.append(orc.acoustic_receive(u, rcvs[s].rcvi, rcvs[s].rcvj, p.NY))
        obs.append(0.6 * tr_ref[s] + 1e-3)
        g_ref = g_ref + orc.acoustic_misfit_gradient(*args, c, *src, rcvs[s].rcvi, rcvs[s].rcvj, obs[s])[1]
    for dtype in (torch.float64, torch.float32):
        plan = ads.AcousticPlan(p, srcs, rcvs, dtype=dtype, nstep=n)
        srcv = plan.pack_srcv([s.srcv for s in srcs])
        ct = torch.as_tensor(c, dtype=dtype, device="cuda")
        ob = plan.pack_traces([torch.as_tensor(o) for o in obs])
        for K in (9, 100):  # launches of every remainder of levels; one segment
            plan.set_blocking(1)
            one = plan.forward(ct, srcv, K)
            plan.set_blocking(2)
            loss, g, tr = plan.gradient(ct, srcv, ob, K, want_traces=True)
            assert torch.equal(tr, one), (dtype, K)
            if dtype == torch.float64:
                for s, t in enumerate(plan.unpack_traces(tr)):
                    assert rel(t.cpu(), tr_ref[s]) < 1e-12, (s, K)
                assert rel(g.cpu(), g_ref) < 1e-10, K
            else:
                assert rel(g.cpu(), g_ref) < 1e-3, K


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("grid", [1, 3, 5])
def test_history_tiles_against_oracle(orc, ads, cuda, kernel, grid):
    """The dense full-history layout, whose rows are not aligned: u, phi, psi of every level, and the
    pullback of a dense cotangent."""
    p, c, srcs, rcvs, n, use = case(ads, orc, GRIDS[grid], kernel, 18)
    k = 0 if kernel == 0 else 1
    Sx, Sy = orc.acoustic_pml(p.NX, p.NY, 10.0, 9.0, p.NPOINTS_PML, p.Rcoef, p.vp_ref, use=use)
    args = (k, p.NX, p.NY, 18, p.DELTAT, 10.0, 9.0, Sx, Sy)
    u, ph, ps = orc.acoustic_forward(*args, c ** 2, srcs[1].srci, srcs[1].srcj, srcs[1].srcv)
    ct = torch.as_tensor(c, device="cuda").requires_grad_(True)
    ap = ads.AcousticPropagatorSolver(p, srcs[1], ct)
    assert rel(ap.u.detach().cpu(), u) < 1e-12
    assert rel(ap.φ.cpu(), ph) < 1e-12
    assert rel(ap.ψ.cpu(), ps) < 1e-12
    gu = np.random.default_rng(3).standard_normal(ap.u.shape)
    gu[:2] = 0.0
    gC = orc.acoustic_adjoint(*args, c ** 2, u, ph, ps, gu.reshape(19, -1))
    gC = gC[0] if isinstance(gC, tuple) else gC
    g = torch.autograd.grad(ap.u, ct, torch.as_tensor(gu, device="cuda"))[0]
    assert rel(g.cpu(), 2.0 * c * np.asarray(gC).reshape(c.shape)) < 1e-10
