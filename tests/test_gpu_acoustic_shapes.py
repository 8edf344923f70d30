"""The shapes of the acoustic plan where they have an effect: the single-level forward's rows, shots and batch
(set_blocking(1)) against the tiles bit for bit, and the adjoint's shots per workgroup against the FP64 oracle
(1e-10, the bound of the other FP64 gradients)."""
import numpy as np
import pytest

from test_gpu_acoustic import SPLITS, T, make_case, oracle_shot, rel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

GRIDS = SPLITS + [dict(NX=70, NY=300, npml=8, use=(True,) * 4)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("grid", range(len(GRIDS)))
def test_single_level_shapes_equal_the_tiles(orc, ads, cuda, kernel, dtype, grid):
    cfg = GRIDS[grid]
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=cfg["NX"], NY=cfg["NY"], NSTEP=33, npml=cfg["npml"], nshots=5,
                                        kernel=kernel, seed=60 + grid, uneven=True)
    p.USE_PML_XMIN, p.USE_PML_XMAX, p.USE_PML_YMIN, p.USE_PML_YMAX = cfg["use"]
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=dtype, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    want = plan.forward(T(c, dtype), srcv, 9).clone()
    plan.set_blocking(1)
    for rows, shots, batch in [(1, 1, 1), (1, 2, 2), (2, 3, 1), (2, 4, 2), (4, 5, 1), (4, 16, 1), (8, 3, 1), (16, 5, 1)]:
        plan.set_shape((rows, shots, batch, 1, 1, 1))
        assert torch.equal(plan.forward(T(c, dtype), srcv, 9), want), (rows, shots, batch)


# 36 and 40 tiles of the first grid for the fewest levels that the rule tries, times 8 shots: more workgroups than
# the card holds at once in FP64, so the levels follow from the tiles' work; the second fits
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("NX,NY,nshots", [(171, 203, 8), (31, 63, 5)])
def test_adjoint_shots_per_workgroup_against_oracle(orc, ads, cuda, kernel, NX, NY, nshots):
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=NX, NY=NY, NSTEP=65, npml=7, nshots=nshots, kernel=kernel,
                                        seed=70, uneven=True)
    obs, g_ref = [], 0.0
    for s in range(nshots):
        obs.append(oracle_shot(orc, p, c, srcs[s], rcvs[s], nstep[s], cmod=1.03 * c))
        g_ref = g_ref + oracle_shot(orc, p, c, srcs[s], rcvs[s], nstep[s], obs=obs[s])[2]
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    for shots in (1, 2, 3, nshots, 32):
        plan.set_shape((2, 16, 1, 2, shots, 1))
        g = plan.gradient(T(c), srcv, plan.pack_traces(obs), 11)[1]
        assert rel(g.cpu(), g_ref) < 1e-10, (shots, rel(g.cpu(), g_ref))
