"""The elastic forward's register tiles (two levels per launch) at the edges of tiles.

FP64 plans step by tiles; against one level per launch (rows set by the caller) the expressions are
the same and only the compiler's contraction differs: the rounding bars of tests/test_gpu_elastic.py
(1e-12 traces, 1e-11 gradients).  Dense histories come from the tiles in both types: the oracle
within that file's 1e-10 / 1e-4.
"""
import numpy as np
import pytest

from test_gpu_elastic import T, make_case, oracle, rel

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# a tile's extent is 32 x 64 cells with a halo of 8: one tile, one row or column more than a tile holds,
# several tiles with plain ones among them
SIZES = [(30, 62), (31, 63), (17, 110), (56, 49), (150, 141)]


@pytest.mark.parametrize("NX,NY", SIZES)
@pytest.mark.parametrize("K", [1, 8, 40])
def test_tiles_match_one_level_per_launch(orc, ads, cuda, NX, NY, K):
    p, models, srcs, rcvs, nstep = make_case(orc, ads, NX=NX, NY=NY, NSTEP=31, npml=5, nshots=2, uneven=True, seed=8)
    mt = [T(m) for m in models]
    out = []
    for rows in (8, 0):
        plan = ads.ElasticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
        plan.set_forward_kernels(1, rows)
        srcv = plan.pack_srcv([s.srcv for s in srcs])
        obs = plan.forward(*[m * f for m, f in zip(mt, (1.02, 0.97, 1.04))], srcv, K).clone()
        L, g, t = plan.gradient(*mt, srcv, obs, K, want_traces=True)
        out.append((obs.cpu(), t.clone().cpu(), float(L), [x.clone().cpu() for x in g]))
    (o0, t0, L0, g0), (o1, t1, L1, g1) = out
    assert rel(o1, o0) <= 1e-12 and rel(t1, t0) <= 1e-12 and abs(L1 - L0) <= 1e-12 * abs(L0)
    for a, b in zip(g1, g0):
        assert rel(a, b) <= 1e-11


@pytest.mark.parametrize("dtype,bar", [(torch.float64, 1e-10), (torch.float32, 1e-4)])
@pytest.mark.parametrize("NX,NY", SIZES)
def test_history_matches_oracle(orc, ads, cuda, NX, NY, dtype, bar):
    p, models, srcs, rcvs, nstep = make_case(orc, ads, NX=NX, NY=NY, NSTEP=25, npml=5, nshots=1, seed=9)
    plan = ads.ElasticPlan(p, srcs, rcvs, dtype=dtype)
    h = plan.forward_history(*[T(m, dtype) for m in models], plan.pack_srcv([srcs[0].srcv])).cpu().numpy()
    _, hist = oracle(orc, p, models, srcs[0], rcvs[0], nstep[0])
    ref = np.stack([np.asarray(hist[k]) for k in range(5)]) if not isinstance(hist, np.ndarray) else hist
    assert rel(h.reshape(-1), ref.reshape(-1)) <= bar
