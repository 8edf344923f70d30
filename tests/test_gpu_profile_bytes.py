"""The profile's bytes of launches that step several levels: the state once per launch and every level once, fewer
than as many single-level launches move, so that a rate formed with them stays below what the memory gives."""
import ctypes as C
import importlib

import pytest

from test_gpu_acoustic import T, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def profiled(lib, L, cls, run):
    L.check(lib.ads_profile_begin())
    run()
    torch.cuda.synchronize()
    L.check(lib.ads_profile_end())
    tm, n, b = C.c_double(), C.c_int64(), C.c_double()
    L.check(lib.ads_profile_query(cls, C.byref(tm), C.byref(n), C.byref(b)))
    return n.value, b.value


@pytest.mark.parametrize("kernel", [0, 1])
def test_acoustic_tiles(orc, ads, cuda, kernel):
    L = importlib.import_module("adseismic_amd._lib")
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=60, NY=50, NSTEP=101, npml=8, nshots=2, kernel=kernel, seed=4)
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    obs = plan.forward(T(1.03 * c), srcv, 100).clone()
    values = 8.0 * 2 * p.NX * p.NY  # bytes of one value per cell and shot
    for cls, single in ((0, 4), (1, 7)):
        n, b = profiled(plan.lib, L, cls, lambda: plan.gradient(T(c), srcv, obs, 100))
        assert n == 100
        assert values * n < b < values * n * single, (cls, b / values / n)
    plan.set_blocking(1)
    n, b = profiled(plan.lib, L, 0, lambda: plan.forward(T(c), srcv, 100))
    assert n == 100 and b >= values * n * 4


def test_elastic_tiles(orc, ads, cuda):
    from test_gpu_elastic import make_case as elastic_case
    L = importlib.import_module("adseismic_amd._lib")
    p, models, srcs, rcvs, nstep = elastic_case(orc, ads, NX=60, NY=50, NSTEP=40, npml=6, nshots=2)
    plan = ads.ElasticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    n, b = profiled(plan.lib, L, 2, lambda: plan.forward(*[T(m) for m in models], srcv, 40))
    values = 8.0 * 2 * p.NX * p.NY
    whole = 13 + 8 * (2 * 6 / 60 + 2 * 6 / 50)  # of a single-level launch, with CPML strips of 6 cells or more
    assert n == 40
    assert values * n * 5 < b < values * n * whole, b / values / n
