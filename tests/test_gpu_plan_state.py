"""A plan holds no state of a call in flight."""
import ctypes as C
import threading

import pytest

from test_gpu_acoustic import T, make_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel", [0, 1])
def test_two_threads_share_a_plan(orc, ads, cuda, kernel):
    """Two threads run one plan, each with a workspace, a stream and a model of its own: every gradient
    equals the one that the plan gives alone, bit for bit."""
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=60, NY=50, NSTEP=150, npml=12, nshots=2, kernel=kernel, seed=4)
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv, K = plan.pack_srcv([s.srcv for s in srcs]), 6
    models = [T(c), T(0.9 * c)]
    obs = plan.forward(T(1.05 * c), srcv, K).clone()
    alone = [plan.gradient(m, srcv, obs, K)[1].clone() for m in models]
    need = plan.workspace_size(K)
    bad = []

    def work(q):
        with torch.cuda.stream(torch.cuda.Stream()):
            ws = torch.empty(need, dtype=torch.uint8, device="cuda")
            g = torch.empty_like(models[q])
            st = torch.cuda.current_stream()
            for it in range(20):
                rc = plan.lib.ads_acoustic_plan_gradient(
                    plan.h, *[C.c_void_p(t.data_ptr()) for t in (models[q], srcv, obs)], None,
                    C.c_void_p(g.data_ptr()), None, C.c_void_p(ws.data_ptr()), need, K, C.c_void_p(st.cuda_stream))
                st.synchronize()
                if rc != 0 or not torch.equal(g, alone[q]):
                    bad.append((q, it, rc))

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not bad, bad
