"""A plan holds no state of a call in flight, a replayed graph belongs to the buffers of its call, and the
settings of a plan hold over their whole range."""
import ctypes as C
import threading

import numpy as np
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


@pytest.mark.parametrize("kernel", [0, 1])
def test_graphs_follow_the_snapshot_count(orc, ads, cuda, kernel):
    """The snapshot count moves the arrays behind the checkpoints within an unchanged workspace buffer: with
    graphs on, a gradient after fewer snapshots and for another model equals the one without graphs, bit
    for bit, and again when the first count returns."""
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=40, NY=36, NSTEP=90, npml=8, nshots=2, kernel=kernel, seed=6)
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv, K = plan.pack_srcv([s.srcv for s in srcs]), 8
    tr = torch.empty(plan.trace_elems, dtype=torch.float64, device="cuda")
    cot = T(np.random.default_rng(1).standard_normal(plan.trace_elems))
    ws = torch.empty(plan.workspace_size(K), dtype=torch.uint8, device="cuda")  # one-level: the largest
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    P = lambda t: C.c_void_p(t.data_ptr())

    def pullback(m):
        g = torch.empty_like(m)
        assert plan.lib.ads_acoustic_plan_forward(plan.h, P(m), P(srcv), P(tr), P(ws), ws.numel(), K, st) == 0
        assert plan.lib.ads_acoustic_plan_backward(plan.h, P(m), P(srcv), P(cot), P(g), P(ws), ws.numel(), K, st) == 0
        torch.cuda.synchronize()
        return g

    steps = [(-1, T(c)), (2, T(0.93 * c)), (0, T(1.04 * c)), (-1, T(0.97 * c))]
    want = []
    for S, m in steps:
        plan.set_snapshots(S)
        want.append(pullback(m))
    plan.set_graph(True)
    for (S, m), w in zip(steps, want):
        plan.set_snapshots(S)
        for _ in range(3):
            assert torch.equal(pullback(m), w), S
    plan.set_graph(False)


def test_shots_per_adjoint_workgroup_up_to_the_largest_int(orc, ads, cuda):
    """set_shape takes any positive number of shots per workgroup; more than the plan has mean all of them."""
    p, c, srcs, rcvs, nstep = make_case(orc, ads, NX=40, NY=36, NSTEP=60, npml=8, nshots=3, kernel=1, seed=7, uneven=True)
    plan = ads.AcousticPlan(p, srcs, rcvs, dtype=torch.float64, nstep=nstep)
    srcv = plan.pack_srcv([s.srcv for s in srcs])
    obs = plan.forward(T(1.03 * c), srcv, 9).clone()
    out = []
    for sg in (3, 4, 2**31 - 1):
        plan.set_shape((2, sg, 1, 2, sg, 1))
        out.append(plan.gradient(T(c), srcv, obs, 9)[1].clone())
    assert torch.equal(out[1], out[0]) and torch.equal(out[2], out[0])
