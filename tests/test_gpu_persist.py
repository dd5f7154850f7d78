"""The resident descent loop (one cooperative launch per step, small meshes) against the three
launches per pass: the same iterates bit for bit, over sizes from one workgroup to the largest it
takes, precisions, materials, fixed and rel-grad steps, external forces, rollbacks, both semantics."""
import sys

import numpy as np
import pytest

import meshgen as M
import phybs_amd as P

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def run(dims, gp, steps=3, twist=30.0, **kw):
    rest, tets = M.bar(*dims, 0.05)
    mask = M.clamp_x0(rest)
    s = P.Solver(rest, tets, mask, P.default_params(graph_passes=gp, **kw))
    s.set_positions(M.twisted_state(rest, *dims, 0.05, twist, 0.01, 1))
    ext = np.zeros_like(rest)
    ext[-5:, 1] = 0.3
    st = [s.step(ext if k == 1 else None) for k in range(steps)]
    out = s.positions(f64=True), s.velocities(), st
    s.close()
    return out


CASES = [
    ((1, 1, 1), dict()),                                                     # 8 nodes: one workgroup
    ((2, 3, 5), dict(precision=P.FP64)),                                     # two
    ((4, 4, 16), dict()),
    ((4, 4, 16), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000)),
    ((4, 4, 16), dict(precision=P.FP64, alpha0=0.4)),                        # rolls back
    ((4, 4, 16), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000, alpha0=0.4)),
    ((4, 4, 16), dict(material=P.MAT_STRETCH)),
    ((5, 3, 9), dict(material=P.MAT_STRETCH, precision=P.FP64, semantics=P.SEM_REF_CPU)),
    ((4, 4, 16), dict(iterations=1)),
    ((4, 4, 16), dict(iterations=0)),
    ((12, 12, 50), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=20000)),
    ((4, 4, 16), dict(iterations=5000)),                                     # ends in rollbacks
    ((6, 6, 40), dict(precision=P.FP64, relgrad_tol=1e-7, max_iterations=9000, profile=[])),  # several launches
    ((17, 18, 60), dict()),                                                  # 110 K tets: two tets per thread
    ((17, 18, 60), dict(precision=P.FP64, material=P.MAT_STRETCH, iterations=40)),
    ((24, 25, 60), dict()),                                                  # 216 K tets
    ((24, 25, 60), dict(precision=P.FP64)),
]


@pytest.mark.parametrize("dims,kw", CASES)
def test_resident_loop_matches_launches(dims, kw):
    say("resident loop", dims, kw)
    xa, va, sa = run(dims, 0, **kw)
    xb, vb, sb = run(dims, 32, **kw)
    say("passes", [q.passes for q in sa], "rollbacks", [q.rollbacks for q in sa], "gpu ms", [round(q.gpu_ms, 2) for q in sa],
        [round(q.gpu_ms, 2) for q in sb])
    for a, b in zip(sa, sb):
        assert (a.passes, a.iterations, a.rollbacks, a.converged, a.alpha) == (b.passes, b.iterations, b.rollbacks, b.converged, b.alpha)
        # FP64 sums of the same terms in another order
        assert a.g_norm == pytest.approx(b.g_norm, rel=1e-11) and a.g0_norm == pytest.approx(b.g0_norm, rel=1e-11)
        assert a.energy == pytest.approx(b.energy, rel=1e-11)
    assert np.array_equal(xa.view(np.uint64), xb.view(np.uint64))
    assert np.array_equal(va[0].view(np.uint32), vb[0].view(np.uint32))


def test_two_threads_step_at_once():
    """Two solvers of one device stepped from two threads, descent and projective dynamics: each gives
    what it gives alone (launches that hold the whole device take turns, they do not block each other)."""
    from concurrent.futures import ThreadPoolExecutor

    rest, tets = M.bar(12, 12, 50, 0.05)
    mask = M.clamp_x0(rest)
    x0 = M.twisted_state(rest, 12, 12, 50, 0.05, 20.0, 0.005, 1)

    def work(kind):
        s = P.Solver(rest, tets, mask, P.default_params(precision=P.FP64))
        s.set_positions(x0)
        for _ in range(6):
            s.pd_step() if kind else s.step()
        out = s.positions(f64=True)
        s.close()
        return out

    alone = [work(k) for k in (0, 1)]
    say("two threads")
    for kinds in ((0, 0), (0, 1), (1, 1)):
        with ThreadPoolExecutor(2) as pool:
            for k, x in zip(kinds, pool.map(work, kinds)):
                assert np.array_equal(x.view(np.uint64), alone[k].view(np.uint64))
