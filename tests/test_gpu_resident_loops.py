"""Which loop a step or solve ran in, and what happens when a resident launch's bounded waits end: the
host sets how often a workgroup looks in vain before it gives up, so every kernel ends by itself, and
the step or solve goes on through the launches from the same start, with their bits."""
import sys

import numpy as np
import pytest

import meshgen as M
import phybs_amd as P

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def solver(dims, **kw):
    rest, tets = M.bar(*dims, 0.05)
    s = P.Solver(rest, tets, M.clamp_x0(rest), P.default_params(**kw))
    s.set_positions(M.twisted_state(rest, *dims, 0.05, 2.0, 0.005, 1))
    return s


def bits(s):
    return s.positions(f64=True).view(np.uint64).copy(), s.velocities()[0].view(np.uint32).copy()


@pytest.mark.parametrize("dims,kw,loop", [
    ((1, 1, 1), dict(), P.LOOP_RESIDENT),
    ((4, 4, 16), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000), P.LOOP_RESIDENT),
    ((17, 18, 60), dict(material=P.MAT_STRETCH), P.LOOP_RESIDENT),
    ((24, 25, 60), dict(precision=P.FP64), P.LOOP_RESIDENT),                # 39,650 nodes
    ((24, 25, 61), dict(), P.LOOP_LAUNCHES),                                # 40,300: more than it takes
    ((4, 4, 16), dict(graph_passes=32), P.LOOP_LAUNCHES),
    ((4, 4, 16), dict(tile_tets=64), P.LOOP_LAUNCHES),
    ((4, 4, 16), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=5000, mixed_switch=1e-3), P.LOOP_LAUNCHES),
])
def test_descent_loop_taken(dims, kw, loop):
    say("loop of a step", dims, kw)
    s = solver(dims, **kw)
    assert s.last_loops() == (P.LOOP_NONE, P.LOOP_NONE)
    s.step()
    assert s.last_loops() == (loop, P.LOOP_NONE)
    s.set_profiling(1)
    s.step()
    assert s.last_loops() == (P.LOOP_LAUNCHES, P.LOOP_NONE)
    s.close()


@pytest.mark.parametrize("precision", [P.FP32, P.FP64])
@pytest.mark.parametrize("dims,blocks,scalar", [((1, 1, 1), True, True), ((16, 16, 60), True, True),
                                                ((20, 20, 80), None, True),   # two shares: 3x3 blocks in FP32
                                                ((30, 30, 135), False, True), ((31, 31, 130), False, False)])
def test_cg_loop_taken(dims, blocks, scalar, precision):
    """3x3 blocks (backward Euler), scalar values (projective dynamics)."""
    say("loop of a solve", dims, precision)
    if blocks is None:
        blocks = precision == P.FP32
    s = solver(dims, precision=precision)
    for call, resident in ((s.implicit_step, blocks), (s.pd_step, scalar)):
        call()
        assert s.last_loops()[1] == (P.LOOP_RESIDENT if resident else P.LOOP_LAUNCHES)
    s.set_profiling(1)
    s.pd_step()
    assert s.last_loops()[1] == P.LOOP_LAUNCHES
    s.close()


@pytest.mark.parametrize("kw", [dict(), dict(precision=P.FP64, relgrad_tol=1e-4, max_iterations=20000)])
def test_descent_goes_on_after_giving_up(kw):
    dims = (12, 12, 50)
    a, b = solver(dims, **kw), solver(dims, graph_passes=32, **kw)
    a.set_resident_polls(1)
    say("descent gives up", kw)
    sa, sb = a.step(), b.step()
    assert a.last_loops()[0] == P.LOOP_GAVE_UP and b.last_loops()[0] == P.LOOP_LAUNCHES
    assert (sa.passes, sa.rollbacks, sa.converged) == (sb.passes, sb.rollbacks, sb.converged)
    for loop in (P.LOOP_LAUNCHES, P.LOOP_RESIDENT):
        for p, q in zip(bits(a), bits(b)):
            assert np.array_equal(p, q)
        if loop == P.LOOP_RESIDENT:
            a.set_resident_polls(0)
        a.step(), b.step()
        assert a.last_loops()[0] == loop
    for p, q in zip(bits(a), bits(b)):
        assert np.array_equal(p, q)
    a.close()
    b.close()


@pytest.mark.parametrize("iterations", [1, 2, 10000])
@pytest.mark.parametrize("kind", ["implicit", "pd"])
def test_solve_goes_on_after_giving_up(kind, iterations):
    """Limits from one look to more than a wait takes, from the first exchange on and on the last one
    alone (a solve that ends after one or two iterations): there, some workgroups see all values and end
    with a result while others give up."""
    dims = (20, 20, 80)

    def step(s):
        if kind == "implicit":
            return s.implicit_step(params=P.implicit_params(cg_max_iterations=iterations)).cg_iterations
        return s.pd_step(params=P.pd_params(cg_max_iterations=iterations, iterations=1)).cg_iterations

    ref = solver(dims)
    ref.set_profiling(1)
    its = step(ref)
    want = bits(ref)
    ref.close()
    for start in (0, 2 * its - 1):
        loops = {}
        for polls in (1, 2, 4, 8, 12, 16, 24, 64):
            s = solver(dims)
            s.set_resident_polls(polls, start)
            say("solve gives up", kind, iterations, start, polls)
            got_its = step(s)
            loops[polls] = s.last_loops()[1]
            assert got_its == its
            for p, q in zip(bits(s), want):
                assert np.array_equal(p, q)
            s.close()
        say("loops", loops)
        assert loops[1] == P.LOOP_GAVE_UP


def test_creation_does_not_pay_for_the_resident_loop():
    """A handle that may never step is created in the time of one that cannot run the resident loop (the
    same tiles, by an explicit size); the first step makes what the loop needs."""
    import time

    rest, tets = M.bar(12, 12, 50, 0.05)
    mask = M.clamp_x0(rest)
    s = P.Solver(rest, tets, mask, P.default_params())
    tile = int(s.get_params().tile_tets)
    s.step()
    assert s.last_loops()[0] == P.LOOP_RESIDENT
    s.close()
    times = {0: [], tile: []}
    for _ in range(15):
        for k in times:
            t0 = time.perf_counter()
            s = P.Solver(rest, tets, mask, P.default_params(tile_tets=k))
            times[k].append(time.perf_counter() - t0)
            s.close()
    med = {k: 1e3 * float(np.median(v[3:])) for k, v in times.items()}
    say("creation, ms by tile size", med)
    assert med[0] <= 1.2 * med[tile]
