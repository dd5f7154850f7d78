"""The resident CG (one cooperative launch per solve) against its three launches per iteration where a
workgroup has the most ghosts: bars of flat and of elongated cells, whose space-filling-curve order cuts
them into runs with about twice the neighbours of a bar of cubes.  Timed solvers launch every CG kernel
by itself; both paths add the same terms in the same order, so counts, positions and velocities are
equal bit for bit."""
import sys

import numpy as np
import pytest

import meshgen as M
import phybs_amd as P

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def flat_case(dims, cell):
    rest, tets = M.bar(*dims, 1.0)
    rest = (rest * np.asarray(cell, np.float32)).astype(np.float32)
    mask = M.clamp_x0(rest)
    size = rest.max(0)
    q = rest / size
    x = rest + (0.01 * size.min() * q[:, :1] * np.sin(3.0 * q[:, [1, 2, 0]] + 1.0)).astype(np.float32)
    return rest, tets, mask, x.astype(np.float32)


# at most 1304 (60x60x33), 1308, 1208 and 386 ghosts per workgroup; a thread of 8 slices' reads 8 components
@pytest.mark.parametrize("precision", [P.FP32, P.FP64])
@pytest.mark.parametrize("dims,cell", [((60, 60, 33), (0.02, 0.02, 0.2)), ((100, 100, 11), (0.02, 0.02, 0.2)),
                                       ((16, 16, 450), (0.05, 0.05, 0.0025)), ((16, 16, 60), (0.02, 0.02, 0.2))])
def test_resident_cg_reads_every_ghost(dims, cell, precision):
    rest, tets, mask, x0 = flat_case(dims, cell)
    say("resident CG", dims, cell, precision, len(rest))
    out = []
    for prof in (0, 1):
        s = P.Solver(rest, tets, mask, P.default_params(precision=precision))
        s.set_positions(x0)
        s.set_profiling(prof)
        st = [s.pd_step() for _ in range(2)]
        out.append(([q.cg_iterations for q in st], s.positions(f64=True), s.velocities()[0]))
        s.close()
    say("its", out[0][0])
    assert np.isfinite(out[0][1]).all() and np.abs(out[0][1] - x0).max() < 0.1 * np.abs(rest).max()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1].view(np.uint64), out[1][1].view(np.uint64))
    assert np.array_equal(out[0][2].view(np.uint32), out[1][2].view(np.uint32))
