"""Training where hidden units are saturated (large negative sums): SiLU is flat there, so its values are
known far better than their sums and almost none of them has to be formed again in FP64."""
import sys
import time

import numpy as np
import pytest

import phybs_amd as P
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu

SCALES = np.ones(7, np.float32)
HIDDEN_BIASES = (1152, 5312, 9472)


def say(*a):
    print("[gpu-test]", *a, flush=True)
    sys.stdout.flush()


def setup(bias, seed, n):
    rest, tets = P.mesh_bar(2, 2, 4, 0.05)
    s = P.Solver(rest, tets, None, P.default_params())
    model = MO.init_params(seed)
    for o in HIDDEN_BIASES:
        model[o:o + 64] = bias
    s.learn_set_model(model, SCALES)
    rng = np.random.default_rng(seed)
    return s, model, rng.normal(0, 1, (n, 18)).astype(np.float32), rng.normal(0, 1, (n, 3)).astype(np.float32)


def bf(a):
    return MO.bf16(a.astype(np.float32)).astype(np.float64)


def loss_grad_64(model, f, t):
    """64 bits with the same BF16 roundings (of inputs, weights and exact hidden activations)."""
    p = list(zip(*MO.unpack(model, np.float64)))
    h, z = [bf(f)], []
    for k, (w, b) in enumerate(p):
        z.append(h[-1] @ bf(w) + b)
        h.append(bf(MO.silu(z[-1])) if k < 3 else z[-1])
    diff = h[-1] - t
    d, g = 2 * diff / diff.size, []
    for k in range(3, -1, -1):
        g = [(h[k].T @ d).reshape(-1), d.sum(0)] + g
        if k:
            d = (d @ bf(p[k][0]).T) * MO.dsilu(z[k - 1])
    return (diff ** 2).mean(), np.concatenate(g)


@pytest.mark.parametrize("bias", [-1.3, -3.0, -6.0, -12.0, "mixed"])
@pytest.mark.parametrize("n", [65, 5003])
def test_gradient_with_saturated_units(n, bias):
    """Against 64 bits.  FP32 rounding of deltas and sums is 2e-7 of the gradient; saturated hidden layers
    leave the output layer's bias gradients, sums over the samples of deltas of either sign, which cancel
    to a part of their size: up to 10 times that.  -1.3 is where SiLU's slope vanishes."""
    s, model, f, t = setup(np.linspace(-14, 4, 64) if bias == "mixed" else bias, n, n)
    loss, g = s.learn_loss_grad(f, t)
    lref, gref = loss_grad_64(model, f, t)
    err = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    say("saturated units", n, bias, "loss", loss, lref, "grad rel err %.2e" % err)
    assert loss == pytest.approx(lref, rel=1e-6) and err <= 2e-6
    s.close()


def test_saturated_units_cost_no_more():
    """A batch of 20,000 samples: units at -8, -12 and -20 against the usual ones, at most twice the time
    (formed again in FP64 they took up to 11 times as long)."""
    times = {}
    for bias in (0.0, -8.0, -12.0, -20.0):
        s, _, f, t = setup(bias, 1, 20000)
        runs = []
        for _ in range(20):
            t0 = time.perf_counter()
            s.learn_loss_grad(f, t)
            runs.append(time.perf_counter() - t0)
        times[bias] = float(np.median(runs[5:]))
        s.close()
    say("saturated units, us a call", {b: round(1e6 * v, 1) for b, v in times.items()})
    assert max(times.values()) <= 2 * times[0.0]


@pytest.mark.parametrize("z", [-80.0, -84.9, -85.1, -90.0, -1e4, -1e20, -1e36, 20.0, 120.0])
def test_units_at_the_ends_of_the_range(z):
    """One unit of the first layer with a bias of z, the others usual: loss and gradient against 64 bits
    (SiLU and its slope are 0 for any large negative z).  Tolerance as above."""
    s, model, f, t = setup(0.0, 3, 257)
    model[1152 + 5] = z
    s.learn_set_model(model, SCALES)
    loss, g = s.learn_loss_grad(f, t)
    with np.errstate(over="ignore"):
        lref, gref = loss_grad_64(model, f, t)
    err = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    say("a unit at", z, "loss", loss, lref, "grad rel err %.2e" % err)
    assert loss == pytest.approx(lref, rel=1e-6) and err <= 2e-6
    s.close()
