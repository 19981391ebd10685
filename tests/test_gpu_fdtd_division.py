"""The leapfrog's division by h^2 through one reciprocal per thread, and the marched interior on
both sides of the size from which it streams past the caches, against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _levels(amd, oracle_mod, n, h, make, steps):
    dt = h / (np.sqrt(3) * 343 * 1.01)
    g = amd.PPPMSolver(n, h, dt, (0, 0, 0), 0, 0.2, 343.0)
    o = oracle_mod.Oracle(n, h, dt, (0, 0, 0), 343.0, 0.2, oracle_mod.FP64)
    for rel in (-1, 0):
        x = make((n ** 3,))
        g.set_grid(rel, x)
        o.set_grid(rel, x)
    for _ in range(steps):
        g.fdtd_step()
        o.fdtd_step()
    a, b = (np.asarray(v).reshape(n, n, n)[2:-2, 2:-2, 2:-2] for v in (g.get_grid(0), o.grid(0)))
    return a, b


def _same(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)].view(np.uint32),
                                                                       b[~np.isnan(b)].view(np.uint32))


@pytest.mark.parametrize("n", [20, 133])  # a thread per column; marched
@pytest.mark.parametrize("h", [1e-3, 0.0098, 7.25, 3e4])
@pytest.mark.parametrize("kind", ["wide", "subnormal", "special"])
def test_division_bitexact(amd, oracle_mod, n, h, kind):
    rng = np.random.default_rng(n)

    def make(shape):
        x = rng.standard_normal(shape)
        if kind == "wide":  # every exponent of FP32
            return (x * 2.0 ** rng.integers(-149, 120, shape)).astype(np.float32)
        if kind == "subnormal":
            return (x * 1e-40).astype(np.float32)
        x = x.astype(np.float32)
        x[rng.random(shape) < 0.3] = 0.0
        x[rng.random(shape) < 0.2] = -0.0
        x[rng.random(shape) < 0.002] = np.inf
        x[rng.random(shape) < 0.002] = np.nan
        return x

    a, b = _levels(amd, oracle_mod, n, h, make, 1)
    assert _same(a, b)


@pytest.mark.parametrize("n", [322, 323])  # three levels just below and just above 384 MB
def test_stream_rule_bitexact(amd, oracle_mod, n):
    rng = np.random.default_rng(n)
    a, b = _levels(amd, oracle_mod, n, 0.01, lambda shape: rng.standard_normal(shape, dtype=np.float32), 2)
    assert _same(a, b)
