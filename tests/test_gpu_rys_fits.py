"""Rys nodes and weights on the device at the ends of the fit intervals and around the large-T limit,
against the exact rule in 50-digit arithmetic.

Tolerance: the fits are good to 1e-15 relative; Estrin's scheme rounds about ten times on the way from
a coefficient to the value, with a sum of |coefficients| below twice the value: 2.5e-15 more.  5e-15."""
import importlib.util
from pathlib import Path

import numpy as np
import pytest

from helpers import bench_molecule
from iqcp_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 7])
def test_gpu_rys_fit_edges(n):
    pytest.importorskip("mpmath")
    src = Path(__file__).parent.parent / "iqcp_amd" / "csrc" / "gen_rys_table.py"
    spec = importlib.util.spec_from_file_location("genrys", src)
    g = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(g)
    tmax = g.tmax_for(n)
    ends = [t for t, _ in g.intervals(n, tmax)][::4] + [tmax]
    T = np.array([v for t in ends for v in (np.nextafter(t, -1.0), t, np.nextafter(t, 1e9), t + 0.11) if v >= 0.0])
    x, w = Engine(bench_molecule("H2O", "sto-3g")).rys_roots(n, T)
    for i, t in enumerate(T):
        ex, ew = g.rys_exact(n, float(t))
        np.testing.assert_allclose(x[i], [float(v) for v in ex], rtol=5e-15)
        np.testing.assert_allclose(w[i], [float(v) for v in ew], rtol=5e-15)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7])
def test_gpu_rys_fit_all_intervals(n):
    """The moments of the rule, sum_i w_i x_i^k = F_k(T) for k < 2n, at, next to and inside every interval of every
    order, against the Boys function in 50-digit arithmetic.  The terms are all positive, each good to k + 1 times
    the tolerance above."""
    mp = pytest.importorskip("mpmath")
    src = Path(__file__).parent.parent / "iqcp_amd" / "csrc" / "gen_rys_table.py"
    spec = importlib.util.spec_from_file_location("genrys", src)
    g = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(g)
    tmax = g.tmax_for(n)
    iv = [(t, h) for t, h in g.intervals(n, tmax)]
    T = np.array([v for t, h in iv for v in (np.nextafter(t, -1.0), t, t + 0.5 * h, t + 0.93 * h) if v >= 0.0])
    x, w = Engine(bench_molecule("H2O", "sto-3g")).rys_roots(n, T)
    for i, t in enumerate(T):
        for k in range(2 * n):
            f = g.boys_mp(k, float(t))
            s = sum(mp.mpf(float(a)) * mp.mpf(float(b)) ** k for a, b in zip(w[i], x[i]))
            assert abs(s / f - 1) < (k + 1) * 5e-15, (t, k)
