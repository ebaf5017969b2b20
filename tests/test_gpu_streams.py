"""Contexts made and destroyed one after the other, many at a time and from several threads: the streams of a
destroyed context are kept for a moment and destroyed by a later call.  J and K are integer sums, so every context's have the same bits; V_xc and
the gradient come from fixed orders of FP64 sums (atomic ones for the gradient's: 1e-10)."""
import threading

import numpy as np
import pytest

from helpers import bench_molecule, random_density
from iqcp_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _use(eng, b, D, ref, xyz, w, xc):
    jk = eng.build_jk(D)
    assert np.array_equal(jk.J, ref["J"]) and np.array_equal(jk.K, ref["K"])
    if xc:
        eng.set_grid(xyz, w)
        assert np.array_equal(eng.xc(D)[0], ref["V"])
        assert np.abs(eng.xc_gradient(D) - ref["g"]).max() < 1e-10


def test_gpu_contexts_in_turn_and_from_threads():
    b = bench_molecule("H2O", "6-31g*")
    rng = np.random.default_rng(1)
    xyz, w = b.xyz[rng.integers(0, b.natom, 500)] + rng.normal(0.0, 1.5, (500, 3)), rng.uniform(0.0, 0.5, 500)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    eng = Engine(b)
    jk = eng.build_jk(D)
    eng.set_grid(xyz, w)
    ref = dict(J=jk.J, K=jk.K, V=eng.xc(D)[0], g=eng.xc_gradient(D))
    eng.build_grid(30)
    e_ks = eng.ks_scf()["energy_total"]
    eng.close()
    for alive in (1, 1, 20, 20, 3):
        engs = [Engine(b) for _ in range(alive)]
        for i, e in enumerate(engs):
            _use(e, b, D, ref, xyz, w, i % 2 == 0)
        for e in engs:
            e.close()
    eng = Engine(b)
    eng.build_grid(30)
    assert abs(eng.ks_scf()["energy_total"] - e_ks) < 1e-8
    eng.close()
    errors = []

    def work(k):
        try:
            for i in range(6):
                e = Engine(b)
                _use(e, b, D, ref, xyz, w, (i + k) % 2 == 0)
                e.close()
        except BaseException as x:  # noqa: BLE001
            errors.append(x)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
