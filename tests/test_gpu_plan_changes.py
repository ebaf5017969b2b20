"""Changes of the options between calls on one context: what a call keeps (the captured Fock graph, the
work plan's lists, the tiles) has to follow."""
import numpy as np
import pytest

from helpers import bench_molecule, random_density
from iqcp_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("between", ["build_jk", "build_fock", "eri_gradient", "rhf_scf", "threshold"])
def test_gpu_fock_graph_follows_the_plan(between):
    """FP64 graph build, a call that plans for other options, FP64 graph build again: the second one is
    captured anew, since the plan that the first one held is gone.  J and K are integer sums, so F has the
    eager build's bits each time."""
    import torch
    b = bench_molecule("H2O", "6-31g*")
    eng = Engine(b)
    D, H = random_density(b.nbf, seed=4, nocc=b.n_occ), np.diag(np.linspace(-2.0, 1.0, b.nbf))
    F = eng.build_fock(H, D)
    dH, dD = torch.tensor(H, device="cuda"), torch.tensor(D, device="cuda")
    dF = torch.empty_like(dD)
    st = torch.cuda.Stream()
    eng.set_graph(True)
    for rep in range(3):
        dF.fill_(7.0)
        torch.cuda.synchronize()
        eng.build_fock_device(dH.data_ptr(), dD.data_ptr(), dF.data_ptr(), 0.5, st.cuda_stream)
        torch.cuda.synchronize()
        assert np.array_equal(dF.cpu().numpy(), F)
        if between == "threshold":
            eng.set_options("fp64", 1e-6, 1e-3)
            eng.build_jk(D)
        else:
            eng.set_options("mixed")
            {"build_jk": lambda: eng.build_jk(D), "build_fock": lambda: eng.build_fock(H, D),
             "eri_gradient": lambda: eng.eri_gradient(D), "rhf_scf": eng.rhf_scf}[between]()
        eng.set_options("fp64")
        # memory freed with the old lists is used by others
        junk = [torch.full((n,), -1, dtype=torch.int32, device="cuda") for n in (1 << 10, 1 << 14, 1 << 18)]
        del junk


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_gpu_tiles_read_before_the_first_build(prec):
    """The tiles read before any build are those that the builds choose, so setting them back changes
    nothing: not the tiles, and not a bit of J and K; and they follow the options."""
    b = bench_molecule("C6H6", "6-31g*")
    D = random_density(b.nbf, seed=4, nocc=b.n_occ)
    eng = Engine(b, precision=prec)
    first = eng.get_tiles()
    jk = eng.build_jk(D)
    assert eng.get_tiles() == first
    other = Engine(b, precision=prec)
    other.set_tiles(other.get_tiles())
    jk2 = other.build_jk(D)
    assert other.get_tiles() == first
    assert np.array_equal(jk2.J, jk.J) and np.array_equal(jk2.K, jk.K)
    eng.set_options(prec, 1e-6, 1e-2)  # far fewer quartets, other tiles; read, then back without a build
    changed = eng.get_tiles()
    eng.set_options(prec)
    assert eng.get_tiles() == first and changed != first
    jk3 = eng.build_jk(D)
    assert np.array_equal(jk3.J, jk.J) and np.array_equal(jk3.K, jk.K)
