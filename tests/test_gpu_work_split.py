"""How a build's quartets are dealt to lanes: several lanes per heavily contracted ket, one lane with
several kets, blocks wider than a bra's kets.  J and K against the oracle's integral-direct build for
the sizes where the split changes (one atom with a 36-primitive core pair, one water, a water dimer,
benzene), every basis, both precisions.

Tolerance: J and K are sums of at most a few thousand products of size <= 10 accumulated in fixed
point with steps of 2^-50 or finer (fixacc.h), and the integrals are good to 1e-14 relative, so 1e-11
absolute leaves two orders; mixed precision adds 2^-20 of quartets below 1e-6 each (test_gpu_eri.py),
a few 1e-12 per quartet over at most 1e3 of them: 1e-9."""
import numpy as np
import pytest

import oracle
from helpers import bench_molecule, random_density
from iqcp_amd import workloads
from iqcp_amd.basis import BasisSet, build_basis
from iqcp_amd.engine import BatchEngine, Engine, QcgError

pytestmark = pytest.mark.gpu


def _mol(name, basis):
    if name == "Ne":
        return build_basis([("Ne", (0.0, 0.0, 0.0))], basis)
    if name == "water2":
        return build_basis(workloads.water_cluster((2, 1, 1), 2.9, 3), basis, units="angstrom")
    return bench_molecule(name, basis)


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 1e-9)])
@pytest.mark.parametrize("name,basis", [("Ne", "6-31g"), ("H2O", "sto-3g"), ("H2O", "6-31g*"), ("H2O", "6-31+g*"),
                                        ("water2", "6-31g*"), ("C6H6", "6-31g")])
def test_gpu_jk_split_over_lanes(name, basis, prec, tol):
    b = _mol(name, basis)
    D = random_density(b.nbf, seed=5, nocc=b.n_occ)
    Jo, Ko, _ = oracle.jk_direct(b, D)
    eng = Engine(b, precision=prec)
    jk = eng.build_jk(D)
    assert np.abs(jk.J - Jo).max() < tol and np.abs(jk.K - Ko).max() < tol
    # another split of the same work (tiles set by the caller, bra primitives in ranges) agrees
    eng.set_tiles([(64, 2)] * 21)
    eng.set_prim_split(3)
    jk2 = eng.build_jk(D)
    assert np.abs(jk2.J - jk.J).max() < tol and np.abs(jk2.K - jk.K).max() < tol


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("mixed", 1e-9)])
@pytest.mark.parametrize("name,basis", [("Ne", "6-31g*"), ("H2O", "6-31+g*"), ("water2", "6-31g*")])
def test_gpu_jk_component_parts(name, basis, prec, tol):
    """Per-lane kernels for every class that has one (the largest in parts of the first shell's
    components) and wavefront kernels for every class that has one, J and K together and alone."""
    b = _mol(name, basis)
    D = random_density(b.nbf, seed=8, nocc=b.n_occ)
    Jo, Ko, _ = oracle.jk_direct(b, D)
    eng = Engine(b, precision=prec)
    for tile in [(64, 1), (0, 1), (256, 2)]:
        eng.set_tiles([tile] * 21)
        jk = eng.build_jk(D)
        assert np.abs(jk.J - Jo).max() < tol and np.abs(jk.K - Ko).max() < tol
        assert np.abs(eng.build_jk(D, want_k=False).J - Jo).max() < tol
        assert np.abs(eng.build_jk(D, want_j=False).K - Ko).max() < tol


@pytest.mark.parametrize("name,basis", [("Ne", "6-31g"), ("H2O", "sto-3g"), ("H2O", "6-31+g*"), ("water2", "6-31g*")])
def test_gpu_tensor_split_over_lanes(name, basis):
    """Every element of the compressed tensor (per-lane and wavefront kernels, lanes per ket), and again
    after a change of the Schwarz threshold (the plan is made per threshold).  Elements are below 10 and
    good to 1e-14 relative: 1e-12 absolute."""
    b = _mol(name, basis)
    eng = Engine(b)
    eri, _ = oracle.eri_compressed(b)
    assert np.abs(eng.eri_compressed() - eri).max() < 1e-12
    eng.set_options("mixed", 1e-6, 1e-6)  # the tensor is FP64 in the mixed option too
    dropped = eng.eri_compressed()
    off = np.abs(dropped - eri) > 1e-12
    assert np.all(dropped[off] == 0.0) and np.all(np.abs(eri[off]) < 1e-6)
    assert off.any() or name != "water2"  # an atom's quartets all survive, a dimer's do not


@pytest.mark.parametrize("name,basis", [("H2O", "sto-3g"), ("H2O", "6-31+g*"), ("water2", "6-31g*"), ("C6H6", "6-31g")])
def test_gpu_eri_gradient_split_over_lanes(name, basis):
    """The ERI gradient (lanes per ket, parts of the first shell's components) against five-point
    differences of 1/2 Tr D J - 1/4 Tr D K for one atom.  Step 0.02: the fourth-order remainder,
    h^4 / 30 times a fifth derivative of order 10, is below 1e-7, and the energies (below 1e3, good to
    1e-13) contribute 1e-10 / 0.02: 1e-6.  With the bra primitives in ranges the same sum is made of other
    partial sums: 1e-10."""
    b = _mol(name, basis)
    D = random_density(b.nbf, seed=6, nocc=b.n_occ)
    eng = Engine(b)
    g = eng.eri_gradient(D)
    assert np.abs(g.sum(axis=0)).max() < 1e-9
    eng.set_prim_split(2)
    assert np.abs(eng.eri_gradient(D) - g).max() < 1e-10
    atoms = [(int(z), x.copy()) for z, x in zip(b.Z, b.xyz)]

    def energy(step, axis):
        moved = [(z, x + (step * np.eye(3)[axis] if i == 1 else 0.0)) for i, (z, x) in enumerate(atoms)]
        jk = Engine(build_basis(moved, basis)).build_jk(D)
        return 0.5 * np.sum(D * jk.J) - 0.25 * np.sum(D * jk.K)

    h = 0.02
    for axis in range(3):
        e = {k: energy(k * h, axis) for k in (-2, -1, 1, 2)}
        fd = (8 * (e[1] - e[-1]) - (e[2] - e[-2])) / (12 * h)
        assert abs(fd - g[1, axis]) < 1e-6


def _long_contractions(n):
    """An s shell of n primitives on one atom and a p shell of n on another, each atom with an s of one and a d
    of two: pairs of n^2, 2 n, n and fewer."""
    ex, co, l, nprim, off, atom = [], [], [], [], [], []
    for a in range(2):
        for s, (ls, m) in enumerate([(a, n), (0, 1), (2, 2)]):
            l.append(ls), nprim.append(m), off.append(len(ex)), atom.append(a)
            ex += list(0.15 * 1.7 ** (np.arange(m) + 0.3 * s))
            co += list(0.5 / m + 0.01 * np.arange(m))
    xyz = np.array([[0.0, 0.1, -0.2], [1.1, 0.4, 0.7]])
    i32 = lambda v: np.array(v, dtype=np.int32)  # noqa: E731
    nc = [(k + 1) * (k + 2) // 2 for k in l]
    return BasisSet(name="long", Z=i32([1, 1]), xyz=xyz, shell_l=i32(l), shell_nprim=i32(nprim), shell_prim_off=i32(off),
                    shell_atom=i32(atom), shell_center=xyz[atom], shell_bf_off=i32(np.cumsum([0] + nc[:-1])),
                    exps=np.array(ex), coefs=np.array(co), nbf=sum(nc), nelec=2)


@pytest.mark.parametrize("n", [15, 16, 17])
def test_gpu_tensor_of_long_contractions(n):
    """The compressed tensor of shell pairs with 225, 256 and 289 primitive pairs.  An element is a sum of up to
    n^4 = 8e4 primitive terms of one sign pattern, each good to 1e-14: 1e-12 of the largest element.  J/K and
    the gradient go to 255 primitive pairs and refuse more, as before."""
    b = _long_contractions(n)
    eng = Engine(b)
    eri, _ = oracle.eri_compressed(b)
    assert np.abs(eng.eri_compressed() - eri).max() < 1e-12 * np.abs(eri).max()
    D = random_density(b.nbf, seed=2, nocc=1)
    if n * n <= 255:
        Jo, Ko, _ = oracle.jk_direct(b, D)
        jk = eng.build_jk(D)
        assert max(np.abs(jk.J - Jo).max(), np.abs(jk.K - Ko).max()) < 1e-11 * np.abs(Jo).max()
    else:
        for call in (eng.build_jk, eng.eri_gradient):
            with pytest.raises(QcgError, match="255 primitive pairs"):
                call(D)


@pytest.mark.parametrize("n", [35, 45, 62])
def test_gpu_jk_rows_of_k_out_of_lds(n):
    """J and K of 525, 675 and 930 functions (neon atoms 40 bohr apart), where first (dd|ss), then the classes
    with nine rows and a staged table, last those without a table keep their K rows in memory; per-lane
    kernels forced for the classes in parts too."""
    b = build_basis([("Ne", (40.0 * (i % 8), 40.0 * (i // 8), 0.0)) for i in range(n)], "6-31g*")
    D = random_density(b.nbf, seed=3, nocc=b.n_occ)
    Jo, Ko, _ = oracle.jk_direct(b, D)
    eng = Engine(b)
    for tile in (None, (64, 1), (256, 2)):
        if tile:
            eng.set_tiles([tile] * 21)
        jk = eng.build_jk(D)
        assert np.abs(jk.J - Jo).max() < 1e-11 * np.abs(Jo).max() and np.abs(jk.K - Ko).max() < 1e-11 * np.abs(Ko).max()
    assert np.abs(eng.build_jk(D, want_j=False).K - Ko).max() < 1e-11 * np.abs(Ko).max()


@pytest.mark.parametrize("names", [["H"], ["H", "He"], ["He", "H2O", "H"], ["CH4", "H", "H2O", "NH3", "He", "C6H6"]])
def test_gpu_batch_ket_arrays(names):
    """Batches whose classes have none, one and several blocks of 256 pairs, atoms of s shells among them: J and K
    of every molecule against the oracle, sums of FP64 terms, 1e-11 of the largest element."""
    bases = [build_basis([(n, (0.1, 0.2, 0.3))], "6-31g*") if n in ("H", "He") else bench_molecule(n, "6-31g*") for n in names]
    Ds = [random_density(b.nbf, seed=3, nocc=max(1, b.n_occ)) for b in bases]
    J, K = BatchEngine(bases).build_jk(Ds)
    for b, D, j, k in zip(bases, Ds, J, K):
        Jo, Ko, _ = oracle.jk_direct(b, D)
        assert np.abs(j - Jo).max() < 1e-11 * np.abs(Jo).max() and np.abs(k - Ko).max() < 1e-11 * np.abs(Ko).max()
