"""The packed FP64 XC build (points sorted into blocks that keep only the functions reaching them) at
the sizes where it can go wrong: grids of 1, 63, 64, 65 and 1000 points, points far from every
function (blocks without any), molecules longer than a function's reach, a change of the precision
option after the grid was made, the library form on the same grid.

Tolerance: V elements are sums over the grid of products of FP64 values of size <= 10 whose weights add
up to the electron number scale; both sides accumulate with rounding below 1e-15 of the largest term
and at most 1e5 terms: 1e-10 absolute, E_xc 1e-10 relative.  The oracle also drops functions below 1e-10
on its 512-point blocks, which is below the same bound after weighting."""
from dataclasses import replace

import numpy as np
import pytest

import oracle
from helpers import bench_molecule, random_density
from iqcp_amd import workloads
from iqcp_amd.basis import build_basis
from iqcp_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _points(b, n, seed, spread=2.5):
    rng = np.random.default_rng(seed)
    at = b.xyz[rng.integers(0, b.natom, n)]
    return at + rng.normal(0.0, spread, (n, 3)), rng.uniform(0.0, 0.5, n)


def _check(b, xyz, w, eng=None):
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    eng = eng or Engine(b)
    eng.set_grid(xyz, w)
    V, E = eng.xc(D)
    chi, grad = oracle.basis_on_grid(b, xyz)
    Vo, Eo, _ = oracle.vxc(chi, grad, w, D)
    assert np.abs(V - Vo).max() < 1e-10 and abs(E - Eo) < 1e-10 * max(1.0, abs(Eo))
    return D, V, E, eng


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 40000])
def test_gpu_packed_point_counts(n):
    _check(bench_molecule("H2O", "6-31g*"), *_points(bench_molecule("H2O", "6-31g*"), n, n))


def test_gpu_packed_far_points_and_long_molecules():
    b = build_basis(workloads.alkane(8, 0.03, 4), "6-31g*", units="angstrom")
    xyz, w = _points(b, 3000, 3)
    far = xyz[:500] + np.array([200.0, 0.0, 0.0])  # no function reaches these
    _check(b, np.concatenate([far, xyz]), np.concatenate([w[:500], w]))
    _check(b, far, w[:500])


@pytest.mark.parametrize("name,basis", [("H2O", "sto-3g"), ("NH3", "6-31+g*"), ("C6H6", "6-31g*")])
def test_gpu_packed_functions_from_radial_parts(name, basis):
    """Blocks without d functions, with tiles of mixed angular momentum, and points out of every reach,
    one of them at infinity, which add nothing."""
    b = bench_molecule(name, basis)
    xyz, w = _points(b, 2000, 5)
    D, V, E, _ = _check(b, xyz, w)
    out = np.array([[1e6, 0.0, 0.0], [0.0, -1e200, 3.0], [np.inf, 0.0, 0.0]])
    eng = Engine(b)
    eng.set_grid(np.concatenate([xyz, out]), np.concatenate([w, np.ones(3)]))
    V2, E2 = eng.xc(D)
    assert np.abs(V2 - V).max() < 1e-10 and abs(E2 - E) < 1e-10 * max(1.0, abs(E))


@pytest.mark.parametrize("n,far,atoms", [(1, 0, 10), (63, 0, 12), (3001, 0, 12), (3001, 700, 10), (3001, 700, 6)])
def test_gpu_mixed_skips_zero_tiles(n, far, atoms):
    """The mixed option's dense kernels leave out K steps and tiles that are zero at their points (a long
    molecule, with points out of every reach in front).  V's elements are sums of FP32 products over at
    most 4e3 points and 234 functions with weights up to 0.5: 6e-8 times a few tens, 1e-5; E_xc 1e-6."""
    b = build_basis(workloads.alkane(atoms, 0.03, 4), "6-31g*", units="angstrom")
    xyz, w = _points(b, n, 7)
    if far:
        xyz = np.concatenate([xyz[:far] + np.array([200.0, 0.0, 0.0]), xyz])
        w = np.concatenate([w[:far], w])
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    eng = Engine(b, precision="mixed")
    eng.set_grid(xyz, w)
    V, E = eng.xc(D)
    chi, grad = oracle.basis_on_grid(b, xyz)
    Vo, Eo, _ = oracle.vxc(chi, grad, w, D)
    assert np.abs(V - Vo).max() < 1e-5 and abs(E - Eo) < 1e-6 * max(1.0, abs(Eo))


def test_gpu_packed_follows_the_options():
    b = bench_molecule("H2O", "6-31g*")
    xyz, w = _points(b, 5000, 8)
    eng = Engine(b, precision="mixed")  # the grid's dense arrays come first
    eng.set_grid(xyz, w)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    Vm, Em = eng.xc(D)
    eng.set_options("fp64")
    _, V, E, _ = _check(b, xyz, w, eng)
    assert np.abs(Vm - V).max() < 1e-4 and abs(Em - E) < 1e-4
    for mode in (1, 2, 0):  # library form on the same grid, then back
        eng.set_xc_mode(mode)
        V1, E1 = eng.xc(D)
        assert np.abs(V1 - V).max() < 1e-10 and abs(E1 - E) < 1e-10 * abs(E)
    eng.set_options("mixed")
    V2, _ = eng.xc(D)
    assert np.array_equal(V2, Vm)


@pytest.mark.parametrize("n", [1, 65, 3000])
def test_gpu_packed_xc_gradient(n):
    """The XC gradient on the packed grid against the oracle's; the sums run over the same products as V
    times basis derivatives below 1e2: 1e-8."""
    b = bench_molecule("H2O", "6-31g*")
    xyz, w = _points(b, n, n, 1.5)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    for prec in ("fp64", "mixed"):  # the gradient is FP64 in both
        eng = Engine(b, precision=prec)
        eng.set_grid(xyz, w)
        g = eng.xc_gradient(D)
        assert np.abs(g - oracle.xc_gradient(b, xyz, w, D)).max() < 1e-8
        assert np.array_equal(eng.xc_gradient(D).shape, (b.natom, 3))


def test_gpu_packed_form_without_room():
    """A grid made for the mixed option whose dense arrays leave no room for the packed ones: the gradient and the
    FP64 build run on the dense arrays.  The card's memory is taken up to 1.9 GB beyond 9 matrices of points by
    functions (Phi, its gradient, X, aow and the FP32 copies); the packed form and its gradient take at least 4 of
    1 GB each.  Tolerances as above."""
    import torch
    b = bench_molecule("C6H6", "6-31g*")
    n = 1_230_000
    unit = 8 * n * b.nbf
    xyz, w = _points(b, 2000, 6)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    ref = Engine(b)
    ref.set_grid(xyz, w)
    (V, E), g = ref.xc(D), ref.xc_gradient(D)
    ref.close()
    eng = Engine(b, precision="mixed")
    eng.eri_gradient(D)
    rep = n // 2000
    big, wb = np.tile(xyz, (rep, 1)), np.tile(w / rep, rep)
    torch.cuda.empty_cache()
    keep = 9 * unit + (14 << 27)
    hog = torch.empty(torch.cuda.mem_get_info()[0] - keep, dtype=torch.uint8, device="cuda")
    try:
        eng.set_grid(big, wb)
        Vm, Em = eng.xc(D)
        g2 = eng.xc_gradient(D)
        eng.set_options("fp64")
        V2, E2 = eng.xc(D)
    finally:
        del hog
        torch.cuda.empty_cache()
    assert np.abs(g2 - g).max() < 1e-8
    assert np.abs(V2 - V).max() < 1e-10 and abs(E2 - E) < 1e-10 * max(1.0, abs(E))
    assert np.abs(Vm - V).max() < 1e-4 and abs(Em - E) < 1e-4


def test_gpu_block_of_more_functions_than_the_packed_kernels_take():
    """One block of 60 points that 380 functions reach: no packed form, so the library form (modes 0 and 1), the
    column-pass MFMA kernels (mode 2) and the library gradient; then points that a part of them reaches."""
    b = build_basis(workloads.water_cluster((5, 2, 2), 2.9, 3), "6-31g*", units="angstrom")
    rng = np.random.default_rng(2)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    eng = Engine(b)
    for _ in range(2):
        xyz, w = b.xyz + rng.normal(0.0, 0.3, b.xyz.shape), rng.uniform(0.0, 0.5, b.natom)
        Vo, Eo, _ = oracle.vxc(*oracle.basis_on_grid(b, xyz), w, D)
        eng.set_grid(xyz, w)
        for mode in (0, 2, 1, 0):
            eng.set_xc_mode(mode)
            V, E = eng.xc(D)
            assert np.abs(V - Vo).max() < 1e-10 and abs(E - Eo) < 1e-10 * max(1.0, abs(Eo)), mode
        assert np.abs(eng.xc_gradient(D) - oracle.xc_gradient(b, xyz, w, D)).max() < 1e-8
        near = b.xyz[0] + rng.normal(0.0, 0.5, (100, 3))
        _check(b, near, rng.uniform(0.0, 0.5, 100), eng)
        assert np.abs(eng.xc_gradient(D) - oracle.xc_gradient(b, near, eng.get_grid()[1], D)).max() < 1e-8


def _reordered(b, order):
    """The basis with its shells in another order."""
    o = np.asarray(order)
    nc = (b.shell_l[o] + 1) * (b.shell_l[o] + 2) // 2
    return replace(b, shell_l=b.shell_l[o], shell_nprim=b.shell_nprim[o], shell_prim_off=b.shell_prim_off[o],
                   shell_atom=b.shell_atom[o], shell_center=np.ascontiguousarray(b.shell_center[o]),
                   shell_bf_off=np.concatenate([[0], np.cumsum(nc)[:-1]]).astype(np.int32))


@pytest.mark.parametrize("first", [1, 2])
def test_gpu_packed_shell_orders(first):
    """Function 0, which stands in for the padding columns of a block, as a p or d function: the p (or d) shells
    first, then the others.  V and E_xc, and the XC gradient twice (its work arrays are kept)."""
    b = bench_molecule("NH3", "6-31+g*")
    b = _reordered(b, np.argsort(b.shell_l != first, kind="stable"))
    assert b.shell_l[0] == first
    xyz, w = _points(b, 2000, 5)
    D, _, _, eng = _check(b, xyz, w)
    g = eng.xc_gradient(D)
    assert np.abs(g - oracle.xc_gradient(b, xyz, w, D)).max() < 1e-8
    eng.xc(random_density(b.nbf, seed=10, nocc=b.n_occ))
    assert np.abs(eng.xc_gradient(D) - g).max() < 1e-10  # its atomic sums arrive in any order


@pytest.mark.parametrize("n", [32767, 32768, 32769, 65537, 131073, 262145, 300000])
def test_gpu_packed_block_sizes(n):
    """Blocks of 64 to 1024 points, the last one full, almost empty or partly filled: V, E_xc and the XC gradient of
    the packed form against the library form on the dense arrays, and the same bits of V from a second set_grid.
    Both are sums of n <= 3e5 terms of size <= 1 rounded below 1e-15 of the largest: 1e-10."""
    b = bench_molecule("H2O", "6-31g*")
    xyz, w = _points(b, n, 3, spread=4.0)
    w = w * (2000.0 / n)
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    eng = Engine(b)
    eng.set_grid(xyz, w)
    V, E = eng.xc(D)
    g = eng.xc_gradient(D)
    eng.set_xc_mode(1)
    Vl, El = eng.xc(D)
    assert np.abs(V - Vl).max() < 1e-10 and abs(E - El) < 1e-10 * max(1.0, abs(El))
    eng.set_xc_mode(0)
    eng.set_grid(xyz, w)
    V2, _ = eng.xc(D)
    assert np.array_equal(V2, V) and np.abs(eng.xc_gradient(D) - g).max() < 1e-10


@pytest.mark.parametrize("n", [10, 11, 16, 18])
def test_gpu_mixed_tiles_of_any_shell_order(n):
    """12 to 22 tiles of 16 functions, the shells in a random order (d shells across two tiles), on a row of waters
    3 angstrom apart, so that most tiles reach few points: the mixed option's V against FP64 products, bounds as
    above."""
    b = build_basis(workloads.water_cluster((n, 1, 1), 3.0, 3), "6-31g*", units="angstrom")
    b = _reordered(b, np.random.default_rng(n).permutation(b.nshell))
    xyz, w = _points(b, 3001, n)
    xyz = xyz[np.argsort(xyz[:, 0])]
    D = random_density(b.nbf, seed=9, nocc=b.n_occ)
    Vo, Eo, _ = oracle.vxc(*oracle.basis_on_grid(b, xyz), w, D)
    eng = Engine(b, precision="mixed")
    eng.set_grid(xyz, w)
    V, E = eng.xc(D)
    assert np.abs(V - Vo).max() < 1e-5 and abs(E - Eo) < 1e-6 * max(1.0, abs(Eo))
