"""The FP32 grid of orthogonal cells: boxes of 16^3 points, atoms farther than
8 half widths summed at 8^3 Chebyshev nodes, beyond 40 half widths at 5^3
(ff_grid_f32.hip box_f32), against
the FP64 oracle where that split can go wrong: too few far atoms for the
polynomial (11, with one Coulomb point 15) and just enough (12, 16), one LDS tile of 256 atoms and one more,
no far atom and no near atom at all, more near atoms than a box lists (512),
partial boxes, unequal steps, both models and stencils, uncharged atoms, an
atom that is not finite.

Bound at every point: |dF| <= 2e-6 S, S the sum over the atoms of the sizes of
the terms that the kernel adds (repulsion and attraction, W / r0^3 and each
w_s (1/r_s^3 - 1/r0^3) of the stencil): a term is rounded some 30 times at 6e-8
each (1.8e-6; the 30 rarely all point one way), and the polynomials add up to
6e-7 of a far atom's force (H, 6 A from a side of its box).  For the dz2 tip S is
the sizes of stencil terms that cancel, so the error as a whole is compared with
that of the sum over every pair too."""

import numpy as np
import pytest

import oracle as O
from ppafm_amd import batch as B
from ppafm_amd import common as C
from ppafm_amd import device as D
from ppafm_amd import molgen as M

pytestmark = pytest.mark.gpu

DZ2 = (np.array([-10.0, 20.0, -10.0, 0.0]), np.array([0.1, 0.0, -0.1, 0.0]))
MONOPOLE = (np.array([-0.1, 0, 0, 0]), np.zeros(4))


def _atoms(xyz, seed, uncharged=False):
    rng = np.random.default_rng(seed)
    Zs = rng.choice([1, 6, 7, 8, 79], len(xyz))
    qs = rng.uniform(-0.3, 0.3, len(xyz))
    if uncharged:
        qs[::2] = 0.0
    return qs, C.REA2LJ(C.getAtomsREA(8, Zs, C.loadSpecies(), alphaFac=-1.0))


def _build(n, L, xyz, qs, cLJs, tip):
    model = D.ff_model(1, with_lj=True, stencil=list(zip(*tip)), with_energy=True, fmax=None)
    return D.ff_build(n, np.diag(L), np.concatenate([xyz, qs[:, None]], 1), cLJs, model, f64=False).download()


def _shell(count, L, lo, hi, seed):
    """Atoms lo to hi A outside the cell."""
    rng = np.random.default_rng(seed)
    out = []
    while len(out) < count:
        p = rng.uniform(-hi, hi + max(L), 3)
        d = np.linalg.norm(np.maximum(np.maximum(-p, p - np.array(L)), 0))
        if lo <= d <= hi:
            out.append(p)
    return np.array(out)


def _bound(n, L, xyz, qs, cLJs, tip, ke=14.399644):
    ax = [np.arange(m) * (l / m) for m, l in zip(n, L)]
    S = np.zeros(n)
    for p, q, (c6, c12) in zip(xyz, qs, cLJs):
        d = [a - v for a, v in zip(ax, p)]
        rxy2 = (d[0] ** 2)[:, None, None] + (d[1] ** 2)[None, :, None]
        r0 = np.sqrt(rxy2 + (d[2] ** 2)[None, None, :])
        t = sum(tip[0]) / r0**3
        t = abs(t) * r0 + abs(sum(w * z for w, z in zip(*tip))) / r0**3
        for w, z in zip(*tip):
            d3 = abs(w) * abs(1 / np.sqrt(rxy2 + ((d[2] + z) ** 2)[None, None, :]) ** 3 - 1 / r0**3)
            t = t + d3 * (r0 + abs(z))
        S += 12 * c12 / r0**13 + 6 * c6 / r0**7 + abs(q) * ke * t
    return 2e-6 * S


def _check(G, FE, bound):
    err = np.linalg.norm(G[..., :3] - FE[..., :3], axis=-1)
    print(f"|dF| / bound: max {(err / bound).max():.2f} p50 {np.median(err / bound):.3f}")
    assert (err <= bound).all()


# name, points, step, near atoms (below the cell, 2.5 A and more), far atoms
CASES = [
    ("11 far atoms", (16, 16, 16), (0.1, 0.1, 0.1), 3, 11),
    ("12 far atoms", (16, 16, 16), (0.1, 0.1, 0.1), 3, 12),
    ("15 far atoms", (16, 16, 16), (0.1, 0.1, 0.1), 3, 15),
    ("16 far atoms", (16, 16, 16), (0.1, 0.1, 0.1), 3, 16),
    ("no near atom", (33, 17, 31), (0.1, 0.1, 0.1), 0, 60),
    ("256 atoms", (20, 35, 18), (0.1, 0.1, 0.1), 6, 250),
    ("257 atoms", (20, 35, 18), (0.1, 0.1, 0.1), 6, 251),
    ("unequal steps", (40, 21, 50), (0.12, 0.08, 0.05), 6, 300),
    ("fine steps", (40, 35, 33), (0.03, 0.03, 0.03), 8, 40),
    ("single plane", (1, 19, 2), (0.1, 0.1, 0.1), 4, 40),
    ("few atoms", (16, 32, 15), (0.1, 0.1, 0.1), 5, 0),
]


@pytest.mark.parametrize("tip", [DZ2, MONOPOLE], ids=["dz2", "monopole"])
@pytest.mark.parametrize("name,n,step,near,far", CASES, ids=[c[0] for c in CASES])
def test_box_grid_vs_oracle(name, n, step, near, far, tip):
    print("case:", name, n, step, near, far, flush=True)
    L = [m * s for m, s in zip(n, step)]
    rng = np.random.default_rng(len(name))
    below = np.stack([rng.uniform(-1, L[0] + 1, near), rng.uniform(-1, L[1] + 1, near), rng.uniform(-4.5, -2.5, near)], 1)
    # the far atoms first, the near ones among the last of their tile
    xyz = np.concatenate([_shell(far, L, 6.5, 30.0, 7) if far else np.zeros((0, 3)), below])
    qs, cLJs = _atoms(xyz, 3, uncharged=True)
    G = _build(n, L, xyz, qs, cLJs, tip)
    FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), np.concatenate([xyz, qs[:, None]], 1), cLJs, *tip)
    _check(G, FE, _bound(n, L, xyz, qs, cLJs, tip))
    de = np.abs(G[..., 3] - FE[..., 3]) / np.maximum(np.abs(FE[..., 3]), 1e-3)
    assert de.max() < 1e-3


@pytest.mark.parametrize("mode", ["dz2", "monopole", "separate"])
@pytest.mark.parametrize("veryfar", [1, 11, 270])
def test_second_set_of_nodes(mode, veryfar):
    """More than one tile of atoms, some beyond 40 half widths (30 A): one, one more than the lane groups, a tile and more."""
    n, L = (17, 20, 33), [1.7, 2.0, 3.3]
    xyz = np.concatenate([_shell(veryfar // 2, L, 34.0, 80.0, 11).reshape(-1, 3), _shell(260, L, 3.0, 29.0, 12),
                          _shell(veryfar - veryfar // 2, L, 34.0, 80.0, 13)])
    qs, cLJs = _atoms(xyz, 8, uncharged=True)
    if mode == "separate":
        model = D.ff_model(0, with_lj=True, stencil=D.PROBE_STENCILS["s"], with_energy=True, coulomb_const=C.CoulombConst,
                           probe_q=M.PROBE_Q, fmax=10.0, fp64_radius=0.0)
        G = D.ff_build(n, np.diag(L), np.concatenate([xyz, qs[:, None]], 1), cLJs, model, f64=False).download()
        FE = O.limit_vec_field(O.lj_ff(n, np.diag(L), xyz, cLJs), 10.0) + M.PROBE_Q * O.limit_vec_field(
            O.coulomb_ff(n, np.diag(L), xyz, qs * C.CoulombConst), 10.0)
        bound = _bound(n, L, xyz, qs, cLJs, ([abs(M.PROBE_Q)], [0.0]))
    else:
        tip = DZ2 if mode == "dz2" else MONOPOLE
        G = _build(n, L, xyz, qs, cLJs, tip)
        FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), np.concatenate([xyz, qs[:, None]], 1), cLJs, *tip)
        bound = _bound(n, L, xyz, qs, cLJs, tip)
    _check(G, FE, bound)


def test_more_near_atoms_than_listed():
    """Wide steps (0.5 A: every atom within 30 A is near): 700 near atoms and 100 far ones."""
    n, L = (17, 16, 16), [8.5, 8.0, 8.0]
    xyz = np.concatenate([_shell(350, L, 3.0, 20.0, 1), _shell(100, L, 40.0, 60.0, 2), _shell(350, L, 3.0, 20.0, 3)])
    qs, cLJs = _atoms(xyz, 5)
    G = _build(n, L, xyz, qs, cLJs, MONOPOLE)
    FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), np.concatenate([xyz, qs[:, None]], 1), cLJs, *MONOPOLE)
    _check(G, FE, _bound(n, L, xyz, qs, cLJs, MONOPOLE))


@pytest.mark.parametrize("with_energy", [True, False])
def test_pp_model_far_atoms(with_energy):
    """Separate LJ and Coulomb sums (the ProbeParticle model's clamps)."""
    n, L = (33, 20, 18), [3.3, 2.0, 1.8]
    rng = np.random.default_rng(2)
    xyz = np.concatenate([_shell(200, L, 6.5, 25.0, 4), rng.uniform([0, 0, -3.5], [3.3, 2.0, -0.8], (5, 3))])
    Zs = rng.choice([1, 6, 7, 8], len(xyz))
    qs = rng.uniform(-0.3, 0.3, len(xyz))
    cLJs = C.getAtomsLJ(M.PROBE_Z, Zs, C.loadSpecies())
    model = D.ff_model(0, with_lj=True, stencil=D.PROBE_STENCILS["s"], with_energy=with_energy, coulomb_const=C.CoulombConst,
                       probe_q=M.PROBE_Q, fmax=10.0, fp64_radius=0.0)
    G = D.ff_build(n, np.diag(L), np.concatenate([xyz, qs[:, None]], 1), cLJs, model, f64=False).download()
    FF = O.limit_vec_field(O.lj_ff(n, np.diag(L), xyz, cLJs), 10.0) + M.PROBE_Q * O.limit_vec_field(
        O.coulomb_ff(n, np.diag(L), xyz, qs * C.CoulombConst), 10.0)
    _check(G, FF, _bound(n, L, xyz, qs, cLJs, ([abs(M.PROBE_Q)], [0.0])))


def test_atom_at_infinity_reaches_every_point():
    """An atom whose position is not finite makes every point NaN, as a sum over all atoms does."""
    n, L = (16, 16, 16), [1.6, 1.6, 1.6]
    xyz = _shell(40, L, 7.0, 12.0, 9)
    xyz[20, 1] = np.nan
    qs, cLJs = _atoms(xyz, 1)
    G = _build(n, L, xyz, qs, cLJs, DZ2)
    assert np.isnan(G[..., 1]).all()


def test_batch_of_many_atoms_equals_single_grids():
    lvec = np.array([[-2.0, -2.0, 3.0], [4.0, 0, 0], [0, 4.0, 0], [0, 0, 4.8]])
    n = (40, 40, 48)
    mols = []
    for k, m in enumerate((5, 300)):
        xyz = _shell(m, [4.0, 4.0, 4.8], 3.0, 25.0, 20 + k) + lvec[0]
        rng = np.random.default_rng(k)
        mols.append((xyz, rng.choice([1, 6, 8], m), np.where(np.arange(m) % 3 == 0, 0.0, rng.uniform(-0.2, 0.2, m))))
    b = B.BatchScan.tilted([lvec] * 2, [n] * 2, pos0s=[(0.0, 0.0, 7.0)] * 2, start=(-1, -1), end=(1, 1), scan_n=(8, 8), nz=10,
                           molecules=mols, grid_f64=False)
    b.run_stages(1)
    b.synchronize()
    for k, (xyz, Zs, qs) in enumerate(mols):
        cLJs = C.REA2LJ(C.getAtomsREA(8, Zs, C.loadSpecies(), alphaFac=-1.0))
        G = D.ff_build(n, lvec[1:], np.concatenate([xyz - lvec[0], qs[:, None]], 1), cLJs, b.model, f64=False).download()
        assert np.array_equal(b.grid(k), G), k
    b.close()


def _offset_bound(n, L, xyz, qs, cLJs, tip, ke=14.399644):
    """_bound, and the rounding of a stencil point's distance: its z is the
    sum of two numbers of up to |dz| and |z|, each rounded at 6e-8, and the
    charge's field changes by at most 2 / rs^3 per A."""
    ax = [np.arange(m) * (l / m) for m, l in zip(n, L)]
    S = _bound(n, L, xyz, qs, cLJs, tip, ke)
    for p, q in zip(xyz, qs):
        d = [a - v for a, v in zip(ax, p)]
        rxy2 = (d[0] ** 2)[:, None, None] + (d[1] ** 2)[None, :, None]
        for w, z in zip(*tip):
            rs = np.sqrt(rxy2 + ((d[2] + z) ** 2)[None, None, :])
            S = S + abs(q * w) * ke * 2 / rs**3 * (6e-8 * (2 * np.abs(d[2]) + abs(z)))[None, None, :]
    return S


@pytest.mark.parametrize("lj", ["without LJ", "zero coefficients", "LJ"])
@pytest.mark.parametrize("step", [0.02, 0.05, 0.1])
@pytest.mark.parametrize("offset", [1.0, -2.5, 3.0, -6.0, 8.0])
def test_stencil_points_reach_the_box(offset, step, lj):
    """Atoms more than 8 half widths from the box whose stencil points (the
    tip's z offset) lie beside the box or inside it, and as many whose points
    stay far away: the first must not be summed at the nodes."""
    n, L = (16, 16, 16), [16 * step] * 3
    rng = np.random.default_rng(7)
    near, lo = 7.5 * step, max(8.2 * 7.5 * step, 2.0 if lj == "LJ" else 0.0)  # half width, distance from the box
    xyz = []
    while len(xyz) < 24:
        p = rng.uniform(-2 * near, L[0] + 2 * near, 3)
        p[2] += offset * rng.uniform(0.8, 1.0)  # its charge at dz + offset: beside the box
        if np.linalg.norm(np.maximum(np.maximum(-p, p - L[0]), 0)) >= lo:
            xyz.append(p)
        elif abs(offset) + 2 * near < lo:  # no such atom at this offset: as close as they come
            xyz.append(p + np.array([0, 0, np.sign(offset) * lo]))
    xyz = np.concatenate([np.array(xyz), _shell(24, L, max(lo, 6.1), 20.0, 3)])
    qs, cLJs = _atoms(xyz, 4)
    if lj != "LJ":
        cLJs = np.zeros_like(cLJs)
    tip = (np.array([-0.1, 0.05, 0, 0]), np.array([0.0, offset, 0, 0]))
    model = D.ff_model(1, with_lj=lj != "without LJ", stencil=list(zip(*tip)), with_energy=True, fmax=None)
    G = D.ff_build(n, np.diag(L), np.concatenate([xyz, qs[:, None]], 1), cLJs, model, f64=False).download()
    FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), np.concatenate([xyz, qs[:, None]], 1), cLJs, *tip)
    _check(G, FE, _offset_bound(n, L, xyz, qs, cLJs, tip))


@pytest.mark.parametrize("offset", [6.0, -31.0])
def test_stencil_points_of_very_far_atoms(offset):
    """More than 256 atoms just beyond 40 half widths (30 A) above and below
    the box, whose stencil points lie within them, at 31 A inside the box."""
    n, L = (17, 16, 16), [1.7, 1.6, 1.6]
    rng = np.random.default_rng(1)
    xyz = np.concatenate([rng.uniform([-3, -3, 0], [4.7, 4.6, 1], (300, 3)), _shell(20, L, 3.0, 12.0, 2)])
    xyz[:300, 2] = np.where(np.arange(300) % 2, L[2] + rng.uniform(30.1, 34, 300), -rng.uniform(30.1, 34, 300))
    qs, cLJs = _atoms(xyz, 6)
    tip = (np.array([-0.1, 0.05, 0, 0]), np.array([0.0, offset, 0, 0]))
    G = _build(n, L, xyz, qs, cLJs, tip)
    FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), np.concatenate([xyz, qs[:, None]], 1), cLJs, *tip)
    _check(G, FE, _offset_bound(n, L, xyz, qs, cLJs, tip))


def _slab(z, half, count):
    """Six layers of a square net of Au atoms below z, displaced at random by
    0.05 A (atoms of one height would all round alike), the count nearest to the axis."""
    rng = np.random.default_rng(1)
    ax = np.arange(-half, half + 2.9, 2.9)
    p = np.stack(np.meshgrid(ax, ax, z - 2.35 * np.arange(6), indexing="ij"), -1).reshape(-1, 3)
    return (p + rng.normal(0, 0.05, p.shape))[np.argsort((p[:, :2] ** 2).sum(1), kind="stable")[:count]] + [0.8, 0.8, 0]


SYSTEMS = ["molecule", "ring", "slab", "far slab"]


@pytest.mark.parametrize("tip", [DZ2, MONOPOLE], ids=["dz2", "monopole"])
@pytest.mark.parametrize("system", SYSTEMS)
def test_error_no_larger_than_of_pair_sums(system, tip):
    """The grid is no further from FP64 than the FP32 sum over every pair, which
    the kernel of sheared cells gives for the same points (a shear of 1e-30): root
    mean square of |dF| and of dE over boxes without near atoms, the dz2 tip
    by its own stencil force.  Rounding alone differs, so 5 % are allowed."""
    n, L = (32, 32, 32), [3.2, 3.2, 3.2]
    xyz = {"molecule": lambda: M.molecule(60, 3)[0] * [1, 1, 1] + [1.6, 1.6, -7.5], "ring": lambda: _shell(200, L, 6.2, 12.0, 4),
           "slab": lambda: _slab(-9.0, 70.0, 3000), "far slab": lambda: _slab(-33.0, 90.0, 3000)}[system]()
    rng = np.random.default_rng(2)
    Zs = np.full(len(xyz), 79) if "slab" in system else rng.choice([1, 6, 7, 8], len(xyz))
    qs = np.zeros(len(xyz)) if "slab" in system else rng.uniform(-0.3, 0.3, len(xyz))
    if "slab" in system:
        qs[::40] = 0.1
    cLJs = C.REA2LJ(C.getAtomsREA(8, Zs, C.loadSpecies(), alphaFac=-1.0))
    xyzq = np.concatenate([xyz, qs[:, None]], 1)
    model = D.ff_model(1, with_lj=True, stencil=list(zip(*tip)), with_energy=True, fmax=None)
    FE = O.ljc_qzs_ff(n, np.array([[0, 0, 0], *np.diag(L)]), xyzq, cLJs, *tip)
    e = []
    for shear in (0.0, 1e-30):
        cell = np.diag(L)
        cell[0, 1] = shear
        d = D.ff_build(n, cell, xyzq, cLJs, model, f64=False).download() - FE
        e.append((np.sqrt((d[..., :3] ** 2).sum(-1).mean()), np.sqrt((d[..., 3] ** 2).mean())))
    F, E = np.sqrt((FE[..., :3] ** 2).sum(-1).mean()), np.sqrt((FE[..., 3] ** 2).mean())
    print(f"{system}: force {e[0][0] / F:.2e} pairs {e[1][0] / F:.2e}, energy {e[0][1] / E:.2e} pairs {e[1][1] / E:.2e}")
    assert e[0][0] <= 1.05 * e[1][0]
    assert e[0][1] <= 1.05 * e[1][1]


@pytest.mark.parametrize("items", [1, 8, 17])
def test_batch_of_small_grids_equals_single_grids(items):
    """A box's slabs in 4 blocks (27 boxes alone, and in a batch), in 2 (8 grids: 216 boxes) and in one (17: 459)
    give the same bits, over partial boxes and slabs too."""
    n, L = (37, 40, 47), np.array([3.7, 4.0, 4.7])
    lvec = np.array([[-2.0, -2.0, 3.0], [L[0], 0, 0], [0, L[1], 0], [0, 0, L[2]]])
    mols = []
    for k in range(items):
        rng = np.random.default_rng(k)
        m = (3, 40, 290)[k % 3]
        mols.append((_shell(m, L, 3.0, 25.0, 20 + k) + lvec[0], rng.choice([1, 6, 8], m), rng.uniform(-0.2, 0.2, m)))
    b = B.BatchScan.tilted([lvec] * items, [n] * items, pos0s=[(0.0, 0.0, 7.0)] * items, start=(-1, -1), end=(1, 1), scan_n=(8, 8),
                           nz=10, molecules=mols, grid_f64=False)
    b.run_stages(1)
    b.synchronize()
    for k, (xyz, Zs, qs) in enumerate(mols):
        cLJs = C.REA2LJ(C.getAtomsREA(8, Zs, C.loadSpecies(), alphaFac=-1.0))
        G = D.ff_build(n, lvec[1:], np.concatenate([xyz - lvec[0], qs[:, None]], 1), cLJs, b.model, f64=False).download()
        assert np.array_equal(b.grid(k), G), k
    b.close()
