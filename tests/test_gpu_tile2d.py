"""The 2-gradient chains as tiles over many workgroups (grid path) against
the oracle, at the edges of the tiles (16 columns by 48 layers owned, a halo
of 8) and of the 8-row segments, for every boundary and stencil they serve."""
import numpy as np
import pytest

from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle

EPS = np.finfo(float).eps


def text(mx, my, comp, geometry, lattice, periodic):
    bounds = ""
    for d in periodic:
        bounds += "lat : L : lowerbound_%s : periodic\nlat : L : upperbound_%s : periodic\n" % (d, d)
    return """
lat : L : gradients : 2
lat : L : geometry : %s
lat : L : n_layers_x : %d
lat : L : n_layers_y : %d
lat : L : lattice_type : %s
%s%smon : A : freedom : free
mon : B : freedom : free
mon : W : freedom : free
mon : A : chi_W : 0.5
mon : B : chi_W : 0.9
mol : pol : composition : %s
mol : pol : freedom : restricted
mol : pol : theta : %r
mol : water : composition : (W)1
mol : water : freedom : solvent
newton : isaac : method : DIIS
""" % (geometry, mx, my, lattice, "lat : L : stencil_full : true\n" if geometry == "planar" else "", bounds, comp,
       0.1 * mx * my)


LATTICES = [("cylindrical", "simple_cubic", ""), ("cylindrical", "hexagonal", ""), ("planar", "simple_cubic", ""),
            ("planar", "simple_cubic", "xy"), ("planar", "simple_cubic", "y"), ("planar", "hexagonal", "x")]
SIZES = [(3, 3, "(A)2", 2), (16, 48, "(A)8", 8), (17, 49, "(A)9", 9), (15, 47, "(A)1(B)16", 17), (33, 5, "(A)17", 17),
         (5, 97, "(A)3(B)1(A)7(B)10", 21), (31, 100, "(B)1(A)24", 25), (48, 7, "(A)25(B)1", 26)]


def check(s, o, N):
    x = np.random.default_rng(o.M).uniform(-0.3, 0.3, o.nvar)
    g, res = s.residual(x)
    go, reso = o.residual(x)
    r, ro = s.results(), o.results()
    # a row is N steps of at most 16 roundings each, GN and the densities sums
    # of positive products of two rows
    tol = 64 * N * EPS
    assert rel_err(r["mol"]["pol"]["GN"], ro["mol"]["pol"]["GN"]) < tol
    for sn in o.seg_names:
        assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < tol
    assert scaled_err(g, go) < 8 * tol


@pytest.mark.gpu
@pytest.mark.parametrize("geometry,lattice,periodic", LATTICES)
def test_tiles_match_oracle(geometry, lattice, periodic):
    from namics_amd import ScfSystem, scf
    for mx, my, comp, N in SIZES:
        t = text(mx, my, comp, geometry, lattice, periodic)
        print(geometry, lattice, periodic, mx, my, comp, flush=True)
        s = ScfSystem(t, mode=scf.MODE_GRID)
        check(s, Oracle(t), N)
        s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("save_memory", [False, True])
def test_large_lattices_take_the_tiles_alone(save_memory):
    """A lattice whose rows do not fit LDS: the call's own choice of path, and
    the same with checkpointed storage (which keeps fewer rows)."""
    from namics_amd import ScfSystem, scf
    t = text(101, 131, "(A)12(B)11", "planar", "simple_cubic", "")
    if save_memory:
        t = t.replace("mol : water : comp", "mol : pol : save_memory : true\nmol : water : comp")
    a, b = ScfSystem(t), ScfSystem(t, mode=scf.MODE_GRID)
    check(a, Oracle(t), 23)
    x = np.random.default_rng(2).uniform(-0.1, 0.1, a.nvar)
    assert np.array_equal(a.residual(x)[0], b.residual(x)[0])
    for s in (a, b):
        s.set_solver(iterationlimit=5)
    assert np.array_equal(a.solve(x)[0], b.solve(x)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("n,tiles", [(2, True), (5, True), (6, False), (12, False)])
def test_batches_change_to_one_workgroup_each(n, tiles):
    """97 x 102 layers, 24 segments: up to five systems of a call run as tiles,
    more in one launch of a workgroup each."""
    from namics_amd import ScfSystem, scf, solve_batch
    t = text(97, 102, "(A)12(B)11", "planar", "simple_cubic", "") + "newton : isaac : iterationlimit : 2\n"
    alone = ScfSystem(t, mode=scf.MODE_GRID if tiles else scf.MODE_FUSED)
    systems = [ScfSystem(t) for _ in range(n)]
    xs = [np.random.default_rng(i).uniform(-0.1, 0.1, alone.nvar) for i in range(n)]
    got, _ = solve_batch(systems, xs)
    for x, y in zip(xs, got):
        assert np.array_equal(alone.solve(x)[0], y)
    for s in systems + [alone]:
        s.close()
