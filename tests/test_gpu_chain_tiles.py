"""The wave-tile chains of 1-gradient lattices against the oracle at the
edges of their tiles (a first-order wave owns 112 positions, a second-order
one 56) and of their row segments (8 and 4 rows), over every boundary and
geometry, with blocks shorter than a segment."""
import numpy as np
import pytest

from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle

EPS = np.finfo(float).eps


def text(layers, comp, markov, geometry, lower, upper):
    wall = ""
    if lower == "surface":
        wall += "mon : S : freedom : frozen\nmon : S : frozen_range : lowerbound\nmon : S : chi_A : -0.7\n"
    if upper == "surface":
        wall += "mon : T : freedom : frozen\nmon : T : frozen_range : upperbound\nmon : T : chi_B : -0.4\n"
    extra = "mol : pol : Markov : 2\nmol : pol : k_stiff : 0.7\n" if markov == 2 else ""
    return """
lat : L : gradients : 1
lat : L : n_layers : %d
lat : L : geometry : %s
%slat : L : lattice_type : simple_cubic
lat : L : lowerbound : %s
lat : L : upperbound : %s
mon : A : freedom : free
mon : B : freedom : free
mon : W : freedom : free
mon : A : chi_W : 0.5
mon : B : chi_W : 0.9
%smol : pol : composition : %s
mol : pol : freedom : free
mol : pol : phibulk : 0.01
%smol : water : composition : (W)1
mol : water : freedom : solvent
newton : isaac : method : DIIS
""" % (layers, geometry, "lat : L : offset_first_layer : 3\n" if geometry == "spherical" else "", lower, upper, wall,
       comp, extra)


# layers + 2 positions: one below, at and above one wave and two waves of
# each order; a lattice smaller than a halo
SIZES = [3, 5, 53, 54, 55, 109, 110, 111, 166, 222, 223]
BOUNDS = [("planar", "surface", "mirror"), ("planar", "mirror", "mirror"), ("planar", "periodic", "periodic"),
          ("planar", "surface", "surface"), ("cylindrical", "mirror", "mirror"), ("spherical", "surface", "mirror"),
          ("spherical", "mirror", "surface")]
# chain lengths around the segments, and blocks that end inside one
COMPS = [("(A)2", 2), ("(A)5", 5), ("(A)8", 8), ("(A)9", 9), ("(A)17", 17), ("(A)3(B)1(A)7(B)20", 31),
         ("(B)1(A)63", 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("markov", [1, 2])
@pytest.mark.parametrize("geometry,lower,upper", BOUNDS)
def test_tiles_match_oracle(geometry, lower, upper, markov):
    from namics_amd import ScfSystem
    for i, layers in enumerate(SIZES):
        comp, N = COMPS[i % len(COMPS)]
        if layers in (54, 110):
            comp, N = COMPS[5]
        t = text(layers, comp, markov, geometry, lower, upper)
        print(geometry, lower, upper, "markov", markov, "layers", layers, comp, flush=True)
        o = Oracle(t)
        s = ScfSystem(t)
        x = np.random.default_rng(layers).uniform(-0.3, 0.3, o.nvar)
        g, res = s.residual(x)
        go, reso = o.residual(x)
        r, ro = s.results(), o.results()
        # a row is N steps of at most 8 roundings each, GN and the densities
        # sums of positive products of two rows
        tol = 32 * N * EPS
        assert rel_err(r["mol"]["pol"]["GN"], ro["mol"]["pol"]["GN"]) < tol
        for sn in o.seg_names:
            assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < tol
        # g subtracts terms of order one over densities of order one
        assert scaled_err(g, go) < 8 * tol
        s.close()


@pytest.mark.gpu
def test_tiles_in_a_wider_launch():
    """A small system gives the same result alone and next to one that
    launches more waves."""
    from namics_amd import ScfSystem, solve_batch
    tiny = text(40, "(A)30", 2, "planar", "surface", "mirror") + "newton : isaac : iterationlimit : 5\n"
    wide = text(400, "(A)30", 2, "planar", "surface", "mirror") + "newton : isaac : iterationlimit : 5\n"
    a, b, c = ScfSystem(tiny), ScfSystem(tiny), ScfSystem(wide)
    x = np.random.default_rng(1).uniform(-0.1, 0.1, a.nvar)
    xa = a.solve(x)[0]
    xs, _ = solve_batch([b, c], [x, np.zeros(c.nvar)])
    assert np.array_equal(xa, xs[0])
