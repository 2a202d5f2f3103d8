"""1-gradient chains that the wave tiles do not serve and one site per thread
does: second order on periodic lattices and on more layers than sixteen waves
own, both orders with a weight on a surface ghost (a tagged segment in the
surface layer); against the oracle."""
import numpy as np
import pytest

from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle
from tests.test_gpu_chain_tiles import text

EPS = np.finfo(float).eps
COMP, N = "(A)3(B)1(A)7(B)20", 31


def check(t):
    from namics_amd import ScfSystem
    o, s = Oracle(t), ScfSystem(t)
    x = np.random.default_rng(o.M).uniform(-0.3, 0.3, o.nvar)
    g, _ = s.residual(x)
    go, _ = o.residual(x)
    r, ro = s.results(), o.results()
    # a row is N steps of at most 8 roundings each, GN and the densities sums
    # of positive products of two rows
    tol = 32 * N * EPS
    for m in o.mol_names:
        assert rel_err(r["mol"][m]["GN"], ro["mol"][m]["GN"]) < tol
    for sn in o.seg_names:
        assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < tol
    assert scaled_err(g, go) < 8 * tol
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("layers,geometry,bound", [(3, "planar", "periodic"), (62, "planar", "periodic"),
                                                   (300, "planar", "periodic"), (1022, "planar", "periodic"),
                                                   (894, "planar", "mirror"), (895, "planar", "mirror"),
                                                   (1022, "planar", "mirror"), (1023, "planar", "mirror"),
                                                   (950, "cylindrical", "mirror"), (950, "spherical", "mirror")])
def test_second_order(layers, geometry, bound):
    check(text(layers, COMP, 2, geometry, bound, bound))


@pytest.mark.gpu
@pytest.mark.parametrize("markov", [1, 2])
@pytest.mark.parametrize("geometry", ["planar", "spherical"])
def test_weight_on_a_surface_ghost(markov, geometry):
    t = text(70, "(A)14(X)1(B)16", markov, geometry, "surface", "mirror")
    t = t.replace("mol : pol : freedom : free\nmol : pol : phibulk : 0.01\n", "mol : pol : freedom : tagged\n")
    check(t + "mon : X : freedom : tagged\nmon : X : tagged_range : lowerbound\n")
