"""The 3-gradient chains of the 6-point stencil as tiles over many workgroups
against the oracle, at the edges of the tiles (24 layers owned in z, 4 to 16
in x and 8 or 16 in y, a halo of 4) and of the launches of four steps, with
mirrors and periodic images, every row kept and checkpoints between them."""
import numpy as np
import pytest

from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle

EPS = np.finfo(float).eps


def text(nx, ny, nz, comp, periodic):
    bounds = ""
    for d in periodic:
        bounds += "lat : L : lowerbound_%s : periodic\nlat : L : upperbound_%s : periodic\n" % (d, d)
    return """
lat : L : gradients : 3
lat : L : n_layers_x : %d
lat : L : n_layers_y : %d
lat : L : n_layers_z : %d
lat : L : lattice_type : simple_cubic
%smon : A : freedom : free
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
""" % (nx, ny, nz, bounds, comp, 0.1 * nx * ny * nz)


SIZES = [(4, 3, 3, "(A)2", 2), (5, 17, 25, "(A)5", 5), (17, 8, 24, "(A)6", 6), (13, 33, 23, "(A)1(B)8", 9),
         (8, 9, 49, "(A)3(B)1(A)6", 10), (25, 16, 7, "(B)1(A)16", 17)]


@pytest.mark.gpu
@pytest.mark.parametrize("periodic", ["", "xyz", "y", "xz"])
def test_boxes_match_oracle(periodic):
    from namics_amd import ScfSystem, scf
    for nx, ny, nz, comp, N in SIZES:
        print(periodic, nx, ny, nz, comp, flush=True)
        t = text(nx, ny, nz, comp, periodic)
        s, o = ScfSystem(t, mode=scf.MODE_GRID), Oracle(t)
        x = np.random.default_rng(o.M).uniform(-0.3, 0.3, o.nvar)
        g, _ = s.residual(x)
        go, _ = o.residual(x)
        r, ro = s.results(), o.results()
        # a row is N steps of 8 roundings, GN and the densities sums of
        # positive products of two rows
        tol = 32 * N * EPS
        assert rel_err(r["mol"]["pol"]["GN"], ro["mol"]["pol"]["GN"]) < tol
        for sn in o.seg_names:
            assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < tol
        assert scaled_err(g, go) < 8 * tol
        # checkpoints: launches are cut at other rows, which moves no bit
        for K in (2, 4, 7):
            if N > 8:
                s.set_checkpoint(K)
                gk, _ = s.residual(x)
                assert np.array_equal(g, gk), K
        s.close()
