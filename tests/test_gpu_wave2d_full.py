"""2-gradient chains in registers where every lane and column lies inside the
lattice (64, 128 or 256 layers) and on shapes that no strip divides: against the
oracle."""
import numpy as np
import pytest

from tests.oracle_lib import Oracle
from tests.test_gpu_tile2d import LATTICES, check, text

FULL = [(8, 64, "(A)2", 2), (24, 64, "(A)3(B)1(A)7", 11), (6, 64, "(A)4", 4), (4, 128, "(A)5", 5), (6, 128, "(A)9", 9),
        (2, 256, "(A)6", 6), (32, 256, "(B)1(A)5", 6)]
EDGES = [(16, 63, "(A)8", 8), (17, 63, "(A)8", 8), (13, 127, "(A)7", 7), (5, 200, "(A)5", 5), (127, 5, "(A)6", 6),
         (16, 65, "(A)4", 4), (16, 83, "(A)1(B)5", 6), (16, 84, "(A)1(B)5", 6)]


@pytest.mark.gpu
@pytest.mark.parametrize("geometry,lattice,periodic", LATTICES)
def test_match_oracle(geometry, lattice, periodic):
    from namics_amd import ScfSystem, scf
    for mx, my, comp, N in FULL + EDGES:
        t = text(mx, my, comp, geometry, lattice, periodic)
        print(geometry, lattice, periodic, mx, my, comp, flush=True)
        s = ScfSystem(t, mode=scf.MODE_FUSED)
        check(s, Oracle(t), N)
        s.close()
