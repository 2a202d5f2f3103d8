"""2-gradient chains in registers where every lane and column lies inside the
lattice (64, 128 or 256 layers) and on shapes that no strip divides, and the
layouts on either side of the line between strips and registers: against the
oracle, and their checkpoint intervals against full storage."""
import numpy as np
import pytest

from tests.oracle_lib import Oracle
from tests.test_gpu_tile2d import LATTICES, check, text

FULL = [(8, 64, "(A)2", 2), (24, 64, "(A)3(B)1(A)7", 11), (6, 64, "(A)4", 4), (4, 128, "(A)5", 5), (6, 128, "(A)9", 9),
        (2, 256, "(A)6", 6), (32, 256, "(B)1(A)5", 6)]
EDGES = [(16, 63, "(A)8", 8), (17, 63, "(A)8", 8), (13, 127, "(A)7", 7), (5, 200, "(A)5", 5), (127, 5, "(A)6", 6),
         (16, 65, "(A)4", 4), (64, 65, "(A)4", 4), (64, 66, "(A)4", 4), (16, 83, "(A)1(B)5", 6), (16, 84, "(A)1(B)5", 6)]


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


@pytest.mark.gpu
@pytest.mark.parametrize("mx,my", [(16, 63), (16, 64), (16, 83), (16, 84), (32, 256), (12, 84)])
def test_checkpoint_intervals_equal_full_storage(mx, my):
    from namics_amd import ScfSystem
    t = text(mx, my, "(B)1(A)12(B)5(A)5", "cylindrical", "simple_cubic", "")
    s = ScfSystem(t)
    assert s.layout()["strip_sx"] > 0
    x = np.random.default_rng(my).uniform(-0.2, 0.2, s.nvar)
    want = s.residual(x)
    for K in (2, 3, 4, 5, 22, 23):
        print(mx, my, "interval", K, flush=True)
        s.set_checkpoint(K)
        g, r = s.residual(x)
        assert r == want[1] and np.array_equal(g, want[0]), K
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nr,nz", [(32, 40), (32, 64), (36, 48)])
def test_tuner_times_registers_and_strips(nr, nz):
    """Registers, every strip width that fits, and the generic chain are
    candidates; a later system of the shape gives the chosen one's bits."""
    from namics_amd import ScfSystem, autotune_forget
    from namics_amd.workloads import brush_cylinder
    autotune_forget()
    t = brush_cylinder(0.5, n_r=nr, n_z=nz, N=60)
    try:
        s = ScfSystem(t)
        x = np.random.default_rng(nz).uniform(-0.05, 0.05, s.nvar)
        default = s.residual(x)[0]
        rep = s.autotune(evals=3)
        widths = [sx for sx in (8, 4) if nr % sx == 0 and nr // sx * nz <= 1024]
        assert [c["strip_sx"] for c in rep["candidates"]] == widths[:1] + widths + [0]
        g = s.residual(x)[0]
        assert np.allclose(g, default, rtol=0, atol=1e-12 * np.abs(default).max())
        later = ScfSystem(t)
        assert np.array_equal(later.residual(x)[0], g)
        s.close()
        later.close()
    finally:
        autotune_forget()
