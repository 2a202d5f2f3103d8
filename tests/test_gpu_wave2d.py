"""The 2-gradient chains that hold the whole lattice in registers (one
workgroup) against the oracle, at the edges of their lanes (64, 128 and 256
layers along y for 1, 2 and 4 per lane) and columns (8, 4 and 2 per wave), for
every boundary and stencil they serve; and their checkpoint intervals, on
chip and through memory, against full storage."""
import numpy as np
import pytest

from tests.oracle_lib import Oracle
from tests.test_gpu_tile2d import LATTICES, check, text

SIZES = [(3, 3, "(A)2", 2), (16, 63, "(A)8", 8), (17, 64, "(A)9", 9), (9, 65, "(A)1(B)5", 6), (12, 127, "(A)7", 7),
         (8, 128, "(A)3(B)1(A)7", 11), (13, 128, "(A)4", 4), (5, 129, "(B)1(A)6", 7), (4, 200, "(A)5", 5),
         (7, 256, "(A)3", 3), (128, 5, "(A)6", 6)]


@pytest.mark.gpu
@pytest.mark.parametrize("geometry,lattice,periodic", LATTICES)
def test_registers_match_oracle(geometry, lattice, periodic):
    from namics_amd import ScfSystem, scf
    for mx, my, comp, N in SIZES:
        t = text(mx, my, comp, geometry, lattice, periodic)
        print(geometry, lattice, periodic, mx, my, comp, flush=True)
        s = ScfSystem(t, mode=scf.MODE_FUSED)
        check(s, Oracle(t), N)
        s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("mx,my", [(16, 40), (16, 101), (64, 128), (8, 200), (32, 256)])
def test_checkpoint_intervals_equal_full_storage(mx, my):
    from namics_amd import ScfSystem
    t = text(mx, my, "(B)1(A)12(B)5(A)5", "cylindrical", "simple_cubic", "")
    s = ScfSystem(t)
    assert s.layout()["strip_sx"] > 0
    x = np.random.default_rng(my).uniform(-0.2, 0.2, s.nvar)
    want = s.residual(x)
    for K in (2, 3, 4, 5, 7, 22, 23, 40):
        print(mx, my, "interval", K, flush=True)
        s.set_checkpoint(K)
        g, r = s.residual(x)
        assert r == want[1] and np.array_equal(g, want[0]), K


@pytest.mark.gpu
def test_tuned_shapes_still_batch():
    """A shape whose layout was tuned on one system serves batches: the tuner
    keeps one workgroup per system where a chain has such a layout."""
    from namics_amd import ScfSystem, autotune_batch, autotune_forget
    from namics_amd.workloads import brush_cylinder
    autotune_forget()
    try:
        for nr, nz in ((64, 128), (43, 101)):
            t = brush_cylinder(0.5, n_r=nr, n_z=nz, N=60)
            s = ScfSystem(t)
            s.autotune(evals=3)
            assert s.layout()["mode"] == "fused"
            s2 = ScfSystem(t)
            autotune_batch([s, s2], evals=1)
            s.close()
            s2.close()
    finally:
        autotune_forget()


@pytest.mark.gpu
def test_tuner_times_the_grid_path_where_nothing_else_runs():
    """Checkpoints off the strips and branched molecules run on the grid path
    alone: the one candidate, which is not remembered for the shape."""
    from namics_amd import ScfSystem, autotune_batch, autotune_forget
    from namics_amd.workloads import brush_cylinder
    from tests.golden.branched_cases import BRANCHED
    autotune_forget()
    plain = brush_cylinder(0.5, n_r=43, n_z=101, N=60)
    try:
        for t in (plain + "mol : brush : save_memory : true\n", BRANCHED["branch2d_lipid"]["text"]):
            s = ScfSystem(t)
            rep = s.autotune(evals=2)
            assert [c["mode"] for c in rep["candidates"]] == ["grid"] and rep["chosen"] == 0
            assert s.layout()["mode"] == "grid"
            s.close()
        s = ScfSystem(plain)
        assert s.layout()["mode"] == "fused"
        autotune_batch([s], evals=1)
        s.close()
    finally:
        autotune_forget()
