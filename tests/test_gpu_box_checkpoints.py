"""Checkpoint intervals of the 3-gradient tile chains against full storage on
a lattice of more tiles than run at once, with the interval 3 whose launches
end at checkpoints among them: given by set_checkpoint, and chosen by the
input's save_memory for chains of 9 and 12 segments; FP64 and FP32 rows."""
import numpy as np
import pytest

from tests.test_gpu_box3d import text

NX, NY, NZ = 96, 120, 128  # 720 tiles, three rounds of the 256 compute units


def box(n, save_memory=False):
    t = text(NX, NY, NZ, "(A)%d(B)%d" % (n // 2, n - n // 2), "xyz")
    if save_memory:
        t += "mol : pol : save_memory : true\n"
    return t


def evaluate(s, x, mixed):
    """The residual, and with FP32 rows the fields after two iterations."""
    if not mixed:
        return s.residual(x)[0]
    s.set_precision(True, 1e-6)
    s.set_solver(iterationlimit=2)
    y, it, res, st = s.solve(x)
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [8, 9, 12, 20, 21])
def test_intervals_equal_full_storage(n, mixed):
    from namics_amd import ScfSystem
    s = ScfSystem(box(n))
    assert s.layout()["mode"] == "grid"
    x = np.random.default_rng(n).uniform(-0.2, 0.2, s.nvar)
    want = evaluate(s, x, mixed)
    for K in (2, 3, 5):
        print(n, "interval", K, flush=True)
        s.set_checkpoint(K)
        assert np.array_equal(evaluate(s, x, mixed), want), K
    s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n", [9, 12])
def test_save_memory_chooses_the_interval(n, mixed):
    from namics_amd import ScfSystem
    s, full = ScfSystem(box(n, save_memory=True)), ScfSystem(box(n))
    assert s.checkpoint_interval() == 3
    x = np.random.default_rng(n).uniform(-0.2, 0.2, s.nvar)
    assert np.array_equal(evaluate(s, x, mixed), evaluate(full, x, mixed))
    s.close()
    full.close()
