"""Batches whose fields share one packed copy (up to 64 KiB per system) next
to systems copied one by one: the results of solving each alone."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("order", [(0, 1), (0, 1, 2), (2, 0, 1), (2, 2), (0, 2)])
def test_batch_equals_alone(order):
    from namics_amd import ScfSystem, solve_batch
    from namics_amd.workloads import brush_cylinder, homopolymer_adsorption
    # 2 blocks of 42, 2 blocks of 4002 (just below 64 KiB), 3 blocks of 66 x 130 (above)
    texts = [homopolymer_adsorption(40, 30, 0.4, -0.5, 1e-3), homopolymer_adsorption(4000, 3, 0.4, -0.5, 1e-3),
             brush_cylinder(0.5, N=20)]
    alone, mixed, xs, want = [], [], [], []
    for k, i in enumerate(order):
        a, b = ScfSystem(texts[i]), ScfSystem(texts[i])
        for s in (a, b):
            s.set_solver(iterationlimit=4)
        x = np.random.default_rng(k).uniform(-0.05, 0.05, a.nvar)
        want.append(a.solve(x))
        alone.append(a)
        mixed.append(b)
        xs.append(x)
    got, infos = solve_batch(mixed, xs)
    for (x, it, res, st), y, (it2, res2, st2) in zip(want, got, infos):
        assert (it, st, res) == (it2, st2, res2)
        assert np.array_equal(x, y)
