"""Branched molecules on 1-gradient lattices: one workgroup with the rows in
LDS (the automatic choice) against the oracle and the grid path, from one
site per thread to several, wherever the molecule stands among the others,
and in a batch."""
import numpy as np
import pytest

from tests.golden.branched_cases import BRANCHED
from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle

ONE = sorted(k for k in BRANCHED if "1d" in k)


def with_layers(text, n):
    lines = text.split("\n")
    return "\n".join("lat : %s : n_layers : %d" % (l.split(":")[1].strip(), n) if ": n_layers :" in l else l
                     for l in lines)


@pytest.mark.gpu
@pytest.mark.parametrize("case", ONE)
@pytest.mark.parametrize("layers", [9, 62, 63, 64, 300])
def test_fused_schedule_matches_oracle_and_grid(case, layers):
    from namics_amd import ScfSystem, scf
    t = with_layers(BRANCHED[case]["text"], layers)
    o = Oracle(t)
    x = np.random.default_rng(layers).uniform(-0.2, 0.2, o.nvar)
    go, _ = o.residual(x)
    ro = o.results()
    for mode in (scf.MODE_AUTO, scf.MODE_GRID):
        s = ScfSystem(t, mode=mode)
        print(case, layers, mode, flush=True)
        g, _ = s.residual(x)
        r = s.results()
        for m in o.mol_names:
            assert rel_err(r["mol"][m]["GN"], ro["mol"][m]["GN"]) < 1e-12
        for sn in o.seg_names:
            assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < 1e-12
        assert scaled_err(g, go) < 1e-11
        s.close()


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["auto", "grid"])
def test_branched_molecule_after_the_solvent(mode):
    """The densities of a branched molecule that is not the first one."""
    from namics_amd import ScfSystem, scf
    t = BRANCHED["branch1d_head"]["text"]
    mols = [l for l in t.split("\n") if l.startswith("mol : surf")]
    t = "\n".join(l for l in t.split("\n") if l not in mols) + "\n".join([""] + mols) + "\n"
    o = Oracle(t)
    assert o.mol_names[-1] == "surf"
    s = ScfSystem(t, mode=scf.MODE_AUTO if mode == "auto" else scf.MODE_GRID)
    x = np.random.default_rng(4).uniform(-0.2, 0.2, o.nvar)
    g, _ = s.residual(x)
    go, _ = o.residual(x)
    r, ro = s.results(), o.results()
    for sn in o.seg_names:
        assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < 1e-12
    assert scaled_err(g, go) < 1e-11


@pytest.mark.gpu
def test_batch_and_alone_agree():
    from namics_amd import ScfSystem, solve_batch
    texts = [with_layers(BRANCHED[c]["text"], n) for c, n in zip(ONE, (20, 80, 40, 150))]
    texts = [t + "newton : isaac : method : DIIS\nnewton : isaac : iterationlimit : 6\n" for t in texts]
    a, b = [ScfSystem(t) for t in texts], [ScfSystem(t) for t in texts]
    xs = [np.random.default_rng(i).uniform(-0.1, 0.1, s.nvar) for i, s in enumerate(a)]
    got, _ = solve_batch(b, xs)
    for s, x, y in zip(a, xs, got):
        assert np.array_equal(s.solve(x)[0], y)


@pytest.mark.gpu
def test_tuning_times_the_fused_schedule():
    """The tuner has both routes of a branched system as candidates, and the
    faster one, the fused one here, stays in use for systems of the shape
    built later."""
    from namics_amd import ScfSystem, autotune_forget, scf
    autotune_forget()
    t = with_layers(BRANCHED["branch1d_head"]["text"], 60)
    try:
        s = ScfSystem(t)
        x = np.random.default_rng(2).uniform(-0.2, 0.2, s.nvar)
        fused = s.residual(x)[0]
        rep = s.autotune(evals=3)
        print(rep, flush=True)
        assert sorted(c["mode"] for c in rep["candidates"]) == ["fused", "grid"]
        assert rep["candidates"][rep["chosen"]]["mode"] == "fused"
        later = ScfSystem(t)
        for k in (s, later):
            assert np.array_equal(k.residual(x)[0], fused)
            k.close()
        grid = ScfSystem(t, mode=scf.MODE_GRID)  # an explicit mode leaves nothing to choose
        assert grid.autotune(evals=1)["candidates"] == []
        grid.close()
    finally:
        autotune_forget()
