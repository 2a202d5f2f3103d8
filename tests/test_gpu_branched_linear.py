"""Branched molecules next to linear ones on 1-gradient lattices: the linear
molecule's end points checkpointed, against the oracle and the grid path;
second-order linear molecules, which the grid path refuses."""
import numpy as np
import pytest

from tests.helpers import rel_err, scaled_err
from tests.oracle_lib import Oracle

EPS = np.finfo(float).eps


def text(layers, N, fjc, extra=""):
    """A branched surfactant and a linear (A)N in a solvent; fjc > 1: a refined
    hexagonal lattice."""
    lattice = "lat : flat : FJC_choices : %d\nlat : flat : lattice_type : hexagonal\n" % (2 * fjc + 1) if fjc > 1 \
        else "lat : flat : lattice_type : simple_cubic\n"
    return """
lat : flat : gradients : 1
lat : flat : n_layers : %d
%smon : A : freedom : free
mon : C : freedom : free
mon : W : freedom : free
mon : A : chi_W : 0.5
mon : C : chi_W : 0.9
mol : surf : composition : (C)6(A)1[(A)2][(C)1](A)1
mol : surf : freedom : restricted
mol : surf : theta : 1.5
mol : pol : composition : (A)%d
mol : pol : freedom : free
mol : pol : phibulk : 0.01
%smol : water : composition : (W)1
mol : water : freedom : solvent
newton : isaac : method : DIIS
""" % (layers, lattice, N, extra)


@pytest.mark.gpu
@pytest.mark.parametrize("fjc", [1, 2, 3])
@pytest.mark.parametrize("how", ["save_memory", "set_checkpoint"])
def test_checkpointed_linear_molecule(fjc, how):
    from namics_amd import ScfSystem, scf
    N = 100
    t = text(30, N, fjc, "mol : pol : save_memory : true\n" if how == "save_memory" else "")
    o = Oracle(t)
    x = np.random.default_rng(fjc).uniform(-0.2, 0.2, o.nvar)
    go, _ = o.residual(x)
    ro = o.results()
    # rows of N steps with 2 fjc + 1 products each, summed over all of them
    tol = 8 * (2 * fjc + 1) * N * EPS
    got = []
    for mode in (scf.MODE_AUTO, scf.MODE_GRID):
        s = ScfSystem(t, mode=mode)
        if how == "set_checkpoint":
            s.set_checkpoint(4)
        assert s.checkpoint_interval() > 1
        print(how, "fjc", fjc, "mode", mode, flush=True)
        g, _ = s.residual(x)
        r = s.results()
        for m in o.mol_names:
            assert rel_err(r["mol"][m]["GN"], ro["mol"][m]["GN"]) < tol
        for sn in o.seg_names:
            assert scaled_err(s.interior(r["seg_phi"][sn]), o.interior(ro["seg_phi"][sn])) < tol
        assert scaled_err(g, go) < 8 * tol
        got.append(g)
        s.close()
    assert np.array_equal(got[0], got[1])


@pytest.mark.gpu
@pytest.mark.parametrize("layers,fjc", [(40, 1), (280, 4)])
def test_second_order_linear_molecule_is_refused(layers, fjc):
    """Also where the branched rows alone fit LDS and the linear ones (18 rows
    of 1128 sites) do not."""
    from namics_amd import ScfError, ScfSystem
    s = ScfSystem(text(layers, 20, fjc, "mol : pol : Markov : 2\nmol : pol : k_stiff : 0.5\n"))
    with pytest.raises(ScfError):
        s.residual(np.zeros(s.nvar))
    s.close()
