"""The live-unit lists of a batch at their edges: classes of one unit, fewer
units than queues or than a wavefront, more than one block of the list, and
molecules that converge many iterations before the others, so that most units
of the late builds are dead.  Every energy within 1e-9 Eh of the molecule's
own run, as for any batch.  Both converge to ||dP|| < 1e-10 and iteration
counts are not compared: the DIIS equations of two electrons are singular, so
that H2's runs at 1e-8 end after 10 to 13 iterations and 2e-9 Eh apart from
one call to the next, with or without a batch."""
import pytest

from geometries import H2, HELIUM, WATER, water_cluster

pytestmark = pytest.mark.gpu

BIG = water_cluster(5, 9.0, seed=8, perturb=True)


@pytest.mark.parametrize("geoms,basis", [([HELIUM, HELIUM], "sto-3g"), ([H2, HELIUM, H2], "6-31g"),
                                         ([WATER, HELIUM], "6-31gs"), ([HELIUM, BIG, H2, WATER], "6-31g")])
def test_units_of_live_molecules(geoms, basis):
    from mmd.batch import run_batch_device
    from mmd.molecule import Molecule
    res = run_batch_device(geoms, basis, group=len(geoms), conver=1e-10)
    for g, r in zip(geoms, res):
        m = Molecule(g, basis)
        m.RHF(doPrint=False, direct=True, conver=1e-10)
        print("%d functions: batch %.10f (%d it)  single %.10f (%d it)" % (r["nbasis"], r["energy"], r["iterations"],
                                                                          m.energy.real, m.iterations))
        assert r["converged"] and m.is_converged
        assert abs(r["energy"] - m.energy.real) < 1e-9
