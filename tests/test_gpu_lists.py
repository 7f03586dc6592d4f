"""The neighbour lists where the build can go wrong: boxes hardly wider than the
ghost shell (a site is a ghost at both faces), a few candidates per site, more than the kept accept bits cover (1024) and more than one group of 64
rounds (4096); rows and reverse lists of more than 64 entries.  Lists, ghosts
and the 2nd list are the oracle's, entry for entry; the reverse list is what the
densities of partners come from (a few thousand double roundings)."""
import numpy as np
import pytest

from tests.conftest import rel_inf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,a", [(2, 3.6), (4, 1.8), (5, 2.4), (6, 1.45), (7, 3.6), (3, 5.0)])
def test_lists_of_sparse_and_dense_boxes(tables, n, a):
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    lat = W.fcc_alloy(n, a=a, seed=n)
    ff, orc = setup(lat, tables, no_i=3), O.make(lat, tables, no_i=3)
    for m in (ff, orc):
        m.force_calc(1)
        m.create_2nd_neigh_lst()
    pairs = [(ff.neighbor_list(), orc.neighbor_list()), (ff.neighbor_list2(), orc.neighbor_list2()),
             (ff.ghosts(), orc.ghosts())]
    for got, want in pairs:
        for g, w in zip(got, want):
            assert np.array_equal(g, w)
    off, nl = pairs[0][0]
    owned = np.bincount(nl[nl < len(off) - 1], minlength=1)
    print(n, a, "row", np.diff(off).max(), "reverse", owned.max(initial=0), flush=True)
    ff.c_d_calc()
    orc.c_d_calc()
    for name in ("E", "dE", "n"):  # the rates of the dense boxes overflow
        assert rel_inf(ff.get(name), orc.get(name)) <= 1e-11, name
    ff.close()
