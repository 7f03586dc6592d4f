"""The neighbour lists where the build can go wrong: boxes hardly wider than the
ghost shell (a site is a ghost at both faces), a few candidates per site, more
than the kept accept bits cover (1024) and more than one group of 64 rounds
(4096); rows and reverse lists of more than 64 entries; boxes with far more bins
than sites, and crowded bins.  Lists, ghosts and the 2nd list are the oracle's,
entry for entry; the reverse list is what the densities of partners come from
(a few thousand double roundings)."""
import numpy as np
import pytest

from tests.conftest import rel_inf

pytestmark = pytest.mark.gpu


def _most_candidates(orc, L, cut):
    """sites and ghosts in the 27 bins (of the shell's width) around an owned site, the largest number"""
    w = cut / L
    b = ((orc.x_all()[:, :3] / L + w) / w).astype(int) + 1
    cnt = np.zeros(b.max(axis=0) + 2, dtype=int)
    np.add.at(cnt, tuple(b.T), 1)
    g = (-1, 0, 1)
    around = sum(np.roll(cnt, (i, j, k), (0, 1, 2)) for i in g for j in g for k in g)
    return around[tuple(b[: orc.natms].T)].max()


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
    # the branch each box stands for
    most = _most_candidates(orc, n * a, tables.rc + 1.2247448713915890 / 5.0 + 0.5)  # alpha_min = 25, skin 0.5
    if a == 1.45:
        assert most > 4096
    elif a in (1.8, 2.4):
        assert 1024 < most <= 4096
    else:
        assert most <= 1024
    if a < 3.0:
        assert np.diff(off).max() > 64 and owned.max() > 64
    ff.c_d_calc()
    orc.c_d_calc()
    for name in ("E", "dE", "n"):  # the rates of the dense boxes overflow
        assert rel_inf(ff.get(name), orc.get(name)) <= 1e-11, name
    ff.close()


@pytest.mark.parametrize("L,n,squeeze", [(100.0, 8, 0.3), (200.0, 6, 1.0), (300.0, 6, 1.0), (300.0, 8, 0.3),
                                         (1500.0, 6, 1.0)])
def test_lists_of_nearly_empty_boxes(tables, L, n, squeeze):
    """4 n^3 sites in two clusters, one across a corner: 8e3 bins (squeezed, several blocks to each by the
    mean of the occupied ones), 5e4 (a block each), 1.7e5 (the list of the occupied ones; squeezed, several
    blocks to each) and 1.8e7 (more than a launch holds blocks)"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    lat = W.fcc_alloy(n, seed=21)
    s = lat.cart * squeeze / L
    s[1::2] += 0.43
    s -= 3.0 / L
    s -= np.floor(s)
    box = W.Lattice(H=np.diag([L] * 3), x=np.ascontiguousarray(np.concatenate([s, lat.x[:, 3:]], axis=1)), c=lat.c,
                    cart=s * L)
    ff, orc = setup(box, tables, no_i=3), O.make(box, tables, no_i=3)
    x = ff.get("x")
    x[3, 0] += 0.8  # past the skin
    for moved in (False, True):
        if moved:
            assert ff.set_x(x) and orc.set_x(x)
        for got, want in ((ff.neighbor_list(), orc.neighbor_list()), (ff.ghosts(), orc.ghosts())):
            for g, w in zip(got, want):
                assert np.array_equal(g, w)
        assert len(orc.neighbor_list()[1]) > 5000 and len(orc.ghosts()[1]) > 100
        en, eo = ff.force_calc(1), orc.force_calc(1)
        # sites to an occupied bin, and more than the 16 of a block where squeezed
        xa, cut = ff.get("x")[:, :3], tables.rc + 1.2247448713915890 / 5.0
        mean = lat.natms / len(np.unique(((xa + cut) / cut).astype(int), axis=0))
        assert mean > 32.0 if squeeze < 1.0 else mean < 16.0
        bound = 1e-12 if squeeze == 1.0 else 1e-11  # more pairs to a site
        assert abs(en[0] - eo[0]) <= bound * abs(eo[0]) and rel_inf(ff.get("f"), orc.get("f")) <= bound
    ff.close()


@pytest.mark.parametrize("L", [8000.0, 9325.0])
def test_box_with_too_many_bins_is_refused(tables, L):
    """2.7e9 bins (negative as a 32-bit product) and 4.3e9 (a small positive one)"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import DMDError, setup
    lat = W.fcc_alloy(2, seed=3)
    box = W.Lattice(H=np.diag([L] * 3), x=lat.x, c=lat.c, cart=lat.x[:, :3] * L)
    with pytest.raises(DMDError) as e:
        setup(box, tables, no_i=3)
    assert e.value.code == -4  # E_RANGE
