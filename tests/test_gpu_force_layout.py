"""The force passes where their layout can go wrong: every rule size (the paired
sums of 3 and 5 points, the general loop of the others), every lanes-per-pair
schedule, one to four types, tables that do not vanish at the cutoff (the points
beyond it read the tables' zero row instead of being tested), and sites with
fewer pairs inside the cut than a round or a half wavefront, and with more; and
the site table of the mobility sweeps, which has the same lanes and edges.
Against the FP64 oracle: forces and densities to 1e-12 (a few hundred double
roundings), 1e-5 with FP32 quadrature sums."""
import numpy as np
import pytest

from tests.conftest import rel_inf

pytestmark = pytest.mark.gpu


def _check(ff, orc, bound):
    en, eo = ff.force_calc(1), orc.force_calc(1)
    assert abs(en[0] - eo[0]) <= bound * abs(eo[0])
    assert rel_inf(en[1:], eo[1:]) <= bound
    for name in ("f", "E", "dE"):
        assert rel_inf(ff.get(name), orc.get(name)) <= bound, name


def _check_rates(ff, orc, bound, names=("E", "dE", "n", "c_d")):
    """the site table through the sweeps that read it; bound: a few hundred double roundings"""
    for m in (ff, orc):
        m.create_2nd_neigh_lst()
        m.c_d_calc()
    for name in names:
        assert rel_inf(ff.get(name), orc.get(name)) <= bound, name


@pytest.mark.parametrize("no_i", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("nt,parts", [(1, 2), (2, 1), (2, 2), (2, 4), (3, 1), (3, 2), (4, 2)])
def test_rules_and_schedules(nt, parts, no_i):
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    tables = W.johnson_tables(elements=("Ni", "Cu", "Pd", "Ag")[:nt], nr=2001, nrho=2001)
    end = 1e-3 * (1.0 + np.arange(nt * nt).reshape(nt, nt))
    tables.rho = tables.rho + end[:, :, None]  # not zero at the cutoff
    tables.rphi = tables.rphi + 1e-3
    lat = W.fcc_alloy(6, nt=nt, seed=40 + no_i)
    for precision, bound in (("fp64", 1e-12), ("mixed", 1e-5)):
        ff = setup(lat, tables, no_i=no_i, precision=precision)
        ff.set_schedule([parts, 4, 0, 2, 0])
        orc = O.make(lat, tables, no_i=no_i)
        _check(ff, orc, bound)
        if parts == 2:
            _check_rates(ff, orc, bound, ("E", "dE", "n", "c_d") if precision == "fp64" else ("E", "dE"))
        ff.close()


@pytest.mark.parametrize("nt,parts", [(1, 4), (2, 4), (3, 4), (4, 1), (4, 4)])
def test_record_runs(nt, parts):
    """rounds of pass 1 that write less than a run of the records, or several"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    tables = W.johnson_tables(elements=("Ni", "Cu", "Pd", "Ag")[:nt], nr=2001, nrho=2001)
    lat = W.fcc_alloy(6, nt=nt, seed=30 + nt)
    orc = O.make(lat, tables, no_i=3)
    for precision, bound in (("fp64", 1e-12), ("mixed", 1e-5)):
        ff = setup(lat, tables, no_i=3, precision=precision)
        ff.set_schedule([parts, 4, 0, 2, 0])
        _check(ff, orc, bound)
        ff.close()


@pytest.mark.parametrize("nt,parts", [(1, 2), (2, 1), (2, 2), (2, 4), (3, 2), (4, 2)])
@pytest.mark.parametrize("lo,hi,odd", [(3000.0, 4000.0, 0), (10.0, 20.0, 0), (3000.0, 4000.0, 3), (10.0, 20.0, 3)])
def test_rounds_without_quadrature(nt, parts, lo, hi, odd):
    """every pair classical, or every pair skipped (rounds that evaluate no rule), and all but those of
    neighbouring cells; energy_calc over the triangle and over every ordered pair (lanes that fetch no row)"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    tables = W.johnson_tables(elements=("Ni", "Cu", "Pd", "Ag")[:nt], nr=2001, nrho=2001)
    lat = W.fcc_alloy(6, nt=nt, seed=70 + nt, alpha_lo=lo, alpha_hi=hi)
    if odd:
        lat.x[: 4 * odd, 3:] = 60.0 if lo < 100.0 else 500.0
    orc = O.make(lat, tables, no_i=3)
    for precision, bound in (("fp64", 1e-12), ("mixed", 1e-5)):
        ff = setup(lat, tables, no_i=3, precision=precision)
        ff.set_schedule([parts, 4, 0, 2, 0])
        _check(ff, orc, bound)
        for full in (False, True):
            ff.set_energy_mode(full)
            orc.set_energy_full(full)
            e, eo = ff.energy_calc(), orc.energy_calc()
            assert abs(e - eo) <= bound * abs(eo)
        ff.set_energy_mode(False)
        orc.set_energy_full(False)
        ff.close()


@pytest.mark.parametrize("no_i", [13, 14])
def test_longest_rules(tables, no_i):
    """the general loop at its end, with and without a point of zero weight"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    lat = W.fcc_alloy(6, seed=no_i)
    for parts in (1, 2, 4):
        ff, orc = setup(lat, tables, no_i=no_i), O.make(lat, tables, no_i=no_i)
        ff.set_schedule([parts, 4, 0, 2, 0])
        _check(ff, orc, 1e-12)
        _check_rates(ff, orc, 1e-12)
        ff.close()


@pytest.mark.parametrize("keep", [1, 2, 5, 33, 200])
def test_few_and_many_pairs(tables, keep):
    """a cluster in a large box: from no pair at all to a whole half wavefront and more"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    lat = W.fcc_alloy(6, seed=9)
    order = np.argsort(np.linalg.norm(lat.cart - lat.cart.mean(axis=0), axis=1), kind="stable")[:keep]
    L = 60.0
    x = lat.x[order].copy()
    x[:, :3] = (lat.cart[order] - lat.cart.mean(axis=0) + 0.5 * L) / L
    # closer than the lattice: up to about 60 pairs inside the cut for one site
    x[:, :3] = 0.5 + (x[:, :3] - 0.5) * 0.85
    box = W.Lattice(H=np.diag([L] * 3), x=np.ascontiguousarray(x), c=np.ascontiguousarray(lat.c[order]),
                    cart=x[:, :3] * L)
    ff = setup(box, tables, no_i=3)
    orc = O.make(box, tables, no_i=3)
    _check(ff, orc, 1e-12)
    _check_rates(ff, orc, 1e-12)
    ff.close()


@pytest.mark.parametrize("no_i", [1, 3, 5])
@pytest.mark.parametrize("alpha_min", [0.25, 1.0, 30.0])
@pytest.mark.parametrize("nt", [1, 2, 4])
def test_widths_far_from_alpha_min(nt, alpha_min, no_i):
    """the site table leaves out the pairs inside the cut (set by alpha_min) whose rules end beyond rc at
    their own widths: with alpha_min far below the widths most pairs near the cut, with alpha_min among
    the pair widths few (and rates beyond e^100, not compared); widths from 20 to 300.  In FP64 with tables that do not vanish at the cutoff
    (with FP32 sums a point within rounding of it would count or not); the bars of the rates above"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    lat = W.fcc_alloy(6, nt=nt, seed=60 + no_i)
    rng = np.random.default_rng(no_i)
    lat.x[:, 3:] = np.exp(rng.uniform(np.log(20.0), np.log(300.0), size=lat.c.shape))
    a = rng.uniform(-0.2, 0.2, size=lat.c.shape)
    for precision, bound in (("fp64", 1e-12), ("mixed", 1e-5)):
        tables = W.johnson_tables(elements=("Ni", "Cu", "Pd", "Ag")[:nt], nr=2001, nrho=2001)
        if precision == "fp64":
            tables.rho = tables.rho + 1e-3
            tables.rphi = tables.rphi + 1e-3
        ff = setup(lat, tables, no_i=no_i, precision=precision, alpha_min=alpha_min)
        orc = O.make(lat, tables, no_i=no_i, alpha_min=alpha_min)
        if precision == "mixed":
            orc.force_calc(1)
            _check_rates(ff, orc, bound, ("E", "dE"))
        else:
            _check(ff, orc, bound)
            _check_rates(ff, orc, bound, ("E", "dE", "n") if alpha_min == 30.0 else ("E", "dE", "n", "c_d"))
        if precision == "fp64" and alpha_min < 30.0:
            cost_o, g_o = orc.calc_g(0, 0.37, a)
            ff.set_vec("a", a)
            assert abs(ff.calc_g(0, 0.37) - cost_o) <= bound * abs(cost_o)
            assert rel_inf(ff.get("g"), g_o) <= bound
        ff.close()
