"""GPU parity at the edges of the DMD force field's input domain, through the
C ABI against the FP64 oracle on the same inputs.

Cases:
  - per-site widths spanning the three regimes of the pair width
    alpha = a_i a_j / (a_i + a_j) (src/ff_dmd_I.cpp:178-180, :261-310): pairs
    skipped at or below alpha_min, Gauss-Hermite quadrature in between, the
    classical EAM branch at or above alpha_max, for every mobility variant;
  - concentrations exactly 0 and 1, inside the 1e-8 margin where calc_ent
    returns 0 (src/ff_dmd_I.cpp:2230-2237) and on its edges;
  - a tilted lower-triangular box whose tilts are lattice translations of
    the crystal (ghosts in s-space, bins of the reduced heights);
  - a cluster in vacuum with isolated sites that have no partner in the cut.
Bars: ghosts and both neighbour lists bit-exact; energy, virial, f, E, dE,
energy_calc, c_d, n, calc_g cost and gradient <= 1e-12 relative (infinity
norm over each array)."""
import numpy as np
import pytest

from tests.conftest import rel_inf

pytestmark = pytest.mark.gpu


def _lattice_from_cart(H, cart, alpha, c):
    from mapp_amd import workload as W
    s = W.x2s(cart, W.m3inv(H))
    x = np.concatenate([s, alpha], axis=1)
    return W.Lattice(H=np.asarray(H, dtype=np.float64), x=np.ascontiguousarray(x),
                     c=np.ascontiguousarray(c), cart=cart)


def regime_counts(orc, alpha_min=25.0, alpha_max=1000.0):
    """number of (pair inside rc, ordered type pair) in each width regime:
    skipped, quadrature, classical"""
    nt = orc.nt
    xa = orc.x_all()
    off, nl = orc.neighbor_list()
    i = np.repeat(np.arange(len(off) - 1), np.diff(off))
    d = xa[i, :3] - xa[nl, :3]
    inr = (d * d).sum(axis=1) < 25.0
    out = np.zeros(3, dtype=np.int64)
    for a in range(nt):
        for b in range(nt):
            ai, aj = xa[i[inr], 3 + a], xa[nl[inr], 3 + b]
            al = ai * aj / (ai + aj)
            out += [(al <= alpha_min).sum(), ((al > alpha_min) & (al < alpha_max)).sum(), (al >= alpha_max).sum()]
    return out


def _check_all(lat, tables, variant="DMD_I", label=""):
    from mapp_amd.dmd import setup
    from oracle import oracle as O
    ff = setup(lat, tables, variant=variant)
    orc = O.make(lat, tables, variant=variant)
    gx, gsrc = ff.ghosts()
    ox, osrc = orc.ghosts()
    assert np.array_equal(gsrc, osrc) and np.array_equal(gx.view(np.uint64), ox.view(np.uint64)), label
    goff, gnl = ff.neighbor_list()
    ooff, onl = orc.neighbor_list()
    assert np.array_equal(goff, ooff) and np.array_equal(gnl, onl), label
    eg, eo = ff.force_calc(1), orc.force_calc(1)
    print(label, "sites", lat.natms, "ghosts", len(osrc), "pairs", len(onl), "energy", eg[0], eo[0], flush=True)
    assert abs(eg[0] - eo[0]) <= 1e-12 * abs(eo[0]), label
    assert rel_inf(eg[1:], eo[1:]) <= 1e-12, label
    for name in ("f", "E", "dE"):
        err = rel_inf(ff.get(name), orc.get(name))
        print(label, name, err, flush=True)
        assert err <= 1e-12, (label, name)
    e1, e2 = ff.energy_calc(), orc.energy_calc()
    assert abs(e1 - e2) <= 1e-12 * abs(e2), label
    ff.create_2nd_neigh_lst()
    orc.create_2nd_neigh_lst()
    goff, gnl = ff.neighbor_list2()
    ooff, onl = orc.neighbor_list2()
    assert np.array_equal(goff, ooff) and np.array_equal(gnl, onl), label
    ff.c_d_calc()
    orc.c_d_calc()
    for name in ("c_d", "n", "E", "dE"):
        err = rel_inf(ff.get(name), orc.get(name))
        print(label, name, err, flush=True)
        assert err <= 1e-12, (label, name)
    a = np.random.default_rng(3).uniform(-0.2, 0.2, size=lat.c.shape)
    cost_o, g_o = orc.calc_g(0, 0.37, a)
    ff.set_vec("a", a)
    cost_g = ff.calc_g(0, 0.37)
    print(label, "calc_g", cost_g, cost_o, rel_inf(ff.get("g"), g_o), flush=True)
    assert abs(cost_g - cost_o) <= 1e-12 * abs(cost_o), label
    assert rel_inf(ff.get("g"), g_o) <= 1e-12, label
    assert abs(ff.calc_g(1, 0.37) - cost_o) <= 1e-12 * abs(cost_o), label
    ff.close()
    return orc


def widths_in_all_regimes(n, seed):
    """FCC n^3 cells whose per-(site, type) widths come from three bands:
    [12, 40] (pairs with them fall at or below alpha_min = 25 or just above),
    [60, 120], [2000, 4000] (pairs of two such widths reach alpha_max = 1000)"""
    from mapp_amd import workload as W
    lat = W.fcc_alloy(n, seed=seed)
    rng = np.random.default_rng(seed + 100)
    nt = lat.c.shape[1]
    band = rng.integers(0, 3, size=(lat.natms, nt))
    lo = np.array([12.0, 60.0, 2000.0])[band]
    hi = np.array([40.0, 120.0, 4000.0])[band]
    lat.x[:, 3:] = rng.uniform(lo, hi)
    return lat


@pytest.mark.parametrize("variant", ["DMD", "DMD_I", "DMD_II"])
def test_widths_in_all_regimes(tables, variant):
    lat = widths_in_all_regimes(6, seed=51)
    orc = _check_all(lat, tables, variant=variant, label=f"widths {variant}")
    counts = regime_counts(orc)
    print("skipped, quadrature, classical (pair, type pair):", counts, flush=True)
    assert (counts > 500).all()


def test_concentration_edges(tables):
    from mapp_amd import workload as W
    lat = W.fcc_alloy(6, seed=52)
    edge = np.array([0.0, 1.0, 5e-9, 1.0 - 5e-9, 1e-8, 1.0 - 1e-8, 2e-8, 1.0 - 2e-8])
    pick = np.random.default_rng(7).integers(0, 2, size=lat.natms).astype(bool)
    cA = lat.c[:, 0].copy()
    cA[pick] = edge[np.arange(pick.sum()) % len(edge)]
    lat.c[:, 0] = cA
    lat.c[:, 1] = 1.0 - cA
    _check_all(lat, tables, label="c edges")


def test_tilted_box(tables):
    """H rows (L,0,0), (2a,L,0), (a,-a,L): the tilts are translations of the
    FCC crystal, so the crystal (not its jitter) continues across every face"""
    from mapp_amd import workload as W
    n, a = 6, 3.6
    cube = W.fcc_alloy(n, a=a, seed=53)
    L = a * n
    H = np.array([[L, 0.0, 0.0], [2 * a, L, 0.0], [a, -a, L]])
    lat = _lattice_from_cart(H, cube.cart, cube.x[:, 3:], cube.c)
    orc = _check_all(lat, tables, label="tilted")
    off, nl = orc.neighbor_list()
    assert len(nl) > 30 * lat.natms


@pytest.mark.parametrize("md", [False, True])
def test_moves_in_a_tilted_box(tables, md):
    """positions moved inside the skin: ghosts follow by H[d][0..d] of each face they crossed, over edges
    and corners; then past it.  Ghosts bit for bit, forces as above"""
    from mapp_amd import workload as W
    from mapp_amd.dmd import setup, setup_eam
    from oracle import oracle as O
    n, a = 6, 3.6
    cube = W.fcc_alloy(n, a=a, seed=55)
    L = a * n
    H = np.array([[L, 0.0, 0.0], [2 * a, L, 0.0], [a, -a, L]])
    lat = _lattice_from_cart(H, cube.cart, cube.x[:, 3:], cube.c)
    if md:
        t = (np.arange(lat.natms) % 3 == 0).astype(np.float64)
        ff = setup_eam(H, lat.x[:, :3].copy(), t, tables)
        orc = O.Oracle(nt=2, variant="EAM")
        orc.set_fs(tables)
        orc.set_params(masses=tables.masses)
        orc.set_system(H, lat.x[:, :3].copy(), t.reshape(-1, 1))
        orc.init(0.5)
    else:
        ff, orc = setup(lat, tables), O.make(lat, tables)
    rng = np.random.default_rng(5)
    x = ff.get("x")
    for far in (False, True):
        x[:, :3] += rng.uniform(-0.04, 0.04, size=(lat.natms, 3))
        x[:, 3:] *= rng.uniform(0.98, 1.02, size=(lat.natms, x.shape[1] - 3))
        if far:
            x[11, 1] += 0.7
        assert ff.set_x(x) is far and orc.set_x(x) is far
        (gx, gsrc), (ox, osrc) = ff.ghosts(), orc.ghosts()
        assert np.array_equal(gsrc, osrc) and np.array_equal(gx.view(np.uint64), ox.view(np.uint64))
        for g, o in zip(ff.neighbor_list(), orc.neighbor_list()):
            assert np.array_equal(g, o)
        eg, eo = ff.force_calc(1), orc.force_calc(1)
        assert abs(eg[0] - eo[0]) <= 1e-12 * abs(eo[0]) and rel_inf(eg[1:], eo[1:]) <= 1e-12
        assert rel_inf(ff.get("f"), orc.get("f")) <= 1e-12
    ff.close()


def test_cluster_in_vacuum(tables):
    """a 3^3-cell FCC cluster (108 sites) in a 40 A box plus four isolated
    sites farther than the list cut from every other site and image"""
    from mapp_amd import workload as W
    rng = np.random.default_rng(54)
    g = np.arange(3)
    cells = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1).reshape(-1, 3)
    basis = np.array([[0, 0, 0], [0.5, 0.5, 0], [0.5, 0, 0.5], [0, 0.5, 0.5]])
    cl = ((cells[:, None, :] + basis[None, :, :]) * 3.6).reshape(-1, 3) + 14.0
    cl += rng.normal(0.0, 0.03, size=cl.shape)
    lone = np.array([[2.0, 2.0, 2.0], [2.0, 34.0, 10.0], [34.0, 2.0, 22.0], [34.0, 34.0, 34.0]])
    cart = np.concatenate([cl, lone])
    nat = len(cart)
    alpha = rng.uniform(60.0, 120.0, size=(nat, 2))
    cA = rng.uniform(0.0, 1.0, size=nat)
    lat = _lattice_from_cart(np.diag([40.0] * 3), cart, alpha, np.stack([cA, 1.0 - cA], axis=1))
    orc = _check_all(lat, tables, label="cluster")
    off, nl = orc.neighbor_list()
    assert (np.diff(off)[-4:] == 0).all()
