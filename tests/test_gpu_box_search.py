"""The calc's localisation (box search over Morton-ordered rows) against the
oracle's tree search, through the C ABI: the counts per type, the lists in
the reference's order after the calc (enkfg_get_localobs walks the trees for
it), and T and w of the calc, which used the box search's lists.

Sizes sit at the edges of the boxes (64 rows a leaf, 64 boxes a level).  The
integer grids put many observations at exactly the radius, 3-4-5 triples and
along an axis, where the reference's search prunes some; a few observations
have no latitude.
"""
import numpy as np
import pytest

import enkfg
import oracle as O

pytestmark = pytest.mark.gpu


def run_case(types, typ, lon, lat, status, status_search, node_lon, node_lat, geographic, m=20, seed=0):
    rng = np.random.default_rng(seed)
    n = len(typ)
    estd = np.full(n, 0.5, np.float32)
    HA = rng.standard_normal((m, n)).astype(np.float32)
    innov = rng.standard_normal(n)
    ob = O.OracleObs(types, typ, lon, lat, estd, status=status_search, status_at_build=status)
    S, s = O.standardise(m, ob, HA, innov)
    ref = O.calc_transforms(1, 1, m, m, 1.0, ob, S, s, node_lon.ravel(), node_lat.ravel(), geographic=geographic)
    E = enkfg.Engine(m, keep_fp64=True)
    E.set_obstypes(types)
    E.set_obs(typ, status, lon, lat, estd)
    E.set_S(HA, innov, standardised=False)
    E.set_obs_status(status_search)
    for again in range(2):
        E.calc_transforms(node_lon, node_lat, geographic=geographic)
        T, w, T64, w64 = E.transforms(fp64=True)
        pn, _, _ = E.diag()
        assert np.array_equal(pn, ref["pnlobs"])
        assert E.stats() == ref["stats"]
        # sums over the local obs in another order: p m additions of 1 / eps
        for a, b in ((T64, ref["T64"]), (w64, ref["w64"])):
            assert np.abs(a - b).max() <= 1e-10 * max(np.abs(b).max(), 1e-300)
        lists = [E.localobs(k, n) for k in range(node_lon.size)] if again == 0 else lists
    for k, (lo, la) in enumerate(zip(node_lon.ravel(), node_lat.ravel())):
        ids, lc = ob.findlocal(lo, la, geographic)
        assert np.array_equal(lists[k][0][:len(ids)], ids) and np.array_equal(lists[k][1][:len(ids)], lc)
    E.close()
    return ref["stats"]["nlobs_sum"]


@pytest.mark.parametrize("n", [1, 63, 64, 65, 4096, 4097, 20000])
def test_box_search_sizes(n):
    """n observations of the first type (random, clustered in profiles at the
    same position), a few of a second with two radii, some not OK, some marked
    bad after set_obs; nodes inside and outside the observations' bounds, one
    without coordinates."""
    print("case box search n=%d" % n, flush=True)
    rng = np.random.default_rng(n)
    n2 = 130
    lon = np.concatenate([rng.uniform(178, 186, n), np.repeat(rng.uniform(178, 186, 13), 10)]).astype(np.float32)
    lat = np.concatenate([rng.uniform(-3, 4, n), np.repeat(rng.uniform(-3, 4, 13), 10)]).astype(np.float32)
    typ = np.concatenate([np.zeros(n, np.int16), np.full(n2, 1, np.int16)])
    o = rng.permutation(n + n2)
    lon, lat, typ = lon[o], lat[o], typ[o]
    status = (rng.random(n + n2) < 0.1).astype(np.int16)
    status2 = np.where(rng.random(n + n2) < 0.1, 5, status).astype(np.int16)
    types = [dict(locrad=[150.0]), dict(locrad=[90.0, 310.5], locweight=[1.0, 2.0])]
    nlon, nlat = np.meshgrid(np.linspace(176.0, 188.0, 11), np.linspace(-6.0, 7.0, 5))
    nlon[0, 3] = np.nan
    assert run_case(types, typ, lon, lat, status, status2, nlon, nlat, 1) > 0


@pytest.mark.parametrize("order", ["random", "sorted"])
@pytest.mark.parametrize("bad", [False, True])
def test_box_search_ties_and_nonfinite(bad, order):
    """An integer grid in plain coordinates and radius 5: observations at
    exactly the radius, some of which the reference's search prunes; with
    `bad`, also observations without a latitude."""
    print("case box search ties bad=%d order=%s" % (bad, order), flush=True)
    rng = np.random.default_rng(4)
    x, y = np.meshgrid(np.arange(40), np.arange(30))
    lon, lat = x.ravel().astype(np.float32), y.ravel().astype(np.float32)
    o = rng.permutation(lon.size) if order == "random" else np.lexsort((lat, lon))
    lon, lat = lon[o], lat[o]
    typ = (np.arange(lon.size) % 2).astype(np.int16)
    if bad:
        lat[[7, 300]] = np.nan
        lat[[17, 400]] = np.inf, -np.inf
        lon[11] = np.nan
    st = np.zeros(lon.size, np.int16)
    types = [dict(locrad=[5.0], geographic=0), dict(locrad=[4.5], geographic=0)]
    nlon, nlat = np.meshgrid(np.arange(1.0, 40.0, 6.0), np.arange(2.0, 30.0, 7.0))
    found = run_case(types, typ, lon, lat, st, st, nlon, nlat, 0)
    r = np.where(typ == 0, 5.0, 4.5)
    near = ((lon[None] - nlon.ravel()[:, None]) ** 2 + (lat[None] - nlat.ravel()[:, None]) ** 2 <= r ** 2).sum()
    assert 0 < found < near, "some observations at the radius are behind a pruned split"


def test_box_search_beyond_one_launch():
    """8.45M nodes and 8 types: more lists (67.6M) than one launch has
    wavefronts for (2^32 threads).  A few observations of each type on planar
    coordinates, at the corners and the middle; every count of the calc (EnOI,
    two members), and lists at the end of the grid."""
    print("case box search beyond one launch", flush=True)
    ni, nj, nt, r = 8192, 1032, 8, 2.5
    rng = np.random.default_rng(8)
    base = np.array([[0.3, 0.4], [8190.2, 0.7], [0.1, 1030.4], [8190.6, 1030.8], [4000.3, 515.2], [8188.9, 1029.7]])
    xy = np.concatenate([base + 0.1 * rng.random(base.shape) for _ in range(nt)]).astype(np.float32)
    typ = np.repeat(np.arange(nt, dtype=np.int16), len(base))
    n = len(typ)
    types = [dict(locrad=[r], geographic=0) for _ in range(nt)]
    estd = np.full(n, 0.5, np.float32)
    st = np.zeros(n, np.int16)
    E = enkfg.Engine(2, mode=enkfg.MODE_ENOI)
    E.set_obstypes(types)
    E.set_obs(typ, st, xy[:, 0], xy[:, 1], estd)
    E.set_S(rng.standard_normal((2, n)).astype(np.float32), rng.standard_normal(n), standardised=False)
    nlon, nlat = np.meshgrid(np.arange(float(ni)), np.arange(float(nj)))
    E.calc_transforms(nlon, nlat, geographic=0)
    pn, _, _ = E.diag()
    want = np.zeros((nt + 1, nj, ni), np.int32)
    for (x, y), t in zip(xy.astype(np.float64), typ):
        i0, j0 = max(int(x) - 4, 0), max(int(y) - 4, 0)
        w = (slice(j0, j0 + 9), slice(i0, i0 + 9))
        hit = (nlon[w] - x) ** 2 + (nlat[w] - y) ** 2 <= r * r
        for q in (t, nt):
            want[q][w] += hit
    assert want[:nt].any(axis=(1, 2)).all()
    assert np.array_equal(pn.reshape(want.shape), want)
    ob = O.OracleObs(types, typ, xy[:, 0], xy[:, 1], estd)
    for k in (0, ni - 1, ni * nj - 1, ni * nj - 2, ni * (nj - 2) + 8190):
        ids, lc = ob.findlocal(nlon.ravel()[k], nlat.ravel()[k], 0)
        got = E.localobs(k, n)
        assert len(ids) and np.array_equal(got[0][:len(ids)], ids) and np.array_equal(got[1][:len(ids)], lc)
    E.close()
