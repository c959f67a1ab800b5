"""The local lists between calls, through the C ABI: which node grid they
belong to, what reads them, and what leaves them as they are."""
import ctypes as C

import numpy as np
import pytest
import torch

import enkfg
import oracle as O
import synth

pytestmark = pytest.mark.gpu


def setup(nmem=8, **kw):
    P = synth.make_problem(**dict(dict(seed=3, nmem=nmem, nobs=1500, nj=24, ni=30, nk=2, locrad=80.0, stride=3), **kw))
    E = enkfg.Engine(nmem, keep_fp64=True)
    E.set_obstypes(P.obstypes)
    E.set_obs(P.obs_type, P.obs_status, P.obs_lon, P.obs_lat, P.obs_estd)
    E.set_S(P.HA, P.innov, standardised=False)
    ob = O.OracleObs(P.obstypes, P.obs_type, P.obs_lon, P.obs_lat, P.obs_estd)
    return P, E, ob


def check_lists(E, ob, lon, lat, nodes):
    for k in nodes:
        ids, lc = ob.findlocal(lon.ravel()[k], lat.ravel()[k])
        got = E.localobs(k, len(ids))
        assert np.array_equal(got[0][:len(ids)], ids) and np.array_equal(got[1][:len(ids)], lc)


@pytest.mark.parametrize("ordered", [False, True])
def test_lists_keep_their_grid_when_transforms_are_set(ordered):
    """enkfg_set_transforms brings a node grid of its own; the lists of the
    calc (or of enkfg_localise) before it stay those of their nodes."""
    print("case lists and set_transforms ordered=%d" % ordered, flush=True)
    P, E, ob = setup()
    if ordered:
        E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
        E.localise(P.node_lon, P.node_lat, stride=P.stride)
    else:
        E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
    nn = P.node_lon.size
    counts = E.local_counts()
    m = E.nmem
    for nj, ni in ((40, 50), (2, 3)):
        E.set_transforms(np.zeros((nj, ni, m, m), np.float32), np.zeros((nj, ni, m), np.float32), P.stride)
        check_lists(E, ob, P.node_lon, P.node_lat, range(min(nn, nj * ni)))
        for bad in (nn, nj * ni) if nn > nj * ni else (nn, nj * ni - 1, nj * ni):
            with pytest.raises(enkfg.EnkfgError):
                E.localobs(bad, 10000)
    E.nnode = 2 * 3
    assert np.array_equal(E.local_counts(), counts[:6])
    E.set_transforms(np.zeros((40, 50, m, m), np.float32), np.zeros((40, 50, m), np.float32), P.stride)
    E.nnode = 40 * 50
    with pytest.raises(enkfg.EnkfgError):
        E.local_counts()
    E.close()


def test_reading_a_list_leaves_the_calc_lists():
    """enkfg_get_localobs after a calc gives the list in the reference's order
    and leaves the lists that the adjoint sums over as they are: one column,
    one node, so that no sum depends on the order of atomics."""
    print("case lists read between two adjoints", flush=True)
    P, E, ob = setup(locrad=400.0)
    lon, lat = P.node_lon[4:5, 5:6].copy(), P.node_lat[4:5, 5:6].copy()
    E.calc_transforms(lon, lat)
    X = torch.randn(1, 1, E.nmem, device="cuda") + 10.0
    dJ = torch.ones(1, 1, device="cuda")
    E.ens_attach(np.ones((1, 1), np.int32), 1, 0, 0, [dict(level=0)], X.data_ptr())
    before = E.adjoint(dJ.data_ptr(), P.nobs)
    assert E.local_counts()[0] > 1000 and np.abs(before[0]).max() > 0
    check_lists(E, ob, lon, lat, [0])
    after = E.adjoint(dJ.data_ptr(), P.nobs)
    assert np.array_equal(before[0], after[0]) and np.array_equal(before[1], after[1])
    E.close()


def test_lists_read_across_runs():
    """1,961 nodes (more than the 1,024 that are ordered together at first, no
    multiple of 8), some without coordinates, read in no order."""
    print("case lists read across runs", flush=True)
    P, E, ob = setup(nj=111, ni=157)
    lon, lat = P.node_lon.copy(), P.node_lat
    assert lon.shape == (37, 53)
    lon[0, 7] = lon[30, 5] = lon[36, 52] = np.nan
    E.calc_transforms(lon, lat, stride=P.stride)
    check_lists(E, ob, lon, lat, [1960, 0, 7, 1023, 1024, 1025, 1599, 63, 64, 1959, 1952, 1951, 1023, 1595, 1960])
    E.close()


def test_a_refused_call_leaves_the_lists():
    """A node grid that is refused (no nodes, no coordinates), by the calc or
    the localisation, leaves the lists of the calc before it."""
    print("case refused node grids", flush=True)
    P, E, ob = setup()
    E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
    lon = P.node_lon.ctypes.data_as(C.POINTER(C.c_double))
    for call in (enkfg.lib().enkfg_calc_transforms, enkfg.lib().enkfg_localise):
        for nd in (enkfg.Nodes(0, 5, 1, 1, lon, lon, None), enkfg.Nodes(2, 2, 1, 1, lon, None, None)):
            assert call(E.h, C.byref(nd)) != 0
            check_lists(E, ob, P.node_lon, P.node_lat, [0, 17])
        assert call(E.h, None) != 0
    assert len(E.local_counts()) == P.node_lon.size
    E.close()


@pytest.mark.parametrize("nj,ni", [(1, 3), (37, 61), (60, 70), (97, 101)])
def test_lists_of_every_grid_size(nj, ni):
    """The walk takes one list a wavefront, several, or tiles of nodes (beyond
    16,384 lists): lists of enkfg_localise and of a run after a calc, two
    obstypes, at the grid's corners and in between."""
    print("case lists %d x %d nodes" % (nj, ni), flush=True)
    P, E, ob = setup(profiles=40)
    assert len(P.obstypes) == 2
    lon, lat = np.meshgrid(np.linspace(P.lon.min() - 0.5, P.lon.max(), ni), np.linspace(P.lat.min(), P.lat.max() + 0.5, nj))
    nn = nj * ni
    nodes = sorted({0, ni - 1, nn // 2, nn - ni, nn - 1, *range(0, nn, 97)} | set(range(max(0, nn - 9), nn)))
    E.localise(lon, lat)
    check_lists(E, ob, lon, lat, nodes)
    E.calc_transforms(lon, lat)
    check_lists(E, ob, lon, lat, nodes)
    E.close()
