"""The tile factorisation (factor_tile.hip) and the Gram tiles it reads, at
the edges of their 16-member tiles: DEnKF calc against the oracle for member
counts that fill their tiles, exceed them by one, or leave most of the last
one empty, through the C ABI.  Columns have fewer and more local obs than
members, and two obstypes, so the per-type traces run on their own matrices.
"""
import numpy as np
import pytest

import enkfg
import oracle as O
import synth

pytestmark = pytest.mark.gpu


def check(m, precision, tolT, tolw, told):
    P = synth.make_problem(seed=m, nmem=m, nobs=700, nj=16, ni=20, nk=3, locrad=60.0, stride=4, profiles=40)
    ob = O.OracleObs(P.obstypes, P.obs_type, P.obs_lon, P.obs_lat, P.obs_estd)
    S, s = O.standardise(m, ob, P.HA, P.innov)
    ref = O.calc_transforms(1, 1, m, m, 0.9, ob, S, s, P.node_lon.ravel(), P.node_lat.ravel())
    E = enkfg.Engine(m, alpha=0.9, precision=precision, keep_fp64=True)
    E.set_obstypes(P.obstypes)
    E.set_obs(P.obs_type, P.obs_status, P.obs_lon, P.obs_lat, P.obs_estd)
    E.set_S(P.HA, P.innov, standardised=False)
    E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
    T, w, T64, w64 = E.transforms(fp64=True)
    pn, pd, ps = E.diag()
    E.close()
    assert np.array_equal(pn, ref["pnlobs"])
    assert np.abs(T64 - ref["T64"]).max() <= tolT * np.abs(ref["T64"]).max()
    assert np.abs(w64 - ref["w64"]).max() <= tolw * np.abs(ref["w64"]).max()
    assert np.abs(pd - ref["pdfs"]).max() <= told * np.abs(ref["pdfs"]).max()
    assert np.array_equal(T.astype(np.float64), T64.astype(np.float32).astype(np.float64))
    # srf = sqrt(tr G / dfs) - 1 is a function of tr G and dfs alone
    ok = ref["pdfs"] > 1e-3
    assert np.abs(ps - ref["psrf"])[ok].max() <= max(1e-5, 2 * told) * (1.0 + np.abs(ref["psrf"])[ok].max())


@pytest.mark.parametrize("m", [2, 15, 16, 17, 32, 33, 48, 64, 65, 80, 81, 95, 112, 113, 128, 145])
def test_factor_tiles_fp64(m):
    """T and w within 1e-10 of the oracle, the FP64 bar (cond(M) m eps is
    below 1e-11 here); dfs and srf are FP32 results."""
    print("case factor tiles fp64 m=%d" % m, flush=True)
    check(m, enkfg.PREC_FP64, 1e-10, 1e-10, 1e-6)


@pytest.mark.parametrize("m", [16, 33, 65, 96])
def test_factor_tiles_mixed(m):
    """Each term of S^T S within 2^-16 (BF16 hi/lo); T = (I + M^-1) / 2 and w
    move by that times the condition of M, below 100 here."""
    print("case factor tiles mixed m=%d" % m, flush=True)
    check(m, enkfg.PREC_MIXED, 2e-3, 2e-3, 2e-3)


@pytest.mark.parametrize("errscale", [1.0, 1e-2, 1e-4])
@pytest.mark.parametrize("m", [2, 3, 5, 7, 8, 15, 16, 17, 33, 48, 64, 65, 80, 81, 97, 112, 113, 128, 129, 145])
def test_factor_etkf_sizes(m, errscale):
    """ETKF (factor_etkf.hip): T = M^-1/2 and w = M^-1 S^T s against the
    eigen-decomposition of M from the oracle's lists, for member counts that
    fill their tiles or leave most of the last one empty, and observation
    errors down to 1e-4 of the ensemble's spread.  The rounding of the sums in
    M, m eps |M|, moves T by that times |M^-1| <= 1 and w by that times |w|,
    and that of S^T s moves w; four times that is allowed."""
    print("case etkf m=%d errscale=%g" % (m, errscale), flush=True)
    P = synth.make_problem(seed=m, nmem=m, nobs=700, nj=16, ni=20, nk=3, locrad=60.0, stride=4, profiles=40)
    estd = (P.obs_estd * errscale).astype(np.float32)
    ob = O.OracleObs(P.obstypes, P.obs_type, P.obs_lon, P.obs_lat, estd)
    S, s = O.standardise(m, ob, P.HA, P.innov)
    E = enkfg.Engine(m, scheme=enkfg.SCHEME_ETKF, keep_fp64=True)
    E.set_obstypes(P.obstypes)
    E.set_obs(P.obs_type, P.obs_status, P.obs_lon, P.obs_lat, estd)
    E.set_S(P.HA, P.innov, standardised=False)
    E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
    T, w, T64, w64 = E.transforms(fp64=True)
    E.close()
    T64, w64 = T64.reshape(-1, m, m), w64.reshape(-1, m)
    eps = np.finfo(np.float64).eps
    for k, (lo, la) in enumerate(zip(P.node_lon.ravel(), P.node_lat.ravel())):
        ids, lc = ob.findlocal(lo, la)
        A = S[:, ids].astype(np.float64) * lc
        b = A @ (s[ids] * lc)
        lam, V = np.linalg.eigh(np.eye(m) + A @ A.T)
        tol = 4 * m * eps * lam[-1]
        assert np.abs(T64[k] - (V / np.sqrt(lam)) @ V.T).max() <= tol
        wr = (V / lam) @ (V.T @ b)
        assert np.abs(w64[k] - wr).max() <= tol * np.abs(wr).max() + 4 * m * eps * (np.abs(A) @ np.abs(s[ids] * lc)).max()


@pytest.mark.parametrize("m", [24, 96, 100, 144])
@pytest.mark.parametrize("errscale", [1e3, 1e5, 3e7])
def test_factor_etkf_weak_observations(m, errscale):
    """dfs = tr(M^-1 G) and srf = sqrt(tr(G) / dfs) - 1 of ETKF columns whose
    observations hardly constrain them: dfs down to 1e-14, far below the
    rounding of m - tr(M^-1).  Both are FP32 results; G has the rounding of
    FP64 sums.  srf is tiny there: it is compared as sqrt(tr(G) / dfs)."""
    print("case etkf weak m=%d errscale=%g" % (m, errscale), flush=True)
    P = synth.make_problem(seed=m, nmem=m, nobs=700, nj=16, ni=20, nk=3, locrad=60.0, stride=4, profiles=40)
    estd = (P.obs_estd * errscale).astype(np.float32)
    ob = O.OracleObs(P.obstypes, P.obs_type, P.obs_lon, P.obs_lat, estd)
    S, s = O.standardise(m, ob, P.HA, P.innov)
    E = enkfg.Engine(m, scheme=enkfg.SCHEME_ETKF)
    E.set_obstypes(P.obstypes)
    E.set_obs(P.obs_type, P.obs_status, P.obs_lon, P.obs_lat, estd)
    E.set_S(P.HA, P.innov, standardised=False)
    E.calc_transforms(P.node_lon, P.node_lat, stride=P.stride)
    _, pd, ps = E.diag()
    E.close()
    pd, ps = pd.reshape(len(P.obstypes) + 1, -1)[-1], ps.reshape(len(P.obstypes) + 1, -1)[-1]
    for k, (lo, la) in enumerate(zip(P.node_lon.ravel(), P.node_lat.ravel())):
        ids, lc = ob.findlocal(lo, la)
        A = S[:, ids].astype(np.float64) * lc
        # the eigenvalues of G: the squares of A's singular values
        lam = np.linalg.svd(A, compute_uv=False) ** 2
        dfs = (lam / (1.0 + lam)).sum()
        assert abs(pd[k] - dfs) <= 4 * np.finfo(np.float32).eps * dfs
        assert abs(ps[k] + 1.0 - np.sqrt(lam.sum() / dfs)) <= 8 * np.finfo(np.float32).eps * np.sqrt(lam.sum() / dfs)
