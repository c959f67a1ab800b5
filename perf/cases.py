"""Performance cases of the analysis engine: the calls that enkf_calc,
enkf_update and a gradient user make, over the sizes, ensembles, schemes,
precisions and observation networks that they meet.

Kinds of case
  calc         enkfg_calc_transforms, then T, w and the diagnostics fetched to
               the host (what enkf_calc writes to transforms.nc and
               enkf_diag.nc, and what the point logs are made of)
  cycle        the calc and the update of the device-resident ensemble in one
               context, no transforms file between them
  update       the update of the device-resident ensemble from transforms that
               were set before
  update_host  the update of host field buffers (the das_updatefields seam)
  he           the ensemble observations from the device-resident ensemble
  adjoint      gradients of a functional of the analysis ensemble

The inputs are synthetic: smooth random ensemble anomalies, a depth profile,
a truth drawn from the same fields, and observation networks of four types
(SST on random points, SLA along tracks, T and S profiles), SST alone, or
clustered tracks and profiles.  The networks, errors, radii and strides are
those of the engine's benchmark and tests.  `order` is the order of the
observations: "random", or "prep", the order enkf_prep writes super-obs in
(type, i, j, k).
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "enkf-c_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "enkf-c_amd"))
import enkfg  # noqa: E402

REARTH = 6371.0
MODES = {"enkf": enkfg.MODE_ENKF, "hybrid": enkfg.MODE_HYBRID, "enoi": enkfg.MODE_ENOI}
SCHEMES = {"denkf": enkfg.SCHEME_DENKF, "etkf": enkfg.SCHEME_ETKF}
PRECS = {"fp64": enkfg.PREC_FP64, "mixed": enkfg.PREC_MIXED}
DEV = "cuda"


def _case(kind, **kw):
    c = dict(kind=kind, mode="enkf", scheme="denkf", prec="fp64", m=96, md=0, nj=100, ni=100, nk=5, stride=3,
             lat0=-50.0, locrad=250.0, density=2.6, net="full", order="random", alpha=1.0, points=0, nlobsmax=0,
             window=0)
    c.update(kw)
    if c["md"] == 0:
        c["md"] = c["m"]
    return c


def listed():
    L = []

    def add(name, kind, **kw):
        L.append(dict(_case(kind, **kw), name=name))

    # the point logs of a run: a handful of columns, all in one call; latency counts
    add("point-logs", "calc", points=9, nj=200, ni=240, nk=20)
    # a small regional ETKF run: 0.1 degree basin, SST only, 24 members, through files
    add("regional-etkf-calc", "calc", scheme="etkf", m=24, nj=100, ni=200, nk=10, lat0=-40.0, locrad=200.0,
        density=1.0, net="sst")
    # the update of that run: 21 fields in host buffers, as enkf_update holds them
    add("regional-update-host", "update_host", m=24, nj=100, ni=200, nk=10, lat0=-40.0)
    # eddy-resolving tile, 96 members, all networks, FP64: the engine's main use
    add("tile-denkf-fp64", "cycle", nj=540, ni=801, nk=10, lat0=-50.0)
    # the same kind of tile in mixed precision, with the super-obs in the order
    # enkf_prep writes them
    add("tile-denkf-mixed-prep", "cycle", prec="mixed", nj=240, ni=450, nk=10, lat0=-20.0, order="prep", alpha=0.8)
    # ETKF on a tile, super-obs order
    add("tile-etkf-fp64-prep", "cycle", scheme="etkf", nj=150, ni=241, nk=5, lat0=10.0, order="prep")
    # hybrid 96 + 48 members, clustered observations (uneven columns), mixed precision
    add("hybrid-clustered-mixed", "cycle", mode="hybrid", prec="mixed", m=144, md=96, nj=240, ni=300, nk=10,
        lat0=-30.0, locrad=150.0, net="clustered")
    # EnOI with a large static ensemble: w and the diagnostics only
    add("enoi-calc", "calc", mode="enoi", m=130, nj=120, ni=181, nk=10, lat0=20.0, locrad=200.0, order="prep")
    # enkf_update on a resident ensemble of 51 layers, two 3D variables and eta
    add("update-fp32", "update", nj=300, ni=401, nk=51)
    # a smaller ensemble whose size is no multiple of anything, mixed precision
    add("update-mixed-ragged", "update", prec="mixed", m=50, nj=200, ni=301, nk=25, stride=4)
    # the ensemble observations of an analysis
    add("ensemble-obs", "he", nj=240, ni=301, nk=11, density=1.0)
    # gradients of a functional over a box (observation impact)
    add("adjoint-ens", "adjoint", nj=150, ni=181, nk=4, locrad=200.0, window=60)
    return L


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["calc", "calc", "cycle", "cycle", "cycle", "update", "update", "update_host", "he", "adjoint"])
    kw = dict(lat0=round(rng.uniform(-60.0, 40.0), 1), stride=rng.choice([2, 3, 3, 4, 5]),
              order=rng.choice(["random", "prep", "prep"]), density=round(rng.uniform(0.5, 2.6), 2),
              locrad=float(rng.randint(100, 250)), nk=_log(rng, 3, 12), alpha=rng.choice([1.0, 1.0, 0.8]),
              prec=rng.choice(["fp64", "fp64", "mixed"]), m=rng.choice([24, 30, 48, 72, 96, 96, 96, 100]))
    if kind == "calc":
        if rng.random() < 0.3:
            kw.update(points=_log(rng, 1, 40), nj=_log(rng, 60, 240), ni=_log(rng, 60, 300))
        else:
            kw.update(nj=_log(rng, 20, 120), ni=_log(rng, 30, 200), m=rng.choice([24, 24, 37, 48, 64]),
                      net=rng.choice(["sst", "full"]))
        if rng.random() < 0.15:
            kw["nlobsmax"] = _log(rng, 50, 800)
        r = rng.random()
        if r < 0.2:
            kw.update(mode="enoi", m=rng.choice([96, 120, 144]))
        elif r < 0.45:
            kw.update(scheme="etkf", prec="fp64")
    elif kind == "cycle":
        kw.update(nj=_log(rng, 60, 320), ni=_log(rng, 80, 500))
        r = rng.random()
        if r < 0.25:
            kw.update(mode="hybrid", m=144, md=96, net="clustered", locrad=150.0, nj=min(kw["nj"], 240),
                      ni=min(kw["ni"], 300))
        elif r < 0.45:
            kw.update(scheme="etkf", nj=min(kw["nj"], 150), ni=min(kw["ni"], 240), m=rng.choice([24, 48, 96]))
    elif kind == "update":
        kw.update(nj=_log(rng, 40, 300), ni=_log(rng, 60, 400), nk=_log(rng, 3, 51),
                  m=rng.choice([24, 37, 48, 50, 96, 96, 120]))
    elif kind == "update_host":
        kw.update(nj=_log(rng, 20, 120), ni=_log(rng, 40, 240), m=rng.choice([24, 36, 50]))
    elif kind == "he":
        kw.update(nj=_log(rng, 60, 240), ni=_log(rng, 80, 300), density=round(rng.uniform(0.1, 1.0), 2))
    else:
        kw.update(nj=_log(rng, 60, 150), ni=_log(rng, 60, 200), window=rng.randint(20, 60), prec="fp64",
                  m=rng.choice([24, 48, 96]), nk=rng.randint(2, 5))
    return _case(kind, **kw)


# ---------------------------------------------------------------------------- inputs
class _Inputs:
    pass


def _smooth(g, n, nj, ni, spacing):
    """n unit-variance smooth random fields [n][nj][ni] (noise every `spacing` cells, interpolated)"""
    cj, ci = max(2, nj // spacing + 2), max(2, ni // spacing + 2)
    c = torch.randn(n, 1, cj, ci, generator=g, device=DEV)
    f = torch.nn.functional.interpolate(c, size=(nj, ni), mode="bicubic", align_corners=True)[:, 0]
    f = f - f.mean(dim=(1, 2), keepdim=True)
    return f / f.std(dim=(1, 2), keepdim=True).clamp_min(1e-3)


def _lonlat(fi, fj, c):
    """curvilinear grid of 0.1 degree"""
    lon = 20.0 + 0.1 * fi + 0.5 * np.sin(math.pi * fj / c["nj"])
    lat = c["lat0"] + 0.1 * fj + 0.3 * np.sin(2.0 * math.pi * fi / c["ni"])
    return lon, lat


def _network(c, rs, inten):
    """fractional indices, layers and types of the observations"""
    nj, ni, nk = c["nj"], c["ni"], c["nk"]
    n = max(8, int(c["density"] * nj * ni))
    cells_km = 0.1 * math.pi / 180.0 * REARTH
    fi, fj, kk, ty = [], [], [], []

    def tracks(n_track, per, km, start=None):
        i0 = rs.uniform(0, ni - 1, n_track) if start is None else start % ni
        j0 = rs.uniform(0, nj - 1, n_track) if start is None else start // ni
        a = rs.uniform(0, 2 * math.pi, n_track)
        s = np.arange(per) * (km / cells_km / per)
        fi.append(np.clip(i0[:, None] + np.cos(a)[:, None] * s, 0, ni - 1).ravel())
        fj.append(np.clip(j0[:, None] + np.sin(a)[:, None] * s, 0, nj - 1).ravel())
        kk.append(np.zeros(n_track * per, np.int64))
        ty.append(np.full(n_track * per, 1, np.int16))

    def profiles(n_prof, start=None):
        pi = rs.uniform(0, ni - 1, n_prof) if start is None else np.clip(start % ni + rs.uniform(-.5, .5, n_prof), 0, ni - 1)
        pj = rs.uniform(0, nj - 1, n_prof) if start is None else np.clip(start // ni + rs.uniform(-.5, .5, n_prof), 0, nj - 1)
        for t in (2, 3):
            fi.append(np.repeat(pi, nk))
            fj.append(np.repeat(pj, nk))
            kk.append(np.tile(np.arange(nk), n_prof))
            ty.append(np.full(n_prof * nk, t, np.int16))

    def sst(k):
        fi.append(rs.uniform(0, ni - 1, k))
        fj.append(rs.uniform(0, nj - 1, k))
        kk.append(np.zeros(k, np.int64))
        ty.append(np.zeros(k, np.int16))

    if c["net"] == "sst":
        sst(n)
    elif c["net"] == "full":
        sst(int(0.6 * n))
        tracks(max(1, int(0.3 * n) // 70), 70, 500.0)
        profiles(max(1, int(0.1 * n) // (2 * nk)))
    else:                       # clustered: log-normal intensity
        p = inten.ravel().astype(np.float64)
        p /= p.sum()
        tracks(max(1, n // 140), 70, 100.0, rs.choice(nj * ni, max(1, n // 140), p=p).astype(np.float64))
        profiles(max(1, n // (4 * nk)), rs.choice(nj * ni, max(1, n // (4 * nk)), p=p).astype(np.float64))
    fi, fj, kk, ty = (np.concatenate(x) for x in (fi, fj, kk, ty))
    if c["order"] == "prep":
        o = np.lexsort((kk, np.floor(fj), np.floor(fi), ty))
    else:
        o = rs.permutation(len(fi))
    return fi[o], fj[o], kk[o], ty[o]


def _inputs(c, seed):
    """every input of the case, from the seed alone"""
    X = _Inputs()
    g = torch.Generator(device=DEV).manual_seed(1000003 * (seed + 1) % (1 << 31))
    rs = np.random.default_rng(seed + 12345)
    nj, ni, nk, m, md = c["nj"], c["ni"], c["nk"], c["m"], c["md"]
    ncell = nj * ni
    X.ncell = ncell
    G = {v: _smooth(g, m + 1, nj, ni, 30) for v in ("temp", "salt", "eta")}    # the last field: the truth
    prof = torch.exp(-torch.arange(nk, device=DEV) / 15.0)
    sd = {"temp": 0.5, "salt": 0.05, "eta": 0.05}
    # layers: 5% land, shallower near it
    if c["kind"] == "he":
        X.nlevels = np.full((nj, ni), nk, np.int32)
    else:
        bath = _smooth(g, 1, nj, ni, 100)[0]
        thr = torch.quantile(bath.flatten()[::max(1, ncell // 100000)], 0.05)
        lev = ((bath - thr) * 40.0).floor().clamp(1, nk)
        X.nlevels = torch.where(bath > thr, lev, torch.zeros_like(lev)).to(torch.int32).cpu().numpy()
    jn, inn = np.arange(0, nj, c["stride"]), np.arange(0, ni, c["stride"])
    fjn, fin = np.meshgrid(jn.astype(float), inn.astype(float), indexing="ij")
    X.nj_s, X.ni_s = len(jn), len(inn)
    if c["points"]:
        fin = rs.uniform(0.1 * ni, 0.9 * ni, (1, c["points"]))
        fjn = rs.uniform(0.1 * nj, 0.9 * nj, (1, c["points"]))
    X.node_lon, X.node_lat = _lonlat(fin, fjn, c)
    X.fields = ([dict(level=k, inflation=1.05, inf_ratio=1.0) for k in range(nk)] * 2
                + [dict(level=0, issurfacevar=1, inflation=1.05, inf_ratio=1.0)])
    X.nf = len(X.fields)

    if c["kind"] in ("calc", "cycle", "he", "adjoint"):
        inten = None
        if c["net"] == "clustered":
            inten = torch.exp(1.2 * _smooth(g, 1, nj, ni, 60)[0]).cpu().numpy()
        fi, fj, kk, ty = _network(c, rs, inten)
        lon, lat = _lonlat(fi, fj, c)
        X.fi, X.fj, X.kk, X.type = fi, fj, kk, ty
        X.lon, X.lat = lon.astype(np.float32), lat.astype(np.float32)
        X.nobs = len(fi)
        X.estd = np.array([0.4, 0.04, 0.05, 0.05], np.float32)[ty]
        X.status = np.zeros(X.nobs, np.int16)
        ot = dict(locrad=[c["locrad"]], rfactor=1.0)
        if c["nlobsmax"]:
            ot["nlobsmax"] = c["nlobsmax"]
        X.obstypes = [dict(ot) for _ in range(4)]
        cell = torch.from_numpy((np.rint(fj).astype(np.int64) * ni + np.rint(fi).astype(np.int64))).to(DEV)
        tyt = torch.from_numpy(ty.astype(np.int64)).to(DEV)
        amp = prof[torch.from_numpy(kk).to(DEV)]
        HA = torch.empty(m + 1, X.nobs, device=DEV)
        for t, v in enumerate(("temp", "eta", "temp", "salt")):
            q = tyt == t
            if bool(q.any()):
                HA[:, q] = G[v].reshape(m + 1, ncell)[:, cell[q]] * (sd[v] * (amp[q] if t >= 2 else 1.0))
        truth = HA[m].double()
        HA = HA[:m]
        HA = HA + 0.02 * 0.05 * torch.randn(HA.shape, generator=g, device=DEV)
        HA = HA - HA.mean(0, keepdim=True)
        X.HA = HA
        err = torch.randn(X.nobs, generator=g, device=DEV, dtype=torch.float64)
        X.innov = truth + err * torch.from_numpy(X.estd).to(DEV).double()
    if c["kind"] != "calc":
        mean = {"temp": 15.0, "salt": 35.0, "eta": 0.0}
        E = torch.empty(X.nf, ncell, m, device=DEV)
        for f in range(X.nf):
            v = "eta" if f == 2 * nk else ("temp" if f < nk else "salt")
            a = G[v][:m].reshape(m, ncell).t() * sd[v]
            if v != "eta":
                a = a * prof[f % nk]
            a = a + 0.1 * sd[v] * torch.randn(ncell, m, generator=g, device=DEV)
            if md < m:          # static members are anomalies
                a[:, :md] += mean[v]
                a[:, md:] -= a[:, md:].mean(1, keepdim=True)
            else:
                a = a + mean[v]
            lv = torch.from_numpy(X.nlevels).to(DEV).reshape(-1)
            a[lv <= X.fields[f]["level"]] = 0.0
            E[f] = a
        X.E = E
    if c["kind"] in ("update", "update_host"):
        # transforms of the size and smoothness the calc gives: symmetric
        # contractions T = I - c^2 V V^T / 2, varying smoothly over the nodes
        n = X.nj_s * X.ni_s
        V = _smooth(g, 4 * m, X.nj_s, X.ni_s, 20).reshape(4, m, n).permute(2, 1, 0) / math.sqrt(m)
        X.T = (torch.eye(m, device=DEV) - 0.2 * V @ V.transpose(1, 2).contiguous())[:, :md].contiguous()
        X.w = (0.3 / m) * _smooth(g, m, X.nj_s, X.ni_s, 20).reshape(m, n).t().contiguous()
    if c["kind"] == "adjoint":
        X.dJ = torch.zeros(X.nf, nj, ni, m, device=DEV)
        h = min(c["window"], nj, ni)
        j0, i0 = (nj - h) // 2, (ni - h) // 2
        X.box = (j0, j0 + h, i0, i0 + h)
        X.dJ[:, j0:j0 + h, i0:i0 + h] = torch.randn(X.nf, h, h, m, generator=g, device=DEV)
        X.dJ = X.dJ.reshape(X.nf, ncell, m)
    return X


def _engine(c):
    return enkfg.Engine(c["m"], nmem_dynamic=c["md"], mode=MODES[c["mode"]], scheme=SCHEMES[c["scheme"]],
                        alpha=c["alpha"], gamma=1.0, precision=PRECS[c["prec"]])


class _State:
    pass


def prepare(case, seed):
    c = case
    X = _inputs(c, seed)
    s = _State()
    s.c = c
    s.eng = _engine(c)
    s.nlevels, s.fields, s.nf, s.stride = X.nlevels, X.fields, X.nf, c["stride"]
    s.node_lon, s.node_lat = X.node_lon, X.node_lat
    kind = c["kind"]
    if kind in ("calc", "cycle", "he", "adjoint"):
        s.eng.set_obstypes(X.obstypes)
        s.eng.set_obs(X.type, X.status, X.lon, X.lat, X.estd)
        s.nobs = X.nobs
    if kind in ("calc", "cycle", "adjoint"):
        s.eng.set_S(X.HA.cpu().numpy(), X.innov.cpu().numpy(), standardised=False)
    if kind in ("cycle", "update", "he", "adjoint"):
        s.E = X.E
        s.eng.ens_attach(X.nlevels, c["stride"], 0, 0, X.fields, s.E.data_ptr())
    if kind == "cycle" and c["mode"] == "hybrid":
        s.E0 = X.E.clone()
    if kind in ("update", "update_host"):
        T = X.T.reshape(X.nj_s, X.ni_s, c["md"], c["m"]).cpu().numpy()
        s.eng.set_transforms(T, X.w.reshape(X.nj_s, X.ni_s, c["m"]).cpu().numpy(), c["stride"])
    if kind == "update_host":
        s.buffers = [np.ascontiguousarray(X.E[f].t().reshape(c["m"], c["nj"], c["ni"]).cpu().numpy())
                     for f in range(X.nf)]
    if kind == "he":
        nk = c["nk"]
        s.hops = [(enkfg.H_SURF, list(range(nk))), (enkfg.H_SURF, [2 * nk]), (enkfg.H_SUBSURF, list(range(nk))),
                  (enkfg.H_SUBSURF, list(range(nk, 2 * nk)))]
        s.fi, s.fj, s.fk = X.fi, X.fj, X.kk.astype(np.float32)
        s.value = np.array([15.0, 0.0, 15.0, 35.0])[X.type] + X.innov.cpu().numpy()
    if kind == "adjoint":
        s.dJ = X.dJ
        s.eng.calc_transforms(s.node_lon, s.node_lat, stride=c["stride"])
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    c, e = s.c, s.eng
    kind = c["kind"]
    if kind == "calc":
        e.calc_transforms(s.node_lon, s.node_lat, stride=s.stride)
        T, w, _, _ = e.transforms()
        n, dfs, srf = e.diag()
        return dict(T=T, w=w, nlobs=n, dfs=dfs, srf=srf) if T is not None else dict(w=w, nlobs=n, dfs=dfs, srf=srf)
    if kind == "cycle":
        flags = 0
        if c["mode"] == "hybrid":
            # the forecast of the cycle; its members are conditioned by the update
            s.E.copy_(s.E0)
            torch.cuda.current_stream().synchronize()
            flags = enkfg.UPD_HYBRID_CONDITION
        e.calc_transforms(s.node_lon, s.node_lat, stride=s.stride)
        e.ens_update(flags)
        n, dfs, srf = e.diag()
        return dict(E=s.E, nlobs=n, dfs=dfs, srf=srf)
    if kind == "update":
        e.ens_update()
        return s.E
    if kind == "update_host":
        e.update_fields(s.nlevels, s.stride, 0, 0, s.fields, s.buffers, 0, c["nj"] - 1)
        return s.buffers
    if kind == "he":
        HA, innov, std = e.calc_HE(s.nlevels, 0, 0, s.hops, s.fi, s.fj, s.fk, s.value)
        return dict(HA=HA, innov=innov, std=std)
    gy, gR, gi = e.adjoint_ens(s.dJ.data_ptr(), s.nobs, s.nf)
    return dict(dJ_dy=gy, dJ_dR=gR, dJ_dinfl=gi)


# ---------------------------------------------------------------------------- work and tolerance
def _nobs(c):
    return c["density"] * c["nj"] * c["ni"]


def _plocal(c):
    """mean observations within the radius of a column"""
    km = 0.1 * math.pi / 180.0 * REARTH
    lat = math.radians(c["lat0"] + 0.05 * c["nj"])
    r = c["locrad"]
    wi, wj = km * math.cos(lat) * c["ni"], km * c["nj"]
    area = min(1.0, 2 * r / wi) * min(1.0, 2 * r / wj) * math.pi / 4 * wi * wj      # of the disc inside the grid
    p = _nobs(c) * area / (wi * wj)
    return min(p, 4.0 * c["nlobsmax"]) if c["nlobsmax"] else p


def work(case):
    c = case
    m, md, ncell = c["m"], c["md"], c["nj"] * c["ni"]
    nn = c["points"] or ((c["nj"] - 1) // c["stride"] + 1) * ((c["ni"] - 1) // c["stride"] + 1)
    nf = 2 * c["nk"] + 1
    nobs = _nobs(c)
    tw = 4.0 * nn * ((md if c["mode"] != "enoi" else 0) * m + m)
    p = _plocal(c)
    cb = 4.0 * m * min(nobs, nn * p) + 8.0 * min(nobs, nn * p) + tw
    cf = nn * (p * (m * (m + 1.0) + 2.0 * m) + 2.0 * m ** 3)
    ub = 4.0 * nf * ncell * (m + md) + tw
    uf = 2.0 * nf * ncell * m * md
    kind = c["kind"]
    if kind == "calc":
        return dict(bytes=cb, flops=cf)
    if kind == "cycle":
        return dict(bytes=cb + ub, flops=cf + uf)
    if kind in ("update", "update_host"):
        return dict(bytes=ub, flops=uf)
    if kind == "he":
        return dict(bytes=min(nobs * 4, nf * ncell) * 4.0 * m + 4.0 * nobs * m + 32.0 * nobs, flops=nobs * m * 12.0)
    h = min(c["window"], c["nj"], c["ni"])
    ns = (h / c["stride"] + 1) ** 2
    return dict(bytes=8.0 * nf * h * h * m + 4.0 * m * nobs + 16.0 * nobs,
                flops=4.0 * nf * h * h * m * md + ns * (p * (m * (m + 1.0) + 2.0 * m * m) + 6.0 * m ** 3))


def tolerance(case):
    """About four times the difference of two orders of the sums: 32-bit
    results of 64-bit algebra (T, w, dfs, srf), the 32-bit products of the
    update beside the 32-bit state, BF16 hi/lo products in mixed precision."""
    c = case
    if c["kind"] == "he":           # anomalies are small differences of 32-bit forecasts
        return dict(rel=5e-6, max=1e-4)
    if c["kind"] == "adjoint":
        return dict(rel=1e-6, max=1e-4)
    if c["kind"] in ("update", "update_host"):
        return dict(rel=5e-7, max=1e-5)
    # T, w, dfs and srf, or the analysis beside dfs and srf
    if c["prec"] == "mixed":        # dfs of a type with few observations varies most
        return dict(rel=5e-3, max=5e-2)
    return dict(rel=1e-6, max=4e-5)


# ---------------------------------------------------------------------------- 64-bit results
def _xyz(lon, lat):
    lo, la = torch.deg2rad(lon), torch.deg2rad(lat)
    return torch.stack([REARTH * torch.cos(lo) * torch.cos(la), REARTH * torch.sin(lo) * torch.cos(la),
                        REARTH * torch.sin(la)], 1)


def _taper(x):
    """Gaspari and Cohn (1999), eq. 4.10, of distance over radius"""
    x = 2.0 * x.clamp(0.0, 1.0)
    a = 1.0 + x ** 2 * (-x ** 3 / 4 + x ** 2 / 2) + 5.0 / 8 * x ** 3 - 5.0 / 3 * x ** 2
    y = x.clamp_min(0.5)
    b = y ** 5 / 12 - y ** 4 / 2 + 5.0 / 8 * y ** 3 + 5.0 / 3 * y ** 2 - 5 * y + 4 - 2.0 / (3 * y)
    return torch.where(x < 1.0, a, b).clamp_min(0.0)


class _Exact:
    """the local analyses of a case in 64 bits"""

    def __init__(self, c, X):
        self.c, self.X = c, X
        self.ob = _xyz(torch.from_numpy(X.lon).to(DEV).double(), torch.from_numpy(X.lat).to(DEV).double())
        self.nd = _xyz(torch.from_numpy(X.node_lon.ravel()).to(DEV), torch.from_numpy(X.node_lat.ravel()).to(DEV))
        self.ty = torch.from_numpy(X.type.astype(np.int64)).to(DEV)
        d = torch.from_numpy(X.estd).to(DEV).double() * math.sqrt(c["m"] - 1)
        self.S = torch.cat([(X.HA.double() / d).t(), torch.zeros(1, c["m"], device=DEV, dtype=torch.float64)])
        self.s = torch.cat([X.innov / d, torch.zeros(1, device=DEV, dtype=torch.float64)])

    def lists(self, nodes):
        """padded ids (nobs = none) and tapers of the nodes' local observations"""
        nobs = self.X.nobs
        cols = []
        for t in range(4):
            w = torch.nonzero(self.ty == t)[:, 0]
            if len(w) == 0:
                continue
            o = self.ob[w]
            d2 = torch.zeros(len(nodes), len(w), device=DEV, dtype=torch.float64)
            for k in range(3):
                d2 += (self.nd[nodes][:, k:k + 1] - o[None, :, k]) ** 2
            if self.c["nlobsmax"]:
                n = min(self.c["nlobsmax"], len(w))
                v, q = torch.topk(d2, n, 1, largest=False)
                cols.append((torch.where(v <= self.c["locrad"] ** 2, w[q], nobs), v))
                continue
            hit = d2 <= self.c["locrad"] ** 2
            n = int(hit.sum(1).max())
            if n == 0:
                continue
            q = torch.argsort((~hit).to(torch.int8), dim=1, stable=True)[:, :n]
            v = d2.gather(1, q)
            cols.append((torch.where(hit.gather(1, q), w[q], nobs), v))
        ids = torch.cat([x for x, _ in cols], 1)
        lc = _taper(torch.cat([v for _, v in cols], 1).sqrt() / self.c["locrad"])
        return ids, lc * (ids < nobs)

    def M(self, ids, lc, S=None):
        """S^T S and S^T s of each node"""
        Sl = (self.S if S is None else S)[ids] * lc[:, :, None]
        sl = self.s[ids] * lc
        return Sl.transpose(1, 2).contiguous() @ Sl, (Sl * sl[:, :, None]).sum(1)

    def root_inverse(self, M):
        """M^(-1/2) by the Denman-Beavers iteration"""
        Y, Z = M.clone(), torch.eye(M.shape[-1], device=DEV, dtype=torch.float64).expand_as(M).contiguous()
        for _ in range(16):
            Y, Z = 0.5 * (Y + torch.linalg.inv(Z)), 0.5 * (Z + torch.linalg.inv(Y))
        return 0.5 * (Z + Z.transpose(1, 2))

    def solve(self, chunk=None):
        """T, w [node], dfs, srf [type + 1][node]"""
        c, X = self.c, self.X
        m, md, nn = c["m"], c["md"], len(self.nd)
        eye = torch.eye(m, device=DEV, dtype=torch.float64)
        chunk = chunk or max(1, min(256, int(3e7 / X.nobs)))
        T = torch.empty(nn, md, m, device=DEV, dtype=torch.float64)
        w = torch.empty(nn, m, device=DEV, dtype=torch.float64)
        dfs = torch.zeros(5, nn, device=DEV, dtype=torch.float64)
        srf = torch.zeros(5, nn, device=DEV, dtype=torch.float64)
        for k0 in range(0, nn, chunk):
            q = torch.arange(k0, min(nn, k0 + chunk), device=DEV)
            ids, lc = self.lists(q)
            tyx = torch.cat([self.ty, torch.full((1,), -1, device=DEV)])[ids]
            G, b = 0.0, 0.0
            for t in range(4):
                on = tyx == t
                if not bool(on.any()):
                    continue
                n = int(on.sum(1).max())
                k = torch.argsort((~on).to(torch.int8), dim=1, stable=True)[:, :n]
                Gt, bt = self.M(torch.where(on, ids, X.nobs).gather(1, k), (lc * on).gather(1, k))
                G, b = G + Gt, b + bt
                self.diag(Gt, dfs[t], srf[t], q, eye)
            Mi = self.diag(G, dfs[4], srf[4], q, eye)
            w[q] = (Mi @ b[:, :, None])[:, :, 0]
            if c["mode"] != "enoi":
                Tn = 0.5 * (eye + Mi) if c["scheme"] == "denkf" else self.root_inverse(eye + G)
                T[q] = (c["alpha"] * (Tn - eye) + eye)[:, :md]
        return T, w, dfs, srf

    def diag(self, G, dfs, srf, q, eye):
        Mi = torch.linalg.inv(eye + G)
        d = (Mi * G).sum((1, 2))
        dfs[q] = d
        srf[q] = torch.where(d > 1e-6, (G.diagonal(dim1=1, dim2=2).sum(1) / d).sqrt() - 1.0, torch.zeros_like(d))
        return Mi


def _node_rows(c, j, nj_s):
    a = min(j // c["stride"], nj_s - 1)
    return a, min(a + 1, nj_s - 1), (j % c["stride"]) / c["stride"]


def _interp_row(c, A, j, i0, i1, nj_s, ni_s):
    """cells i0 .. i1 - 1 of row j of the node field A [nj_s][ni_s][...]"""
    a, b, wj = _node_rows(c, j, nj_s)
    R = A[a] * (1 - wj) + A[b] * wj
    i = torch.arange(i0, i1, device=DEV)
    p = (i // c["stride"]).clamp_max(ni_s - 1)
    q = (p + 1).clamp_max(ni_s - 1)
    wi = ((i % c["stride"]).double() / c["stride"]).reshape([-1] + [1] * (R.dim() - 1))
    return R[p] * (1 - wi) + R[q] * wi


def _analyse(c, v, T, w, infl, ratio):
    """the analysis of v [field][cell][m] with T [cell][md][m] and w [cell][m]"""
    m, md = c["m"], c["md"]
    xf = v[:, :, :md].mean(2, keepdim=True)
    A = v - xf
    va = (A.transpose(0, 1).contiguous() @ T.transpose(1, 2).contiguous()).transpose(0, 1)
    xa = xf + (A * w[None]).sum(2, keepdim=True)
    kd = math.sqrt((m - 1.0) / (md - 1.0)) if c["mode"] == "hybrid" else 1.0
    va, vf = va / kd, A[:, :, :md] / kd
    f2, a2 = (vf ** 2).sum(2, keepdim=True), (va ** 2).sum(2, keepdim=True)
    raw = torch.where(a2 > 0, (f2 / a2.clamp_min(1e-300)).sqrt() * ratio + 1.0 - ratio, infl)
    f = torch.where(raw < infl, raw, infl)
    f = torch.where(f - 1.0 > 1e-6, f, torch.ones_like(f))
    return va * f + xa


def _update(c, X, T, w):
    """the analysis ensemble [field][cell][m]"""
    nj, ni, m, md = c["nj"], c["ni"], c["m"], c["md"]
    T = T.reshape(X.nj_s, X.ni_s, md, m)
    w = w.reshape(X.nj_s, X.ni_s, m)
    out = X.E.double()
    one = torch.tensor(float(np.float32(1.05)), device=DEV, dtype=torch.float64)
    lv = torch.from_numpy(X.nlevels).to(DEV)
    lev = torch.tensor([f["level"] for f in X.fields], device=DEV)
    for j in range(nj):
        sl = slice(j * ni, (j + 1) * ni)
        v = out[:, sl]
        if c["mode"] == "hybrid":
            ms = m - md
            mean = v[:, :, :md].mean(2, keepdim=True)
            v = torch.cat([(v[:, :, :md] - mean) * math.sqrt((m - 1.0) / (md - 1.0)) + mean,
                           v[:, :, md:] * math.sqrt((m - 1.0) / (ms - 1.0)) + mean], 2)
        Xa = _analyse(c, v, _interp_row(c, T, j, 0, ni, X.nj_s, X.ni_s),
                      _interp_row(c, w, j, 0, ni, X.nj_s, X.ni_s), one, 1.0)
        wet = (lv[j][None] > lev[:, None])[:, :, None]
        out[:, sl] = torch.where(wet, torch.cat([Xa, v[:, :, md:]], 2), torch.zeros_like(v))
    return out


def _exact_adjoint(c, X):
    m, md, nj, ni = c["m"], c["md"], c["nj"], c["ni"]
    ex = _Exact(c, X)
    j0, j1, i0, i1 = X.box
    st = c["stride"]
    a0, a1 = j0 // st, min((j1 - 1) // st + 1, X.nj_s - 1)
    b0, b1 = i0 // st, min((i1 - 1) // st + 1, X.ni_s - 1)
    nodes = torch.tensor([a * X.ni_s + b for a in range(a0, a1 + 1) for b in range(b0, b1 + 1)], device=DEV)
    eye = torch.eye(m, device=DEV, dtype=torch.float64)
    y = torch.zeros(X.nobs + 1, device=DEV, dtype=torch.float64)
    R = torch.cat([torch.from_numpy(X.estd).to(DEV).double() ** 2, torch.ones(1, device=DEV, dtype=torch.float64)])
    HA = torch.cat([X.HA.double().t(), torch.zeros(1, m, device=DEV, dtype=torch.float64)])
    y[:-1] = X.innov

    def columns(ids, lc, yl, Rl):
        d = (Rl * (m - 1)).sqrt()
        S = HA[ids] * (lc / d)[:, :, None]
        M = eye + S.transpose(1, 2).contiguous() @ S
        Mi = torch.linalg.inv(M)
        w = (Mi @ (S * (yl * lc / d)[:, :, None]).sum(1)[:, :, None])[:, :, 0]
        return (c["alpha"] * (0.5 * (eye + Mi) - eye) + eye)[:, :md], w

    T = torch.zeros(X.nj_s * X.ni_s, md, m, device=DEV, dtype=torch.float64)
    w = torch.zeros(X.nj_s * X.ni_s, m, device=DEV, dtype=torch.float64)
    chunk = 16
    parts = []
    for k in range(0, len(nodes), chunk):
        q = nodes[k:k + chunk]
        ids, lc = ex.lists(q)
        parts.append((q, ids, lc))
        T[q], w[q] = columns(ids, lc, y[ids], R[ids])
    gT, gw = torch.zeros_like(T), torch.zeros_like(w)
    gi = torch.zeros(X.nf, device=DEV, dtype=torch.float64)
    infl = torch.full((X.nf,), float(np.float32(1.05)), device=DEV, dtype=torch.float64)
    lv = torch.from_numpy(X.nlevels).to(DEV)
    lev = torch.tensor([f["level"] for f in X.fields], device=DEV)
    for j in range(j0, j1):
        Tj, wj, fl = T.clone().requires_grad_(), w.clone().requires_grad_(), infl.clone().requires_grad_()
        sl = slice(j * ni + i0, j * ni + i1)
        Xa = _analyse(c, X.E[:, sl].double(),
                      _interp_row(c, Tj.reshape(X.nj_s, X.ni_s, md, m), j, i0, i1, X.nj_s, X.ni_s),
                      _interp_row(c, wj.reshape(X.nj_s, X.ni_s, m), j, i0, i1, X.nj_s, X.ni_s), fl[:, None, None], 1.0)
        wet = (lv[j, i0:i1][None] > lev[:, None])[:, :, None]
        J = (torch.where(wet, Xa, torch.zeros_like(Xa)) * X.dJ[:, sl, :md].double()).sum()
        a, b, f = torch.autograd.grad(J, (Tj, wj, fl))
        gT += a
        gw += b
        gi += f
    gy, gR = torch.zeros_like(y), torch.zeros_like(R)
    for q, ids, lc in parts:
        yl, Rl = y[ids].requires_grad_(), R[ids].requires_grad_()
        Tn, wn = columns(ids, lc, yl, Rl)
        a, b = torch.autograd.grad((Tn, wn), (yl, Rl), (gT[q], gw[q]))
        gy.index_put_((ids.reshape(-1),), a.reshape(-1), accumulate=True)
        gR.index_put_((ids.reshape(-1),), b.reshape(-1), accumulate=True)
    return dict(dJ_dy=gy[:-1], dJ_dR=gR[:-1], dJ_dinfl=gi)


def _exact_he(c, X):
    """bilinear interpolation on whole layers, anomalies, innovations and spread"""
    ni, nj, nk, m = c["ni"], c["nj"], c["nk"], c["m"]
    f = np.where(X.type == 1, 2 * nk, np.where(X.type == 3, nk + X.kk, np.where(X.type == 2, X.kk, 0)))
    f = torch.from_numpy(f).to(DEV)
    fi, fj = torch.from_numpy(X.fi).to(DEV), torch.from_numpy(X.fj).to(DEV)
    i1, j1 = fi.floor().long(), fj.floor().long()
    i2, j2 = fi.ceil().long().clamp_max(ni - 1), fj.ceil().long().clamp_max(nj - 1)
    a, b = (fi - i1)[:, None], (fj - j1)[:, None]
    HA = torch.empty(X.nobs, m, device=DEV, dtype=torch.float64)
    for o in range(0, X.nobs, 100000):
        q = slice(o, o + 100000)
        at = lambda j, i: X.E[f[q], j[q] * ni + i[q]].double()  # noqa: E731
        HA[q] = ((1 - b[q]) * ((1 - a[q]) * at(j1, i1) + a[q] * at(j1, i2))
                 + b[q] * ((1 - a[q]) * at(j2, i1) + a[q] * at(j2, i2)))
    mean = HA.mean(1)
    HA = HA - mean[:, None]
    value = torch.from_numpy(np.array([15.0, 0.0, 15.0, 35.0])[X.type]).to(DEV) + X.innov
    return dict(HA=HA.t().contiguous(), innov=value - mean, std=(HA ** 2).sum(1).div(m - 1).sqrt())


def exact(case, seed):
    c = case
    X = _inputs(c, seed)
    kind = c["kind"]
    if kind == "he":
        return _exact_he(c, X)
    if kind == "adjoint":
        return _exact_adjoint(c, X)
    if kind in ("update", "update_host"):
        E = _update(c, X, X.T.double(), X.w.double())
        if kind == "update":
            return E
        return [E[f].t().reshape(c["m"], c["nj"], c["ni"]) for f in range(X.nf)]
    T, w, dfs, srf = _Exact(c, X).solve()
    if kind == "cycle":
        return dict(E=_update(c, X, T, w), nlobs=None, dfs=dfs, srf=srf)
    if c["mode"] == "enoi":
        return dict(w=w, nlobs=None, dfs=dfs, srf=srf)
    return dict(T=T, w=w, nlobs=None, dfs=dfs, srf=srf)
