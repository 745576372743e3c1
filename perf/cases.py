"""The measured cases: what programs that use this library have it do, over its real range.

A GCM calls crm() once per physics step on whatever columns a rank holds, so most cases are one
call (crm_hip_run_device, crm_hip_run or crm_hip_run_many): from one physics chunk of 16 columns,
where every substep is a string of short dependent launches, to the 4096 instances that fill the
device; 2D and 3D CRMs of every column count, the level counts of the reference's configurations
and others, both precisions, the mean-state acceleration that production runs use, host and device
arrays.  The others are the microphysics network (training step and inference) and the GCM-side
code around the call.

Inputs: tropical soundings drawn per instance (the distribution of crm_inputs.make_case), noise in
the lowest levels, and in a part of the instances a moist raining updraft and an ice cloud, so that
every microphysics branch is taken as it is in a run.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "acme-ecp_amd"))

import crm_glue  # noqa: E402
import crm_inputs  # noqa: E402
from crm_hip import CrmHip, DeviceCase, run_many  # noqa: E402
from crm_mlp import NIN, NOUT, CrmMlp, init_params, unpack  # noqa: E402
from crm_views import CrmCase, OUT_GRID, OUT_PLEV, RAD_ORDER, STATE_ORDER  # noqa: E402

DEV = "cuda:0"
DT_GL = 1200.0  # the GCM physics step [s]

# Output members of one value per column, returned in groups of one unit.
COL_GROUPS = {"precip": ["precc", "precl", "precsc", "precsl"], "cover": ["cltot", "clhgh", "clmed", "cllow"],
              "coltend": ["prectend", "precstend"], "levels": ["jt_crm", "mx_crm"],
              "surface": ["taux", "tauy", "z0m", "timing_factor"]}

# The five size classes of an uneven batch: ncrms, nx, ny, nz.
UNEVEN = [(2048, 16, 1, 28), (1024, 32, 1, 28), (1024, 64, 1, 58), (256, 128, 1, 58), (128, 8, 8, 28)]


def _crm(name, n, nx, ny, nz, rad, prec="fp64", entry="device", accel=0, tuned=False, coriolis=False):
    c = {"kind": "crm", "n": n, "nx": nx, "ny": ny, "nz": nz, "nx_rad": rad[0], "ny_rad": rad[1], "prec": prec,
         "entry": entry, "accel": accel, "tuned": tuned, "coriolis": coriolis}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the operational 2D configuration (64 columns, 58 levels, 16 radiation columns), a batch
        # that fills the device, launch shapes tuned once as the benchmark does
        _crm("sp1v1_4096_fp64", 4096, 64, 1, 58, (16, 1), tuned=True),
        # the same batch in mixed precision, as a caller that never tunes gets it
        _crm("sp1v1_4096_mixed", 4096, 64, 1, 58, (16, 1), "mixed"),
        # one physics chunk of 16 GCM columns: the smallest call, latency and launches
        _crm("chunk_16x32x28", 16, 32, 1, 28, (8, 1)),
        # the columns of one rank through the drop-in entry on host arrays
        _crm("rank_866x32x28_host", 866, 32, 1, 28, (32, 1), entry="host"),
        # wide CRMs: two waves per instance, half of the device
        _crm("wide_256x128x58", 256, 128, 1, 58, (16, 1)),
        # the fast configuration's 3D CRM: 4 x 4 columns
        _crm("fast_1024x4x4x28", 1024, 4, 4, 28, (1, 1)),
        # 3D with Coriolis, a level count without a compiled-in loop, odd batch, mixed precision
        _crm("cube_333x8x8x40_mixed", 333, 8, 8, 40, (4, 2), "mixed", coriolis=True),
        # production's mean-state acceleration (factor 3: a quarter of the substeps)
        _crm("accel_500x64x58", 500, 64, 1, 58, (16, 1), accel=3),
        # every size class of an uneven batch advanced together, a stream per class
        {"kind": "uneven", "name": "uneven_batch", "scale": 1.0, "prec": "fp64"},
        # one training step of the microphysics network at the training batch
        {"kind": "mlp_train", "name": "mlp_train_16384", "rows": 16384},
        # the network on every grid point of a 1024 x 64 x 58 batch
        {"kind": "mlp_infer", "name": "mlp_infer_1024x64x58", "rows": 1024 * 64 * 58},
        # the GCM-side code around one call on a node's columns
        {"kind": "gcm", "name": "gcm_4096x60", "n": 4096, "nz": 58, "nrad": 16},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["crm", "uneven", "mlp_train", "mlp_infer", "gcm"], [12, 1, 2, 2, 2])[0]
    if kind == "uneven":
        return {"kind": kind, "scale": round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3),
                "prec": rng.choice(["fp64", "mixed"])}
    if kind == "mlp_train":
        return {"kind": kind, "rows": _log_int(rng, 500, 65536)}
    if kind == "mlp_infer":
        return {"kind": kind, "rows": _log_int(rng, 1000, 4000000)}
    if kind == "gcm":
        return {"kind": kind, "n": _log_int(rng, 16, 4096), "nz": rng.choice([28, 40, 58]),
                "nrad": rng.choice([1, 4, 16, 64])}
    nx, ny = rng.choice([(8, 1), (16, 1), (32, 1), (32, 1), (64, 1), (64, 1), (64, 1), (128, 1), (8, 8), (4, 4)])
    nz = rng.choice([28, 28, 58, 58, rng.randint(16, 64)])
    rx = 2 ** rng.randint(0, int(math.log2(nx)))
    ry = 2 ** rng.randint(0, int(math.log2(ny)))
    # at most a quarter of the largest batch's cells, so that a draw is cheap and sizes are spread
    most = min(4096, 4096 * 64 * 58 // 4 // (nx * ny * nz))
    n = _log_int(rng, 1, most)
    accel = rng.choice([0, 0, 0, 0, 3])
    return _crm(None, n, nx, ny, nz, (rx, ry), rng.choice(["fp64", "fp64", "mixed"]),
                "host" if n * nx * ny * nz < 2000000 and rng.random() < 0.2 else "device", accel,
                coriolis=ny > 1 and rng.random() < 0.3)


# ---- inputs ---------------------------------------------------------------------------------
def _grid(nz):
    """Column spacing [m] and substep [s] of the configurations with nz levels."""
    return (1000.0, 5.0) if nz > 48 else (2000.0, 10.0) if nz > 32 else (4000.0, 20.0)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _columns(n, nz, seed):
    """Tropical soundings of n GCM columns with nz + 2 levels (numpy, GCM level order)."""
    rng = np.random.default_rng(seed)
    sst, rh, shear = rng.uniform(290.0, 304.0, (n, 1)), rng.uniform(0.6, 0.9, (n, 1)), rng.uniform(0.0, 10.0, (n, 1))
    dzb, dzm, ztop = crm_inputs.GRIDS.get(nz, (80.0, 1600.0, 24000.0 * nz / 28.0))
    zi = crm_inputs.stretched_interfaces(nz, dzb, dzm, min(ztop, 40000.0))
    zi = np.concatenate([zi, zi[-1] + (zi[-1] - zi[-2]) * np.array([1.0, 2.0])])
    zint, zmid = zi[::-1][None, :], (0.5 * (zi[1:] + zi[:-1]))[::-1][None, :]
    t, qv, u, pm, pi = crm_inputs.sounding_profiles(zmid, zint, sst, rh, shear)
    one = np.ones((n, 1))
    return {"zmid": zmid * one, "zint": zint * one, "tl": t, "ql": qv, "pmid": pm, "pint": pi,
            "pdel": pi[:, 1:] - pi[:, :-1], "ul": u}


def _dev(a):
    """A (columns, levels) array as the device tensor (levels, columns)."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.float64).T)).to(DEV)


def _crm_case(n, nx, ny, nz, nx_rad, ny_rad, seed):
    dx, dt = _grid(nz)
    case = CrmCase(n, nz + 2, nx, ny, nz, dx, dt, nx_rad=nx_rad, ny_rad=ny_rad)
    case.lat[:] = np.linspace(-0.5, 0.5, n)
    plev, col = nz + 2, _columns(n, nz, seed)
    sh, lh = 15.0, 100.0
    inp = {k: v.copy() for k, v in col.items()}
    inp["vl"] = 0.5 * col["ul"] if ny > 1 else np.zeros_like(col["ul"])
    inp["qccl"] = inp["qiil"] = np.zeros_like(col["ul"])
    # the surface fluxes, as the caller's flux bypass delivers them
    pd = col["pdel"][:, -1]
    inp["tl"][:, -1] += crm_inputs.G * sh * DT_GL / (crm_inputs.CP * pd)
    inp["ql"][:, -1] += crm_inputs.G * (lh / crm_inputs.LV) * DT_GL / pd
    arrays = {"inp": {k: _dev(v) for k, v in inp.items()}}
    zero = np.zeros(n)
    cols = {"ps": col["pint"][:, -1], "phis": zero, "ocnfrac": zero + 1.0, "tau00": zero,
            "wndls": np.abs(col["ul"][:, -1]), "bflxls": sh / crm_inputs.CP + 0.61 * col["tl"][:, -1] * lh / crm_inputs.LV,
            "fluxu00": zero, "fluxv00": zero, "fluxt00": zero, "fluxq00": zero}
    arrays["inp"].update({k: _dev(v) for k, v in cols.items()})

    g = _gen(seed)
    shape = (nz, ny, nx, n)

    def crm_levels(a):  # (columns, levels) in GCM order -> (nz, 1, 1, n), CRM order
        return _dev(a[:, ::-1][:, :nz])[:, None, None, :]

    def rand(*s):
        return torch.rand(*s, generator=g, device=DEV, dtype=torch.float64)

    t = crm_levels(col["tl"]).expand(shape).contiguous()
    qt = crm_levels(col["ql"]).expand(shape).contiguous()
    u = crm_levels(col["ul"]).expand(shape).contiguous()
    v = crm_levels(inp["vl"]).expand(shape).contiguous()
    t[:5] += 0.2 * rand(5, ny, nx, n) - 0.1
    qn, qp, w = torch.zeros_like(t), torch.zeros_like(t), torch.zeros_like(t)
    # a third of the instances convect: a cloudy raining updraft over a sixth of the columns
    # (at least three), an ice cloud with snow aloft, and noise in the winds
    conv = torch.arange(n, device=DEV) % 3 == 0
    i = torch.arange(nx, device=DEV)[:, None]
    at = torch.arange(n, device=DEV)[None, :]
    plume = conv & ((i - 3 * at) % nx < max(3, nx // 6))                     # (nx, n)
    klo, khi = max(1, nz // 12), max(3, nz // 2)
    # the moisture of the plume: a little above saturation at the sounding's temperature
    qs = crm_levels(crm_inputs.qsatw(col["tl"], col["pmid"] / 100.0)).expand(shape)[klo:khi]
    rows = slice(0, max(1, ny // 3))
    m = plume[None, None].expand(khi - klo, ny, nx, n).clone()
    m[:, rows.stop:] = False
    qn[klo:khi] = torch.where(m, 1.5e-3 * (1.0 + 0.3 * rand(*m.shape)), 0.0)
    qt[klo:khi] = torch.where(m, 1.01 * qs + qn[klo:khi], qt[klo:khi])
    qp[klo:khi] = torch.where(m, 2.0e-3 * rand(*m.shape), 0.0)
    # the updraft grows with height, as the layers do (vertical Courant numbers as in a run)
    rise = torch.arange(khi - klo, device=DEV, dtype=torch.float64)[:, None, None, None] / (khi - klo)
    w[klo:khi] = torch.where(m, (0.5 + 3.5 * rise) * (0.75 + 0.5 * rand(*m.shape)), 0.0)
    ice = conv[None, None, None] & (t < 245.0) & (t > 225.0) & (i[None, None] >= nx // 2) & \
        (i[None, None] < nx // 2 + max(2, nx // 8))
    qn = torch.where(ice, 2.0e-4, qn)
    qt = torch.where(ice, qt + 2.0e-4, qt)
    qp = torch.where(ice, 5.0e-4, qp)
    u += conv * (2.0 * rand(*shape) - 1.0)
    if ny > 1:
        v += conv * (2.0 * rand(*shape) - 1.0)
    w[1:] += conv * (0.4 * rand(nz - 1, ny, nx, n) - 0.2)
    arrays["state"] = {"u_wind": u, "v_wind": v, "w_wind": w, "temperature": t, "qt": qt, "qp": qp, "qn": qn}

    def zeros(*s):
        return torch.zeros(s, dtype=torch.float64, device=DEV)

    # radiative cooling of 1.5 K a day in the troposphere
    arrays["rad"] = {k: zeros(nz, ny_rad, nx_rad, n) for k in RAD_ORDER}
    arrays["rad"]["qrad"].copy_((-1.5 / 86400.0) * (crm_levels(col["zmid"]) < 15000.0))
    out = {k: zeros(*shape) for k in OUT_GRID}
    out["prec_crm"] = zeros(ny, nx, n)
    groups = {k: zeros(len(v), n) for k, v in COL_GROUPS.items()}
    for k, v in COL_GROUPS.items():
        out.update({f: groups[k][j] for j, f in enumerate(v)})
    out.update({k: zeros(plev, n) for k in OUT_PLEV})
    arrays["out"] = out
    dc = DeviceCase.__new__(DeviceCase)
    dc.case, dc.torch, dc.arrays = case, torch, arrays
    return dc, groups


def _to_host(dc):
    """The same columns as a host program holds them: numpy arrays in Fortran order."""
    for group in ("inp", "state", "rad", "out"):
        dst = getattr(dc.case, group)
        for k, t in dc.arrays[group].items():
            dst[k] = np.asfortranarray(t.cpu().numpy().T)
    return dc.case


def _prepare_crm(c, seed):
    dc, groups = _crm_case(c["n"], c["nx"], c["ny"], c["nz"], c["nx_rad"], c["ny_rad"], seed)
    hip = CrmHip(0, c["prec"])
    if c["coriolis"]:
        hip.set_coriolis(True)
    if c["accel"]:
        hip.accel_init(True, float(c["accel"]), True)
    if c["tuned"]:
        scratch, _ = _crm_case(c["n"], c["nx"], c["ny"], c["nz"], c["nx_rad"], c["ny_rad"], seed)
        hip.autotune(scratch, 12 * dc.case.dt)
        del scratch
    if c["entry"] == "host":
        return {"hip": hip, "case": _to_host(dc)}
    torch.cuda.synchronize()
    return {"hip": hip, "dc": dc, "groups": groups}


def _network(seed):
    """A network with the normalisation that recorded pairs give (crm_mlp.fit_norm)."""
    m = CrmMlp(0)
    mean = np.array([262.0, 540.0, 0.72, 4.5e-3, 4.0e-5, 2.0e-5, 3.0e-5, 2.0e-5, 0.0])
    scale = np.array([28.0, 290.0, 0.33, 5.5e-3, 2.2e-4, 7.0e-5, 2.0e-4, 1.0e-4, 0.5])
    oscale = np.array([4.0e-7, 4.0e-7, 8.0e-8, 9.0e-8, 4.0e-8, 1.0e-3])
    m.set_norm(mean, scale, oscale)
    m.set_params(init_params(seed % 1000))
    return m, mean, scale, oscale


def _points(rows, seed, mean, scale):
    g = _gen(seed)
    z = torch.randn((rows, NIN), generator=g, device=DEV)
    x = torch.from_numpy(mean).float().to(DEV) + z * torch.from_numpy(scale).float().to(DEV)
    x[:, 3:8] = x[:, 3:8].clamp_min(0.0)
    return x.contiguous(), g


def _targets(x, g, mean, scale, oscale):
    z = (x - torch.from_numpy(mean).float().to(DEV)) / torch.from_numpy(scale).float().to(DEV)
    y = torch.stack([torch.tanh(z[:, j] * z[:, j + 1]) + 0.5 * z[:, j + 3] for j in range(NOUT)], 1)
    y += 0.1 * torch.randn(y.shape, generator=g, device=DEV)
    return (y * torch.from_numpy(oscale).float().to(DEV)).contiguous()


def _prepare_gcm(c, seed):
    n, nz, nrad = c["n"], c["nz"], c["nrad"]
    pver = nz + 2
    dc, _ = _crm_case(n, nrad, 1, nz, nrad, 1, seed)
    g = _gen(seed + 1)

    def rand(*s):
        return torch.rand(*s, generator=g, device=DEV, dtype=torch.float64)

    a = dc.arrays["inp"]
    st = {"zm": a["zmid"].clone(), "zi": a["zint"].clone(), "t": a["tl"].clone(), "qv": a["ql"].clone(),
          "qcl": 1e-5 * rand(pver, n), "qci": 1e-5 * rand(pver, n), "ps": a["ps"].reshape(n).clone(),
          "pmid": a["pmid"].clone(), "pint": a["pint"].clone(), "pdel": a["pdel"].clone(),
          "phis": 100.0 * rand(n), "u": a["ul"].clone(), "v": 2.0 * rand(pver, n) - 1.0}
    srf = {"ocnfrac": rand(n), "wsx": 0.1 * rand(n), "wsy": 0.1 * rand(n), "shf": 30.0 * rand(n),
           "lhf": 200.0 * rand(n)}
    r = dc.arrays["rad"]
    r["temperature"].copy_(st["t"].flip(0)[:nz, None, None, :].expand_as(r["temperature"]))
    r["qv"].copy_(st["qv"].flip(0)[:nz, None, None, :].expand_as(r["qv"]))
    cloudy = rand(*r["cld"].shape) < 0.4
    for k, amp in (("qc", 1e-4), ("qi", 1e-5), ("cld", 1.0)):
        r[k].copy_(torch.where(cloudy, amp * rand(*r[k].shape), 0.0))
    for k in ("sltend", "qltend", "qcltend", "qiltend", "precc", "precl", "precsc", "precsl"):
        t = dc.arrays["out"][k]
        t.copy_(1e-3 * rand(*t.shape))
    s = {"hip": CrmHip(0), "dc": dc, "n": n, "nz": nz, "nrad": nrad, "st": st, "srf": srf,
         "angle": 6.28 * rand(n), "cflx": 1e-4 * rand(n),
         "cloud": {k: rand(pver, n) for k in crm_glue.CLOUD},
         # the radiation's heating of this step, in and above the CRM columns
         "qrs_in": 1e-2 * rand(pver, n), "qrl_in": -1e-2 * rand(pver, n),
         "qrs_crm": 1e-5 * rand(nz, 1, nrad, n), "qrl_crm": -1e-5 * rand(nz, 1, nrad, n),
         "qrs": torch.empty(pver, n, dtype=torch.float64, device=DEV),
         "qrl": torch.empty(pver, n, dtype=torch.float64, device=DEV),
         "bypass": [torch.empty(pver, n, dtype=torch.float64, device=DEV) for _ in range(2)],
         "ptend": {k: torch.empty(pver, n, dtype=torch.float64, device=DEV) for k in ("s", "qv", "qcl", "qci")},
         "flux": torch.empty(n, dtype=torch.float64, device=DEV),
         "cols": {k: torch.empty(pver, nrad, n, dtype=torch.float64, device=DEV) for k in crm_glue.RAD_COLUMN},
         "flx": {"vap": 1e-4 * rand(n), "cnd": 1e-7 * rand(n), "ice": 1e-8 * rand(n), "sen": 30.0 * rand(n)}}
    s["cur"] = {"te": 2.6e9 * (1.0 + 0.01 * rand(n)), "tw": 40.0 + 10.0 * rand(n)}
    for k in ("tnd", "rer"):
        s[k] = {f: torch.zeros(n, dtype=torch.float64, device=DEV) for f in ("te", "tw")}
    torch.cuda.synchronize()
    return s


def prepare(case, seed):
    kind = case["kind"]
    if kind == "crm":
        s = _prepare_crm(case, seed)
    elif kind == "uneven":
        cl = [(max(1, int(n * case["scale"])), nx, ny, nz) for n, nx, ny, nz in UNEVEN]
        made = [_crm_case(n, nx, ny, nz, nx, ny, seed + j) for j, (n, nx, ny, nz) in enumerate(cl)]
        s = {"hips": [CrmHip(0, case["prec"]) for _ in cl], "dcs": [m[0] for m in made], "groups": [m[1] for m in made]}
        torch.cuda.synchronize()
    elif kind == "gcm":
        s = _prepare_gcm(case, seed)
    else:
        m, mean, scale, oscale = _network(seed)
        x, g = _points(case["rows"], seed, mean, scale)
        s = {"m": m, "x": x}
        if kind == "mlp_train":
            s["t"] = _targets(x, g, mean, scale, oscale)
        torch.cuda.synchronize()
    return dict(s, kind=kind)


# ---- one pass -------------------------------------------------------------------------------
def _run_gcm(s):
    hip, dc, n, nz, nrad = s["hip"], s["dc"], s["n"], s["nz"], s["nrad"]
    pver, pdel = nz + 2, s["st"]["pdel"]
    # what the radiation hands over in this step
    s["qrs"].copy_(s["qrs_in"])
    s["qrl"].copy_(s["qrl_in"])
    crm_glue.rad_qrad(hip, n, n, nrad, nz, s["qrs_crm"], s["qrl_crm"], dc)
    crm_glue.gcm_input(hip, n, n, pver, nz, nrad, s["st"], s["srf"], s["angle"], dc)
    crm_glue.flux_bypass(hip, n, n, pver, pdel, s["srf"]["shf"], s["cflx"], *s["bypass"])
    crm_glue.rad_columns(hip, n, n, pver, nz, nrad, s["st"], s["cloud"], dc, s["cols"])
    crm_glue.gcm_tend(hip, n, n, pver, nz, nrad, pdel, dc, s["qrs"], s["qrl"], s["ptend"], s["flux"])
    crm_glue.check_energy_chng(hip, n, n, pver, s["st"], DT_GL, s["flx"], s["cur"], s["tnd"], s["rer"])
    a = dc.arrays
    keep = ("tl", "ul", "vl", "zint", "bflxls", "wndls", "tau00")
    return {"inp": {k: a["inp"][k] for k in keep}, "qrad": a["rad"]["qrad"], "bypass": s["bypass"],
            "cols": s["cols"], "ptend": s["ptend"], "flux": s["flux"], "qrs": s["qrs"], "qrl": s["qrl"],
            "precc": a["out"]["precc"], "cur": s["cur"], "tnd": s["tnd"], "rer": s["rer"]}


def run(state):
    kind = state["kind"]
    if kind == "mlp_infer":
        return state["m"].forward(state["x"])
    if kind == "mlp_train":
        loss = state["m"].train_step(state["x"], state["t"], 1e-3)
        return {"loss": loss, "params": state["m"].params()}
    if kind == "gcm":
        return _run_gcm(state)
    if kind == "uneven":
        run_many(state["hips"], state["dcs"], DT_GL)
        return [{"state": dc.arrays["state"], "t_rad": dc.arrays["rad"]["temperature"],
                 "sltend": dc.arrays["out"]["sltend"], "qltend": dc.arrays["out"]["qltend"],
                 "precip": g["precip"], "cover": g["cover"]}
                for dc, g in zip(state["dcs"], state["groups"])]
    if "case" in state:  # host arrays
        c = state["case"]
        state["hip"].run(c, DT_GL)
        return {"state": c.state, "rad": {k: c.rad[k] for k in RAD_ORDER[1:]},
                "grid": {k: c.out[k] for k in OUT_GRID + ["prec_crm"]}, "plev": {k: c.out[k] for k in OUT_PLEV},
                "precc": c.out["precc"], "precl": c.out["precl"], "cltot": c.out["cltot"], "z0m": c.out["z0m"]}
    state["hip"].run_device(state["dc"], DT_GL)
    a = state["dc"].arrays
    return {"state": {k: a["state"][k] for k in STATE_ORDER}, "rad": {k: a["rad"][k] for k in RAD_ORDER[1:]},
            "grid": {k: a["out"][k] for k in OUT_GRID + ["prec_crm"]}, "plev": {k: a["out"][k] for k in OUT_PLEV},
            "cols": state["groups"]}


# ---- work -----------------------------------------------------------------------------------
def _crm_work(n, nx, ny, nz, prec, accel):
    """Prognostics read and written once per substep and the Adams-Bashforth history (16 words per
    cell in 2D, 21 in 3D), and about 1000 operations per cell and substep with the transforms."""
    steps = DT_GL / _grid(nz)[1] / (1 + accel)
    cells = n * nx * ny * nz * steps
    words = 21 if ny > 1 else 16
    return {"bytes": cells * words * (4 if prec == "mixed" else 8), "flops": cells * (1000 + 4 * nx * ny)}


def work(case):
    kind = case["kind"]
    net = NIN * 128 + 2 * 128 * 128 + 128 * NOUT
    if kind == "mlp_infer":
        return {"bytes": 4 * case["rows"] * (NIN + NOUT), "flops": 2 * net * case["rows"]}
    if kind == "mlp_train":
        return {"bytes": 4 * case["rows"] * (NIN + NOUT) + 7 * 4 * net, "flops": 6 * net * case["rows"]}
    if kind == "gcm":
        cells = case["n"] * (case["nz"] + 2)
        return {"bytes": 8 * (cells * 60 + cells * case["nrad"] * 20), "flops": cells * (100 + 20 * case["nrad"])}
    if kind == "uneven":
        parts = [_crm_work(max(1, int(n * case["scale"])), nx, ny, nz, case["prec"], 0) for n, nx, ny, nz in UNEVEN]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    return _crm_work(case["n"], case["nx"], case["ny"], case["nz"], case["prec"], case["accel"])


# ---- 64-bit values --------------------------------------------------------------------------
def _forward64(x, norm, mats):
    mean, scale = norm
    h = [(x.double() - torch.from_numpy(mean.astype(np.float32)).double().to(DEV)) /
         torch.from_numpy(scale.astype(np.float32)).double().to(DEV)]
    for j in range(4):
        z = h[-1] @ mats[2 * j] + mats[2 * j + 1]
        h.append(z.clamp_min(0.0) if j < 3 else z)
    return h


def _exact_mlp(case, seed):
    s = prepare(case, seed)
    _, mean, scale, oscale = _network(seed)
    osc = torch.from_numpy(oscale.astype(np.float32)).double().to(DEV)
    mats = [torch.from_numpy(a.astype(np.float64)).to(DEV) for a in unpack(init_params(seed % 1000))]
    if case["kind"] == "mlp_infer":
        return torch.cat([_forward64(x, (mean, scale), mats)[-1] * osc for x in s["x"].split(1 << 20)])
    h = _forward64(s["x"], (mean, scale), mats)
    d = h[4] - s["t"].double() / osc
    loss = (d * d).mean()
    grad, up = [None] * 8, 2.0 * d / d.numel()
    for j in (3, 2, 1, 0):
        grad[2 * j], grad[2 * j + 1] = h[j].t() @ up, up.sum(0)
        if j:
            up = (up @ mats[2 * j].t()) * (h[j] > 0)
    # the first Adam step: the bias-corrected moments are the gradient and its square
    new = [w - 1e-3 * g / (g.abs() + 1e-8) for w, g in zip(mats, grad)]
    return {"loss": float(loss), "params": torch.cat([w.reshape(-1) for w in new])}


def _exact_gcm(case, seed):
    s = prepare(case, seed)
    G, CP, LV, LI = 9.80616, 1.00464e3, 2.501e6, 3.337e5
    n, nz, nrad = case["n"], case["nz"], case["nrad"]
    pver, st, a, srf = nz + 2, s["st"], s["dc"].arrays, s["srf"]
    dp = st["pdel"]
    dpc = dp.flip(0)[:nz, None, None, :]
    ca, sa = torch.cos(s["angle"]), torch.sin(s["angle"])
    inp = {"tl": st["t"], "ul": st["u"] * ca + st["v"] * sa, "vl": st["v"] * ca - st["u"] * sa, "zint": st["zi"],
           "bflxls": (srf["shf"] / CP + float(np.float32(0.61)) * st["t"][-1] * srf["lhf"] / LV)[None],
           "wndls": torch.sqrt(st["u"][-1] ** 2 + st["v"][-1] ** 2)[None],
           "tau00": torch.sqrt(srf["wsx"] ** 2 + srf["wsy"] ** 2)[None]}
    inp = {k: v.reshape(a["inp"][k].shape) for k, v in inp.items()}
    qrad = (s["qrs_crm"] + s["qrl_crm"]) / dpc * dpc
    by = [torch.zeros_like(dp), torch.zeros_like(dp)]
    by[0][-1], by[1][-1] = G / dp[-1] * srf["shf"], G / dp[-1] * s["cflx"]
    cols = {}
    r = {k: a["rad"][k].reshape(nz, nrad, n) for k in ("temperature", "qv", "qc", "qi", "cld")}
    dpr, cloudy = dpc.reshape(nz, 1, n), r["cld"] > 0
    floor = r["cld"].clamp_min(0.01)
    qtot = torch.where(cloudy, r["qc"] + r["qi"], 1.0)
    low = {"t": r["temperature"], "qv": r["qv"].clamp_min(1e-9), "qc": r["qc"], "qi": r["qi"], "cld": r["cld"],
           "fice": torch.where(cloudy, r["qi"] / qtot, 0.0),
           "cicewp": torch.where(cloudy, r["qi"] * dpr / G / floor, 0.0),
           "cliqwp": torch.where(cloudy, r["qc"] * dpr / G / floor, 0.0)}
    top = {"t": st["t"], "qv": st["qv"], "qc": st["qcl"], "qi": st["qci"], **s["cloud"]}
    for k in crm_glue.RAD_COLUMN:
        cols[k] = torch.cat([top[k][:pver - nz, None, :].expand(pver - nz, nrad, n), low[k].flip(0)])
    qrs, qrl = s["qrs_in"] / dp, s["qrl_in"] / dp
    o = a["out"]
    pt = {"s": o["sltend"].clone(), "qv": o["qltend"], "qcl": o["qcltend"], "qci": o["qiltend"]}
    pt["s"][:pver - nz + 2] = (qrs + qrl)[:pver - nz + 2]
    ke = (0.5 * (st["u"] ** 2 + st["v"] ** 2) * dp / G).sum(0)
    se = (st["t"] * CP * dp / G).sum(0) + st["phis"] * st["ps"] / G
    wv, wl, wi = ((st[k] * dp / G).sum(0) for k in ("qv", "qcl", "qci"))
    te, tw = se + ke + (LV + LI) * wv + LI * wl, wv + wl + wi
    f = s["flx"]
    dte = f["vap"] * (LV + LI) - (f["cnd"] - f["ice"]) * 1000.0 * LI + f["sen"]
    dtw = f["vap"] - f["cnd"] * 1000.0
    rer = {"te": (s["cur"]["te"] + dte * DT_GL - te) / s["cur"]["te"],
           "tw": (s["cur"]["tw"] + dtw * DT_GL - tw) / s["cur"]["tw"]}
    return {"inp": inp, "qrad": qrad, "bypass": by, "cols": cols, "ptend": pt,
            "flux": ((qrs + qrl) * dp / G).sum(0), "qrs": qrs, "qrl": qrl, "precc": o["precc"] + o["precl"],
            "cur": {"te": te, "tw": tw}, "tnd": {"te": dte, "tw": dtw}, "rer": rer}


def exact(case, seed):
    """The network and the GCM-side code in 64 bits; a whole crm() call has no short closed form."""
    if case["kind"] in ("mlp_infer", "mlp_train"):
        return _exact_mlp(case, seed)
    return _exact_gcm(case, seed) if case["kind"] == "gcm" else None
