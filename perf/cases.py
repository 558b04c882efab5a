"""The calls whose speed matters to a host of the column step.

A case is a dict of plain values; listed() names the ones that are always
timed, draw() makes more of the same ranges.  prepare() makes what a host
holds before the call (the state on the GPU, or in host memory for the
host-array path, and an initialised context), run() is one pass through the
public entry points.

Columns come from the repository's generator (tempo_amd/generator.py): one or
two cloud layers of 2-4 km in an otherwise clear column, so that about a
fifth of the points hold hydrometeors.  A step updates its state in place;
between two steps a host's dynamics hands it new fields, which the device
passes model by one copy of the prognostic fields.
"""
import math

import numpy as np
import torch

from tempo_amd import generator as gen
from tempo_amd import host
from tempo_amd.autograd import tempo_step

PROGNOSTIC = ("t", "qv", "qc", "qr", "qi", "qs", "qg", "ni", "nr", "nc", "nwfa", "nifa", "ng", "qb")
INPUTS = ("p", "w", "dz")
# the 3-D diagnostics that hosts ask for by default (the radiation's radii, reflectivity)
DIAG3 = ("refl10cm", "re_cloud", "re_ice", "re_snow")
# differentiated inputs of the repository's gradient benchmark
WRT = ("t", "qv", "qc", "qr", "qi", "qs", "qg", "nc", "nr")
DT = 20.0


def _step(name, columns, levels, bits=32, **more):
    case = dict(kind="step", columns=columns, levels=levels, bits=bits, aerosol=False, hail=False, uneven=False,
                convective=False, options=False)
    case.update(more)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a single-column model, FP64 as a Fortran host steps by default: the
        # smallest call, nothing but launches and latency
        _step("column", 1, 60, bits=64),
        # one tile of a regional model (the repository's CPU-sized configuration)
        _step("tile", 1024, 60),
        # the headline configuration: an aerosol-aware batch
        _step("aerosol", 100_000, 90, aerosol=True),
        # terrain-following columns of 30 to 128 active levels, hail-aware,
        # convective: unequal work per column, many sedimentation substeps
        _step("uneven", 131_072, 128, hail=True, uneven=True, convective=True),
        # the largest configuration: aerosol- and hail-aware, a quarter convective
        _step("largest", 262_144, 90, aerosol=True, hail=True, convective=True),
        # the FP64 step, as hosts run it that need the reference's results
        _step("fp64", 25_000, 90, bits=64, aerosol=True),
        # more than 128 levels, an odd number of columns
        _step("deep", 8_191, 160, aerosol=True),
        # the run-time options together: semi-Lagrangian sedimentation,
        # melting-layer reflectivity, cloud number from the network
        _step("options", 10_007, 59, hail=True, options=True),
        # gradient of a loss on precipitation and reflectivity (assimilation, learning)
        dict(name="adjoint", kind="adjoint", columns=16_384, levels=64, bits=32, aerosol=True, hail=False, steps=1),
        # tangent-linear step (the inner loop of a variational assimilation)
        dict(name="tangent", kind="tangent", columns=8_192, levels=64, bits=32, aerosol=True, hail=True),
        # a Fortran host's arrays in ordinary host memory, transfers included
        dict(name="host", kind="host", columns=20_000, levels=60, bits=64, aerosol=True, hail=False),
        # the public check routines on the points of a tile (a host recomputes
        # its effective-radius inputs after advection), and the surface emissions
        dict(name="checks", kind="checks", points=1_000_000, bits=32),
    ]


# cost of a point-column of each kind against the plain FP32 step, rough: a
# drawn case stays within the largest listed one
_MOST = 262_144 * 90


def _between(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(("step", "adjoint", "tangent", "host", "checks"), (12, 2, 2, 2, 1))[0]
    if kind == "checks":
        return dict(kind="checks", points=_between(rng, 1_000, 4_000_000), bits=rng.choice((32, 64)))
    bits = rng.choices((32, 64), (3, 1))[0]
    if kind == "step":
        uneven = rng.random() < 0.2
        options = not uneven and rng.random() < 0.2
        levels = rng.randint(96, 128) if uneven else rng.randint(30, 160) if rng.random() < 0.3 else rng.randint(40, 100)
        cost = (6 if bits == 64 else 1) * (20 if options else 3 if levels > 128 else 1)
        aerosol = not options and rng.random() < 0.6
        return _step(None, _between(rng, 1, _MOST // (levels * cost)), levels, bits=bits, aerosol=aerosol,
                     hail=rng.random() < 0.5, uneven=uneven, convective=rng.random() < 0.4, options=options)
    levels = rng.randint(40, 90)
    if kind == "adjoint":
        steps = rng.choice((1, 1, 2))
        return dict(kind=kind, columns=_between(rng, 64, 16_384 // steps // (6 if bits == 64 else 1)), levels=levels,
                    bits=bits, aerosol=rng.random() < 0.7, hail=rng.random() < 0.5, steps=steps)
    return dict(kind=kind, columns=_between(rng, 64, 8_192 if kind == "tangent" else 40_000), levels=levels, bits=bits,
                aerosol=rng.random() < 0.7, hail=rng.random() < 0.5)


def _workload(case):
    """the generator's description of the case's columns: 16 km of atmosphere,
    or layers stretched from 25 m for the uneven ones"""
    nz = case["levels"]
    w = dict(ncol=case["columns"], nz=nz, dz=16000.0 / nz, dt=DT, aerosol=case["aerosol"], hail=case["hail"],
             seed=1, ragged=bool(case.get("uneven")), itimestep=2)
    if case.get("convective"):
        w["convective"] = 0.25
    if case.get("uneven"):
        w.update(dz=200.0, dz_sfc=25.0, dz_growth=1.06)
    return w


def _columns(case, seed, dtype):
    gen.WORKLOADS["case"] = _workload(case)
    try:
        return gen.generate_torch("case", col0=(seed // 30_000) % 1000 * 4096, seed=1 + seed % 30_000, dtype=dtype)
    finally:
        del gen.WORKLOADS["case"]


_contexts = {}


def _context(case):
    """one context per set of flags, initialised once as a host does"""
    flags = dict(aerosolaware_flag=int(bool(case.get("aerosol"))), hailaware_flag=int(bool(case.get("hail"))))
    if case.get("options"):
        flags.update(semi_sedi_flag=1, refl10cm_from_melting_flag=1, ml_for_nc_flag=1)
    key = tuple(sorted(flags.items()))
    if key not in _contexts:
        _contexts[key] = host.TempoHip(**flags)
    return _contexts[key]


def _stacked(fields, names):
    """the named (nz, ncol) fields as contiguous views of one buffer"""
    buf = torch.stack([fields[n] for n in names])
    return buf, {n: buf[i] for i, n in enumerate(names)}


def _diags(nz, ncol, dtype):
    d = {n: torch.zeros(ncol, dtype=dtype, device="cuda") for n in host.DIAG2_NAMES}
    d.update({n: torch.zeros((nz, ncol), dtype=dtype, device="cuda") for n in DIAG3})
    return d


def prepare(case, seed):
    dtype = torch.float32 if case["bits"] == 32 else torch.float64
    if case["kind"] == "checks":
        return _prepare_checks(case, seed, dtype)
    s = dict(kind=case["kind"], ctx=_context(case))
    fields, meta = _columns(case, seed, dtype)
    nz, ncol = fields["p"].shape
    names = [n for n in PROGNOSTIC if n in fields]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def noise(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=dtype)
    if case["kind"] == "host":
        s["state"] = {k: v.double().cpu().numpy() for k, v in fields.items()}
        s["names"] = names
        s["diags"] = {n: np.zeros(ncol) for n in host.DIAG2_NAMES}
        s["diags"].update({n: np.zeros((nz, ncol)) for n in DIAG3})
        s["precision"] = host.FP32 if case["bits"] == 32 else host.FP64
        return s
    if case["kind"] == "adjoint":
        s["state"] = fields
        s["steps"] = case["steps"]
        s["wrt"] = [n for n in WRT if n in fields]
        for n in s["wrt"]:
            fields[n].requires_grad_(True)
        s["rows"] = [nz // 16, 3 * nz // 10, 6 * nz // 10]
        s["weight2"], s["weight3"] = 1.0 + 0.1 * noise(ncol), 0.01 * (1.0 + 0.1 * noise(len(s["rows"]), ncol))
        return s
    s["given"], _ = _stacked(fields, names)
    s["work"] = torch.empty_like(s["given"])
    s["fields"] = {n: s["work"][i] for i, n in enumerate(names)}
    s["state"] = dict(s["fields"], **{n: fields[n] for n in INPUTS})
    s["nlev"] = meta.get("nlev")
    if case["kind"] == "tangent":
        s["given_tangent"] = 0.01 * s["given"].abs() * noise(*s["given"].shape)
        s["work_tangent"] = torch.empty_like(s["given"])
        s["tangent"] = {n: s["work_tangent"][i] for i, n in enumerate(names)}
        return s
    s["diags"] = _diags(nz, ncol, dtype)
    return s


def run(s):
    if s["kind"] == "checks":
        return _run_checks(s)
    ctx = s["ctx"]
    if s["kind"] == "step":
        s["work"].copy_(s["given"])
        ctx.run(s["state"], DT, 2, nlev=s["nlev"], diags=s["diags"])
        return dict(state=s["fields"], diags=s["diags"])
    if s["kind"] == "host":
        # in place, step after step, as the host's time loop does
        ctx.run_host(s["state"], DT, 2, precision=s["precision"], diags=s["diags"])
        return dict(state={n: s["state"][n] for n in s["names"]}, diags=s["diags"])
    if s["kind"] == "tangent":
        s["work"].copy_(s["given"])
        s["work_tangent"].copy_(s["given_tangent"])
        d, dt_, _ = ctx.tlm(s["state"], s["tangent"], DT, 2)
        two = ("rain_precip", "snow_liquid_equiv_precip", "refl10cm")
        return dict(state=s["fields"], tangent=s["tangent"], diags={n: d[n] for n in two},
                    diag_tangent={n: dt_[n] for n in two})
    state, loss = dict(s["state"]), 0.0
    for k in range(s["steps"]):
        out = tempo_step(ctx, DT, 2 + k, state)
        precip = (out["rain_precip"] + out["ice_liquid_equiv_precip"] + out["snow_liquid_equiv_precip"] +
                  out["graupel_liquid_equiv_precip"])
        loss = loss + (s["weight2"] * precip).sum() + (s["weight3"] * out["refl10cm"][s["rows"]]).sum()
        state.update({n: v for n, v in out.items() if n in state})
    grads = torch.autograd.grad(loss, [s["state"][n] for n in s["wrt"]])
    return dict(grads=dict(zip(s["wrt"], grads)), precip=precip.detach(), refl10cm=out["refl10cm"].detach(),
                t=out["t"].detach(), qv=out["qv"].detach())


def work(case):
    size = case["bits"] // 8
    if case["kind"] == "checks":  # rows read and written once, the presence flags are 4 bytes
        ins, outs = 5 + 5 + 3 + 2, 8 + 7 + 3
        return dict(bytes=case["points"] * (size * (ins + outs) + 4 * 3), flops=0)
    ncol, nz = case["columns"], case["levels"]
    prog = 9 + (3 if case["aerosol"] else 0) + (2 if case["hail"] else 0)
    points = ncol * nz * (0.62 if case.get("uneven") else 1.0)
    ins, outs = prog + len(INPUTS), prog + len(DIAG3)
    if case["kind"] == "host":
        size = 8  # the host's arrays are FP64 in either precision of the step
    if case["kind"] == "adjoint":  # per step: the step, and its inputs and cotangents in, gradients out
        back = ins + 1 + len(WRT)
        return dict(bytes=case["steps"] * size * points * (ins + outs + back), flops=0)
    if case["kind"] == "tangent":
        return dict(bytes=size * points * 2 * (prog + prog + 1) + size * points * len(INPUTS), flops=0)
    return dict(bytes=size * (points * (ins + outs) + len(host.DIAG2_NAMES) * ncol), flops=0)


# ---- the check routines and the surface emissions ----

CHECKS = {"cloud": ("qc1d", "nc1d", "qcten", "ncten"), "ice": ("qi1d", "ni1d", "qiten", "niten"),
          "snow": ("qs1d", "qsten")}
OUTS = {"cloud": ("rc", "nc", "ilamc", "mvd_c"), "ice": ("ri", "ni", "ilami"), "snow": ("rs",)}
FLAGS = {"cloud": "l_qc", "ice": "l_qi", "snow": "l_qs"}


def _check_inputs(case, seed, dtype, device):
    """points after advection: 60 % cloud-free, lognormal masses and numbers, small tendencies"""
    n = case["points"]
    r = torch.Generator(device=device).manual_seed(seed)

    def uniform(lo, hi):
        return (lo + (hi - lo) * torch.rand(n, generator=r, device=device, dtype=torch.float64)).to(dtype)

    def lognormal(median, sigma):
        return (median * torch.exp(sigma * torch.randn(n, generator=r, device=device, dtype=torch.float64))).to(dtype)
    x = dict(rho=uniform(0.3, 1.2))
    for which, names in CHECKS.items():
        on = torch.rand(n, generator=r, device=device) < 0.4
        q = torch.where(on, lognormal(1e-4, 1.0), torch.zeros((), dtype=dtype, device=device))
        x[names[0]] = q
        if which != "snow":
            number = lognormal(1e8 if which == "cloud" else 1e5, 1.0)
            x[names[1]] = torch.where(on, number, torch.zeros((), dtype=dtype, device=device))
            x[names[3]] = x[names[1]] * uniform(-1e-3, 1e-3)
        x["qsten" if which == "snow" else names[2]] = q * uniform(-1e-3, 1e-3)
    x["nwfa"], x["nwfa2d"] = lognormal(3e8, 1.0), lognormal(1e4, 1.0)
    return x


def _prepare_checks(case, seed, dtype):
    x = _check_inputs(case, seed, dtype, "cuda")
    n = case["points"]
    s = dict(kind="checks", ctx=_context(dict(aerosol=True, hail=False)), rho=x["rho"], nwfa2d=x["nwfa2d"], args={})
    inout = [k for names in CHECKS.values() for k in names] + ["nwfa"]
    s["given"], _ = _stacked(x, inout)
    s["work"] = torch.empty_like(s["given"])
    view = {k: s["work"][i] for i, k in enumerate(inout)}
    for which, names in CHECKS.items():
        a = dict(rho=s["rho"], **{k: view[k] for k in names})
        a.update({k: torch.zeros(n, dtype=dtype, device="cuda") for k in OUTS[which]})
        a[FLAGS[which]] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["args"][which] = a
    s["nwfa"] = view["nwfa"].view(1, n)
    return s


def _run_checks(s):
    s["work"].copy_(s["given"])
    for which, a in s["args"].items():
        s["ctx"].check_and_update(which, a, DT)
    s["ctx"].surface_emissions(s["nwfa"], s["nwfa2d"], DT)
    return dict({w: {k: v for k, v in a.items() if k != "rho"} for w, a in s["args"].items()}, nwfa=s["nwfa"])


def exact(case, seed):
    """The check routines and the emissions in 64 bits.  The step itself is
    several thousand lines of threshold physics with 975 MB of lookup tables:
    nothing outside the repository states it in 64 bits, so its outputs and
    derivatives have no such value here."""
    if case["kind"] != "checks":
        return None
    dtype = torch.float32 if case["bits"] == 32 else torch.float64
    x = {k: v.double() for k, v in _check_inputs(case, seed, dtype, "cuda").items()}
    rho, pi = x["rho"], 3.1415926536
    r1, r2, d0c, d0r, d0s = 1e-12, 1e-6, 1e-6, 50e-6, 300e-6

    def pick(on, a, b):
        return torch.where(on, a, torch.as_tensor(b, dtype=torch.float64, device=a.device))
    # cloud: gamma distribution with shape nu of the number
    am_r = pi * 1000.0 / 6.0
    q, n, qt, nt = (x[k] for k in CHECKS["cloud"])
    q2 = q + qt * DT
    on = q2 > r1
    rc = pick(on, q2 * rho, r1)

    def shape(nc):
        return torch.where(1e9 / nc >= 12.5, 15.0, torch.clamp(torch.floor(1e9 / nc + 0.5) + 2.0, max=15.0))

    def gammas(nu):  # gamma(nu + 4) / gamma(nu + 1)
        return (nu + 3.0) * (nu + 2.0) * (nu + 1.0)
    raw = torch.clamp((n + nt * DT) * rho, min=2.0)
    hit = (raw <= 2.0) | (raw > 1999e6)
    nc = torch.clamp(raw, max=1999e6)
    nu = shape(nc)
    lam = (nc * am_r * gammas(nu) / rc) ** (1.0 / 3.0)
    size = (nu + 4.0) / lam
    hit = hit | (size < d0c) | (size > 2.0 * d0r)
    lam = torch.where(size < d0c, (nu + 4.0) / d0c, torch.where(size > 2.0 * d0r, (nu + 4.0) / (2.0 * d0r), lam))
    nc = rc / (am_r * gammas(nu)) * lam ** 3
    nt2 = torch.where(hit, (nc / rho - n) / DT, nt)
    n2 = torch.maximum(2.0 / rho, torch.minimum(q2 / (am_r * gammas(nu)) * lam ** 3, 1999e6 / rho))
    nu = shape(nc)
    ilam = (rc / (nc * am_r * gammas(nu))) ** (1.0 / 3.0)
    cloud = dict(qc1d=pick(on, q2, 0.0), nc1d=pick(on, n2, 0.0), qcten=torch.where(on, qt, -q / DT),
                 ncten=torch.where(on, nt2, -n / DT), rc=rc, nc=pick(on, nc, 2.0), ilamc=pick(on, ilam, 0.0),
                 mvd_c=pick(on, torch.clamp((nu + 3.672) * ilam, d0c, d0r), d0c), l_qc=None)
    # ice: exponential distribution
    am_i = pi * 890.0 / 6.0
    q, n, qt, nt = (x[k] for k in CHECKS["ice"])
    q2 = q + qt * DT
    on = q2 > r1
    ri = pick(on, q2 * rho, r1)
    ni = torch.clamp((n + nt * DT) * rho, min=r2)
    small = ni <= r2
    lam5, lams = torch.full_like(ri, 4.0 / 5e-6), torch.full_like(ri, 4.0 / d0s)
    cap = torch.full_like(ri, 4999e3)
    ni = torch.where(small, torch.minimum(cap, ri / (6.0 * am_i) * lam5 ** 3), ni)
    lam = (am_i * 6.0 * ni / ri) ** (1.0 / 3.0)
    size = 4.0 / lam
    lo, hi = size < 5e-6, size > d0s
    lam = torch.where(lo, lam5, torch.where(hi, lams, lam))
    ni = torch.where(lo, torch.minimum(cap, ri / (6.0 * am_i) * lam5 ** 3), torch.where(hi, ri / (6.0 * am_i) * lams ** 3, ni))
    nt2 = torch.where(small | lo | hi, (ni / rho - n) / DT, nt)
    n2 = torch.maximum(r2 / rho, torch.minimum(q2 / (6.0 * am_i) * lam ** 3, 4999e3 / rho))
    ice = dict(qi1d=pick(on, q2, 0.0), ni1d=pick(on, n2, 0.0), qiten=torch.where(on, qt, -q / DT),
               niten=torch.where(on, nt2, -n / DT), ri=ri, ni=pick(on, ni, r2), ilami=pick(on, 1.0 / lam, 0.0), l_qi=None)
    q, qt = (x[k] for k in CHECKS["snow"])
    q2 = q + qt * DT
    on = q2 > r1
    snow = dict(qs1d=pick(on, q2, 0.0), qsten=torch.where(on, qt, -q / DT), rs=pick(on, q2 * rho, r1), l_qs=None)
    return dict(cloud=cloud, ice=ice, snow=snow, nwfa=(x["nwfa"] + x["nwfa2d"] * DT).view(1, -1))
