"""The transport work whose speed is followed, and its inputs.

Every case is a call, or a short sequence of calls, of the public Python
interface (``AdvectionDiffusion``, ``Transport``, ``thomasz``, ``thomas3d`` and
the producers) on seeded synthetic basins with the structure MOHID's own
modules give their fields: land and KFloor masks, layer thicknesses, areas and
volumes, divergence-free fluxes, and the vertical flux from continuity.

Device fields are tensors of shape (nK, nJ, nI) over Size = WorkSize +/- 1,
which is the Fortran layout of an (nI, nJ, nK) array.
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

NULL_REAL = -9.9e15          # the reference's value on land
UPWIND1, TVD = 1, 4          # advection methods
MUSCL, SUPERBEE = 3, 4       # limiters
SCHEMES = {"upwind": (UPWIND1, SUPERBEE), "superbee": (TVD, SUPERBEE), "muscl": (TVD, MUSCL)}
F64 = torch.float64


def _case(name, kind, ni, nj, nk, **kw):
    c = dict(name=name, kind=kind, ni=ni, nj=nj, nk=nk, vertical="cartesian", land=0.0,
             ragged=False, tracers=1, scheme="superbee", dt=60.0, steps=1, precision="fp64",
             implicit="none", coastal=False)
    c.update(kw)
    return c


def listed():
    return [
        # one property of a small model, a call per step: launches and waits count
        _case("call_small_upwind", "call", 100, 100, 20, scheme="upwind"),
        # one property of a sigma-layer model, TVD, a call per step
        _case("call_sigma_tvd", "call", 512, 512, 50, vertical="sigma", dt=30.0),
        # a step of eight properties, one call each, over a ragged bathymetry with
        # odd sizes; the later calls of the step share the first one's coefficients
        _case("call_properties_ragged", "call", 517, 389, 37, land=0.30, ragged=True, tracers=8),
        # the same loop from a Fortran program whose arrays live in host memory
        _case("call_host_properties", "host", 203, 171, 25, land=0.30, ragged=True, tracers=3),
        # a coastal model: open boundary, river discharges around each call, and
        # the cell fluxes that box budgets read
        _case("call_coastal_options", "call", 301, 253, 31, land=0.20, ragged=True, tracers=2,
              scheme="muscl", coastal=True),
        # a model coupled every step: tracers, geometry and hydrodynamics go in, one
        # step, tracers come out for the sources and sinks of the other modules
        _case("coupled_step", "coupled", 301, 263, 30, vertical="sigma", land=0.15, tracers=5,
              dt=30.0),
        # a small batched run, where the launches of the step loop count
        _case("run_small", "run", 100, 100, 20, land=0.20, ragged=True, tracers=3, steps=20),
        # the headline workload: 8 tracers, 30 % land, KFloor 5..40
        _case("run_headline", "run", 1024, 1024, 40, land=0.30, ragged=True, tracers=8, steps=5),
        # a deep sigma model in the fast mode, 25 % land, full columns
        _case("run_fast_sigma", "run", 1024, 1024, 60, vertical="sigma", land=0.25, tracers=4,
              dt=20.0, steps=5, precision="fast"),
        # implicit horizontal advection, the direction alternating every step
        _case("run_implicit", "run", 512, 512, 40, land=0.30, ragged=True, tracers=8, steps=2,
              implicit="x"),
        # the tridiagonal solvers alone, for modules that assemble their own rows:
        # columns, lines along j and lines along i
        _case("solvers", "solvers", 512, 512, 50, land=0.25),
        # continuity, volumes and areas of a moving sigma grid, every step
        _case("producers", "producers", 512, 512, 50, vertical="sigma", land=0.25, dt=30.0),
    ]


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["call", "call", "call", "host", "coupled", "run", "run", "run", "run",
                       "solvers", "producers"])
    most = {"host": 1_000_000, "coupled": 8_000_000, "run": 40_000_000}.get(kind, 14_000_000)

    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    nk = size(5, 60)
    ni, nj = size(30, 1024), size(30, 1024)
    while ni * nj * nk > most:
        ni, nj = max(30, int(ni * 0.8)), max(30, int(nj * 0.8))
    vertical = rng.choice(["cartesian", "sigma"])
    c = _case("", kind, ni, nj, nk, vertical=vertical, land=rng.choice([0.0, 0.15, 0.25, 0.30]),
              ragged=vertical == "cartesian" and rng.random() < 0.7,
              dt=rng.choice([20.0, 30.0, 60.0]))
    del c["name"]
    if kind in ("call", "host"):
        c["scheme"] = rng.choice(["upwind", "superbee", "superbee", "muscl"])
        c["tracers"] = rng.choice([1, 1, 2, 3, 5])
        c["coastal"] = kind == "call" and rng.random() < 0.25
    elif kind in ("coupled", "run"):
        c["tracers"] = rng.choice([1, 2, 3, 4, 5, 6, 8])
        c["scheme"] = rng.choice(["superbee", "superbee", "superbee", "upwind"])
    if kind == "run":
        c["steps"] = rng.choice([1, 2, 5])
        c["precision"] = rng.choice(["fp64", "fp64", "fast"])
        c["implicit"] = rng.choice(["none", "none", "x", "y"])
    return c


# ---------------------------------------------------------------------------
# Inputs
def _smooth(g, ny, nx, modes=8, vanish=False):
    """A smooth seeded field on [0, 1]^2; with vanish it is zero on the edge."""
    dev = g.device
    y = torch.arange(ny, dtype=F64, device=dev) / max(ny - 1, 1)
    x = torch.arange(nx, dtype=F64, device=dev) / max(nx - 1, 1)
    p, q = torch.randint(1, 5, (2, modes, 1), generator=g, device=dev).to(F64)
    a = torch.randn((modes, 1, 1), generator=g, device=dev, dtype=F64)
    s = torch.rand((2, modes, 1), generator=g, device=dev, dtype=F64) * (2 * math.pi)
    if vanish:
        fy, fx = torch.sin(math.pi * p * y), torch.sin(math.pi * q * x)
    else:
        fy, fx = torch.cos(math.pi * p * y + s[0]), torch.cos(math.pi * q * x + s[1])
    return (a * fy[:, :, None] * fx[:, None, :]).sum(0)


def _basin(c, seed):
    """Geometry, hydrodynamics and tracers of a case, as a running model holds them."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    ni, nj, nk = c["ni"], c["nj"], c["nk"]
    nI, nJ, nK = ni + 2, nj + 2, nk + 2
    dev = g.device

    def rand(*shape):
        return torch.rand(shape, generator=g, device=dev, dtype=F64)

    def zeros(*shape):
        return torch.zeros(shape, device=dev, dtype=F64)

    # ---- land and KFloor
    wet = torch.ones((nj, ni), dtype=torch.bool, device=dev)
    if c["land"] > 0:
        noise, amp = zeros(nj, ni), 1.0
        for o in range(5):
            m = 4 * 2 ** o
            noise += amp * torch.nn.functional.interpolate(
                (2 * rand(1, 1, m + 1, m + 1) - 1), size=(nj, ni), mode="bilinear",
                align_corners=True)[0, 0]
            amp *= 0.5
        flat = noise.flatten()
        wet = noise > flat.sort().values[int(c["land"] * (flat.numel() - 1))]
    for _ in range(2):           # no isolated water column
        w = torch.nn.functional.pad(wet, (1, 1, 1, 1))
        wet = wet & (w[:-2, 1:-1] | w[2:, 1:-1] | w[1:-1, :-2] | w[1:-1, 2:])
    KF = torch.full((nJ, nI), nk + 1, dtype=torch.int32, device=dev)
    kf = torch.ones((nj, ni), dtype=torch.int32, device=dev)
    if c["ragged"]:
        kf = torch.randint(max(1, nk // 8), nk + 1, (nj, ni), generator=g, device=dev,
                           dtype=torch.int32)
    KF[1:-1, 1:-1] = torch.where(wet, kf, torch.full_like(kf, nk + 1))
    W2 = torch.zeros((nJ, nI), dtype=torch.bool, device=dev)
    W2[1:-1, 1:-1] = wet
    inner = torch.zeros_like(W2)
    inner[1:-1, 1:-1] = True
    k = torch.arange(nK, device=dev, dtype=torch.int32)[:, None, None]
    ink = (k >= 1) & (k <= nk)
    water = W2 & (k >= KF) & ink

    # ---- layers and horizontal metrics
    if c["vertical"] == "sigma":
        b = _smooth(g, nJ, nI)
        b = (b - b.min()) / (b.max() - b.min()).clamp_min(1e-30)
        layer = (5.0 + 195.0 * b) / nk
    else:
        layer = torch.full((nJ, nI), 2.0, dtype=F64, device=dev)
    DWZ = torch.where(water, layer, 0.0)
    surf = 1.0 + 0.05 * _smooth(g, nJ, nI, 4) / 4.0       # the moving surface layer
    DWZ[nk] = DWZ[nk] * surf.clamp(0.8, 1.2)
    wx = 500.0 * (1.0 + 0.2 * torch.sin(torch.arange(nJ, device=dev, dtype=F64) / 40.0))
    hy = 500.0 * (1.0 + 0.2 * torch.cos(torch.arange(nI, device=dev, dtype=F64) / 50.0))
    DUX = wx[:, None].expand(nJ, nI).contiguous()
    DVY = hy[None, :].expand(nJ, nI).contiguous()
    DZX, DZY = DUX.clone(), DVY.clone()
    DZX[:-1] = (DUX[:-1] + DUX[1:]) / 2
    DZY[:, :-1] = (DVY[:, :-1] + DVY[:, 1:]) / 2
    up = torch.zeros_like(DWZ)
    up[:-1] = DWZ[1:]
    DZZ = torch.where(water, (up + DWZ) / 2, 0.0)
    DUZ, DVZ = torch.zeros_like(DWZ), torch.zeros_like(DWZ)
    DUZ[:, 1:] = torch.where(water[:, 1:] & water[:, :-1],
                             (DWZ[:, 1:] * DUX[:-1] + DWZ[:, :-1] * DUX[1:]) /
                             (DUX[:-1] + DUX[1:]), 0.0)
    DVZ[:, :, 1:] = torch.where(water[:, :, 1:] & water[:, :, :-1],
                                (DWZ[:, :, 1:] * DVY[:, :-1] + DWZ[:, :, :-1] * DVY[:, 1:]) /
                                (DVY[:, :-1] + DVY[:, 1:]), 0.0)
    nominal = DUX * DVY * float(layer.mean())
    VolumeZ = torch.where(water, DUX * DVY * DWZ, nominal)
    VolumeZOld = VolumeZ.clone()
    VolumeZOld[nk] = VolumeZ[nk] * (1.0 + 0.01 * _smooth(g, nJ, nI, 4) / 4.0).clamp(0.95, 1.05)

    # ---- compute faces and open points
    cfu, cfv = torch.zeros_like(water), torch.zeros_like(water)
    cfu[:, 2:-1, 1:-1] = (water[:, 2:-1] & water[:, 1:-2])[:, :, 1:-1]
    cfv[:, 1:-1, 2:-1] = (water[:, :, 2:-1] & water[:, :, 1:-2])[:, 1:-1]
    top = torch.zeros_like(W2)
    top[:-1] |= cfu[nk, :-1] | cfu[nk, 1:]
    top[:, :-1] |= cfv[nk, :, :-1] | cfv[nk, :, 1:]
    cfw = top & (k >= KF + 1) & ink
    opn = torch.zeros_like(water)
    opn[:, :-1] |= cfu[:, :-1] | cfu[:, 1:]
    opn[:, :, :-1] |= cfv[:, :, :-1] | cfv[:, :, 1:]
    opn |= cfw
    opn[:-1] |= cfw[1:]
    opn &= inner & ink
    land = inner & ink & ~water

    # ---- fluxes: a streamfunction plus an overturning mode, w from continuity
    psi = _smooth(g, nj + 1, ni + 1, vanish=True)
    L = torch.nn.functional.pad(~wet, (1, 1, 1, 1), value=True)
    psi[L[:-1, :-1] | L[1:, :-1] | L[:-1, 1:] | L[1:, 1:]] = 0.0
    Tx, Ty = zeros(nJ, nI), zeros(nJ, nI)
    Tx[1:-1, 1:-1] = psi[:-1, 1:] - psi[:-1, :-1]
    Ty[1:-1, 1:-1] = -(psi[1:, :-1] - psi[:-1, :-1])
    peak = max(float(Tx.abs().max()), float(Ty.abs().max()), 1e-30)
    A = torch.zeros((2, nJ, nI), dtype=F64, device=dev)
    for q in range(2):
        s = _smooth(g, nj, ni)
        A[q, 1:-1, 1:-1] = 0.3 * peak * s / s.abs().max().clamp_min(1e-30)

    def layered(T2, A2, kface, cf):
        n = (nk - kface + 1).clamp_min(1).to(F64)
        mode = torch.cos(math.pi * ((k - kface) + 0.5) / n)
        return torch.where(cf, (T2 + A2 * mode) / n, 0.0)

    kfu, kfv = KF.clone(), KF.clone()
    kfu[1:] = torch.maximum(KF[1:], KF[:-1])
    kfv[:, 1:] = torch.maximum(KF[:, 1:], KF[:, :-1])
    Qx, Qy = layered(Tx, A[0], kfu, cfu), layered(Ty, A[1], kfv, cfv)
    AreaU, AreaV = DUZ * DVY, DVZ * DUX
    speed = torch.maximum((Qx.abs() / AreaU.clamp_min(1e-30)).max(),
                          (Qy.abs() / AreaV.clamp_min(1e-30)).max()).clamp_min(1e-30)
    Qx, Qy = Qx * (0.5 / speed), Qy * (0.5 / speed)
    div = torch.zeros_like(Qx)
    div[:, :-1] += Qx[:, :-1] - Qx[:, 1:]
    div[:, :, :-1] += Qy[:, :, :-1] - Qy[:, :, 1:]
    div = torch.where(water, div, 0.0)
    Qz = torch.where(cfw, torch.cumsum(div, 0) - div, 0.0)
    visc = 1.0 + 99.0 * rand(nK, nJ, nI)
    diffv = torch.exp(math.log(1e-6) + (math.log(1e-2) - math.log(1e-6)) * rand(nK, nJ, nI))

    geom = dict(DUX=DUX, DVY=DVY, DZX=DZX, DZY=DZY, KFloorZ=KF, AreaU=AreaU, AreaV=AreaV,
                DZZ=DZZ, DWZ=DWZ)
    i32 = torch.int32
    hydro = dict(Wflux_X=Qx, Wflux_Y=Qy, Wflux_Z=Qz, VolumeZOld=VolumeZOld, VolumeZ=VolumeZ,
                 OpenPoints3D=opn.to(i32), LandPoints3D=land.to(i32),
                 ComputeFacesU3D=cfu.to(i32), ComputeFacesV3D=cfv.to(i32),
                 ComputeFacesW3D=cfw.to(i32), WaterPoints3D=water.to(i32), Visc_H=visc,
                 Diff_V=diffv)
    # temperature, salinity, then log-normal nutrients
    tracers = []
    if c["kind"] not in ("solvers", "producers"):
        for t in range(c["tracers"]):
            if c["tracers"] >= 2 and t < 2:
                v = rand(nK, nJ, nI) * (20.0, 6.0)[t] + (5.0, 30.0)[t]
            else:
                v = torch.exp(torch.randn((nK, nJ, nI), generator=g, device=dev, dtype=F64))
            tracers.append(torch.where(inner & ink, torch.where(water, v, NULL_REAL), 0.0))
    method, limiter = SCHEMES[c["scheme"]]
    params = dict(schmidt_H=1.0, SchmidtCoef_V=1.0, SchmidtBackground_V=0.0, AdvMethodH=method,
                  TVDLimitationH=limiter, AdvMethodV=method, TVDLimitationV=limiter,
                  Upwind2H=method == TVD, Upwind2V=method == TVD, VolumeRelMax=1.5,
                  DTProp=c["dt"], ImpExp_AdvV=1.0, ImpExp_DifV=1.0,
                  ImpExp_AdvXX=float(c["implicit"] == "x"),
                  ImpExp_AdvYY=float(c["implicit"] == "y"), ImpExp_DifH=0.0, NullDif=False,
                  # WaterProperties' rule for the optimised path
                  Optimize=c["scheme"] == "superbee" and c["tracers"] >= 2)
    size, ws = (0, ni + 1, 0, nj + 1, 0, nk + 1), (1, ni, 1, nj, 1, nk)
    b = SimpleNamespace(size=size, ws=ws, geom=geom, hydro=hydro, tracers=tracers,
                        params=params, DUZ=DUZ, DVZ=DVZ, disch=None)
    if c["coastal"]:
        edge = inner.clone()
        edge[2:-2, 2:-2] = False
        hydro["BoundaryPoints2D"] = (edge & W2).to(i32)
        params.update(ReferenceProp=torch.full_like(Qx, 2.0), BoundaryCondition=1,
                      DecayTime=3600.0, CellFluxes=True)
        jj, ii = torch.nonzero(W2 & ~edge, as_tuple=True)
        pick = torch.randperm(len(ii), generator=g, device=dev)[:8]
        ii, jj = ii[pick].tolist(), jj[pick].tolist()
        n = len(ii)
        b.disch = dict(flow=[1.5 + 0.25 * q for q in range(n)], conc=[5.0] * n,
                       concMF=[1.0] * n, I=ii, J=jj, K=[nk] * n, Kmin=[-9999999] * n,
                       Kmax=[-9999999] * n, vert=[1] * n, ignore=[0] * n, ncells=[1] * n,
                       bypass=[0] * n)
    return b


def _rows(c, seed):
    """Diagonally dominant rows of the stand-alone solvers, and the water columns."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    shape = (c["nk"] + 2, c["nj"] + 2, c["ni"] + 2)
    r = [torch.rand(shape, generator=g, device="cuda", dtype=F64) for _ in range(4)]
    D, F = -0.9 * r[0], -0.9 * r[1]
    E = 1.0 + r[0] + r[1]
    TI = 35.0 * r[2]
    wp = torch.zeros(shape, dtype=torch.int32, device="cuda")
    wp[1:-1, 1:-1, 1:-1] = (r[3][-2, 1:-1, 1:-1] >= c["land"]).to(torch.int32)
    return D, E, F, TI, wp


# ---------------------------------------------------------------------------
class _Tracer:
    """A tracer of a batched handle where it lies in device memory; keeps the
    handle alive."""

    def __init__(self, tr, index, shape):
        import ctypes as ct

        from mohid_amd import _lib as L
        ptr, stride = ct.c_void_p(), ct.c_int64()
        L.check("tracer_ptr", L.lib().mgpu_transport_tracer_ptr(
            tr._h, index, ct.byref(ptr), ct.byref(stride)))
        self.owner = tr
        s = int(stride.value) * 8
        nK, nJ, nI = shape
        self.__cuda_array_interface__ = dict(
            shape=shape, typestr="<f8", strides=(s * nI * nJ, s * nI, s), version=2,
            data=(ptr.value, False))


def _host(t):
    """A device field as the Fortran-ordered host array it mirrors."""
    return t.cpu().numpy().T


def prepare(case, seed):
    from mohid_amd import _lib as L
    from mohid_amd.advection_diffusion import AdvectionDiffusion, Transport
    s = SimpleNamespace(kind=case["kind"], case=case)
    ni, nj, nk = case["ni"], case["nj"], case["nk"]
    if s.kind == "solvers":
        s.rows = _rows(case, seed)
        s.res = [torch.zeros_like(s.rows[0]) for _ in range(3)]
        s.size, s.ws = (0, ni + 1, 0, nj + 1, 0, nk + 1), (1, ni, 1, nj, 1, nk)
        return s
    b = s.b = _basin(case, seed)
    if s.kind != "producers":
        b.DUZ = b.DVZ = None
    if s.kind == "producers":
        s.out = {n: torch.zeros_like(b.DUZ)
                 for n in ("Qz", "VolumeZ", "VolumeU", "VolumeV", "AreaU", "AreaV")}
        s.DXX, s.DYY = b.geom["DUX"], b.geom["DVY"]
    elif s.kind == "host":
        s.geom = {n: _host(v) for n, v in b.geom.items()}
        s.hydro = {n: _host(v) for n, v in b.hydro.items()}
        s.props = [_host(t).copy(order="F") for t in b.tracers]
        s.ad = AdvectionDiffusion(b.size, b.ws, s.geom)
        b.tracers = b.hydro = b.geom = None
    elif s.kind == "call":
        s.ad = AdvectionDiffusion(b.size, b.ws, b.geom)
        s.props = b.tracers
    else:
        s.tr = Transport(b.size, b.ws, b.geom, case["tracers"],
                         precision=L.MGPU_PREC_FAST if case["precision"] == "fast" else
                         L.MGPU_PREC_FP64)
        if s.kind == "run":
            s.shape = tuple(b.tracers[0].shape)
            s.tr.set_hydro(b.hydro, b.params)
            for t, p in enumerate(b.tracers):
                s.tr.set_tracer(t, p)
            b.tracers = b.hydro = b.geom = None      # the handle keeps its own
        else:
            s.props = b.tracers
    return s


def run(state):
    """One pass; returns every field it computes, whole."""
    s, c = state, state.case
    if s.kind == "solvers":
        from mohid_amd.advection_diffusion import thomas3d, thomasz
        D, E, F, TI, wp = s.rows
        ni, nj, nk = c["ni"], c["nj"], c["nk"]
        thomasz(s.size, s.ws, D, E, F, TI, wp, s.res[0])
        thomas3d(s.size, 1, ni, 1, nj, 1, nk, 0, 1, D, E, F, TI, s.res[1])
        thomas3d(s.size, 1, nj, 1, ni, 1, nk, 1, 0, D, E, F, TI, s.res[2])
        return list(s.res)
    b = s.b
    if s.kind == "producers":
        from mohid_amd import producers as P
        h, g, o = b.hydro, b.geom, s.out
        P.compute_volumes(b.size, b.ws, g["DWZ"], g["DUX"], g["DVY"], o["VolumeZ"],
                          o["VolumeU"], o["VolumeV"])
        P.compute_areas(b.size, b.ws, b.DUZ, b.DVZ, s.DXX, s.DYY, o["AreaU"], o["AreaV"])
        P.waterflux_z(b.size, b.ws, h["Wflux_X"], h["Wflux_Y"], o["Qz"], h["ComputeFacesU3D"],
                      h["ComputeFacesV3D"], h["WaterPoints3D"], c["dt"], o["VolumeZ"],
                      h["VolumeZOld"])
        return dict(o)
    if s.kind in ("call", "host"):
        hydro = s.hydro if s.kind == "host" else b.hydro
        fluxes = []
        for t, p in enumerate(s.props):
            if b.disch:
                s.ad.set_discharges(b.disch)
            s.ad(p, hydro, b.params, first_property=t == 0)
            if b.disch:
                s.ad.unset_discharges()
                fluxes.append(s.ad.fluxes(like=p))
        # host fields as the (k, j, i) tensors the device ones are
        return {"props": [p.T if s.kind == "host" else p for p in s.props], "fluxes": fluxes}
    if s.kind == "coupled":
        for t, p in enumerate(s.props):
            s.tr.set_tracer(t, p)
        s.tr.set_geometry(b.geom)
        s.tr.set_hydro(b.hydro, b.params)
        s.tr.run(1)
        for t, p in enumerate(s.props):
            s.tr.get_tracer(t, out=p)
        return list(s.props)
    s.tr.run(c["steps"])
    return [torch.as_tensor(_Tracer(s.tr, t, s.shape), device="cuda")
            for t in range(c["tracers"])]


# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every field the path needs once and the tracers in and out, per
    step; flops: the arithmetic of a cell's faces, row and solve."""
    n = case["ni"] * case["nj"] * case["nk"]
    wet = n * (1.0 - case["land"]) * (0.56 if case["ragged"] else 1.0)
    T = case["tracers"]
    if case["kind"] == "solvers":        # four rows in, one solution out, three solves
        return {"bytes": 40.0 * n * (3.0 - case["land"]), "flops": 8.0 * n * 3}
    if case["kind"] == "producers":
        # DWZ in and three volumes out; two thicknesses in and two areas out;
        # fluxes, volumes and three masks in and the vertical flux out
        return {"bytes": n * (32.0 + 32.0 + 52.0), "flops": 20.0 * n}
    flops = 110.0 * wet * T * case["steps"]
    if case["kind"] == "run":
        # 8 shared fields read by every step, each tracer in and out
        return {"bytes": case["steps"] * wet * (16.0 * T + 64.0), "flops": flops}
    # eleven fields of the wet cells and six masks of all cells, once a step
    bytes_ = wet * 88.0 + n * 24.0 + wet * 16.0 * T
    if case["kind"] == "host":
        bytes_ = n * (11 * 8.0 + 24.0) + n * 16.0 * T
    if case["coastal"]:
        bytes_ += n * 48.0 * T           # six flux arrays out
    return {"bytes": bytes_, "flops": flops}


# ---------------------------------------------------------------------------
# What run() returns, in plain 64-bit torch.
def _sh(x, dim, o, fill=0.0):
    """y[n] = x[n + o] along dim, `fill` past the ends."""
    y = torch.full_like(x, fill)
    n = x.shape[dim]
    if o >= 0:
        y.narrow(dim, 0, n - o).copy_(x.narrow(dim, o, n - o))
    else:
        y.narrow(dim, -o, n + o).copy_(x.narrow(dim, 0, n + o))
    return y


def _coef(c, P, V, du, opn, Q, dim):
    """The advective flux of the face between a cell and the one before it
    along dim is D * P[n-1] + E * P[n]."""
    om1, om2, op1 = _sh(opn, dim, -1, False), _sh(opn, dim, -2, False), _sh(opn, dim, 1, False)
    pos = Q > 0.0
    D, E = torch.where(pos, Q, 0.0), torch.where(pos, 0.0, Q)
    if c["scheme"] != "upwind":
        Pm, Vm, dm = _sh(P, dim, -1), _sh(V, dim, -1, 1.0), _sh(du, dim, -1)
        down, upst = torch.where(pos, P, Pm), torch.where(pos, Pm, P)
        far = torch.where(pos, _sh(P, dim, -2), _sh(P, dim, 1))
        near = ~torch.where(pos, om2, op1)
        cr = Q * c["dt"] / torch.where(pos, Vm, V)
        s1 = du + dm
        s0 = torch.where(pos, dm + _sh(du, dim, -2), du + _sh(du, dim, 1))
        dc = (down - upst) / s1
        dc = torch.where(dc.abs() < 1e-16, torch.where(dc >= 0.0, 1e-16, -1e-16).to(F64), dc)
        r = (upst - far) / s0 / dc
        if c["scheme"] == "superbee":
            th = torch.maximum((2.0 * r).clamp(max=1.0).clamp(min=0.0), r.clamp(max=2.0))
        else:
            th = torch.minimum((2.0 * r).clamp(max=2.0), (1.0 + r) / 2.0).clamp(min=0.0)
        th = 0.5 * th * (1.0 - cr)
        th = torch.where(near, 0.0, th)
        D = torch.where(pos, Q * (1.0 - th), Q * th)
        E = torch.where(pos, Q * th, Q * (1.0 - th))
    both = opn & om1
    return torch.where(both, D, 0.0), torch.where(both, E, 0.0)


def _thomas(D, E, F, TI, dim):
    """x of D x[n-1] + E x[n] + F x[n+1] = TI along dim, from the first row."""
    Dn, En, Fn, Tn = (a.unbind(dim) for a in (D, E, F, TI))
    W, G = [-Fn[0] / En[0]], [Tn[0] / En[0]]
    for n in range(1, len(Dn)):
        aux = En[n] + Dn[n] * W[-1]
        W.append(-Fn[n] / aux)
        G.append((Tn[n] - Dn[n] * G[-1]) / aux)
    x = [G[-1]]
    for n in range(len(Dn) - 2, -1, -1):
        x.append(W[n] * x[-1] + G[n])
    return torch.stack(x[::-1], dim)


def _advance(c, b, P, axis):
    """One step of one tracer; axis: the implicit horizontal direction ("x",
    "y") or "none".  Returns the new tracer and the cell fluxes."""
    h, g, nk, dt = b.hydro, b.geom, c["nk"], c["dt"]
    m = {n: h[n] == 1 for n in ("OpenPoints3D", "LandPoints3D", "ComputeFacesU3D",
                                "ComputeFacesV3D", "ComputeFacesW3D", "WaterPoints3D")}
    opn, cfu, cfv, cfw = (m[n] for n in ("OpenPoints3D", "ComputeFacesU3D", "ComputeFacesV3D",
                                         "ComputeFacesW3D"))
    V, Vo, DUX, DVY = h["VolumeZ"], h["VolumeZOld"], g["DUX"], g["DVY"]
    dv = dt / V
    # face conductances
    nu = h["Visc_H"]
    DUXm, DVYm = _sh(DUX, 0, -1, 1.0), _sh(DVY, 1, -1, 1.0)
    cu = torch.where(cfu, (nu * DUXm + _sh(nu, 1, -1) * DUX) / (DUX + DUXm) * g["AreaU"] /
                     _sh(g["DZX"], 0, -1, 1.0), 0.0)
    cv = torch.where(cfv, (nu * DVYm + _sh(nu, 2, -1) * DVY) / (DVY + DVYm) * g["AreaV"] /
                     _sh(g["DZY"], 1, -1, 1.0), 0.0)
    cw = torch.where(cfw, h["Diff_V"] * DUX * DVY / _sh(g["DZZ"], 0, -1, 1.0), 0.0)
    # volume variation and horizontal diffusion
    TI = torch.where(opn, P * (Vo / V), P)
    if b.disch:
        for q, (i, j, k) in enumerate(zip(b.disch["I"], b.disch["J"], b.disch["K"])):
            if opn[k, j, i]:
                TI[k, j, i] += b.disch["flow"][q] * dv[k, j, i] * b.disch["conc"][q]
    fx, fy = cu * (P - _sh(P, 1, -1)), cv * (P - _sh(P, 2, -1))
    difx, dify = -fx, -fy
    TI = TI - fx * dv + _sh(fx, 1, 1) * dv - fy * dv + _sh(fy, 2, 1) * dv
    # horizontal advection, explicit directions
    Dx, Ex = (torch.where(cfu, a, 0.0) for a in
              _coef(c, P, V, DUX.expand_as(P), opn, h["Wflux_X"], 1))
    Dy, Ey = (torch.where(cfv, a, 0.0) for a in
              _coef(c, P, V, DVY.expand_as(P), opn, h["Wflux_Y"], 2))
    advx, advy = Dx * _sh(P, 1, -1) + Ex * P, Dy * _sh(P, 2, -1) + Ey * P
    if axis != "x":
        TI = TI + advx * dv - _sh(advx, 1, 1) * dv
    if axis != "y":
        TI = TI + advy * dv - _sh(advy, 2, 1) * dv
    E0 = torch.ones_like(TI)
    if axis == "none":
        E0[nk] = torch.where(opn[nk], 1.0 + dv[nk] * h["Wflux_Z"][nk + 1], 1.0)
    else:
        d = 1 if axis == "x" else 2
        Df, Ef = (Dx, Ex) if axis == "x" else (Dy, Ey)
        El = torch.ones_like(TI)
        El[nk] = torch.where(opn[nk], 1.0 + dv[nk] * h["Wflux_Z"][nk + 1], 1.0)
        rows = [0.0 - Df * dv, El - Ef * dv + _sh(Df, d, 1) * dv, _sh(Ef, d, 1) * dv, TI]
        n = P.shape[d]
        for q, v in enumerate((0.0, 1.0, 0.0, 0.0)):          # the ghost end row
            rows[q].narrow(d, n - 1, 1).fill_(v)
        o = 2 if d == 1 else 1                                # the lines of the WorkSize
        cut = [a[1:-1].narrow(d, 1, n - 1).narrow(o, 1, P.shape[o] - 2) for a in rows]
        P = P.clone()
        P[1:-1].narrow(d, 1, n - 1).narrow(o, 1, P.shape[o] - 2).copy_(_thomas(*cut, d))
        TI = P.clone()
    # vertical rows
    Dz, Ez = _coef(c, P, V, g["DWZ"], opn, h["Wflux_Z"], 0)
    build = cfw & opn[nk] if nk > 1 else torch.zeros_like(cfw)
    Dz, Ez = torch.where(build, Dz, 0.0), torch.where(build, Ez, 0.0)
    if nk == 1:
        cw = torch.zeros_like(cw)
    cwt, Dt, Et = _sh(cw, 0, 1), _sh(Dz, 0, 1), _sh(Ez, 0, 1)
    for a in (cwt, Dt, Et):
        a[nk] = 0.0
    D = (-cw - Dz) * dv
    E = E0 + (cw + cwt - Ez + Dt) * dv
    F = (-cwt + Et) * dv
    if c["coastal"]:
        bp, tdec = h["BoundaryPoints2D"] == 1, 1.0 / (1.0 + b.params["DecayTime"] / dt)
        X, Y, Z = (torch.where(f, h[q], 0.0) for f, q in
                   ((cfu, "Wflux_X"), (cfv, "Wflux_Y"), (cfw, "Wflux_Z")))
        wf = X - _sh(X, 1, 1) + Y - _sh(Y, 2, 1) + Z - _sh(Z, 0, 1) - (V - Vo) / dt
        kk = torch.arange(P.shape[0], device=P.device)[:, None, None]
        at = bp & opn & (kk >= g["KFloorZ"]) & (kk <= nk)
        ext = P * (1.0 - tdec) + b.params["ReferenceProp"] * tdec
        TI = torch.where(at & (wf < 0.0), TI - wf * ext * dv, TI)
        E = torch.where(at & ~(wf < 0.0), E + wf * dv, E)
    TI = torch.where(m["LandPoints3D"], NULL_REAL, TI)
    D[nk + 1], E[nk + 1], F[nk + 1], TI[nk + 1] = 0.0, 1.0, 0.0, 0.0
    if axis != "none":
        TI[nk + 1] = P[nk + 1]
    x = _thomas(D[1:], E[1:], F[1:], TI[1:], 0)
    out = P.clone()
    out[1:] = torch.where(m["WaterPoints3D"][nk], x, P[1:])
    flux = {}
    if c["coastal"]:
        flux = dict(AdvFluxX=advx, AdvFluxY=advy, DifFluxX=difx, DifFluxY=dify,
                    AdvFluxZ=Dz * _sh(out, 0, -1) + Ez * out,
                    DifFluxZ=-cw * (out - _sh(out, 0, -1)))
        flux = {n: torch.where(m[f], v, 0.0) for (n, v), f in zip(
            flux.items(), ["ComputeFacesU3D", "ComputeFacesV3D"] * 2 + ["ComputeFacesW3D"] * 2)}
    return out, flux


def exact(case, seed):
    c = case
    if c["kind"] == "solvers":
        D, E, F, TI, wp = _rows(c, seed)
        res = [torch.zeros_like(D) for _ in range(3)]
        rows = (D, E, F, TI)
        x = _thomas(*(a[1:, 1:-1, 1:-1] for a in rows), 0)
        res[0][1:, 1:-1, 1:-1] = torch.where(wp[-2, 1:-1, 1:-1] == 1, x, 0.0)
        res[1][1:-1, 1:, 1:-1] = _thomas(*(a[1:-1, 1:, 1:-1] for a in rows), 1)
        res[2][1:-1, 1:-1, 1:] = _thomas(*(a[1:-1, 1:-1, 1:] for a in rows), 2)
        return res
    b = _basin(c, seed)
    if c["kind"] == "producers":
        h, g = b.hydro, b.geom
        o = {n: torch.zeros_like(b.DUZ)
             for n in ("Qz", "VolumeZ", "VolumeU", "VolumeV", "AreaU", "AreaV")}
        i = (slice(1, -1),) * 3
        v = g["DWZ"] * g["DUX"] * g["DVY"]
        o["VolumeZ"][i] = v[i]
        o["VolumeU"][1:-1, 2:-1, 1:-1] = ((v[:, 1:-2] + v[:, 2:-1]) / 2)[1:-1, :, 1:-1]
        o["VolumeV"][1:-1, 1:-1, 2:-1] = ((v[:, :, 1:-2] + v[:, :, 2:-1]) / 2)[1:-1, 1:-1]
        o["AreaU"][i] = (b.DUZ * g["DVY"])[i]
        o["AreaV"][i] = (b.DVZ * g["DUX"])[i]
        X, Y = h["Wflux_X"] * h["ComputeFacesU3D"], h["Wflux_Y"] * h["ComputeFacesV3D"]
        d = X - _sh(X, 1, 1) + Y - _sh(Y, 2, 1) - (v - h["VolumeZOld"]) / c["dt"]
        wp = h["WaterPoints3D"] == 1
        for k in range(1, c["nk"] + 1):
            o["Qz"][k + 1] = torch.where(wp[k], o["Qz"][k] + d[k], o["Qz"][k + 1])
        return o
    props, fluxes = [], []
    for P in b.tracers:
        axis = c["implicit"]
        for _ in range(c["steps"]):
            P, flux = _advance(c, b, P, axis)
            axis = {"x": "y", "y": "x"}.get(axis, axis)
        props.append(P)
        if flux:
            fluxes.append(flux)
    if c["kind"] in ("call", "host"):
        return {"props": props, "fluxes": fluxes}
    return props

