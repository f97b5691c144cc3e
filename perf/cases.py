"""The measured work of this framework: what a SCALE-RM host or a Python program
has it do, through the public entry points of scale_amd.hip, over the sizes and
options of the repository's benchmark and tests.

Kinds of a case (all FP64 unless ``mixed``):

* ``short``     one RK4 short step of the resident model (filter, four HEVI
                stages, combination): the benchmark's headline step;
* ``large``     one large step: preparation, short step, RK3 tracers;
* ``adjoint``   a checkpointed forward of a few large steps and its adjoint;
* ``batch``     the same for several member models at once (terrain);
* ``ensemble``  one large step of an ensemble of uneven members, mixed
                precision, replayed from a graph;
* ``dropin``    one HEVI stage on host Fortran arrays, as a Fortran host calls it.

``exact`` is a plain torch FP64 restatement on periodic interior arrays
(levels, y, x), written from the scheme's equations.
"""
import math

import numpy as np
import torch

from scale_amd import hip, inputs

GRAV, RDRY, CPDRY, P00 = 9.80665, 287.04, 1004.64, 1.0e5
CPOVCV = CPDRY / (CPDRY - RDRY)
EPS = float(np.finfo(np.float64).eps)
BV2 = 1.5e-4  # Brunt-Vaisala frequency squared of the base state [1/s2]
STATE = ("DENS", "MOMZ", "MOMX", "MOMY", "RHOT")
# members of the ensemble and the terrain batch: (imax, jmax, kmax)
ENSEMBLE = ((96, 96, 48), (128, 128, 64), (96, 96, 48), (192, 192, 64), (96, 96, 48), (128, 128, 64))
CASE = dict(kind="large", imax=64, jmax=64, kmax=48, dx=500.0, dz0=250.0, dz1=250.0, scheme=3, tracers=0,
            tracer_scheme=3, fct=True, mixed=False, height=0.0, steps=0, every=0, members=1)


def _case(name=None, **kw):
    c = dict(CASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest earnest run: the dry warm bubble of the tests and of the reference's own test set
        _case("bubble 40x40x80", imax=40, jmax=40, kmax=80, tracers=1, fct=False),
        # an odd domain with the reference's default tracer scheme, central dynamics, stretched levels
        _case("ragged 97x61x45 CD4 Koren", imax=97, jmax=61, kmax=45, dz0=80.0, dz1=500.0, scheme=4, tracers=2,
              tracer_scheme=31),
        # an ordinary single-GPU domain with the benchmark's three limited tracers
        _case("large 128x128x64", imax=128, jmax=128, kmax=64, tracers=3),
        # the same at a size that fills the device: most of the step is tracer advection
        _case("large 320x320x96", imax=320, jmax=320, kmax=96, dx=1000.0, dz0=60.0, dz1=400.0, tracers=3),
        # the headline benchmark: FP64 short step at its full size
        _case("short 512x512x128", kind="short", imax=512, jmax=512, kmax=128, dx=1000.0, dz0=50.0, dz1=400.0),
        # FP32 dynamics with the FP64 solve (the reference's single-precision build), large domain
        _case("mixed 512x384x96", imax=512, jmax=384, kmax=96, dx=1000.0, dz0=60.0, dz1=400.0, tracers=1, mixed=True),
        # flow over a mountain, the batched adjoint's member size: Coriolis force and a sponge layer
        _case("terrain 128x128x64", imax=128, jmax=128, kmax=64, tracers=1, height=500.0),
        # a larger ragged domain over terrain: the general-metrics path is the reference's only path
        _case("terrain 301x259x80", imax=301, jmax=259, kmax=80, tracers=1, height=500.0),
        # sensitivities: the benchmark's adjoint domain
        _case("adjoint 128x128x64", kind="adjoint", imax=128, jmax=128, kmax=64, steps=8, every=4),
        # sensitivities of several mountain flows at once
        _case("batch adjoint 3x64x48x40", kind="batch", imax=64, jmax=48, kmax=40, height=500.0, steps=4, every=2,
              members=3),
        # uneven ensemble members advanced together
        _case("ensemble 6 members", kind="ensemble", tracers=1, mixed=True, members=6),
        # a Fortran host's call: every array crosses PCIe
        _case("dropin 128x128x64", kind="dropin", imax=128, jmax=128, kmax=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["short", "large", "large", "large", "mixed", "terrain", "terrain", "adjoint", "batch", "ensemble",
                       "dropin"])
    kmax = rng.randint(24, 128)
    scheme = rng.choice([3, 3, 4])
    dz0, dz1 = rng.choice([(250.0, 250.0), (60.0, 400.0), (100.0, 300.0)])
    if (dz0 + dz1) * kmax / 2 > 30000.0:
        kmax = int(60000.0 / (dz0 + dz1))
    c = dict(kmax=kmax, scheme=scheme, dz0=dz0, dz1=dz1)
    if kind == "short":
        return _case(kind="short", imax=_log(rng, 30, 512), jmax=_log(rng, 30, 512), **c)
    if kind in ("large", "mixed", "terrain"):
        top = 384 if kind != "terrain" else 256
        return _case(imax=_log(rng, 30, top), jmax=_log(rng, 30, top), tracers=rng.randint(0, 3 if kind == "large" else 1),
                     tracer_scheme=rng.choice([3, 31, 4]), fct=rng.random() < 0.7, mixed=kind == "mixed",
                     height=rng.choice([200.0, 500.0]) if kind == "terrain" else 0.0, **c)
    if kind == "adjoint":
        c["kmax"] = min(kmax, 64)
        return _case(kind="adjoint", imax=_log(rng, 24, 128), jmax=_log(rng, 24, 128), steps=rng.randint(2, 8), every=2,
                     height=rng.choice([0.0, 300.0]), **c)
    if kind == "batch":
        c["kmax"] = min(kmax, 48)
        return _case(kind="batch", imax=_log(rng, 24, 64), jmax=_log(rng, 24, 64), steps=rng.randint(2, 4), every=2,
                     height=rng.choice([0.0, 300.0, 500.0]), members=rng.randint(2, 4), **c)
    if kind == "ensemble":
        return _case(kind="ensemble", tracers=1, mixed=rng.random() < 0.7, members=rng.randint(2, 6),
                     imax=rng.randint(0, 40))  # imax: shrinks the members, for odd sizes
    return _case(kind="dropin", imax=_log(rng, 24, 128), jmax=_log(rng, 24, 128), height=rng.choice([0.0, 300.0]),
                 **dict(c, kmax=min(kmax, 64)))


# ---- inputs: made from the seed on the GPU -------------------------------------
class _Grid1D:
    """1-D grid: level thicknesses with two ghost levels each side (CDZ, FDZ), centre and face heights."""

    def __init__(self, c):
        n = c["kmax"]
        dz = [c["dz0"] + (c["dz1"] - c["dz0"]) * k / max(n - 1, 1) for k in range(n)]
        self.dz = np.array(dz)
        self.cdz = np.array([dz[0]] * 2 + dz + [dz[-1]] * 2)
        self.fz = np.concatenate([[0.0], np.cumsum(self.cdz)]) - 2 * dz[0]
        self.cz = 0.5 * (self.fz[1:] + self.fz[:-1])
        self.cdz = self.fz[1:] - self.fz[:-1]
        self.fdz = self.cz[1:] - self.cz[:-1]
        self.dx = c["dx"]
        self.dt = 1.0 if c["dx"] <= 500.0 else 2.0
        self.top = self.fz[n + 2]
        self.wdamp = np.zeros(n + 4)
        if c["height"] > 0.0:  # sponge layer over the upper 30 %
            h = 0.7 * self.top
            f = self.fz[1:]
            w = np.where(f >= h, 0.5 * (1.0 - np.cos(math.pi * (f - h) / (self.top - h))), 0.0) / 300.0
            w[:2], w[n + 2:] = w[2], w[n + 1]
            self.wdamp = w
        self.f0 = 1.0e-4 if c["height"] > 0.0 else 0.0


def _surface(c):
    """Surface height (jmax, imax): a bell-shaped mountain in the centre."""
    i = (torch.arange(c["imax"], device="cuda", dtype=torch.float64) + 0.5) * c["dx"]
    j = (torch.arange(c["jmax"], device="cuda", dtype=torch.float64) + 0.5) * c["dx"]
    x, y = i[None, :] - 0.5 * c["imax"] * c["dx"], j[:, None] - 0.5 * c["jmax"] * c["dx"]
    return c["height"] / (1.0 + (x / 5000.0) ** 2 + (y / 5000.0) ** 2)


def _fields(c, seed):
    """The state, reference state and tracers on the interior (levels, y, x), with the ghost levels of the
    reference pressure: stably stratified air with sheared wind, smooth waves in v and w, a warm bubble and noise."""
    g = _Grid1D(c)
    K, J, I = c["kmax"], c["jmax"], c["imax"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    f64 = dict(device="cuda", dtype=torch.float64)
    zeta = torch.tensor(g.cz, **f64)[:, None, None]
    zs = _surface(c)[None] if c["height"] > 0.0 else torch.zeros(1, 1, 1, **f64)
    z = ((g.top - zs) / g.top * zeta + zs).expand(K + 4, J, I)  # heights of the centres
    theta = 300.0 * torch.exp(BV2 / GRAV * z)
    pi = 1.0 - GRAV ** 2 / (CPDRY * BV2 * 300.0) * (1.0 - torch.exp(-BV2 / GRAV * z))
    pres = P00 * pi ** (CPDRY / RDRY)
    dens = pres / (RDRY * theta * pi)
    # the pressure just outside the domain that the hydrostatic balance across KS and KE gives
    rpres = pres.clone()
    rpres[1] = pres[3] - dens[2] * GRAV * (z[1] - z[3])
    rpres[K + 2] = pres[K] - dens[K + 1] * GRAV * (z[K + 2] - z[K])
    s = slice(2, K + 2)
    x = (torch.arange(I, **f64) + 0.5)[None, None, :] / I
    y = (torch.arange(J, **f64) + 0.5)[None, :, None] / J
    zn = z[s] / g.top
    ph = torch.rand(6, generator=gen, **f64) * 2 * math.pi
    tw = 2 * math.pi
    r2 = ((x - 0.5) * I * g.dx / 2000.0) ** 2 + ((y - 0.5) * J * g.dx / 2000.0) ** 2 + ((z[s] - 2000.0) / 2000.0) ** 2
    th = theta[s] + 2.0 * torch.cos(0.5 * math.pi * torch.sqrt(r2.clamp(max=1.0))) ** 2
    th = th + 0.1 * torch.randn(K, J, I, generator=gen, **f64)
    u = 5.0 + 15.0 * (z[s] / 10000.0).clamp(max=1.0) + torch.sin(tw * y + ph[0]) * torch.cos(math.pi * zn)
    v = 2.0 * torch.sin(tw * x + ph[1]) * torch.cos(math.pi * zn + ph[2])
    w = 0.3 * torch.sin(tw * x + ph[3]) * torch.cos(tw * y + ph[4]) * torch.sin(math.pi * zn)
    d = dens[s].contiguous()
    st = dict(DENS=d, MOMZ=d * w, MOMX=d * u, MOMY=d * v, RHOT=d * th)
    st["MOMZ"][-1] = 0.0
    tr = []
    for q in range(c["tracers"]):
        if q % 3 == 0:  # a smooth blob
            r = ((x - 0.3) / 0.15) ** 2 + ((y - 0.5) / 0.15) ** 2 + ((zn - 0.2) / 0.15) ** 2
            tr.append(1.0e-3 * torch.cos(0.5 * math.pi * torch.sqrt(r.clamp(max=1.0))) ** 2)
        elif q % 3 == 1:  # a top hat
            tr.append(torch.where(((x - 0.5).abs() < 0.2) & ((y - 0.5).abs() < 0.2) & (zn < 0.3), 1.0e-3, 0.0).to(torch.float64))
        else:  # a filled field
            tr.append(1.0e-3 * (1.0 + 0.1 * torch.randn(K, J, I, generator=gen, **f64)))
    ref = dict(REF_dens=dens, REF_pott=theta, REF_pres=rpres)
    return g, st, ref, [t.contiguous() for t in tr]


def _halo(a):
    """Periodic two-cell halo in y and x."""
    a = torch.cat([a[:, :, -2:], a, a[:, :, :2]], 2)
    return torch.cat([a[:, -2:], a, a[:, :2]], 1)


def _ghost(a, name):
    """Two ghost levels each side: zero for MOMZ, the boundary level's values otherwise."""
    e = torch.zeros_like(a[:1]) if name == "MOMZ" else None
    lo, hi = (e, e) if name == "MOMZ" else (a[:1], a[-1:])
    return torch.cat([lo, lo, a, hi, hi], 0)


def _host(a):
    """(levels, y, x[, components]) on the GPU -> NumPy (KA, IA, JA[, ...]) in Fortran order."""
    return a.permute(*range(a.dim() - 1, 2, -1), 1, 2, 0).contiguous().cpu().numpy().T


def _grid(c, g):
    return inputs.Grid(c["kmax"], c["imax"], c["jmax"], g.dx, g.dx, g.dz)


def _metric(c, g):
    """1-D grid arrays and unit map factors."""
    IA, JA = c["imax"] + 4, c["jmax"] + 4
    m = dict(CDZ=g.cdz, FDZ=g.fdz, RCDZ=1.0 / g.cdz, RFDZ=1.0 / g.fdz, MAPF=np.ones((IA, JA, 2, 4), order="F"), J33G=1.0)
    for ax, n in (("X", IA), ("Y", JA)):
        m.update({"CD" + ax: np.full(n, g.dx), "FD" + ax: np.full(n - 1, g.dx), "RCD" + ax: np.full(n, 1.0 / g.dx),
                  "RFD" + ax: np.full(n - 1, 1.0 / g.dx)})
    return m


class _View:
    """A resident field of a context as a tensor: keeps the context alive."""

    def __init__(self, ctx, fid, shape):
        self.ctx = ctx
        p = hip.C.POINTER(hip.C.c_double)()
        rc = hip.load_library().scale_hip_model_device_ptr(ctx._h, hip.C.c_int32(fid), hip.C.byref(p))
        if rc != 0:
            raise RuntimeError("scale_hip_model_device_ptr failed")
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8", version=2,
                                             data=(hip.C.cast(p, hip.C.c_void_p).value, False))


def _outputs(ctx, c):
    """The model's state (whole arrays) and, on the interior where alone they are defined, its mass and theta
    fluxes and tracers, as tensors of the resident buffers."""
    g = ctx.grid
    shape = (g.KA, g.JA, g.IA)
    inner = (Ellipsis, slice(2, -2), slice(2, -2), slice(2, -2))
    dev = lambda fid, sh=shape: torch.as_tensor(_View(ctx, fid, sh), device="cuda")  # noqa: E731
    out = {k: dev(hip.FIELD[k]) for k in STATE}
    if not c["mixed"] and c["kind"] in ("short", "large"):
        out["mflx_hi"] = dev(hip.FIELD["mflx_hi"], (3,) + shape)[inner]
        out["tflx_hi"] = dev(hip.FIELD["tflx_hi"], (3,) + shape)[inner]
    for q in range(c["tracers"]):
        out["QTRC%d" % q] = dev(hip.QTRC_BASE + q)[inner]
    return out


def _model(c, seed):
    """A context whose resident model holds the case's inputs."""
    g, st, ref, tr = _fields(c, seed)
    ctx = hip.Context(_grid(c, g), c["scheme"], c["tracer_scheme"])
    zs = _halo(_surface(c)[None])[0].T.contiguous().cpu().numpy() if c["height"] > 0.0 else \
        np.zeros((c["imax"] + 4, c["jmax"] + 4))
    ctx.set_terrain(_metric(c, g), g.fz, np.asfortranarray(zs))
    ctx.model_create(g.dt, g.dt, c["tracers"], fct_tracer=c["fct"], mixed_precision=c["mixed"])
    for k, v in ref.items():
        ctx.model_set(k, _host(_halo(v)))
    for k, v in st.items():
        ctx.model_set(k, _host(_halo(_ghost(v, k))))
    ctx.model_set("CORIOLI", np.full((1, c["imax"] + 4, c["jmax"] + 4), g.f0, order="F"))
    ctx.model_set("wdamp_coef", g.wdamp)
    for q, v in enumerate(tr):
        ctx.model_set(hip.QTRC_BASE + q, _host(_halo(_ghost(v, "QTRC"))))
    ctx.synchronize()
    return ctx


def _sensitivity(c, seed):
    """Adjoints of the final state of an objective on a box in the middle, scaled by the fields' magnitudes."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed) + 1)
    K, J, I = c["kmax"], c["jmax"], c["imax"]
    out = {}
    for k, scale in zip(STATE, (1.0, 1.0, 0.1, 1.0, 1.0 / 300.0)):
        a = torch.zeros(K, J, I, device="cuda", dtype=torch.float64)
        b = (slice(1, K // 2), slice(J // 4, J - J // 4), slice(I // 4, I - I // 4))
        a[b] = scale * (1.0 + 0.2 * torch.randn(a[b].shape, generator=gen, device="cuda", dtype=torch.float64))
        e = torch.zeros(2, J, I, device="cuda", dtype=torch.float64)
        out[k] = _host(torch.nn.functional.pad(torch.cat([e, a, e], 0), (2, 2, 2, 2)))
    return out


def _members(c):
    """The cases of an ensemble's members."""
    out = []
    for m in range(c["members"]):
        i, j, k = ENSEMBLE[m % len(ENSEMBLE)]
        less = c["imax"] if c["imax"] < 48 else 0
        out.append(dict(c, imax=i - less, jmax=j - less // 2, kmax=k))
    return out


def prepare(case, seed):
    c = dict(CASE, **case)
    kind = c["kind"]
    if kind in ("short", "large", "adjoint"):
        ctx = _model(c, seed)
        s = dict(kind=kind, ctx=ctx, c=c, out=_outputs(ctx, c))
        if kind == "short":
            ctx.model_prepare()
        if kind == "adjoint":
            s["xb"] = _sensitivity(c, seed)
        return s
    if kind == "batch":
        ctxs = [_model(c, seed + 1000 * m) for m in range(c["members"])]
        return dict(kind=kind, ctxs=ctxs, c=c, xbs=[_sensitivity(c, seed + 1000 * m) for m in range(c["members"])],
                    out=[_outputs(x, c) for x in ctxs])
    if kind == "ensemble":
        ctxs = [_model(m, seed + 1000 * q) for q, m in enumerate(_members(c))]
        ens = hip.Ensemble(ctxs)
        ens.set_graph(True)
        return dict(kind=kind, ens=ens, c=c, out=[_outputs(x, c) for x in ctxs])
    # dropin: the host's own arrays
    g, st, ref, _ = _fields(c, seed)
    ctx = hip.Context(_grid(c, g), c["scheme"], c["scheme"])
    P = _prep(c, g, st, ref)
    nd = _filter(c, g, st, ref, g.dt)
    h = {k: _host(_halo(_ghost(v, k))) for k, v in st.items()}
    g1 = ctx.grid
    z = lambda *e: np.zeros((g1.KA, g1.IA, g1.JA) + e, order="F")  # noqa: E731
    num_diff = torch.zeros(3, 5, g1.KA, g1.JA, g1.IA, device="cuda", dtype=torch.float64)
    for (v, d), a in nd.items():
        num_diff[d, v, 2:-2] = _halo(a)
    M = _metrics(c, g)
    full = lambda a: _halo(a.expand(-1, c["jmax"], c["imax"]))  # noqa: E731
    met = {n: np.asfortranarray(np.stack([_host(full(a)) for a in M[n]], 3)) for n in ("G", "J13", "J23")}
    return dict(kind=kind, ctx=ctx, c=c, g=g, st=h, m=_metric(c, g), met=met, PHI=_host(full(M["phi"])),
                num_diff=num_diff.permute(0, 1, 3, 4, 2).contiguous().cpu().numpy().transpose(4, 3, 2, 1, 0), zero=z(),
                pres={k: _host(_halo(P[k + "_all"])) for k in ("DPRES0", "RT2P", "REF_rhot")}, REF_dens=_host(_halo(ref["REF_dens"])),
                cor=np.full((1, g1.IA, g1.JA), g.f0, order="F"), out={k + "_RK": h[k].copy(order="F") for k in STATE},
                flux=dict(mflx_hi=z(3), tflx_hi=z(3)))


def run(state):
    kind = state["kind"]
    if kind == "large":
        state["ctx"].model_large_step(1)
        return state["out"]
    if kind == "short":
        state["ctx"].model_short_step(1)
        return state["out"]
    if kind == "adjoint":
        state["ctx"].model_forward_checkpointed(state["c"]["steps"], state["c"]["every"])
        return dict(state["out"], **{k + "_b": v for k, v in state["ctx"].model_adjoint(state["xb"]).items()})
    if kind == "batch":
        hip.batch_forward_checkpointed(state["ctxs"], state["c"]["steps"], state["c"]["every"])
        xb = hip.batch_adjoint(state["ctxs"], state["xbs"])
        return [dict(o, **{k + "_b": v for k, v in b.items()}) for o, b in zip(state["out"], xb)]
    if kind == "ensemble":
        state["ens"].large_step(1)
        return state["out"]
    s, m, met, p = state["st"], state["m"], state["met"], state["pres"]
    o, f, z, g = state["out"], state["flux"], state["zero"], state["g"]
    state["ctx"].ATMOS_DYN_Tstep_short_fvm_hevi(
        *[o[k + "_RK"] for k in STATE], None, f["mflx_hi"], f["tflx_hi"], *[s[k] for k in STATE], *[s[k] for k in STATE],
        z, z, z, z, z, None, None, p["DPRES0"], p["RT2P"], state["cor"], state["num_diff"], g.wdamp, 0.0, z,
        False, False, True, m["CDZ"], m["FDZ"], m["FDX"], m["FDY"], m["RCDZ"], m["RCDX"], m["RCDY"], m["RFDZ"], m["RFDX"],
        m["RFDY"], state["PHI"], met["G"], met["J13"], met["J23"], m["J33G"], m["MAPF"], state["REF_dens"], p["REF_rhot"],
        False, False, False, False, g.dt, False)
    inner = (slice(2, -2), slice(2, -2), slice(2, -2))
    return dict({k: v[inner] for k, v in o.items()}, mflx_hi=f["mflx_hi"][inner], tflx_hi=f["tflx_hi"][inner])


# ---- what a pass cannot do without ---------------------------------------------
def _points(c):
    return c["imax"] * c["jmax"] * c["kmax"]


def work(case):
    """Inputs read once and outputs written once, in the storage type of the dynamics, and the operations of the
    sweeps (counted per interior point from the scheme: about 800 a stage, 300 the filter, 100 a tracer stage,
    350 the limited one; the adjoint twice the forward's)."""
    c = dict(CASE, **case)
    if c["kind"] == "ensemble":
        w = [work(dict(m, kind="large")) for m in _members(c)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if c["kind"] == "batch":
        w = work(dict(c, kind="adjoint"))
        return {k: v * c["members"] for k, v in w.items()}
    n = _points(c)
    b = 4 if c["mixed"] else 8
    metrics = 22 * 8 if c["height"] > 0.0 else 0
    if c["kind"] == "dropin":  # 5 + 5 state, 5 tendencies, 4 pressure and reference, 15 filter in; 5 + 6 out
        return {"bytes": float(n * (34 * 8 + 11 * 8 + metrics)), "flops": 800.0 * n}
    step = n * (5 * b + 3 * 8 + 11 * b + metrics)  # state and reference state in; state and fluxes out
    flops = n * (4 * 800.0 + 300.0)
    if c["kind"] == "short":
        return {"bytes": float(step), "flops": flops}
    if c["kind"] == "large":
        return {"bytes": float(step + n * 16 * c["tracers"]),
                "flops": flops + n * c["tracers"] * (200.0 + (350.0 if c["fct"] else 100.0))}
    # the adjoint: the state in, the state and its adjoint in and out, per step one state kept and read again
    return {"bytes": float(n * 8 * (5 + 3 + 5 + 10 + 10 * c["steps"]) + n * metrics), "flops": 3.0 * c["steps"] * flops}


def tolerance(case):
    c = dict(CASE, **case)
    if c["mixed"]:
        # four times the FP32 dynamics' distance from the FP64 restatement (1.8e-6, in w, the small difference of
        # large terms)
        return {"rel": 8e-6}
    # four times the FP64 paths' largest distance from the restatement, whose sums have another order (9e-14, in w)
    return {"rel": 4e-13}


# ---- plain FP64 restatement ------------------------------------------------------
def _x(a, n):
    return torch.roll(a, -n, 2)


def _y(a, n):
    return torch.roll(a, -n, 1)


def _sign(v, size=1.0):
    return torch.copysign(torch.full_like(v, size), v)


def _koren(v1, v2, v3):
    z1 = EPS - torch.copysign(torch.full_like(v1, EPS), (v1 - v2).abs() - EPS)
    z2 = EPS - torch.copysign(torch.full_like(v1, EPS), (v2 - v3).abs() - EPS)
    r2 = 2.0 * (v1 - v2 + z1 * z2) / (v2 - v3 + z2)
    return torch.minimum(r2, ((1.0 + r2) / 3.0).clamp(max=2.0)).clamp(min=0.0)


def _face(s, qm, q0, q1, q2, vel):
    """Value at the face between q0 and q1."""
    if s == 31:
        return (q0 + 0.5 * _koren(q1, q0, qm) * (q0 - qm)) * (0.5 + _sign(vel, 0.5)) \
            + (q1 + 0.5 * _koren(q0, q1, q2) * (q1 - q2)) * (0.5 - _sign(vel, 0.5))
    cd = 7.0 / 12.0 * (q1 + q0) - 1.0 / 12.0 * (q2 + qm)
    return cd if s == 4 else cd - (3.0 / 12.0 * (q1 - q0) - 1.0 / 12.0 * (q2 - qm)) * _sign(vel)


def _low(s, q0, q1, q2, vel):
    """Value at the lowest face."""
    up, dn = 0.5 + _sign(vel, 0.5), 0.5 - _sign(vel, 0.5)
    if s == 31:
        return q0 * up + (q1 + 0.5 * _koren(q0, q1, q2) * (q1 - q2)) * dn
    return 0.5 * (q0 + q1) if s == 4 else 0.5 * (q0 + q1) * up + (2.0 * q0 + 5.0 * q1 - q2) / 6.0 * dn


def _high(s, qm, q0, q1, vel):
    """Value at the highest face."""
    up, dn = 0.5 + _sign(vel, 0.5), 0.5 - _sign(vel, 0.5)
    if s == 31:
        return (q0 + 0.5 * _koren(qm, q0, q1) * (q0 - q1)) * up + q1 * dn
    return 0.5 * (q0 + q1) if s == 4 else (2.0 * q1 + 5.0 * q0 - qm) / 6.0 * up + 0.5 * (q0 + q1) * dn


def _zface(s, q, vel):
    """Values at the inner horizontal faces of a column field."""
    return torch.cat([_low(s, q[:1], q[1:2], q[2:3], vel[:1]), _face(s, q[:-3], q[1:-2], q[2:-1], q[3:], vel[1:-1]),
                      _high(s, q[-3:-2], q[-2:-1], q[-1:], vel[-1:])])


def _dz(f):
    """Difference of the inner faces' fluxes across each cell, zero at both ends."""
    return torch.cat([f[:1], f[1:] - f[:-1], -f[-1:]])


XYZ, XYW, UYW, XVW, UYZ, XVZ, UVZ = range(7)


def _metrics(c, g):
    """GSQRT, J13G and J23G (7 components each) and PHI of Gal-Chen heights on all levels; one column when flat."""
    f64 = dict(device="cuda", dtype=torch.float64)
    col = lambda a: torch.tensor(a, **f64)[:, None, None]  # noqa: E731
    if c["height"] <= 0.0:
        one = torch.ones(c["kmax"] + 4, 1, 1, **f64)
        return dict(G=[one] * 7, J13=[one * 0.0] * 7, J23=[one * 0.0] * 7, phi=GRAV * col(g.cz))
    zx = _surface(c)[None]
    zu, zv = 0.5 * (zx + _x(zx, 1)), 0.5 * (zx + _y(zx, 1))
    zuv = 0.25 * (zx + _x(zx, 1) + _y(zx, 1) + _x(_y(zx, 1), 1))
    h = lambda zs, a: (g.top - zs) / g.top * col(a) + zs  # noqa: E731
    C = [h(a, g.cz) for a in (zx, zu, zv, zuv)]
    F = [h(a, g.fz) for a in (zx, zu, zv, zuv)]
    full = lambda f: (f[1:] - f[:-1]) / col(g.cdz)  # noqa: E731
    def half(a):
        d = (a[1:] - a[:-1]) / col(g.fdz)
        return torch.cat([d, d[-1:]])
    G = [full(F[0]), half(C[0]), half(C[1]), half(C[2]), full(F[1]), full(F[2]), full(F[3])]
    T = [f[1:] for f in F]
    bx = lambda a: -(a - _x(a, -1)) / g.dx  # noqa: E731
    fx = lambda a: -(_x(a, 1) - a) / g.dx  # noqa: E731
    by = lambda a: -(a - _y(a, -1)) / g.dx  # noqa: E731
    fy = lambda a: -(_y(a, 1) - a) / g.dx  # noqa: E731
    J13 = [bx(C[1]), bx(T[1]), fx(T[0]), bx(T[3]), fx(C[0]), bx(C[3]), fx(C[2])]
    J23 = [by(C[2]), by(T[2]), by(T[3]), fy(T[0]), by(C[3]), fy(C[0]), fy(C[1])]
    return dict(G=G, J13=J13, J23=J23, phi=GRAV * C[0])


def _prep(c, g, st, ref):
    """Pressure terms of the large step's start; the _all arrays hold the ghost levels too."""
    T = st["RHOT"]
    pres = P00 * (RDRY * T / P00) ** CPOVCV
    rp = ref["REF_pres"]
    d0 = pres - rp[2:-2]
    lo, hi = d0[1:2] + (rp[3:4] - rp[1:2]), d0[-2:-1] + (rp[-4:-3] - rp[-2:-1])
    o = torch.zeros_like(lo)
    rt2p = CPOVCV * pres / T
    return dict(DPRES0=d0, lo=lo, hi=hi, RT2P=rt2p, REF_rhot=T, DPRES0_all=torch.cat([o, lo, d0, hi, o]),
                RT2P_all=torch.cat([o, o, rt2p, o, o]), REF_rhot_all=torch.cat([o, o, T, o, o]))


def _filter(c, g, st, ref, dt):
    """Fourth-order numerical diffusion fluxes {(variable, direction z/x/y)} with coefficient 1e-4."""
    f64 = dict(device="cuda", dtype=torch.float64)
    col = lambda a: torch.tensor(np.asarray(a), **f64)[:, None, None]  # noqa: E731
    cdz, fdz = col(g.cdz[2:-2]), col(g.fdz[2:-2])  # K and K-1 values
    k4 = 1.0e-4 / 16.0 / dt
    D, W, U, V, T = (st[k] for k in STATE)

    def third_z(p):  # at the inner faces, mirrored about the lowest and highest level
        d1 = (p[1:] - p[:-1]) / fdz
        d2 = torch.cat([2.0 * d1[:1], d1[1:] - d1[:-1], -2.0 * d1[-1:]]) / cdz
        return (d2[1:] - d2[:-1]) / fdz

    def third_w(p):  # of a face field p (levels 0..K-2) at the cells 1..K-2; p mirrored below, zero above
        q = torch.cat([p[1:2], p, torch.zeros_like(p[:1])])  # faces -1..K-1
        d1 = (q[1:] - q[:-1]) / cdz  # cells 0..K-1
        d2 = (d1[1:] - d1[:-1]) / fdz  # faces 0..K-2
        return (d2[1:] - d2[:-1]) / cdz[1:-1]

    def third(p, sh, half):  # centred fields at the face ahead (half = 0), face fields at the cell (half = 1)
        o = 0 if half else 1
        return (sh(p, 1 + o) - 3.0 * sh(p, o) + 3.0 * sh(p, o - 1) - sh(p, o - 2)) / g.dx ** 3

    x4 = k4 * g.dx ** 4
    z4, w4 = k4 * cdz ** 4, k4 * fdz ** 4
    pad = lambda a, n=1: torch.nn.functional.pad(a, (0, 0, 0, 0, 0, n))  # noqa: E731
    up = lambda a: a[1:] + a[:-1]  # noqa: E731
    nd = {}
    p = D - ref["REF_dens"][2:-2]
    nd[0, 0] = pad(third_z(p) * z4[:-1])
    nd[0, 1], nd[0, 2] = third(p, _x, 0) * x4, third(p, _y, 0) * x4
    p = 2.0 * W[:-1] / up(D)
    nd[1, 0] = torch.nn.functional.pad(third_w(p) * w4[1:] * D[1:-1], (0, 0, 0, 0, 1, 1))
    nd[1, 1] = pad(third(p, _x, 0) * x4 * 0.25 * up(D + _x(D, 1)))
    nd[1, 2] = pad(third(p, _y, 0) * x4 * 0.25 * up(D + _y(D, 1)))
    for v, m, own, oth in ((2, U, 1, 2), (3, V, 2, 1)):
        so, st_ = (_x, _y) if own == 1 else (_y, _x)
        p = 2.0 * m / (so(D, 1) + D)
        nd[v, 0] = pad(third_z(p) * z4[:-1] * 0.25 * up(so(D, 1) + D))
        nd[v, own] = third(p, so, 1) * x4 * D
        nd[v, oth] = third(p, st_, 0) * x4 * 0.25 * (D + so(D, 1) + st_(D, 1) + so(st_(D, 1), 1))
    p = T / D - ref["REF_pott"][2:-2]
    nd[4, 0] = pad(third_z(p) * z4[:-1] * 0.5 * up(D))
    nd[4, 1], nd[4, 2] = third(p, _x, 0) * x4 * 0.5 * (_x(D, 1) + D), third(p, _y, 0) * x4 * 0.5 * (_y(D, 1) + D)
    return nd


def _stage(c, g, M, s0, s, ref, P, nd, dt):
    """One HEVI stage: the five updated fields and the mass and theta fluxes."""
    f64 = dict(device="cuda", dtype=torch.float64)
    col = lambda a: torch.tensor(np.asarray(a), **f64)[:, None, None]  # noqa: E731
    K, sch, rd = c["kmax"], c["scheme"], 1.0 / g.dx
    cdzg = col(g.cdz)  # with ghost levels
    cdz, rfdz = cdzg[2:-2], 1.0 / col(g.fdz[2:-2])
    G = [a[2:-2] for a in M["G"]]
    J13, J23 = [a[2:-2] for a in M["J13"]], [a[2:-2] for a in M["J23"]]
    D, W, U, V, T = (s[k] for k in STATE)
    D0, W0, U0, V0, T0 = (s0[k] for k in STATE)
    refd = ref["REF_dens"][2:-2]
    phi = M["phi"]
    dp = P["DPRES0"] + P["RT2P"] * (T - P["REF_rhot"])
    dpe = torch.cat([P["lo"] - D[:1] * (phi[1:2] - phi[3:4]), dp, P["hi"] - D[-1:] * (phi[-2:-1] - phi[-4:-3])])

    def f2h(comp, n, off=0):
        """Weights of the upper and lower level at the faces off..off+n-1 above level KS."""
        q = (cdzg * M["G"][comp])[2 + off:3 + off + n]
        return q[:-1] / (q[1:] + q[:-1]), q[1:] / (q[1:] + q[:-1])

    # continuity
    ux, vy = U + _x(U, -1), V + _y(V, -1)
    mz = J13[XYW][:-1] * 0.25 * (ux[1:] + ux[:-1]) + J23[XYW][:-1] * 0.25 * (vy[1:] + vy[:-1]) + G[XYW][:-1] * nd[0, 0][:-1]
    mx, my = G[UYZ] * (U + nd[0, 1]), G[XVZ] * (V + nd[0, 2])
    hdiv = lambda fx, fy: (fx - _x(fx, -1)) * rd + (fy - _y(fy, -1)) * rd  # noqa: E731
    Sr = -(_dz(mz) / cdz + hdiv(mx, my)) / G[XYZ]
    # vertical momentum, explicit part
    vz = 0.5 * (W[:-2] + W[1:-1]) / D[1:-1]
    zf = lambda v: torch.cat([_low(sch, W[:1], W[1:2], W[2:3], v[:1]),  # noqa: E731
                              _face(sch, W[:-3], W[1:-2], W[2:-1], W[3:], v[1:])])
    qz = vz * zf(vz) + G[XYZ][1:-1] * nd[1, 0][1:-1]
    for mom, J in ((ux, J13), (vy, J23)):
        v = 0.5 * mom / D
        v = torch.cat([0.5 * (v[1:2] + v[:1]), v[2:-1]]) * J[XYZ][1:-1]
        qz = qz + v * zf(v)
    hf = []
    for mom, sh, comp, d in ((U, _x, UYW, 1), (V, _y, XVW, 2)):
        a, b = f2h(comp, K - 1)
        dd = 0.5 * (D + sh(D, 1))
        v = (a * mom[1:] + b * mom[:-1]) / (a * dd[1:] + b * dd[:-1])
        w = W[:-1]
        hf.append(G[comp][:-1] * (v * _face(sch, sh(w, -1), w, sh(w, 1), sh(w, 2), v) + nd[1, d][:-1]))
    Sw = -(_dz(qz) * rfdz + hdiv(*hf)) / G[XYW][:-1] - col(g.wdamp[2:-3]) * W0[:-1]
    # theta
    th = T / D
    tz = mz * _zface(sch, th, mz) + G[XYW][:-1] * nd[4, 0][:-1]
    tx = mx * _face(sch, _x(th, -1), th, _x(th, 1), _x(th, 2), mx) + G[UYZ] * nd[4, 1]
    ty = my * _face(sch, _y(th, -1), th, _y(th, 1), _y(th, 2), my) + G[XVZ] * nd[4, 2]
    St = -(_dz(tz) / cdz + hdiv(tx, ty)) / G[XYZ]
    # implicit vertical solve
    pt = _zface(sch, th, W[:-1])
    A = dt * dt * P["RT2P"] / cdz / G[XYZ]
    B = GRAV * dt * dt / (cdz[1:] + cdz[:-1])
    gw = G[XYW][:-1]
    F1 = -(pt[1:] * rfdz[:-1] * A[1:-1] + B[:-1]) / gw[:-1]
    F2 = 1.0 + pt * rfdz * (A[1:] + A[:-1]) / gw
    F3 = -(pt[:-1] * rfdz[1:] * A[1:-1] - B[1:]) / gw[1:]
    a, b = f2h(XYZ, K - 1)
    e1, r1 = dp + P["RT2P"] * dt * St, D - refd + Sr * dt
    C = W[:-1] + dt * (-(e1[1:] - e1[:-1]) * rfdz / gw - GRAV * (a * r1[1:] + b * r1[:-1]) + Sw)
    e, f = [], []
    for k in range(K - 1):
        den = F2[k] if k == 0 else F2[k] + F3[k - 1] * e[-1]
        rhs = C[k] if k == 0 else C[k] - F3[k - 1] * f[-1]
        if k < K - 2:
            e.append(-F1[k] / den)
        f.append(rhs / den)
    sol = [f[-1]]
    for k in range(K - 3, -1, -1):
        sol.append(e[k] * sol[-1] + f[k])
    C = torch.stack(sol[::-1])
    out = {"DENS": D0 + dt * (-_dz(C) / cdz / G[XYZ] + Sr), "RHOT": T0 + dt * (-_dz(C * pt) / cdz / G[XYZ] + St),
           "MOMZ": torch.cat([W0[:-1] + (C - W[:-1]), torch.zeros_like(W[:1])])}
    # horizontal momentum, x then y
    for name, m, m0, o, so, sn, v, zc, hc, J, Jo, jw, cf in (
            ("MOMX", U, U0, V, _x, _y, 2, UYW, UYZ, J13, J23, M["J13"], 0.25 * g.f0),
            ("MOMY", V, V0, U, _y, _x, 3, XVW, XVZ, J23, J13, M["J23"], -0.25 * g.f0)):
        own, oth = (1, 2) if v == 2 else (2, 1)
        dd = 0.5 * (D + so(D, 1))
        a, b = f2h(zc, K - 1)
        vel = 0.5 * (W + so(W, 1))[:-1] / (a * dd[1:] + b * dd[:-1])
        qz = vel * _zface(sch, m, vel) + G[zc][:-1] * nd[v, 0][:-1]
        a, b = f2h(hc, K - 1)
        den = a * dd[1:] + b * dd[:-1]
        o4 = 0.25 * (o + so(o, 1) + sn(o, -1) + so(sn(o, -1), 1))
        for q, jj in ((m, J), (o4, Jo)):
            vel = (a * q[1:] + b * q[:-1]) / den * jj[zc][:-1]
            qz = qz + vel * _zface(sch, m, vel)
        vel = 0.5 * (m + so(m, -1)) / D
        qo = G[XYZ] * (vel * _face(sch, so(m, -2), so(m, -1), m, so(m, 1), vel) + nd[v, own])
        vel = 0.5 * (o + so(o, 1)) / (0.25 * (D + so(D, 1) + sn(D, 1) + so(sn(D, 1), 1)))
        qn = G[UVZ] * (vel * _face(sch, sn(m, -1), m, sn(m, 1), sn(m, 2), vel) + nd[v, oth])
        adv = -_dz(qz) / cdz - ((so(qo, 1) - qo) * rd + (qn - sn(qn, -1)) * rd)
        gp = G[XYZ] * dp
        d2 = 0.5 * (so(dpe, 1) + dpe)
        a, b = f2h(hc, K)
        a2, b2 = (a, b) if v == 2 else f2h(hc, K, -1)  # the lower face's weights: as the reference has them
        pg = (so(gp, 1) - gp) * rd + (jw[zc][2:-2] * (a * d2[2:] + b * d2[1:-1])
                                      - jw[zc][1:-3] * (a2 * d2[1:-1] + b2 * d2[:-2])) / cdz
        out[name] = m0 + dt * ((adv - pg) / G[hc] + cf * 4.0 * o4)
    top = torch.zeros_like(W[:1])
    return out, [torch.cat([mz + C, top]), mx, my], [torch.cat([tz + C * pt, top]), tx, ty]


def _short_step(c, g, M, st, ref, P):
    """RK4 short step: the state, and the mass and theta fluxes averaged over the stages."""
    nd = _filter(c, g, st, ref, g.dt)
    r, mf, tf, s = [], None, None, st
    for q, (dt, w) in enumerate(((g.dt / 2, 1.0), (g.dt / 2, 2.0), (g.dt, 2.0), (g.dt, 1.0))):
        s, m, t = _stage(c, g, M, st, s, ref, P, nd, dt)
        r.append(s)
        mf = [w * a for a in m] if mf is None else [a + w * b for a, b in zip(mf, m)]
        tf = [w * a for a in t] if tf is None else [a + w * b for a, b in zip(tf, t)]
    new = {k: (2.0 * r[0][k] + 4.0 * r[1][k] + 2.0 * r[2][k] + r[3][k] - 3.0 * st[k]) / 6.0 for k in STATE}
    return new, [a / 6.0 for a in mf], [a / 6.0 for a in tf]


def _fct_weights(rw, ru, rv):
    """Weights of the 14 upstream points along the wind."""
    h = lambda v: _sign(v, 0.5)  # noqa: E731
    ugev, ugew, vgew = (h(a.abs() - b.abs()) + 0.5 for a, b in ((ru, rv), (ru, rw), (rv, rw)))
    uz, vz, wz = (h(a.abs() - EPS) - 0.5 for a in (ru, rv, rw))
    suv, suw, svw = h(ru * rv) + 0.5, h(ru * rw) + 0.5, h(rv * rw) + 0.5
    wu, vu = (rw / (ru + uz) * (1.0 + uz)).abs(), (rv / (ru + uz) * (1.0 + uz)).abs()
    uv, wv = (ru / (rv + vz) * (1.0 + vz)).abs(), (rw / (rv + vz) * (1.0 + vz)).abs()
    uw, vw = (ru / (rw + wz) * (1.0 + wz)).abs(), (rv / (rw + wz) * (1.0 + wz)).abs()
    um, vm = ugev * ugew * (1.0 + uz), (1.0 - ugev) * vgew
    wm = 1.0 - ugev * ugew - vm
    c3 = um * vu * wu + vm * uv * wv + wm * uw * vw
    cuw = (1.0 - vm) * (ugew * wu * (1.0 - vu) + (1.0 - ugew) * uw * (1.0 - vw))
    cvw = (1.0 - um) * (vgew * wv * (1.0 - uv) + (1.0 - vgew) * vw * (1.0 - uw))
    cuv = (1.0 - wm) * (ugev * vu * (1.0 - wu) + (1.0 - ugev) * uv * (1.0 - wv))
    nuv, nuw, nvw = 1.0 - suv, 1.0 - suw, 1.0 - svw
    return {(0, 0, 0): -ugev * ugew * uz, (1, 0, 0): wm * (1.0 - uw) * (1.0 - vw), (0, 1, 0): um * (1.0 - vu) * (1.0 - wu),
            (0, 0, 1): vm * (1.0 - uv) * (1.0 - wv), (1, 1, 1): suv * suw * c3, (1, -1, 1): nuv * nuw * c3,
            (1, 1, -1): nuv * suw * c3, (1, -1, -1): suv * nuw * c3, (1, 1, 0): suw * cuw, (1, -1, 0): nuw * cuw,
            (1, 0, 1): svw * cvw, (1, 0, -1): nvw * cvw, (0, 1, 1): suv * cuv, (0, 1, -1): nuv * cuv}


def _tracer_stage(c, g, M, q, q0, D0, D, mf, dt, fct):
    """One tracer stage with (fct) or without the flux limiter."""
    col = torch.tensor(g.cdz[2:-2], device="cuda", dtype=torch.float64)[:, None, None]
    G, rd, sch = M["G"][XYZ][2:-2], 1.0 / g.dx, c["tracer_scheme"]
    mz, mx, my = mf[0][:-1], mf[1], mf[2]
    hz = mz * _zface(sch, q, mz)
    hx = mx * _face(sch, _x(q, -1), q, _x(q, 1), _x(q, 2), mx)
    hy = my * _face(sch, _y(q, -1), q, _y(q, 1), _y(q, 2), my)
    div = lambda z, x, y: (_dz(z) / col + (x - _x(x, -1)) * rd + (y - _y(y, -1)) * rd) / G  # noqa: E731
    if fct:
        up = lambda a, b, v: 0.5 * v * (a + b) - 0.5 * v.abs() * (b - a)  # noqa: E731
        lz, lx, ly = up(q0[:-1], q0[1:], mz), up(q0, _x(q0, 1), mx), up(q0, _y(q0, 1), my)
        az, ax, ay = hz - lz, hx - lx, hy - ly
        lo = (q0 * D0 - dt * div(lz, lx, ly)) / D
        zero = torch.zeros_like(q[:1])
        zb, zt = torch.cat([zero, az]), torch.cat([az, zero])  # lower and upper face of each cell
        pos, neg = (lambda a: a.clamp(min=0.0)), (lambda a: a.clamp(max=0.0))  # noqa: E731
        pp = dt * ((pos(zb) - neg(zt)) / col + (pos(_x(ax, -1)) - neg(ax)) * rd + (pos(_y(ay, -1)) - neg(ay)) * rd) / G
        pm = dt * ((pos(zt) - neg(zb)) / col + (pos(ax) - neg(_x(ax, -1))) * rd + (pos(ay) - neg(_y(ay, -1))) * rd) / G
        sz = torch.cat([mz[:1], mz[1:] + mz[:-1], mz[-1:]]) / col
        wt = _fct_weights(sz, (mx + _x(mx, -1)) * rd, (my + _y(my, -1)) * rd)
        big, small = torch.maximum(q0, lo), torch.minimum(q0, lo)
        for p in (q0, lo):
            above, below = torch.cat([p[1:], p[-1:]]), torch.cat([p[:1], p[:-1]])
            qa, qb = 0.0, 0.0
            for (k, i, j), w in wt.items():
                qa = qa + w * _y(_x(above if k else p, i), j)
                # the mirrored point; two of the fourteen weights look at y-1 on both sides, as in the reference
                bj = j if (k, i, j) in ((0, 1, -1), (1, 0, -1)) else -j
                qb = qb + w * _y(_x(below if k else p, -i), bj)
            big, small = torch.maximum(big, torch.maximum(qa, qb)), torch.minimum(small, torch.minimum(qa, qb))
        def ratio(room, p):
            z = 0.5 - _sign(p - EPS, 0.5)
            return (room * D * (1.0 - z) / (p - z)).clamp(max=1.0)
        rp, rm = ratio(big - lo, pp), ratio(lo - small, pm)
        def limit(a, rp1, rm1, rp0, rm0):
            d = 0.5 + _sign(a, 0.5)
            return a * (torch.minimum(rp1, rm0) * d + torch.minimum(rp0, rm1) * (1.0 - d)) - a
        hz = hz + limit(az, rp[1:], rm[1:], rp[:-1], rm[:-1])
        hx = hx + limit(ax, _x(rp, 1), _x(rm, 1), rp, rm)
        hy = hy + limit(ay, _y(rp, 1), _y(rm, 1), rp, rm)
    return (q0 * D0 - dt * div(hz, hx, hy)) / D


def _large_step(c, g, M, st, ref, tr):
    P = _prep(c, g, st, ref)
    new, mf, tf = _short_step(c, g, M, st, ref, P)
    D0, D = st["DENS"], new["DENS"]
    qs = []
    for q0 in tr:
        q = _tracer_stage(c, g, M, q0, q0, D0, D0 + (D - D0) / 3.0, mf, g.dt / 3.0, False)
        q = _tracer_stage(c, g, M, q, q0, D0, D0 + (D - D0) * 0.5, mf, g.dt / 2.0, False)
        qs.append(_tracer_stage(c, g, M, q, q0, D0, D, mf, g.dt, c["fct"]))
    return new, mf, tf, qs


def exact(case, seed):
    c = dict(CASE, **case)
    if c["kind"] in ("adjoint", "batch"):
        return None  # adjoints of whole arrays, each halo cell an input of its own: no plain restatement here
    if c["kind"] == "ensemble":
        return [exact(dict(m, kind="large"), seed + 1000 * q) for q, m in enumerate(_members(c))]
    g, st, ref, tr = _fields(c, seed)
    M = _metrics(c, g)
    if c["kind"] == "dropin":
        o, mf, tf = _stage(c, g, M, st, st, ref, _prep(c, g, st, ref), _filter(c, g, st, ref, g.dt), g.dt)
        f = lambda a: _host(torch.stack(a, 3).permute(0, 1, 2, 3))  # noqa: E731
        return dict({k + "_RK": _host(v) for k, v in o.items()}, mflx_hi=f(mf), tflx_hi=f(tf))
    if c["kind"] == "short":
        new, mf, tf = _short_step(c, g, M, st, ref, _prep(c, g, st, ref))
        qs = []
    else:
        new, mf, tf, qs = _large_step(c, g, M, st, ref, tr)
    out = {k: _halo(_ghost(v, k)) for k, v in new.items()}
    if not c["mixed"]:
        out.update(mflx_hi=torch.stack(mf), tflx_hi=torch.stack(tf))
    out.update({"QTRC%d" % q: a for q, a in enumerate(qs)})
    return out
