"""The workloads that are timed: one large time step of a forecast (or of a batch of forecasts) through the public
entry points, over the sizes, options and arithmetics the library is used with.

A pass is one `RK3.step(1)` (a batch: one `Batch.step(1)`) on domains whose state stays on the GPU, as a forecast's
time loop runs it; its outputs are the prognostic fields after the step, zero-copy views of the domain's storage.
Kinds of domain:

  igw, squall, straka   the x-z slices of the idealized runs (dry gravity waves; moist convection with Kessler; a
                        density current with second-order diffusion)
  bubble                a dry 3-D domain as the ensembles and the forecast server hold them, periodic or open
  real                  a real-data-shaped domain: terrain, hybrid coordinate, map factors, Coriolis, six moist
                        species with the positive-definite limiter, specified lateral boundaries, and at
                        convection-permitting spacing sixth-order diffusion
  ensemble              a batch of dry 3-D domains of uneven sizes, one graph per step
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from cppwrf_amd import _abi as A
from cppwrf_amd.dyn import Batch, Case, Context, Grid, RK3

STATE = {"u": A.MI_U, "v": A.MI_V, "w": A.MI_W, "t": A.MI_T, "ph": A.MI_PH, "mu": A.MI_MU, "p": A.MI_P, "al": A.MI_AL}
G, RD, T0, P0 = 9.81, 287.0, 300.0, 1.0e5
CP = 3.5 * RD
CPOVCV = CP / (CP - RD)
BW = A.MI_SPEC_BDY_WIDTH
SPECIES = (1.0, 0.05, 0.02, 0.01, 0.01, 0.005)  # qv, then cloud, rain, ice, snow, graupel as fractions of it


def listed():
    return [
        # the smallest calls: x-z slices, where launches and latency are all there is
        {"name": "igw 300x10 f64", "kind": "igw", "nx": 300, "nz": 10, "f32": False},
        {"name": "squall 120x40 f64", "kind": "squall", "nx": 120, "nz": 40, "f32": False},
        {"name": "straka 512x64 f64", "kind": "straka", "nx": 512, "nz": 64, "f32": False},
        # one small 3-D forecast, the size the examples and the smoke runs use
        {"name": "bubble 64x64x40 f32", "kind": "bubble", "nx": 64, "ny": 64, "nz": 40, "dx": 1000.0, "open": False, "f32": True},
        # one forecast with radiative boundaries, odd sizes
        {"name": "bubble 97x75x35 open f64", "kind": "bubble", "nx": 97, "ny": 75, "nz": 35, "dx": 3000.0, "open": True,
         "f32": False},
        # one request of the forecast server, in its usual arithmetic
        {"name": "bubble 219x173x44 f32", "kind": "bubble", "nx": 219, "ny": 173, "nz": 44, "dx": 6000.0, "open": False,
         "f32": True},
        # an ensemble of uneven members advanced together, in both arithmetics
        {"name": "ensemble 8 f32", "kind": "ensemble", "members": 8, "sizes": 2024, "f32": True},
        {"name": "ensemble 8 f64", "kind": "ensemble", "members": 8, "sizes": 2024, "f32": False},
        # the regional real-data domain at 15 km
        {"name": "real 119x89x44 f32", "kind": "real", "nx": 119, "ny": 89, "nz": 44, "dx": 15000.0, "f32": True},
        {"name": "real 119x89x44 f64", "kind": "real", "nx": 119, "ny": 89, "nz": 44, "dx": 15000.0, "f32": False},
        # the large convection-permitting real-data domain at 3 km
        {"name": "real 425x300x50 f32", "kind": "real", "nx": 425, "ny": 300, "nz": 50, "dx": 3000.0, "f32": True},
        {"name": "real 425x300x50 f64", "kind": "real", "nx": 425, "ny": 300, "nz": 50, "dx": 3000.0, "f32": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    f32 = rng.random() < 0.6
    kind = rng.choice(["igw", "squall", "straka", "bubble", "bubble", "bubble", "real", "real", "real", "ensemble"])
    if kind == "igw":
        return {"kind": kind, "nx": _log_int(rng, 100, 1000), "nz": _log_int(rng, 10, 100), "f32": f32}
    if kind == "squall":
        return {"kind": kind, "nx": rng.randint(80, 240), "nz": rng.randint(36, 60), "f32": f32}
    if kind == "straka":
        return {"kind": kind, "nx": rng.randint(256, 520), "nz": rng.randint(32, 64), "f32": f32}
    if kind == "bubble":
        return {"kind": kind, "nx": rng.randint(50, 300), "ny": rng.randint(50, 300), "nz": rng.randint(30, 60),
                "dx": round(rng.uniform(3000.0, 15000.0), 1), "open": rng.random() < 0.25, "f32": f32}
    if kind == "real":
        nx, ny = _log_int(rng, 60, 424), _log_int(rng, 60, 299)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": rng.randint(35, 50), "dx": rng.choice([3000.0, 9000.0, 15000.0]),
                "f32": f32}
    return {"kind": kind, "members": rng.randint(2, 8), "sizes": rng.randrange(1 << 20), "f32": f32}


# ------------------------------------------------------------------------------------------------ the cases' setups
def _sizes(case):
    """(nx, ny, nz, dx) of every domain of a case"""
    k = case["kind"]
    if k == "ensemble":  # nx 60-220, ny 60-180, nz 35/44/50, dx 3-15 km
        rng = np.random.default_rng(case["sizes"])
        out = []
        for _ in range(case["members"]):
            nx, ny = int(rng.integers(60, 221)), int(rng.integers(60, 181))
            out.append((nx, ny, int(rng.choice([35, 44, 50])), float(rng.uniform(3000.0, 15000.0))))
        return out
    if k in ("bubble", "real"):
        return [(case["nx"], case["ny"], case["nz"], case["dx"])]
    return [(case["nx"], 1, case["nz"], {"straka": 100.0}.get(k, 1000.0))]


def _options(case, dx):
    """the parameters of a domain, keywords of Case.params / default_params"""
    k = case["kind"]
    kw = {"precision": A.MI_FP32_BULK if case["f32"] else A.MI_FP64}
    if k == "squall":
        kw.update(n_moist=3, n_scalars=3, mp_physics=1)
    elif k == "straka":
        kw.update(diff_opt=1, khdif=75.0, kvdif=75.0, pr_inv=1.0)
    elif k in ("bubble", "ensemble"):
        kw.update(time_step_sound=6, damp_opt=3, zdamp=5000.0)
    elif k == "real":
        kw.update(time_step_sound=6 if dx < 5000.0 else 4, damp_opt=3, zdamp=5000.0, dampcoef=0.2, n_moist=6, n_scalars=6,
                  moist_adv_opt=1, terrain=1, mapped=1, coriolis=1)
        if dx < 5000.0:
            kw.update(diff_6th_opt=1, diff_6th_factor=0.12)
    return kw


def _idealized(case, q, seed):
    """domain q of an idealized case: (Case, {name: initial field}), the fields perturbed from the seed"""
    nx, ny, nz, dx = _sizes(case)[q]
    k = case["kind"]
    if k == "igw":
        c = Case(A.MI_CASE_IGW, Grid(nx, 1, nz, 1000.0, 1000.0, 6.0), 10000.0)
    elif k == "squall":
        c = Case.squall2d(nx, nz)
    elif k == "straka":
        c = Case.straka(nx, nz)
    else:
        bc = A.MI_BC_OPEN if case.get("open") else A.MI_BC_PERIODIC
        c = Case.bubble3d(nx, ny, nz, dx=dx, ztop=20000.0, dt=6.0 * dx / 1000.0, seed=seed + 7919 * q, noise_amp=0.05, bc=bc)
    rng = np.random.default_rng([seed, q])
    fields = {n: c.field(f) for n, f in STATE.items()}
    amp_t, amp_u = (0.5, 1.0) if k in ("bubble", "ensemble") else (0.02, 0.1)  # as the ensemble's members; less for slices
    fields["t"] += rng.uniform(-amp_t, amp_t, size=fields["t"].shape)
    du = rng.uniform(-amp_u, amp_u, size=fields["u"].shape)
    du[..., -1] = du[..., 0]  # the periodic face
    fields["u"] += du
    if ny > 1:
        dv = rng.uniform(-amp_u, amp_u, size=fields["v"].shape)
        dv[:, -1] = dv[:, 0]
        fields["v"] += dv
    if case["f32"]:  # the values the domain stores (mu stays in 64 bits)
        fields = {n: f if n == "mu" else f.astype(np.float32).astype(np.float64) for n, f in fields.items()}
    return c, fields


class _Span:
    """a strided window of a domain's device memory for torch.as_tensor; the tensor keeps it, and so the domain, alive"""

    def __init__(self, owner, addr, shape, strides, f32):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (addr, False), "shape": shape, "strides": strides,
                                         "typestr": "<f4" if f32 else "<f8", "version": 2}


def _view(rk, fid, halo=0):
    """a field of a domain as a tensor over its storage, (levels, rows, points), `halo` halo points on each side"""
    v = rk.field_view(fid)
    e, hy = v.elem_bytes, halo if v.ny > 1 else 0
    shape = (v.nz, v.ny + 2 * hy, v.nx + 2 * halo)
    strides = (v.stride_k * e, v.stride_j * e, e)
    return torch.as_tensor(_Span(rk, v.data - (hy * v.stride_j + halo) * e, shape, strides, e == 4), device="cuda")


def _bind(rk, fid, values):
    """a field initialised from a tensor, in a buffer that the caller owns (returned)"""
    lay = rk.field_layout(fid)
    buf = torch.zeros(lay.alloc_elems, dtype=torch.float32 if lay.elem_bytes == 4 else torch.float64, device="cuda")
    buf.as_strided((lay.nz, lay.ny, lay.nx), (lay.stride_k, lay.stride_j, 1), lay.offset).copy_(values)
    torch.cuda.synchronize()
    rk.bind(fid, buf.data_ptr(), buf.numel() * buf.element_size())
    return buf


# US standard atmosphere up to 32 km: pressure at a height, height at a pressure, temperature
_LAYERS = ((0.0, 288.15, -0.0065), (11000.0, 216.65, 0.0), (20000.0, 216.65, 0.001))


def _std_tables():
    out, p = [], 101325.0
    for n, (z0, t0, lapse) in enumerate(_LAYERS):
        out.append((z0, t0, lapse, p))
        if n + 1 < len(_LAYERS):
            dz = _LAYERS[n + 1][0] - z0
            p *= math.exp(-9.80665 * dz / (287.053 * t0)) if lapse == 0 else ((t0 + lapse * dz) / t0) ** (-9.80665 / (287.053 * lapse))
    return out


def _std_p(z):
    out = torch.zeros_like(z)
    for z0, t0, lapse, p0 in _std_tables():
        dz = z - z0
        p = p0 * torch.exp(-9.80665 * dz / (287.053 * t0)) if lapse == 0 else p0 * ((t0 + lapse * dz) / t0).clamp(min=0.1) ** (-9.80665 / (287.053 * lapse))
        out = torch.where(z >= z0, p, out)
    return out


def _std_z(p):
    out = torch.zeros_like(p)
    for z0, t0, lapse, p0 in _std_tables():
        r = p / p0
        z = z0 - 287.053 * t0 / 9.80665 * torch.log(r) if lapse == 0 else z0 + t0 / lapse * (r ** (-287.053 * lapse / 9.80665) - 1.0)
        out = torch.where((p <= p0) | (z0 == 0.0), z, out)
    return out


def _std_t(z):
    out = torch.zeros_like(z)
    for z0, t0, lapse, _ in _std_tables():
        out = torch.where((z >= z0) | (z0 == 0.0), t0 + lapse * (z - z0), out)
    return out


def _real(ctx, case, seed):
    """a real-data-shaped domain: seeded hills, standard atmosphere, jets with +-1 m/s of noise, map factors, Coriolis,
    patchy moist species, slowly drifting boundary data"""
    nx, ny, nz, dx = _sizes(case)[0]
    dt = 6.0 * dx / 1000.0
    small = Case.hills(10, 10, nz, dx=dx, dt=dt, bc=A.MI_BC_SPECIFIED)  # the level coefficients (50 hPa top, hybrid)
    lv = small.levels
    rk = RK3(ctx, Grid(nx, ny, nz, dx, dx, dt, A.MI_BC_SPECIFIED, A.MI_BC_SPECIFIED), A.default_params(**_options(case, dx)),
             levels=lv)
    f8 = dict(dtype=torch.float64, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    host = np.random.default_rng(seed)
    uni = lambda *s: 2.0 * torch.rand(*s, generator=gen, **f8) - 1.0  # noqa: E731
    co = {n: torch.tensor(np.ctypeslib.as_array(getattr(lv, n), shape=(nz + (n[-1] == "f"),)).copy(), **f8).view(-1, 1, 1)
          for n in ("c1h", "c2h", "c3h", "c4h", "c1f", "c2f", "dnw")}
    x = (torch.arange(nx, **f8) + 0.5) * dx
    y = (torch.arange(ny, **f8) + 0.5) * dx
    ht = torch.zeros(1, ny, nx, **f8)
    wide = (10000.0, 60000.0) if dx < 5000.0 else (30000.0, 150000.0)
    for _ in range(12):
        cx, cy, h, w = host.uniform(0, nx * dx), host.uniform(0, ny * dx), host.uniform(0, 2500.0), host.uniform(*wide)
        ht += h * torch.exp(-((x - cx) / w) ** 2)[None, None, :] * torch.exp(-((y - cy) / w) ** 2)[None, :, None]
    ht = 3000.0 * torch.tanh(ht / 3000.0)
    mf = lambda i, j: 1.0 + 0.05 * torch.sin(math.pi * i / nx)[None, None, :] * torch.cos(math.pi * j / ny)[None, :, None]  # noqa: E731
    im, iu = torch.arange(nx, **f8) + 0.5, torch.arange(nx + 1, **f8)
    jm, jv = torch.arange(ny, **f8) + 0.5, torch.arange(ny + 1, **f8)
    mt, mu_, mv = mf(im, jm), mf(iu, jm), mf(im, jv)
    lat = (30.0 + 20.0 * jm / ny)[None, :, None].expand(1, ny, nx) * math.pi / 180.0
    # dry hydrostatic base state, column by column; the moist initial state in theta_m
    mub = _std_p(ht) - lv.p_top
    pb = co["c3h"] * mub + co["c4h"] + lv.p_top
    z = _std_z(pb)
    tk = _std_t(z)
    tb = tk * (P0 / pb) ** (RD / CP)
    alb = RD / P0 * tb * (pb / P0) ** (-1.0 / CPOVCV)
    es = 611.2 * torch.exp(17.67 * (tk - 273.15) / (tk - 29.65))
    qv = torch.where(z < 10000.0, 0.8 - 0.7 * z / 10000.0, torch.full_like(z, 0.1)) * 0.622 * es / (pb - es)
    th = tb * (1.0 + 461.6 / RD * qv)
    al = RD / P0 * th * (pb / P0) ** (-1.0 / CPOVCV) - alb
    layer = -co["dnw"] * (co["c1h"] * mub + co["c2h"])
    up = lambda s: torch.cat([torch.zeros(1, ny, nx, **f8), torch.cumsum(s, 0)])  # noqa: E731
    phb, ph = G * ht + up(layer * alb), up(layer * al)
    jet = lambda amp: amp * torch.exp(-((z - 10000.0) / 4000.0) ** 2)  # noqa: E731
    uj, vj = jet(host.uniform(5.0, 40.0)), jet(host.uniform(5.0, 40.0))
    u = torch.cat([uj, uj[:, :, -1:]], 2) + uni(nz, ny, nx + 1)
    v = torch.cat([vj, vj[:, -1:]], 1) + uni(nz, ny + 1, nx)
    t = th - T0
    zero = torch.zeros(1, ny, nx, **f8)
    fields = {A.MI_MUB: mub, A.MI_PB: pb, A.MI_ALB: alb, A.MI_PHB: phb, A.MI_T_INIT: tb - T0, A.MI_HT: ht, A.MI_MSFTX: mt,
              A.MI_MSFTY: mt, A.MI_MSFUX: mu_, A.MI_MSFUY: mu_, A.MI_MSFVX: mv, A.MI_MSFVY: mv, A.MI_MSFVX_INV: 1.0 / mv,
              A.MI_F: 1.45842e-4 * torch.sin(lat), A.MI_E: 1.45842e-4 * torch.cos(lat), A.MI_U: u, A.MI_V: v,
              A.MI_W: torch.zeros(nz + 1, ny, nx, **f8), A.MI_T: t, A.MI_PH: ph, A.MI_MU: zero, A.MI_P: torch.zeros_like(t),
              A.MI_AL: al}
    rk.buffers = [_bind(rk, fid, a) for fid, a in fields.items()]  # as long as the domain
    q = [f * qv * (1.0 if n == 0 else torch.rand(nz, ny, nx, generator=gen, **f8) > 0.7) for n, f in enumerate(SPECIES)]
    for n, a in enumerate(q):  # halos too: the outer rows copied outward, as the lateral boundaries' fill
        _view(rk, A.MI_Q + n, 3).copy_(torch.nn.functional.pad(a[None], (3, 3, 3, 3), mode="replicate")[0])
    # boundary data: the initial outer rows, coupled, and tendencies of a slow oscillation (half a metre per second and
    # a tenth of a kelvin over a day)
    muu = torch.cat([mub[:, :, :1], 0.5 * (mub[:, :, 1:] + mub[:, :, :-1]), mub[:, :, -1:]], 2)
    muv = torch.cat([mub[:, :1], 0.5 * (mub[:, 1:] + mub[:, :-1]), mub[:, -1:]], 1)
    mass = lambda m, s: co["c1" + s] * m + co["c2" + s]  # noqa: E731
    coupled = {A.MI_BDY_U: (u, mass(muu, "h") / mu_, 0.5), A.MI_BDY_V: (v, mass(muv, "h") / mv, 0.5),
               A.MI_BDY_T: (t, mass(mub, "h"), 0.1), A.MI_BDY_PH: (ph, mass(mub, "f"), 0.0),
               A.MI_BDY_MU: (zero, torch.ones_like(zero), 0.0), A.MI_BDY_Q: (q[0], mass(mub, "h"), 0.0)}
    for var, (a, m, amp) in coupled.items():
        for side in range(4):
            def ring(b):
                b = b.flip(2) if side == A.MI_BDY_XE else b.flip(1) if side == A.MI_BDY_YE else b
                return b[:, :, :BW].permute(2, 0, 1) if side < 2 else b[:, :BW].permute(1, 0, 2)
            val = ring(a * m).contiguous()
            pos = torch.arange(val.shape[2], **f8) / val.shape[2]
            ten = amp * 2.0 * math.pi / 86400.0 * ring(m.expand_as(a)) * torch.cos(2.0 * math.pi * (pos + host.uniform()))
            rk.bdy_set(var, side, val.cpu().numpy(), ten.cpu().numpy())
    rk.calc_p_rho_phi(1)  # p from the state
    rk.sync()
    return rk


def prepare(case, seed):
    stream = torch.cuda.Stream()
    ctx = Context(0, stream=stream.cuda_stream)
    if case["kind"] == "real":
        rks = [_real(ctx, case, seed)]
    else:
        rks = []
        for q in range(len(_sizes(case))):
            c, fields = _idealized(case, q, seed)
            rk = RK3(ctx, c.grid, c.params(**_options(case, c.grid.dx)), c)
            for n, a in fields.items():
                rk.set_field(STATE[n], a)
            rks.append(rk)
    state = {"ctx": ctx, "stream": stream, "domains": rks,
             "views": [{n: _view(rk, f) for n, f in STATE.items()} for rk in rks],
             "scalars": rks[0].params.n_scalars}
    if case["kind"] == "ensemble":
        state["batch"] = Batch(ctx, rks)
    return state


def run(state):
    """one large time step; the fields after it, ordered before what the caller's stream does next"""
    if "batch" in state:
        state["batch"].step(1)
    else:
        state["domains"][0].step(1)
    torch.cuda.current_stream().wait_stream(state["stream"])
    if "batch" in state:
        return state["views"]
    out = dict(state["views"][0])
    for n in range(state["scalars"]):  # a scalar's two buffers swap at every stage
        out["q%d" % n] = _view(state["domains"][0], A.MI_Q + n)
    return out


def work(case):
    """One step reads the prognostic state, the scalars and the base state and writes the state and the scalars.  The
    operations per point: a dry RK stage about 620 (prep 40, tendencies 420, acoustic set-up 90, recoupling with a
    power 70) and an acoustic substep 190; a scalar 110 per stage and 260 more with the limiter at the last stage."""
    by = fl = 0.0
    for nx, ny, nz, dx in _sizes(case):
        kw = _options(case, dx)
        pts, e = float(nx * ny * nz), 4 if case["f32"] else 8
        n_sound = kw.get("time_step_sound") or {"igw": 4, "squall": 4, "straka": 6}[case["kind"]]
        subs, nsc = 1 + n_sound // 2 + n_sound, kw.get("n_scalars", 0)
        by += pts * (2 * (7 + nsc) * e + (32 if kw.get("terrain") else 0))
        fl += pts * (3 * 620 + 190 * subs + nsc * (3 * 110 + 260) + (100 if kw.get("diff_6th_opt") else 0))
    return {"bytes": by, "flops": fl}


# ------------------------------------------------------------------------------------------------ the step in 64 bits
def exact(case, seed):
    """The dry step over flat ground with periodic sides and constant map factors (igw, bubble, ensemble), restated in
    torch's float64 from the discrete equations of the ARW solver.  The other kinds (Kessler, diffusion, open and
    specified sides, terrain, limited scalars) have no such restatement here."""
    if case["kind"] == "ensemble":
        return [_dry_step(*_idealized(case, q, seed), True) for q in range(case["members"])]
    if case["kind"] == "igw" or (case["kind"] == "bubble" and not case["open"]):
        return _dry_step(*_idealized(case, 0, seed), case["kind"] == "bubble")
    return None


def _dry_step(c, fields, damped):
    nx, ny, nz, g = c.grid.nx, c.grid.ny, c.grid.nz, c.grid
    f8 = dict(dtype=torch.float64, device="cuda")
    lv = c.levels
    col = lambda n, m: torch.tensor(np.ctypeslib.as_array(getattr(lv, n), shape=(m,)).copy(), **f8).view(-1, 1, 1)  # noqa: E731
    dnw, rdnw, c1h, c2h = (col(n, nz) for n in ("dnw", "rdnw", "c1h", "c2h"))
    rdn, fnm, fnp, c1f, c2f = (col(n, nz + 1) for n in ("rdn", "fnm", "fnp", "c1f", "c2f"))
    fnm_, fnp_, rdn_ = fnm[1:nz], fnp[1:nz], rdn[1:nz]
    prof = lambda f: torch.tensor(c.profile(f), **f8).view(-1, 1, 1)  # noqa: E731
    pb, alb, phb, mub = prof(A.MI_PB), prof(A.MI_ALB), prof(A.MI_PHB), float(c.field(A.MI_MUB)[0, 0, 0])
    s = {n: torch.tensor(a, **f8) for n, a in fields.items()}
    u, v, w, t, ph, mu, p, al = (s[n] for n in ("u", "v", "w", "t", "ph", "mu", "p", "al"))
    u, v = u[..., :nx], v[:, :ny]
    rdx, rdy, two_d = lv.rdx, lv.rdy, ny == 1
    eps, smdiv, emdiv, dampcoef, zdamp = 0.1, 0.1, 0.01, 0.2, 5000.0
    emdx, emdy = emdiv / rdx, 0.0 if two_d else emdiv / rdy
    n_sound = 6 if damped else max(2 * (int(300.0 * g.dt / g.dx - 0.01) + 1), 4)
    zrow = torch.zeros(1, ny, nx, **f8)
    X, Y = -1, -2
    at = lambda a, d, n: torch.roll(a, -n, d) if not (two_d and d == Y) else a  # noqa: E731  the value n points on

    def flux5(q, vel, d):  # 5th-order upwind flux at the face between points -1 and 0 along d
        qs = [at(q, d, n) for n in range(-3, 3)]
        sg = torch.where(vel >= 0, 1.0, -1.0)
        return vel * ((37 * (qs[3] + qs[2]) - 8 * (qs[4] + qs[1]) + (qs[5] + qs[0])) / 60 -
                      sg * ((qs[5] - qs[0]) - 5 * (qs[4] - qs[1]) + 10 * (qs[3] - qs[2])) / 60)

    def flux3(q, vel):  # 3rd-order upwind along the levels, between levels 1 and 2 of each run of four
        a, b, e, f = q[:-3], q[1:-2], q[2:-1], q[3:]
        sg = torch.where(-vel >= 0, 1.0, -1.0)
        return vel * ((7 * (e + b) - (f + a)) / 12 + sg * ((f - a) - 3 * (e - b)) / 12)

    def vflux(q, vel):  # vertical flux of a mass-level field at levels 0..nz, vel at levels 1..nz-1
        second = vel * (fnm_ * q[1:] + fnp_ * q[:-1])
        f = second.clone()
        f[1:-1] = flux3(q, vel[1:-1])
        return torch.cat([zrow, f, zrow])

    def at_w(q):  # a mass-level field at w levels 1..nz-1
        return fnm_ * q[1:] + fnp_ * q[:-1]

    def dpn(q):  # the pressure sum of two columns at w levels 0..nz
        lo = 0.5 * (lv.cf1 * q[0] + lv.cf2 * q[1] + lv.cf3 * q[2])
        return torch.cat([lo[None], 0.5 * at_w(q), zrow])

    def pgf(d, rd, mface, ph_, alt, p_, al_, php, mu_):
        dd = lambda a: a - at(a, d, -1)  # noqa: E731
        ss = lambda a: a + at(a, d, -1)  # noqa: E731
        dn = dpn(ss(p_))
        return (0.5 * rd * (c1h * mface + c2h) * (dd(ph_[1:]) + dd(ph_[:-1]) + ss(alt) * dd(p_)) +
                rd * dd(php) * (rdnw * (dn[1:] - dn[:-1]) - 0.5 * c1h * ss(mu_)))

    u1, v1, w1, t1, ph1, mu1 = u, v, w, t, ph, mu
    mudf = zrow
    for rk in (1, 2, 3):
        dts = g.dt / 3.0 if rk == 1 else g.dt / n_sound
        ns = 1 if rk == 1 else n_sound // 2 if rk == 2 else n_sound
        # -------- the stage's coupled fields
        mut = mu + mub
        muu, muv = 0.5 * (mut + at(mut, X, -1)), 0.5 * (mut + at(mut, Y, -1))
        Mh, Mf, Mu, Mv = c1h * mut + c2h, c1f * mut + c2f, c1h * muu + c2h, c1h * muv + c2h
        ru, rv, rw, alt = u * Mu, v * Mv, w * Mf, al + alb
        full = phb + ph
        php = 0.5 * (full[1:] + full[:-1])
        dv = dnw * (rdx * (at(ru, X, 1) - ru) + rdy * (at(rv, Y, 1) - rv))
        ww = torch.cat([zrow, -torch.cumsum(dnw * c1h * dv.sum(0, keepdim=True) + dv, 0)[:-1], zrow])
        # -------- tendencies
        wi = ww[1:nz]
        rw4 = 0.5 * (rw[1:] + rw[:-1])
        fx = flux5(u, 0.5 * (ru + at(ru, X, -1)), X)
        ut = -rdx * (at(fx, X, 1) - fx)
        fy = flux5(u, 0.5 * (rv + at(rv, X, -1)), Y)
        ut = ut - rdy * (at(fy, Y, 1) - fy)
        fz = vflux(u, 0.5 * (wi + at(wi, X, -1)))
        ut = ut - rdnw * (fz[1:] - fz[:-1]) - pgf(X, rdx, muu, ph, alt, p, al, php, mu)
        ut = ut - u / 6370.0e3 * 0.5 * (rw4 + at(rw4, X, -1))
        vt = torch.zeros_like(v)
        if not two_d:
            fx = flux5(v, 0.5 * (ru + at(ru, Y, -1)), X)
            fy = flux5(v, 0.5 * (rv + at(rv, Y, -1)), Y)
            fz = vflux(v, 0.5 * (wi + at(wi, Y, -1)))
            vt = -rdx * (at(fx, X, 1) - fx) - rdy * (at(fy, Y, 1) - fy) - rdnw * (fz[1:] - fz[:-1])
            vt = vt - pgf(Y, rdy, muv, ph, alt, p, al, php, mu) - v / 6370.0e3 * 0.5 * (rw4 + at(rw4, Y, -1))
        up = lambda r: torch.cat([at_w(r), (2 - fnm[nz - 1]) * r[-1:] - fnp[nz - 1] * r[-2:-1]])  # noqa: E731  w levels 1..nz
        fx, fy = flux5(w[1:], up(ru), X), flux5(w[1:], up(rv), Y)
        wt = -rdx * (at(fx, X, 1) - fx) - rdy * (at(fy, Y, 1) - fy)
        wm = 0.5 * (ww[1:] + ww[:-1])
        fz = wm * 0.5 * (w[1:] + w[:-1])
        fz[1:-1] = flux3(w, wm[1:-1])
        wt[:-1] += -rdn_ * (fz[1:] - fz[:-1]) + G * (rdn_ * (p[1:] - p[:-1]) - c1f[1:nz] * mu)
        mid = lambda a, d: 0.5 * at_w(a + at(a, d, 1))  # noqa: E731
        wt[:-1] += (mid(ru, X) * mid(u, X) + mid(rv, Y) * mid(v, Y)) / 6370.0e3
        wt[-1:] += 2 * rdn[nz - 1] * fz[-1:] + G * (-2 * rdnw[nz - 1] * p[-1:] - c1f[nz] * mu)
        fx, fy, fz = flux5(t, ru, X), flux5(t, rv, Y), vflux(t, wi)
        tt = -rdx * (at(fx, X, 1) - fx) - rdy * (at(fy, Y, 1) - fy) - rdnw * (fz[1:] - fz[:-1])
        wd = wm * rdnw * (full[1:] - full[:-1])
        pt = torch.cat([-at_w(wd), zrow]) + Mf[1:] * G * w[1:]
        for d, rd, m, q in ((Y, rdy, muv, v), (X, rdx, muu, u)):
            vel = torch.cat([0.25 * (q[1:] + q[:-1]), 0.5 * (lv.cfn * q[-1:] + lv.cfn1 * q[-2:-1])]) * (c1f[1:] * m + c2f[1:])
            gr = 45 * (at(ph, d, 1) - at(ph, d, -1)) - 9 * (at(ph, d, 2) - at(ph, d, -2)) + at(ph, d, 3) - at(ph, d, -3)
            pt = pt - rd * (vel + at(vel, d, 1)) * gr[1:] / 60
        # -------- the acoustic steps' variables and coefficients
        mts = mub + mu1
        us, vs, ws, ts, phs, mus, ww1 = u, v, w, t, ph, mu, ww
        mfu, mfv = (muu, muv) if rk == 1 else (0.5 * (mts + at(mts, X, -1)), 0.5 * (mts + at(mts, Y, -1)))
        ucs, vcs = Mu * us, Mv * vs
        u, v = (c1h * mfu + c2h) * u1 - ucs, (c1h * mfv + c2h) * v1 - vcs
        w, t, ph, mu = (c1f * mts + c2f) * w1 - Mf * ws, (c1h * mts + c2h) * t1 - Mh * ts, ph1 - phs, mu1 - mus
        muts = mts
        c2a = CPOVCV * (pb + p) / alt

        def p_rho():
            m = c1h * muts + c2h
            a = -(alt * c1h * mu + rdnw * (ph[1:] - ph[:-1])) / m
            return c2a * (alt * (t - c1h * mu * ts) / (m * (T0 + ts)) - a), a

        p, al = p_rho()
        pm1 = p
        cof = (0.5 * dts * G * (1 + eps)) ** 2
        a_, b_, c_ = (torch.zeros(nz + 1, ny, nx, **f8) for _ in range(3))
        a_[2:nz] = -cof * rdn[2:nz] * rdnw[1:nz - 1] * c2a[1:-1] / (Mh[1:-1] * Mf[1:nz - 1])
        a_[nz] = (-2 * cof * rdnw[-1] ** 2 * c2a[-1] / (Mh[-1] * Mf[nz - 1]))
        b_[1:nz] = 1 + cof * rdn_ * (rdnw[1:] * c2a[1:] / (Mh[1:] * Mf[1:nz]) + rdnw[:-1] * c2a[:-1] / (Mh[:-1] * Mf[1:nz]))
        b_[nz] = 1 + 2 * cof * rdnw[-1] ** 2 * c2a[-1] / (Mh[-1] * Mf[nz])
        c_[1:nz] = -cof * rdn_ * rdnw[1:] * c2a[1:] / (Mh[1:] * Mf[2:])
        alpha, gamma = torch.zeros_like(a_), torch.zeros_like(a_)
        for k in range(1, nz + 1):
            alpha[k] = 1 / (b_[k] - a_[k] * gamma[k - 1])
            gamma[k] = c_[k] * alpha[k]
        damp = torch.zeros_like(w)
        if damped:
            hgt = (phs + phb) / G
            over = hgt - (hgt[-1:] - zdamp)
            damp = torch.where(over >= 0, dts * dampcoef * torch.sin(0.5 * math.pi * over / zdamp) ** 2, damp)
            damp[0] = 0
        if rk == 1:
            mudf = zrow
        cw = c2a * rdnw / Mh
        for it in range(1, ns + 1):
            du = ut * dts - dts * pgf(X, rdx, muu, ph, alt, p, al, php, mu) - c1h * emdx * (mudf - at(mudf, X, -1))
            if not two_d:
                v = v + dts * vt - dts * pgf(Y, rdy, muv, ph, alt, p, al, php, mu) - c1h * emdy * (mudf - at(mudf, Y, -1))
            u = u + du
            dv = rdx * (at(u + ucs, X, 1) - (u + ucs)) + rdy * (at(v + vcs, Y, 1) - (v + vcs))
            mudf = (dnw * dv).sum(0, keepdim=True)
            old, mu = mu, mu + dts * mudf
            muts = mut + mu
            ave = 0.5 * ((1 + eps) * mu + (1 - eps) * old)
            ww = torch.cat([zrow, -torch.cumsum(dnw * (c1h * mudf + dv), 0)[:-1] - ww1[1:nz], zrow])
            wdt = torch.cat([zrow, ww[1:nz] * at_w(ts), zrow])
            hf = 0.5 * rdx * (at(u, X, 1) * (at(ts, X, 1) + ts) - u * (ts + at(ts, X, -1)))
            hf = hf + 0.5 * rdy * (at(v, Y, 1) * (at(ts, Y, 1) + ts) - v * (ts + at(ts, Y, -1)))
            old_t, t = t, t + dts * tt - dts * (hf + rdnw * (wdt[1:] - wdt[:-1]))
            tav = (0.5 * ((1 + eps) * t + (1 - eps) * old_t) + c1h * ave * T0) / ((c1h * muts + c2h) * (T0 + ts))
            wdn = 0.5 * (ww[1:] + ww[:-1]) * rdnw * ((phs + phb)[1:] - (phs + phb)[:-1])
            rr = dts * (pt + 0.5 * G * (1 - eps) * w[1:])
            rr[:-1] -= dts * at_w(wdn)
            R = torch.cat([zrow, ph[1:] + rr / Mf[1:]])
            dph = (1 + eps) * (R[1:] - R[:-1]) + (1 - eps) * (ph[1:] - ph[:-1])
            we = w + torch.cat([zrow, dts * wt])
            we[1:nz] += 0.5 * dts * G * rdn_ * (cw[1:] * dph[1:] - cw[:-1] * dph[:-1])
            ca = c2a * alt * tav
            we[1:nz] += dts * G * (rdn_ * (ca[1:] - ca[:-1]) - c1f[1:nz] * ave)
            we[nz:] += -dts * G * rdnw[-1] ** 2 * c2a[-1:] / Mh[-1:] * dph[-1:] - dts * G * (2 * rdnw[-1] * ca[-1:] + c1f[nz] * ave)
            we[0] = 0
            for k in range(1, nz + 1):
                we[k] = (we[k] - a_[k] * we[k - 1]) * alpha[k]
            for k in range(nz - 1, 0, -1):
                we[k] = we[k] - gamma[k] * we[k + 1]
            w = (we - damp * Mf * ws) / (1 + damp)
            ph = torch.cat([ph[:1], R[1:] + 0.5 * dts * G * (1 + eps) * w[1:] / (c1f * muts + c2f)[1:]])
            pn, al = p_rho()
            p, pm1 = pn + smdiv * (pn - pm1), pn
        # -------- back to the full fields
        mfu, mfv = 0.5 * (muts + at(muts, X, -1)), 0.5 * (muts + at(muts, Y, -1))
        u, v = (u + ucs) / (c1h * mfu + c2h), (v + vcs) / (c1h * mfv + c2h)
        w, t = (w + ws * Mf) / (c1f * muts + c2f), (t + ts * Mh) / (c1h * muts + c2h)
        ph, mu = ph + phs, mu + mus
        al = -(alb * c1h * mu + rdnw * (ph[1:] - ph[:-1])) / (c1h * muts + c2h)
        p = P0 * (RD * (T0 + t) / (P0 * (al + alb))) ** CPOVCV - pb
    u = torch.cat([u, u[..., :1]], -1)
    if not two_d:
        v = torch.cat([v, v[:, :1]], -2)
    return {"u": u, "v": v, "w": w, "t": t, "ph": ph, "mu": mu, "p": p, "al": al}
