"""What the stepper is timed on: the calls a user's program makes, over the range of sizes and
options it makes them with.

Five kinds of pass:

``run``      one whole simulation through ``openem_amd.run``: tables, upload, stepping, readout
             (a sweep of small simulations is many of these: launches and set-up count);
``step``     ``Stepper.run`` on a scene resident on the GPU, then the monitors and the energies
             (what a long simulation of a large scene spends its time on);
``pool``     a batch of small scenes stepped together by the serving pool, each set up, read out
             and released;
``grad``     one inverse-design gradient through ``overlap_power_gradient``;
``segment``  one checkpointed segment of a gradient on a resident scene: reload, recompute with
             the design recorded, step the adjoint back, read the gradient.

The media are those of the package's scene builders: the seeded box soup (PML on all faces,
2-pole Lorentz boxes, a dipole), the Lorentz sphere, the plane-wave slab, a graded index with a
value of its own in every cell, the Bloch unit cell with metal cylinders, and the waveguide bend
with a design region.  Every number is formed here with numpy; the package receives it as a
``Scene``, and :func:`exact` steps the same numbers in float64 with torch.
"""

from __future__ import annotations

import numpy as np
import torch

import openem_amd
from openem_amd import _lib, adjoint, cpml, grid, model, serving, solver, tables, waveform

EPS0, MU0, ETA0, C0 = 8.8541878128e-12, 1.25663706212e-6, 376.7303136668535, 299792458.0

#: passes a resident scene's step tables cover (a pass continues where the last one ended)
RESIDENT_PASSES = 400


def listed():
    return [
        # the smallest: a periodic slab transmission, launches and set-up dominate
        dict(name="run_slab_30x30x174", kind="run", medium="slab", nx=30, ny=30, nz=174,
             steps=2000, nf=11),
        # a small dispersive simulation, 64 cells a side
        dict(name="run_soup_64", kind="run", medium="soup", nx=64, ny=64, nz=64, steps=1500, nf=9),
        # odd sides, graded z spacing, field-time probes
        dict(name="run_sphere_97x89x103", kind="run", medium="sphere", nx=97, ny=89, nz=103,
             steps=1200, nf=5),
        # oblique incidence on a small Bloch cell with metal: complex fields, TF/SF faces
        dict(name="run_bloch_tfsf_64x64x200", kind="run", medium="cell", nx=64, ny=64, nz=200,
             steps=800, nf=7, tfsf=True),
        # ordinary resident scenes: below and above where one scene fills the GPU
        dict(name="step_soup_160", kind="step", medium="soup", nx=160, ny=160, nz=160, steps=512,
             nf=5),
        dict(name="step_graded_150x133x141", kind="step", medium="graded", nx=150, ny=133, nz=141,
             steps=512, nf=5),
        dict(name="step_soup_250x230x210", kind="step", medium="soup", nx=250, ny=230, nz=210,
             steps=192, nf=3),
        # the largest resident scenes, complex and real fields
        dict(name="step_bloch_192x192x480", kind="step", medium="cell", nx=192, ny=192, nz=480,
             steps=128, nf=2, tfsf=False),
        dict(name="step_soup_512", kind="step", medium="soup", nx=512, ny=512, nz=512, steps=64,
             nf=1),
        # a serving batch of ten scenes of mixed kinds and sides
        dict(name="pool_10x64-144", kind="pool", medium="mixed", scenes=10, side_lo=64,
             side_hi=144, steps=600, nf=7),
        # inverse design on a bend: a whole small gradient, a segment of a large one
        dict(name="grad_bend_120x120x44", kind="grad", medium="bend", nx=120, ny=120, nz=44,
             steps=1000, nf=1, design=48),
        dict(name="segment_bend_400x400x48", kind="segment", medium="bend", nx=400, ny=400, nz=48,
             steps=64, nf=1, design=160),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["run", "run", "step", "step", "step", "pool", "grad", "segment"])
    if kind == "run":
        medium = rng.choice(["slab", "soup", "sphere", "cell"])
        if medium == "slab":
            s = dict(nx=side(8, 64), ny=side(8, 64), nz=side(100, 260))
        elif medium == "cell":
            s = dict(nx=side(40, 72), ny=side(40, 72), nz=side(120, 220), tfsf=True)
        else:
            s = dict(nx=side(56, 112), ny=side(56, 112), nz=side(56, 112))
        return dict(kind=kind, medium=medium, steps=rng.randint(500, 1200), nf=rng.randint(3, 11),
                    **s)
    if kind == "step":
        medium = rng.choice(["soup", "soup", "sphere", "graded", "cell"])
        if medium == "graded":
            s = dict(nx=side(96, 176), ny=side(96, 176), nz=side(96, 176))
        elif medium == "cell":
            s = dict(nx=side(96, 180), ny=side(96, 180), nz=side(200, 480), tfsf=False)
        else:
            s = dict(nx=side(120, 420), ny=side(120, 300), nz=side(120, 260))
        cells = s["nx"] * s["ny"] * s["nz"]
        return dict(kind=kind, medium=medium, steps=max(64, min(512, int(2e9 // cells))),
                    nf=rng.randint(1, 4), **s)
    if kind == "pool":
        lo = side(56, 96)
        return dict(kind=kind, medium="mixed", scenes=rng.randint(4, 12), side_lo=lo,
                    side_hi=min(152, side(lo + 8, 160)), steps=rng.randint(250, 500),
                    nf=rng.randint(5, 9))
    n = side(84, 128) if kind == "grad" else side(160, 400)
    return dict(kind=kind, medium="bend", nx=n, ny=side(n, n + 24), nz=side(36, 64),
                steps=rng.randint(500, 800) if kind == "grad" else rng.randint(32, 64), nf=1,
                design=max(16, int(0.4 * n)))


# ------------------------------------------------------------------ numbers of a scene --------

def _pulse(t, f0, fwidth):
    """tidy3d's Gaussian pulse with its DC component removed (complex amplitude at times t)."""
    tw = 1.0 / (2.0 * np.pi * fwidth)
    w0, ts = 2.0 * np.pi * f0, t - 5.0 * tw
    return np.exp(-1j * w0 * t - ts ** 2 / (2.0 * tw ** 2)) * (1j + ts / tw ** 2 / w0)


def _lorentz(de, w0, delta):
    r = np.sqrt(w0 * w0 - delta * delta)
    return complex(-delta, -r), complex(0.0, de * w0 * w0 / (2.0 * r))


def _cpml(depth, dl, dt):
    """(a, b, 1/kappa) at normalised depths of a face (tidy3d's default grading)."""
    sig = 1.5 / (ETA0 * dl) * depth ** 3
    kap = 1.0 + 2.0 * depth ** 3
    b = np.exp(-(dt / EPS0) * sig / kap)
    return np.where(sig > 0, (b - 1.0) / kap, 0.0), b, 1.0 / kap


def _model(c, seed, part=0):
    """Every number of the case's scene as numpy arrays (``part``: which scene of a batch)."""
    rng = np.random.default_rng([seed, part, 7])
    medium = c["medium"]
    shape = (c["nx"], c["ny"], c["nz"])
    nx, ny, nz = shape
    d0 = 10e-9 if medium == "cell" else 20e-9
    dls = [np.full(n, d0) for n in shape]
    if medium == "sphere":
        dls[2] = d0 * (1.0 + 0.25 * np.sin(np.linspace(0.0, np.pi, nz)) ** 2)
        dls[2][:12], dls[2][-12:] = dls[2][12], dls[2][-13]
    bounds = {"slab": ("Periodic", "Periodic", "PML"),
              "cell": ("BlochBoundary", "BlochBoundary", "PML")}.get(medium, ("PML",) * 3)
    layers = [12 if b == "PML" else 0 for b in bounds]
    if medium == "bend" and nz < 48:
        layers[2] = 8
    dt = 0.99 / (C0 * np.sqrt(sum(1.0 / d.min() ** 2 for d in dls)))
    resident = c["kind"] in ("step", "segment")
    n_total = c["steps"] * (RESIDENT_PASSES if c["kind"] == "step" else 1)
    m = dict(shape=shape, dls=dls, bounds=bounds, layers=layers, dt=dt, steps=c["steps"],
             n_total=n_total, sigma=None, mat=None, poles=[], bloch=(0.0, 0.0, 0.0), dipoles=[],
             plane=None, mode=None, tfsf=None, flux=[], boxes=[], probes=[], warm=None)
    t = np.arange(n_total + 1) * dt
    inner = [(lo, n - lo) for lo, n in zip(layers, shape)]
    f0 = 4e14 if medium == "cell" else 1.934e14 if medium == "bend" else 2.5e14
    fw = (0.1 if medium == "bend" else 0.4) * f0
    m["freqs"] = np.linspace(0.85 * f0, 1.15 * f0, c["nf"]) if c["nf"] > 1 else np.array([f0])

    if medium == "slab":
        thick = int(rng.integers(10, 20))
        eps = np.ones(shape)
        eps[:, :, nz // 2: nz // 2 + thick] = rng.uniform(2.0, 12.0)
        m["eps"] = [eps] * 3
        m["plane"] = (18, _pulse(t, f0, fw).real,
                      _pulse(t + 0.5 * dt + 0.5 * d0 / C0, f0, fw).real / ETA0)
        m["flux"] = [(2, nz - 18), (2, 15)]
    elif medium == "graded":
        eps = np.empty(shape)
        ax = [np.linspace(0, 1, n) for n in shape]
        p = rng.uniform(0, 6.28, 6)
        eps[:] = (4.0 + np.sin(9 * ax[0] + p[0])[:, None, None] * np.cos(7 * ax[1] + p[1])[None, :, None]
                  + np.cos(8 * ax[2] + p[2])[None, None, :])
        eps += 0.2 * rng.random(shape)
        m["eps"] = [eps, eps + 0.01, eps + 0.02]
    elif medium in ("soup", "sphere"):
        mat = np.full(shape, -1, np.int32)
        eps = np.ones(shape)
        if medium == "soup":
            for q in range(32):
                s = rng.integers(4, 65, size=3)
                lo = [int(rng.integers(a, b)) - int(x) // 2 for (a, b), x in zip(inner, s)]
                sl = tuple(slice(max(a, o), min(b, o + int(x)))
                           for (a, b), o, x in zip(inner, lo, s))
                lor = q % 2 == 1
                eps[sl] = rng.uniform(1.0, 4.0 if lor else 12.0)
                mat[sl] = len(m["poles"]) if lor else -1
                if lor:
                    m["poles"].append([_lorentz(rng.uniform(0.5, 3.0), rng.uniform(1e14, 8e14), 1e13)
                                       for _ in range(2)])
        else:
            r = rng.uniform(0.15, 0.35) * min(b - a for a, b in inner)
            g = [np.arange(n) - (n - 1) / 2.0 for n in shape]
            inside = (g[0][:, None, None] ** 2 + g[1][None, :, None] ** 2
                      + g[2][None, None, :] ** 2) <= r * r
            eps[inside] = rng.uniform(1.0, 4.0)
            mat[inside] = 0
            m["poles"].append([_lorentz(rng.uniform(0.5, 3.0), rng.uniform(1e14, 8e14), 1e13)])
        m["eps"], m["mat"] = [eps] * 3, mat
    elif medium == "cell":
        th, ph = np.deg2rad(30.0), np.deg2rad(45.0)
        k0 = 2.0 * np.pi * f0 / C0 * np.sin(th)
        kx, ky = k0 * np.cos(ph), k0 * np.sin(ph)
        m["bloch"] = (kx * nx * d0 / (2 * np.pi), ky * ny * d0 / (2 * np.pi), 0.0)
        k_sub = int(0.35 * nz)
        eps, mat = np.ones(shape), np.full(shape, -1, np.int32)
        eps[:, :, :k_sub] = 2.1
        xs, ys = np.arange(nx) + 0.5, np.arange(ny) + 0.5
        for i in range(3):
            for j in range(3):
                r = rng.uniform(2.0, 6.0)
                ins = ((xs[:, None] - (i + 0.5) * nx / 3) ** 2
                       + (ys[None, :] - (j + 0.5) * ny / 3) ** 2) <= r * r
                mat[ins, k_sub: k_sub + 20] = 0
        wp, gam = 1.37e16, 1e14
        m["poles"] = [[(complex(-gam, 0.0), complex(-wp * wp / (2 * gam), 0.0)),
                       _lorentz(1.0, 4e15, 2e14), _lorentz(0.6, 6e15, 3e14)]]
        eps[mat >= 0] = 1.0
        m["eps"], m["mat"] = [eps] * 3, mat
        m["sigma"] = np.where(mat >= 0, EPS0 * wp * wp / gam, 0.0)
        lo_k, hi_k = max(16, k_sub - 20), min(nz - 20, k_sub + 50)
        if c["tfsf"]:
            line = np.where(np.arange(nz) < k_sub, 2.1, 1.0)
            m["tfsf"] = dict(lo=(0, 0, lo_k), hi=(nx, ny, hi_k), k=(kx, ky),
                             j=(np.cos(ph), np.sin(ph)), line=line, phase=rng.uniform(0, 6.28))
        m["flux"] = [(2, hi_k + 4), (2, lo_k - 4)]
    elif medium == "bend":
        npx, cx, cy, cz = c["design"], nx // 2, ny // 2, nz // 2
        eps = np.full(shape, 2.1)
        zs = slice(cz - 5, cz + 6)
        dx, dy = cx - npx // 2, cy - npx // 2
        eps[:dx, cy - 12: cy + 13, zs] = 12.1
        eps[cx - 12: cx + 13, dy + npx:, zs] = 12.1
        u = np.linspace(0, 3 * np.pi, npx)
        p = rng.uniform(0, 6.28, 4)
        pix = 7.1 + 1.2 * (np.sin(u + p[0])[:, None] * np.cos(2 * u + p[1])[None, :]
                           + np.cos(1.4 * u + p[2])[:, None] * np.sin(u + p[3])[None, :])
        pix = pix + 0.5 * rng.random((npx, npx))
        eps[dx: dx + npx, dy: dy + npx, zs] = pix[:, :, None]
        m["eps"] = [eps] * 3
        ii, jj, kk = np.meshgrid(np.arange(dx, dx + npx), np.arange(dy, dy + npx),
                                 np.arange(cz - 5, cz + 6), indexing="ij")
        cells = ((ii * ny + jj) * nz + kk).ravel()
        m["comp"] = np.repeat(np.arange(3, dtype=np.int32), cells.size)
        m["cell"] = np.tile(cells.astype(np.int32), 3)
        yy, zz = np.arange(ny) - cy, np.arange(nz) - cz
        g = np.exp(-(yy[:, None] / 11.0) ** 2 - (zz[None, :] / 7.0) ** 2)
        g[(np.abs(yy) > 24)[:, None] | (np.abs(zz) > 14)[None, :]] = 0.0
        m["mode"] = (layers[0] + 6, g, g * 2.7 / ETA0, _pulse(t, f0, fw),
                     _pulse(t + 0.5 * dt, f0, fw))
        # a whole run looks at the far end of the output guide, a segment just behind the design
        km = ny - layers[1] - 8 if c["kind"] == "grad" else dy + npx + 4
        xx = np.arange(nx) - cx
        w = np.exp(-(xx[:, None] / 11.0) ** 2 - (zz[None, :] / 7.0) ** 2)
        w[(np.abs(xx) > 24)[:, None] | (np.abs(zz) > 14)[None, :]] = 0.0
        if c["kind"] == "segment":
            m["target"] = (km, w * np.exp(0.05j * xx)[:, None])
            m["target_tab"] = np.exp(2j * np.pi * f0 * (np.arange(n_total) + 1.0) * dt)
        else:
            m["flux"] = [(1, km)]
            k = np.zeros((4, nx, nz), np.complex128)
            k[0], k[3] = 2.7 / ETA0 * w, w
            m["weights"] = k * np.exp(0.05j * xx)[None, :, None] * 1e12

    if medium in ("soup", "sphere", "graded") or (medium == "cell" and not c["tfsf"]):
        amp = 1e-20 * _pulse(t + 0.5 * dt, f0, fw) / np.prod([d[n // 2] for d, n in zip(dls, shape)])
        if resident:
            amp = amp * 100.0                # visible beside the warm fields
        m["dipoles"] = [(2, (nx // 2, ny // 2, nz // 2), amp)]
        if medium != "cell":
            m["flux"] = [(2, nz - 16), (0, nx - 17), (1, ny - 18)]
    if resident:
        # the fields of a running simulation: a few long waves
        m["warm"] = [[(rng.uniform(-1, 1) * (1.0 if f < 3 else 1.0 / ETA0),
                       rng.uniform(-0.3, 0.3, 3), rng.uniform(0, 6.28)) for _ in range(3)]
                     for f in range(6)]
    if c["kind"] == "run" and medium == "sphere":
        m["probes"] = [((nx // 2 - 2, ny // 2 - 2, nz // 2 + 4), (4, 4, 3))]
    if c["kind"] == "step" and c["nx"] * c["ny"] * c["nz"] > 32e6:
        m["flux"] = []
        m["boxes"] = [((16, 16, nz // 2), (nx - 32, ny - 32, 1))]
    return m


def _warm_field(m, f, dev):
    """Initial field component ``f`` (float32 or complex64, rounded once, both sides read it)."""
    cplx = any(m["bloch"])
    out = None
    for amp, k, ph in m["warm"][f]:
        e = [torch.exp(1j * k[a] * torch.arange(n, dtype=torch.float64, device=dev))
             for a, n in enumerate(m["shape"])]
        v = (amp * np.exp(1j * ph)) * (e[0][:, None, None] * e[1][None, :, None]).to(torch.complex64) \
            * e[2].to(torch.complex64)[None, None, :]
        v = v if cplx else v.real
        out = v if out is None else out + v
    return out.to(torch.complex64 if cplx else torch.float32)


def _pole_numbers(m):
    """Per material (A - 1, B) of the trapezoidal pole update and sum 2 Re B."""
    out = []
    for poles in m["poles"]:
        a, r = (np.array([p[q] for p in poles]) for q in (0, 1))
        den = 1.0 - a * m["dt"] / 2.0
        b = r * m["dt"] / 2.0 / den
        out.append(((1.0 + a * m["dt"] / 2.0) / den - 1.0, b, 2.0 * b.real.sum()))
    return out


def _faces(m):
    """The CPML coefficients of every absorbing face, increasing global index."""
    out = {}
    for ax, n in enumerate(m["layers"]):
        if not n:
            continue
        for side in ("lo", "hi"):
            dl = m["dls"][ax][0 if side == "lo" else -1]
            p = np.arange(n, dtype=np.float64)
            de, dh = (n - p, n - p - 0.5) if side == "lo" else (p, p + 0.5)
            out[ax, side] = _cpml(de / n, dl, m["dt"]) + _cpml(dh / n, dl, m["dt"])
    return out


# ------------------------------------------------------------------ the package's side --------

def _scene(m):
    dt, shape = m["dt"], m["shape"]
    axes = [grid.Axis(np.concatenate([[0.0], np.cumsum(d)]), b, b)
            for d, b in zip(m["dls"], m["bounds"])]
    disp = None
    if m["poles"] and (m["mat"] >= 0).any():
        cells = np.flatnonzero(m["mat"].reshape(-1) >= 0)
        mid = m["mat"].reshape(-1)[cells]
        num = _pole_numbers(m)
        np_ = len(num[0][0])
        am1, b = np.stack([x[0] for x in num]), np.stack([x[1] for x in num])
        disp = model.Dispersion(
            comp=np.repeat(np.arange(3, dtype=np.int32), cells.size),
            cell=np.tile(cells.astype(np.int32), 3),
            pole_ofs=(np.arange(3 * cells.size + 1) * np_).astype(np.int32),
            am1=np.tile(am1[mid].reshape(-1), 3), b=np.tile(b[mid].reshape(-1), 3),
            g=np.tile(np.array([x[2] for x in num])[mid], 3))
    kw = {}
    if m["sigma"] is not None:
        kw.update(sigma_ex=m["sigma"], sigma_ey=m["sigma"], sigma_ez=m["sigma"])
    zero = np.zeros(m["n_total"] + 1)
    if m["plane"] is not None:
        ks, ex, hy = m["plane"]
        wf = waveform.Waveform(ex, ex, ex + 0j, ex + 0j, dt)
        kw["sources"] = [model.PlaneWaveSource(2, ks, +1, 0, wf, ex, hy)]
    kw["dipoles"] = [model.PointDipole(comp, np.array([idx]), np.ones(1), waveform.Waveform(
        zero, amp.real.copy(), zero + 0j, amp, dt)) for comp, idx, amp in m["dipoles"]]
    if m["mode"] is not None:
        ks, e, h, ae, ah = m["mode"]
        kw["mode_sources"] = [model.ModeSource(ks, +1, e + 0j, 0j * e, 0j * h, h + 0j, ae, ah, 2.7)]
    if m["tfsf"] is not None:
        f0 = m["freqs"].mean()
        t = np.arange(m["n_total"] + 1) * dt
        a0, a1 = (_pulse(x, f0, 0.4 * f0) * np.exp(1j * m["tfsf"]["phase"]) for x in (t, t + 0.5 * dt))
        kw["tfsf_sources"] = [model.TFSFSource(
            m["tfsf"]["lo"], m["tfsf"]["hi"], -1, waveform.Waveform(a0.real.copy(), a1.real.copy(), a0, a1, dt),
            open_axes=(0, 1), kxy=m["tfsf"]["k"], jxy=m["tfsf"]["j"],
            eps_line=(m["tfsf"]["line"], m["tfsf"]["line"]))]
    kw["field_time_monitors"] = [model.FieldTimeMonitor(f"t{q}", (0, 2, 4), o, b, 0, m["n_total"], 8,
                                                        m["n_total"] // 8)
                                 for q, (o, b) in enumerate(m["probes"])]
    return model.Scene(
        grid=grid.Grid(*axes), dt=dt, num_time_steps=m["n_total"], eps_ex=m["eps"][0],
        eps_ey=m["eps"][1], eps_ez=m["eps"][2],
        pml={k: cpml.PMLCoeffs(*v) for k, v in _faces(m).items()}, dispersion=disp,
        bloch_k=m["bloch"],
        flux_monitors=[model.FluxMonitor(f"f{q}", a, km, +1, m["freqs"])
                       for q, (a, km) in enumerate(m["flux"])],
        field_monitors=[model.FieldMonitor(f"b{q}", m["freqs"], o, b)
                        for q, (o, b) in enumerate(m["boxes"])], **kw)


def _parts(c):
    """The scenes of a serving batch."""
    n = c["scenes"]
    out = []
    for q in range(n):
        s = int(round(c["side_lo"] * (c["side_hi"] / c["side_lo"]) ** (q / max(n - 1, 1))))
        out.append(dict(kind="part", medium=("soup", "sphere", "slab")[q % 3], nx=s, ny=s, nz=s,
                        steps=c["steps"] + 40 * q, nf=c["nf"]))
    return out


class _Batch:
    """A serving pool and the step tables of the scenes that wait for it."""

    def __init__(self, tabs):
        self.tabs = tabs
        need = sum(serving.device_bytes(t) for t in tabs)
        self.pool = serving.Pool(int(1.1 * need) + (64 << 20))

    def __del__(self):
        self.pool.close()


def prepare(case, seed):
    c = case
    if c["kind"] == "pool":
        tabs = [tables.build(_scene(_model(p, seed, q))) for q, p in enumerate(_parts(c))]
        for t in tabs:
            t.material_classes()
        return dict(case=c, batch=_Batch(tabs))
    m = _model(c, seed)
    sc = _scene(m)
    if c["kind"] in ("run", "grad"):
        return dict(case=c, scene=sc, weights=m.get("weights"), comp=m.get("comp"), cell=m.get("cell"))
    st = solver.Stepper(tables.build(sc))
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    for f in range(6):
        st.write_field(f, _warm_field(m, f, dev).cpu().numpy())
    if c["kind"] == "step":
        st.setup_energy()
        return dict(case=c, stepper=st, steps=c["steps"])
    lib, ctx, P = st.lib, st.ctx, _lib.ptr
    comp, cell = m["comp"], m["cell"]
    co = adjoint.design_coefficients(st.tabs, comp, cell)
    _lib.check(lib, lib.oem_adjoint_setup(ctx, comp.size, P(comp), P(cell), *[P(x) for x in co],
                                          c["steps"]))
    for mag, fc, cells, z in _target_lists(m):
        tab = np.ascontiguousarray(m["target_tab"]).view(np.float64)
        z = np.ascontiguousarray(z, np.complex64).view(np.float32)
        _lib.check(lib, lib.oem_adjoint_objective(ctx, mag, cells.size, P(np.full(cells.size, fc, np.int32)),
                                                  P(cells), P(z), P(tab)))
    _lib.check(lib, lib.oem_checkpoint_alloc(ctx, 1))
    _lib.check(lib, lib.oem_checkpoint_save(ctx, 0))
    return dict(case=c, stepper=st, steps=c["steps"], n=comp.size)


def _target_lists(m):
    """The objective's points on the output plane (normal y): (magnetic, component, cells, z)."""
    (nx, ny, nz), (km, w) = m["shape"], m["target"]
    ii, kk = np.nonzero(w)
    at = lambda j: ((ii * ny + j) * nz + kk).astype(np.int32)  # noqa: E731
    z = w[ii, kk]
    return [(0, 0, at(km), z), (0, 2, at(km), 0.5 * z), (1, 0, at(km), 150.0 * z),
            (1, 0, at(km - 1), 150.0 * z), (1, 2, at(km), 90.0 * z), (1, 2, at(km - 1), 90.0 * z)]


def run(state):
    kind = state["case"]["kind"]
    if kind == "run":
        r = openem_amd.run(state["scene"], verbose=False, use_shutoff=False)
        return dict(phasors={k: v.data for k, v in r.phasors.items()}, time=r.time_samples)
    if kind == "step":
        st = state["stepper"]
        st.run(state["steps"])
        return dict(monitors=[st.read_monitor(i) for i in range(len(st.mon_ids))], energy=st.energy())
    if kind == "pool":
        b = state["batch"]
        sts = [solver.Stepper(t, pool=b.pool) for t in b.tabs]
        b.pool.run_to_completion(sts)
        out = [[st.read_monitor(i) for i in range(len(st.mon_ids))] for st in sts]
        for st in sts:
            st.close()
        return out
    if kind == "grad":
        g = adjoint.overlap_power_gradient(state["scene"], "f0", state["weights"], state["comp"],
                                           state["cell"])
        return dict(J=g.J, a=np.array([g.a_plus]), grad=g.grad)
    st, n = state["stepper"], state["steps"]
    lib, ctx = st.lib, st.ctx
    _lib.check(lib, lib.oem_checkpoint_load(ctx, 0))
    _lib.check(lib, lib.oem_adjoint_record(ctx, n))
    _lib.check(lib, lib.oem_adjoint_back(ctx, n))
    out = np.empty(state["n"], np.float64)
    _lib.check(lib, lib.oem_adjoint_gradient(ctx, _lib.ptr(out), out.size))
    return out


def work(case):
    c = case
    if c["kind"] == "pool":
        w = [work(p) for p in _parts(c)]
        return dict(bytes=sum(x["bytes"] for x in w), flops=sum(x["flops"] for x in w))
    n = c["nx"] * c["ny"] * c["nz"]
    wide = 2 if c["medium"] == "cell" else 1
    # a step reads and writes E and H once, reads the material of each cell, and reads and
    # writes four psi components of each face pair's layers
    per = 48 * wide + (24 if c["medium"] == "graded" else 2)
    lay = [0 if c["medium"] in ("slab", "cell") and a < 2 else 24 for a in range(3)]
    psi = sum(32 * wide * n * la / s for la, s in zip(lay, (c["nx"], c["ny"], c["nz"])))
    b, f = c["steps"] * (per * n + psi), c["steps"] * 42.0 * wide * n
    if c["kind"] in ("grad", "segment"):     # and the adjoint step the same, plus the record
        b, f = 2 * b + 2 * c["steps"] * 12.0 * 11 * c["design"] ** 2, 2 * f
    return dict(bytes=float(b), flops=float(f))


# ------------------------------------------------------------------ the same in 64 bits -------

class _Stepper64:
    """The scene's time step in float64 (complex128 on a Bloch cell), as plain torch."""

    def __init__(self, m, eps=None):
        self.m = m
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.cplx = any(m["bloch"])
        self.dtype = torch.complex128 if self.cplx else torch.float64
        shape, dt = m["shape"], m["dt"]
        z = lambda: torch.zeros(shape, dtype=self.dtype, device=self.dev)  # noqa: E731
        self.E, self.H = [z() for _ in range(3)], [z() for _ in range(3)]
        self.ax = []
        faces = _faces(m)
        for a in range(3):
            dl, n = m["dls"][a], shape[a]
            per = m["bounds"][a] != "PML"
            dual = 0.5 * (dl + np.roll(dl, 1))
            if not per:
                dual[0] = dl[0]
            co = [np.zeros(n), np.ones(n), np.ones(n), np.zeros(n), np.ones(n), np.ones(n)]
            for side in ("lo", "hi"):
                if (a, side) in faces:
                    la = m["layers"][a]
                    for v, f in zip(co, faces[a, side]):
                        v[slice(0, la) if side == "lo" else slice(n - la, n)] = f
            pec = np.ones(n)
            if not per:
                pec[0] = 0.0
            ph = np.exp(2j * np.pi * m["bloch"][a]) if self.cplx else 1.0
            self.ax.append(dict(idp=self._b(1.0 / dl, a), idd=self._b(1.0 / dual, a), dl=dl,
                                dual=dual, pec=self._b(pec, a), hi=ph if per else 0.0,
                                lo=1.0 / ph if per else 0.0, pml=bool(m["layers"][a]),
                                e=[self._b(v, a) for v in co[:3]], h=[self._b(v, a) for v in co[3:]]))
        self.psi = {}
        T = lambda v: torch.as_tensor(v, device=self.dev)  # noqa: E731
        self.num = _pole_numbers(m)
        self.cells, self.P, self.Q = [], [], []
        g = None
        if m["mat"] is not None:
            flat = T(m["mat"]).reshape(-1)
            g = torch.zeros(shape, dtype=torch.float64, device=self.dev)
            for q, (am1, b, gg) in enumerate(self.num):
                idx = torch.nonzero(flat == q).reshape(-1)
                self.cells.append(idx)
                g.view(-1)[idx] = gg
                for s in (self.P, self.Q):
                    s.append([torch.zeros((len(am1), idx.numel()), dtype=torch.complex128,
                                          device=self.dev) for _ in range(3)])
        self.ca, self.cb, seen = [], [], {}
        for c in range(3):
            e = eps[c] if eps is not None else m["eps"][c]
            if id(e) not in seen:
                t = e if eps is not None else T(e)
                s = 0.0 if m["sigma"] is None else T(m["sigma"]) * (dt / (2.0 * EPS0))
                den = t + s + (0.0 if g is None else g)
                seen[id(e)] = ((t - s) / den, (dt / EPS0) / den)
            self.ca.append(seen[id(e)][0])
            self.cb.append(seen[id(e)][1])
        self.n = 0
        if m["warm"] is not None:
            for f in range(6):
                (self.E if f < 3 else self.H)[f % 3] = _warm_field(m, f, self.dev).to(self.dtype)

    def _b(self, v, a):
        s = [1, 1, 1]
        s[a] = -1
        return torch.as_tensor(np.ascontiguousarray(v), device=self.dev).reshape(s)

    def _diff(self, F, a, fwd, key):
        A, n = self.ax[a], F.shape[a]
        if fwd:
            d = (torch.cat([F.narrow(a, 1, n - 1), F.narrow(a, 0, 1) * A["hi"]], a) - F) * A["idp"]
        else:
            d = (F - torch.cat([F.narrow(a, n - 1, 1) * A["lo"], F.narrow(a, 0, n - 1)], a)) * A["idd"]
        if not A["pml"]:
            return d
        ca, cb, ik = A["h" if fwd else "e"]
        psi = self.psi.get(key)
        psi = d * ca if psi is None else torch.addcmul(psi * cb, d, ca)
        self.psi[key] = psi
        return torch.addcmul(psi, d, ik)

    def step(self):
        m, n, E, H = self.m, self.n, self.E, self.H
        ch, ax = m["dt"] / MU0, self.ax
        H = [H[c] - ch * (self._diff(E[(c + 2) % 3], (c + 1) % 3, True, ("h", c, 0))
                          - self._diff(E[(c + 1) % 3], (c + 2) % 3, True, ("h", c, 1)))
             for c in range(3)]
        if m["plane"] is not None:
            ks, ex, hy = m["plane"]
            H[1][:, :, ks - 1] += ch / ax[2]["dl"][ks - 1] * ex[n]
        if m["mode"] is not None:
            ks, e, h, ae, ah = m["mode"]
            v = torch.as_tensor(ch / ax[0]["dl"][ks - 1] * e * ae[n].real, device=self.dev)
            H[2] = H[2].clone()
            H[2][ks - 1] += v
        hist = [None] * 3
        for q, (am1, b, _) in enumerate(self.num):
            am1, b = (torch.as_tensor(x, device=self.dev)[:, None] for x in (am1, b))
            for c in range(3):
                en = E[c].reshape(-1)[self.cells[q]]
                w = 0.0
                for S, x, unit in ((self.P, en.real, 1.0), (self.Q, en.imag if self.cplx else None, 1j)):
                    if x is None:
                        continue
                    dP = am1 * S[q][c] + b * x
                    S[q][c] = S[q][c] + dP
                    w = w + unit * 2.0 * dP.real.sum(0)
                if hist[c] is None:
                    hist[c] = torch.zeros(m["shape"], dtype=self.dtype, device=self.dev)
                hist[c].view(-1)[self.cells[q]] = w.to(self.dtype)
        new = []
        for c in range(3):
            u, v = (c + 1) % 3, (c + 2) % 3
            s = self._diff(H[v], u, False, ("e", c, 0)) - self._diff(H[u], v, False, ("e", c, 1))
            if hist[c] is not None:
                s = s - (EPS0 / m["dt"]) * hist[c]
            x = self.ca[c] * E[c] + self.cb[c] * s
            for a in (u, v):
                if m["bounds"][a] == "PML":
                    x = x * ax[a]["pec"]
            new.append(x)
        E = new
        if m["plane"] is not None:
            E[0][:, :, ks] += self.cb[0][:, :, ks] / ax[2]["dual"][ks] * hy[n]
        if m["mode"] is not None:
            v = torch.as_tensor(h * ah[n].real / ax[0]["dual"][ks], device=self.dev)
            E[1] = E[1].clone()
            E[1][ks] += self.cb[1][ks] * v
        for c, idx, amp in m["dipoles"]:
            E[c][idx] -= self.cb[c][idx] * (amp[n] if self.cplx else amp[n].real)
        for q, (am1, b, _) in enumerate(self.num):
            b = torch.as_tensor(b, device=self.dev)[:, None]
            for c in range(3):
                en = E[c].reshape(-1)[self.cells[q]]
                self.P[q][c] = self.P[q][c] + b * en.real
                if self.cplx:
                    self.Q[q][c] = self.Q[q][c] + b * en.imag
        self.E, self.H = E, H
        self.n += 1


def _plane(s, a, km):
    t1, t2 = [x for x in range(3) if x != a]
    at = lambda F, k: F.select(a, k)  # noqa: E731
    return [at(s.E[t1], km), at(s.E[t2], km), 0.5 * (at(s.H[t1], km) + at(s.H[t1], km - 1)),
            0.5 * (at(s.H[t2], km) + at(s.H[t2], km - 1))]


def _accumulate(s, acc, n):
    """Add the step's samples to the monitors' phasors (E at (n+1) dt, H at (n+1/2) dt)."""
    m = s.m
    w = 2.0 * np.pi * m["freqs"]
    ph = [torch.as_tensor(np.exp(1j * w * (n + o) * m["dt"]), device=s.dev) for o in (1.0, 0.5)]
    vals = [_plane(s, a, km) for a, km in m["flux"]]
    for o, b in m["boxes"]:
        sl = tuple(slice(x, x + y) for x, y in zip(o, b))
        vals.append([F[sl] for F in s.E + s.H])
    for q, v in enumerate(vals):
        half = len(v) // 2
        add = torch.stack([x[None] * ph[0 if k < half else 1].reshape((-1,) + (1,) * x.dim())
                           for k, x in enumerate(v)])
        acc[q] = add if acc[q] is None else acc[q] + add
    return acc


def _energies(s):
    out = torch.zeros(3, dtype=torch.float64, device=s.dev)
    for c in range(3):
        L = [s._b(A["dl"] if a == c else A["dual"], a) for a, A in enumerate(s.ax)]
        V = L[0] * L[1] * L[2]
        e2 = V * s.E[c].abs() ** 2
        out[0] += e2.sum()
        out[1] += (e2 * torch.as_tensor(s.m["eps"][c], device=s.dev)).sum()
        out[2] += (V * s.H[c].abs() ** 2).sum()
    return out.cpu().numpy()


def exact(case, seed):
    c = case
    if c["kind"] == "pool":
        return [exact(p, (seed, q)) for q, p in enumerate(_parts(c))]
    seed, part = seed if isinstance(seed, tuple) else (seed, None)
    m = _model(c, seed, part or 0)
    if m["tfsf"] is not None:
        return None                          # its incident line is a simulation of its own
    host = lambda acc: [x.cpu().numpy() for x in acc]  # noqa: E731
    if c["kind"] in ("run", "step", "part"):
        s, acc = _Stepper64(m), [None] * (len(m["flux"]) + len(m["boxes"]))
        probes = [np.zeros((3, m["n_total"] // 8) + b) for _, b in m["probes"]]
        with torch.no_grad():
            for n in range(c["steps"]):
                s.step()
                acc = _accumulate(s, acc, n)
                for (o, b), out in zip(m["probes"], probes):
                    sl = tuple(slice(x, x + y) for x, y in zip(o, b))
                    for k, F in enumerate((s.E[0], s.E[2], s.H[1])):
                        for mm, wt in ((n + 1, 1.0 if k < 2 else 0.5), (n, 0.0 if k < 2 else 0.5)):
                            if mm % 8 == 0 and mm // 8 < out.shape[1] and wt:
                                out[k, mm // 8] += wt * F[sl].cpu().numpy()
            if part is not None:
                return host(acc)
            if c["kind"] == "step":
                return dict(monitors=host(acc), energy=_energies(s))
        last = (c["steps"] - 1) // 8 + 1
        return dict(phasors={f"f{q}": x for q, x in enumerate(host(acc))},
                    time={f"t{q}": x[:, :last] for q, x in enumerate(probes)})
    # gradients: the same step, differentiated by torch
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    comp, cell = (torch.as_tensor(m[k], device=dev).long() for k in ("comp", "cell"))
    eps = [torch.as_tensor(e, device=dev).clone() for e in m["eps"]]
    p = torch.stack(eps).reshape(3, -1)[comp, cell].clone().requires_grad_(True)
    eps = list(torch.stack(eps).reshape(3, -1).index_put((comp, cell), p).reshape((3,) + m["shape"]))
    s = _Stepper64(m, eps)
    if c["kind"] == "grad":
        acc = [None]
        for n in range(c["steps"]):
            s.step()
            acc = _accumulate(s, acc, n)
        a = (acc[0][:, 0] * torch.as_tensor(m["weights"], device=dev)).sum()
        J = a.abs() ** 2
        J.backward()
        return dict(J=float(J.detach()), a=a.detach().cpu().numpy()[None], grad=p.grad.cpu().numpy())
    J = 0.0
    lists = [(mag, fc, torch.as_tensor(cells, device=dev).long(), np.complex64(z))
             for mag, fc, cells, z in _target_lists(m)]
    for n in range(c["steps"]):
        s.step()
        for mag, fc, cells, z in lists:
            w = torch.as_tensor((z.astype(np.complex128) * m["target_tab"][n]).real, device=dev)
            J = J + (w * (s.H if mag else s.E)[fc].reshape(-1)[cells]).sum()
    J.backward()
    return p.grad.cpu().numpy()
