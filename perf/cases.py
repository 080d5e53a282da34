"""Workloads whose speed is measured, through the framework's public entry points.

Each case is one thing that a user's program does with ``kwave_amd``:

* ``call``    a whole ``kspace_first_order`` / ``kspace_first_order_as`` call on host data: tables, upload,
              time loop, read-back (the drop-in use; small grids, where latency and launches count);
* ``steps``   a ``Simulation`` that the program keeps, advanced by a run of time steps, then its sensor data
              (2-D grids also the pressure field) read: long acoustic runs, where the time loop is all that counts;
* ``elastic`` the same with an ``ElasticSimulation``;
* ``firings`` the same with a stacked transmit sequence (``Simulation.firings``);
* ``grad``    a whole ``gradient_c0`` call: misfit gradient of a transmit sequence (forward, recompute, adjoint).

Results of Float32 runs come back from the library as Float32 values widened to Float64; they are returned here
in the type they were computed in.  ``exact`` restates the same schemes in torch, in Float64.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "k-wave-julia_amd"))

import kwave_amd as K  # noqa: E402

DX = 1e-4
MANY = 2_000_000     # Nt of kept simulations: far more steps than a program takes


def _smooth_number(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


SMOOTH = [n for n in range(8, 1025) if _smooth_number(n)]


def listed():
    def acoustic(name, kind, n, steps, dtype, **kw):
        n = tuple(n) + (1,) * (3 - len(n))
        base = dict(name=name, kind=kind, nx=n[0], ny=n[1], nz=n[2], steps=steps, dtype=dtype, het=True, absorb=True,
                    nonlinear=False, source="p", maps="native", axisym=False, pml=20)
        base.update(kw)
        return base

    return [
        # the smallest whole call: a 1-D pulse, double precision (the default data_cast); latency is all there is
        acoustic("call 1d 512 f64", "call", (512,), 1200, "f64", het=False, absorb=False, source="p0"),
        # the 2-D homogeneous 128 x 128 configuration with its full record length, double precision
        acoustic("call 2d 128x128 f64", "call", (128, 128), 1208, "f64", het=False, absorb=False),
        # a whole single-precision call on a grid of no special size: photoacoustic p0 (smoothed, as by default)
        acoustic("call 2d 300x251 f32", "call", (300, 251), 500, "f32", source="p0"),
        # one 2-D simulation of ordinary size, kept by the program and advanced (ultrasound imaging, inversion loops)
        acoustic("steps 2d 512x512 f32", "steps", (512, 512), 300, "f32"),
        # a small 3-D grid: all fields fit the last-level cache, launches are short
        acoustic("steps 3d 128^3 f32", "steps", (128, 128, 128), 150, "f32", nonlinear=True),
        # the framework's headline: heterogeneous absorbing nonlinear 256^3, single precision
        acoustic("steps 3d 256^3 f32", "steps", (256, 256, 256), 60, "f32", nonlinear=True),
        # sides of small prime factors but no power of two, as programs size their grids
        acoustic("steps 3d 240x216x150 f32", "steps", (240, 216, 150), 60, "f32", nonlinear=True, pml=10),
        # double precision in 3-D (the reference's default type), unequal sides
        acoustic("steps 3d 192x160x128 f64", "steps", (192, 160, 128), 60, "f64", nonlinear=True, pml=10),
        # the largest: half of the 512^3 layered workload, medium maps stored as Float16 offsets
        acoustic("steps 3d 512x512x256 f32 f16", "steps", (512, 512, 256), 12, "f32", nonlinear=True, maps="f16"),
        # elastic wave propagation through layers (transcranial, nondestructive testing)
        dict(name="elastic 3d 256x256x128 f32", kind="elastic", nx=256, ny=256, nz=128, steps=40, dtype="f32", pml=10),
        # waveform inversion: misfit gradient of a ring's transmit sequence
        dict(name="grad 2d 256x256 f32", kind="grad", nx=256, ny=256, firings=16, steps=200, every=50, dtype="f32",
             pml=20),
        # a transmit sequence: one firing per element on one grid and medium, run as one stacked simulation
        dict(name="firings 2d 320x200x24 f32", kind="firings", nx=320, ny=200, firings=24, steps=100, dtype="f32",
             pml=20),
    ]


def _length(rng, lo, hi):
    """An axis length: half of them products of 2, 3 and 5 (what grids are mostly sized to), half any."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(SMOOTH, key=lambda s: (abs(s - n), s)) if rng.random() < 0.5 else n


def _planned(rng, lo, hi):
    """An axis length that the adjoint and the elastic solver take."""
    have = [n for n in (48, 64, 72, 80, 96, 100, 125, 128, 144, 160, 192, 200, 225, 243, 256, 320, 384, 400, 512, 640,
                        768, 1024) if lo <= n <= hi]
    return rng.choice(have)


def draw(rng):
    kind = rng.choice(("call", "call", "steps", "steps", "steps", "elastic", "firings", "grad"))
    dtype = rng.choice(("f32", "f32", "f64"))
    if kind in ("call", "steps"):
        nd = rng.choice((1, 2, 2)) if kind == "call" else rng.choice((2, 3, 3))
        lo, hi = {1: (64, 1024), 2: (64, 400) if kind == "call" else (100, 1000), 3: (48, 320)}[nd]
        n = [_length(rng, lo, hi) for _ in range(nd)]
        while nd == 3 and n[0] * n[1] * n[2] > 256 ** 3:
            n[n.index(max(n))] = _length(rng, lo, max(n) * 3 // 4)
        vox = int(np.prod(n))
        steps = rng.randint(150, 900) if kind == "call" else max(20, min(300, int(6e8 / vox)) - rng.randint(0, 9))
        if kind == "steps" and nd == 2:
            steps = min(steps, min(n))      # the field that is read back still holds the waves
        het = rng.random() < 0.7
        axisym = kind == "call" and nd == 2 and rng.random() < 0.2
        return dict(kind=kind, nx=n[0], ny=n[1] if nd > 1 else 1, nz=n[2] if nd > 2 else 1, steps=steps, dtype=dtype,
                    het=het, absorb=rng.random() < 0.6, nonlinear=rng.random() < 0.4,
                    source=rng.choice(("p", "p0", "u", "tr") if kind == "call" and not axisym else ("p", "u")),
                    maps="f16" if kind == "steps" and het and dtype == "f32" and rng.random() < 0.25 else "native",
                    axisym=axisym, pml=rng.randint(6, 20))
    if kind == "elastic":
        nd = rng.choice((2, 3))
        n = [_planned(rng, 48 if nd == 3 else 100, 256 if nd == 3 else 768) for _ in range(nd)]
        vox = int(np.prod(n))
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2] if nd > 2 else 1, dtype=dtype, pml=rng.randint(6, 16),
                    steps=max(20, min(200, int(3e8 / vox)) - rng.randint(0, 9)))
    if kind == "firings":
        return dict(kind=kind, nx=_planned(rng, 100, 512), ny=_planned(rng, 100, 512), firings=rng.randint(2, 40),
                    steps=rng.randint(50, 100), dtype=dtype, pml=rng.randint(10, 20))
    return dict(kind="grad", nx=_planned(rng, 128, 320), ny=_planned(rng, 128, 320), firings=rng.randint(1, 20),
                steps=rng.randint(100, 200), every=rng.choice((20, 50)), dtype=dtype, pml=rng.randint(10, 20))


# ---------------------------------------------------------------------------
# inputs: numbers of a problem, made from the seed alone
# ---------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _sides(case):
    return [case[k] for k in ("nx", "ny", "nz") if case.get(k, 1) > 1]


def _axes(n, dev):
    """Index vectors broadcastable over a (z, y, x) array."""
    nd = len(n)
    return [torch.arange(n[a], device=dev, dtype=torch.float64).reshape([-1 if d == nd - 1 - a else 1 for d in range(nd)])
            for a in range(nd)]


def _blobs(n, rng, count, lo, hi, width, dev):
    """Sum of Gaussian inclusions, as a (z, y, x) Float64 tensor."""
    out = torch.zeros(list(reversed(n)), dtype=torch.float64, device=dev)
    ax = _axes(n, dev)
    for _ in range(count):
        amp = float(rng.uniform(lo, hi))
        g = None
        for a, x in enumerate(ax):
            c, w = float(rng.uniform(0.15, 0.85)) * n[a], max(2.5, float(rng.uniform(*width)) * min(n))
            e = torch.exp(-((x - c) / w) ** 2 / 2)
            g = e if g is None else g * e
        out += amp * g
    return out


def _host(t):
    """(z, y, x) tensor -> column-major (x, y, z) array, as the framework takes its maps."""
    return t.cpu().numpy().T


def _burst(dt, f0, cycles, columns):
    """Gaussian tone burst in at most `columns` samples and one zero column (the last value is re-added after)."""
    n = min(columns, int(round(cycles / f0 / dt)))
    t = np.arange(n) * dt
    mid = cycles / f0 / 2
    s = np.sin(2 * math.pi * f0 * t) * np.exp(-((t - mid) / (mid / cycles)) ** 2 / 2)
    return np.concatenate([s, [0.0]])


def _problem(case, seed):
    """Everything that defines an acoustic run, as numbers (maps as (z, y, x) tensors, indices column-major)."""
    rng, dev = np.random.default_rng(seed), _device()
    n = _sides(case)
    nd, vox = len(n), int(np.prod(n))
    pml = min(case["pml"], min(n) // 4)
    q = dict(n=n, pml=pml, steps=case["steps"], absorb=None, bona=6.0 if case["nonlinear"] else None, p0=None,
             p=None, u=None, tr=None, axisym=case["axisym"])
    if case["het"]:
        q["c0"] = 1500.0 + _blobs(n, rng, 6, -100.0, 120.0, (0.03, 0.12), dev)
        q["rho0"] = 1000.0 + _blobs(n, rng, 6, -80.0, 100.0, (0.03, 0.12), dev)
    else:
        q["c0"], q["rho0"] = float(rng.uniform(1450, 1550)), float(rng.uniform(950, 1050))
    cmax = float(q["c0"].max()) if case["het"] else q["c0"]
    q["dt"] = 0.3 * DX / cmax
    if case["absorb"]:
        q["absorb"] = (float(rng.uniform(0.4, 0.8)), 1.5)
    # sources: an aperture on the first rows after the PML along the last axis
    plane = vox // n[-1]
    idx = np.arange(plane) + plane * pml if nd > 1 else np.array([n[0] // 3])
    f0 = 1500.0 / (8 * DX)
    if case["source"] in ("p", "u"):
        burst = _burst(q["dt"], f0, 3, 120)
        w = 1.0 + 0.5 * np.cos(np.arange(idx.size) * float(rng.uniform(0.01, 0.05)) + float(rng.uniform(0, 6)))
        if case["source"] == "p":
            q["p"] = (idx, 1e5 * w[:, None] * burst[None, :])
        else:
            q["u"] = (idx, [0.05 * float(rng.uniform(0.5, 1)) * w[:, None] * burst[None, :] for _ in range(nd)])
    if case["source"] == "tr":
        t = np.arange(case["steps"])[None, :]
        ph = rng.uniform(0, 2 * math.pi, (idx.size, 2))
        q["tr"] = 1e4 * (np.sin(0.11 * t + ph[:, :1]) + 0.5 * np.sin(0.037 * t + ph[:, 1:]))
    elif case["source"] == "p0" or case["kind"] == "steps":
        # steps: a wave field that fills the grid from the first step on
        q["p0"] = _blobs(n, rng, 10, 2e4, 2e5, (0.03, 0.08), dev)
    # sensors: two crossed planes (3-D), two crossed lines (2-D), a few points (1-D); TR: the aperture itself
    mask = torch.zeros(list(reversed(n)), dtype=torch.bool, device=dev)
    if case["source"] == "tr":
        mask.reshape(-1)[torch.from_numpy(idx).to(dev)] = True
    elif nd == 1:
        mask[[n[0] // 4, n[0] // 2, n[0] - n[0] // 4]] = True
    else:
        mask[(3 * n[-1]) // 4] = True
        mask[:, n[-2] // 2] = True
    q["mask"] = mask
    q["smooth"] = case["kind"] == "call"
    q["record"] = (["p_final"] if case["source"] == "tr" else
                   ["p", "p_max", "u_rms"] if case["kind"] == "call" else ["p_max", "p_min"])
    return q


def _kgrid(n, dt, Nt):
    kg = K.KWaveGrid(*[v for k in n for v in (k, DX)])
    kg.dt, kg.Nt = dt, Nt
    return kg


def _np(v):
    return _host(v) if torch.is_tensor(v) else v


def _mask_of(idx, n):
    m = np.zeros(int(np.prod(n)), dtype=bool)
    m[idx] = True
    return m.reshape(n, order="F")


def _model(q, Nt):
    """The framework's own objects for a problem: (kgrid, medium, source, sensor)."""
    n = q["n"]
    ab = dict(alpha_coeff=q["absorb"][0], alpha_power=q["absorb"][1], alpha_mode="stokes") if q["absorb"] else {}
    med = K.KWaveMedium(sound_speed=_np(q["c0"]), density=_np(q["rho0"]), BonA=q["bona"], **ab)
    src = {}
    if q["p0"] is not None:
        src["p0"] = _np(q["p0"])
    if q["p"]:
        src.update(p_mask=_mask_of(q["p"][0], n), p=q["p"][1])
    if q["u"]:
        src.update(u_mask=_mask_of(q["u"][0], n), **dict(zip(("ux", "uy", "uz"), q["u"][1])))
    sen = K.KWaveSensor(mask=_host(q["mask"]), record=q["record"], time_reversal_boundary_data=q["tr"])
    return _kgrid(n, q["dt"], Nt), med, K.KWaveSource(**src), sen


def _elastic_problem(case, seed):
    rng, dev = np.random.default_rng(seed), _device()
    n = _sides(case)
    solid = (_axes(n, dev)[-1] >= n[-1] * float(rng.uniform(0.45, 0.55))).to(torch.float64)
    noise = _blobs(n, rng, 6, -40.0, 40.0, (0.03, 0.1), dev)
    q = dict(n=n, pml=min(case["pml"], min(n) // 4), steps=case["steps"],
             cp=1540.0 + 1460.0 * solid + noise, cs=(1500.0 * solid).expand(noise.shape).contiguous(),
             rho0=1000.0 + 900.0 * solid + noise, p0=_blobs(n, rng, 8, 2e4, 2e5, (0.03, 0.08), dev))
    q["dt"] = 0.3 * DX / float(q["cp"].max())
    q["mask"] = torch.zeros(list(reversed(n)), dtype=torch.bool, device=dev)
    q["mask"][n[-1] // 2 - 4] = True
    q["record"] = ["p_max", "p_min", "u_max"]
    return q


def _ring_problem(case, seed):
    rng, dev = np.random.default_rng(seed), _device()
    n, m = _sides(case), 64
    c0 = 1500.0 + _blobs(n, rng, 5, -40.0, 60.0, (0.04, 0.12), dev)
    dt = 0.3 * DX / 1650.0
    ang = 2 * math.pi * np.arange(m) / m
    ix = np.round(n[0] / 2 + 0.36 * n[0] * np.cos(ang)).astype(int)
    iy = np.round(n[1] / 2 + 0.36 * n[1] * np.sin(ang)).astype(int)
    ring = np.unique(ix + n[0] * iy)
    px, py = ring % n[0], ring // n[0]
    f0 = 1500.0 / (8 * DX)
    burst = _burst(dt, f0, 2, 100)
    fire = rng.choice(ring.size, size=case["firings"], replace=case["firings"] > ring.size)
    obs, t = [], (np.arange(case["steps"]) + 1) * dt
    for k in fire:      # observations: straight-ray arrivals of the burst at another speed
        r = np.hypot(px - px[k], py - py[k]) * DX
        late = t[None, :] - (r / float(rng.uniform(1460, 1540)))[:, None]
        mid = 1.0 / f0
        s = np.sin(2 * math.pi * f0 * late) * np.exp(-((late - mid) / (mid / 2)) ** 2 / 2)
        obs.append(np.where(late > 0, s, 0.0) * (0.05 / np.sqrt(1 + r / DX))[:, None])
    return dict(n=n, pml=min(case["pml"], min(n) // 4), dt=dt, steps=case["steps"], c0=c0, rho0=1000.0, ring=ring,
                fire=ring[fire], burst=burst, obs=obs)


def _firing_problems(case, seed):
    """A transmit sequence: one problem per element of an aperture, on one grid and medium."""
    rng = np.random.default_rng(seed)
    one = dict(case, nz=1, het=True, absorb=True, nonlinear=False, source="none", axisym=False)
    q = _problem(one, seed)
    n = q["n"]
    q["rho0"] = 1000.0
    out = []
    for x in rng.choice(n[0] - 2 * q["pml"] - 2, size=case["firings"], replace=True):
        burst = 1e5 * float(rng.uniform(0.5, 1.5)) * _burst(q["dt"], 1500.0 / (8 * DX), 3, 120)
        idx = q["pml"] + int(x) + np.arange(2) + n[0] * (q["pml"] + 1)
        out.append(dict(q, p=(idx, np.stack([burst, burst]))))
    return out


# ---------------------------------------------------------------------------
# what a program holds before the call, and the call
# ---------------------------------------------------------------------------

def _cast(case):
    return np.float64 if case["dtype"] == "f64" else np.float32


def prepare(case, seed):
    T = _cast(case)
    if case["kind"] in ("call", "steps"):
        q = _problem(case, seed)
        kw = dict(pml_size=q["pml"], pml_alpha=2.0, data_cast=T)
        if case["kind"] == "call":
            kg, med, src, sen = _model(q, q["steps"])
            return dict(case=case, args=(kg, med, src, sen), kw=kw)
        kg, med, src, sen = _model(q, MANY)
        desc, keep, _ = K.build_desc(kg, med, src, sen, smooth_p0=False,
                                     medium_storage=np.float16 if case["maps"] == "f16" else None, **kw)
        return dict(case=case, sim=K.Simulation(desc, keep), record=q["record"])
    if case["kind"] == "elastic":
        q = _elastic_problem(case, seed)
        med = K.ElasticMedium(sound_speed_compression=_host(q["cp"]), sound_speed_shear=_host(q["cs"]),
                              density=_host(q["rho0"]))
        sen = K.KWaveSensor(mask=_host(q["mask"]), record=q["record"])
        from kwave_amd.elastic import build_elastic_desc
        desc, keep, _ = build_elastic_desc(_kgrid(q["n"], q["dt"], MANY), med, K.ElasticSource(p0=_host(q["p0"])), sen,
                                           pml_size=q["pml"], pml_alpha=2.0, data_cast=T)
        return dict(case=case, sim=K.ElasticSimulation(desc, keep), record=q["record"])
    if case["kind"] == "firings":
        descs, keeps = [], []
        for q in _firing_problems(case, seed):
            d, k, _ = K.build_desc(*_model(q, MANY), pml_size=q["pml"], pml_alpha=2.0, smooth_p0=False, data_cast=T)
            descs.append(d)
            keeps.append(k)
        return dict(case=case, sim=K.Simulation.firings(descs, keeps), record=["p_max", "p_min"])
    q = _ring_problem(case, seed)
    ring = _mask_of(q["ring"], q["n"])
    srcs = [K.KWaveSource(p_mask=_mask_of([f], q["n"]), p=q["burst"][None, :]) for f in q["fire"]]
    sens = [K.KWaveSensor(mask=ring, record=["p"])] * len(srcs)
    return dict(case=case, args=(_kgrid(q["n"], q["dt"], q["steps"]),
                                 K.KWaveMedium(sound_speed=_host(q["c0"]), density=q["rho0"]), srcs, sens, q["obs"]),
                kw=dict(checkpoint_every=case["every"], data_cast=T, pml_size=q["pml"], pml_alpha=2.0, smooth_p0=False))


def run(state):
    case = state["case"]
    T = _cast(case)
    if case["kind"] == "call":
        solve = K.kspace_first_order_as if case["axisym"] else K.kspace_first_order
        out = solve(*state["args"], **state["kw"])
        return {f: out[f].astype(T, copy=False) for f in out.keys()}
    if case["kind"] == "grad":
        loss, g = K.gradient_c0(*state["args"], **state["kw"])
        return {"loss": loss, "grad": g.astype(T, copy=False)}
    sim = state["sim"]
    sim.run(case["steps"])
    out = {f: sim.sensor(f).astype(T, copy=False) for f in state["record"]}
    if case["kind"] == "steps" and case["nz"] == 1:
        out["field"] = sim.field("p").astype(T, copy=False)
    return out


def work(case):
    """Every evolving field read and written once per step, every map read once; one transform pair per derivative
    and one for the equation of state, 2.5 N log2 N each way."""
    s = 8 if case["dtype"] == "f64" else 4
    n = _sides(case)
    nd, vox = len(n), int(np.prod(n))
    logs = sum(math.log2(k) for k in n)
    if case["kind"] == "elastic":
        fields = 5 if nd == 2 else 9
        return {"bytes": vox * case["steps"] * (2 * fields + 3) * s,
                "flops": vox * case["steps"] * (2 * nd * 5 * logs + 40)}
    if case["kind"] == "grad":
        return {"bytes": vox * case["firings"] * case["steps"] * 26 * s,
                "flops": vox * case["firings"] * case["steps"] * 4 * (15 * logs + 30)}
    if case["kind"] == "firings":
        return {"bytes": vox * case["firings"] * case["steps"] * 11 * s,
                "flops": vox * case["firings"] * case["steps"] * (15 * logs + 30)}
    maps = (2 * (2 if case["maps"] == "f16" else s)) if case["het"] else 0
    return {"bytes": vox * case["steps"] * (2 * (1 + 2 * nd) * s + maps),
            "flops": vox * case["steps"] * (15 * logs + 30)}


# ---------------------------------------------------------------------------
# the same schemes in torch, Float64
# ---------------------------------------------------------------------------

def _k(n):
    return 2 * math.pi / DX * np.fft.fftfreq(n)


def _dim(nd, a):
    return nd - 1 - a


def _along(v, nd, a):
    return v.reshape([-1 if d == _dim(nd, a) else 1 for d in range(nd)])


def _derivative(n, dev):
    """f, axis, sign -> staggered spectral derivative of a (z, y, x) array."""
    nd, mult = len(n), {}
    for a in range(nd):
        k = np.abs(_k(n[a])[: n[a] // 2 + 1])
        if n[a] % 2 == 0:
            k[-1] *= -1     # the Nyquist wavenumber is negative
        for sign in (1, -1):
            mult[a, sign] = _along(torch.from_numpy(1j * k * np.exp(sign * 1j * k * DX / 2)).to(dev), nd, a)

    def d(f, a, sign):
        x = _dim(nd, a) - nd
        return torch.fft.irfft(mult[a, sign] * torch.fft.rfft(f, dim=x), n=n[a], dim=x)
    return d


def _pml(n, size, dt, nd, a, dev, staggered):
    v = np.ones(n)
    for i in range(size):
        pos = (size - i - (0.5 if staggered else 0.0)) / size
        v[i] = v[n - 1 - i] = math.exp(-2.0 * pos ** 4 * dt)
    return _along(torch.from_numpy(v).to(dev), nd, a)


def _stagger(m, nd, a):
    return (m + torch.roll(m, -1, _dim(nd, a))) / 2 if torch.is_tensor(m) else m


def _smooth(p0, n):
    out = p0.to(torch.complex128)
    for a in range(len(n)):
        i = np.arange(n[a])
        w = 0.42 - 0.5 * np.cos(2 * math.pi * i / (n[a] - 1)) + 0.08 * np.cos(4 * math.pi * i / (n[a] - 1))
        d = _dim(len(n), a)
        out = torch.fft.ifft(torch.fft.fft(out, dim=d) * _along(torch.from_numpy(np.fft.fftshift(w)).to(p0.device), len(n), a),
                             dim=d)
    return out.real * (p0.abs().max() / out.real.abs().max())


def _quantized(m):
    off = float(np.round((float(m.min()) + float(m.max())) / 2))
    return (m - off).to(torch.float16).to(torch.float64) + off


def _acoustic(q, dev, each, c0=None):
    """Runs a problem; each(t, p, u) after every step.  Returns p."""
    n, nd, dt = q["n"], len(q["n"]), q["dt"]
    c0, rho0 = q["c0"] if c0 is None else c0, q["rho0"]
    maps = torch.is_tensor(c0)
    c_ref = c0.mean() if maps else torch.tensor(c0, dtype=torch.float64, device=dev)
    D = _derivative(n, dev)
    P = [_pml(n[a], q["pml"], dt, nd, a, dev, False) for a in range(nd)]
    S = [_pml(n[a], q["pml"], dt, nd, a, dev, True) for a in range(nd)]
    k2 = sum(_along(torch.from_numpy((_k(n[a])[: n[a] // 2 + 1] if a == 0 else _k(n[a])) ** 2).to(dev), nd, a)
             for a in range(nd))
    k = torch.sqrt(k2)
    arg = c_ref * k * dt / 2
    kappa = torch.where(k == 0, torch.ones_like(arg), torch.sin(arg) / torch.where(k == 0, torch.ones_like(arg), arg))
    n1 = n2 = None
    if q["absorb"]:
        al, y = q["absorb"]
        a_np = al * (1e-2 / (20 * math.log10(math.e))) * (2 * math.pi * 1e6) ** (-y)
        n1 = -2 * a_np * c_ref ** (y - 1) * k ** y
        n2 = None if maps else 2 * a_np * c_ref ** (y - 1) * math.tan(math.pi * y / 2) * k ** (y - 1)
    rsg = [_stagger(rho0, nd, a) for a in range(nd)]
    shape = list(reversed(n))
    zero = torch.zeros(shape, dtype=torch.float64, device=dev)
    p, u, r = zero, [zero] * nd, [zero] * nd
    before = zero
    if q["p0"] is not None and q["tr"] is None:
        p = _smooth(q["p0"], n) if q["smooth"] else q["p0"]
        r = [p / (nd * c0 ** 2)] * nd
        u = [-dt / (2 * rsg[a]) * D(p, a, 1) for a in range(nd)]
    at = lambda i: torch.from_numpy(np.asarray(i)).to(dev)  # noqa: E731
    col = lambda s, t: torch.from_numpy(np.ascontiguousarray(s[:, min(t, s.shape[1]) - 1])).to(dev)  # noqa: E731
    put = lambda f, i, v: f.reshape(-1).index_put((i,), v, accumulate=True).reshape(shape)  # noqa: E731
    c_at = lambda i: c0.reshape(-1)[i] if maps else c0  # noqa: E731
    if q["p"]:
        pi = at(q["p"][0])
        psig = torch.from_numpy(q["p"][1]).to(dev) / (nd * (c_at(pi) ** 2)[:, None] if maps else nd * c0 ** 2)
    if q["u"]:
        ui = at(q["u"][0])
    if q["tr"] is not None:
        ti = torch.nonzero(q["mask"].reshape(-1)).reshape(-1)
    if q["axisym"]:
        rad = np.abs((np.arange(n[1]) - (n[1] - 1) / 2) * DX)
        rad[rad == 0] = DX / 2
        inv_r = _along(torch.from_numpy(1.0 / rad).to(dev), nd, 1)
    eos = lambda x: x if q["bona"] is None else x * (1 + q["bona"] / 2 * x / rho0)  # noqa: E731
    dims = list(range(nd))
    for t in range(1, q["steps"] + 1):
        if q["tr"] is not None:
            v = col(q["tr"], q["steps"] - t + 1) / (nd * c_at(ti) ** 2)
            r = [x.reshape(-1).index_put((ti,), v).reshape(shape) for x in r]
        u = [S[a] * (S[a] * u[a] - dt / rsg[a] * D(p, a, 1)) for a in range(nd)]
        if q["u"]:
            u = [put(u[a], ui, col(q["u"][1][a], t)) for a in range(nd)]
        du = [D(u[a], a, -1) for a in range(nd)]
        if q["axisym"]:
            du[1] = du[1] + u[1] * inv_r
        r = [P[a] * (P[a] * r[a] - dt * rho0 * du[a]) for a in range(nd)]
        if q["p"]:
            r = [put(x, pi, psig[:, min(t, psig.shape[1]) - 1]) for x in r]
        tot = sum(r)
        f = torch.fft.rfftn(eos(tot) * c0 ** 2, dim=dims)
        if n1 is not None:
            f = f * (1 + n1)
        if n2 is not None:
            # no value at k = 0: the dispersion operator's k^(y-1) is 0 there for y > 1
            f = f - n2 * torch.fft.rfftn((eos(tot) - eos(before)) / dt * c0 ** 2, dim=dims)
        p = torch.fft.irfftn(kappa * f, s=shape, dim=dims)
        before = tot
        each(t, p, u)
    return p


def _sensed(q, run):
    """Sensor data as recorded by run(each)."""
    i = torch.nonzero(q["mask"].reshape(-1)).reshape(-1)
    got = {}

    def each(t, p, u):
        v = p.reshape(-1)[i]
        for f in q["record"]:
            if f == "p":
                got.setdefault("p", []).append(v)
            elif f == "p_final":
                got[f] = v
            elif f == "p_max":
                got[f] = v if f not in got else torch.maximum(got[f], v)
            elif f == "p_min":
                got[f] = v if f not in got else torch.minimum(got[f], v)
            else:
                w = sum(x.reshape(-1)[i] ** 2 for x in u)
                if f == "u_rms":
                    got[f] = w if f not in got else got[f] + w
                else:
                    got[f] = torch.sqrt(w) if f not in got else torch.maximum(got[f], torch.sqrt(w))
    p = run(each)
    if "u_rms" in got:
        got["u_rms"] = torch.sqrt(got["u_rms"] / q["steps"])
    if "p" in got:
        got["p"] = torch.stack(got["p"], dim=1)
    if q.get("tr") is not None:
        got["p_final"] = p.reshape(-1)
    return {f: v.cpu().numpy() for f, v in got.items()}, p


def _elastic(q, dev, each):
    n, nd, dt = q["n"], len(q["n"]), q["dt"]
    D = _derivative(n, dev)
    P = [_pml(n[a], q["pml"], dt, nd, a, dev, False) for a in range(nd)]
    S = [_pml(n[a], q["pml"], dt, nd, a, dev, True) for a in range(nd)]
    lam, mu = q["rho0"] * (q["cp"] ** 2 - 2 * q["cs"] ** 2), q["rho0"] * q["cs"] ** 2
    rsg = [_stagger(q["rho0"], nd, a) for a in range(nd)]
    zero = torch.zeros_like(q["p0"])
    v = [zero] * nd
    s = {(a, b): -q["p0"] if a == b else zero for a in range(nd) for b in range(a, nd)}
    for t in range(1, q["steps"] + 1):
        for a in range(nd):
            v[a] = S[a] * (S[a] * v[a] + dt / rsg[a] * sum(D(s[min(a, b), max(a, b)], b, 1) for b in range(nd)))
        dv = [[D(v[a], b, -1) for b in range(nd)] for a in range(nd)]
        div = sum(dv[a][a] for a in range(nd))
        for a in range(nd):
            s[a, a] = P[a] * (P[a] * s[a, a] + dt * (lam * div + 2 * mu * dv[a][a]))
            for b in range(a + 1, nd):
                s[a, b] = P[a] * P[b] * (s[a, b] + dt * mu * (dv[a][b] + dv[b][a]))
        p = -sum(s[a, a] for a in range(nd)) / nd
        each(t, p, v)
    return p


def exact(case, seed):
    dev = _device()
    if case["kind"] == "elastic":
        q = _elastic_problem(case, seed)
        return _sensed(q, lambda each: _elastic(q, dev, each))[0]
    if case["kind"] == "firings":
        each = [_sensed(q, lambda f, q=q: _acoustic(q, dev, f))[0] for q in _firing_problems(case, seed)]
        return {f: np.concatenate([o[f] for o in each]) for f in each[0]}
    if case["kind"] == "grad":
        q = _ring_problem(case, seed)
        q.update(absorb=None, bona=None, p0=None, u=None, tr=None, axisym=False, smooth=False)
        c0 = q["c0"].clone().requires_grad_(True)
        ring = torch.from_numpy(q["ring"]).to(dev)
        loss = 0.0
        for f, obs in zip(q["fire"], q["obs"]):
            one = dict(q, p=(np.array([f]), q["burst"][None, :]))
            o, terms = torch.from_numpy(obs).to(dev), []
            _acoustic(one, dev, lambda t, p, u: terms.append(((p.reshape(-1)[ring] - o[:, t - 1]) ** 2).sum()), c0)
            part = 0.5 * sum(terms)
            part.backward()
            loss += float(part.detach())
        return {"loss": np.float64(loss), "grad": c0.grad.cpu().numpy().T}
    q = _problem(case, seed)
    if case["maps"] == "f16":
        q["c0"], q["rho0"] = _quantized(q["c0"]), _quantized(q["rho0"])
    out, p = _sensed(q, lambda each: _acoustic(q, dev, each))
    if case["kind"] == "steps" and case["nz"] == 1:
        out["field"] = p.cpu().numpy().T
    return out
