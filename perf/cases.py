"""Performance cases of the framework: the work its users have it do, through its public entry points.

``listed()`` gives the fixed cases, ``draw(rng)`` more of the same ranges.  A
case is a dict of plain values; ``prepare`` makes its inputs and the plan,
network or buffers a program keeps, ``run`` is one pass, ``work`` the bytes
and operations that pass cannot do without, ``exact`` the same outputs from
plain numpy/torch in 64 bits where that takes seconds.

Kinds of case:

``step``   one meteorological step through the drop-in calls on host data
           (``vertical_profiles`` then ``steady_state_transport_solver``)
``solve``  one device-resident solve (``solve_device``): a footprint, or the
           dispersion of a surface flux at several levels
``batch``  towers x timesteps in one plan (``FootprintBatch.run``), one grid
           for all or a mix of grids with arbitrary halos
``fft2``   the 2-D FFT drop-in on device tensors
``serve``  footprints served by the learned surrogate with its FP64 gate
``train``  one gradient step of the surrogate on freshly solved points
``km01``   Kormann-Meixner footprints of a series of measurements
"""

import math
import random

import numpy as np
import torch

KARMAN = 0.4


# ------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: one half-hour of a tower through the reference's own two functions,
        # grid, domain and single precision of its regression fixtures (padded 960 x 384)
        dict(name="step_64x128", kind="step", nx=64, ny=128, xmax=100.0, ymax=700.0, n=16),
        # one production footprint on device data: 512^2 modes, 2 km, column to 100 m
        dict(name="footprint_512", kind="solve", footprint=True, nx=512, ny=512, xmax=2000.0, ymax=2000.0, n=26,
             height=100.0, halo=None, nlev=1, precision="double", fast=False),
        # dispersion of a surface flux on the production grid, nine output levels up to the measurement height
        dict(name="plume_512_9lev", kind="solve", footprint=False, nx=512, ny=512, xmax=2000.0, ymax=2000.0, n=26,
             height=None, halo=None, nlev=9, precision="double", fast=False),
        # dispersion on a grid and halo nobody tuned for (padded 486 x 364), single precision output
        dict(name="plume_250x186_f32", kind="solve", footprint=False, nx=250, ny=186, xmax=1100.0, ymax=900.0, n=20,
             height=None, halo=520.0, nlev=4, precision="single", fast=False),
        # serving scale: 128 footprints of 512^2 modes x 64 steps in one plan (the benchmark's batch)
        dict(name="batch_128x512", kind="batch", count=128, nx=512, ny=512, xmax=2000.0, ymax=2000.0, n=26,
             height=100.0, halo=None, mix=0, precision="double", fast=False),
        # two days of half-hours on a small grid
        dict(name="batch_96x128", kind="batch", count=96, nx=128, ny=128, xmax=1000.0, ymax=1000.0, n=19,
             height=None, halo=None, mix=0, precision="single", fast=False),
        # a tower network: every tower its own grid, domain and halo, odd sizes among them
        dict(name="batch_mixed_32", kind="batch", count=32, nx=300, ny=240, xmax=1200.0, ymax=1000.0, n=20,
             height=None, halo=None, mix=11, precision="double", fast=False),
        # the FFT backend on a large power of two, complex128 forward
        dict(name="fft2_2048", kind="fft2", batch=2, n0=2048, n1=2048, single=False, inverse=False),
        # and on a ragged stack of complex64 fields, inverse
        dict(name="ifft2_1001x1386_c64", kind="fft2", batch=4, n0=1001, n1=1386, single=True, inverse=True),
        # the surrogate serving a batch of production footprints
        dict(name="serve_24x512", kind="serve", count=24, nx=512, tol=1e-3),
        # one training step of the surrogate at its own batch size
        dict(name="train_65536", kind="train", points=65536, nmet=256),
        # a day of half-hourly Kormann-Meixner footprints on a 2 m grid
        dict(name="km01_48x300", kind="km01", count=48, nx=300, ny=300, res=2.0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["step", "solve", "solve", "batch", "batch", "fft2", "serve", "train", "km01"])
    if kind == "step":
        return dict(kind=kind, nx=2 * _log_int(rng, 16, 80), ny=2 * _log_int(rng, 16, 80),
                    xmax=round(rng.uniform(100.0, 800.0), 1), ymax=round(rng.uniform(100.0, 800.0), 1),
                    n=rng.randint(10, 32))
    if kind == "solve":
        fp = rng.random() < 0.5
        nx, ny = _log_int(rng, 48, 512), _log_int(rng, 48, 512)
        if not fp:  # a dispersion solve takes even grids (as its modes are)
            nx, ny = nx + nx % 2, ny + ny % 2
        d = round(rng.uniform(2.5, 6.0), 2)
        return dict(kind=kind, footprint=fp, nx=nx, ny=ny, xmax=round(d * nx, 1), ymax=round(d * ny, 1),
                    n=rng.randint(12, 32), height=None,
                    halo=None if rng.random() < 0.5 else round(d * rng.uniform(0.4, 1.1) * max(nx, ny), 1),
                    nlev=1 if fp else rng.randint(1, 9), precision=rng.choice(["single", "double"]),
                    fast=fp and rng.random() < 0.25)
    if kind == "batch":
        nx, ny = _log_int(rng, 48, 512), _log_int(rng, 48, 512)
        count = _log_int(rng, 2, max(2, min(128, (1 << 23) // (nx * ny))))
        d = round(rng.uniform(2.5, 6.0), 2)
        return dict(kind=kind, count=count, nx=nx, ny=ny, xmax=round(d * nx, 1), ymax=round(d * ny, 1),
                    n=rng.randint(12, 32), height=None,
                    halo=None if rng.random() < 0.5 else round(d * rng.uniform(0.4, 1.1) * max(nx, ny), 1),
                    mix=rng.choice([0, rng.randint(1, 999)]), precision=rng.choice(["single", "double"]),
                    fast=rng.random() < 0.2)
    if kind == "fft2":
        n0, n1 = _log_int(rng, 48, 3000), _log_int(rng, 48, 3000)
        if rng.random() < 0.5:
            n0, n1 = 8 * max(1, n0 // 8), 8 * max(1, n1 // 8)
        return dict(kind=kind, batch=_log_int(rng, 1, max(1, min(64, (1 << 23) // (n0 * n1)))), n0=n0, n1=n1,
                    single=rng.random() < 0.5, inverse=rng.random() < 0.5)
    if kind == "serve":
        return dict(kind=kind, count=_log_int(rng, 2, 24), nx=2 * _log_int(rng, 64, 256), tol=1e-3)
    if kind == "train":
        return dict(kind=kind, points=256 * _log_int(rng, 16, 256), nmet=_log_int(rng, 16, 512))
    return dict(kind=kind, count=_log_int(rng, 2, 48), nx=_log_int(rng, 60, 300), ny=_log_int(rng, 60, 300),
                res=float(rng.choice([1, 2, 5])))


# ------------------------------------------------------------------ inputs
def _psi(x):
    """Businger-Dyer psi(z/L)."""
    x = np.asarray(x, dtype=np.float64)
    xi = np.maximum(1.0 - 16.0 * x, 0.0) ** 0.25
    unstable = -2.0 * np.log(0.5 * (1.0 + xi)) - np.log(0.5 * (1.0 + xi * xi)) + 2.0 * np.arctan(xi) - 0.5 * np.pi
    return np.where(x > 0.0, 5.0 * x, unstable)


def _mets(count, seed, zm=None):
    """Seeded meteorology: friction velocity, Obukhov length of either sign,
    roughness, direction, and the wind speed the log law gives with them."""
    r = random.Random(1000003 * seed + 17)
    out = []
    for _ in range(count):
        h = zm if zm is not None else r.uniform(6.0, 20.0)
        us, z0 = r.uniform(0.2, 0.6), h * math.exp(r.uniform(math.log(0.003), math.log(0.02)))
        mol = -math.exp(r.uniform(math.log(20.0), math.log(300.0))) if r.random() < 0.6 else r.uniform(60.0, 400.0)
        speed = us / KARMAN * (math.log(h / z0) + float(_psi(h / mol)))
        wd = math.radians(r.uniform(0.0, 360.0))
        out.append(dict(meas_height=h, ustar=us, mol=mol, wind=(-speed * math.sin(wd), -speed * math.cos(wd))))
    return out


def _geometries(case):
    """(nx, ny, xmax, ymax, halo) of each footprint of a batch; a mix varies
    every one of them by its own generator, not by the seed of the inputs."""
    if not case["mix"]:
        return [(case["nx"], case["ny"], case["xmax"], case["ymax"], case["halo"])] * case["count"]
    r = random.Random(case["mix"])
    out = []
    for _ in range(case["count"]):
        s, t = r.uniform(0.4, 1.0), r.uniform(0.4, 1.0)
        nx, ny = max(16, int(s * case["nx"])), max(16, int(t * case["ny"]))
        dx, dy = case["xmax"] / case["nx"], case["ymax"] / case["ny"]
        halo = None if r.random() < 0.4 else r.uniform(0.4, 1.0) * max(nx * dx, ny * dy)
        out.append((nx, ny, nx * dx, ny * dy, halo))
    return out


def _even(n):
    return n - n % 2


def _source(nx, ny, xmax, ymax, seed):
    """Surface flux: twelve seeded Gaussian patches (float64, on the host)."""
    r = random.Random(7919 * seed + 3)
    x, y = np.arange(nx) * (xmax / nx), np.arange(ny) * (ymax / ny)
    q = np.zeros((ny, nx))
    for _ in range(12):
        cx, cy = r.uniform(0.1, 0.9) * xmax, r.uniform(0.1, 0.9) * ymax
        s = r.uniform(0.02, 0.08) * max(xmax, ymax)
        q += r.uniform(0.5, 2.0) * np.outer(np.exp(-((y - cy) ** 2) / (2 * s * s)),
                                            np.exp(-((x - cx) ** 2) / (2 * s * s)))
    return q


def _levels(case):
    return sorted({int(round(v)) for v in np.linspace(0 if case["nlev"] > 1 else case["n"], case["n"], case["nlev"])})


def _specs(case, seed):
    from bldfm_amd.batch import FootprintSpec

    zm = 15.0 if case["height"] else None
    return [FootprintSpec(nx=nx, ny=ny, domain=(xm, ym), modes=(_even(nx), _even(ny)), meas_pt=(0.5 * xm, 0.5 * ym),
                          n=case["n"], domain_height=case["height"], halo=halo, **m)
            for (nx, ny, xm, ym, halo), m in zip(_geometries(case), _mets(case["count"], seed, zm))]


def _km01_records(case, seed):
    r = random.Random(104729 * seed + 5)
    half_x, half_y = 0.5 * case["nx"] * case["res"], 0.5 * case["ny"] * case["res"]
    out = []
    for m in _mets(case["count"], seed):
        ws = math.hypot(*m["wind"])
        z0 = m["meas_height"] * math.exp(float(_psi(m["meas_height"] / m["mol"])) - KARMAN * ws / m["ustar"])
        out.append(dict(zm=m["meas_height"], z0=z0, ws=ws, ustar=m["ustar"], mo_len=m["mol"],
                        sigma_v=r.uniform(0.4, 1.2), grid_domain=(-half_x, half_x, -half_y, half_y),
                        grid_res=case["res"], mxy=(0.0, 0.0), wd=r.uniform(0.0, 360.0)))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return dict(case=case, met=_mets(1, seed, 10.0)[0], q0=np.zeros((case["ny"], case["nx"])))
    if kind == "solve":
        from bldfm_amd.pbl_model import vertical_profiles

        met = _mets(1, seed, 15.0)[0]
        z, prof = vertical_profiles(case["n"], closure="MOST", domain_height=case["height"], **met)
        q0 = (np.zeros((case["ny"], case["nx"])) if case["footprint"]
              else _source(case["nx"], case["ny"], case["xmax"], case["ymax"], seed))
        return dict(case=case, z=z, prof=prof, q0=torch.as_tensor(q0, device="cuda"), levels=_levels(case))
    if kind == "batch":
        from bldfm_amd.batch import FootprintBatch

        return dict(case=case, fb=FootprintBatch(_specs(case, seed), precision=case["precision"], fast=case["fast"]))
    if kind == "fft2":
        g = torch.Generator(device="cuda").manual_seed(seed)
        dt = torch.complex64 if case["single"] else torch.complex128
        return dict(case=case, x=torch.randn(case["batch"], case["n0"], case["n1"], dtype=dt, device="cuda", generator=g))
    if kind == "serve":
        from bldfm_amd import surrogate
        from bldfm_amd.batch import FootprintBatch, FootprintSpec

        net = surrogate.SurrogateNet.load(surrogate.DEFAULT_CHECKPOINT)
        h = net.hull
        ext = 2000.0 * case["nx"] / 512
        specs = [FootprintSpec(nx=case["nx"], ny=case["nx"], domain=(ext, ext), modes=(case["nx"], case["nx"]),
                               meas_pt=(0.5 * ext, 0.5 * ext), n=h.n, closure=h.closure,
                               domain_height=h.top_ratio * m["meas_height"], **m)
                 for m in _mets(case["count"], seed, 15.0)]
        return dict(case=case, fb=FootprintBatch(specs, precision="double", surrogate=net, tol=case["tol"]), net=net)
    if kind == "train":
        from bldfm_amd import surrogate

        net = surrogate.SurrogateNet.load(surrogate.DEFAULT_CHECKPOINT)
        ms = surrogate.MetSet(surrogate.sample_met(case["nmet"], seed, net.hull), net.hull)
        g = torch.Generator(device="cuda").manual_seed(seed)
        mids, kxy = net.sample_points(ms, case["points"] // surrogate.TRANSFER_BLOCK, g)
        ws = torch.empty(case["points"] * net.bytes_per_point, dtype=torch.uint8, device="cuda")
        return dict(case=case, net=net, ms=ms, mids=mids, kxy=kxy, ws=ws)
    return dict(case=case, records=_km01_records(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        from bldfm_amd.pbl_model import vertical_profiles
        from bldfm_amd.solver import steady_state_transport_solver

        z, prof = vertical_profiles(case["n"], **state["met"])
        dom = (case["xmax"], case["ymax"])
        return steady_state_transport_solver(state["q0"], z, prof, dom, case["n"], modes=(case["nx"], case["ny"]),
                                             meas_pt=(0.5 * dom[0], 0.0), footprint=True)
    if kind == "solve":
        from bldfm_amd.solver import solve_device

        dom = (case["xmax"], case["ymax"])
        conc, flx, _ = solve_device(state["q0"], state["z"], state["prof"], dom, state["levels"],
                                    modes=(_even(case["nx"]), _even(case["ny"])),
                                    meas_pt=(0.5 * dom[0], 0.5 * dom[1]) if case["footprint"] else (0.0, 0.0),
                                    footprint=case["footprint"], halo=case["halo"], precision=case["precision"],
                                    fast=case["fast"])
        return conc, flx
    if kind in ("batch", "serve"):
        state["fb"].run()
        return state["fb"].conc, state["fb"].flx
    if kind == "fft2":
        from bldfm_amd import fft_manager

        return fft_manager.ifft2(state["x"], norm="ortho") if case["inverse"] else fft_manager.fft2(state["x"])
    if kind == "train":
        net = state["net"]
        g = state["ms"].solve(state["mids"], state["kxy"])
        net.grad.zero_()
        loss = net.grad_step(state["ms"], state["mids"].repeat_interleave(2), state["kxy"], g, ws=state["ws"])
        return dict(g=g, loss=loss, grad=net.grad)
    from bldfm_amd.ffm_kormann_meixner import estimate_footprints

    return [f for _, _, f in estimate_footprints(state["records"])]


# -------------------------------------------------------------------- work
def _padded(nx, ny, xmax, ymax, halo):
    halo = max(xmax, ymax) if halo is None else halo
    return nx + 2 * int(halo / (xmax / nx)), ny + 2 * int(halo / (ymax / ny))


def _steps(n, zm, height):
    """Vertical intervals of the log-stretched grid, about: n below zm, the
    top where 1 - e^{-z/(2 zm)} has grown by height's share."""
    top = 2.0 * zm if height is None else height
    return int(n * (1.0 - math.exp(-top / (2.0 * zm))) / (1.0 - math.exp(-0.5)))


def _solve_work(nx, ny, xmax, ymax, halo, steps, nlev, footprint, out_bytes):
    """One solve: its outputs written once (its flux read once), 80 operations
    per half-plane mode and vertical step, and per output level the
    transforms of the retained band onto the cropped grid at 5 N log2 N."""
    nxe, nye = _padded(nx, ny, xmax, ymax, halo)
    mx, my = min(_even(nx), nxe), min(_even(ny), nye)
    fft = 5.0 * (mx * nye * math.log2(nye) + ny * nxe * math.log2(nxe))
    return dict(bytes=2.0 * nlev * nx * ny * out_bytes + (0 if footprint else 8.0 * nx * ny),
                flops=80.0 * 0.5 * mx * my * steps + fft * nlev + (0 if footprint else 0.5 * fft))


def work(case):
    kind = case["kind"]
    if kind == "step":
        w = _solve_work(case["nx"], case["ny"], case["xmax"], case["ymax"], None, _steps(case["n"], 10.0, None), 1, True, 8)
        return w
    if kind == "solve":
        f32 = case["precision"] == "single" and not case["footprint"]
        return _solve_work(case["nx"], case["ny"], case["xmax"], case["ymax"], case["halo"],
                           _steps(case["n"], 15.0, case["height"]), len(_levels(case)), case["footprint"],
                           4 if f32 else 8)
    if kind == "batch":
        w = [_solve_work(*g, _steps(case["n"], 15.0, case["height"]), 1, True, 8) for g in _geometries(case)]
        return dict(bytes=sum(v["bytes"] for v in w), flops=sum(v["flops"] for v in w))
    if kind == "fft2":
        n = case["batch"] * case["n0"] * case["n1"]
        return dict(bytes=2.0 * n * (8 if case["single"] else 16), flops=5.0 * n * math.log2(case["n0"] * case["n1"]))
    if kind == "serve":  # the network on every half-plane mode, 1 % of them solved, the transforms
        n = case["nx"]
        w = _solve_work(n, n, 1.0, 1.0, None, 0, 1, True, 8)
        return dict(bytes=case["count"] * w["bytes"],
                    flops=case["count"] * (w["flops"] + 0.5 * n * n * (573440.0 + 0.01 * 80 * 64)))
    if kind == "train":  # forward, backward and weight gradients; the FP64 targets at 64 steps
        p = case["points"]
        return dict(bytes=p * 32.0 + 4.0 * 290000, flops=p * (3 * 573440.0 + 80 * 64))
    cells = case["count"] * case["nx"] * case["ny"]
    return dict(bytes=8.0 * cells, flops=100.0 * cells)


# ------------------------------------------------------------- exact values
def _profiles_exact(n, met, height):
    """MOST profiles on the log-stretched grid (numpy, float64)."""
    zm, us, mol = met["meas_height"], met["ustar"], met["mol"]
    um, vm = met["wind"]
    speed = np.sqrt(um**2 + vm**2)
    z0 = zm * np.exp(-KARMAN * speed / us + float(_psi(zm / mol)))
    h, top = 2.0 * zm, 2.0 * zm if height is None else height
    bb = zm / (np.exp(-z0 / h) - np.exp(-zm / h))
    aa = bb * np.exp(-z0 / h)
    dzeta = zm / n
    zeta = np.arange(0.0, float(aa - bb * np.exp(-top / h)) + dzeta, dzeta)
    z = -h * np.log(-(zeta - aa) / bb)
    absu = us / KARMAN * (np.log(z / z0) + _psi(z / mol))
    x = z / mol
    phi = np.where(x > 0.0, 1.0 + 5.0 * x, np.maximum(1.0 - 16.0 * x, 1e-300) ** -0.5)
    K = KARMAN * us * z / phi
    return z, (um / speed * absu, vm / speed * absu, K, K, K)


def _march_exact(z, prof, lx, ly, q0, levels):
    """Both initial-value problems over every mode and the shooting
    combination: p^ and q^ at ``levels`` (a list), complex arrays like lx."""
    u, v, Kx, Ky, Kz = prof

    def mul(a, b):  # a complex product rounds its products and sums one by one
        return a[0] * b[0] - a[1] * b[1], a[0] * b[1] + a[1] * b[0]

    one, zero = np.ones_like(lx), np.zeros_like(lx)
    st = [(one, zero), (zero, zero), (zero, zero), (np.real(q0) * one, np.imag(q0) * one)]
    lx2, ly2 = lx * lx, ly * ly
    snap = {}
    for i in range(len(z)):
        if i in levels:
            snap[i] = [a + 1j * b for a, b in st]
        if i == len(z) - 1:
            break
        ki, h = 1.0 / Kz[i], z[i + 1] - z[i]
        h2, h3 = h * h, h * (h * h)
        T = (-(Kx[i] * lx2 + Ky[i] * ly2), -(u[i] * lx + v[i] * ly))
        sa, sb, sc = 0.5 * ki, (1.0 / 6.0) * (ki * ki), (1.0 / 6.0) * ki
        a = (1.0 - sa * T[0] * h2, -(sa * T[1] * h2))
        b = (-ki * h - sb * T[0] * h3, -(sb * T[1] * h3))
        t2 = mul(T, T)
        c = (T[0] * h - sc * t2[0] * h3, T[1] * h - sc * t2[1] * h3)
        new = []
        for p, q in ((st[0], st[1]), (st[2], st[3])):
            ap, bq, cp, aq = mul(a, p), mul(b, q), mul(c, p), mul(a, q)
            new += [(ap[0] + bq[0], ap[1] + bq[1]), (cp[0] + aq[0], cp[1] + aq[1])]
        st = new
    p1, q1, p2, q2 = (a + 1j * b for a, b in st)
    ki = 1.0 / Kz[-1]
    lam = np.sqrt(Kx[-1] * ki * lx2 + Ky[-1] * ki * ly2 + 1j * (u[-1] * ki * lx + v[-1] * ki * ly))
    with np.errstate(invalid="ignore", divide="ignore"):
        al = -(q2 - Kz[-1] * lam * p2) / (q1 - Kz[-1] * lam * p1)
    return [(al * snap[i][0] + snap[i][2], al * snap[i][1] + snap[i][3]) for i in levels]


def _solve_exact(nx, ny, xmax, ymax, halo, modes, meas_pt, footprint, q, z, prof, levels):
    """(conc, flx), each (levels, ny, nx), by numpy's FFT on the padded grid."""
    halo = max(xmax, ymax) if halo is None else halo
    dx, dy = xmax / nx, ymax / ny
    px, py = int(halo / dx), int(halo / dy)
    nxe, nye = nx + 2 * px, ny + 2 * py
    mx, my = modes if modes[0] <= nxe and modes[1] <= nye else (nxe, nye)
    Lx, Ly = mx + 2 * ((nxe - mx) // 2), my + 2 * ((nye - my) // 2)
    fx, fy = (np.fft.fftfreq(m, d=1.0 / m) for m in (mx, my))
    lx, ly = np.meshgrid(2.0 * np.pi / dx / nxe * fx, 2.0 * np.pi / dy / nye * fy)
    ix, iy = np.rint(fx).astype(int) % Lx, np.rint(fy).astype(int) % Ly
    if footprint:
        q0 = np.full((my, mx), (1.0 / nxe) * (1.0 / nye), dtype=complex)
    else:
        pad = np.zeros((nye, nxe))
        pad[py:py + ny, px:px + nx] = q
        q0 = np.fft.fft2(pad, norm="forward")[np.ix_(iy, ix)]
    got = _march_exact(z, prof, lx, ly, q0, levels)
    p00 = 0.0
    at0 = {}
    for i in range(len(z)):
        at0[i] = p00
        if i < len(z) - 1:
            p00 = p00 - q0[0, 0] * (z[i + 1] - z[i]) * (0.5 / prof[4][i] + 0.5 / prof[4][i + 1])
    sh = np.exp(1j * (lx * (meas_pt[0] + halo) + ly * (meas_pt[1] + halo))) if footprint else 1.0
    # the output keeps what the inverse transform of Lx x Ly points leaves of the crop
    nxo, nyo = min(nxe - px, Lx) - px, min(nye - py, Ly) - py
    out = np.empty((2, len(levels), nyo, nxo))
    for k, (i, (p, f)) in enumerate(zip(levels, got)):
        p[0, 0], f[0, 0] = at0[i], q0[0, 0]
        for m, X in enumerate((p * sh, f * sh)):
            full = np.zeros((Ly, Lx), dtype=complex)
            full[np.ix_(iy, ix)] = X
            r = np.fft.fft2(full) if footprint else np.fft.ifft2(full, norm="forward")
            out[m, k] = r.real[py:py + nyo, px:px + nxo]
    return out[0], out[1]


def _km01_exact(r):
    k, zm, L = KARMAN, r["zm"], r["mo_len"]
    if L < 0:
        a = 1.0 - 16.0 * zm / L
        phim, phic, n = a**-0.25, a**-0.5, (1.0 - 24.0 * zm / L) / a
    else:
        phim = phic = 1.0 + 5.0 * zm / L
        n = 1.0 / phim
    m = r["ustar"] * phim / (k * r["ws"])
    kappa = k * zm * r["ustar"] / (phic * zm**n)
    U = r["ustar"] * (math.log(zm / r["z0"]) + float(_psi(zm / L))) / (k * zm**m)
    s = 2.0 + m - n
    mu, Xi = (1.0 + m) / s, U * zm**s / (s * s * kappa)
    A = U / (math.gamma(1.0 / s) * r["sigma_v"]) * (kappa * s * s / U) ** (m / s)
    x0, x1, y0, y1 = r["grid_domain"]
    gx, gy = np.meshgrid(np.arange(x0 + 0.5 * r["grid_res"], x1, r["grid_res"]),
                         np.arange(y1 - 0.5 * r["grid_res"], y0, -r["grid_res"]))
    rho, th = np.hypot(gx, gy), np.arctan2(gy, gx) + np.deg2rad(r["wd"]) - 0.5 * np.pi
    x, y = rho * np.cos(th), rho * np.sin(th)
    f = np.zeros_like(x)
    up = x > 0.0
    xu, yu = x[up], y[up]
    f[up] = (r["grid_res"] ** 2 / math.sqrt(2.0 * math.pi) * Xi**mu * A * xu ** (m / s - 2.0 - mu)
             * np.exp(-Xi / xu - 0.5 * (math.gamma(mu) * yu * A * xu ** (m / s - 1.0)) ** 2))
    return f


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        met = _mets(1, seed, 10.0)[0]
        z, prof = _profiles_exact(case["n"], met, None)
        dom = (case["xmax"], case["ymax"])
        c, f = _solve_exact(case["nx"], case["ny"], *dom, None, (case["nx"], case["ny"]), (0.5 * dom[0], 0.0), True,
                            None, z, prof, [case["n"]])
        X, Y = np.meshgrid(np.arange(case["nx"]) * (dom[0] / case["nx"]), np.arange(case["ny"]) * (dom[1] / case["ny"]))
        return (X, Y, np.full(X.shape, z[case["n"]])), c[0], f[0]
    if kind == "solve":
        z, prof = _profiles_exact(case["n"], _mets(1, seed, 15.0)[0], case["height"])
        dom = (case["xmax"], case["ymax"])
        q = None if case["footprint"] else _source(case["nx"], case["ny"], *dom, seed)
        return _solve_exact(case["nx"], case["ny"], *dom, case["halo"], (_even(case["nx"]), _even(case["ny"])),
                            (0.5 * dom[0], 0.5 * dom[1]), case["footprint"], q, z, prof, _levels(case))
    if kind == "batch":
        geo = _geometries(case)
        # about 1 us a mode and step in numpy: larger batches take over 20 seconds
        if sum(g[0] * g[1] for g in geo) * _steps(case["n"], 15.0, case["height"]) > 6e7:
            return None
        conc, flx = [], []
        for (nx, ny, xm, ym, halo), m in zip(geo, _mets(case["count"], seed, 15.0 if case["height"] else None)):
            z, prof = _profiles_exact(case["n"], m, case["height"])
            c, f = _solve_exact(nx, ny, xm, ym, halo, (_even(nx), _even(ny)), (0.5 * xm, 0.5 * ym), True, None, z,
                                prof, [case["n"]])
            conc.append(c.ravel())
            flx.append(f.ravel())
        return np.concatenate(conc), np.concatenate(flx)
    if kind == "fft2":
        x = prepare(case, seed)["x"].cpu().numpy().astype(np.complex128)
        return np.fft.ifft2(x, norm="ortho") if case["inverse"] else np.fft.fft2(x)
    if kind == "km01":
        return [_km01_exact(r) for r in _km01_records(case, seed)]
    # serve, train: the outputs are those of a bf16 network, whose products in 64 bits would need the
    # package's own features and checkpoint; they are held to the start's outputs
    return None
