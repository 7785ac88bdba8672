"""The work that users of this framework have it do, as measurable cases.

Four kinds of case, each through public entry points:

* ``mirror``: one loop body of a driver written against the Melvin-style
  classes (``Simulation``, ``Variable``, ``Integrator``, ...), as the
  reference's examples write it: the drop-in use.
* ``transforms``: ``SpectralTransformer.to_spectral`` and ``to_physical``
  on their own, as drivers use them for initial conditions and output.
* ``fused``: ``fused.Batch`` steps of one or many fully spectral simulations.
* ``fdz``: ``fdz.FdzBatch`` steps of one or many Rayleigh-Benard simulations.

``listed()`` gives the named cases and ``draw(rng)`` more of the same
ranges; ``prepare`` builds a case's simulations from a seed, ``run`` makes
one pass, ``work`` counts the bytes and operations a pass cannot do
without, and ``exact`` restates the pass in 64-bit torch / numpy.
"""
import math

import numpy as np
import torch

import __graft_entry__

melvin = __graft_entry__.load_package()
fdz, fused, utility = melvin.fdz, melvin.fused, melvin.utility

TWO_PI = 2.0 * math.pi
NFIELD = {"vortex": 1, "ink": 2, "ddc": 3, "mhd": 2}


def listed():
    return [
        # the drop-in user's Taylor-Green loop: small arrays, many calls
        {"name": "mirror_tgv_256_f64", "kind": "mirror", "flow": "vortex", "nx": 256, "nz": 256,
         "dtype": "f64", "ab": 2, "fd": 2},
        # the drop-in user's Kelvin-Helmholtz loop with ink at the size of the precision study
        {"name": "mirror_kh_1024_f64", "kind": "mirror", "flow": "ink", "nx": 1024, "nz": 1024,
         "dtype": "f64", "ab": 4, "fd": 2},
        # the drop-in user's Rayleigh-Benard loop (Fourier x, FD z), odd nz
        {"name": "mirror_rbc_1024x513_f64", "kind": "mirror", "flow": "rbc", "nx": 1024, "nz": 513,
         "dtype": "f64", "ab": 2, "fd": 2},
        # transforms alone, both directions, single precision, not square
        {"name": "transforms_2048x1024_f32", "kind": "transforms", "nx": 2048, "nz": 1024,
         "dtype": "f32"},
        # one small FP64 simulation run for many loops with the CFL ticker on
        # the device: launches and latency count
        {"name": "tgv_256_f64", "kind": "fused", "flow": "vortex", "sizes": "256", "dtype": "f64",
         "ab": 2, "fd": 2, "steps": 100, "mode": "device"},
        # the plain FP64 simulation of the benchmark
        {"name": "kh_1024_f64", "kind": "fused", "flow": "ink", "sizes": "1024", "dtype": "f64",
         "ab": 4, "fd": 2, "steps": 4, "mode": "step"},
        # the benchmark's batched FP32 form: bandwidth counts
        {"name": "kh_1024_f32_batch16", "kind": "fused", "flow": "ink",
         "sizes": ",".join(["1024"] * 16), "dtype": "f32", "ab": 4, "fd": 2, "steps": 4,
         "mode": "step"},
        # a double-diffusive parameter study on mixed grids, graph-captured
        {"name": "ddc_mixed_f32_batch10", "kind": "fused", "flow": "ddc",
         "sizes": "1024,128,512,256,512,1024,128,256,512,256", "dtype": "f32", "ab": 2, "fd": 2,
         "steps": 20, "mode": "graph"},
        # resistive tearing (two stages per step), fourth-order differences
        {"name": "mhd_512_f32_batch4", "kind": "fused", "flow": "mhd", "sizes": "512,512,512,512",
         "dtype": "f32", "ab": 2, "fd": 4, "steps": 4, "mode": "step"},
        # what a serving batch holds: vortex pairs of very different sizes
        {"name": "vortex_mixed_f32_batch8", "kind": "fused", "flow": "vortex",
         "sizes": "2048,256,1024,256,512,2048,512,256", "dtype": "f32", "ab": 2, "fd": 2,
         "steps": 4, "mode": "step"},
        # the Rayleigh-Benard configuration: predictor-corrector, FP32 with
        # FP64 solves, CFL ticker on the device
        {"name": "rbc_1024x513_f32_pc", "kind": "fdz", "sizes": "1024x513", "scheme": "pc",
         "dtype": "f32", "ab": 2, "fd": 2, "steps": 20, "mode": "device"},
        # a Rayleigh-number study with the reference's explicit scheme, FP64,
        # ragged sizes (order 4 needs the wide wall band)
        {"name": "rbc_ragged_f64_batch6", "kind": "fdz",
         "sizes": "256x129,512x257,64x33,512x200,128x100,256x65", "scheme": "explicit",
         "dtype": "f64", "ab": 2, "fd": 4, "steps": 4, "mode": "step"},
    ]


def draw(rng):
    kind = rng.choice(["mirror", "mirror", "transforms", "fused", "fused", "fused", "fdz", "fdz"])
    p2 = lambda lo, hi: 1 << rng.randint(lo, hi)  # noqa: E731
    logu = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    c = {"kind": kind, "dtype": rng.choice(["f64", "f32"])}
    if kind == "mirror":
        c.update(flow=rng.choice(["vortex", "ink", "rbc"]), nx=p2(5, 11), ab=rng.choice([2, 4]),
                 fd=rng.choice([2, 4]))
        c["nz"] = logu(17, 1025) if c["flow"] == "rbc" else p2(5, 11)
    elif kind == "transforms":
        c.update(nx=p2(4, 12), nz=p2(4, 11))
    elif kind == "fused":
        c.update(flow=rng.choice(["vortex", "ink", "ddc", "mhd"]), ab=rng.choice([2, 4]),
                 fd=rng.choice([2, 4]), mode=rng.choice(["step", "graph"]), steps=4)
        most = min(12, 64 // (2 * NFIELD[c["flow"]]))
        top = 10 if c["dtype"] == "f64" else 11
        n, room, sizes = rng.randint(1, most), 1 << 22, []
        for _ in range(n):
            s = p2(5, top)
            if s * s <= room:
                sizes.append(s)
                room -= s * s
        c["sizes"] = ",".join(str(s) for s in sizes or [256])
    else:
        c.update(scheme=rng.choice(["explicit", "semi-implicit", "pc"]), ab=rng.choice([2, 4]),
                 fd=rng.choice([2, 4]), mode=rng.choice(["step", "graph"]), steps=4)
        c["sizes"] = ",".join("%dx%d" % (p2(5, 10), logu(17, 700)) for _ in range(rng.randint(1, 6)))
    return c


# ---------------------------------------------------------------------------
# Inputs: smooth random fields of a few dozen modes with the profiles of the
# flows they stand for, formed in 64 bits on the GPU from the seed alone.
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _grid(nx, nz, lx, lz):
    x = torch.arange(nx, device="cuda", dtype=torch.float64) * (lx / nx)
    z = torch.arange(nz, device="cuda", dtype=torch.float64) * (lz / nz)
    return x[:, None], z[None, :]


def _modes(g, x, z, lx, lz):
    """Random combination of the Fourier modes kx in [1, n], kz in [0, n], n
    an eighth of the grid, amplitudes falling off as 1 / |k|: a developed
    field, whose advection is well above the rounding of its products."""
    n = max(2, min(x.numel(), z.numel()) // 8)
    k = torch.arange(1, n + 1, device="cuda", dtype=torch.float64)
    m = torch.arange(0, n + 1, device="cuda", dtype=torch.float64)
    r = torch.rand((2, n, n + 1), generator=g, device="cuda", dtype=torch.float64)
    a = (2 * r[0] - 1) / torch.hypot(k[:, None], m[None, :])
    ph = TWO_PI * r[1]
    ax, az = TWO_PI / lx * x * k[None, :], TWO_PI / lz * z.T * m[None, :]
    # cos(ax + az + ph) expanded so that each product is a small contraction
    c, s = torch.cos(ax), torch.sin(ax)
    cz, sz = torch.cos(az), torch.sin(az)
    ac, as_ = a * torch.cos(ph), a * torch.sin(ph)
    return ((c @ ac - s @ as_) @ cz.T) - ((s @ ac + c @ as_) @ sz.T)


def _noise(g, nx, nz, amp):
    return amp * (2 * torch.rand((nx, nz), generator=g, device="cuda", dtype=torch.float64) - 1)


def _flow(flow, nx, nz, seed):
    """(lx, lz, dt, coeff, param, physical fields) of a fully spectral flow."""
    g = _gen(seed)
    if flow == "vortex":  # Taylor-Green vortex with a perturbation
        lx = lz = TWO_PI
        x, z = _grid(nx, nz, lx, lz)
        f = [2 * torch.sin(x) * torch.sin(z) + _modes(g, x, z, lx, lz)]
        coeff, param = [1e-2], []
    elif flow == "ink":  # double shear layer with a passive scalar
        lx = lz = 2.0
        x, z = _grid(nx, nz, lx, lz)
        a, b = (z - 0.5) / 0.05, (z - 1.5) / 0.05
        w = (1 / torch.cosh(a) ** 2 - 1 / torch.cosh(b) ** 2) / 0.05
        u = torch.tanh(a) - torch.tanh(b)
        f = [w + 5 * _modes(g, x, z, lx, lz) + _noise(g, nx, nz, 1e-3),
             u + _modes(g, x, z, lx, lz)]
        coeff, param = [1e-4, 1e-4], []
    elif flow == "ddc":  # double-diffusive convection
        lx = lz = 1e5 ** 0.25
        x, z = _grid(nx, nz, lx, lz)
        f = [0.1 * _modes(g, x, z, lx, lz) for _ in range(3)]
        coeff, param = [7.0, 1.0, 0.01], [7.0, 1.5]
    else:  # resistive tearing: a double current sheet
        lx = lz = 1.0
        x, z = _grid(nx, nz, lx, lz)
        j = torch.zeros_like(z)
        for k in range(-2, 3):
            j = j + (1 / torch.cosh((z - 0.25 - k) / 0.1) ** 2
                     - 1 / torch.cosh((z - 0.75 - k) / 0.1) ** 2) / 0.1
        f = [_modes(g, x, z, lx, lz), j + _modes(g, x, z, lx, lz)]
        coeff, param = [1e-4, 1e-4], []
    return lx, lz, 0.05 * min(lx / nx, lz / nz), coeff, param, f


def _rbc(nx, nz, seed):
    """(lx, lz, dt, Pr, Ra, w, T) of a Rayleigh-Benard roll pattern."""
    lx, lz, pr, ra = 2.0, 1.0, 1.0, 1e6
    g = _gen(seed)
    x, z = _grid(nx, nz, lx, lz)
    bump = torch.sin(math.pi * z / lz) ** 2
    w = 500.0 * bump * _modes(g, x, z, lx, lz)
    t = 1.0 - z / lz + 0.2 * bump * _modes(g, x, z, lx, lz) + _noise(g, nx, nz, 1e-3)
    dz, dx = lz / nz, lx / nx
    return lx, lz, min(2e-5 * min(dx, dz), dz * dz / 64), pr, ra, w, t


def _spec(f):
    """Compact spectrum (2 nn + 1, nm) of a real field, normalised."""
    nx, nz = f.shape
    nn, nm = (nx - 1) // 3, (nz - 1) // 3
    s = torch.fft.fft(torch.fft.rfft(f, dim=1)[:, :nm], dim=0) / (nx * nz)
    return torch.cat([s[: nn + 1], s[nx - nn:]], dim=0)


def _spec_x(f):
    """Fourier-x / FD-z spectrum (nn, nz) of a real field, normalised."""
    nx = f.shape[0]
    return torch.fft.rfft(f, dim=0)[: (nx - 1) // 3] / nx


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _mirror_state(case, seed):
    nx, nz, flow = case["nx"], case["nz"], case["flow"]
    rbc = flow == "rbc"
    if rbc:
        lx, lz, dt, pr, ra, *fields = _rbc(nx, nz, seed)
        spectra = [_spec_x(f) for f in fields]
    else:
        lx, lz, dt, coeff, _, fields = _flow(flow, nx, nz, seed)
        spectra = [_spec(f) for f in fields]
    prm = {"nx": nx, "nz": nz, "lx": lx, "lz": lz, "final_time": 1e9, "initial_dt": dt,
           "integrator_order": case["ab"], "spatial_derivative_order": case["fd"],
           "precision": "double" if case["dtype"] == "f64" else "single"}
    if rbc:
        prm.update(integrator="explicit", discretisation=["spectral", "fdm"])
    p = melvin.Parameters(prm)
    sim = melvin.Simulation(p, melvin.hip)
    B = melvin.BasisFunctions
    bfs = [B.COMPLEX_EXP, B.FDM if rbc else B.COMPLEX_EXP]
    names = ["w", "tmp"] if rbc else ["w", "ink"][: len(spectra)]
    var = [sim.make_variable(n, bfs) for n in names]
    dvar = [sim.make_derivative("d" + n) for n in names]
    psi, ux, uz = (sim.make_variable(n, bfs) for n in ("psi", "ux", "uz"))
    sim.init_laplacian_solver(bfs)
    sim.config_cfl(ux, uz)
    for v, s in zip(var, spectra):
        v.load(s)
    st = {"case": case, "sim": sim, "p": p, "var": var, "dvar": dvar, "psi": psi, "ux": ux,
          "uz": uz}
    st.update({"Pr": pr, "Ra": ra} if rbc else {"coeff": coeff})
    return st


def _mirror_run(st):
    sim, psi, ux, uz = st["sim"], st["psi"], st["ux"], st["uz"]
    w = st["var"][0]
    utility.calc_velocity_from_vorticity(w, psi, ux, uz, sim.get_laplacian_solver())
    if st["case"]["flow"] == "rbc":
        (w, tmp), (dw, dtmp) = st["var"], st["dvar"]
        pr, ra = st["Pr"], st["Ra"]
        diffusion_term = pr * w.snabla2()
        dw[:] = -w.vec_dot_nabla(ux.getp(), uz.getp()) - pr * ra * tmp.sddx()
        sim._integrator.integrate(w, dw, diffusion_term)
        diffusion_term = tmp.snabla2()
        dtmp[:] = -tmp.vec_dot_nabla(ux.getp(), uz.getp())
        sim._integrator.integrate(tmp, dtmp, diffusion_term)
        k = 2 if st["case"]["fd"] == 4 else 1
        w[1:, :k] = 0.0
        w[1:, -k:] = 0.0
        psi[1:, :k] = 0.0
        psi[1:, -k:] = 0.0
        tmp[0, :k] = 1.0
        tmp[0, -k:] = 0.0
        tmp[1:, :k] = 0.0
        tmp[1:, -k:] = 0.0
        psi[0, :] = 0.0
        w[0, :] = 0.0
    else:
        for v, dv, c in zip(st["var"], st["dvar"], st["coeff"]):
            lin_op = c * v.lap()
            dv[:] = -v.vec_dot_nabla(ux.getp(), uz.getp())
            sim._integrator.integrate(v, dv, lin_op)
    sim.end_loop()
    return {"var": [v.gets() for v in st["var"]], "rhs": [d.get_all() for d in st["dvar"]],
            "psi": psi.gets(), "ux": ux.getp(), "uz": uz.getp()}


def _sizes(case):
    return [s.split("x") if "x" in s else (s, s) for s in case["sizes"].split(",")]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "mirror":
        return _mirror_state(case, seed)
    if kind == "transforms":
        nx, nz = case["nx"], case["nz"]
        p = melvin.Parameters({"nx": nx, "nz": nz, "lx": 2.0, "lz": 2.0, "final_time": 1.0,
                               "precision": "double" if case["dtype"] == "f64" else "single"})
        phys, spec = _transform_inputs(nx, nz, seed)
        real, cplx = ((torch.float64, torch.complex128) if case["dtype"] == "f64"
                      else (torch.float32, torch.complex64))
        return {"case": case, "st": melvin.SpectralTransformer(p, melvin.hip),
                "phys": phys.to(real).contiguous(), "spec": spec.to(cplx).contiguous()}
    jobs = []
    for i, (nx, nz) in enumerate(_sizes(case)):
        nx, nz = int(nx), int(nz)
        if kind == "fdz":
            lx, lz, dt, pr, ra, w, t = _rbc(nx, nz, seed + 1000 * i)
            job = fdz.FdzJob(nx, nz, lx, lz, Pr=pr, Ra=ra, dtype=case["dtype"], dt=dt,
                             scheme=case["scheme"], ab_order=case["ab"], fd_order=case["fd"])
            job.set_state([_spec_x(w), _spec_x(t)])
        else:
            flow = case["flow"]
            lx, lz, dt, coeff, param, f = _flow(flow, nx, nz, seed + 1000 * i)
            job = fused.Job({"vortex": "vorticity", "ink": "vorticity"}.get(flow, flow), nx, nz,
                            lx, lz, dtype=case["dtype"], dt=dt, coeff=coeff, param=param,
                            ab_order=case["ab"], fd_order=case["fd"])
            job.set_state([_spec(a) for a in f])
        jobs.append(job)
    batch = fdz.FdzBatch(jobs) if kind == "fdz" else fused.Batch(jobs)
    return {"case": case, "jobs": jobs, "batch": batch}


def _transform_inputs(nx, nz, seed):
    g = _gen(seed)
    x, z = _grid(nx, nz, 2.0, 2.0)
    phys = _modes(g, x, z, 2.0, 2.0) + _noise(g, nx, nz, 1e-2)
    return phys, _spec(_modes(g, x, z, 2.0, 2.0) + _noise(g, nx, nz, 1e-2))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "mirror":
        return _mirror_run(state)
    if kind == "transforms":
        st = state["st"]
        return {"spec": st.to_spectral(state["phys"]), "phys": st.to_physical(state["spec"])}
    batch, n = state["batch"], case["steps"]
    if case["mode"] == "device":
        (fdz if kind == "fdz" else fused).run_device(batch, n, chunk=n)
    elif case["mode"] == "graph":
        batch.graph_step(n)
    else:
        batch.step(n)
    if kind == "fdz":
        return [{"state": j.buf[j.parity], "rhs": j.hist} for j in state["jobs"]]
    # (the device arrays are kz-major; views in the reference's (rows, nm) layout)
    return [{"state": j.current(), "rhs": [h.transpose(1, 2) for h in j.hist]}
            for j in state["jobs"]]


# ---------------------------------------------------------------------------
# The least a pass moves and computes: per step, the state read and written,
# the history ring's other levels read and its new level written (nothing of
# the passes between), and the transforms' butterflies with the pointwise
# arithmetic.
# ---------------------------------------------------------------------------
def _fft2(nx, nz):
    """Operations of one real 2-D transform, dealiased columns along x."""
    return 2.5 * nx * nz * math.log2(nz) + 5.0 * (nz // 3) * nx * math.log2(nx)


def work(case):
    kind = case["kind"]
    r = 8 if case["dtype"] == "f64" else 4
    c = 2 * r
    if kind == "transforms":
        nx, nz = case["nx"], case["nz"]
        s = (2 * ((nx - 1) // 3) + 1) * ((nz - 1) // 3)
        return {"bytes": 2 * (nx * nz * r + s * c), "flops": 2 * _fft2(nx, nz)}
    total = {"bytes": 0.0, "flops": 0.0}
    sizes = [(case["nx"], case["nz"])] if kind == "mirror" else _sizes(case)
    steps = 1 if kind == "mirror" else case["steps"]
    for nx, nz in sizes:
        nx, nz = int(nx), int(nz)
        nn = (nx - 1) // 3
        if kind == "fdz" or case.get("flow") == "rbc":
            nf, s = 2, nn * nz
            evals = 2 if case.get("scheme") == "pc" else 1
            fl = evals * (8 * 2.5 * nx * nz * math.log2(nx) + 12 * nx * nz + 3 * 30 * s)
            by = nf * s * c * (2 + case["ab"])
        else:
            nf, s = NFIELD[case["flow"]], (2 * nn + 1) * ((nz - 1) // 3)
            inv, fwd = (7, 2) if case["flow"] == "mhd" else (nf + 2, nf)
            fl = (inv + fwd) * _fft2(nx, nz) + 8 * nf * nx * nz + 30 * nf * s
            by = nf * s * c * (2 + case["ab"])
        if kind == "mirror":  # the loop body's psi, ux and uz are results too
            by += s * c + 2 * nx * nz * r
        total["bytes"] += steps * by
        total["flops"] += steps * fl
    return total


# ---------------------------------------------------------------------------
# 64-bit restatement
# ---------------------------------------------------------------------------
def _phys(s, nx, nz):
    """Real field of a compact spectrum (the imaginary part of the kz = 0
    term is dropped after the x transform, as a c2r transform does)."""
    nn = (nx - 1) // 3
    a = torch.zeros((nx, s.shape[1]), dtype=torch.complex128, device=s.device)
    a[: nn + 1] = s[: nn + 1]
    a[nx - nn:] = s[nn + 1:]
    a = torch.fft.ifft(a, dim=0) * nx
    b = torch.zeros((nx, nz // 2 + 1), dtype=torch.complex128, device=s.device)
    b[:, : s.shape[1]] = a
    b[:, 0] = b[:, 0].real
    return torch.fft.irfft(b, n=nz, dim=1) * nz


def _phys_x(s, nx):
    b = torch.zeros((nx // 2 + 1, s.shape[1]), dtype=torch.complex128, device=s.device)
    b[: s.shape[0]] = s
    b[0] = b[0].real
    return torch.fft.irfft(b, n=nx, dim=0) * nx


def _diff(f, h, order, dim, periodic=True):
    r = lambda k: torch.roll(f, -k, dims=dim)  # noqa: E731
    if order == 2:
        d, w = (r(1) - r(-1)) / (2 * h), 1
    else:
        d, w = (-0.25 * r(2) + 2 * r(1) - 2 * r(-1) + 0.25 * r(-2)) / (3 * h), 2
    if not periodic:
        d = d.clone()
        d.narrow(dim, 0, w).zero_()
        d.narrow(dim, f.shape[dim] - w, w).zero_()
    return d


def _diff2_z(f, h, order):
    r = lambda k: torch.roll(f, -k, dims=1)  # noqa: E731
    if order == 2:
        d, w = (r(1) - 2 * f + r(-1)) / h ** 2, 1
    else:
        d, w = (-r(2) / 12 + 4 / 3 * r(1) - 5 / 2 * f + 4 / 3 * r(-1) - r(-2) / 12) / h ** 2, 2
    d[:, :w] = 0
    d[:, -w:] = 0
    return d


def _ab(ring, cur, dt):
    q = ring.shape[0]
    h = lambda i: ring[(cur - i) % q]  # noqa: E731
    if q == 2:
        return dt / 2 * (3 * h(0) - h(1))
    return dt / 24 * (55 * h(0) - 59 * h(1) + 37 * h(2) - 9 * h(3))


def _held(s, dtype):
    """A spectrum as a driver's single- or double-precision variable holds it."""
    return s.to(torch.complex64).to(torch.complex128) if dtype == "f32" else s


def _exact_spectral(flow, nx, nz, ab, fd, steps, seed, held="f64"):
    """(states, rings, psi, ux, uz) after `steps` steps of a spectral flow."""
    lx, lz, dt, coeff, param, f = _flow(flow, nx, nz, seed)
    s = [_held(_spec(a), held) for a in f]
    nn, nm = (nx - 1) // 3, (nz - 1) // 3
    n = torch.cat([torch.arange(nn + 1), torch.arange(-nn, 0)]).to("cuda", torch.float64)[:, None]
    m = torch.arange(nm, device="cuda", dtype=torch.float64)[None, :]
    ikx, ikz = 1j * TWO_PI / lx * n, 1j * TWO_PI / lz * m
    lap = -(TWO_PI / lx * n) ** 2 - (TWO_PI / lz * m) ** 2
    inv = lap.clone()
    inv[0, 0] = 1.0
    ring = [torch.zeros((ab,) + tuple(s[0].shape), dtype=torch.complex128, device="cuda") for _ in s]
    dx, dz = lx / nx, lz / nz

    def vel(w):
        p = -w / inv
        return p, _phys(-ikz * p, nx, nz), _phys(ikx * p, nx, nz)

    def adv(g, u, v):
        return _spec(_diff(u * g, dx, fd, 0) + _diff(v * g, dz, fd, 1))

    for k in range(steps):
        cur = k % ab

        def update(i, rhs):
            ring[i][cur] = rhs
            lin = coeff[i] * lap
            return ((1 + 0.49 * dt * lin) * s[i] + _ab(ring[i], cur, dt)) / (1 - 0.51 * dt * lin)

        psi, ux, uz = vel(s[0])
        if flow == "mhd":
            _, bx, bz = vel(s[1])
            w, j = _phys(s[0], nx, nz), _phys(s[1], nx, nz)
            s[0] = update(0, -adv(w, ux, uz) + adv(j, bx, bz))
            s[1] = update(1, -adv(j, ux, uz) + adv(_phys(s[0], nx, nz), bx, bz))
        else:
            rhs = [-adv(_phys(a, nx, nz), ux, uz) for a in s]
            if flow == "ddc":
                rhs[0] = rhs[0] + param[0] * ikx * (s[2] - s[1])
                rhs[1] = rhs[1] - ikx * psi
                rhs[2] = rhs[2] - ikx * psi / param[1]
            s = [update(i, rhs[i]) for i in range(len(s))]
            if flow == "ddc":
                s[1][:, 0] = 0
                s[2][:, 0] = 0
    return s, ring, psi, ux, uz


def _tridiag(lo, dg, rhs):
    """Per-row tridiagonal solve along z, identity first and last rows,
    interior bands (lo, dg[row], lo); rows of `rhs` (numpy)."""
    nz = rhs.shape[1]
    c = np.zeros((rhs.shape[0], nz))
    d = np.array(rhs)
    for j in range(1, nz - 1):
        r = 1.0 / (dg - lo * c[:, j - 1])
        c[:, j] = lo * r
        d[:, j] = (rhs[:, j] - lo * d[:, j - 1]) * r
    for j in range(nz - 2, 0, -1):
        d[:, j] -= c[:, j] * d[:, j + 1]
    return d


def _exact_rbc(nx, nz, scheme, ab, fd, steps, seed, held="f64"):
    """(states, rings, psi, ux, uz) after `steps` steps of Rayleigh-Benard."""
    lx, lz, dt, pr, ra, w0, t0 = _rbc(nx, nz, seed)
    s = [_held(_spec_x(a), held) for a in (w0, t0)]
    nn = s[0].shape[0]
    dx, dz = lx / nx, lz / nz
    kx = TWO_PI / lx * torch.arange(nn, device="cuda", dtype=torch.float64)[:, None]
    k2 = (kx ** 2)[:, 0].cpu().numpy()
    wall = 1 if fd == 2 else 2
    coeff = [pr, 1.0]
    ring = [torch.zeros((ab,) + tuple(a.shape), dtype=torch.complex128, device="cuda") for a in s]

    def solve(lo, dg, rhs):
        return torch.from_numpy(_tridiag(lo, dg, rhs.cpu().numpy())).cuda()

    def explicit_terms(v):
        psi = solve(1 / dz ** 2, -(k2 + 2 / dz ** 2), -v[0])
        ux = _phys_x(-_diff(psi, dz, fd, 1, False), nx)
        uz = _phys_x(1j * kx * psi, nx)
        rhs = []
        for a in v:
            f = _phys_x(a, nx)
            rhs.append(-_spec_x(_diff(ux * f, dx, fd, 0) + _diff(uz * f, dz, fd, 1, False)))
        rhs[0] = rhs[0] - pr * ra * 1j * kx * v[1]
        return psi, ux, uz, rhs

    def walls(v):
        w, t = v
        w[:, :wall], w[:, -wall:], w[0] = 0, 0, 0
        t[:, :wall], t[:, -wall:] = 0, 0
        t[0, :wall] = 1
        return v

    def implicit(i, e):
        lap = -(kx ** 2) * s[i] + _diff2_z(s[i], dz, 2)
        lap[:, 0], lap[:, -1] = 0, 0
        a = 0.51 * dt * coeff[i]
        return s[i] + solve(-a / dz ** 2, 1 + a * (k2 + 2 / dz ** 2), dt * coeff[i] * lap + e)

    for k in range(steps):
        cur = k % ab
        psi, ux, uz, rhs = explicit_terms(s)
        for i in range(2):
            if scheme == "explicit":
                rhs[i] = rhs[i] + coeff[i] * (-(kx ** 2) * s[i] + _diff2_z(s[i], dz, fd))
            ring[i][cur] = rhs[i]
        if scheme == "explicit":
            s = walls([s[i] + _ab(ring[i], cur, dt) for i in range(2)])
            continue
        new = walls([implicit(i, _ab(ring[i], cur, dt)) for i in range(2)])
        if scheme == "pc":
            nxt = (cur + 1) % ab
            rhs = explicit_terms(new)[3]
            e = []
            for i in range(2):
                ring[i][nxt] = rhs[i]
                h = lambda b: ring[i][(nxt - b) % ab]  # noqa: E731
                e.append(dt / 2 * (h(0) + h(1)) if ab == 2 else
                         dt / 24 * (9 * h(0) + 19 * h(1) - 5 * h(2) + h(3)))
            new = walls([implicit(i, e[i]) for i in range(2)])
        s = new
    psi = psi.clone()
    psi[:, :wall], psi[:, -wall:], psi[0] = 0, 0, 0
    return s, ring, psi, ux, uz


def exact(case, seed):
    kind = case["kind"]
    if kind == "transforms":
        # the values the call is given are the rounded ones
        phys, spec = _transform_inputs(case["nx"], case["nz"], seed)
        if case["dtype"] == "f32":
            phys, spec = phys.float().double(), spec.to(torch.complex64).to(torch.complex128)
        return {"spec": _spec(phys), "phys": _phys(spec, case["nx"], case["nz"])}
    if kind == "mirror":
        if case["flow"] == "rbc":
            s, ring, psi, ux, uz = _exact_rbc(case["nx"], case["nz"], "explicit", case["ab"],
                                              case["fd"], 1, seed, case["dtype"])
        else:
            s, ring, psi, ux, uz = _exact_spectral(case["flow"], case["nx"], case["nz"],
                                                   case["ab"], case["fd"], 1, seed, case["dtype"])
        return {"var": s, "rhs": ring, "psi": psi, "ux": ux, "uz": uz}
    out = []
    for i, (nx, nz) in enumerate(_sizes(case)):
        args = (case["ab"], case["fd"], case["steps"], seed + 1000 * i)
        if kind == "fdz":
            s, ring = _exact_rbc(int(nx), int(nz), case["scheme"], *args)[:2]
        else:
            s, ring = _exact_spectral(case["flow"], int(nx), int(nz), *args)[:2]
        out.append({"state": s, "rhs": ring})
    return out
