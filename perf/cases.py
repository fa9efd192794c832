"""The particle-mesh work that programs on this framework do, as cases that can be timed and checked.

Five families, each through the public Python entry points:

  step     the PM driver's inner loop: lf.pm_step (deposit, Poisson solve, gather, kick, drift)
           twice per pass, so that the second step's fields carry the first step's particle update
  driver   the same physics call by call, the way a program written against the reference spells
           it: projection_init, *_project, *_comm, FFT, Green, inverse FFT, updateHalo,
           updateVel (whose max |v| sets the next time step), moveParticles
  project  one projection of the particles (density, momentum, stress) with its ghost fold and
           halo, as the source term of a field equation
  fft      a transform to k space and one back into another field
  diffpm   loss and gradients of the differentiable PM run with respect to the initial particles

Positions are a displaced lattice (the usual start of a simulation), uniform, or clustered blobs.
Particles of a case with "upload" come from arrays of the caller's and have a 64-bit result to be
compared with; the larger cases use the container's own initial conditions.  Box length 1, total
mass 1, ghost width 1 unless a case says otherwise.
"""
import math

import torch

import latfield2_amd as lf
from latfield2_amd.diffpm import DiffPM, pm_density_loss

DT = 1e-3
FFT_SIZES = sorted({m << k for m in (1, 3, 5) for k in range(11) if 8 <= (m << k) <= 1024})
KINDS = {"scalar": (lf.PROJ_SCALAR, 1), "vector": (lf.PROJ_VECTOR, 3), "vecvec": (lf.PROJ_VECVEC, 6),
         "vector_ngp": (lf.PROJ_VECTOR_NGP, 3), "tensor_ngp": (lf.PROJ_SYMTENSOR_NGP, 6)}
CALLS = {"scalar": (lf.scalarProjectionCIC_project, lf.scalarProjectionCIC_comm),
         "vector": (lf.vectorProjectionCIC_project, lf.vectorProjectionCIC_comm),
         "vecvec": (lf.VecVecProjectionCIC_project, lf.VecVecProjectionCIC_comm),
         "vector_ngp": (lf.vectorProjectionCICNGP_project, lf.vectorProjectionCICNGP_comm),
         "tensor_ngp": (lf.symtensorProjectionCICNGP_project, lf.symtensorProjectionCICNGP_comm)}


def listed():
    return [
        # a small force test: 64^3 mesh, 32^3 particles at rest; launches and latency count
        dict(name="step_64", family="step", N=64, np=32 ** 3, ic="lattice", sigma=0.5, sigma_v=0.0, dtype="f32",
             fixed=False, masses=False, upload=True),
        # the common production size on one card: one particle per cell, barely displaced
        dict(name="step_256", family="step", N=256, np=256 ** 3, ic="lattice", sigma=0.3, sigma_v=0.01, dtype="f32",
             fixed=False, masses=False, upload=False),
        # the largest: an evolved, strongly clustered mesh (most particles in dense blobs)
        dict(name="step_512_blobs", family="step", N=512, np=512 ** 3, ic="blobs", sigma=2.0, sigma_v=0.01, dtype="f32",
             fixed=False, masses=False, upload=False),
        # the same step in double precision, the reference's default Real
        dict(name="step_f64_256", family="step", N=256, np=256 ** 3, ic="lattice", sigma=0.3, sigma_v=0.01, dtype="f64",
             fixed=False, masses=False, upload=False),
        # the bit-reproducible integer deposit, for runs that have to repeat exactly
        dict(name="step_fixed_128", family="step", N=128, np=128 ** 3, ic="lattice", sigma=0.5, sigma_v=0.01,
             dtype="f32", fixed=True, masses=False, upload=True),
        # a reference program's loop, recompiled: double precision, a size that is no power of two
        dict(name="driver_f64_96", family="driver", N=96, np=96 ** 3, ic="lattice", sigma=0.5, sigma_v=0.01,
             dtype="f64", upload=True),
        # the same loop in single precision on particles without any order
        dict(name="driver_128", family="driver", N=128, np=1_500_007, ic="uniform", sigma=0.0, sigma_v=0.01,
             dtype="f32", upload=True),
        # momentum density of particles of different masses on a mesh of an odd number of bricks
        dict(name="project_vector_120", family="project", kind="vector", N=120, np=1_000_003, ic="blobs", sigma=6.0,
             sigma_v=0.05, dtype="f32", masses=True, target="calls", halo=1, upload=True),
        # the stress tensor of a whole simulation, the widest projection
        dict(name="project_vecvec_256", family="project", kind="vecvec", N=256, np=256 ** 3, ic="lattice", sigma=1.0,
             sigma_v=0.05, dtype="f32", masses=False, target="calls", halo=1, upload=False),
        # a large vector field to k space and back (vector modes of a metric)
        dict(name="fft_vector_512", family="fft", N=512, C=3, halo=1, khalo=0, dtype="f32", c2c=False),
        # one evaluation of an optimizer that fits initial conditions: loss and all gradients
        dict(name="diffpm_128", family="diffpm", N=128, np=128 ** 3, nsteps=10, ic="lattice", sigma=0.5, sigma_v=0.0,
             dtype="f32"),
        # the same in double precision on a small mesh, as gradient checks and samplers run it
        dict(name="diffpm_f64_32", family="diffpm", N=32, np=32 ** 3, nsteps=3, ic="lattice", sigma=0.5, sigma_v=0.05,
             dtype="f64"),
    ]


def _between(rng, lo, hi):
    """an integer of [lo, hi], spread over the logarithm"""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _near(rng, sizes, lo, hi):
    t = _between(rng, lo, hi)
    return min((s for s in sizes if lo <= s <= hi), key=lambda s: abs(math.log(s / t)))


def draw(rng):
    family = rng.choice(["step", "step", "step", "driver", "driver", "project", "project", "project", "fft", "fft",
                         "diffpm", "diffpm"])
    f64 = rng.random() < 0.3
    c = dict(family=family)
    if family == "fft":
        c2c = rng.random() < 0.3
        most = {1: 640 if c2c or f64 else 1024, 3: 320 if c2c or f64 else 512, 6: 256 if c2c else 384}
        C = 1 if c2c else rng.choice([1, 1, 3] if f64 else [1, 1, 3, 6])
        return dict(c, N=_near(rng, FFT_SIZES, 16, most[C]), C=C, halo=rng.choice([0, 1, 1, 2]), khalo=rng.choice([0, 0, 1]),
                    dtype="f64" if f64 else "f32", c2c=c2c)
    if family == "diffpm":
        N = rng.choice([16, 32, 64, 128])
        return dict(c, N=N, np=_between(rng, N ** 3 // 8, N ** 3), nsteps=rng.randint(1, 10 if N < 128 or not f64 else 5),
                    ic="uniform" if rng.random() < 0.3 else "lattice", sigma=round(rng.uniform(0.2, 1.0), 3),
                    sigma_v=rng.choice([0.0, 0.05]), dtype="f64" if f64 else "f32")
    if family == "project":
        # a mesh that no FFT limits: every multiple of 4
        N = 4 * _between(rng, 6, 48 if f64 else 64)
    else:
        N = _near(rng, FFT_SIZES, 16, 192 if f64 else 384)
    np_ = _between(rng, N ** 3 // 8, N ** 3 * 2 if N <= 128 else N ** 3)
    ic = rng.choice(["lattice", "lattice", "uniform", "blobs"])
    if ic == "lattice":
        np_ = round(np_ ** (1 / 3)) ** 3
    c.update(N=N, np=np_, ic=ic, sigma=round(rng.uniform(0.2, 1.0) if ic == "lattice" else rng.uniform(1.0, 6.0), 3),
             sigma_v=rng.choice([0.01, 0.05]), dtype="f64" if f64 else "f32", upload=np_ <= 3_000_000)
    if family == "step":
        c.update(fixed=not f64 and rng.random() < 0.25, masses=c["upload"] and rng.random() < 0.25)
    if family == "project":
        c.update(kind=rng.choice(list(KINDS)), masses=c["upload"] and rng.random() < 0.4,
                  target=rng.choice(["calls", "calls", "set"]), halo=rng.choice([1, 1, 2]))
    return c


# ---------------------------------------------------------------- inputs
def _type(case):
    return torch.float32 if case["dtype"] == "f32" else torch.float64


def _code(case):
    return lf.F32 if case["dtype"] == "f32" else lf.F64


def _particles(case, seed):
    """positions in the box, velocities and masses, in 64 bits on the card"""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)
    n, N = case["np"], case["N"]
    kw = dict(generator=g, device="cuda", dtype=torch.float64)
    if case["ic"] == "lattice":
        ng = math.ceil(round(n ** (1 / 3), 9))
        i = torch.arange(n, device="cuda")
        pos = torch.stack([i % ng, i // ng % ng, i // (ng * ng)], 1).double() / ng
        pos = pos + torch.randn((n, 3), **kw) * (case["sigma"] / N)
    elif case["ic"] == "uniform":
        pos = torch.rand((n, 3), **kw)
    else:  # four fifths in blobs of unequal weight, the rest spread
        nb = max(4, n // 4096)
        weight = torch.rand(nb, **kw).clamp_min(1e-3) ** (-1 / 1.5)
        which = torch.multinomial(weight, n, replacement=True, generator=g)
        pos = torch.rand((nb, 3), **kw)[which] + torch.randn((n, 3), **kw) * (case["sigma"] / N)
        pos = torch.where(torch.rand((n, 1), **kw) < 0.8, pos, torch.rand((n, 3), **kw))
    pos = pos - torch.floor(pos)
    pos = torch.where(pos >= 1.0, torch.zeros_like(pos), pos)
    vel = torch.randn((n, 3), **kw) * case["sigma_v"]
    mass = (0.5 + torch.rand(n, **kw)) / n
    return pos, vel, mass


def _container(case, seed):
    n, masses = case["np"], bool(case.get("masses"))
    parts = lf.Particles(case["N"], n, _code(case), per_particle_mass=masses, mass=1.0 / n)
    if case["upload"]:
        pos, vel, mass = _particles(case, seed)
        parts.addParticles(pos.cpu().numpy(), vel.cpu().numpy(), mass.cpu().numpy() if masses else None)
    elif case["ic"] == "lattice":
        parts.ic_lattice(round(n ** (1 / 3)), case["sigma"], case["sigma_v"], seed)
    elif case["ic"] == "uniform":
        parts.ic_uniform(n, case["sigma_v"], seed)
    else:
        parts.ic_blobs(n, max(4, min(4096, n // 4096)), 1.5, case["sigma"], 0.2, case["sigma_v"], seed)
    return parts


def _field_values(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)
    shape = (case["N"],) * 3 + (case["C"],) + ((2,) if case["c2c"] else ())
    return torch.randn(shape, generator=g, device="cuda", dtype=_type(case))


def _diffpm_inputs(case, seed):
    """initial positions and velocities and the target density of a differentiable run, in its type"""
    pos, vel, _ = _particles(case, seed)
    t = _type(case)
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 19)
    target = 1 + 0.5 * torch.randn((case["N"],) * 3, generator=g, device="cuda", dtype=t)
    return pos.to(t), vel.to(t), target


def prepare(case, seed):
    lf.load()
    s = dict(case=case)
    f = case["family"]
    code = _code(case)
    if f == "fft":
        lat = lf.Lattice(3, case["N"], case["halo"])
        if case["c2c"]:
            make = lambda h: lf.CField(lf.Lattice(3, case["N"], h), case["C"], code)  # noqa: E731
            s["r"], s["k"], s["back"] = make(case["halo"]), make(case["khalo"]), make(case["halo"])
        else:
            s["r"], s["back"] = lf.Field(lat, case["C"], code), lf.Field(lat, case["C"], code)
            s["k"] = lf.KField(lat, case["khalo"], case["C"], code)
        s["r"].interior().copy_(_field_values(case, seed))
        s["there"], s["home"] = lf.PlanFFT(s["r"], s["k"]), lf.PlanFFT(s["back"], s["k"])
        return s
    if f == "diffpm":
        pos, vel, s["target"] = _diffpm_inputs(case, seed)
        s["pos"], s["vel"] = pos.requires_grad_(), vel.requires_grad_()
        s["model"] = DiffPM(case["N"], case["np"], case["nsteps"], 1.0 / case["np"], 0.02, code)
        return s
    s["parts"] = _container(case, seed)
    lat = lf.Lattice(3, case["N"], case.get("halo", 1))
    if f == "project":
        s["field"] = lf.Field(lat, KINDS[case["kind"]][1], code)
        return s
    s["rho"], s["phi"] = lf.Field(lat, 1, code), lf.Field(lat, 1, code)
    if f == "step":
        s["plan"] = lf.PlanFFT(s["rho"], None)
    else:
        s["k"] = lf.KField(lat, 0, 1, code)
        s["there"], s["home"] = lf.PlanFFT(s["rho"], s["k"]), lf.PlanFFT(s["phi"], s["k"])
    return s


# ---------------------------------------------------------------- a pass
def run(s):
    return globals()["_run_" + s["case"]["family"]](s, s["case"])


def _run_step(s, case):
    acc = lf.ACC_FIXED64 if case["fixed"] else lf.ACC_NATIVE
    for _ in range(2):
        lf.pm_step(s["parts"], s["plan"], s["rho"], s["phi"], DT, DT, acc)
    return {"rho": s["rho"].t, "phi": s["phi"].t}


def _run_driver(s, case):
    parts, rho, phi, k = s["parts"], s["rho"], s["phi"], s["k"]
    lf.projection_init(rho)
    lf.scalarProjectionCIC_project(parts, rho)
    lf.scalarProjectionCIC_comm(rho)
    s["there"].execute(lf.FFT_FORWARD)
    lf.poisson_green(k, scale=1.0 / case["N"] ** 3)
    s["home"].execute(lf.FFT_BACKWARD)
    phi.updateHalo()
    rho.updateHalo()
    vmax = parts.updateVel(lf.updateVel_cicKick, DT, [phi], 1)
    parts.moveParticles(lf.move_particles_simple, DT)
    return {"rho": rho.t, "k": k.t, "phi": phi.t, "vmax": vmax}


def _run_project(s, case):
    field, parts = s["field"], s["parts"]
    if case["target"] == "calls":
        project, comm = CALLS[case["kind"]]
        lf.projection_init(field)
        project(parts, field)
        comm(field)
    else:
        parts.deposit(KINDS[case["kind"]][0], field, lf.DEP_PERIODIC_SET)
    field.updateHalo()
    return field.t


def _run_fft(s, case):
    s["there"].execute(lf.FFT_FORWARD)
    s["home"].execute(lf.FFT_BACKWARD)
    return {"k": s["k"].t, "back": s["back"].t}


def _run_diffpm(s, case):
    s["pos"].grad = s["vel"].grad = None
    loss = pm_density_loss(s["pos"], s["vel"], s["target"], s["model"])
    loss.backward()
    return {"loss": loss, "pos": s["pos"].grad, "vel": s["vel"].grad}


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    N, es = case["N"], 4 if case["dtype"] == "f32" else 8
    V = N ** 3
    f = case["family"]
    if f == "fft":
        C = case["C"]
        k = (V if case["c2c"] else (N // 2 + 1) * N * N) * C * 2 * es
        r = V * C * es * (2 if case["c2c"] else 1)
        return {"bytes": 2 * (r + k), "flops": 2 * (5 if case["c2c"] else 2.5) * V * C * math.log2(V)}
    n = case["np"]
    state = n * (4 + 6 * es if case["dtype"] == "f32" else 6 * es)  # positions and velocities as they are kept
    solve = 5 * V * math.log2(V) + 4 * V
    if f == "step":
        return {"bytes": 2 * (2 * state + 2 * V * es), "flops": 2 * (solve + 150.0 * n)}
    if f == "driver":
        return {"bytes": 2 * state + V * es * 4, "flops": solve + 150.0 * n}
    if f == "project":
        C = KINDS[case["kind"]][1]
        read = n * (4 + 3 * es if case["dtype"] == "f32" else 3 * es) + (n * 3 * es if C > 1 else 0)
        return {"bytes": read + V * C * es + (n * es if case["masses"] else 0), "flops": 24.0 * n * C}
    # forward: every step reads and writes the particles; backward: reads them, and the adjoints twice
    steps = case["nsteps"]
    return {"bytes": steps * (2 * state + state + 4 * n * 6 * es) + 4 * n * 3 * es + V * es,
            "flops": steps * (3 * solve + 900.0 * n)}


# ---------------------------------------------------------------- the same in 64 bits
def _corners(pos, N):
    x = pos * N
    c = torch.floor(x)
    return c.long() % N, x - c


def _sites(c, off, N):
    """flat index [z, y, x] of the sites c + off"""
    i = [(c[:, d] + off[d]) % N for d in range(3)]
    return (i[2] * N + i[1]) * N + i[0]


def _axis(u, how):
    """(site offset, weight) pairs of one axis: vertices, links (half a cell up) or the nearest"""
    if how == "nearest":
        return [(0, torch.ones_like(u))]
    if how == "link":
        t = u - 0.5
        return [(-1, (-t).clamp_min(0)), (0, 1 - t.abs()), (1, t.clamp_min(0))]
    return [(0, 1 - u), (1, u)]


def _deposit(pos, q, N, how=("vertex",) * 3):
    c, u = _corners(pos, N)
    f = torch.zeros(N ** 3, dtype=torch.float64, device=pos.device)
    ax = [_axis(u[:, d], how[d]) for d in range(3)]
    for k, wz in ax[2]:
        for j, wy in ax[1]:
            for i, wx in ax[0]:
                f = f.index_add(0, _sites(c, (i, j, k), N), q * wx * wy * wz)
    return f.reshape(N, N, N)


def _potential(rho, want_k=False):
    N = rho.shape[0]
    s = 4.0 * N * N * torch.sin(math.pi * torch.arange(N, device=rho.device, dtype=torch.float64) / N) ** 2
    k2 = s[:, None, None] + s[None, :, None] + s[None, None, : N // 2 + 1]
    k2[0, 0, 0] = 1.0
    k = torch.fft.rfftn(rho) * (-1.0 / k2)
    k[0, 0, 0] = 0.0
    phi = torch.fft.irfftn(k, s=(N, N, N))
    return (phi, k / N ** 3) if want_k else phi


def _accel(phi, pos):
    N = phi.shape[0]
    c, u = _corners(pos, N)
    F = [-(torch.roll(phi, -1, 2 - d) - torch.roll(phi, 1, 2 - d)).reshape(-1) * (N / 2) for d in range(3)]
    a = [0.0, 0.0, 0.0]
    for k, wz in _axis(u[:, 2], "vertex"):
        for j, wy in _axis(u[:, 1], "vertex"):
            for i, wx in _axis(u[:, 0], "vertex"):
                at, w = _sites(c, (i, j, k), N), wx * wy * wz
                a = [a[d] + w * F[d][at] for d in range(3)]
    return torch.stack(a, 1)


def _padded(f, h):
    """[z, y, x(, c)] with h periodic ghost sites, as a Field of the framework stores it"""
    f = f if f.dim() == 4 else f[..., None]
    for d in range(3):
        n = f.shape[d]
        f = f.index_select(d, torch.arange(-h, n + h, device=f.device) % n)
    return f


def _inside(f, h):
    """the same with the ghosts zero"""
    f = f if f.dim() == 4 else f[..., None]
    return torch.nn.functional.pad(f, (0, 0) + (h, h) * 3)


def exact(case, seed):
    f = case["family"]
    if f == "fft":
        return _exact_fft(case, seed)
    if f == "diffpm":
        return _exact_diffpm(case, seed)
    if not case["upload"]:
        return None
    pos, vel, mass = _particles(case, seed)
    N, n = case["N"], case["np"]
    q = mass * N ** 3 if case.get("masses") else torch.full((n,), N ** 3 / n, dtype=torch.float64, device="cuda")
    if f == "project":
        return _exact_project(case, pos, vel, q)
    if f == "driver":
        rho = _deposit(pos, q, N)
        phi, k = _potential(rho, True)
        v = vel + DT * _accel(phi, pos)
        return {"rho": _padded(rho, 1), "k": torch.view_as_real(k.permute(1, 0, 2).contiguous())[..., None, :],
                "phi": _padded(phi, 1), "vmax": float(v.square().sum(1).max().sqrt())}
    for _ in range(2):
        rho = _deposit(pos, q, N)
        phi = _potential(rho)
        vel = vel + DT * _accel(phi, pos)
        pos = pos + DT * vel
        pos = pos - torch.floor(pos)
    # the step leaves its fields' ghosts alone or clears them
    return {"rho": _inside(rho, 1), "phi": _inside(phi, 1)}


def _exact_project(case, pos, vel, q):
    N, kind = case["N"], case["kind"]
    axes = ("x", "y", "z")
    pairs = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)]
    how = "nearest" if kind.endswith("ngp") else "link"
    if kind == "scalar":
        comps = [_deposit(pos, q, N)]
    elif kind.startswith("vector"):
        comps = [_deposit(pos, q * vel[:, a], N, [how if d == a else "vertex" for d in range(3)])
                 for a in range(len(axes))]
    else:
        comps = [_deposit(pos, q * vel[:, a] * vel[:, b], N,
                          [how if a != b and d in (a, b) else "vertex" for d in range(3)]) for a, b in pairs]
    return _padded(torch.stack(comps, -1), case["halo"])


def _exact_fft(case, seed):
    N, C = case["N"], case["C"]
    if N ** 3 * C > 1024 ** 3:
        return None
    v = _field_values(case, seed).double()
    if case["c2c"]:
        z = torch.view_as_complex(v)
        k = torch.fft.fftn(z, dim=(0, 1, 2)).permute(1, 2, 0, 3)  # [kz, ky, kx] -> storage [ky, kx, kz]
        k = torch.view_as_real(k.contiguous()).flatten(3)
        return {"k": _inside(k, case["khalo"]).unflatten(3, (C, 2)),
                "back": _inside(v.flatten(3) * N ** 3, case["halo"]).unflatten(3, (C, 2))}
    k = torch.fft.rfftn(v, dim=(0, 1, 2))
    k = torch.view_as_real(k.permute(1, 0, 2, 3).contiguous()).flatten(3)  # storage [ky, kz, kx]
    return {"k": _inside(k, case["khalo"]).unflatten(3, (C, 2)), "back": _inside(v * N ** 3, case["halo"])}


def _exact_diffpm(case, seed):
    N, n, dt = case["N"], case["np"], 0.02
    pos0, vel0, target = (t.double() for t in _diffpm_inputs(case, seed))
    pos0, vel0 = pos0.requires_grad_(), vel0.requires_grad_()
    q = torch.full((n,), N ** 3 / n, dtype=torch.float64, device="cuda")

    def step(x, v):
        v = v + dt * _accel(_potential(_deposit(x, q, N)), x)
        return x + dt * v, v

    from torch.utils.checkpoint import checkpoint
    x, v = pos0, vel0
    for _ in range(case["nsteps"]):
        x, v = checkpoint(step, x, v, use_reentrant=False)
    loss = (_deposit(x, q, N) - target).square().sum()
    gp, gv = torch.autograd.grad(loss, (pos0, vel0))
    return {"loss": loss.detach(), "pos": gp, "vel": gv}
