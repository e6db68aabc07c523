"""The work that users of this library have it do, as cases that can be timed.

Paths, each through the public entry points:

  derivs       tree build, density iteration, primitive variables and force of
               all particles on arrays resident in HBM (integrator.derivs, the
               reference's deriv.f90): every step of a run on a global
               timestep and the synchronisation steps of a run on bins.
  step         one whole leapfrog step inside the library
               (integrator.evolve_graph) on a global timestep.
  substep      one substep on block timesteps (integrator.evolve_graph) with a
               chosen fraction of the particles active.
  grad_density tree, density iteration and the adjoint of the density
               summation on HBM arrays: one iteration of gradient relaxation.
  grad_step    forward and backward of one differentiable leapfrog step
               through torch.autograd (adjoint.leapfrog_step, host tensors).

Set-ups are those of phantom_amd.setups (uniform box, shock tube, MHD and dust
box, polytrope), drawn on the GPU so that they are quick to make.  Every pass
starts from the same positions and smoothing lengths: one device copy restores
the arrays that the pass advances, standing for the predictor that moves them
in a run.
"""
import functools
import math

import numpy as np
import torch

from phantom_amd import abi, adjoint, integrator, setups, sph
from phantom_amd.device import DeviceArray as D

PI_PH = 3.1415926536  # the reference's pi (physcon.f90:23)
GAMMA = 5.0 / 3.0
BOX = (-0.5, 0.5)
# part of the particles in each bin of the block-timestep runs (setups.LEVELS_4):
# substeps 64, 32, 8 and 1 of 64 have 1, 1/2, 1/8 and 1/64 of them active
NBINMAX = 6


def listed():
    return [
        # the smallest calls: a test-sized box, where launches and latency are all
        dict(name="box_4k", path="derivs", setup="box", nx=16, ny=16, nz=16, kernel="cubic", gas="isothermal",
             precision="fp64"),
        # the 64^3 isothermal box (the small configuration of the benchmark)
        dict(name="box_262k", path="derivs", setup="box", nx=64, ny=64, nz=64, kernel="cubic", gas="isothermal",
             precision="fp64"),
        # the benchmark's default: 8.4M adiabatic particles, the largest that is run in earnest
        dict(name="box_8M", path="derivs", setup="box", nx=256, ny=256, nz=128, kernel="cubic", gas="adiabatic",
             precision="fp64"),
        # the 1.1M-particle shock tube on its lattice, quintic kernel (the start of a run)
        dict(name="tube_1M", path="derivs", setup="tube", ny=58, kernel="quintic", gas="adiabatic",
             precision="fp64"),
        # 128^3 ideal MHD with one-fluid dust, quintic kernel, all particles active
        dict(name="mhd_dust_2M", path="derivs", setup="mhd_dust", nx=128, ny=128, nz=128, kernel="quintic",
             gas="adiabatic", precision="fp64"),
        # block timesteps: an ordinary substep (1/8 active) of the same box
        dict(name="substep_8th_2M", path="substep", setup="mhd_dust", nx=128, ny=128, nz=128, kernel="quintic",
             gas="adiabatic", precision="fp64", substep=8),
        # block timesteps: the deepest substep (1/64 active), the most frequent one, on an odd box
        dict(name="substep_64th_1M", path="substep", setup="mhd_dust", nx=101, ny=97, nz=103, kernel="quintic",
             gas="adiabatic", precision="fp64", substep=1),
        # a global-timestep run of an adiabatic box in mixed precision, odd sizes
        dict(name="step_mixed_850k", path="step", setup="box", nx=95, ny=101, nz=89, kernel="cubic",
             gas="adiabatic", precision="mixed"),
        # a small self-gravitating star (stellar tests, relaxation)
        dict(name="star_30k", path="derivs", setup="polytrope", n=30000, kernel="cubic", gas="adiabatic",
             precision="fp64"),
        # the self-gravitating n = 1.5 polytrope of the benchmark
        dict(name="star_1M", path="derivs", setup="polytrope", n=1048576, kernel="cubic", gas="adiabatic",
             precision="fp64"),
        # the density adjoint of gradient relaxation, n = 3 polytrope
        dict(name="grad_density_500k", path="grad_density", setup="relaxation", n=500000, kernel="cubic",
             gas="adiabatic", precision="fp64"),
        # forward and backward of a differentiable step
        dict(name="grad_step_100k", path="grad_step", setup="box", nx=47, ny=45, nz=48, kernel="cubic",
             gas="isothermal", precision="fp64"),
    ]


def draw(rng):
    path = rng.choice(["derivs"] * 4 + ["step", "substep", "grad_density", "grad_step"])
    kernel = rng.choice(["cubic", "quintic"])

    def size(lo, hi):
        return math.exp(rng.uniform(math.log(lo), math.log(hi)))

    def sides(n):
        m = n ** (1.0 / 3.0)
        s = [max(14, int(round(m * rng.uniform(0.8, 1.25)))) for _ in range(3)]
        return dict(zip(("nx", "ny", "nz"), s))

    if path == "grad_density":
        return dict(path=path, setup="relaxation", n=int(size(20e3, 700e3)), kernel="cubic", gas="adiabatic",
                    precision="fp64")
    if path == "grad_step":
        return dict(path=path, setup="box", **sides(size(10e3, 200e3)), kernel=kernel, gas="isothermal",
                    precision="fp64")
    if path == "substep":
        return dict(path=path, setup="mhd_dust", **sides(size(100e3, 1.6e6)), kernel=kernel, gas="adiabatic",
                    precision="fp64", substep=rng.choice([64, 32, 8, 1]))
    if path == "step":
        return dict(path=path, setup="box", **sides(size(10e3, 2.5e6)), kernel=kernel, gas="adiabatic",
                    precision=rng.choice(["fp64", "mixed"]))
    setup = rng.choice(["box", "box", "tube", "mhd_dust", "polytrope"])
    if setup == "box":
        gas, precision = rng.choice([("isothermal", "fp64"), ("adiabatic", "fp64"), ("adiabatic", "mixed")])
        return dict(path=path, setup=setup, **sides(size(4e3, 5e6)), kernel=kernel, gas=gas, precision=precision)
    if setup == "tube":
        return dict(path=path, setup=setup, ny=int(size(14, 70)), kernel=kernel, gas="adiabatic",
                    precision=rng.choice(["fp64", "mixed"]))
    if setup == "mhd_dust":
        return dict(path=path, setup=setup, **sides(size(10e3, 2e6)), kernel=kernel, gas="adiabatic",
                    precision="fp64")
    return dict(path=path, setup=setup, n=int(size(10e3, 1.5e6)), kernel="cubic", gas="adiabatic",
                precision=rng.choice(["fp64", "fp64", "mixed"]))


# ----------------------------------------------------------------------------
# particle sets
# ----------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) % (2 ** 31))
    return g


def _rand(g, shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(shape, generator=g, dtype=torch.float64, device="cuda")


def _lattice(nx, ny, nz, lo, hi):
    ax = [lo[c] + (torch.arange(m, dtype=torch.float64, device="cuda") + 0.5) * ((hi[c] - lo[c]) / m)
          for c, m in enumerate((nx, ny, nz))]
    z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")  # x fastest, as set_unifdis
    return torch.stack([x.ravel(), y.ravel(), z.ravel()], dim=1)


@functools.lru_cache(maxsize=None)
def _lane_emden(nindex):
    return setups.lane_emden(nindex, dxi=1e-3)


def _hfact(case):
    return 1.2 if case["kernel"] == "cubic" else 1.0


def _particles(case, seed):
    """Tensors x (n,3), h, v, u, alpha (n,3) and, with MHD and dust, B/rho and
    the dust variable; the particle mass, box and hfact."""
    g = _gen(seed)
    hf = _hfact(case)
    d = dict(lo=(BOX[0],) * 3, hi=(BOX[1],) * 3, hfact=hf, radkern=2.0 if case["kernel"] == "cubic" else 3.0)
    if case["setup"] in ("box", "mhd_dust"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        dx = 1.0 / max(nx, ny, nz)  # cubic cells: the box follows the sides
        d["lo"], d["hi"] = tuple(-0.5 * dx * m for m in (nx, ny, nz)), tuple(0.5 * dx * m for m in (nx, ny, nz))
        x = _lattice(nx, ny, nz, d["lo"], d["hi"])
        n = x.shape[0]
        x += _rand(g, (n, 3), -0.05 * dx, 0.05 * dx)
        h = torch.full((n,), hf * dx, dtype=torch.float64, device="cuda")
        side = [d["hi"][c] - d["lo"][c] for c in range(3)]
        sx, sy = ((x[:, c] - d["lo"][c]) / side[c] for c in (0, 1))
        phase = _rand(g, (2,))
        v = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
        if case["setup"] == "box":  # shear flow of setups.uniform_box
            d["pmass"] = side[0] * side[1] * side[2] / n
            v[:, 0] = 0.1 * torch.sin(2 * PI_PH * (sy + phase[0]))
            u = torch.full((n,), 1.5, dtype=torch.float64, device="cuda")
        else:  # Orszag-Tang-type flow with dust of setups.mhd_dust_box
            rho0, P0 = 25.0 / (36.0 * PI_PH), 5.0 / (12.0 * PI_PH)
            d["pmass"] = rho0 * side[0] * side[1] * side[2] / n
            v[:, 0] = -torch.sin(2 * PI_PH * (sy + phase[0]))
            v[:, 1] = torch.sin(2 * PI_PH * (sx + phase[1]))
            v[:, 2] = 0.01
            eps = torch.exp(_rand(g, (n,), math.log(0.01), math.log(0.5)))
            u = P0 / ((GAMMA - 1.0) * rho0 * (1.0 - eps))
            B = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
            B[:, 0] = -torch.sin(2 * PI_PH * (sy + phase[0])) / (math.sqrt(4 * PI_PH) * rho0)
            B[:, 1] = torch.sin(4 * PI_PH * (sx + phase[1])) / (math.sqrt(4 * PI_PH) * rho0)
            d["Bevol"], d["dustevol"], d["rho0"] = B, torch.sqrt(eps / (1.0 - eps)), rho0
    elif case["setup"] == "tube":
        ny = case["ny"]
        dx = 0.1 / ny
        nxl = int(round(0.5 / dx))
        left = _lattice(nxl, ny, ny, (-0.5, -0.05, -0.05), (0.0, 0.05, 0.05))
        right = _lattice(nxl // 2, ny // 2, ny // 2, (0.0, -0.05, -0.05), (0.5, 0.05, 0.05))
        x = torch.cat([left, right])
        n, nl = x.shape[0], left.shape[0]
        d["lo"], d["hi"] = (-0.5, -0.05, -0.05), (0.5, 0.05, 0.05)
        d["pmass"] = (0.5 * 0.01 + 0.125 * 0.5 * 0.01) / n
        h = torch.full((n,), hf * dx, dtype=torch.float64, device="cuda")
        h[nl:] = 2.0 * hf * dx
        v = 0.01 * torch.randn((n, 3), generator=g, dtype=torch.float64, device="cuda")
        u = torch.full((n,), 1.0 / (GAMMA - 1.0), dtype=torch.float64, device="cuda")
        u[nl:] = 0.1 / ((GAMMA - 1.0) * 0.125)
    else:  # polytropes: a jittered lattice in the unit sphere stretched to the Lane-Emden profile
        nindex = 1.5 if case["setup"] == "polytrope" else 3.0
        nside = int(round((case["n"] * 6.0 / math.pi) ** (1.0 / 3.0)))
        dx = 2.0 / nside
        x = _lattice(nside, nside, nside, (-1.0,) * 3, (1.0,) * 3)
        x = x[torch.sqrt((x * x).sum(dim=1)) < 1.0 - 0.18 * dx]  # inside the sphere wherever the jitter puts them
        x = x + _rand(g, x.shape, -0.1 * dx, 0.1 * dx)
        r0 = torch.sqrt((x * x).sum(dim=1))
        n = x.shape[0]
        xi, th, dth = _lane_emden(nindex)
        xi1 = xi[-1]
        menc = -(xi * xi) * dth
        q = r0.cpu().numpy()
        r = np.interp(q ** 3, menc / menc[-1], xi / xi1)
        x = x * torch.from_numpy(r / np.maximum(q, 1e-300)).cuda()[:, None]
        rho_c = xi1 / (4.0 * math.pi * (-dth[-1]))
        K = 4.0 * math.pi / xi1 ** 2 * rho_c ** (1.0 - 1.0 / nindex) / (nindex + 1.0)
        rho = torch.from_numpy(np.maximum(rho_c * np.interp(r * xi1, xi, th) ** nindex, 1e-3 * rho_c)).cuda()
        d["pmass"] = 1.0 / n
        d["lo"], d["hi"] = (-2.0,) * 3, (2.0,) * 3
        h = hf * (d["pmass"] / rho) ** (1.0 / 3.0)
        if nindex == 3.0:  # relaxation starts from a noisy star
            x = x + 0.02 * h[:, None] * torch.randn((n, 3), generator=g, dtype=torch.float64, device="cuda")
        v = 0.01 * torch.randn((n, 3), generator=g, dtype=torch.float64, device="cuda")
        u = K * rho ** (1.0 / nindex) * (1.5 if nindex == 1.5 else 3.0)
    alpha = torch.zeros((x.shape[0], 3), dtype=torch.float32, device="cuda")
    alpha[:, 0] = _rand(g, (x.shape[0],)).float()
    L = [d["hi"][c] - d["lo"][c] for c in range(3)]
    if case["setup"] in ("box", "mhd_dust"):  # the jitter may carry a particle over the edge
        for c in range(3):
            xc = x[:, c]
            x[:, c] = torch.where(xc < d["lo"][c], xc + L[c], torch.where(xc > d["hi"][c], xc - L[c], xc))
    d.update(x=x, h=h, v=v, u=u, alpha=alpha, gen=g)
    return d


def _params(case, d):
    p = abi.default_params(abi.KERNEL_CUBIC if case["kernel"] == "cubic" else abi.KERNEL_QUINTIC)
    p.xmin, p.ymin, p.zmin = d["lo"]
    p.xmax, p.ymax, p.zmax = d["hi"]
    p.massoftype_gas = d["pmass"]
    p.maxp = d["x"].shape[0]
    p.precision = abi.PREC_MIXED if case["precision"] == "mixed" else abi.PREC_FP64
    if case["gas"] == "isothermal":
        p.maxvxyzu, p.ieos, p.polyk = 3, 1, 1.0
    else:
        p.maxvxyzu, p.ieos, p.gamma = 4, 2, GAMMA
    if case["setup"] == "mhd_dust":
        p.mhd, p.use_dustfrac, p.ndustsmall, p.idrag = 1, 1, 1, 2
        p.K_code = d["rho0"] * 0.99
    if case["setup"] in ("polytrope", "relaxation"):
        p.periodic = 0
        p.gravity = 1 if case["setup"] == "polytrope" else 0
        p.tree_accuracy = 0.5
        if case["setup"] == "relaxation":
            p.gamma = 4.0 / 3.0
    if case["path"] == "substep":
        p.ind_timesteps = 1
        p.dtmax = 0.016
    return p


class _View:
    """A device array of the library's callers as the tensor of the same memory."""

    def __init__(self, a):
        self.keep = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr=a.dtype.str, data=(a.ptr, False), version=2)


def _tensor(a):
    return torch.as_tensor(_View(a), device="cuda")


def _np(t):
    return None if t is None else t.cpu().numpy()


# ----------------------------------------------------------------------------
# states and passes
# ----------------------------------------------------------------------------
# arrays that a pass advances, restored before it
_MOVES = ("xyzh", "vxyzu", "fxyzu", "alphaind", "divcurlv", "eos_vars", "Bevol", "dBevol", "dustevol", "ddustevol",
          "ibin", "ibin_old", "ibin_wake", "twas")
_DERIVS_OUT = ("xyzh", "gradh", "divcurlv", "dvdx", "alphaind", "eos_vars", "fxyzu", "divcurlB", "dBevol", "divBsymm",
               "dustfrac", "ddustevol", "deltav", "tstop")
_STEP_OUT = ("xyzh", "vxyzu", "fxyzu", "alphaind", "gradh", "divcurlv", "Bevol", "dBevol", "dustevol", "ddustevol",
             "ibin", "ibin_wake", "twas")


def prepare(case, seed):
    d = _particles(case, seed)
    p = _params(case, d)
    n = d["x"].shape[0]
    xyzh = torch.cat([d["x"], d["h"][:, None]], dim=1)
    vxyzu = torch.cat([d["v"], d["u"][:, None]], dim=1)[:, :p.maxvxyzu].contiguous()
    ctx = sph.Context(p)
    st = dict(case=case, ctx=ctx, p=p, n=n)
    g = d["gen"]
    if case["path"] == "grad_step":
        st["h0"] = d["h"].cpu()
        st["x"] = d["x"].cpu().requires_grad_(True)
        st["v"] = d["v"].cpu().requires_grad_(True)
        st["gx"] = _rand(g, (n, 3), -1.0, 1.0).cpu()
        st["gv"] = _rand(g, (n, 3), -1.0, 1.0).cpu()
        st["dt"] = 0.1 * float(d["h"].min())
        return st
    if case["path"] == "grad_density":
        st["xyzh"], st["vxyzu"] = D.from_numpy(_np(xyzh)), D.from_numpy(_np(vxyzu))
        st["out"] = dict(divcurlv=D((n, 1), np.float32), alphaind=D.from_numpy(_np(d["alpha"])),
                         gradh=D((n, 1), np.float32), dvdx=D((n, 9), np.float32))
        st["rhobar"] = D.from_numpy(_np(_rand(g, (n,), -1.0, 1.0)))
        st["dxyz"] = D((n, 3), np.float64)
        ctx.maketree(st["xyzh"], leaf=False)  # the h that the last iteration of the relaxation converged to
        ctx.densityiterate(1, st["xyzh"], st["vxyzu"], **st["out"])
        st["t"] = {k: _tensor(st[k]) for k in ("xyzh", "dxyz")}
        start = st["t"]["xyzh"].clone()
        start[:, 3] *= 1.0 + _rand(g, (n,), -1e-3, 1e-3)  # as the moved positions leave it
        st["start"] = start
        return st
    s = integrator.State(p, _np(xyzh), _np(vxyzu), _np(d["alpha"]), Bevol=_np(d.get("Bevol")),
                         dustevol=_np(d.get("dustevol")), device=case["path"] != "substep")
    if case["path"] == "substep":
        s.enable_bins(0)
        integrator.init_ind(ctx, s)
        perm = torch.randperm(n, generator=g, device="cuda").cpu().numpy()
        b = np.zeros(n, np.int8)
        at = 0
        for k, (lev, frac) in enumerate(setups.LEVELS_4):
            to = n if k == len(setups.LEVELS_4) - 1 else at + int(round(frac * n))
            b[perm[at:to]] = lev
            at = to
        s.ibin[:] = b
        s.ibin_old[:] = b
        s.ibin_wake[:] = 0
        s.nbinmax = NBINMAX
        s.twas[:] = 0.5 * (p.dtmax / 2.0 ** b.astype(np.float64))
        s = s.copy(device=True)
        st["istepfrac"] = case["substep"] - 1
    else:
        integrator.init_global(ctx, s)  # the first derivatives of a run
    st["s"] = s
    st["t"] = {k: _tensor(getattr(s, k)) for k in integrator.State.ARRAYS if getattr(s, k) is not None}
    if p.gravity:
        st["t"]["poten"] = _tensor(ctx._poten)
    if case["path"] == "derivs":
        if case["setup"] == "polytrope":
            # the h of the last step, off by what a step's prediction leaves
            start = st["t"]["xyzh"].clone()
            start[:, 3] *= 1.0 + _rand(g, (n,), -1e-3, 1e-3)
        else:
            start = xyzh.clone()
        moves = ["xyzh"]
        st["save"] = [start]
    else:
        moves = [k for k in _MOVES if k in st["t"]]
        st["save"] = [st["t"][k].clone() for k in moves]
        st["scalars"] = {k: getattr(s, k) for k in integrator.State.SCALARS}
        if case["path"] == "step":
            st["dt"] = min(s.dtforce, s.dtcourant)
    st["moves"] = [st["t"][k] for k in moves]
    return st


def run(st):
    path, ctx = st["case"]["path"], st["ctx"]
    if path == "grad_step":
        st["x"].grad = st["v"].grad = None
        x1, v1 = adjoint.leapfrog_step(st["x"], st["v"], st["h0"], st["dt"], ctx)
        torch.autograd.backward([x1, v1], [st["gx"], st["gv"]])
        return dict(x=x1.detach(), v=v1.detach(), dx=st["x"].grad, dv=st["v"].grad)
    if path == "grad_density":
        st["t"]["xyzh"].copy_(st["start"])
        ctx.maketree(st["xyzh"], leaf=False)
        ctx.densityiterate(1, st["xyzh"], st["vxyzu"], **st["out"])
        ctx.density_vjp(st["xyzh"], rhobar=st["rhobar"], dxyz=st["dxyz"])
        return dict(st["t"])
    s, t = st["s"], st["t"]
    for a, b in zip(st["moves"], st["save"]):
        a.copy_(b)
    if path == "derivs":
        dt = integrator.derivs(ctx, 1, s)
        out = {k: t[k] for k in _DERIVS_OUT + ("poten",) if k in t}
        out["dt"] = float(dt)
        return out
    for k, v in st["scalars"].items():
        setattr(s, k, v)
    if path == "step":
        _, _, dt, _ = integrator.evolve_graph(ctx, s, 1, dt=st["dt"])
        return dict({k: t[k] for k in _STEP_OUT if k in t}, dt=float(dt))
    s.istepfrac = st["istepfrac"]
    _, _, _, o = integrator.evolve_graph(ctx, s, 1, time=st["istepfrac"] / 64.0 * st["p"].dtmax)
    return dict({k: t[k] for k in _STEP_OUT if k in t}, nactive=int(o[0]["nactive"]), nbinmax=int(s.nbinmax))


# ----------------------------------------------------------------------------
# the least work of a pass
# ----------------------------------------------------------------------------
def _count(case):
    if "nx" in case:
        return case["nx"] * case["ny"] * case["nz"]
    if "n" in case:
        return case["n"]
    ny = case["ny"]
    nxl = int(round(5 * ny))
    return nxl * ny * ny + (nxl // 2) * (ny // 2) ** 2


def work(case):
    """Arrays of the caller read and written once, and the arithmetic of the
    interacting pairs: 2.5 passes of the h iteration (34 operations a pair),
    one of all density sums (102, MHD 34 more) and the pair force (124, MHD
    110 and dust 40 more); a density or step adjoint has the forward sums and a
    pass of the same size back.  With self-gravity about 1000 near particles
    of 20 operations."""
    n = _count(case)
    ngb = 4.0 / 3.0 * math.pi * ((2.0 if case["kernel"] == "cubic" else 3.0) * _hfact(case)) ** 3
    mhd = case["setup"] == "mhd_dust"
    act = n * case["substep"] / 64.0 if case["path"] == "substep" else float(n)
    if case["path"] == "substep" and case["substep"] == 32:
        act = n * 0.5
    dens = 2.5 * 34 + 102 + (34 if mhd else 0)
    force = 124 + (150 if mhd else 0)
    per = 32 * 2 + 32 * 2 + 8 + 4 + 36 + 12 + 24 + 32 + (16 + 32 * 2 + 4 + 8 * 3 + 24 + 8 if mhd else 0)
    if case["path"] == "grad_density":
        return dict(bytes=n * (32 * 2 + 32 + 8 + 24), flops=n * ngb * (dens + 102))
    if case["path"] == "grad_step":
        return dict(bytes=n * 8 * (3 * 6 + 2), flops=n * ngb * 2 * (2 * dens + 2 * force))
    flops = act * ngb * (dens + force)
    if case["setup"] == "polytrope":
        flops += act * 1000 * 20
    extra = 0
    if case["path"] in ("step", "substep"):
        extra = n * (32 * 6 + (32 * 6 if mhd else 0))
    return dict(bytes=act * per + extra, flops=flops)


# ----------------------------------------------------------------------------
# the same in 64 bits with torch alone: density and hydrodynamic force of
# periodic boxes (pairs from a grid of cells)
# ----------------------------------------------------------------------------
def _kernel(case, q):
    if case["kernel"] == "cubic":
        a, b = (2.0 - q).clamp(min=0.0), (1.0 - q).clamp(min=0.0)
        return 0.25 * a ** 3 - b ** 3, -0.75 * a ** 2 + 3.0 * b ** 2
    a, b, c = ((k - q).clamp(min=0.0) for k in (3.0, 2.0, 1.0))
    return a ** 5 - 6.0 * b ** 5 + 15.0 * c ** 5, -5.0 * (a ** 4 - 6.0 * b ** 4 + 15.0 * c ** 4)


class _Pairs:
    """The particles in cells no smaller than the largest kernel radius."""

    def __init__(self, x, lo, hi, radius):
        self.x = x
        self.L = torch.tensor([h - l for l, h in zip(lo, hi)], dtype=torch.float64, device=x.device)
        m = [max(3, int(float(s) / radius)) for s in self.L]
        assert all(float(s) / k >= radius * 0.999999 for s, k in zip(self.L, m)), "box too small for the grid"
        m_t = torch.tensor(m, device=x.device)
        c = torch.minimum(((x - torch.tensor(lo, device=x.device)) / self.L * m_t).long().clamp(min=0), m_t - 1)
        cell = (c[:, 2] * m[1] + c[:, 1]) * m[0] + c[:, 0]
        order = torch.argsort(cell)
        cnt = torch.bincount(cell, minlength=m[0] * m[1] * m[2])
        first = torch.cumsum(cnt, 0) - cnt
        M = int(cnt.max())
        tab = torch.full((cnt.numel(), M), -1, dtype=torch.long, device=x.device)
        tab[cell[order], torch.arange(x.shape[0], device=x.device) - first[cell[order]]] = order
        self.tab = tab
        k = torch.arange(cnt.numel(), device=x.device)
        kx, ky, kz = k % m[0], (k // m[0]) % m[1], k // (m[0] * m[1])
        nb = []
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                for e in (-1, 0, 1):
                    nb.append((((kz + a) % m[2]) * m[1] + (ky + b) % m[1]) * m[0] + (kx + e) % m[0])
        self.nb = torch.stack(nb, dim=1)

    def chunks(self, most=60_000_000):
        M = self.tab.shape[1]
        step = max(1, most // (M * 27 * M))
        for k in range(0, self.tab.shape[0], step):
            i = self.tab[k:k + step].reshape(-1)
            rows = torch.nonzero(i >= 0).squeeze(1)
            i = i[rows]
            j = self.tab[self.nb[k:k + step][rows // M]].reshape(rows.numel(), 27 * M)
            ok = (j >= 0) & (j != i[:, None])
            j = j.clamp(min=0)
            dx = self.x[i][:, None, :] - self.x[j]
            dx = dx - self.L * torch.round(dx / self.L)
            yield i, j, ok, dx, (dx * dx).sum(dim=2)


def exact(case, seed):
    if case["path"] != "derivs" or case["setup"] == "polytrope" or _count(case) > 1_300_000:
        return None
    d = _particles(case, seed)
    x, pm, hf, R = d["x"], d["pmass"], d["hfact"], d["radkern"]
    n = x.shape[0]
    hydro = case["setup"] != "mhd_dust"
    cn = 1.0 / PI_PH if case["kernel"] == "cubic" else 1.0 / (120.0 * PI_PH)
    w0 = 1.0 if case["kernel"] == "cubic" else 66.0
    if any((b - a) / 3.0 < 1.3 * R * float(d["h"].max()) for a, b in zip(d["lo"], d["hi"])):
        return None  # the grid needs three cells a side
    pairs = _Pairs(x, d["lo"], d["hi"], 1.2 * R * float(d["h"].max()))
    v, u, h0 = d["v"], d["u"], d["h"]

    def rhoh(h):
        return pm * (hf / h) ** 3

    # h iteration (dens.F90:1382-1466), each particle until it converges
    h = h0.clone()
    todo = torch.ones(n, dtype=torch.bool, device=x.device)
    rho, gh = torch.empty_like(h), torch.empty_like(h)
    for _ in range(30):
        for i, j, ok, dx, r2 in pairs.chunks():
            q = torch.sqrt(r2) / h[i][:, None]
            w, gw = _kernel(case, q)
            w, gw = torch.where(ok, w, 0.0), torch.where(ok, gw, 0.0)
            new = todo[i]
            rho[i] = torch.where(new, cn * pm * (w.sum(1) + w0) / h[i] ** 3, rho[i])
            gh[i] = torch.where(new, cn * pm * ((-q * gw - 3.0 * w).sum(1) - 3.0 * w0) / h[i] ** 4, gh[i])
        om = 1.0 + h / (3.0 * rhoh(h)) * gh
        hn = h + (rhoh(h) - rho) * h / (3.0 * rhoh(h)) / om
        hn = torch.minimum(torch.maximum(hn, 0.8 * h), 1.2 * h)
        todo = todo & ~((hn - h).abs() / h0 < 1e-4)
        if not bool(todo.any()):
            break
        h = torch.where(todo, hn, h)
    hsum = h
    gradh = (1.0 / om).float()
    h = hf * (pm / rho) ** (1.0 / 3.0)
    # primitive variables
    iso = case["gas"] == "isothermal"
    if hydro:
        P = rhoh(h) * (1.0 if iso else (GAMMA - 1.0) * u)
        cs = torch.ones_like(h) if iso else torch.sqrt(GAMMA * (GAMMA - 1.0) * u)
    # pair force (force.F90:1227-2056)
    f = torch.zeros((n, 4), dtype=torch.float64, device=x.device)
    divv = torch.empty_like(h)
    al, gd = d["alpha"][:, 0].double(), gradh.double()
    rh = rhoh(h)
    dtc = dtf = math.inf
    for i, j, ok, dx, r2 in pairs.chunks():
        r = torch.sqrt(r2)
        hi, hj = h[i][:, None], h[j]
        gi = torch.where(ok & (r < R * hi), _kernel(case, r / hi)[1], 0.0) * cn * gd[i][:, None] / hi ** 4
        gj = torch.where(ok & (r < R * hj), _kernel(case, r / hj)[1], 0.0) * cn * gd[j] / hj ** 4
        un = torch.where(ok[:, :, None], dx / r[:, :, None], 0.0)
        pv = ((v[i][:, None, :] - v[j]) * un).sum(dim=2)
        divv[i] = -pm * (pv * gi).sum(1) / rh[i]
        if not hydro:
            continue
        ci, cj, ri, rj = cs[i][:, None], cs[j], rh[i][:, None], rh[j]
        near = ok & ((r < R * hi) | (r < R * hj))
        vs = torch.where(near, torch.maximum(ci, cj) - 2.0 * pv, 0.0).amax(dim=1).clamp(min=0.0)
        app = pv < 0.0
        qi = torch.where(app, -0.5 / ri * (al[i][:, None] * ci - 2.0 * pv).clamp(min=0.0) * pv, 0.0)
        qj = torch.where(app, -0.5 / rj * (al[j] * cj - 2.0 * pv).clamp(min=0.0) * pv, 0.0)
        Pi, Pj = P[i][:, None], P[j]
        gp = pm * ((Pi / ri ** 2 + qi) * gi + (Pj / rj ** 2 + qj) * gj)
        f[i, :3] = -(un * gp[:, :, None]).sum(1)
        dti = 0.3 * h[i] / torch.maximum(vs, cs[i])
        dtc = min(dtc, float(dti.min()))
        if not iso:
            vu = torch.sqrt((Pi - Pj).abs() * 2.0 / (ri + rj))
            cond = vu * (u[i][:, None] - u[j]) * 0.5 * pm * (gi / ri + gj / rj)
            f4 = P[i] / rh[i] ** 2 * pm * (pv * gi).sum(1) + (pm * qi * pv * gi).sum(1) + cond.sum(1)
            low = u[i] + dti * f4 < 2.2e-16
            f[i, 3] = torch.where(low, f4 / (1.0 - dti * f4 / u[i]), f4)
        a = torch.sqrt((f[i, :3] ** 2).sum(1))
        dtf = min(dtf, float((0.25 * torch.sqrt(h[i] / a)).min()))
    # velocity gradients and d(div v)/dt of the density pass (exact linear)
    dvdx, dda = torch.empty((n, 9), dtype=torch.float64, device=x.device), torch.empty_like(h)
    for i, j, ok, dx, r2 in pairs.chunks():
        r = torch.sqrt(r2)
        gw = torch.where(ok, _kernel(case, r / hsum[i][:, None])[1], 0.0)
        un = torch.where(ok[:, :, None], dx * (gw / r)[:, :, None], 0.0)
        rr = -torch.einsum("pka,pkb->pab", dx, un)
        inv = torch.linalg.inv(rr)
        dv = torch.einsum("pka,pkb->pab", v[i][:, None, :] - v[j], un)
        G = -torch.einsum("pab,pbc->pac", dv, inv)
        dvdx[i] = G.reshape(-1, 9)
        if hydro:
            da = torch.einsum("pka,pkb->pab", f[i][:, None, :3] - f[j][:, :, :3], un)
            diva = -torch.einsum("pab,pba->p", da, inv)
            dda[i] = diva - torch.einsum("pab,pba->p", G, G)
    out = dict(xyzh=torch.cat([x, h[:, None]], 1), gradh=gradh[:, None], divcurlv=divv[:, None], dvdx=dvdx)
    if hydro:
        tr = (dvdx[:, 0] + dvdx[:, 4] + dvdx[:, 8])
        curl2 = (dvdx[:, 7] - dvdx[:, 5]) ** 2 + (dvdx[:, 2] - dvdx[:, 6]) ** 2 + (dvdx[:, 3] - dvdx[:, 1]) ** 2
        fac = (-tr).clamp(min=0.0) ** 2
        xil = torch.where(fac + curl2 > 2.2e-16, fac / (fac + curl2), 1.0)
        aloc = (10.0 * h * h * xil * (-dda).clamp(min=0.0) / cs ** 2).clamp(max=1.0)
        out["alphaind"] = torch.stack([al, aloc, dda], dim=1)
        out["eos_vars"] = torch.stack([P, cs, torch.zeros_like(P)], dim=1)
        out["fxyzu"] = f if not iso else f[:, :3]
        out["dt"] = min(dtc, dtf, 1e29)
    else:
        for k in ("alphaind", "eos_vars", "fxyzu", "divcurlB", "dBevol", "divBsymm", "dustfrac", "ddustevol",
                  "deltav", "tstop", "dt"):
            out[k] = None
    return out
