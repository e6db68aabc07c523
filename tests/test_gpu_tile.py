"""The density and force passes (tiles: one workgroup per tree node, candidates
in LDS) against the oracle at the sizes where their forms change: sets whose
nodes hold other than 64 particles, boxes too small for one periodic offset per
leaf (which lists search), groups with more candidates or longer lists than a
tile holds (the large form, and beyond it the list kernels), and active
fractions on both sides of one half.  test_paths asks for the path of each case
besides.
Neighbour and iteration counts are exact; h and each force component agree to
1e-12 of the rms (the parity tests' FP64 tolerance: sums of a few hundred FP64
terms in another order, a few 1e-16 each)."""
import numpy as np
import pytest

from phantom_amd import abi, setups, sph
from tests import parity

pytestmark = pytest.mark.gpu


def _noisy_star():
    return setups.relaxation_target(n=9000, seed=7)


def _active(frac):
    s = setups.uniform_box(nx=18, ny=16, nz=20, seed=3, isothermal=False,
                           box=(-0.45, 0.45, -0.4, 0.4, -0.5, 0.5))
    return setups.with_levels(s, [(0, 1.0 - frac), (2, frac)], nbinmax=2, istepfrac=1)


CASES = {
    "box_67_per_node_cubic": lambda: setups.uniform_box(nx=17, ny=18, nz=14, seed=3, isothermal=False,
                                                         box=(-0.425, 0.425, -0.45, 0.45, -0.35, 0.35)),
    "box_quintic": lambda: setups.uniform_box(nx=20, ny=19, nz=21, seed=4, kernel=abi.KERNEL_QUINTIC,
                                               box=(-0.5, 0.5, -0.475, 0.475, -0.525, 0.525)),
    "small_box_quintic": lambda: setups.uniform_box(nx=12, seed=5, kernel=abi.KERNEL_QUINTIC),
    "random_box_h_times_4": lambda: setups.random_box(n=7000, seed=12),
    "random_box_quintic": lambda: setups.random_box(n=5000, seed=13, kernel=abi.KERNEL_QUINTIC),
    "tube_interface": lambda: setups.shock_tube(ny=16),
    "noisy_star": _noisy_star,
    "mhd_dust_odd": lambda: setups.mhd_dust_box(nx=15, jitter=0.05, kernel=abi.KERNEL_CUBIC),
    "active_0.45": lambda: _active(0.45),
    "active_0.55": lambda: _active(0.55),
}


def check(setup, tol_dudt=1e-12):
    """The setup on the GPU against the oracle; how the GPU searched."""
    g = parity.run_gpu(setup)
    o = parity.run_oracle(setup)
    act = setup["iphase"] > 0 if setup.get("iphase") is not None else np.ones(len(setup["xyzh"]), bool)
    np.testing.assert_array_equal(g["nneigh"][act], o["dens"]["nneigh"][act])
    np.testing.assert_array_equal(g["nits"][act], o["dens"]["nits"][act])
    assert parity.rel_rms(g["xyzh"][:, 3], o["xyzh"][:, 3]) <= 1e-12
    for k in ("gradh", "dvdx"):
        # FP32 outputs: one unit in the last place of values up to the rms,
        # relative above it
        assert parity.rel_err(np.asarray(g["dens"][k])[act], np.asarray(o["dens"][k])[act]) <= 2.4e-7, k
    ncomp = 4 if setup["params"].maxvxyzu >= 4 else 3
    f, fo = g["force"]["fxyzu"][act], o["force"]["fxyzu"][act]
    rms = np.sqrt(np.mean((fo[:, :3] ** 2).sum(axis=1)))
    assert np.max(np.abs(f[:, :3] - fo[:, :3])) <= 1e-12 * rms
    if ncomp == 4:
        assert parity.rel_rms(f[:, 3], fo[:, 3]) <= tol_dudt
    if setup["params"].mhd:
        for c in range(4):
            assert parity.rel_rms(g["force"]["dBevol"][:, c], o["force"]["dBevol"][:, c]) <= 1e-12, c
        assert parity.rel_rms(g["force"]["ddustevol"], o["force"]["ddustevol"]) <= 1e-12
    if setup.get("bins") is not None:
        np.testing.assert_array_equal(g["force"]["ibin"], o["force"]["ibin"])
    st = g["ctx"].get_search_stats()
    g["ctx"].close()
    return st


@pytest.mark.parametrize("name", list(CASES))
def test_tiles_match_oracle(name, gpu):
    setup = CASES[name]()
    print(f"\n[case {name}] n={setup['xyzh'].shape[0]}", flush=True)
    check(setup)


@pytest.mark.parametrize("kernel", [abi.KERNEL_CUBIC, abi.KERNEL_QUINTIC])
def test_thin_box_keeps_its_lists(kernel, gpu):
    """A periodic box with 12 particles along z, too thin for any tile: the
    density pass makes lists of all particles, and the force pass uses them
    (no list of its own, none for particles run again)."""
    setup = setups.uniform_box(nx=40, ny=40, nz=12, seed=9, kernel=kernel, box=(-0.5, 0.5, -0.5, 0.5, -0.15, 0.15))
    g = parity.run_gpu(setup)
    kernels = [nm for nm, _ in g["ctx"].timings()]
    g["ctx"].close()
    assert "force" in kernels and not any(k.startswith("force_list") for k in kernels), kernels
    o = parity.run_oracle(setup)
    np.testing.assert_array_equal(g["nneigh"], o["dens"]["nneigh"])
    np.testing.assert_array_equal(g["nits"], o["dens"]["nits"])
    assert parity.rel_rms(g["xyzh"][:, 3], o["xyzh"][:, 3]) <= 1e-12
    for c in range(3):
        assert parity.rel_rms(g["force"]["fxyzu"][:, c], o["force"]["fxyzu"][:, c]) <= 1e-12, c


def _open_levels(frac, kernel, nx, ny, nz):
    s = setups.uniform_box(nx=nx, ny=ny, nz=nz, seed=3, kernel=kernel, isothermal=False,
                           box=(-0.025 * nx, 0.025 * nx, -0.025 * ny, 0.025 * ny, -0.025 * nz, 0.025 * nz))
    s["params"].periodic = 0
    return s if frac == 1.0 else setups.with_levels(s, [(0, 1.0 - frac), (2, frac)], nbinmax=2, istepfrac=1)


# 5760 particles: groups of up to 64; 4284: of up to 80
DISPATCH = [(0.45, abi.KERNEL_CUBIC, (18, 16, 20), False), (0.55, abi.KERNEL_CUBIC, (18, 16, 20), True),
            (0.55, abi.KERNEL_QUINTIC, (18, 16, 20), True), (0.55, abi.KERNEL_CUBIC, (17, 18, 14), False),
            (0.7, abi.KERNEL_CUBIC, (17, 18, 14), True), (0.8, abi.KERNEL_QUINTIC, (17, 18, 14), False),
            (0.95, abi.KERNEL_QUINTIC, (17, 18, 14), True), (1.0, abi.KERNEL_CUBIC, (17, 18, 14), True),
            (1.0, abi.KERNEL_QUINTIC, (17, 18, 14), True)]


@pytest.mark.parametrize("frac,kernel,n,tiles", DISPATCH)
def test_active_fraction_and_kernel_choose_the_search(frac, kernel, n, tiles, gpu):
    print(f"\n[case {frac} {kernel} {n}]", flush=True)
    st = check(_open_levels(frac, kernel, *n))
    assert (st["tiles"] > 0) == tiles, st


# lists of 128 groups (cubic) take 2 MB, those of groups in the large form, which
# have room for all here, 21 MiB; lists of all particles 16.9 MiB at 256 entries
@pytest.mark.parametrize("caps,tiles", [("dlist=16", True), ("budget_kib=18432", False), ("budget_kib=32768", True),
                                        ("lists=1", False)])
def test_budget_of_the_tiles_own_lists(caps, tiles, gpu, monkeypatch):
    """Tiles run while their own lists fit in the list budget, whatever the
    capacity of the list kernels' buffers."""
    monkeypatch.setenv("PHSPH_CAPS", caps)
    print(f"\n[case {caps}]", flush=True)
    st = check(_open_levels(1.0, abi.KERNEL_CUBIC, 18, 16, 20))
    assert (st["tiles"] > 0) == tiles, st


def test_outgrown_particles_count_once(gpu):
    """The search radius of the next call goes by how many particles outgrew
    their lists (more than 1/200: wider).  A group that is run again in the large
    form, for a list that is too long, meets its outgrown particles twice: 30 of
    8192 here, in groups with one such list each."""
    setup = setups.uniform_box(nx=32, ny=16, nz=16, seed=8, box=(-1.0, 1.0, -0.5, 0.5, -0.5, 0.5))
    p = setup["params"]
    p.tolh = 2e-3  # above 1e-3 the lists do not serve the force pass and the radius goes by this count alone
    n = setup["xyzh"].shape[0]
    cell = np.floor((setup["xyzh"][:, :3] - [-1.0, -0.5, -0.5]) * 16.0).astype(int)
    block, local = cell // 4, cell % 4  # nodes of 64 particles: 4 x 4 x 4 lattice cells
    some = (block[:, 0] * 16 + block[:, 1] * 4 + block[:, 2]) % 4 == 1
    ids = np.flatnonzero(some & (local == 1).all(axis=1))[:30]
    keep = {tuple(b) for b in block[ids]}
    big = [i for i in np.flatnonzero(some & (local == 2).all(axis=1)) if tuple(block[i]) in keep]
    assert len(ids) == len(big) == 30
    ctx = sph.Context(p)
    xyzh = setup["xyzh"].copy()
    for k in range(3):
        if k == 2:
            assert ctx.get_tuning()["search_radius"] == 1.03
            xyzh[ids, 3] *= 0.9
            xyzh[big, 3] *= 1.25
        ctx.maketree(xyzh)
        ctx.densityiterate(1, xyzh, setup["vxyzu"], alphaind=setup["alphaind"].copy())
    st, radius = ctx.get_search_stats(), ctx.get_tuning()["search_radius"]
    ctx.close()
    assert st["tiles"] == 128 and st["large"] == 30 and st["again"] >= 30, st
    assert 200 * 30 <= n < 2 * 200 * 30 and radius == 1.03


def _huge_h():
    """One particle reaches all others: its group has every leaf a candidate."""
    s = setups.uniform_box(nx=32, seed=6, isothermal=False)
    s["params"].periodic = 0
    s["xyzh"][5000, 3] = 0.6
    return s


# setup, PHSPH_CAPS and what get_search_stats must say: [tiles, large form,
# force by tiles], True: some, False: none, None: either
PATHS = {
    "tile4_cubic": (lambda: setups.uniform_box(nx=24, seed=3, isothermal=False), "", [True, False, True]),
    "tile4_quintic": (lambda: setups.uniform_box(nx=24, seed=3, kernel=abi.KERNEL_QUINTIC), "", [True, None, True]),
    "tile5_cubic": (lambda: setups.uniform_box(nx=20, seed=3), "", [True, False, True]),
    "tile5_quintic": (lambda: setups.uniform_box(nx=26, seed=3, kernel=abi.KERNEL_QUINTIC, isothermal=False), "",
                      [True, None, True]),
    "tile4_mhd_dust": (lambda: setups.mhd_dust_box(nx=24, jitter=0.05), "", [True, None, True]),
    "tile5_mhd_dust": (lambda: setups.mhd_dust_box(nx=26, jitter=0.05, kernel=abi.KERNEL_CUBIC), "",
                       [True, False, True]),
    "tile4_part_active": (lambda: setups.with_levels(setups.uniform_box(nx=24, seed=3, isothermal=False),
                                                     [(0, 0.4), (2, 0.6)], nbinmax=2, istepfrac=1), "",
                          [True, False, True]),
    "large_interface": (lambda: setups.shock_tube(ny=16), "", [True, True, True]),
    "large_noisy": (_noisy_star, "", [True, True, None]),
    "large_quintic": (lambda: setups.random_box(n=30000, seed=5, kernel=abi.KERNEL_QUINTIC, hmin_frac=0.9,
                                                hmax_frac=1.1), "", [True, True, None]),
    # room for one group in the large form: the others are handed back
    "no_room_large": (_noisy_star, "tlarge=1", [True, True, None]),
    # every walk's first stack too small, with tiles and with the groups run again
    "deep_walks": (_noisy_star, "wstack=8", [True, True, None]),
    "deep_walks_box": (lambda: setups.uniform_box(nx=20, seed=3), "wstack=2", [True, False, True]),
    # candidate lists of 4 leaves that grow, and the exact offsets that follow where
    # a uniform length does not fit: 512 tiles take 7.84 MB, 4096 leaves a group 8.4 MB
    "few_candidates": (lambda: setups.uniform_box(nx=24, seed=3), "gcand=4", [True, False, True]),
    "exact_candidates": (_huge_h, "gcand=4,tlarge=1,budget_kib=7900", [True, None, None]),
}


@pytest.mark.parametrize("name", list(PATHS))
def test_paths(name, gpu, monkeypatch):
    setup, caps, want = PATHS[name]
    if caps:
        monkeypatch.setenv("PHSPH_CAPS", caps)
    print(f"\n[case {name}]", flush=True)
    # particles of equal pressure and different u: the conductivity of du/dt goes
    # by the root of a pressure difference that is rounding (1e-16 of P) alone, so
    # the list kernels are 2.2e-12 from the oracle on the larger set too
    st = check(setup(), tol_dudt=1e-11 if "mhd" in name else 1e-12)
    for k, w in zip(("tiles", "large", "force_tiles"), want):
        assert w is None or (st[k] > 0) == w, st
    assert (st["deep"] > 0) == ("wstack" in caps), st
    if name == "no_room_large":
        assert st["large"] > 1


def test_handed_back_particles_have_every_list_attempt(gpu, monkeypatch):
    """Lists grow from one entry to the 2048 of the twelfth attempt: smoothing
    lengths 2.5 times too large give lists of about 1200, which no tile holds."""
    monkeypatch.setenv("PHSPH_CAPS", "dlist=1")
    s = _open_levels(1.0, abi.KERNEL_CUBIC, 18, 16, 20)
    s["xyzh"][:, 3] *= 2.5
    st = check(s)
    assert st["tiles"] > 0 and st["again"] > 0, st


# random positions and h, about 55 particles a group, at the widest search radius
# (that of a context's first call)
@pytest.mark.parametrize("kernel,n,tiles", [(abi.KERNEL_QUINTIC, 40000, True), (abi.KERNEL_QUINTIC, 80000, False),
                                            (abi.KERNEL_CUBIC, 40000, True), (abi.KERNEL_CUBIC, 80000, False)])
def test_uneven_sets_with_many_groups_go_by_lists(kernel, n, tiles, gpu):
    print(f"\n[case {kernel} {n}]", flush=True)
    st = check(setups.random_box(n=n, seed=21, kernel=kernel, hmin_frac=0.7, hmax_frac=1.3))
    assert (st["tiles"] > 0) == tiles, st


# after three calls, at the narrowest: the h of random positions differ by 1.45
# within a group, and h with a factor of two between neighbours by more
@pytest.mark.parametrize("n,factor,tiles", [(80000, 1.0, True), (160000, 1.0, True), (80000, 2.0, True),
                                            (160000, 2.0, False)])
def test_uneven_cubic_sets_at_the_narrow_radius(n, factor, tiles, gpu):
    print(f"\n[case {n} {factor}]", flush=True)
    s = setups.random_box(n=n, seed=22, hmin_frac=1.0, hmax_frac=1.0)
    ctx = sph.Context(s["params"])
    for k in range(4):
        if k == 3:
            assert ctx.get_tuning()["search_radius"] == 1.03
            s["xyzh"][::2, 3] *= factor  # above the converged h: none outgrows its list
        xyzh = s["xyzh"].copy()
        ctx.maketree(xyzh)
        ctx.densityiterate(1, xyzh, s["vxyzu"], alphaind=s["alphaind"].copy())
        if k < 3:
            s["xyzh"][:, 3] = xyzh[:, 3]
    st = ctx.get_search_stats()
    nneigh, nits = ctx.get_particle_stats(n)
    ctx.close()
    assert (st["tiles"] > 0) == tiles, st
    o = parity.run_oracle(s)
    np.testing.assert_array_equal(nneigh, o["dens"]["nneigh"])
    np.testing.assert_array_equal(nits, o["dens"]["nits"])
    assert parity.rel_rms(xyzh[:, 3], o["xyzh"][:, 3]) <= 1e-12
