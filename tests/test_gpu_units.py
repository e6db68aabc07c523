"""Any unit of length: sets whose lengths are far outside what a 32-bit square
holds (1.2e-38 to 3.4e38) give the oracle's neighbour and iteration counts
exactly, and h, gradh and (after icall = 1) forces to the parity tolerances, as
the same set in lengths of order one does.  Where icall = 0 no second pass
could mend a short neighbour list."""
import numpy as np
import pytest

from phantom_amd import abi, setups
from tests import parity

pytestmark = pytest.mark.gpu


def scaled(setup, s):
    """The set with every length in units 1/s of the old one, at the same
    densities and velocities."""
    p = setup["params"]
    setup["xyzh"] = setup["xyzh"] * s
    for k in ("xmin", "xmax", "ymin", "ymax", "zmin", "zmax"):
        setattr(p, k, getattr(p, k) * s)
    p.massoftype_gas *= s ** 3
    return setup


def _box(s, periodic=1, kernel=abi.KERNEL_CUBIC):
    setup = setups.uniform_box(nx=18, ny=16, nz=20, seed=3, kernel=kernel, box=(-0.45, 0.45, -0.4, 0.4, -0.5, 0.5))
    setup["params"].periodic = periodic
    return scaled(setup, s)


def _random(s):
    setup = setups.random_box(n=5000, seed=12, hmin_frac=0.8, hmax_frac=1.2)
    setup["params"].periodic = 0
    return scaled(setup, s)


CASES = {"box_1": lambda: _box(1.0)}
# below about 1e-15 every node is as large as the whole set (the reference
# adds epsilon to its size), so that no periodic offset per group is safe
CASES.update({f"box_{s:g}": (lambda s=s: _box(s)) for s in (1e18, 8e19, 1e21, 1e25)})
CASES.update({f"open_{s:g}": (lambda s=s: _box(s, periodic=0)) for s in (1e20, 1e-17, 1e-20, 1e-22, 1e-25)})
CASES.update({f"open_quintic_{s:g}": (lambda s=s: _box(s, periodic=0, kernel=abi.KERNEL_QUINTIC))
              for s in (3e20, 1e-21)})
CASES.update({f"random_{s:g}": (lambda s=s: _random(s)) for s in (1e20, 1e-21)})


@pytest.mark.parametrize("icall", [1, 0])
@pytest.mark.parametrize("name", list(CASES))
def test_length_unit(name, icall, gpu):
    setup = CASES[name]()
    print(f"\n[case {name}] n={setup['xyzh'].shape[0]} icall {icall}", flush=True)
    g = parity.run_gpu(setup, icall=icall)
    o = parity.run_oracle(setup, icall=icall)
    g["ctx"].close()
    np.testing.assert_array_equal(g["nneigh"], o["dens"]["nneigh"])
    np.testing.assert_array_equal(g["nits"], o["dens"]["nits"])
    assert parity.rel_rms(g["xyzh"][:, 3], o["xyzh"][:, 3]) <= 1e-12
    assert parity.rel_err(np.asarray(g["dens"]["gradh"]), np.asarray(o["dens"]["gradh"])) <= 2.4e-7
    if icall == 0:  # the oracle's force search goes by the tree's h, not by the one stored
        return
    f, fo = g["force"]["fxyzu"][:, :3], o["force"]["fxyzu"][:, :3]
    rms = np.sqrt(np.mean((fo ** 2).sum(axis=1)))
    assert np.max(np.abs(f - fo)) <= 1e-12 * rms


# where the epsilon that the reference adds to a separation (dens.F90:664-670)
# is small beside it, of its size, and far above it
@pytest.mark.parametrize("name", ["open_1", "open_1e-06", "box_1e-12", "open_1e-13", "open_1e-15", "open_1e-20"])
def test_small_lengths_velocity_gradients(name, gpu):
    kind, s = name.split("_")
    setup = _box(float(s), periodic=int(kind == "box"))
    print(f"\n[case {name}] n={setup['xyzh'].shape[0]}", flush=True)
    g = parity.run_gpu(setup)
    o = parity.run_oracle(setup)
    g["ctx"].close()
    # FP32 outputs: one unit in the last place of values up to the rms, relative above it
    for k in ("dvdx", "divcurlv"):
        assert parity.rel_err(np.asarray(g["dens"][k]), np.asarray(o["dens"][k])) <= 2.4e-7, k
    assert parity.rel_err(g["alphaind"][:, 2], o["alphaind"][:, 2]) <= 2.4e-7
