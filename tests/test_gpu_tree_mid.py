"""Nodes split by one workgroup (more than 1024 and at most 16384 particles):
sizes at both ends of the range and one past them, unequal children, particles
on the split plane (sequential sums inside the workgroup) and coincident ones
(halved in place), against the oracle's sequential build."""
import numpy as np
import pytest

from oracle import oracle
from phantom_amd import setups, sph
from tests import parity

pytestmark = pytest.mark.gpu


def _random(n):
    return setups.random_box(n=n, seed=n)


def _clumped(n):
    s = setups.random_box(n=n, seed=3)
    r = s["xyzh"]
    r[: n // 3, :3] = 0.2 + 0.02 * r[: n // 3, :3]
    s["params"].maxp = 16 * n  # levels that ids number (the build refuses deeper trees)
    return s


def _coincident(n):
    s = setups.random_box(n=n, seed=4)
    s["xyzh"][: n // 2, :3] = s["xyzh"][0, :3]
    s["params"].maxp = 16 * n
    return s


CASES = {f"random_{n}": (lambda n=n: _random(n)) for n in (1024, 1025, 2051, 16384, 16385, 33333)}
CASES["clumped_16000"] = lambda: _clumped(16000)
CASES["coincident_3000"] = lambda: _coincident(3000)
CASES["lattice_24"] = lambda: setups.uniform_box(nx=24, seed=1, jitter=0.0)


@pytest.mark.parametrize("name", list(CASES))
def test_mid_nodes(name, gpu):
    setup = CASES[name]()
    p = setup["params"]
    print(f"\n[case {name}] n={setup['xyzh'].shape[0]}", flush=True)
    ctx = sph.Context(p)
    leaf, ncells = ctx.maketree(setup["xyzh"].copy())
    gt = ctx.get_tree()
    ctx.close()
    o = oracle.Oracle(p)
    o.maketree(setup["xyzh"].copy())
    ot = o.get_tree()
    assert ncells == ot["ncells"]
    np.testing.assert_array_equal(leaf, ot["leaf_is_active"])
    used = parity.reachable_nodes(ot)
    np.testing.assert_array_equal(gt["inoderange"][used], ot["inoderange"][used])
    np.testing.assert_array_equal(gt["inodeparts"], ot["inodeparts"])
    for f in ("leftchild", "rightchild", "parent", "hmax"):
        np.testing.assert_array_equal(gt["node"][f][used], ot["node"][f][used])
    # |S_seq - S| <= 2 gamma_{n-1} sum|a_i|, as in test_gpu_tree_large
    u = 2.0 ** -53
    nn = (ot["inoderange"][used, 1] - ot["inoderange"][used, 0] + 1).astype(np.float64)
    xmax = np.max(np.abs(setup["xyzh"][:, :3]))
    tol = 2.0 * nn * u / (1.0 - nn * u) * xmax + 4 * u * xmax
    dx = np.max(np.abs(gt["node"]["xcen"][used] - ot["node"]["xcen"][used]), axis=1)
    assert np.all(dx <= tol), np.max(dx / tol)
    ds = np.abs(gt["node"]["size"][used] - ot["node"]["size"][used])
    assert np.all(ds <= 2 * tol + 1e-15), np.max(ds / (2 * tol + 1e-15))
