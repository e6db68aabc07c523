"""Sparse active sets, searched by one wavefront per particle: few and single
active particles, lists longer than the separations kept in LDS (256), leaf
batches that end anywhere, small periodic boxes, against the oracle with the
tolerances of test_gpu_tile."""
import pytest

from phantom_amd import abi, setups
from tests import test_gpu_tile

pytestmark = pytest.mark.gpu


def _sparse(frac, hfac=1.0, **kw):
    s = setups.uniform_box(seed=3, isothermal=False, **kw)
    s["xyzh"][:, 3] *= hfac
    return setups.with_levels(s, [(0, 1.0 - frac), (2, frac)], nbinmax=2, istepfrac=1)


CASES = {
    "one_in_64": lambda: _sparse(1.0 / 64.0, nx=18, ny=16, nz=20, box=(-0.45, 0.45, -0.4, 0.4, -0.5, 0.5)),
    "one_in_8_quintic": lambda: _sparse(0.125, nx=16, kernel=abi.KERNEL_QUINTIC),
    "long_lists": lambda: _sparse(0.1, hfac=1.9, nx=18),
    "few": lambda: _sparse(0.0007, nx=16),
    "small_box": lambda: _sparse(0.3, nx=10, kernel=abi.KERNEL_QUINTIC),
}


@pytest.mark.parametrize("name", list(CASES))
def test_sparse_sets_match_oracle(name, gpu, monkeypatch):
    monkeypatch.setitem(test_gpu_tile.CASES, name, CASES[name])
    test_gpu_tile.test_tiles_match_oracle(name, gpu)
