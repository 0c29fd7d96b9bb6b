"""Resident kernels on meshes whose last tile is far shorter than the others
(fewer 16-node units, down to one node's worth), so that some of its waves own
no node: bitwise equal to the pair kernel."""
import numpy as np
import pytest

from test_gpu_units import _run, _sphere

pytestmark = pytest.mark.gpu


# nodes on 256 compute units: tiles of ceil(n / 256), last tile n mod that
@pytest.mark.parametrize("n", [4412, 9002, 12252, 15212])
def test_exact_short_last_tile(pkg, tmp_path, n):
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: exact, short last tile, N={n}", flush=True)
    want = _run(pkg, prob, [7], kernel="pair", exact=True)
    assert np.isfinite(want).all() and not np.array_equal(want, prob.H_init)
    assert np.array_equal(_run(pkg, prob, [7], exact=True), want)


@pytest.mark.parametrize("n", [9002, 12252, 52228, 65796, 76548])
def test_fast_short_last_tile(pkg, tmp_path, n):
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: fast mode, short last tile, N={n}", flush=True)
    want = _run(pkg, prob, [7], kernel="pair")
    assert np.isfinite(want).all() and not np.array_equal(want, prob.H_init)
    assert np.array_equal(_run(pkg, prob, [7]), want)
