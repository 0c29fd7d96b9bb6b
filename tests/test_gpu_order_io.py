"""State I/O of reordered single states on both sides of the sizes that the
host reorders itself (16 KB to 4096 nodes), in every host layout and both precisions:
round trip, and the device copy against a context in the host's node order."""
import numpy as np
import pytest

from test_gpu_state_io import _device_state, _problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("layout", ["cfdl", "sfdl", "default"])
@pytest.mark.parametrize("kib", [15, 16, 17, 63, 64, 65, 127, 128, 129])
def test_reordered_round_trip(pkg, tmp_path, kib, layout, fp32):
    n = kib * 1024 // (16 if fp32 else 32)
    prob = _problem(pkg, tmp_path, n, layout, fp32)
    print(f"case: reordered state of {kib} KiB, {layout} fp32={fp32}", flush=True)
    kind = np.float32 if fp32 else np.float64
    H = np.random.default_rng(n).standard_normal(4 * prob.patch_size).astype(kind)
    dev = {}
    for order in ("host", "hilbert"):
        with pkg.runtime.HipContext(prob, fp32=fp32, kernel="lane" if fp32 else "pair",
                                    order=order) as ctx:
            ctx.set_state(H)
            dev[order] = _device_state(pkg, ctx, (prob.patch_size, 4), kind)
            assert np.array_equal(ctx.get_state(), H)
    assert np.array_equal(dev["host"], H[prob.svm_index()])
    a, b = (v[np.lexsort(v.T)] for v in (dev["host"], dev["hilbert"]))
    assert np.array_equal(a, b) and not np.array_equal(dev["host"], dev["hilbert"])
