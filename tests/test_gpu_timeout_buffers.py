"""A read-back after a resident launch whose wait timed out reports the error
and leaves the caller's buffer alone, on every read-back path.  The time-out is
forced from the host with a limit of one poll on the kernel's own bounded
wait (every wave still exits)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,kw", [
    (10242, dict(kernel="resident", order="hilbert")),   # reordered into the pinned ring
    (10242, dict(fp32=True)),
    (70001, dict()),                                     # plain copy, several ring slots
    (70001, dict(order="hilbert"))])                     # reordered on the device, then the ring
def test_buffer_survives_a_time_out(pkg, tmp_path, monkeypatch, n, kw):
    fp32 = kw.get("fp32", False)
    prob = _sphere(pkg, tmp_path, n, fp32=fp32)
    print(f"case: read-back after a forced time-out, N={n} {kw}", flush=True)
    lib = pkg.runtime.lib()
    get = lib.swe_hip_get_state32 if fp32 else lib.swe_hip_get_state
    buf = np.full(4 * prob.patch_size, -7.25, np.float32 if fp32 else np.float64)
    ptr = buf.ctypes.data_as(C.POINTER(C.c_float if fp32 else C.c_double))
    monkeypatch.setenv("SWE_HIP_RESIDENT_SPIN_LIMIT", "1")
    errors = 0
    with pkg.runtime.HipContext(prob, **kw) as ctx:
        for _ in range(20):   # a time-out is likely in every launch, certain in some
            ctx.set_state(prob.H_init)
            ctx.rk_steps(30)
            rc = get(ctx.handle, 0, ptr)
            if rc:
                assert rc == -3 and (buf == -7.25).all()
                errors += 1
            else:
                buf[:] = -7.25
        assert errors > 0
