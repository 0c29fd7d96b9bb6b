"""Contexts that share a mesh share the unit records of the form they run: a
further context takes the device memory of its own state only, every context
computes the same bits, and the records live exactly as long as a context that
uses them, whichever is destroyed first."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu


def _free(pkg):
    """Free device memory, through the HIP runtime the library itself uses."""
    free, total = C.c_size_t(), C.c_size_t()
    info = pkg.runtime.lib().hipMemGetInfo
    info.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    assert info(C.byref(free), C.byref(total)) == 0
    return free.value


def _steps(ctx, H, members, k=6):
    ctx.set_state(H, members - 1)
    ctx.rk_steps(k)
    return ctx.get_state(members - 1)


@pytest.mark.parametrize("n,members,kw", [
    (100004, 1, {}), (500004, 1, {}), (100004, 1, dict(fp32=True, kernel="auto")),
    (100004, 2, {}), (50004, 16, {}), (10004, 1, dict(exact=True))])
def test_records_are_shared(pkg, tmp_path, n, members, kw):
    prob = _sphere(pkg, tmp_path, n, fp32=kw.get("fp32", False))
    print(f"case: shared records N={n} members={members} {kw}", flush=True)
    H = prob.H_init
    kind = 4 if kw.get("fp32") else 8
    owner = "lane" if kw.get("fp32") else "pair"
    with pkg.runtime.HipContext(prob, kernel=owner, fp32=kw.get("fp32", False),
                                exact=kw.get("exact", False)) as base:
        want = _steps(base, H, 1)
        if kw.get("fp32"):   # AUTO sums as PAIR at this size
            with pkg.runtime.HipContext(prob, share=base, kernel="pair", fp32=True) as ref:
                want = _steps(ref, H, 1)
        # the runtime's own first-use allocations (cooperative queue) come first
        with pkg.runtime.HipContext(prob, members=members, share=base, **kw) as ctx:
            assert np.array_equal(_steps(ctx, H, members), want)
        start = _free(pkg)
        one = pkg.runtime.HipContext(prob, members=members, share=base, **kw)
        first = start - _free(pkg)
        two = pkg.runtime.HipContext(prob, members=members, share=base, **kw)
        second = start - first - _free(pkg)
        # H, two K, D and the staging state; D of streamed units in memory;
        # allocations are rounded up to 2 MiB
        state = (16 * members + 4 + 8) * kind * n + (10 << 20)
        assert second <= state, (first, second)
        if n > 20000:
            assert first >= 1024 * n * kind // 8
        assert two.device_bytes() == one.device_bytes()
        assert np.array_equal(_steps(one, H, members), want)
        one.close()
        assert np.array_equal(_steps(two, H, members), want)
        with pkg.runtime.HipContext(prob, members=members, share=base, **kw) as three:
            two.close()
            assert np.array_equal(_steps(three, H, members), want)
        assert _free(pkg) >= start - (12 << 20)   # the records are gone with their last user
        with pkg.runtime.HipContext(prob, members=members, share=base, **kw) as again:
            assert np.array_equal(_steps(again, H, members), want)


def test_forms_do_not_mix(pkg, tmp_path):
    """Single states, ensembles of items of 8 and of 16 members and the exact form
    on one mesh at once."""
    prob = _sphere(pkg, tmp_path, 9002)
    print("case: four forms of records on one mesh, N=9002", flush=True)
    H = prob.H_init
    with pkg.runtime.HipContext(prob, kernel="pair") as base, \
            pkg.runtime.HipContext(prob, share=base, kernel="pair", exact=True) as ref:
        want = {False: _steps(base, H, 1), True: _steps(ref, H, 1)}
        ctxs = [(pkg.runtime.HipContext(prob, members=m, exact=e, share=base), m, e)
                for m, e in ((1, False), (1, True), (2, False), (10, False), (1, False))]
        for ctx, m, e in ctxs + ctxs[::-1]:
            assert np.array_equal(_steps(ctx, H, m), want[e]), (m, e)
        for ctx, m, e in ctxs[:3]:
            ctx.close()
        for ctx, m, e in ctxs[3:]:
            assert np.array_equal(_steps(ctx, H, m), want[e]), (m, e)
            ctx.close()
