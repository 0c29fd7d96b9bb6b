"""Server batches that hold two kernels: which one a launch takes (the
member-lane tiles are built, and counted, by the first launch that wants them),
the bits of members that live through both, and the budget."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu


class _Bytes(C.Structure):
    _fields_ = [("records", C.c_longlong), ("tiles", C.c_longlong)]


def _batch(pkg, prob, slots, room=1 << 40):
    """A batch context as the server creates it."""
    rt = pkg.runtime
    L = rt.lib()
    L.swe_hip_batch_create.argtypes = [C.POINTER(rt.SweHipStatic), C.POINTER(rt.SweHipOptions),
                                       C.c_longlong, C.POINTER(C.c_void_p), C.POINTER(_Bytes)]
    L.swe_hip_batch_alone.argtypes = [C.c_void_p, C.c_int]
    s, keep = rt.static_from_problem(prob)
    o = rt.SweHipOptions(slots, 0, 0, 32, None, 0, 0, rt.ORDERS["hilbert"], 1, 0, 0, 0)
    h, b = C.c_void_p(), _Bytes()
    assert L.swe_hip_batch_create(C.byref(s), C.byref(o), room, C.byref(h), C.byref(b)) == 0
    ctx = object.__new__(rt.HipContext)
    ctx.prob, ctx.members, ctx.exact, ctx.fp32 = prob, slots, False, False
    ctx.n_state, ctx._share, ctx._h = 4 * prob.patch_size, None, h
    return ctx, b


@pytest.mark.parametrize("n,few", [(640, None), (2560, 48), (10244, 48)])
def test_launches_take_the_faster_kernel(pkg, tmp_path, n, few):
    """64 slots: k_stage_tspec when full (at N = 640 always), else the matrix cores."""
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: batch of 64 slots, N={n}", flush=True)
    size = prob.compute_size
    rng = np.random.default_rng(n)
    H = [prob.H_init * (1.0 + 1e-3 * rng.standard_normal(prob.H_init.shape)) for _ in range(64)]
    ctx, b = _batch(pkg, prob, 64)
    alone = pkg.runtime.lib().swe_hip_batch_alone
    with ctx, pkg.runtime.HipContext(prob, kernel="pair") as one:
        assert 1024 * size < b.records < 1350 * size and b.tiles == 2048 * size
        records = ctx.device_bytes()
        for m in range(64):
            ctx.set_state(H[m], m)
        done = 0
        for active, by_itself, tiles in ([(16, 1, True)] if few is None else
                                         [(few, 1, False), (64, 0, False), (64, 1, True),
                                          (few, 1, True), (64, 1, True), (64, 0, True)]):
            alone(ctx.handle, by_itself)
            ctx.set_active(active)
            ctx.rk_steps(3)
            done += 3
            extra = ctx.device_bytes() - records
            assert (0 < extra <= b.tiles) == tiles, (active, by_itself, extra)
        for m in (0, 15):   # advanced by every call
            one.set_state(H[m])
            one.rk_steps(done)
            assert np.array_equal(ctx.get_state(m), one.get_state()), m


def test_no_room_keeps_the_tiles_alone(pkg, tmp_path):
    prob = _sphere(pkg, tmp_path, 2560)
    print("case: batch without room for two kernels, N=2560", flush=True)
    size = prob.compute_size
    ctx, b = _batch(pkg, prob, 32, room=3000 * size)
    with ctx, pkg.runtime.HipContext(prob, members=32, member_block=32, tiled=1,
                                     order="hilbert") as tiled:
        assert (b.records, b.tiles) == (0, 0)
        assert ctx.device_bytes() == tiled.device_bytes()


@pytest.mark.parametrize("cap_batches", [1, 3, 1000])
def test_full_and_partial_batches_equal_solo(pkg, cap_batches):
    """64 members at once on one mesh (a full batch with nothing beside it), then
    few, then two meshes; in a budget of one batch, of three and of many."""
    m = pkg.mesh
    probs = [pkg.host.Problem(m.case_path(n, seed=1), use_rcm=True, layout="cfdl")
             for n in (642, 2562)]
    print(f"case: server with room for {cap_batches} batches", flush=True)
    rng = np.random.default_rng(cap_batches)
    size = probs[1].compute_size
    cap = cap_batches * size * (31 * 36 + 17 * 8 + 32 + 128 * 64 + 2048)
    reqs = []

    def add(mesh, members, steps, at):
        H = probs[mesh].H_init
        reqs.append(pkg.serve.Request(
            mesh=mesh, inits=[H * (1.0 + 1e-3 * rng.standard_normal(H.shape))
                              for _ in range(members)], nsteps=steps, tag=len(reqs),
            arrival_s=at))
    for mesh, members, steps in ((1, 64, 9), (1, 5, 7), (0, 64, 6), (0, 3, 5), (1, 40, 4)):
        add(mesh, members, steps, 0.0)
    with pkg.serve.Server(hbm_cap_bytes=cap, slots=64, member_block=32, chunk_steps=3,
                          tiled=True) as srv:
        for p in probs:
            srv.add_mesh(p)
        stats = [srv.run([r])["requests_done"] for r in reqs[:2]]   # one after the other
        stats = srv.run(reqs[2:])                                   # the rest at once
    assert stats["requests_done"] == len(reqs)
    assert stats["hbm_peak"] <= cap
    ctxs = [pkg.runtime.HipContext(p) for p in probs]
    for r in reqs:
        for k in {0, len(r.inits) // 2, len(r.inits) - 1}:
            ctx = ctxs[r.mesh]
            ctx.set_state(r.inits[k])
            ctx.rk_steps(r.nsteps)
            assert np.array_equal(ctx.get_state(), r.results[k]), (r.tag, k)
    for c in ctxs:
        c.close()
