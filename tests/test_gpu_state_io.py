"""State upload and read-back: whole states below, at and beyond the slots of
the pinned ring, through the reordering kernels and as plain copies, in every
host layout, precision and for ensembles.  The device copy is checked too
([node][var][member] in the device node order)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(pkg, tmp_path, n, layout, fp32):
    """n nodes on a spiral whose stencils are the next 31 nodes."""
    m = pkg.mesh
    i = np.arange(n) + 0.5
    z = 1.0 - 2.0 * i / n
    lon = i * (np.pi * (3.0 - np.sqrt(5.0)))
    r = np.sqrt(1.0 - z * z)
    X = np.stack([r * np.cos(lon), r * np.sin(lon), z], 1)
    idx = ((np.arange(n)[:, None] + np.arange(31)) % n).astype(np.int32)
    W = np.zeros((n, 31))
    p_u, p_v, p_w = m.projection_rows(X)
    H = np.arange(4.0 * n).reshape(n, 4)
    case = m.SweCase(n_nodes=n, nnbr=31, a=m.A_EARTH, gh0=1.0, dt=1.0, gamma=1.0, X=X, f=z, ghm=z,
                     p_u=p_u, p_v=p_v, p_w=p_w, gradghm=p_u, Dx=W, Dy=W, Dz=W, L=W, idx=idx,
                     H_init=H, H_final=H)
    path = str(tmp_path / "spiral.bin")
    m.write_bin(path, case)
    return pkg.host.Problem(path, use_rcm=False, layout=layout, simd=4, fp32=fp32)


def _device_state(pkg, ctx, shape, kind):
    """Copy of the context's device state through the HIP runtime the library
    itself uses."""
    out = np.empty(shape, kind)
    copy = pkg.runtime.lib().hipMemcpy
    copy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    assert copy(out.ctypes.data, ctx.state_device_ptr(), out.nbytes, 2) == 0
    return out


@pytest.mark.parametrize("n,layout,fp32,members,order", [
    (642, "cfdl", False, 1, "host"), (642, "sfdl", False, 1, "hilbert"),
    (642, "default", True, 1, "host"), (642, "cfdl_sfdl", True, 1, "morton"),
    (642, "sfdl", False, 4, "host"), (16384, "cfdl", False, 1, "host"),
    (16388, "cfdl", False, 1, "host"), (65536, "cfdl", False, 1, "hilbert"),
    (65540, "cfdl", False, 1, "hilbert"), (65540, "default", False, 2, "host"),
    (131076, "cfdl", True, 1, "hilbert"), (100004, "cfdl", False, 1, "host"),
    (150004, "sfdl", False, 1, "morton")])
def test_state_round_trip(pkg, tmp_path, n, layout, fp32, members, order):
    prob = _problem(pkg, tmp_path, n, layout, fp32)
    print(f"case: state I/O N={n} {layout} fp32={fp32} members={members} {order}", flush=True)
    rng = np.random.default_rng(n)
    kind = np.float32 if fp32 else np.float64
    kernel = "lane" if fp32 else ("pair" if members == 1 else "auto")
    H = [rng.standard_normal(4 * prob.patch_size).astype(kind) for _ in range(members)]
    with pkg.runtime.HipContext(prob, members=members, fp32=fp32, kernel=kernel,
                                order=order) as ctx:
        for m in range(members):
            ctx.set_state(H[m], m)
        dev = _device_state(pkg, ctx, (prob.patch_size, 4, members), kind)
        back = [ctx.get_state(m) for m in range(members)]
    for m in range(members):
        assert np.array_equal(back[m], H[m])
        want = H[m][prob.svm_index()]
        got = dev[:, :, m]
        if order != "host":   # another node order: the same rows
            want, got = (a[np.lexsort(a.T)] for a in (want, got))
        assert np.array_equal(got, want)
