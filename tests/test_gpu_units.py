"""The matrix-core resident kernels (k_steps_units, k_steps_units32), which AUTO
contexts run in fast mode, against the stage kernels: bitwise equal, because
the FP64 and FP32 matrix instructions round every product-sum like the
fused multiply-add they replace and the sums keep their order.  Sizes on both
sides of every change of plan: one, two and four 4-node groups per wave, one
and two resident units per wave, the first mesh whose units stream their weights
(LDS tables, then tables in memory, then records past the last-level cache), a last tile with a ragged unit, padded
nodes outside every stencil."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sphere(pkg, tmp_path, n, fp32=False):
    """A Fibonacci sphere with nearest-neighbour stencils and small random
    weights (the values only have to keep a few steps finite)."""
    rng = np.random.default_rng(n)
    i = np.arange(n) + 0.5
    z = 1.0 - 2.0 * i / n
    lon = i * (np.pi * (3.0 - np.sqrt(5.0)))
    r = np.sqrt(1.0 - z * z)
    X = np.stack([r * np.cos(lon), r * np.sin(lon), z], 1)
    m = pkg.mesh
    idx = m.stencils(X, 31)
    W = rng.standard_normal((4, n, 31)) * np.array([2.0, 2.0, 2.0, 5.0]).reshape(4, 1, 1)
    p_u, p_v, p_w = m.projection_rows(X)
    H = rng.standard_normal((n, 4)) * [10.0, 10.0, 10.0, 100.0]
    case = m.SweCase(n_nodes=n, nnbr=31, a=m.A_EARTH, gh0=5.0e4, dt=20.0, gamma=-1e-5, X=X,
                     f=2.0 * m.OMEGA * X[:, 2], ghm=rng.random(n) * 1e3, p_u=p_u, p_v=p_v, p_w=p_w,
                     gradghm=rng.standard_normal((n, 3)) * 1e-3, Dx=W[0], Dy=W[1], Dz=W[2],
                     L=W[3], idx=idx, H_init=H, H_final=H)
    path = str(tmp_path / "sphere.bin")
    m.write_bin(path, case)
    return pkg.host.Problem(path, use_rcm=True, layout="cfdl", simd=4, fp32=fp32)


def _run(pkg, prob, calls, **kw):
    with pkg.runtime.HipContext(prob, **kw) as ctx:
        ctx.set_state(prob.H_init)
        for k in calls:
            ctx.rk_steps(k)
        return ctx.get_state()


@pytest.mark.parametrize("n,order", [(1000, "host"), (4100, "morton"), (8192, "host"),
                                     (8193, "host"), (32769, "host"), (49152, "hilbert"),
                                     (49153, "host"), (65536, "hilbert"), (65537, "host"),
                                     (120001, "morton"), (300001, "host")])
def test_fp64_auto_bitwise_vs_pair(pkg, tmp_path, n, order):
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: FP64 units N={n} order={order}, calls of 5, 1 and 4 steps", flush=True)
    want = _run(pkg, prob, [10], kernel="pair")
    got = _run(pkg, prob, [5, 1, 4], order=order, slot_block=16 if order == "morton" else 0)
    assert np.isfinite(want).all() and not np.array_equal(want, prob.H_init)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n,kernel", [(1000, "lane"), (32769, "lane"), (65536, "lane"),
                                      (65537, "pair"), (120001, "pair"), (262144, "pair"),
                                      (300001, "lane"), (400001, "lane"), (620001, "lane")])
def test_fp32_auto_bitwise_vs_stage_kernel(pkg, tmp_path, n, kernel):
    """AUTO keeps the partial sums of the stage kernel it ran at that size:
    two per stencil sum (PAIR) from 65536 to 262144 nodes, else one (LANE)."""
    prob = _sphere(pkg, tmp_path, n, fp32=True)
    print(f"case: FP32 units N={n} against {kernel}, calls of 5 and 4 steps", flush=True)
    want = _run(pkg, prob, [9], fp32=True, kernel=kernel)
    got = _run(pkg, prob, [5, 4], fp32=True)
    assert np.isfinite(want).all() and not np.array_equal(want, prob.H_init.astype(np.float32))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n,order", [(1000, "host"), (4097, "morton"), (16384, "host"),
                                     (16385, "host")])
def test_exact_auto_bitwise_vs_pair(pkg, tmp_path, n, order):
    """k_steps_exact up to 64 nodes per compute unit, k_steps_resident above."""
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: exact N={n} order={order}, calls of 5, 1 and 4 steps", flush=True)
    want = _run(pkg, prob, [10], kernel="pair", exact=True)
    got = _run(pkg, prob, [5, 1, 4], exact=True, order=order,
               slot_block=16 if order == "morton" else 0)
    assert np.isfinite(want).all() and not np.array_equal(want, prob.H_init)
    assert np.array_equal(got, want)


def test_auto_calls_of_one_step_above_the_register_size(pkg, tmp_path):
    """Above 256 nodes per compute unit every call length runs the same sums."""
    prob = _sphere(pkg, tmp_path, 70001, fp32=True)
    print("case: FP32 units N=70001, calls of 1, 2 and 3 steps", flush=True)
    assert np.array_equal(_run(pkg, prob, [1, 2, 3], fp32=True), _run(pkg, prob, [6], fp32=True))


@pytest.mark.parametrize("members", [1, 16])
def test_tuner_choice_runs_the_same_bits(pkg, tmp_path, members):
    """Above RESIDENT's sizes the tuner times the streaming form too, and for
    ensembles the matrix-core kernel whatever divides the member count."""
    prob = _sphere(pkg, tmp_path, 70001 if members == 1 else 3000)
    print(f"case: tuner, {members} member(s), {prob.n_nodes} nodes", flush=True)
    with pkg.runtime.HipContext(prob, kernel="pair", order="hilbert") as base:
        opts, ms = base.tune(members, steps=3)
        assert ms > 0 and (opts["kernel"] in ("auto", "pair", "tile"))
        with pkg.runtime.HipContext(prob, share=base, **opts) as ctx:
            ctx.set_state(prob.H_init, members - 1)
            ctx.rk_steps(4)
            got = ctx.get_state(members - 1)
        base.set_state(prob.H_init)
        base.rk_steps(4)
        assert np.array_equal(got, base.get_state())
