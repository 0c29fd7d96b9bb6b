"""Drop-in substeps as one fused kernel (timing off) against the separate
RHS and axpy kernels (timing on): bitwise equal for any order of calls, with
an RHS evaluation and whole steps in between, on every kernel family."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CALLS = [0, 1, 2, 3, 0, 1, "rhs", 2, 3, 0, 1, 1, 3, 3, 2, "steps", "none", 0, 2, "rhs", 1, 3]


def _run(pkg, prob, timing, members, **kw):
    with pkg.runtime.HipContext(prob, members=members, **kw) as ctx:
        rng = np.random.default_rng(3)
        for m in range(members):
            ctx.set_state(prob.H_init * (1.0 + 1e-3 * rng.standard_normal()), m)
        ctx.set_timing(timing)
        out = []
        for c in CALLS:
            if c == "rhs":
                out.append(ctx.eval_rhs(prob.H_init, members - 1))
            elif c == "steps":
                ctx.rk_steps(2)
                ctx.rk_substep(0)
            elif c == "none":
                ctx.rk_steps(0)
            else:
                ctx.rk_substep(c)
        return out + [ctx.get_state(m) for m in range(members)]


@pytest.mark.parametrize("members,kw", [
    (1, {}), (1, dict(exact=True)), (1, dict(kernel="quadw")), (1, dict(kernel="tile")),
    (1, dict(fp32=True)), (1, dict(fp32=True, exact=True)), (1, dict(fp32=True, kernel="quad")),
    (1, dict(fp32=True, kernel="tile")), (4, {}), (64, dict(member_block=64)),
    (32, dict(member_block=32, tiled=1, order="hilbert"))])
def test_fused_substeps_bitwise(pkg, members, kw):
    prob = pkg.host.Problem(pkg.mesh.case_path(642, seed=1), use_rcm=True, layout="cfdl", simd=4,
                            fp32=kw.get("fp32", False))
    print(f"case: fused substeps N=642 members={members} {kw}", flush=True)
    want = _run(pkg, prob, True, members, **kw)
    got = _run(pkg, prob, False, members, **kw)
    for a, b in zip(got, want):
        assert np.isfinite(b).all()
        assert np.array_equal(a, b)
