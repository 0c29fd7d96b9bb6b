"""States with infinities, NaN, subnormal numbers and the largest finite ones
through the matrix-core and exact unit kernels: the values of the stage kernels,
and no member of an ensemble touched by another's.  Every case first checks that
the context did not fall back to the kernel it is compared with: its unit tables
or records are in its device bytes."""
import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu

# small meshes take one step (4 hops), so that not every node is reached
RESIDENT = dict(kernel="resident", order="hilbert")
KINDS = ("inf", "nan", "subnormal", "largest", "zero")


def _state(prob, kind, kind_rng, dtype):
    H = prob.H_init.astype(dtype).copy()
    some = kind_rng.choice(prob.n_nodes, 3, replace=False) * 4 + kind_rng.integers(0, 4, 3)
    tiny = np.finfo(dtype).smallest_subnormal
    if kind == "inf":
        H[some] = [np.inf, -np.inf, np.inf]
    elif kind == "nan":
        H[some] = np.nan
    elif kind == "subnormal":   # every product and most sums are subnormal
        H[:] = (kind_rng.integers(-2000, 2000, H.shape) * float(tiny)).astype(dtype)
    elif kind == "largest":
        H[some] = np.finfo(dtype).max
    else:
        H[:] = 0.0
        H[some] = -0.0
    return H


_last = {}


def _mesh(pkg, tmp_path, n, fp32):
    if (n, fp32) not in _last:   # the kinds of one mesh run in a row
        _last.clear()
        _last[n, fp32] = _sphere(pkg, tmp_path, n, fp32=fp32)
    return _last[n, fp32]


def _same(a, b):
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,kw,ref,table", [
    (1000, RESIDENT, "pair", 1024), (9002, {}, "pair", 1024), (49152, {}, "pair", 1024),
    (66004, {}, "pair", 1024), (300004, {}, "pair", 1024),
    (4412, dict(exact=True, **RESIDENT), "pair", 64),
    (9002, dict(fp32=True), "lane", 512), (66004, dict(fp32=True), "pair", 512),
    (300004, dict(fp32=True), "lane", 512)])
def test_single_states(pkg, tmp_path, n, kw, ref, table, kind):
    fp32 = kw.get("fp32", False)
    dtype = np.float32 if fp32 else np.float64
    prob = _mesh(pkg, tmp_path, n, fp32)
    print(f"case: {kind} states, N={n} {kw} against {ref}", flush=True)
    H = _state(prob, kind, np.random.default_rng(n), dtype)
    out = []
    steps = 1 if "kernel" in kw else 4
    with pkg.runtime.HipContext(prob, **{**kw, "kernel": ref}) as one, \
            pkg.runtime.HipContext(prob, **kw) as auto:
        assert auto.device_bytes() - one.device_bytes() >= table * n, "fell back"
        for ctx in (one, auto):
            ctx.set_state(H)
            ctx.rk_steps(steps)
            out.append(ctx.get_state())
    assert _same(*out)
    if kind in ("inf", "nan"):
        assert not np.isfinite(out[0]).all() and np.isfinite(out[0]).any()
    if kind == "subnormal":
        assert (out[0] != 0).any() and not np.array_equal(out[0], H)


@pytest.mark.parametrize("n,members", [(2562, 2), (2562, 10), (40962, 2), (40962, 8),
                                       (40962, 24), (81000, 4)])
def test_ensemble_members_stay_apart(pkg, tmp_path, n, members):
    """Every member a kind of its own, the others ordinary; N = 40962 and 81000 reach
    the whole-tile rounds of both item shapes (64 tiles per XCD and more)."""
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: special members, N={n} members={members}", flush=True)
    rng = np.random.default_rng(n + members)
    H = [_state(prob, KINDS[m % 5], rng, np.float64) if m % 2 else
         prob.H_init * (1.0 + 1e-3 * rng.standard_normal(prob.H_init.shape))
         for m in range(members)]
    active = members - members // 4
    size = prob.compute_size
    with pkg.runtime.HipContext(prob, kernel="pair") as one, \
            pkg.runtime.HipContext(prob, members=members) as ens:
        assert ens.device_bytes() - 128 * size * members >= 1024 * size, "fell back"
        for call, act in ((2, members), (1, active)):
            for m in range(members):
                ens.set_state(H[m], m)
            ens.set_active(act)
            ens.rk_steps(call)
            for m in range(act):
                one.set_state(H[m])
                one.rk_steps(call)
                assert _same(ens.get_state(m), one.get_state()), (call, m)
        assert _same(ens.eval_rhs(H[1], 1), one.eval_rhs(H[1]))
