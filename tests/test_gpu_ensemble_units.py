"""The matrix-core ensemble kernel (fast mode, the caller naming no member
block, or LDS tiles): every member's bits are those of its single-state run,
for member counts on both sides of an item's 8 or 16, a ragged last tile, idle
slots, evaluations and substeps; a mesh whose tiles do not fit falls back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _states(prob, members, seed):
    rng = np.random.default_rng(seed)
    return [prob.H_init * (1.0 + 1e-3 * rng.standard_normal(prob.H_init.shape))
            for _ in range(members)]


@pytest.mark.parametrize("n,members,kw", [
    (642, 2, {}), (642, 6, {}), (642, 8, {}), (2562, 10, {}), (642, 16, {}), (2562, 24, {}),
    (10242, 4, dict(order="hilbert")), (10242, 40, dict(order="morton", slot_block=16)),
    (2562, 96, dict(member_block=32, tiled=1, order="hilbert")),
    (10242, 96, dict(member_block=32, tiled=1, order="hilbert"))])
def test_members_equal_single_runs(pkg, n, members, kw):
    prob = pkg.host.Problem(pkg.mesh.case_path(n, seed=1), use_rcm=True, layout="cfdl")
    print(f"case: ensemble units N={n} members={members} {kw}", flush=True)
    H = _states(prob, members, n + members)
    some = sorted({0, 1, members // 2, members - 1})
    active = members - members // 4
    with pkg.runtime.HipContext(prob, kernel="pair") as one, \
            pkg.runtime.HipContext(prob, members=members, **kw) as ens:
        for m in range(members):
            ens.set_state(H[m], m)
        ens.rk_steps(3)
        for s in range(4):
            ens.rk_substep(s)
        for m in some:
            one.set_state(H[m])
            one.rk_steps(4)
            assert np.array_equal(ens.get_state(m), one.get_state()), m
        assert np.array_equal(ens.eval_rhs(H[0], members - 1), one.eval_rhs(H[0]))
        for m in range(members):
            ens.set_state(H[m], m)
        ens.set_active(active)
        ens.rk_steps(2)
        for m in [m for m in some if m < active]:
            one.set_state(H[m])
            one.rk_steps(2)
            assert np.array_equal(ens.get_state(m), one.get_state()), m


def test_scattered_stencils_fall_back(pkg, tmp_path):
    """Stencils of random nodes: a tile's rows exceed the LDS."""
    m = pkg.mesh
    case = m.read_bin(m.case_path(2562, seed=1))
    rng = np.random.default_rng(2)
    case.idx = rng.integers(0, 2562, case.idx.shape).astype(np.int32)
    case.idx[:, 0] = np.arange(2562)
    for nm in ("Dx", "Dy", "Dz", "L"):
        setattr(case, nm, rng.standard_normal(case.idx.shape) * 1e-3)
    path = str(tmp_path / "scattered.bin")
    m.write_bin(path, case)
    prob = pkg.host.Problem(path, use_rcm=False, layout="cfdl")
    print("case: ensemble on scattered stencils, N=2562", flush=True)
    H = _states(prob, 4, 1)
    with pkg.runtime.HipContext(prob, kernel="pair") as one, \
            pkg.runtime.HipContext(prob, members=4) as ens:
        for k in range(4):
            ens.set_state(H[k], k)
        ens.rk_steps(2)
        one.set_state(H[3])
        one.rk_steps(2)
        assert np.array_equal(ens.get_state(3), one.get_state())


@pytest.mark.parametrize("members", [4, 16])
def test_tiles_with_too_many_rows_are_cut(pkg, tmp_path, members):
    """Three random neighbours per node in a part of the mesh: its tiles exceed
    an item's rows, their halves do not, and the kernel still runs (its records
    are in the context's bytes)."""
    m = pkg.mesh
    case = m.read_bin(m.case_path(2562, seed=1))
    rng = np.random.default_rng(3)
    some = np.flatnonzero(case.X[:, 2] > 0.8)
    case.idx[some, 28:] = rng.integers(0, 2562, (len(some), 3))
    path = str(tmp_path / "cut.bin")
    m.write_bin(path, case)
    prob = pkg.host.Problem(path, use_rcm=False, layout="cfdl")
    print(f"case: ensemble with cut tiles, N=2562 members={members}", flush=True)
    H = _states(prob, members, 1)
    with pkg.runtime.HipContext(prob, kernel="pair") as one, \
            pkg.runtime.HipContext(prob, members=members) as ens:
        n = prob.compute_size
        assert ens.device_bytes() > 4 * 32 * n * members + 1024 * n
        for k in range(members):
            ens.set_state(H[k], k)
        ens.rk_steps(2)
        for k in (0, members - 1):
            one.set_state(H[k])
            one.rk_steps(2)
            assert np.array_equal(ens.get_state(k), one.get_state()), k


def test_untiled_server_batches_hold_what_admission_counts(pkg):
    """member_block 0 in a server: no records beside the static data and the
    slots' states, which is all that admission counts for an untiled batch."""
    prob = pkg.host.Problem(pkg.mesh.case_path(642, seed=1), use_rcm=True, layout="cfdl")
    print("case: server with member_block 0, N=642", flush=True)
    peak = {}
    for mb in (0, 4):
        req = pkg.serve.Request(mesh=0, inits=_states(prob, 3, 1), nsteps=2, tag=0, arrival_s=0.0)
        with pkg.serve.Server(slots=4, member_block=mb) as srv:
            srv.add_mesh(prob)
            peak[mb] = srv.run([req])["hbm_peak"]
    assert peak[0] == peak[4]
