"""Which ensembles that name no member block run the matrix-core kernel (its
records, more than 1 KB per node, are in the context's bytes), on both sides of
each line of the rule on 256 compute units, and that the bits do not depend on it."""
import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,members,records", [
    (640, 2, True), (640, 64, False),            # 64 does not divide, or does; half a turn
    (1000, 192, True), (1000, 128, False),       # 48 and 32 items of 64 in the first turn
    (508, 256, False), (512, 320, True),         # two tiles per XCD
    (2560, 128, False), (3240, 128, True),       # 69 % and 81 % of two turns
    (4840, 64, False), (6760, 64, True)])        # 59 % and 84 %
def test_default_kernel_rule(pkg, tmp_path, n, members, records):
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: default ensemble N={n} members={members}", flush=True)
    rng = np.random.default_rng(n)
    some = sorted({0, members // 2, members - 1})
    H = {m: prob.H_init * (1.0 + 1e-3 * rng.standard_normal(prob.H_init.shape)) for m in some}
    size = prob.compute_size
    with pkg.runtime.HipContext(prob, kernel="pair") as one, \
            pkg.runtime.HipContext(prob, members=members) as ens:
        extra = ens.device_bytes() - 4 * 32 * size * members - 32 * size
        assert (extra > 1024 * size) == records
        for m in range(members):
            ens.set_state(H.get(m, H[0]), m)
        ens.rk_steps(3)
        for m in some:
            one.set_state(H[m])
            one.rk_steps(3)
            assert np.array_equal(ens.get_state(m), one.get_state()), m


@pytest.mark.parametrize("n,members,records", [
    (12252, 64, False), (16000, 32, False),      # full, but in three and two turns
    (16000, 64, True), (10244, 96, True),        # 98 % and 96 % of four
    (2560, 96, False), (10240, 64, False)])      # 52 % and 84 %
def test_tiled_kernel_rule(pkg, tmp_path, n, members, records):
    """Tiled contexts: the matrix-core kernel shows as item records without the
    member-lane tiles' node-major copies (1280 bytes per node)."""
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: tiled ensemble N={n} members={members}", flush=True)
    size = prob.compute_size
    with pkg.runtime.HipContext(prob, kernel="pair", order="hilbert") as one, \
            pkg.runtime.HipContext(prob, members=members, member_block=32, tiled=1,
                                   share=one) as ens:
        extra = ens.device_bytes() - 4 * 32 * size * members - 32 * size
        assert (1024 * size < extra < 1350 * size) == records, extra / size
        for m in range(members):
            ens.set_state(prob.H_init, m)
        ens.rk_steps(3)
        one.set_state(prob.H_init)
        one.rk_steps(3)
        assert np.array_equal(ens.get_state(members - 1), one.get_state())
