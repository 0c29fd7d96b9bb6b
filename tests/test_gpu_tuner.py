"""swe_hip_tune_ex over ensembles: the candidates that run the matrix-core kernel
whatever tile shape they name are timed as one, the library's own choice."""
import numpy as np
import pytest

from test_gpu_units import _sphere

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,members", [(10244, 96), (16000, 64)])
def test_one_candidate_runs_the_matrix_core_kernel(pkg, tmp_path, n, members):
    prob = _sphere(pkg, tmp_path, n)
    print(f"case: tuner, tiled shapes that share a kernel, N={n} members={members}", flush=True)
    with pkg.runtime.HipContext(prob, kernel="pair", order="hilbert") as base:
        for _ in range(5):
            opts, ms = base.tune(members, steps=5)
            assert ms > 0 and not opts["tiled"], opts
        with pkg.runtime.HipContext(prob, share=base, **opts) as ctx:
            ctx.set_state(prob.H_init, members - 1)
            ctx.rk_steps(2)
            got = ctx.get_state(members - 1)
        base.set_state(prob.H_init)
        base.rk_steps(2)
        assert np.array_equal(got, base.get_state())
