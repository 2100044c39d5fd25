"""The second Gram-Schmidt pass of a single small instance (at most 64
reduction chunks: its updates sum the multi-dot partials themselves, and the
end of the step resumes after the pass while the next step, already enqueued,
skips itself).  With the pass on every column, on none and at the default
threshold the solves reach the same fixed point; and with the cycles launched
directly (kernel timing on), where every step is waited for and none is
enqueued ahead, they take the same iterates to the bit."""
import numpy as np
import pytest

import oracle_lib as O
from product_util import glhip

pytestmark = pytest.mark.gpu
G = glhip()


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", [(8, 8, 8), (3, 3, 4)], ids=["8x8x8", "3x3x4"])
def test_second_pass_of_a_small_instance(n, fp32):
    # 729 nodes (13 chunks) and 80 nodes (a chunk and a remainder)
    p, t, D = 20.0, 0.5, 20.0
    m = G.Mesh(1, n, (-20, -20, -D / 2), (20, 20, D / 2), [1, 1, 1, 1, 0, 0])
    ctx = G.Context(0)
    try:
        ctx.upload_mesh(m)
        ctx.set_materials(np.array([O.coef(p, t)]))
        U0 = O.initial_guess(m.n_nodes, O.matep(p, t)["gap_B"], amp=0.05, seed=60)
        out = {}
        for ratio in (0.01, 1.0, 0.0):
            ctx.set_reorth(ratio)
            for timing in (False, True):
                print("second pass", n, "fp32" if fp32 else "fp64", "ratio", ratio, "direct", timing, flush=True)
                ctx.set_timing(timing)
                ctx.set_solution(U0)
                st = ctx.newton_solve(rtol=1e-10, max_newton=60, lin_tol=1e-2, restart=40, fp32=fp32)
                print(st, flush=True)
                assert st["converged"] == 1.0
                assert st["r_final"] <= 1e-10 * st["r0"] * (1 + 1e-6)
                out[ratio, timing] = (st["gmres_its"], st["F"], ctx.solution())
            ctx.set_timing(False)
            a, b = out[ratio, False], out[ratio, True]
            assert a[0] == b[0] and a[1] == b[1] and np.array_equal(a[2], b[2])
        ref = out[0.01, False]
        for (ratio, _), (its, F, U) in out.items():
            assert abs(F - ref[1]) <= 1e-10 * abs(ref[1]), ratio
        assert abs(out[1.0, False][0] - ref[0]) <= 0.1 * ref[0] + 5
    finally:
        ctx.close()
