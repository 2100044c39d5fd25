"""Products with the assembled Jacobian from its upper triangle against the
whole matrix read back: both sides of the block count at which they start
(4096), rows of one to 125 blocks (steps of 3, columns held 63 at a time),
a condensed adaptive matrix, and a batch.  FP64 sums of at most 125 x 18
terms: 1e-13 of the largest row; the FP32 matrix's sums are FP64, rounded once
to FP32: 1e-6."""
import numpy as np
import pytest

from product_util import adaptive_forest, glhip, initial_state

pytestmark = pytest.mark.gpu
G = glhip()
WALLS = [2, 2, 3, 3, 4, 4]


def _mesh(kind, n):
    if kind == "adaptive":
        return adaptive_forest(G, n, [-4.0] * 3, [4.0] * 3, WALLS, 2).mesh()
    if kind == "batch":
        ms = [G.Mesh(1, (k, 4, 3), [-k, -4, -3], [k, 4, 3], WALLS) for k in n]
        return G.Mesh.concat(ms)
    hi = np.array(n, float) * kind
    return G.Mesh(kind, n, -hi, hi, WALLS)


@pytest.mark.parametrize("kind,n", [(1, (4, 5, 5)), (1, (5, 5, 5)), (1, (17, 3, 40)), (2, (2, 2, 2)), (2, (40, 1, 1)),
                                    (2, (5, 4, 3)), ("adaptive", (5, 4, 4)), ("batch", (9, 4, 15))])
def test_upper_triangle_product_matches_the_matrix(kind, n):
    mesh = _mesh(kind, n)
    a = mesh.arrays()
    rp, col = a["row_ptr"].astype(np.int64), a["col"]
    print("symmetric product", kind, n, "blocks", col.size, flush=True)
    ctx = G.Context(0)
    try:
        ctx.set_material_pt(24.0, 0.75, bt=2.0)
        ctx.upload_mesh(mesh)
        ctx.set_solution(initial_state(mesh.n_nodes, 24.0, 0.75, 0.05, 1))
        x = np.random.default_rng(3).standard_normal(mesh.n_nodes * 18)
        row = np.repeat(np.arange(mesh.n_nodes), np.diff(rp))
        for fp32, tol in ((False, 1e-13), (True, 1e-6)):
            ctx.assemble(J=True, R=True, fp32=fp32)
            J = np.asarray(ctx.jacobian()).reshape(-1, 18, 18)
            xv = (x.astype(np.float32).astype(np.float64) if fp32 else x).reshape(-1, 18)
            y = np.zeros((mesh.n_nodes, 18))
            np.add.at(y, row, np.einsum("bij,bj->bi", J, xv[col]))
            assert np.abs(ctx.apply_jacobian(x).reshape(-1, 18) - y).max() <= tol * np.abs(y).max()
    finally:
        ctx.close()
