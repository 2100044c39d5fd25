"""GMRES through the Gram-Schmidt kernels at the edges of their chunks: fewer
values than a chunk, a whole number of chunks, an FP32 chunk that ends with a
pair of values, the long chunks of large instances, and a batch whose second
instance starts at an odd node (FP32 loads aligned to 8 bytes only).  A wrong
or missing value in a product or an update leaves a false residual estimate,
so the residual of the returned update, formed by the product itself, is held
to the tolerance of the solve (with the slack of its own rounding)."""
import numpy as np
import pytest

import oracle_lib as O
from product_util import glhip, initial_state

pytestmark = pytest.mark.gpu
G = glhip()
Z = [1, 1, 1, 1, 0, 0]
P, T = 24.0, 0.75

# cells of the instances: 486 dofs (2 mod 4), 9216 = 9 * 1024, 1350, 1.15e6
# (chunks of 4096), and a batch of 27 and 75 nodes
CASES = [[(2, 2, 2)], [(7, 7, 7)], [(4, 4, 2)], [(39, 39, 39)], [(2, 2, 2), (4, 4, 2), (7, 7, 7)]]


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("cells", CASES, ids=["-".join("x".join(map(str, n)) for n in c) for c in CASES])
def test_gmres_update_has_the_residual_it_reports(cells, fp32):
    meshes = [G.Mesh(1, n, -0.6 * np.array(n), 0.6 * np.array(n), Z) for n in cells]
    mesh = G.Mesh.concat(meshes) if len(meshes) > 1 else meshes[0]
    print("nodes", mesh.n_nodes, "instances", mesh.n_inst, flush=True)
    ctx = G.Context(0)
    try:
        ctx.upload_mesh(mesh)
        ctx.set_materials(np.array([O.coef(P, T)] * len(cells)))
        ctx.set_solution(initial_state(mesh.n_nodes, P, T, 0.05, 1))
        ctx.assemble(J=True, R=True, matrix_free=True, fp32=fp32)
        rtol = 1e-6
        its, rel = ctx.solve(rtol=rtol, maxit=2000, restart=30)
        b, x = ctx.rhs(), ctx.update()
        # FP32: the product itself is good to 2e-6 of its terms
        res = np.linalg.norm(b - ctx.apply_jacobian(x)) / np.linalg.norm(b)
        print("its", its, "reported", rel, "residual", res, flush=True)
        assert rel <= rtol
        assert res <= rtol * 1.001 + (4e-6 if fp32 else 0.0)
    finally:
        ctx.close()
