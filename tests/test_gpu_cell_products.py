"""The cell loop of the residual and of the matrix-free product at the edges
of its launch shapes, against the oracle's cell loop (orc_cells_apply):
single cells, workgroups that are not full (7 cells each, 8 ranges of cells),
and both sides of the cell counts at which the thread mapping changes (Q2
FP64 1536, Q2 FP32 3072, Q1 512).  FP64 to 1e-12, the FP32 form to 2e-6, the
bounds of the other parity tests."""
import numpy as np
import pytest

import oracle_lib as O
from product_util import glhip, initial_state

pytestmark = pytest.mark.gpu
G = glhip()
Z = [1, 1, 1, 1, 0, 0]
WALLS = [2, 2, 3, 3, 4, 4]

# degree, cells per direction, boundary ids, bt
CASES = [
    (2, (1, 1, 1), WALLS, 2.0),
    (2, (7, 1, 1), Z, 1.0e10),
    (2, (3, 3, 1), WALLS, 2.0),
    (2, (16, 12, 8), Z, 1.0e10),      # 1536
    (2, (29, 53, 1), WALLS, 2.0),     # 1537
    (2, (16, 16, 12), WALLS, 2.0),    # 3072
    (2, (439, 7, 1), Z, 1.0e10),      # 3073
    (1, (1, 1, 1), WALLS, 2.0),
    (1, (5, 3, 1), Z, 1.0e10),
    (1, (8, 8, 8), WALLS, 2.0),       # 512
    (1, (27, 19, 1), WALLS, 2.0),     # 513
    (1, (57, 8, 1), Z, 1.0e10),       # 8 ranges of 57 = 8 * 7 + 1 cells
]


@pytest.fixture(scope="module")
def ctx():
    c = G.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("deg,n,sides,bt", CASES, ids=["q%d_%dx%dx%d" % (c[0], *c[1]) for c in CASES])
def test_residual_and_product_match_the_oracle_cell_loop(ctx, deg, n, sides, bt):
    p, t = 24.0, 0.75
    hi = np.array([1.3, 1.1, 0.9]) * deg * np.array(n) / 2
    mesh = G.Mesh(deg, n, -hi, hi, sides)
    print("cells", mesh.n_cells, flush=True)
    ctx.set_material_pt(p, t, bt=bt)
    ctx.upload_mesh(mesh)
    ctx.set_solution(initial_state(mesh.n_nodes, p, t, 0.05, 1))
    U = ctx.solution()
    x = np.random.default_rng(2).standard_normal(U.size)
    r, (y,) = O.cells_apply(deg, mesh.arrays(), mesh.n_nodes, O.coef(p, t, bt=bt), U, X=[x])
    for fp32, tol in ((False, 1e-12), (True, 2e-6)):
        ctx.assemble(J=True, R=True, matrix_free=True, fp32=fp32)
        assert np.abs(ctx.rhs() - r).max() <= 1e-12 * np.abs(r).max()
        assert np.abs(ctx.apply_jacobian(x) - y).max() <= tol * np.abs(y).max()


# cells of a colour below and above the counts at which its pairs go to
# several workgroups
ASM_CASES = [(1, (3, 2, 2)), (1, (20, 18, 16)), (2, (2, 2, 1)), (2, (9, 9, 9)), (2, (18, 16, 29))]


@pytest.mark.parametrize("deg,n", ASM_CASES, ids=["q%d_%dx%dx%d" % (c[0], *c[1]) for c in ASM_CASES])
def test_assembled_product_matches_the_oracle_cell_loop(ctx, deg, n):
    p, t, bt = 24.0, 0.75, 2.0
    hi = np.array([1.3, 1.1, 0.9]) * deg * np.array(n) / 2
    mesh = G.Mesh(deg, n, -hi, hi, WALLS)
    print("cells", mesh.n_cells, flush=True)
    ctx.set_material_pt(p, t, bt=bt)
    ctx.upload_mesh(mesh)
    ctx.set_solution(initial_state(mesh.n_nodes, p, t, 0.05, 1))
    U = ctx.solution()
    x = np.random.default_rng(3).standard_normal(U.size)
    _, (y,) = O.cells_apply(deg, mesh.arrays(), mesh.n_nodes, O.coef(p, t, bt=bt), U, X=[x], rhs=False)
    for fp32, tol in ((False, 1e-12), (True, 2e-6)):
        ctx.assemble(J=True, R=False, fp32=fp32)
        assert np.abs(ctx.apply_jacobian(x) - y).max() <= tol * np.abs(y).max()


# one chunk of cells and several (3640 Q2 or 12300 Q1 cells each): nodes whose
# cells lie in different chunks are written by one and added to by the others
DIAG_CASES = [(1, (1, 1, 1)), (1, (24, 23, 23)), (2, (3, 1, 2)), (2, (11, 21, 17))]


@pytest.mark.parametrize("deg,n", DIAG_CASES, ids=["q%d_%dx%dx%d" % (c[0], *c[1]) for c in DIAG_CASES])
def test_matrix_free_diagonal_blocks_match_the_assembled_ones(ctx, deg, n):
    p, t, bt = 24.0, 0.75, 2.0
    hi = np.array([1.3, 1.1, 0.9]) * deg * np.array(n) / 2
    mesh = G.Mesh(deg, n, -hi, hi, WALLS)
    print("cells", mesh.n_cells, flush=True)
    ctx.set_material_pt(p, t, bt=bt)
    ctx.upload_mesh(mesh)
    ctx.set_solution(initial_state(mesh.n_nodes, p, t, 0.05, 1))
    ctx.assemble(J=True, R=False)
    D = ctx.diagonal_blocks()
    for fp32 in (False, True):  # the blocks are FP64 in both
        ctx.assemble(J=True, R=False, matrix_free=True, fp32=fp32)
        assert np.abs(ctx.diagonal_blocks() - D).max() <= 1e-12 * np.abs(D).max()
