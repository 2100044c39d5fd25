"""Calls that run out of device memory, and the calls after them, with the
library's host code on hip_host.cpp's runtime (no GPU, no kernels)."""
import pytest

import hip_host

NET = """
rng = np.random.default_rng(0)
X = rng.uniform(-1, 1, (70, 6)).astype(np.float32)
Y = rng.standard_normal((70, 18)).astype(np.float32)
def zeros(n):
    return np.zeros((n, 6), np.float32), np.zeros((n, 18), np.float32)
def trained():
    net = G.MLP(n_freq=32, sigma=1.0, width=%d, depth=2, n_out=18, seed=1)
    net.set_data(X, Y)
    net.train(1, batch=128)
    assert H.hh_bad() == 0
    return net
def refused(f, *a):
    try:
        f(*a)
        return False
    except G.GLHError as e:
        assert "out of memory" in str(e), e
        return True
"""


@pytest.mark.parametrize("width", [64, 320])
def test_training_after_a_refused_gradient_takes_its_buffers_again(width):
    # a gradient of 2^16 rows that does not get all of its buffers, for every
    # place at which the memory can end: some of the training batch's are gone
    # by then, so training has to take them again and capture its step anew
    hip_host.run(NET % width + """
for k in range(64):
    net = trained()
    H.hh_limit(H.hh_used() + k * (65536 * 64))
    out = refused(net.loss_grad, *zeros(65536))
    H.hh_limit(NO_LIMIT)
    if not out:
        break
    n = H.hh_captures()
    net.train(1, batch=128)
    assert H.hh_bad() == 0 and H.hh_captures() == n + 1, (k, H.hh_bad(), H.hh_captures(), n)
    net.loss_grad(X, Y)
    net.predict(X)
    net.train(1, batch=128)
    assert H.hh_bad() == 0
    net.close()
assert k > 3, k
""")


@pytest.mark.parametrize("width", [64, 320])
def test_refused_data_leaves_none_to_train_on(width):
    hip_host.run(NET % width + """
net = trained()
n = 1 << 20
for room in (0, n * 6 * 4):  # neither array, or the points alone
    H.hh_limit(H.hh_used() + room)
    assert refused(net.set_data, *zeros(n))
    H.hh_limit(NO_LIMIT)
    try:
        net.train(1, batch=128)
        raise AssertionError("trained on data that is gone")
    except G.GLHError as e:
        assert "no training data" in str(e), e
    net.set_data(X, Y)
    net.train(1, batch=128)
    assert H.hh_bad() == 0
""")


def test_a_refused_mesh_leaves_none():
    # a mesh of other degree and size that does not get all of its buffers,
    # for every place at which the memory can end
    hip_host.run("""
small = G.Mesh(2, (1, 1, 1), (-2, -2, -2), (2, 2, 2), [1, 1, 1, 1, 0, 0])
large = adaptive_forest(G, (6, 6, 6), (-5, -5, -6), (5, 5, 6), [1, 1, 1, 1, 0, 0], 1, 0, frac=0.3).mesh()
U = initial_state(small.n_nodes, 20.0, 0.5, 0.05, 1)
ctx = G.Context(0)
ctx.set_material_pt(20.0, 0.5)
for k in range(4096):
    ctx.upload_mesh(small)
    ctx.set_solution(U)
    ctx.assemble()
    ctx.solve()
    H.hh_limit(H.hh_used() + k * 2000)
    out = False
    try:
        ctx.upload_mesh(large)
    except G.GLHError as e:
        assert "out of memory" in str(e), e
        out = True
    H.hh_limit(NO_LIMIT)
    if not out:
        break
    for f in (lambda: ctx.assemble(), lambda: ctx.residual_norm(), lambda: ctx.set_solution(U), lambda: ctx.solve(),
              lambda: ctx.newton_solve(), lambda: ctx.newton_step(), lambda: ctx.solution()):
        try:
            f()
            raise AssertionError("a call went through without a mesh")
        except G.GLHError as e:
            assert "no mesh uploaded" in str(e), e
assert k > 20, k
""")


@pytest.mark.parametrize("mesh", ["box", "hanging"])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("matrix_free", [False, True])
def test_what_fits_without_the_scratch_of_the_faster_paths_is_not_refused(mesh, fp32, matrix_free):
    # The memory that a solve holds at its end, less the upper-triangle
    # products' map and scratch (4 + 18 * 8 bytes a block) or, matrix-free, the
    # setup's shares of the diagonal blocks (171 * 8 doubles a Q1 cell): with
    # that much the same calls go through, twice, and with a block less than
    # that they are refused for the buffers that they cannot do without.
    hip_host.run("""
mesh, fp32, mf = %r, %r, %r
if mesh == "box":
    m = G.Mesh(1, (9, 8, 7), (-4, -4, -4), (4, 4, 4), [1, 1, 1, 1, 0, 0])
else:
    m = adaptive_forest(G, (6, 6, 6), (-5, -5, -6), (5, 5, 6), [1, 1, 1, 1, 0, 0], 1, 0, frac=0.3).mesh()
    assert m.constraints()["n_hanging"] > 0
assert m.nnzb >= 4096, m.nnzb
U = initial_state(m.n_nodes, 20.0, 0.5, 0.05, 1)
def calls(ctx):
    ctx.set_material_pt(20.0, 0.5)
    ctx.upload_mesh(m)
    ctx.set_solution(U)
    for _ in range(2):
        ctx.assemble(fp32=fp32, matrix_free=mf)
        ctx.solve(rtol=1e-3, restart=100)  # a basis larger than the scratch: that is there before it
        ctx.newton_step()
        ctx.apply_jacobian(U)
H.hh_limit(NO_LIMIT)
ctx = G.Context(0)
n0 = H.hh_used()
calls(ctx)
held = H.hh_used() - n0
ctx.close()
assert H.hh_used() <= n0
spare = 171 * 8 * 8 * m.n_cells if mf else 148 * m.nnzb
ctx = G.Context(0)
fills = H.hh_launches(b"k_sym_fill")
least = H.hh_used() + held - spare + (171 * 8 * 8 if mf else 0)  # a setup needs one cell's shares
H.hh_limit(least)
calls(ctx)
whole = H.hh_launches(b"k_spmv_up")
calls(ctx)
assert mf or H.hh_launches(b"k_spmv_up") == whole, "upper-triangle products without their scratch"
if not mf:
    # the blocks below the diagonal are there for whoever reads them (in FP32
    # the norms' zeros end the solve before its basis: the scratch stays away)
    assert mesh == "hanging" or fp32 or H.hh_launches(b"k_sym_fill") > fills
    n = H.hh_launches(b"k_sym_fill")
    ctx.jacobian()
    assert H.hh_launches(b"k_sym_fill") == n
ctx.close()
ctx = G.Context(0)
H.hh_limit(least - 324 * 8)
try:
    calls(ctx)
    raise AssertionError("the limit was not the least")
except G.GLHError as e:
    assert "out of memory" in str(e), e
""" % (mesh, fp32, matrix_free))
