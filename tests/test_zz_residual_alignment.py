"""glh_residual_into on buffers aligned to a double and no better (a view from
an odd value on): the same bits as on whole allocations, and nothing written
beside them; Q1 and Q2 boxes, a batch and a mesh with hanging nodes."""
import numpy as np
import pytest

import oracle_lib as O
from product_util import adaptive_forest, glhip, initial_state
from test_zz_no_alloc import _Dev

pytestmark = pytest.mark.gpu
G = glhip()
Z = [1, 1, 1, 1, 0, 0]


def _mesh(name):
    if name == "hanging":
        return adaptive_forest(G, (3, 3, 3), (-5, -5, -6), (5, 5, 6), Z, 1, 0, frac=0.3).mesh()
    box = [G.Mesh(2 if name == "q2" else 1, n, (-3, -3, -3), (3, 3, 3), Z) for n in ((3, 4, 2), (2, 2, 2))]
    return G.Mesh.concat(box) if name == "batch" else box[0]


@pytest.mark.parametrize("name", ["q1", "q2", "batch", "hanging"])
def test_buffers_aligned_to_a_double(name):
    print("residual alignment", name, flush=True)
    p, t = 22.0, 0.8
    m = _mesh(name)
    n, s = m.n_nodes * 18, m.n_inst
    ctx, dev = G.Context(0), _Dev()
    try:
        ctx.upload_mesh(m)
        ctx.set_materials(np.array([O.coef(p, t)] * s))
        U = initial_state(m.n_nodes, p, t, 0.05, 1)
        out = []
        for off in (0, 1):
            # values before and after stay as they are
            Ud = dev.upload(np.concatenate([np.full(off, np.nan), U, np.full(2, np.nan)]))
            Rd = dev.upload(np.full(n + off + 2, 7.0))
            Nd = dev.upload(np.full(s + off + 2, 7.0))
            assert dev.hip.hipDeviceSynchronize() == 0
            ctx.residual_into(Ud + 8 * off, Rd + 8 * off, Nd + 8 * off)
            R, N = dev.download(Rd, n + off + 2), dev.download(Nd, s + off + 2)
            assert np.all(R[:off] == 7.0) and np.all(R[off + n:] == 7.0)
            assert np.all(N[:off] == 7.0) and np.all(N[off + s:] == 7.0)
            out.append((R[off:off + n], N[off:off + s]))
        assert np.all(np.isfinite(out[0][0])) and np.all(out[0][1] > 0)
        assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    finally:
        dev.close()
        ctx.close()
