"""The decode GEMV on row-major tensors (csrc/ns_gemv_row.hip) against the oracle and the slab kernel:
row counts around a step's rows and past one round of workgroups, rows that end inside a wave's 16
super-blocks, fill it, and need 2, 3, 4 and more waves, and a tensor whose last block ends the buffer."""
import numpy as np
import pytest

import ns_oracle as O
import nsffn as N
from helpers import rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    c = N.Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


@pytest.mark.parametrize("rows,nb", [(1, 1), (7, 15), (9, 16), (64, 17), (33, 33), (130, 47), (5, 60), (66, 65),
                                     (3, 256), (8199, 3)])
@pytest.mark.parametrize("qtype", [N.Q4_K, N.Q6_K], ids=["q4k", "q6k"])
def test_gemv_row(ctx, tune, qtype, rows, nb):
    cols = nb * 256
    host = N.synth_weights(qtype, 0x60 + nb, rows, cols)
    w = torch.from_numpy(host).cuda()
    x = N.synth_normal_f32(0x61, cols)
    xd = torch.from_numpy(x).cuda()
    y = torch.full((rows + 1,), float("nan"), dtype=torch.float32, device="cuda")
    ctx.matmul(w, qtype, N.ROW_MAJOR, cols, rows, 1, xd, y)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[rows])
    assert rel_err(got[:rows], O.gemv(qtype, O.ROW_MAJOR, host, cols, rows, x)) <= 1e-3
    # the slab kernel sums the same exact products in another order: 24 bits over cols terms
    tune("gemv_row", 0)
    z = torch.empty(rows, dtype=torch.float32, device="cuda")
    ctx.matmul(w, qtype, N.ROW_MAJOR, cols, rows, 1, xd, z)
    torch.cuda.synchronize()
    assert rel_err(got[:rows], z.cpu().numpy()) <= 2.0 ** -24 * 8 * np.sqrt(cols)
