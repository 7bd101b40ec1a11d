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
                                     (3, 256), (8199, 3), (8199, 9), (4097, 130)])
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


@pytest.mark.parametrize("qtype,rows,nb,same", [
    (N.Q4_K, 32768, 1, True), (N.Q4_K, 32768, 4, True), (N.Q4_K, 32768, 5, False), (N.Q4_K, 8193, 65, True),
    (N.Q4_K, 8192, 1, False), (N.Q4_K, 4096, 65, False), (N.Q6_K, 32768, 8, True), (N.Q6_K, 32768, 9, False),
    (N.Q6_K, 32768, 17, True), (N.Q6_K, 32768, 28, False), (N.Q6_K, 8193, 8, True), (N.Q6_K, 4097, 4, True),
    (N.Q6_K, 4096, 1, False), (N.Q6_K, 4097, 127, True), (N.Q6_K, 4097, 128, False)])
def test_short_rows_on_the_slab_kernel(ctx, tune, qtype, rows, nb, same):
    """Which kernel many rows of few super-blocks run on (the row kernel took up to 6 times as long there): the
    two sum in different orders, so the slab kernel's bits tell it."""
    cols = nb * 256
    w = torch.from_numpy(N.synth_weights(qtype, 0x62, rows, cols)).cuda()
    x = torch.from_numpy(N.synth_normal_f32(0x63, cols)).cuda()
    y = [torch.empty(rows, dtype=torch.float32, device="cuda") for _ in range(2)]
    ctx.matmul(w, qtype, N.ROW_MAJOR, cols, rows, 1, x, y[0])
    tune("gemv_row", 0)
    ctx.matmul(w, qtype, N.ROW_MAJOR, cols, rows, 1, x, y[1])
    torch.cuda.synchronize()
    assert torch.equal(y[0], y[1]) == same
