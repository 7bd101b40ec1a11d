"""Batch 2-4 on tensors of more slabs than one round of workgroups holds (csrc/ns_gemv_mfma.hip, the
streaming form): the same numbers as from calls on 65,536-row pieces, which give every wave one slab.
Slab counts just past one round and just past a half-full last one, that leave waves of the last step without
a slab, and of three steps; one, two, three and fifteen super-blocks per row."""
import pytest

import nsffn as N

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

PIECE = 65536


@pytest.mark.parametrize("rows,nb,batch", [(131136, 2, 2), (131136, 1, 3), (196672, 3, 4), (262144, 15, 3), (270400, 2, 4),
                                           (229440, 3, 2), (361472, 2, 4)])
@pytest.mark.parametrize("half", [False, True], ids=["fp32", "fp16"])
@pytest.mark.parametrize("qtype", [N.Q4_K, N.Q6_K], ids=["q4k", "q6k"])
def test_streaming_matches_pieces(qtype, half, rows, nb, batch):
    cols, size = nb * 256, N.BLOCK_BYTES[qtype]
    ctx = N.Context(0)
    ctx.set_tuning("gemm_skinny", 0)  # fp16 Q4_K stays on this kernel
    g = torch.Generator(device="cuda").manual_seed(rows + nb)
    blk = torch.randint(0, 256, (rows * nb, size), dtype=torch.uint8, device="cuda", generator=g)
    factors = (0, 2, 4) if qtype == N.Q4_K else (208, 210)
    for a, b in zip(factors, factors[1:]):
        blk[:, a:b] = torch.full((rows * nb, 1), 1e-4, device="cuda").half().view(torch.uint8)
    w = torch.empty_like(blk).view(-1)
    N.retile_device(blk.view(-1), w, qtype, cols, rows, N.ROW_MAJOR, N.CDNA4)
    x = torch.randn(batch, cols, device="cuda", generator=g)
    x = x.half() if half else x
    y = torch.full((batch, rows), float("nan"), device="cuda")
    ctx.matmul(w, qtype, N.CDNA4, cols, rows, batch, x, y, half_input=half)
    for r0 in range(0, rows, PIECE):
        n = min(PIECE, rows - r0)
        z = torch.empty(batch, n, device="cuda")
        ctx.matmul(w[r0 * nb * size:(r0 + n) * nb * size], qtype, N.CDNA4, cols, n, batch, x, z, half_input=half)
        if n == PIECE:  # (a shorter piece splits its columns: other sums)
            assert torch.equal(y[:, r0:r0 + n], z), r0
        else:
            assert torch.allclose(y[:, r0:r0 + n], z, rtol=0, atol=2.0 ** -24 * 8 * cols ** 0.5 * float(z.abs().max())), r0
    ctx.close()
