"""The prefill GEMM for few tokens (csrc/ns_gemm_skinny.hip) against the oracle, at the edges of its
tiles: one token past a 32-token tile and the largest batch of each tile height, a last column tile
that is partly past the rows, more super-block groups than super-blocks and a remainder of them,
split K over workgroups, both wave splits (4 or 8 super-block groups).

Bars: the repository's 1e-3 (FP32 mode) and, against the FP16-mode oracle, 1e-3 (5e-3 for the
pair, whose h is fp16 of a product of two rounded sums).
"""
import numpy as np
import pytest

import ns_oracle as O
import nsffn as N
from helpers import f16_value, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

LNAME = {N.CDNA4: "cdna4", N.ROW_MAJOR: "rowmajor"}
# (rows, cols, batch): tiles of 32, 64 and 128 tokens, 1 to 17 super-blocks
SHAPES = [(64, 256, 5), (192, 768, 32), (320, 1024, 33), (128, 2304, 64), (192, 1280, 65), (64, 4352, 128)]


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    c = N.Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


def weights(qtype, seed, rows, cols, layout):
    host = N.synth_weights(qtype, seed, rows, cols)
    lay = host if layout == N.ROW_MAJOR else N.retile(host, qtype, cols, rows, N.ROW_MAJOR, layout)
    return host, torch.from_numpy(np.ascontiguousarray(lay)).cuda()


def tokens(seed, batch, cols):
    bits = N.synth_normal_f16(seed, batch * cols).reshape(batch, cols)
    return bits, torch.from_numpy(bits.view(np.int16)).cuda()


@pytest.mark.parametrize("wk,kparts", [(4, 1), (8, 1), (4, 3), (8, 2), (0, 0)],
                         ids=["wk4", "wk8", "wk4_split3", "wk8_split2", "plan"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("qtype", [N.Q4_K, N.Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("mode", ["fp32_cdna4", "fp16_cdna4", "fp32_rowmajor"])
def test_skinny_matmul(ctx, tune, mode, qtype, shape, wk, kparts):
    rows, cols, batch = shape
    layout, fast = (N.ROW_MAJOR if mode.endswith("rowmajor") else N.CDNA4), mode.startswith("fp16")
    if layout == N.ROW_MAJOR:
        rows -= 11  # ragged: the row-major layout has no 64-row rule
    tune("gemm_skinny", 128)
    tune("skinny_wk", wk)
    tune("gemm_kparts", min(kparts, cols // 256))
    host, w = weights(qtype, 0x51, rows, cols, layout)
    bits, x = tokens(0x52, batch, cols)
    y = torch.full((batch + 1, rows), float("nan"), dtype=torch.float32, device="cuda")
    ctx.ffn_down(w, qtype, layout, cols, rows, batch, x, y, half_input=True, fast_swa=fast)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.isnan(got[batch]).all()  # nothing past the batch is written
    ref = O.gemm(qtype, O.ROW_MAJOR, host, cols, rows, batch, bits, 1 if fast else 0)
    assert rel_err(got[:batch], ref) <= 1e-3


@pytest.mark.parametrize("wk,kparts", [(4, 1), (8, 2), (0, 0)], ids=["wk4", "wk8_split2", "plan"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("fast", [False, True], ids=["fp32", "fp16"])
def test_skinny_gate_up(ctx, tune, fast, shape, wk, kparts):
    rows, cols, batch = shape
    tune("gemm_skinny", 128)
    tune("skinny_wk", wk)
    tune("gemm_kparts", min(kparts, cols // 256))
    hg, wg = weights(N.Q4_K, 0x53, rows, cols, N.CDNA4)
    hu, wu = weights(N.Q4_K, 0x54, rows, cols, N.CDNA4)
    bits, x = tokens(0x55, batch, cols)
    h = torch.full((batch + 1, rows), 0x7E00, dtype=torch.int16, device="cuda")
    ctx.gate_up_geglu_rm32(wg, wu, N.CDNA4, cols, rows, batch, x, h, fast)
    torch.cuda.synchronize()
    got = h.cpu().numpy()
    assert (got[batch] == 0x7E00).all()
    ref = O.gate_up_geglu_prefill(O.ROW_MAJOR, hg, hu, cols, rows, batch, bits, 1 if fast else 0)
    assert rel_err(f16_value(got[:batch].view(np.uint16)), ref) <= (5e-3 if fast else 1e-3)


def test_skinny_exact_min_term_and_large_sums(ctx, tune):
    """FP32 mode, blocks with d = 0 (the output is the min term alone) on activations whose 32-wide
    groups sum past fp16's range: the three-piece group sums lose nothing (float64 closed form)."""
    tune("gemm_skinny", 128)
    cols, rows, batch = 768, 64, 40
    host = N.synth_weights(N.Q4_K, 0x56, rows, cols).copy()
    host.reshape(-1, 144)[:, 0:2] = 0
    w = torch.from_numpy(N.retile(host, N.Q4_K, cols, rows, N.ROW_MAJOR, N.CDNA4)).cuda()
    x = (np.random.RandomState(7).randn(batch, cols) * 3.0 + 2100.0).astype(np.float16)
    y = torch.empty((batch, rows), dtype=torch.float32, device="cuda")
    ctx.matmul(w, N.Q4_K, N.CDNA4, cols, rows, batch, torch.from_numpy(x.view(np.int16)).cuda(), y, half_input=True)
    torch.cuda.synchronize()
    want = x.astype(np.float64) @ O.dequant_rows(N.Q4_K, O.ROW_MAJOR, host, cols, rows, 0, rows).astype(np.float64).T
    # 24 block groups of exact products, each sum and product rounded to 24 bits
    assert rel_err(y.cpu().numpy(), want) <= 64 * 2.0 ** -24


@pytest.mark.parametrize("batch", [2, 4, 31, 33, 70])
@pytest.mark.parametrize("v", ["q4", "q6", "tied"])
@pytest.mark.parametrize("layout", [N.ROW_MAJOR, N.CDNA4], ids=LNAME.get)
def test_qkv_one_launch(ctx, tune, layout, v, batch):
    """Q, K and V as column tiles of one launch equal the three projections by themselves up to the sum's
    order (one launch may split K differently), ragged rows included; Q6_K scales span -128..127, where
    batch 2-4 has to stay exact (24-bit sums), and the tied V is K bit for bit."""
    cols, q_rows, kv_rows = 1280, 320, 192
    if layout == N.ROW_MAJOR:
        q_rows, kv_rows = 331, 135
    vt = N.Q6_K if v == "q6" else N.Q4_K
    host, dev = zip(*(weights(t, 0x57 + i, r, cols, N.ROW_MAJOR) for i, (t, r) in
                      enumerate(((N.Q4_K, q_rows), (N.Q4_K, kv_rows), (vt, kv_rows)))))
    if v == "q6":
        host[2].reshape(-1, 210)[:, 192:208] = np.random.RandomState(3).randint(0, 256, (kv_rows * cols // 256, 16))
    dev = [torch.from_numpy(np.ascontiguousarray(h if layout == N.ROW_MAJOR else
                                                 N.retile(h, t, cols, r, N.ROW_MAJOR, layout))).cuda()
           for h, (t, r) in zip(host, ((N.Q4_K, q_rows), (N.Q4_K, kv_rows), (vt, kv_rows)))]
    bits, x = tokens(0x5A, batch, cols)
    out = [torch.full((batch, r), float("nan"), dtype=torch.float32, device="cuda") for r in (q_rows, kv_rows, kv_rows)]
    ctx.qkv(dev[0], dev[1], None if v == "tied" else dev[2], vt, layout, cols, q_rows, kv_rows, batch, x, *out)
    torch.cuda.synchronize()
    got = [o.cpu().numpy() for o in out]
    xf = bits.view(np.float16).astype(np.float64)
    for i, (t, r) in enumerate(((N.Q4_K, q_rows), (N.Q4_K, kv_rows), (vt, kv_rows))):
        if i == 2 and v == "tied":
            assert np.array_equal(got[2].view(np.uint32), got[1].view(np.uint32))
            continue
        want = xf @ O.dequant_rows(t, O.ROW_MAJOR, host[i], cols, r, 0, r).astype(np.float64).T
        # sums of 24-bit roundings; Q6_K above 4 tokens may round sc*(v-32) to 11 bits
        bar = 1e-3 if t == N.Q6_K and batch > 4 else 64 * 2.0 ** -24
        assert rel_err(got[i], want) <= bar, i


@pytest.mark.parametrize("batch", [2, 3, 4])
@pytest.mark.parametrize("qtype,layout", [(N.Q4_K, N.CDNA4), (N.Q4_K, N.ROW_MAJOR), (N.Q6_K, N.ROW_MAJOR)],
                         ids=["q4k-cdna4", "q4k-rowmajor", "q6k-rowmajor"])
def test_small_batch_fp16_exact(ctx, qtype, layout, batch):
    """Batch 2-4 with fp16 x where this kernel takes it: 24-bit sums of exact products, Q6_K scales over the
    whole int8 range; an x that is not 16-byte aligned gives the same (by the small-batch kernels)."""
    cols, rows = 2304, 192
    host = N.synth_weights(qtype, 0x5B, rows, cols).copy()
    if qtype == N.Q6_K:
        host.reshape(-1, 210)[:, 192:208] = np.random.RandomState(4).randint(0, 256, (rows * cols // 256, 16))
    img = host if layout == N.ROW_MAJOR else N.retile(host, qtype, cols, rows, N.ROW_MAJOR, layout)
    w = torch.from_numpy(np.ascontiguousarray(img)).cuda()
    bits, x = tokens(0x5C, batch, cols)
    want = bits.view(np.float16).astype(np.float64) @ O.dequant_rows(qtype, O.ROW_MAJOR, host, cols, rows, 0, rows).astype(np.float64).T
    shifted = torch.empty(batch * cols + 4, dtype=torch.int16, device="cuda")[4:]
    shifted.copy_(x.reshape(-1))
    for xin in (x, shifted):
        y = torch.empty((batch, rows), dtype=torch.float32, device="cuda")
        ctx.matmul(w, qtype, layout, cols, rows, batch, xin, y, half_input=True)
        torch.cuda.synchronize()
        assert rel_err(y.cpu().numpy(), want) <= 64 * 2.0 ** -24


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")], ids=str)
@pytest.mark.parametrize("layout", [N.CDNA4, N.ROW_MAJOR], ids=LNAME.get)
@pytest.mark.parametrize("batch", [32, 50])
def test_group_sums_keep_tokens_apart(ctx, layout, batch, value):
    """Q4_K, FP32 mode: x values that are not finite reach their own token's outputs alone, though the group
    sums of a wave's tokens share MFMA instructions; the others are bit for bit what they are without them."""
    cols, rows = 1280, 192
    _, w = weights(N.Q4_K, 0x5D, rows, cols, layout)
    _, x = tokens(0x5E, batch, cols)
    bad = x.clone()
    for t, c in ((3, 17), (batch - 1, cols - 1)):
        bad.view(torch.float16)[t, c] = value
    y = [torch.empty((batch, rows), dtype=torch.float32, device="cuda") for _ in range(2)]
    for xin, out in zip((x, bad), y):
        ctx.ffn_down(w, N.Q4_K, layout, cols, rows, batch, xin, out, half_input=True, fast_swa=False)
    torch.cuda.synchronize()
    clean, got = (t.cpu().numpy() for t in y)
    hit = np.zeros(batch, bool)
    hit[[3, batch - 1]] = True
    assert np.array_equal(got[~hit].view(np.uint32), clean[~hit].view(np.uint32))
    assert not np.isfinite(got[hit]).any()


def sum_error(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("batch", [2, 3, 4])
@pytest.mark.parametrize("qtype,layout", [(N.Q4_K, N.CDNA4), (N.Q4_K, N.ROW_MAJOR), (N.Q6_K, N.ROW_MAJOR)],
                         ids=["q4k-cdna4", "q4k-rowmajor", "q6k-rowmajor"])
@pytest.mark.parametrize("rows,cols", [(2048, 3840), (1024, 15360)])
def test_small_batch_sums_no_worse(ctx, tune, qtype, layout, rows, cols, batch):
    """Batch 2-4 with fp16 x: the sums are no further from 64 bits than the small-batch kernels', for one matrix
    and for Q, K and V in one launch.  5% above them is the spread of a 2-norm over 12,288 roundings and more."""
    host, w = weights(qtype, 0x5F, rows, cols, layout)
    dense = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    ctx.dequant(w, qtype, layout, cols, rows, 0, rows, out_f32=dense)
    wt = dense.double().t().contiguous()
    _, q4 = (host, w) if qtype == N.Q4_K else weights(N.Q4_K, 0x60, rows, cols, layout)
    err = {}
    for skinny in (-1, 0):
        tune("gemm_skinny", skinny)
        err[skinny] = np.zeros(2)
        for seed in range(6):
            _, x = tokens(0x61 + seed, batch, cols)
            want = x.view(torch.float16).double() @ wt
            y, q, k, v = (torch.empty((batch, rows), dtype=torch.float32, device="cuda") for _ in range(4))
            ctx.matmul(w, qtype, layout, cols, rows, batch, x, y, half_input=True)
            ctx.qkv(q4, q4, w, qtype, layout, cols, rows, rows, batch, x, q, k, v)
            err[skinny] += [sum_error(y, want), sum_error(v, want)]
    assert (err[-1] <= 1.05 * err[0]).all(), err


@pytest.mark.parametrize("qtype,layout,rows,nb,batch,tile", [
    (N.Q6_K, N.CDNA4, 65536, 1, 217, True), (N.Q4_K, N.CDNA4, 131072, 1, 65, True), (N.Q4_K, N.ROW_MAJOR, 15360, 1, 933, True),
    (N.Q6_K, N.ROW_MAJOR, 32768, 1, 1023, True), (N.Q6_K, N.CDNA4, 4096, 16, 1687, True), (N.Q4_K, N.CDNA4, 15360, 15, 1024, True),
    (N.Q4_K, N.CDNA4, 4096, 15, 157, False), (N.Q4_K, N.ROW_MAJOR, 2048, 15, 1024, False), (N.Q6_K, N.ROW_MAJOR, 2048, 15, 500, False),
    (N.Q6_K, N.CDNA4, 3840, 60, 64, False),
    (N.Q4_K, N.CDNA4, 262144, 2, 3, True), (N.Q4_K, N.CDNA4, 65536, 15, 2, True), (N.Q4_K, N.ROW_MAJOR, 64, 16, 2, True),
    (N.Q6_K, N.ROW_MAJOR, 2048, 4, 4, True), (N.Q6_K, N.ROW_MAJOR, 64, 15, 3, True), (N.Q4_K, N.CDNA4, 32768, 15, 3, False),
    (N.Q4_K, N.ROW_MAJOR, 4096, 15, 3, False), (N.Q6_K, N.ROW_MAJOR, 3840, 60, 3, False)])
def test_route_by_the_faster_kernel(ctx, tune, qtype, layout, rows, nb, batch, tile):
    """FP32 mode: which of the two kernels runs, on shapes where one of them takes 1.1 to 3 times as long.  They sum
    in different orders, so the tile or small-batch kernel's bits tell it."""
    cols = nb * 256
    _, w = weights(qtype, 0x65, rows, cols, layout)
    _, x = tokens(0x66, batch, cols)
    y = [torch.empty((batch, rows), dtype=torch.float32, device="cuda") for _ in range(2)]
    for out, skinny in zip(y, (-1, 0)):
        tune("gemm_skinny", skinny)
        ctx.matmul(w, qtype, layout, cols, rows, batch, x, out, half_input=True)
    torch.cuda.synchronize()
    assert torch.equal(y[0], y[1]) == tile
