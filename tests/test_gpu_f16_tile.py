"""The FP16-mode prefill GEMM's 128-token tile (f16_mi 4, csrc/ns_gemm_f16.hip): against the oracle at
ragged batches around its tiles, and bit for bit against the 256-token tile (the same parts in the same
order), with the split-K finished by the reduce-scatter, also where a part owns half an MFMA tile
(8 parts, and 16 of the 256-token tile), and by the last arrival."""
import numpy as np
import pytest

import ns_oracle as O
import nsffn as N
from helpers import f16_value, rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    c = N.Context(0)
    c.set_tuning("gemm_skinny", 0)
    yield c
    torch.cuda.synchronize()
    c.close()


def weights(qtype, seed, rows, cols):
    host = N.synth_weights(qtype, seed, rows, cols)
    return host, torch.from_numpy(N.retile(host, qtype, cols, rows, N.ROW_MAJOR, N.CDNA4)).cuda()


@pytest.mark.parametrize("kparts", [1, 2, 3, 8])
@pytest.mark.parametrize("batch", [127, 129, 300])
@pytest.mark.parametrize("qtype", [N.Q4_K, N.Q6_K], ids=["q4k", "q6k"])
def test_f16_tile128_down(ctx, tune, qtype, batch, kparts):
    cols, rows = 2304, 320
    tune("gemm_kparts", kparts)
    host, w = weights(qtype, 0x71, rows, cols)
    bits = N.synth_normal_f16(0x72, batch * cols).reshape(batch, cols)
    x = torch.from_numpy(bits.view(np.int16)).cuda()
    got = {}
    for mi in (4, 8):
        tune("f16_mi", mi)
        for rs in (1, 0):
            tune("gemm_rs", rs)
            y = torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda")
            ctx.ffn_down(w, qtype, N.CDNA4, cols, rows, batch, x, y, half_input=True, fast_swa=True)
            torch.cuda.synchronize()
            got[mi, rs] = y.cpu().numpy()
    assert rel_err(got[4, 1], O.gemm(qtype, O.ROW_MAJOR, host, cols, rows, batch, bits, 1)) <= 1e-3
    for k in got:
        assert np.array_equal(got[k].view(np.uint32), got[4, 1].view(np.uint32)), k


@pytest.mark.parametrize("kparts", [1, 4])
@pytest.mark.parametrize("batch", [129, 256])
def test_f16_tile128_gate_up(ctx, tune, batch, kparts):
    cols, rows = 1024, 320
    tune("gemm_kparts", kparts)  # the plans of the two tiles may split K differently
    hg, wg = weights(N.Q4_K, 0x73, rows, cols)
    hu, wu = weights(N.Q4_K, 0x74, rows, cols)
    bits = N.synth_normal_f16(0x75, batch * cols).reshape(batch, cols)
    x = torch.from_numpy(bits.view(np.int16)).cuda()
    out = []
    for mi in (4, 8):
        tune("f16_mi", mi)
        h = torch.empty((batch, rows), dtype=torch.int16, device="cuda")
        ctx.gate_up_geglu_rm32(wg, wu, N.CDNA4, cols, rows, batch, x, h, True)
        torch.cuda.synchronize()
        out.append(h.cpu().numpy())
    assert rel_err(f16_value(out[0].view(np.uint16)), O.gate_up_geglu_prefill(O.ROW_MAJOR, hg, hu, cols, rows, batch, bits, 1)) <= 5e-3
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("value", [1, 5, 16])
def test_f16_unknown_tile_forces_nothing(ctx, tune, value):
    """Values of f16_mi that name no tile leave the plan's: the same bits."""
    cols, rows, batch = 1024, 192, 140
    _, w = weights(N.Q4_K, 0x76, rows, cols)
    x = torch.from_numpy(N.synth_normal_f16(0x77, batch * cols).view(np.int16)).cuda()
    y = [torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
    for out, mi in zip(y, (0, value)):
        tune("f16_mi", mi)
        ctx.ffn_down(w, N.Q4_K, N.CDNA4, cols, rows, batch, x, out, half_input=True, fast_swa=True)
    torch.cuda.synchronize()
    assert torch.isfinite(y[0]).all() and torch.equal(y[0], y[1])


@pytest.mark.parametrize("qtype", [N.Q4_K, N.Q6_K], ids=["q4k", "q6k"])
def test_f16_tile256_sixteen_parts(ctx, tune, qtype):
    """16 K parts of the 256-token tile, the most that the plan takes: each part finishes one 16-token unit of the
    reduce-scatter, bit for bit what the last arrival adds up; a ragged second token tile and column tile."""
    cols, rows, batch = 8192, 320, 300
    host, w = weights(qtype, 0x78, rows, cols)
    bits = N.synth_normal_f16(0x79, batch * cols).reshape(batch, cols)
    x = torch.from_numpy(bits.view(np.int16)).cuda()
    tune("f16_mi", 8)
    tune("gemm_kparts", 16)
    y = [torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
    for rs, out in enumerate(y):
        tune("gemm_rs", rs)
        ctx.ffn_down(w, qtype, N.CDNA4, cols, rows, batch, x, out, half_input=True, fast_swa=True)
    torch.cuda.synchronize()
    last, scatter = (t.cpu().numpy() for t in y)
    assert np.array_equal(last.view(np.uint32), scatter.view(np.uint32))
    assert rel_err(scatter, O.gemm(qtype, O.ROW_MAJOR, host, cols, rows, batch, bits, 1)) <= 1e-3
