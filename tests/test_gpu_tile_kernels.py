"""The 128- and 256-token tile GEMMs and the small-batch kernels at the batches that the few-token GEMM takes
by default: the prefill and small-batch tests of the other modules once more, on a context that never selects
it (gemm_skinny 0)."""
import numpy as np
import pytest

import ns_oracle as O
import nsffn as N
from helpers import rel_err

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_edge_cases import test_special_blocks_gate_up, test_special_blocks_gemm  # noqa: E402,F401
from test_gpu_fp16_mode import (test_fp16_gate_up_one_hot, test_fp16_mode_rounds_once_at_the_end,  # noqa: E402,F401
                                test_fp16_tiles_one_hot_bit_exact)
from test_gpu_large_inputs import (test_gate_up_prefill_large_group_sums, test_q4k_prefill_large_group_sums,  # noqa: E402,F401
                                   test_q4k_prefill_some_tokens_rescaled)
from test_gpu_parity import (test_prefill_down_small, test_prefill_gate_up_small,  # noqa: E402,F401
                             test_prefill_q6k_down_many_parts, test_prefill_split_k)
from test_gpu_q6k_scales import (test_prefill_down_full_range_scales,  # noqa: E402,F401
                                 test_prefill_down_full_range_scales_power_of_two_d)
from test_gpu_shape_sweep import test_gate_up_sweep, test_prefill_sweep, test_small_batch_sweep  # noqa: E402,F401
from test_gpu_small_batch import test_ffn_down_small_batch_half_input, test_matmul_small_batch  # noqa: E402,F401


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    c = N.Context(0)
    c.set_tuning("gemm_skinny", 0)
    yield c
    torch.cuda.synchronize()
    c.close()


@pytest.mark.parametrize("qtype,cols,rows,batch,kparts", [(N.Q4_K, 2304, 2496, 1000, 3), (N.Q4_K, 6400, 2496, 1020, 5),
                                                          (N.Q6_K, 4096, 3264, 1200, 3), (N.Q6_K, 8192, 2752, 700, 7)],
                         ids=["q4k-3parts", "q4k-5parts", "q6k-3parts", "q6k-7parts"])
def test_odd_parts(ctx, tune, qtype, cols, rows, batch, kparts):
    """FP32-mode splits of K that are no power of two, on ragged tiles: the terms are those of one part, so the
    two results differ by the order of 24-bit sums; and the repository's 1e-3 against the dequantised weights."""
    host = N.synth_weights(qtype, 0x61, rows, cols)
    w = torch.from_numpy(np.ascontiguousarray(N.retile(host, qtype, cols, rows, N.ROW_MAJOR, N.CDNA4))).cuda()
    bits = N.synth_normal_f16(0x62, batch * cols).reshape(batch, cols)
    x = torch.from_numpy(bits.view(np.int16)).cuda()
    y = [torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
    for out, parts in zip(y, (kparts, 1)):
        tune("gemm_kparts", parts)
        ctx.ffn_down(w, qtype, N.CDNA4, cols, rows, batch, x, out, half_input=True, fast_swa=False)
    torch.cuda.synchronize()
    split, one = (t.cpu().numpy() for t in y)
    assert rel_err(split, one) <= 64 * 2.0 ** -24
    want = bits.view(np.float16).astype(np.float32) @ O.dequant_rows(qtype, O.ROW_MAJOR, host, cols, rows, 0, rows).T
    assert rel_err(split, want) <= 1e-3


@pytest.mark.parametrize("batch,kparts", [(600, 8), (1300, 4)])
@pytest.mark.parametrize("qtype,layout", [(N.Q6_K, N.CDNA4), (N.Q4_K, N.ROW_MAJOR), (N.Q6_K, N.NSMFFN)],
                         ids=["q6k-cdna4", "q4k-rowmajor", "q6k-nsmffn"])
def test_down_parts_keep_their_chains(ctx, tune, qtype, layout, batch, kparts):
    """FP32 mode, 3840 x 15360: no fewer K parts than the power of two that fills the device, so no longer chains
    of fp32 sums (against 64 bits a Q6_K down in 4 parts is 1.42 times as far off as in 8): the planned result is
    that of 8 parts (3 x 15 tiles of 256 tokens) and of 4 parts (6 x 15) bit for bit.  (Q4_K on CDNA4 may take fewer:
    test_q4k_min_term.)"""
    cols, rows = 15360, 3840
    host = N.synth_weights(qtype, 0x63, rows, cols)
    img = host if layout == N.ROW_MAJOR else N.retile(host, qtype, cols, rows, N.ROW_MAJOR, layout)
    w = torch.from_numpy(np.ascontiguousarray(img)).cuda()
    x = torch.from_numpy(N.synth_normal_f16(0x64, batch * cols).reshape(batch, cols).view(np.int16)).cuda()
    y = [torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda") for _ in range(2)]
    for out, parts in zip(y, (0, kparts)):
        tune("gemm_kparts", parts)
        ctx.ffn_down(w, qtype, layout, cols, rows, batch, x, out, half_input=True, fast_swa=False)
    torch.cuda.synchronize()
    assert torch.isfinite(y[0]).all()
    assert torch.equal(y[0].view(torch.int32), y[1].view(torch.int32))


@pytest.mark.parametrize("cols,rows,batch,kparts,was", [(3840, 512, 70, 1, 1.142e-6), (3840, 512, 70, 0, 1.082e-6),
                                                        (15360, 3840, 600, 0, 1.253e-6), (21504, 256, 130, 1, 1.626e-6)])
def test_q4k_min_term(ctx, tune, cols, rows, batch, kparts, was):
    """Q4_K on CDNA4, FP32 mode, against 64 bits.  The min term's second fragment, an fp16 subnormal, kept 17 of its 22
    bits, which put the outputs `was` off with 1, 4, 8 (the power of two: 6 now) and 1 K parts.  Scaled, what is left is
    the fp32 sums: 6.9e-7, 5.8e-7, 8.9e-7 and 1.38e-6 (84 super-blocks in one chain, the longest that the estimate makes)."""
    host = N.synth_weights(N.Q4_K, 0x65, rows, cols)
    w = torch.from_numpy(np.ascontiguousarray(N.retile(host, N.Q4_K, cols, rows, N.ROW_MAJOR, N.CDNA4))).cuda()
    x = torch.from_numpy(N.synth_normal_f16(0x66, batch * cols).reshape(batch, cols).view(np.int16)).cuda()
    dense = torch.empty((rows, cols), dtype=torch.float32, device="cuda")
    ctx.dequant(w, N.Q4_K, N.CDNA4, cols, rows, 0, rows, out_f32=dense)
    want = x.view(torch.float16).double() @ dense.double().t().contiguous()
    y = torch.full((batch, rows), float("nan"), dtype=torch.float32, device="cuda")
    tune("gemm_kparts", kparts)
    ctx.matmul(w, N.Q4_K, N.CDNA4, cols, rows, batch, x, y, half_input=True)
    assert float((y.double() - want).norm() / want.norm()) <= 0.9 * was
