"""The 128- and 256-token tile GEMMs at the batches that the few-token GEMM takes by default: the
prefill tests of the other modules once more, on a context that never selects it (gemm_skinny 0)."""
import pytest

import nsffn as N

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
from test_gpu_shape_sweep import test_gate_up_sweep, test_prefill_sweep  # noqa: E402,F401


@pytest.fixture(scope="module")
def ctx():
    assert torch.cuda.is_available(), "GPU tests need a visible MI355X"
    c = N.Context(0)
    c.set_tuning("gemm_skinny", 0)
    yield c
    torch.cuda.synchronize()
    c.close()
