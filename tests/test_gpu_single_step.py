"""Single-step launches (csrc/rln_single.h) at the edges of their splits.

One row per team of waves: rows that fill their last wave by a part of a lane
row, idle waves and lanes, teams past the last row, and both sides of the rule
that hands larger launches to the walking kernels. Every output element is
checked against the oracle (parity.check_full_tensor: mask and `updated`
bitwise, the rest against float64 at the parity bar).
"""

import pytest
import torch

from gfx1010_kernels import _C
from parity import check_full_tensor, generator_state
from test_gpu_configs import check_parameter_gradients, device_inputs

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _run(rows, hidden, branch_dtype, normalized_dtype, dropout_p):
    print(f"[single step] rows={rows} H={hidden} {branch_dtype} {normalized_dtype} "
          f"p={dropout_p}", flush=True)
    inputs, grads = device_inputs(rows, hidden, branch_dtype, seed=3 * hidden + rows)
    grads = (grads[0], grads[1].to(normalized_dtype))
    torch.cuda.manual_seed(hidden + rows)
    seed, offset = generator_state()
    outputs = _C.residual_layer_norm_forward(*inputs, dropout_p, EPS, True, 128,
                                             normalized_dtype=normalized_dtype)
    gradients = _C.residual_layer_norm_backward(
        grads[0], grads[1], outputs[0], inputs[2], outputs[2], outputs[3], outputs[4], dropout_p,
        True, branch_dtype == torch.float16, 128, 64, 64, 1, True, branch_dtype)
    reference_stream = hidden in (128, 256, 384, 512, 768, 1024)
    check_full_tensor(inputs, grads, outputs, gradients, dropout_p, EPS, seed, offset,
                      threads=128 if reference_stream else 0, what=f"{rows} x {hidden}")
    check_parameter_gradients(outputs[0], grads[1], gradients)


# One, two, three, four and more waves per row, one to three slots per lane,
# whole and ragged; rows that leave teams of a block without one.
@pytest.mark.parametrize("rows", [1, 3, 5, 130])
@pytest.mark.parametrize("hidden", [128, 192, 256, 320, 512, 576, 768, 832, 1024, 1088, 1536, 1600,
                                    2048, 2112, 3072, 3136, 4096, 4160, 6144, 6208, 8192])
def test_small_rows(rows, hidden):
    branch, normalized = [(torch.float16, torch.float32), (torch.bfloat16, torch.bfloat16),
                          (torch.float32, torch.float16)][(hidden // 64 + rows) % 3]
    _run(rows, hidden, branch, normalized, 0.1)


# The forward's last single-step row count and the first walked one.
@pytest.mark.parametrize("hidden,rows,dropout_p", [
    (128, 6144, 0.1), (256, 6144, 0.2), (384, (1 << 21) // 384, 0.1), (768, (1 << 21) // 768, 0.1),
    (1280, (1 << 21) // 1280, 0.1), (1344, (1 << 20) // 1344, 0.1), (4096, 256, 0.0),
    (4160, (1 << 20) // 4160, 0.1), (4160, (1 << 17) // 4160, 0.0), (8192, 16, 0.0)])
@pytest.mark.parametrize("above", [0, 1])
def test_forward_switch(hidden, rows, dropout_p, above):
    _run(rows + above, hidden, torch.float16, torch.float32, dropout_p)
