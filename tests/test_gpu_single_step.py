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


# The backward's last single-step row count and the first walked one.
@pytest.mark.parametrize("hidden,rows", [(128, (1 << 22) // 128), (256, (1 << 23) // 256),
                                         (768, (12 << 20) // 768), (1088, (6 << 20) // 1088),
                                         (4096, (1 << 23) // 4096), (6208, (1 << 24) // 6208),
                                         # the staggered walking backward among them
                                         (768, 7679), (768, 7680), (768, 9216)])
@pytest.mark.parametrize("above", [0, 1])
def test_backward_switch(hidden, rows, above):
    _run(rows + above, hidden, torch.float16, torch.bfloat16, 0.1)


def _row_outputs(rows, hidden, inputs, grads, branch_dtype, dropout_p, deterministic=False):
    """Forward and backward over the first `rows` rows, without weight/bias sums."""
    from test_gpu_schedules import run

    out = run((inputs[0], inputs[1], inputs[2], inputs[3], *grads), rows, torch.float32,
              dropout_p, deterministic)
    return {name: out[name] for name in ("updated", "normalized", "mean", "rstd", "mask", "grad_x",
                                         "grad_branch")}, out["parameters"]


@pytest.mark.parametrize("hidden", [128, 192, 256, 320, 384, 512, 576, 768, 832, 1024, 1088, 1600,
                                    2048, 2112, 2880, 4096, 4160, 7168, 8192])
@pytest.mark.parametrize("dropout_p", [0.0, 0.1])
def test_single_step_rows_equal_walked_rows(hidden, dropout_p):
    """A row's outputs are the same bits from the single-step kernels (a few
    rows) and from the walking ones (enough rows to be above both rules; rows
    of 768 and 6657-8192 columns stay below the sizes that change the walking
    backward's own sums)."""
    many = (1 << 24) // hidden + 3
    inputs, grads = device_inputs(many, hidden, torch.bfloat16, seed=hidden)
    print(f"[single step] rows {many} against 77 H={hidden} p={dropout_p}", flush=True)
    walked, _ = _row_outputs(many, hidden, inputs, grads, torch.bfloat16, dropout_p)
    single, _ = _row_outputs(77, hidden, inputs, grads, torch.bfloat16, dropout_p)
    for name, value in single.items():
        if name == "mask":
            count = value.numel() if dropout_p else 0
            assert torch.equal(value[:count], walked[name][:count])
        else:
            integer = {4: torch.int32, 2: torch.int16}[value.element_size()]
            assert torch.equal(value.view(integer), walked[name][:77].view(integer)), name


@pytest.mark.parametrize("rows,hidden", [(3, 384), (300, 192), (4096, 128), (4097, 128),
                                         (9000, 256), (16384, 512), (16385, 512), (500, 2880),
                                         (33, 8192), (3072, 128), (3073, 128), (3072, 256),
                                         (3073, 256), (4096, 512), (4097, 512), (3072, 1024),
                                         (3073, 1024), (1365, 3072), (1366, 3072), (1228, 5120),
                                         (1229, 5120), (1536, 8192), (1537, 8192)])
def test_deterministic_partials(rows, hidden):
    """Fixed-order weight/bias sums of single-step launches: chunks of few and
    many rows, and the row counts that hand over to the walking backward. Bit
    for bit the same twice, at the parity bar against float64."""
    from test_gpu_schedules import check_parameter_sums, run

    print(f"[single step] deterministic rows={rows} H={hidden}", flush=True)
    inputs, grads = device_inputs(rows, hidden, torch.float16, seed=rows + hidden)
    case = (*inputs, *grads)
    first = run(case, rows, torch.float32, 0.1, True)
    second = run(case, rows, torch.float32, 0.1, True)
    assert torch.equal(first["parameters"], second["parameters"])
    check_parameter_sums(first, grads[1], rows)


@pytest.mark.parametrize("over", ["grad_normalized", "updated"])
@pytest.mark.parametrize("rows,hidden", [(100, 768), (40, 2880), (2047, 768), (4097, 768),
                                         (6145, 768), (12291, 384), (4096, 832), (4096, 1024)])
def test_gradients_written_over_their_inputs(rows, hidden, over):
    """grad_x in the memory of grad_normalized or `updated`: the same results
    as in memory of its own."""
    from gfx1010_kernels import _cabi

    inputs, grads = device_inputs(rows, hidden, torch.float32, seed=rows)
    updated, _, mean, rstd, mask = _C.residual_layer_norm_forward(*inputs, 0.1, EPS, True, 128)
    print(f"[single step] grad_x over {over} rows={rows} H={hidden}", flush=True)
    results = []
    for in_place in (False, True):
        saved = dict(grad_normalized=grads[1].clone(), updated=updated.clone())
        grad_x = saved[over] if in_place else torch.empty_like(updated)
        grad_branch = torch.empty_like(updated)
        sums = torch.zeros(2, hidden, device="cuda")
        _cabi.backward(
            grads[0].data_ptr(), saved["grad_normalized"].data_ptr(), saved["updated"].data_ptr(),
            inputs[2].data_ptr(), mean.data_ptr(), rstd.data_ptr(), mask.data_ptr(),
            grad_x.data_ptr(), grad_branch.data_ptr(), _cabi.RLN_DTYPE_F32, sums[0].data_ptr(),
            sums[1].data_ptr(), rows, hidden, 0.1, True, False, None, 0,
            torch.cuda.current_stream().cuda_stream, accumulate_parameters=True)
        torch.cuda.synchronize()
        results.append((grad_x, grad_branch, sums))
    assert torch.equal(results[0][0], results[1][0])
    assert torch.equal(results[0][1], results[1][1])
    separate, shared = results[0][2], results[1][2]
    if rows <= 100:
        # Two fp32 orders of sums over at most 100 values of order one.
        assert torch.allclose(separate, shared, rtol=1e-5, atol=1e-4)
    # Sums of n values of order one in two fp32 orders of at most 300 additions per
    # term (rows of a wave or chunk, then blocks): 2^-24 * sqrt(300) = 1e-6 of the
    # sums' norm, ten times that allowed.
    assert ((separate - shared).norm(dim=1) <= 1e-5 * separate.norm(dim=1)).all()


@pytest.mark.parametrize("rows,hidden", [(341, 768), (512, 1024), (64, 4096), (257, 2880), (5792, 128),
                                         (11585, 128), (772, 960), (4369, 960), (252, 4160),
                                         (712, 4160), (337, 6208), (675, 6208)])
def test_misaligned_launches_match_aligned_ones(rows, hidden):
    """Both sides of the lines from which element accesses walk: row outputs are
    the aligned launch's bits, weight/bias sums at the parity bar."""
    from test_gpu_schedules import ROW_OUTPUTS, assert_same_bits, check_parameter_sums, empty, run

    print(f"[single step] misaligned rows={rows} H={hidden}", flush=True)
    inputs, grads = device_inputs(rows, hidden, torch.bfloat16, seed=rows + hidden)
    aligned_case = (*inputs, *grads)
    shifted_case = tuple(empty(t.shape, t.dtype, shift=1).copy_(t) for t in aligned_case)
    aligned = run(aligned_case, rows, torch.float32, 0.1, False)
    shifted = run(shifted_case, rows, torch.float32, 0.1, False, shift=1)
    for name in (*ROW_OUTPUTS, "mask"):
        assert_same_bits(shifted[name], aligned[name], name)
    check_parameter_sums(shifted, grads[1], rows)
