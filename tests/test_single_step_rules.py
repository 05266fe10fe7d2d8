"""The host rules of the single-step kernels (csrc/rln_single.h), on the CPU.

tests/sanitize/rln_rules.hip compiles the rules with the host sanitizers and
answers queries about them; nothing reaches a device.
"""

import os
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent / "sanitize"
HIDDEN = range(128, 8193, 64)


@pytest.fixture(scope="module")
def ask():
    """ask(queries): one list of integers per query line."""
    if not Path("/opt/rocm/bin/hipcc").exists():
        pytest.skip("no hipcc")
    build = subprocess.run(["make", "-s", "-C", str(HERE), "rln_rules"], capture_output=True,
                           text=True, timeout=600)
    assert build.returncode == 0, build.stdout + build.stderr
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")

    def run(queries):
        lines = [" ".join(str(int(v)) if not isinstance(v, str) else v for v in query)
                 for query in queries]
        result = subprocess.run([str(HERE / "rln_rules")], input="\n".join(lines) + "\n",
                                capture_output=True, text=True, timeout=300, env=env)
        assert result.returncode == 0, result.stderr
        answers = [[int(v) for v in line.split()] for line in result.stdout.splitlines()]
        assert len(answers) == len(lines)
        return answers

    return run


def test_row_sums_stay_inside_their_lds_array(ask):
    """Every row of every split reads its sums from inside the block's array
    (rows of 1025-1216 columns share a block of four waves, two rows of two)."""
    queries = [("lds", pass_, rows, hidden) for pass_ in (0, 1) for hidden in HIDDEN
               for rows in (1, 5, 2048, 8192, 8193, 12291, 65536)]
    for query, (size, end) in zip(queries, ask(queries)):
        assert end <= size, query


F32, F16, BF16 = 0, 1, 2
GRAD_UPDATED, GRAD_NORMALIZED, DROPOUT, PARAMETERS, PARTIALS = 1, 2, 4, 8, 16
EVERYTHING = GRAD_UPDATED | GRAD_NORMALIZED | DROPOUT | PARAMETERS


def test_row_counts_whose_bytes_overflow(ask):
    """The C ABI accepts every rows * hidden that fits int64; the choice of the
    backward's kernel must not overflow on the bytes of such tensors."""
    queries = [("backward", (2**63 - 1) // hidden, hidden, F32, F32, flags, over, 1)
               for hidden in (128, 768, 8192) for over in range(5)
               for flags in (EVERYTHING, EVERYTHING | PARTIALS)]
    assert ask(queries) == [[0]] * len(queries)


@pytest.mark.parametrize("hidden", [128, 768, 2880])
def test_gradients_over_inputs_walk(ask, hidden):
    """Gradients in the memory of what the slab blocks read take the walking
    kernels; without weight/bias sums there are no slab blocks."""
    for over in range(5):
        answers = ask([("backward", 100, hidden, F16, F32, EVERYTHING, over, 1),
                       ("backward", 100, hidden, F16, F32, EVERYTHING & ~PARAMETERS, over, 1)])
        assert answers == [[int(over == 0)], [1]]


# (rows, hidden, branch, grad_normalized, flags, single-step?) on both sides of
# lines beside which rln_single.h gives both sides' times.
NONE = EVERYTHING & ~PARAMETERS
NO_GRAD_NORMALIZED = NONE & ~GRAD_NORMALIZED
MISALIGNED = [
    (5792, 128, F16, F32, EVERYTHING, 1), (11585, 128, F32, F32, EVERYTHING, 0),
    (5461, 768, F32, F32, EVERYTHING, 1), (6553, 640, BF16, BF16, EVERYTHING, 1),
    (772, 960, F16, F32, EVERYTHING, 1), (4369, 960, F32, F32, EVERYTHING, 0),
    (252, 4160, F16, F32, EVERYTHING, 1), (712, 4160, F16, F32, EVERYTHING, 0),
    (682, 6144, F32, F32, EVERYTHING, 0), (337, 6208, F32, F32, EVERYTHING, 1),
    (675, 6208, F32, F32, EVERYTHING, 0),
    (204, 1280, F16, F32, NONE, 1), (579, 1280, F16, F32, NONE, 0),
    (21, 3072, F16, F32, NONE, 0), (482, 3072, F16, F32, NONE, 0),
]


def test_misaligned_backward_lines(ask):
    """Element accesses take the walking backward where it is the faster one."""
    assert ask([("backward", *case[:5], 0, 0) for case in MISALIGNED]) \
        == [[case[5]] for case in MISALIGNED]


def test_misaligned_forward_lines(ask):
    """Element accesses: single-step for small launches of up to 4096 columns,
    write-through below 2^23 elements at every row length."""
    cases = [(341, 768, 1, 1, 1), (1365, 768, 1, 0, 1), (512, 1024, 1, 1, 1), (64, 4096, 1, 1, 1),
             (257, 2880, 1, 0, 1), (1927, 1088, 1, 0, 1),
             (12, 5120, 0, 0, 1), (64, 8192, 1, 0, 1), (7414, 1600, 1, 0, 0),
             (10485, 1600, 1, 0, 0), (65536, 256, 1, 0, 0), (5242, 1600, 1, 0, 1)]
    assert ask([("forward", *case[:3], 0) for case in cases]) == [list(case[3:]) for case in cases]


def test_deterministic_route_ignores_alignment(ask):
    """Deterministic weight/bias sums are the same bits for tensors of any
    alignment: the kernel that groups them is chosen without it."""
    queries = [("backward", rows, hidden, F16, F32, EVERYTHING | PARTIALS, 0)
               for hidden in HIDDEN for rows in (1, 60, 300, 1000, 3000, 9000, 20000)]
    assert ask([(*q, 0) for q in queries]) == ask([(*q, 1) for q in queries])


WITHOUT_SUMS = [
    (241, 3072, F16, F32, NONE, 1), (482, 3072, F16, F32, NONE, 0), (512, 4096, F32, F32, NONE, 0),
    (682, 6144, BF16, BF16, NONE, 0), (682, 6144, BF16, BF16, EVERYTHING, 1),
    (42, 3072, F16, F32, NO_GRAD_NORMALIZED, 0), (42, 3072, F16, F32, NONE, 1),
    (241, 3072, F16, F32, NO_GRAD_NORMALIZED, 1), (85, 6144, F16, F32, NO_GRAD_NORMALIZED, 1),
    (512, 2048, F16, F32, NONE, 1), (579, 1280, F16, F32, NONE, 0), (655, 1600, F16, F32, NONE, 0),
    (724, 2048, F32, F32, NONE, 0), (724, 2048, F32, F32, EVERYTHING, 1),
    (926, 1600, F16, F32, NONE, 1), (1170, 1792, F32, F32, NONE, 0),
    (431, 2432, F16, F32, NONE, 1), (862, 2432, F16, F32, NONE, 0),
    (4096, 128, F16, F32, NO_GRAD_NORMALIZED, 0), (4096, 128, F16, F32, NONE, 1),
    (5792, 128, F16, F32, NO_GRAD_NORMALIZED, 1),
    (362, 8192, F16, F32, NONE, 1), (512, 8192, F32, F32, NONE, 0), (512, 8192, F32, F32, EVERYTHING, 1),
    (1170, 7168, F16, F32, NONE, 1),
]


def test_backward_lines_without_sums(ask):
    """Frozen parameters, or no grad_normalized: the walking backward where its
    grid is full in its first or second row step."""
    assert ask([("backward", *case[:5], 0, 1) for case in WITHOUT_SUMS]) \
        == [[case[5]] for case in WITHOUT_SUMS]


DETERMINISTIC = [
    (2896, 128, 1), (4096, 128, 0), (1365, 192, 1), (1930, 192, 0), (1448, 256, 1), (5792, 256, 0),
    (2730, 768, 1), (5461, 768, 0), (3276, 640, 1), (13107, 640, 0), (2048, 1024, 1), (8192, 1024, 0),
    (1310, 1600, 1), (3707, 1600, 0), (965, 3072, 1), (1655, 3584, 0), (819, 5120, 1), (1638, 5120, 0),
    (827, 7168, 1), (2702, 6208, 0),
]


def test_deterministic_backward_lines(ask):
    """Fixed-order sums: the walking backward past the lines of their own."""
    assert ask([("backward", rows, hidden, F16, F32, EVERYTHING | PARTIALS, 0, 1)
                for rows, hidden, _ in DETERMINISTIC]) == [[case[2]] for case in DETERMINISTIC]


def test_lines_of_32_bit_tensors_and_long_rows(ask):
    """A 32-bit branch and gradient pass over to the walk earlier, and so do rows of
    3073-4095 columns."""
    cases = [(2621, 1600, F32, F32, EVERYTHING, 1), (3707, 1600, F32, F32, EVERYTHING, 0),
             (3707, 1600, F16, F32, EVERYTHING, 1), (3707, 1600, F32, F32, NONE, 0),
             (827, 3584, F32, F32, EVERYTHING, 1), (1170, 3584, F32, F32, EVERYTHING, 0),
             (1655, 3584, F16, F32, EVERYTHING, 0), (512, 8192, F16, F32, NONE, 1),
             (1448, 8192, F16, F32, NONE, 0)]
    assert ask([("backward", *case[:5], 0, 1) for case in cases]) == [[case[5]] for case in cases]


def test_forward_lines(ask):
    """Aligned forwards: (rows, hidden, dropout) single-step and write-through."""
    cases = [(4096, 128, 0, 1, 1), (5792, 128, 0, 0, 1), (5792, 128, 1, 1, 1), (5792, 256, 0, 1, 1),
             (5405, 6208, 1, 0, 1), (5792, 8192, 1, 0, 0), (9362, 7168, 1, 0, 0),
             (8192, 8192, 0, 0, 1), (8193, 8192, 0, 0, 0), (16384, 4096, 1, 0, 1)]
    assert ask([("forward", *case[:3], 1) for case in cases]) == [list(case[3:]) for case in cases]


def test_768_columns_with_32_bit_gradients_walk_from_7168_rows(ask):
    """One line, whatever shape the walk has above it; 16-bit gradients, launches
    without sums and the neighbouring row lengths keep theirs."""
    rows = (6912, 7167, 7168, 7679, 7680, 8192, 9216, 9217, 16384)
    for branch in (F16, F32):
        assert ask([("backward", r, 768, branch, F32, EVERYTHING, 0, 1) for r in rows]) \
            == [[int(r < 7168)] for r in rows]
    for hidden, grad_normalized, flags in ((768, BF16, EVERYTHING), (768, F32, NONE),
                                           (704, F32, EVERYTHING), (832, F32, EVERYTHING)):
        assert ask([("backward", r, hidden, F16, grad_normalized, flags, 0, 1) for r in rows]) \
            == [[int(r * hidden <= 12 << 20)] for r in rows]


def test_launches_named_after_walking_shapes_walk(ask):
    """The GPU tests of the walking backward's shapes and schedules run in place or
    deterministic: both take the walk at their sizes."""
    import test_gpu_launch_shapes as shapes
    import test_gpu_schedules as schedules

    in_place = [(768, rows) for rows, _ in shapes.TWELVE_WAVE_CASES]
    in_place += [(384, rows) for rows, _ in shapes.NINE_WAVE_CASES]
    in_place += [(hidden, rows) for hidden, rows, _ in shapes.STAGGERED_WIDE_CASES]
    in_place += schedules.RING_CASES
    deterministic = [(hidden, rows) for hidden, rows, _ in shapes.STAGGERED_SHAPES]
    queries = [("backward", rows, hidden, F16, F32, flags, 2, 1) for hidden, rows in in_place
               for flags in (EVERYTHING, EVERYTHING | PARTIALS)]
    queries += [("backward", rows, hidden, F16, F32, EVERYTHING | PARTIALS, 0, aligned)
                for hidden, rows in deterministic for aligned in (0, 1)]
    assert ask(queries) == [[0]] * len(queries)


def test_bench_names_the_kernel_the_rules_choose(ask):
    """bench.py's roofline names the kernel a workload launches; its copy of the
    rules agrees with the library's over sizes, dtypes and modes."""
    import random
    from dataclasses import replace

    from test_bench_cli import _bench_module

    bench = _bench_module()
    code = {"f32": F32, "f16": F16, "bf16": BF16}
    rng = random.Random(19)
    workloads = [bench.C1, *bench.sweep_workloads()]
    for hidden in HIDDEN:
        for _ in range(24):
            rows = max(1, round(2 ** rng.uniform(14, 25) / hidden))
            workloads.append(replace(
                bench.C1, rows=rows, hidden=hidden, branch=rng.choice(list(code)),
                normalized=rng.choice(list(code)), dropout_p=rng.choice([0.0, 0.1]),
                deterministic=rng.random() < 0.3, training=rng.random() < 0.8))
    queries = []
    for w in workloads:
        flags = GRAD_UPDATED | GRAD_NORMALIZED | PARAMETERS | (PARTIALS if w.deterministic else 0)
        queries.append(("forward", w.rows, w.hidden, w.dropping, 1))
        queries.append(("backward", w.rows, w.hidden, code[w.branch], code[w.normalized], flags, 0, 1))
    answers = ask(queries)
    for w, forward, backward in zip(workloads, answers[::2], answers[1::2]):
        named = [("single" in bench.launched_kernel(f"rln_{pass_}_kernel", w))
                 for pass_ in ("forward", "backward")]
        assert named == [bool(forward[0]), bool(backward[0])], w
