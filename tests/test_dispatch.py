"""The dispatch rule replayed against a measured MI355X sweep, as the reference
replays its Metal sweeps through select_gemm (tests/test_mlx_modules.py:553,
1007). tests/golden/dispatch_sweep_mi355x.json holds the time of every kernel
the library can run for each (27B linear shape, batch), measured by
tests/golden/sweep_dispatch.py; the rule must pick one within 15 % of the
fastest everywhere."""

from __future__ import annotations

import json

import pytest
import torch

from tests.conftest import GOLDEN
from ternel_amd import _lib
from ternel_amd.kernels import linear_kernel
from ternel_amd.layout import PackedTensorLayout
from ternel_amd.modules import select_kernel

SWEEP = json.loads((GOLDEN / "dispatch_sweep_mi355x.json").read_text())
NAMES = {100: "lut23", 1: "tile", 2: "direct", 3: "wide"}


@pytest.mark.parametrize("row", SWEEP["rows"], ids=lambda r: f"{r['shape']}-M{r['M']}")
def test_the_rule_picks_a_kernel_within_15_percent_of_the_fastest(row) -> None:
    code = _lib.lib().ternel_tq1_linear_kernel(row["M"], row["N"], row["K"], _lib.DTYPE_F16)
    chosen = NAMES[code]
    times = row["us"]
    assert chosen in times, f"the rule picked {chosen}, which the sweep did not time"
    assert times[chosen] <= 1.15 * min(times.values()), (chosen, times)


def test_the_module_dispatch_follows_the_library() -> None:
    for row in SWEEP["rows"]:
        layout = PackedTensorLayout.for_tensor(row["N"], row["K"])
        code = _lib.lib().ternel_tq1_linear_kernel(row["M"], row["N"], row["K"], _lib.DTYPE_F16)
        assert select_kernel(layout, row["M"], torch.float16) == ("lut23" if code == 100 else "gemm")


def test_fp32_activations_take_the_lut_kernel_and_bf16_the_wide_form() -> None:
    handle = _lib.lib()
    for M in (1, 3, 8, 64, 512, 2048):
        assert handle.ternel_tq1_linear_kernel(M, 17408, 5120, _lib.DTYPE_F32) == 100
        # bf16: the LUT23 kernel where fp16 takes it, the wide form (3) above
        fp16 = handle.ternel_tq1_linear_kernel(M, 17408, 5120, _lib.DTYPE_F16)
        assert handle.ternel_tq1_linear_kernel(M, 17408, 5120, _lib.DTYPE_BF16) == (100 if fp16 == 100 else 3)


def test_the_sweep_covers_every_regime() -> None:
    chosen = {NAMES[_lib.lib().ternel_tq1_linear_kernel(r["M"], r["N"], r["K"], _lib.DTYPE_F16)] for r in SWEEP["rows"]}
    assert chosen == {"lut23", "direct", "wide", "tile"}


def direct_split(M: int, rows: int, groups: int) -> int:
    """K chunks of the direct form, from the partials its workspace holds (a
    quad of sums per lane of four waves, per 8 activation rows and 128 rows)."""
    need = _lib.lib().ternel_tq1_gemm_workspace_bytes(M, rows, groups * 128, 2, 0)
    quads = 8 if M > 32 else -(-M // 8)
    return max(1, (need - 65536) // (-(-rows // 128) * 4 * quads * 1024)) if need else 1


@pytest.mark.parametrize("M", (8, 16, 32, 64))
@pytest.mark.parametrize("rows", (256, 1024, 4096, 17408))
def test_every_group_count_splits_over_the_chip(M, rows) -> None:
    """Prime and almost prime group counts as well: about a workgroup per CU (at
    64 rows, half of that, where a split would cost more), or chunks of at most
    12 groups."""
    blocks = -(-rows // 128)
    for groups in range(1, 141):
        k = direct_split(M, rows, groups)
        assert 1 <= k <= groups
        assert blocks * k >= (192 if M <= 32 else 128) or -(-groups // k) <= 12, (groups, k)


def test_the_27b_widths_split_into_equal_chunks() -> None:
    for M, rows, groups, k in ((8, 17408, 40, 5), (8, 8192, 40, 5), (8, 5120, 136, 17), (8, 5120, 48, 6),
                               (8, 34816, 40, 5), (32, 8192, 40, 10), (32, 5120, 48, 6), (8, 1024, 40, 10),
                               (8, 4096, 32, 8)):
        assert direct_split(M, rows, groups) == k, (M, rows, groups)


def test_what_the_matmul_path_refuses_it_refuses_for_every_kernel() -> None:
    """More K chunks than a LUT23 launch takes, in a batch that the trit kernel
    would run: refused before any launch, with and without a workspace."""
    handle = _lib.lib()
    columns = (65536 * 4 + 1) * 128
    aligned = 1 << 20  # never read: the call is refused first
    for M in (4, 8, 64):
        assert handle.ternel_tq1_matmul_workspace_bytes(M, 256, columns, 0, 0) == 0
        for rc in (handle.ternel_tq1_matmul(aligned, aligned, aligned, M, 512, columns, _lib.DTYPE_F16, 0, 0, None, 0, None),
                   handle.ternel_tq1_matmul_noalloc(aligned, aligned, aligned, M, 512, columns, _lib.DTYPE_F16, 0, 0,
                                                    None)):
            assert rc == _lib.TERNEL_TQ1_EINVAL
            assert "K too large for one launch" in _lib.last_error()
        assert handle.ternel_tq1_swiglu(aligned, aligned, aligned, M, 512, columns, _lib.DTYPE_F32, None, 0,
                                        None) == _lib.TERNEL_TQ1_EINVAL
        assert "K too large for one launch" in _lib.last_error()


def test_the_reported_kernel_is_one_the_path_can_launch() -> None:
    handle = _lib.lib()
    seen = set()
    for dtype, code in ((torch.float16, _lib.DTYPE_F16), (torch.bfloat16, _lib.DTYPE_BF16), (torch.float32, _lib.DTYPE_F32)):
        for rows, columns in ((48, 5120), (1024, 5120), (4096, 4096), (5120, 17408), (8192, 5120), (17408, 5120)):
            layout = PackedTensorLayout.for_tensor(rows, columns)
            for M in (1, 2, 3, 4, 6, 8, 24, 33, 64, 100, 128, 400, 600, 2048):
                name = linear_kernel(layout, M, dtype)
                seen.add(name)
                path = handle.ternel_tq1_linear_kernel(M, rows, columns, code)
                if path == 100:
                    assert name in ("lut23", "strip", "trit")
                    assert name != "strip" or M == 1
                elif path == 2:
                    assert name == "trit"
                else:
                    assert name in ("trit", NAMES[path])
                # the workspace that the launch needs tells the trit kernel's split from the wide form's
                if name == "wide":
                    assert handle.ternel_tq1_linear_workspace_bytes(M, rows, columns, code) > 65536
    assert seen == {"lut23", "strip", "trit", "wide", "tile"}
    assert handle.ternel_tq1_linear_launches(0, 64, 128, 0) == _lib.TERNEL_TQ1_EINVAL


# Both sides of the lines between the LUT23 and the trit kernel (and, fp16 above 64 rows, the tile
# form) as measured on an MI355X: the kernel that was the faster one, or within 5 % of it.
LINES = [
    # fp16 and bf16 batches of the matmul path: 2 rows, then 3 and 4
    (torch.float16, 17408, 5120, 2, "trit"), (torch.float16, 17408, 10752, 2, "lut23"),
    (torch.float16, 8192, 5120, 2, "lut23"), (torch.float16, 5120, 6144, 2, "lut23"),
    (torch.bfloat16, 1024, 5120, 2, "trit"), (torch.bfloat16, 512, 10752, 2, "lut23"),
    (torch.float16, 256, 10752, 3, "lut23"), (torch.float16, 320, 5120, 3, "trit"),
    (torch.bfloat16, 160, 7168, 4, "lut23"), (torch.float16, 48, 5120, 4, "lut23"),
    # fp32: too few rows or groups, then enough, at each tile width; odd group counts
    (torch.float32, 17408, 5120, 4, "lut23"), (torch.float32, 17408, 5120, 6, "trit"),
    (torch.float32, 4096, 5120, 6, "lut23"), (torch.float32, 8192, 5120, 9, "trit"),
    (torch.float32, 2048, 3072, 16, "lut23"), (torch.float32, 4096, 5120, 16, "trit"),
    (torch.float32, 949, 5120, 24, "lut23"), (torch.float32, 8192, 5120, 24, "trit"),
    (torch.float32, 219, 1152, 61, "lut23"), (torch.float32, 512, 8192, 48, "lut23"),
    (torch.float32, 2048, 8192, 48, "trit"), (torch.float32, 1024, 1664, 64, "lut23"),
    (torch.float32, 2048, 4736, 4, "trit"), (torch.float32, 2048, 5120, 4, "lut23"),
    (torch.float32, 64, 4736, 9, "trit"), (torch.float32, 64, 4736, 4, "lut23"),
    (torch.float32, 136, 2688, 47, "lut23"), (torch.float32, 2862, 1408, 35, "lut23"),
    (torch.float16, 1447, 10368, 2, "trit"), (torch.bfloat16, 145, 5248, 4, "trit"),
    # fp16 above the direct form: short rows under 64 KiB keep the tile form
    (torch.float16, 57, 1152, 90, "tile"), (torch.float16, 54, 3584, 375, "trit"), (torch.float16, 1024, 5120, 128, "trit"),
    (torch.bfloat16, 57, 1152, 90, "trit"),
]


@pytest.mark.parametrize(("dtype", "rows", "columns", "batch", "kernel"), LINES)
def test_each_side_of_a_line_runs_its_faster_kernel(dtype, rows, columns, batch, kernel) -> None:
    assert linear_kernel(PackedTensorLayout.for_tensor(rows, columns), batch, dtype) == kernel


def test_a_form_asked_for_by_name_is_the_one_that_runs() -> None:
    """bf16, a shape the trit kernel runs unsplit and so without a workspace: the
    wide form always needs one, and is refused for the lack of it."""
    handle = _lib.lib()
    rows, columns = 256, 128
    assert linear_kernel(PackedTensorLayout.for_tensor(rows, columns), 8, torch.bfloat16) == "trit"
    aligned = 1 << 20  # never read
    rc = handle.ternel_tq1_gemm(aligned, aligned, aligned, 8, rows, columns, _lib.DTYPE_BF16, 3, 0, None, 0, None)
    assert rc == _lib.TERNEL_TQ1_EINVAL
    assert "workspace of 0 bytes" in _lib.last_error()


def test_a_given_split_moves_no_batch_to_the_direct_form() -> None:
    """AUTO with a k_split at 49-64 rows on a small matrix: one K chunk runs the
    wide form (whose workspace holds more than partials), several the tile
    form; without one the direct form, up to 48 rows in any case."""
    size = _lib.lib().ternel_tq1_gemm_workspace_bytes
    rows, columns = 4096, 4096
    for M in (49, 56, 64):
        assert size(M, rows, columns, 0, 0) == size(M, rows, columns, 2, 0)
        assert size(M, rows, columns, 0, 1) == size(M, rows, columns, 3, 1)
        assert size(M, rows, columns, 0, 4) == size(M, rows, columns, 1, 4)
    for k_split in (0, 1, 4):
        assert size(48, rows, columns, 0, k_split) == size(48, rows, columns, 2, k_split)


KERNEL_SWEEP = json.loads((GOLDEN / "kernel_sweep_mi355x.json").read_text())
# Where another kernel was more than 15 % faster: the tile form splits K only by divisors of the group
# count (67 and 74 here), as does the LUT23 kernel's automatic choice in chunks of 1 or 2 groups.
SLOWER = {(4096, 8576, 100), (4096, 8576, 203), (4096, 8576, 384), (2048, 9472, 203), (2048, 9472, 384), (2048, 9472, 768),
          (1024, 16768, 1), (2048, 9472, 2)}


@pytest.mark.parametrize("row", KERNEL_SWEEP["rows"], ids=lambda r: f"{r['N']}x{r['K']}-{r['dtype']}-M{r['M']}")
def test_the_dispatch_runs_the_kernel_of_the_sweep(row) -> None:
    """The kernel that was timed is the one that runs, within 15 % of any other."""
    layout = PackedTensorLayout.for_tensor(row["N"], row["K"])
    assert linear_kernel(layout, row["M"], getattr(torch, row["dtype"])) == row["runs"]
    others = [us for name, us in row["us"].items() if name != "dispatch"]
    if (row["N"], row["K"], row["M"]) not in SLOWER or row["dtype"] != "float16":
        assert row["us"]["dispatch"] <= 1.15 * min(others, default=row["us"]["dispatch"]), row["us"]


def test_the_kernel_sweep_covers_every_kernel_of_every_type() -> None:
    runs = {(row["dtype"], row["runs"]) for row in KERNEL_SWEEP["rows"]}
    assert runs == {(t, k) for t in ("float16", "bfloat16") for k in ("strip", "lut23", "trit", "wide")} | \
        {("float16", "tile")} | {("float32", k) for k in ("strip", "lut23", "trit")}


@pytest.mark.parametrize("name", ("ternel_tq1_linear_workspace_bytes", "ternel_tq1_swiglu_workspace_bytes"))
def test_a_bf16_workspace_for_the_largest_batch_holds_the_smaller_ones(name) -> None:
    size = getattr(_lib.lib(), name)
    for rows, columns in ((34816, 5120), (8192, 5120), (5120, 6144), (4096, 4096), (1024, 5120), (300, 1152)):
        for largest in (512, 768, 2048):
            need = size(largest, rows, columns, _lib.DTYPE_BF16)
            assert max(size(M, rows, columns, _lib.DTYPE_BF16) for M in range(33, largest)) <= need, (rows, columns)
