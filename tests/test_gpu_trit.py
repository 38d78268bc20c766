"""The trit kernel (small batches of fp16, bf16 and fp32 activations) against the fp64 oracle, and
the SwiGLU epilogues of the MFMA kernels against the linear they follow.

Shapes sit where it can go wrong: row counts that are no multiple of a wave's
32 or a workgroup's 128 rows, group counts below, at and past its windows (1,
5, 9 and 17 groups unsplit, 40 split), batches on both sides of its 8-, 16-, 32-
and 64-row tiles, several tiles in a launch and in several launches. Products of an activation with
-1, 0 or +1 are exact (fp32 as three bf16 terms), so an output is held to the
fp32 summation bound plus one rounding to its type.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import tq1_oracle as O
from tests.gpu_util import layout, pack, random_blocks, to_dev
from ternel_amd import _lib, synthetic
from ternel_amd.kernels import (GemmConfig, linear_kernel, pack_weights, tq1_gemm_words, tq1_linear_words,
                                tq1_matmul_words, tq1_swiglu_words)

pytestmark = pytest.mark.gpu

ROUNDOFF = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def activations(batch: int, columns: int, dtype: torch.dtype, seed: int) -> torch.Tensor:
    rng = np.random.default_rng(seed)
    x = rng.normal(0.0, 1.0, size=(batch, columns))
    if dtype != torch.float16:
        x *= 10.0 ** rng.integers(-6, 7, size=columns)  # far past fp16's range
    return to_dev(x.astype(np.float32)).to(dtype)


def bound(x: np.ndarray, blocks: np.ndarray, want: np.ndarray, dtype: torch.dtype) -> np.ndarray:
    rows, groups, _ = blocks.shape
    weights = O.dense_weights(blocks, rows=rows, columns=groups * 128)
    sums = (128 + groups) * float(np.finfo(np.float32).eps) * (np.abs(x) @ np.abs(weights).T)
    return sums + ROUNDOFF[dtype] * (np.abs(want) + sums) + 2.0 ** -25 * (dtype == torch.float16)


SHAPES = ((130, 128), (300, 640), (257, 1152), (96, 2176), (1024, 5120))
CASES = [(dtype, rows, columns, batch) for dtype in (torch.float16, torch.bfloat16)
         for rows, columns in SHAPES for batch in (5, 8, 9, 17, 32, 33, 64)]
# tiles of 64 rows and the remainder of a batch past them, split and unsplit
CASES += [(dtype, rows, columns, batch) for dtype in (torch.float16, torch.bfloat16)
          for rows, columns, batch in ((257, 1152, 65), (1024, 5120, 130), (300, 640, 203), (4100, 1024, 193))]
# fp32: matrices large enough for the trit kernel at each tile width, and (LUT23) small ones
CASES += [(torch.float32, 5121, 4608, 8), (torch.float32, 2562, 4608, 15), (torch.float32, 300, 640, 77),
          (torch.float32, 257, 1152, 130), (torch.float32, 130, 128, 65)]


@pytest.mark.parametrize(("dtype", "rows", "columns", "batch"), CASES)
def test_small_batches_match_the_oracle(dtype, rows, columns, batch) -> None:
    print(f"trit: {dtype} rows={rows} columns={columns} batch={batch}", flush=True)
    blocks = random_blocks(rows, columns, seed=rows + columns + batch)
    packed, lay = pack(blocks), layout(rows, columns)
    x = activations(batch, columns, dtype, seed=batch)
    got = tq1_linear_words(packed, x, layout=lay)
    assert torch.equal(got, tq1_linear_words(packed, x, layout=lay))  # the same bits twice
    x64 = x.double().cpu().numpy()
    want = O.oracle_matmul(blocks, x64, rows=rows, columns=columns)
    assert (np.abs(got.double().cpu().numpy() - want) <= bound(x64, blocks, want, dtype)).all()


# the trit kernel's tiles, then the wide form's (fp16 takes it from 64 tiles of
# 256 rows on); an output width that no 16-byte store divides, and one it does
SWIGLU = [(dtype, 1030, 1152, batch) for dtype in (torch.float16, torch.bfloat16) for batch in (2, 7, 30, 64)]
SWIGLU += [(torch.bfloat16, 1030, 1152, 70), (torch.bfloat16, 1030, 1152, 800), (torch.bfloat16, 1024, 1152, 800),
           (torch.bfloat16, 60006, 1024, 70), (torch.float16, 60000, 1024, 70), (torch.float16, 16390, 256, 800)]


@pytest.mark.parametrize(("dtype", "rows", "columns", "batch"), SWIGLU)
def test_the_fused_swiglu_is_the_linear_and_the_elementwise_step(dtype, rows, columns, batch) -> None:
    packed, lay = pack(random_blocks(rows, columns, seed=batch)), layout(rows, columns)
    x = to_dev(np.random.default_rng(batch).normal(0.0, 0.3, size=(batch, columns)).astype(np.float32)).to(dtype)
    both = tq1_linear_words(packed, x, layout=lay).float()
    gate, up = both[:, 0::2], both[:, 1::2]
    want = (gate / (1.0 + torch.exp(-gate)) * up).to(dtype).float()
    diff = (tq1_swiglu_words(packed, x, layout=lay).float() - want).abs()
    # expf against torch's exp, then one rounding: at most a step of the type
    assert bool((diff <= want.abs() * 2 * ROUNDOFF[dtype] + 2.0 ** -24).all())


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16, torch.float32))
def test_non_finite_values_follow_the_entry_point(dtype) -> None:
    """The GEMM path computes (t - 1) * scale (a zero trit of a non-finite scale
    is NaN), the matmul path scale * sum as the LUT23 kernel does."""
    rows, columns, batch = 640, 640, 80 if dtype == torch.float32 else 6
    blocks = random_blocks(rows, columns, seed=3)
    bits = {5: 0x7C00, 70: 0xFC00, 300: 0x7E00}  # +inf, -inf, NaN in a row's second group
    for row, value in bits.items():
        blocks[row, 1, 0:2] = np.frombuffer(np.uint16(value).tobytes(), dtype=np.uint8)
    packed, lay = pack(blocks), layout(rows, columns)
    x = to_dev(np.random.default_rng(4).normal(0.0, 1.0, size=(batch, columns)).astype(np.float32)).to(dtype)
    x[1, 7], x[2, 639] = float("inf"), float("nan")
    x64 = x.double().cpu().numpy()
    with np.errstate(invalid="ignore"):
        products = O.oracle_matmul(blocks, x64, rows=rows, columns=columns)
        tables = O.lut23_matmul(blocks, x64.astype(np.float32), rows=rows, columns=columns)
    if dtype != torch.float32:
        got = tq1_linear_words(packed, x, layout=lay).float().cpu().numpy()
        assert O.compare(got, products)["pattern_mismatches"] == 0
    got = tq1_matmul_words(packed, x, layout=lay).float().cpu().numpy()
    assert O.compare(got, tables)["pattern_mismatches"] == 0


def test_a_swiglu_reduction_that_gives_up_writes_nan() -> None:
    """The wide form's bounded wait driven to give up from the host: every
    output is the fused value or NaN, some are NaN, and the error word is set."""
    rows, columns, batch = 1030, 5120, 800
    packed, lay = pack(random_blocks(rows, columns, seed=5)), layout(rows, columns)
    x = to_dev(np.random.default_rng(5).normal(0.0, 0.3, size=(batch, columns)).astype(np.float32)).to(torch.bfloat16)
    want = tq1_swiglu_words(packed, x, layout=lay)
    handle = _lib.lib()
    need = handle.ternel_tq1_swiglu_workspace_bytes(batch, rows, columns, _lib.DTYPE_BF16)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    out = torch.zeros((batch, rows // 2), dtype=torch.bfloat16, device="cuda")
    old = handle.ternel_tq1_set_spin_limit(-1)
    try:
        _lib.check(handle.ternel_tq1_swiglu(packed.data_ptr(), x.data_ptr(), out.data_ptr(), batch, rows, columns,
                                            _lib.DTYPE_BF16, ws.data_ptr(), need, 0))
        torch.cuda.synchronize()
    finally:
        handle.ternel_tq1_set_spin_limit(old)
    word = ctypes.c_int(0)
    _lib.check(handle.ternel_tq1_workspace_error(ws.data_ptr(), need, ctypes.byref(word), 0))
    nan = torch.isnan(out)
    assert word.value == 2 and bool(nan.any())
    assert torch.equal(out[~nan], want[~nan])


def test_a_row_of_more_than_2_gib_of_packed_words() -> None:
    """One K chunk whose last groups lie past 2^31 bytes of the tile's words:
    blocks of scale 0 but for two at the far end, trits all -1, so an output is
    minus those groups' activations, times their scales, exactly."""
    rows, groups = 64, 2 ** 31 // 1792 + 11
    columns = groups * 128
    packed = torch.zeros((1, groups, 7, 64), dtype=torch.int32, device="cuda")
    packed[0, groups - 1, 0, :] = 0x3C00  # word 0: the scale (1.0) and code bytes 0 and 1
    packed[0, groups - 9, 0, :] = 0x4000  # 2.0
    x = torch.zeros((2, columns), dtype=torch.float16, device="cuda")
    x[0, (groups - 1) * 128:] = 1.0
    x[1, (groups - 9) * 128:(groups - 8) * 128] = 0.5
    got = tq1_gemm_words(packed, x, layout=layout(rows, columns), config=GemmConfig(form="direct", k_split=1))
    want = torch.tensor([[-128.0], [-128.0]], dtype=torch.float16, device="cuda").expand(2, rows)
    assert torch.equal(got, want)


# group counts that no chunk of 4 or 8 divides: K chunks with a shorter last one, of one group (5,
# 9, 37, 73), two (74) and three (67), at each tile width, over batch tiles and through the fused SwiGLU
ODD_GROUPS = [(dtype, rows, groups, batch) for rows, groups in ((1024, 37), (1030, 67), (300, 5), (386, 74))
              for dtype, batches in ((torch.float16, (2, 3, 8, 16, 32, 64, 130)), (torch.bfloat16, (3, 8, 32, 50)),
                                     (torch.float32, (40, 70))) for batch in batches]
ODD_GROUPS += [(torch.float32, 4096, 67, 9), (torch.float32, 4096, 37, 24), (torch.float32, 2560, 73, 16)]


@pytest.mark.parametrize(("dtype", "rows", "groups", "batch"), ODD_GROUPS)
def test_group_counts_without_divisors_match_the_oracle(dtype, rows, groups, batch) -> None:
    print(f"trit: {dtype} rows={rows} groups={groups} batch={batch}", flush=True)
    columns = groups * 128
    blocks = random_blocks(rows, columns, seed=rows + groups + batch)
    packed, lay = pack(blocks), layout(rows, columns)
    x = activations(batch, columns, dtype, seed=batch)
    got = tq1_linear_words(packed, x, layout=lay)
    assert torch.equal(got, tq1_linear_words(packed, x, layout=lay))
    sample = np.unique(np.r_[0:64, rows - 70:rows, np.random.default_rng(batch).integers(0, rows, 200)])
    x64 = x.double().cpu().numpy()
    want = O.oracle_matmul(blocks[sample], x64, rows=len(sample), columns=columns)
    assert (np.abs(got.double().cpu().numpy()[:, sample] - want) <= bound(x64, blocks[sample], want, dtype)).all()
    z = tq1_swiglu_words(packed, x[:, :].mul(0.01), layout=lay).float()
    both = tq1_linear_words(packed, x[:, :].mul(0.01), layout=lay).float()
    gate, up = both[:, 0::2], both[:, 1::2]
    silu = (gate / (1.0 + torch.exp(-gate)) * up).to(dtype).float()
    finite = torch.isfinite(silu)
    assert bool(((z - silu).abs() <= silu.abs() * 4 * ROUNDOFF[dtype] + 2.0 ** -24)[finite].all())


# fp32 activations down to the last bits of the subnormals and up to near the largest value (group sums
# of random signs stay finite): the three bf16 terms hold every finite value exactly, so the bound is
# the summation one, with the spacing of the subnormals once per rounding
@pytest.mark.parametrize("exponent", (-148, -140, -130, -126, -120, -110, -60, 110))
@pytest.mark.parametrize(("rows", "columns", "batch"), ((8192, 1152, 7), (4100, 4608, 16), (4100, 4608, 24)))
def test_fp32_values_of_any_magnitude_match_the_oracle(rows, columns, batch, exponent) -> None:
    print(f"trit: fp32 rows={rows} columns={columns} batch={batch} 2^{exponent}", flush=True)
    lay = layout(rows, columns)
    assert linear_kernel(lay, batch, torch.float32) == "trit"
    blocks = random_blocks(rows, columns, seed=rows + batch)
    rng = np.random.default_rng(1000 + batch - exponent)
    x = to_dev((rng.normal(0.0, 1.0, size=(batch, columns)) * 2.0 ** exponent).astype(np.float32))
    got = tq1_linear_words(pack(blocks), x, layout=lay)
    sample = np.unique(np.r_[0:64, rows - 70:rows, rng.integers(0, rows, 200)])
    x64 = x.double().cpu().numpy()
    want = O.oracle_matmul(blocks[sample], x64, rows=len(sample), columns=columns)
    weights = O.dense_weights(blocks[sample], rows=len(sample), columns=columns)
    sums = (128 + columns // 128) * 2.0 ** -23 * (np.abs(x64) @ np.abs(weights).T) + (columns // 64) * 2.0 ** -149
    assert (np.abs(got.double().cpu().numpy()[:, sample] - want) <= sums).all()


@pytest.mark.parametrize("batch", (64, 63))
def test_a_batch_of_several_launches(batch) -> None:
    """fp32 on down's shape: 17 K chunks whose partials leave room for one batch
    tile of 32 rows within the matmul path's limit, so two launches share the
    counters, the second one short; linear and SwiGLU."""
    rows, columns = 5120, 17408
    lay = layout(rows, columns)
    assert linear_kernel(lay, batch, torch.float32) == "trit"
    # one tile's partials, rather than two: 17 chunks of 40 row blocks x 4 waves x 4 quads
    need = _lib.lib().ternel_tq1_matmul_workspace_bytes(batch, rows, columns, 0, 0)
    tile = 17 * 40 * 4 * 4 * 1024
    assert tile <= (16 << 20) < 2 * tile and need >= 65536 + tile
    blocks = synthetic.device_blocks(rows, columns, seed=synthetic.SEED_BASE + 5)
    packed = pack_weights(blocks, layout=lay)
    x = synthetic.device_activations(batch, columns, seed=batch).to(torch.float32) * 0.05
    got = tq1_linear_words(packed, x, layout=lay)
    assert torch.equal(got, tq1_linear_words(packed, x, layout=lay))
    sample = np.sort(np.random.default_rng(batch).choice(rows // 2, size=64, replace=False))
    pairs = np.stack([2 * sample, 2 * sample + 1], axis=1).reshape(-1)
    sampled = blocks[torch.from_numpy(pairs).cuda()].cpu().numpy()
    x64 = x.double().cpu().numpy()
    want = O.oracle_matmul(sampled, x64, rows=len(pairs), columns=columns)
    assert (np.abs(got.double().cpu().numpy()[:, pairs] - want) <= bound(x64, sampled, want, torch.float32)).all()
    gate, up = got[:, 0::2], got[:, 1::2]
    silu = gate / (1.0 + torch.exp(-gate)) * up
    diff = (tq1_swiglu_words(packed, x, layout=lay) - silu).abs()
    assert bool((diff <= silu.abs() * 4 * ROUNDOFF[torch.float32] + 2.0 ** -126).all())


def test_fp32_non_finite_values_follow_the_lut23_oracle() -> None:
    """As above for fp32, on a matrix large enough for the trit kernel, at 16
    and 24 rows a tile."""
    rows, columns = 4096, 1152
    for batch in (16, 72):
        lay = layout(rows, columns)
        assert linear_kernel(lay, batch, torch.float32) == "trit"
        blocks = random_blocks(rows, columns, seed=3)
        for row, value in {5: 0x7C00, 70: 0xFC00, 300: 0x7E00, rows - 1: 0x7C00}.items():
            blocks[row, 1, 0:2] = np.frombuffer(np.uint16(value).tobytes(), dtype=np.uint8)
        x = to_dev(np.random.default_rng(4).normal(0.0, 1.0, size=(batch, columns)).astype(np.float32))
        x[1, 7], x[2, 639], x[batch - 1, 1151] = float("inf"), float("nan"), -float("inf")
        sample = np.r_[0:96, 280:320, rows - 40:rows]
        tables = O.lut23_matmul(blocks[sample], x.cpu().numpy(), rows=len(sample), columns=columns)
        got = tq1_linear_words(pack(blocks), x, layout=lay).cpu().numpy()[:, sample]
        assert O.compare(got, tables)["pattern_mismatches"] == 0
