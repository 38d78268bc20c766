"""Sweep of the present kernels on an MI355X: for each (shape, activation type,
batch) the time of what the library's dispatch runs, by name, and of every other
kernel that can be asked for, timed as sweep_dispatch.py times (cold weight
ring, launches replayed from one HIP graph). Shapes are the 27B linears', and
small, odd and short-rowed ones. Writes the fixture that tests/test_dispatch.py
replays through ``kernels.linear_kernel``.

    python tests/golden/sweep_kernels.py OUT.json     # on a GPU box
"""

from __future__ import annotations

import json
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[2]))

from tests.golden.sweep_dispatch import graph_us  # noqa: E402
from ternel_amd import synthetic  # noqa: E402
from ternel_amd.kernels import (GemmConfig, MatmulConfig, linear_kernel, pack_weights, tq1_gemm_words,  # noqa: E402
                                tq1_linear_words, tq1_matmul_words)
from ternel_amd.layout import PackedTensorLayout  # noqa: E402

SHAPES = ((17408, 5120), (34816, 5120), (5120, 17408), (8192, 5120), (5120, 6144), (4096, 4096), (1024, 5120), (48, 5120),
          (4096, 8576), (1024, 16768), (2048, 9472), (300, 1152))
BATCHES = (1, 2, 3, 4, 6, 8, 16, 24, 32, 48, 64, 100, 203, 384, 768)
RING_BYTES = 400 << 20
F16, BF16, F32 = torch.float16, torch.bfloat16, torch.float32


def alternatives(dtype, M: int) -> dict:
    forms = {}
    if M <= (64 if dtype == F32 else 16):
        forms["lut23"] = lambda w, x, lay: tq1_matmul_words(w, x, layout=lay, config=MatmulConfig(batch_tile=1))
    for form in {F16: ("direct", "wide", "tile"), BF16: ("wide",), F32: ()}[dtype]:
        if M <= 64 or form != "direct":
            forms[form] = lambda w, x, lay, form=form: tq1_gemm_words(w, x, layout=lay, config=GemmConfig(form=form))
    return forms


def main(out: str) -> None:
    rows = []
    for N, K in SHAPES:
        lay = PackedTensorLayout.for_tensor(N, K)
        ring = max(2, min(256, RING_BYTES // lay.payload_bytes))
        first = pack_weights(synthetic.device_blocks(N, K, seed=1), layout=lay)
        weights = [first] + [first.clone() for _ in range(ring - 1)]
        for dtype in (F16, BF16, F32):
            for M in BATCHES:
                if dtype == F32 and M > 64:
                    continue
                x = synthetic.device_activations(M, K, seed=M).to(dtype)
                launches = max(4, min(2 * ring, 4096 // M))
                kernels = {"dispatch": lambda w, x, lay: tq1_linear_words(w, x, layout=lay), **alternatives(dtype, M)}
                times = {name: round(min(graph_us(lambda i, fn=fn: fn(weights[i % ring], x, lay), launches)
                                         for _ in range(2)), 2) for name, fn in kernels.items()}
                rows.append({"N": N, "K": K, "dtype": str(dtype).split(".")[1], "M": M,
                             "runs": linear_kernel(lay, M, dtype), "us": times})
        print(json.dumps(rows[-1]), flush=True)
        del weights
    Path(out).write_text(json.dumps({
        "device": torch.cuda.get_device_name(0),
        "method": "cold weight ring, launches replayed from one HIP graph, events around it, the better of two",
        "rows": rows,
    }, indent=0) + "\n")


if __name__ == "__main__":
    main(sys.argv[1])
