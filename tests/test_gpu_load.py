"""The load pass (permutation into the packed words with the byte scan folded in)
against the index formula and the separate scan, at the edges of its 64-row x
8-group tiles."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.gpu_util import layout, random_blocks, to_dev
from ternel_amd.format import FormatError, count_invalid_bytes
from ternel_amd.kernels import pack_weights, packed_shape, unpack_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", (1, 63, 64, 65, 520))
@pytest.mark.parametrize("groups", (1, 7, 8, 9, 40))
def test_a_checked_load_is_the_permutation_and_the_scan(rows: int, groups: int) -> None:
    blocks = random_blocks(rows, groups * 128, seed=rows + groups)
    lay = layout(rows, groups * 128)
    packed = pack_weights(to_dev(blocks), layout=lay, validate=True)
    words = np.zeros(packed_shape(lay), dtype=np.uint32)
    source = blocks.reshape(rows, groups, 28).view(np.uint32).reshape(rows, groups, 7)
    for r in range(rows):
        words[r // 64, :, :, r % 64] = source[r]
    np.testing.assert_array_equal(packed.cpu().numpy().view(np.uint32), words)
    assert torch.equal(packed, pack_weights(to_dev(blocks), layout=lay))
    np.testing.assert_array_equal(unpack_weights(packed, layout=lay).cpu().numpy(), blocks)

    rng = np.random.default_rng(rows * groups)
    bad = blocks.copy()
    bad[..., 2:] = rng.integers(0, 256, size=bad[..., 2:].shape, dtype=np.uint8)
    bad[rows - 1, groups - 1, 27], bad[0, 0, 2] = 27, 243  # the last tail and the first code byte at least
    regular, tail = int((bad[..., 2:27] > 242).sum()), int((bad[..., 27] > 26).sum())
    assert count_invalid_bytes(to_dev(bad)) == (regular, tail)
    with pytest.raises(FormatError, match=rf"regular={regular} \(max 242\), tail={tail} \(max 26\)"):
        pack_weights(to_dev(bad), layout=lay, validate=True)
