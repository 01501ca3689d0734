"""Parity of the per-row int8 decode kernel for every way its waves take a row's batches (in turn by one or by
two, or one contiguous range per wave; chosen by the wave's share) at shares around the rule's edges, with row
lengths at and next to whole batches, pairs and turns, in one block and in several blocks per row. Bar as the
other attention tests: max abs <= 2e-3, max rel <= 1e-2."""
from __future__ import annotations

import pytest
import torch

from helpers import SEED, assert_close
from test_gpu_attention import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
def test_shares_around_the_rule(device, D):
    tpl = 1024 // D
    batch = 4 * tpl
    span = 40 * batch + tpl
    lengths = [0, 1, batch, 2 * batch + 1, 6 * batch - 1, 12 * batch, 13 * batch + 1, 16 * batch, 17 * batch - 1,
               32 * batch + 3, span - 1, span]
    c = Case(device, len(lengths), 2, D, lengths, span, q_dtype=torch.bfloat16, scratch_dtype=torch.bfloat16,
             seed=SEED + 7 * D)
    ref, ref16 = c.reference(), c.reference(history_bf16=True)
    # Shares of 1 to 12 batches: whole, a tile short, a tile over.
    for split in sorted({max(tpl, k * batch + e * tpl) for k in (1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 12) for e in (-1, 0, 1)}):
        print(f"D={D} split={split}", flush=True)
        assert_close(c.run(split), ref, what=f"D={D} split={split}")
        if split % batch == 0:
            assert_close(c.run(split, bf16_history=True), ref16, what=f"D={D} split={split} bf16 history")
