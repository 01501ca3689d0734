"""Parity of the per-row int8 decode kernel with and without early batches: with the lengths on the device only,
every wave requests its first batches before its row's length arrives; with ragged host lengths, where too many of
those would lie past their row's history, it waits for the length and requests what the row has. Waves end with
0, 1, 2, 3 or more batches on either way, in one block and in several blocks per row. Both give the same bits (the
order of the sums is the plan's, not the requests'). Bar as the other attention tests: max abs <= 2e-3, max rel
<= 1e-2."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import SEED, assert_close
from test_gpu_attention import Case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16_history", [False, True])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_with_and_without_early_batches(device, D, bf16_history):
    batch = 4096 // D  # four load tiles of 1024 / D tokens
    for waves in (1, 3, 8, 19):  # 19: several blocks per row
        for share in (1, 2, 3, 4):
            span = waves * share * batch
            edges = {0, 1, batch, batch + 1, waves * batch, waves * batch + 1, 2 * waves * batch - 1,
                     2 * waves * batch + 1, 3 * waves * batch + batch // 2}
            lengths = [span] + sorted(x for x in edges if x < span)
            c = Case(device, len(lengths), 2, D, lengths, span + 1, q_dtype=torch.bfloat16,
                     scratch_dtype=torch.bfloat16, seed=SEED + D + waves)
            print(f"D={D} waves={waves} share={share}", flush=True)
            kw = dict(max_past=span, bf16_history=bf16_history)
            early, late = c.run(share * batch, **kw), c.run(share * batch, past_host=lengths, **kw)
            assert_close(early, c.reference(history_bf16=bf16_history), what=f"D={D} {waves} waves of {share} batches")
            np.testing.assert_array_equal(early, late)
