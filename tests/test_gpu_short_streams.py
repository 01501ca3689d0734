"""Parity of the per-row int8 decode kernel where its waves change path: ranges of one and two batches (K and V
requested at once) and just beyond them (the ring), lengths around those edges, every operand dtype at the
least alignment it may have (one element past an aligned base), and head and row counts that are no powers of
two. Bar as the other attention tests: max abs <= 2e-3, max rel <= 1e-2."""
from __future__ import annotations

import pytest
import torch

from helpers import SEED, assert_close
from test_gpu_attention import Case

pytestmark = pytest.mark.gpu


def shifted(t: torch.Tensor) -> torch.Tensor:
    """The same values one element past an aligned base."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_edges_of_the_stream_paths(device, D, dtype):
    tpl = 1024 // D  # tokens per load tile; a batch is four tiles
    batch = 4 * tpl
    lengths = [0, 1, batch - 1, batch, batch + 1, 2 * batch - 1, 2 * batch, 2 * batch + 1, 3 * batch + tpl,
               7 * batch - 3, 8 * batch + 5]
    c = Case(device, len(lengths), 3, D, lengths, 8 * batch + 5, q_dtype=dtype, scratch_dtype=dtype, seed=SEED + D)
    c.q, c.sk, c.sv = shifted(c.q), shifted(c.sk), shifted(c.sv)
    ref, ref16 = c.reference(), c.reference(history_bf16=True)
    for split in (tpl, batch - tpl, batch, batch + tpl, 2 * batch, 2 * batch + tpl, 4 * batch, 0):
        print(f"D={D} {dtype} split={split}", flush=True)
        assert_close(c.run(split), ref, what=f"D={D} split={split}")
        assert_close(c.run(split, bf16_history=True), ref16, what=f"D={D} split={split} bf16 history")
