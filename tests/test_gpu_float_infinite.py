"""Infinite values in a float KV store reach the output as the plain softmax has them: the channel that holds one
is infinite, every other channel finite. The value lies in the share of the row's last wave (and not in its
last token), for blocks of one to twelve waves and for rows of several blocks: the combines of a block's and of a
row's records may not give the records that are not there a say."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import ppk
from helpers import SEED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("waves,blocks", [(1, 1), (2, 1), (3, 1), (5, 1), (7, 1), (8, 1), (9, 1), (12, 1), (18, 2), (39, 3),
                                          (144, 9), (272, 17)])
@pytest.mark.parametrize("D", [64, 256])
def test_infinite_value_in_the_last_wave(device, kv, waves, blocks, D):
    share, rows, heads = 32, 4, 2  # 32 tokens: whole batches at every width, so no token is read twice
    n = waves * share
    rng = np.random.default_rng(SEED + waves + D)
    k = torch.from_numpy(rng.standard_normal((rows, n, D), dtype=np.float32)).to(device).to(kv)
    v = torch.from_numpy(rng.standard_normal((rows, n, D), dtype=np.float32)).to(device).to(kv)
    q = torch.from_numpy(rng.standard_normal((rows, 1, D), dtype=np.float32)).to(device)
    at = n - share + 3
    v[0, at, 5] = float("inf")
    v[1, at, D - 1] = float("-inf")
    lengths = torch.full((rows // heads,), n, dtype=torch.int32, device=device)
    args, _ = ppk.fused_attention.decode_attention_args(q, k, v, lengths, heads, share)
    info = ppk.fused_attention.plan_info(args, ppk.context(device))
    assert (info["nsplits"], info["waves_per_block"]) == (blocks, waves // blocks)
    out = ppk.fused_attention.decode_attention(q, k, v, lengths, heads, share)
    torch.cuda.synchronize()
    got = out.reshape(rows, D).double().cpu().numpy()
    kk, vv, qq = k.double().cpu(), v.double().cpu(), q.double().cpu()
    p = torch.softmax((kk * qq).sum(-1) / np.sqrt(D), -1)
    want = (p[..., None] * vv).sum(1).numpy()
    assert np.isposinf(want[0, 5]) and np.isneginf(want[1, D - 1])
    np.testing.assert_allclose(got, want, rtol=1e-2, atol=1e-4)
