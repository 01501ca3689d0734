"""Parity of the per-row int8 decode kernel for every way its waves take a row's batches (in turn by one or by
two, or one contiguous range per wave; chosen by the wave's share and the grid) at shares around the rule's
edges, with row lengths at and next to whole batches, pairs and turns. Shares of 1 to 12 batches run over a span of
40 batches: up to four batches that is several blocks per row, above it one. Turns of two over several blocks,
shares around 32 batches and the long contiguous ranges of a full grid have their own shapes. Bar as the other
attention tests: max abs <= 2e-3, max rel <= 1e-2."""
from __future__ import annotations

import math

import pytest
import torch

import ppk
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


# (head_dim, sequences, heads, batches per share, waves per row, blocks per row)
LONG = [
    (64, 12, 2, 6, 20, 3),     # turns of two over three blocks, the row's last pair cut short
    (128, 12, 2, 8, 17, 3),
    (256, 12, 2, 12, 24, 3),
    (64, 10, 2, 31, 3, 1),     # pairs within 1/16 of the share
    (64, 10, 2, 32, 3, 1),     # from 32 batches on: turns of one
    (128, 10, 2, 33, 5, 1),
    (128, 16, 16, 16, 8, 1),   # one eight-wave block on every CU: pairs up to 16 batches,
    (128, 16, 16, 17, 8, 1),   # contiguous ranges above
    (256, 15, 16, 19, 8, 1),
    (128, 7, 16, 18, 16, 2),   # 224 blocks: just too few for that rule
]


@pytest.mark.parametrize("D,B,H,share,waves,blocks", LONG)
def test_long_shares(device, D, B, H, share, waves, blocks):
    batch = 4096 // D
    split = share * batch
    span = waves * split - batch // 2
    edges = [0, 1, batch, 2 * batch * waves, 2 * batch * waves + 1, 3 * batch * waves - 1, split - 1, split, split + 1,
             span - 2 * batch, span - 1]
    lens = [span] + [min(edges[i % len(edges)], span) for i in range(B - 1)]
    rows, cap = B * H, span + 1
    g = torch.Generator(device=device).manual_seed(SEED + D + share)
    codes = [torch.randint(-127, 128, (rows, cap, D), generator=g, device=device, dtype=torch.int8) for _ in range(2)]
    scales = [torch.rand((rows, cap), generator=g, device=device) * 0.02 + 0.005 for _ in range(2)]
    q, sk, sv = (torch.randn((rows, 1, D), generator=g, device=device) for _ in range(3))
    past = torch.tensor(lens, dtype=torch.int32, device=device)
    args, _ = ppk.int8_kv_ops.attention_args(q, codes[0].view(torch.uint8), codes[1].view(torch.uint8), *scales, sk, sv,
                                             past, H, split, max_past=span)
    info = ppk.int8_kv_ops.plan_info(args, ppk.context(device))
    assert (info["split_tokens"], info["nsplits"]) == (split, blocks)
    got = ppk.attention(q, codes[0].view(torch.uint8), codes[1].view(torch.uint8), *scales, sk, sv, past, H, split,
                        max_past=span)
    torch.cuda.synchronize()
    for b, n in enumerate(lens):
        r = slice(b * H, (b + 1) * H)
        k, v = (torch.cat([c[r, :n].double() * s[r, :n, None].double(), t[r].double()], 1)
                for c, s, t in ((codes[0], scales[0], sk), (codes[1], scales[1], sv)))
        p = torch.softmax((k * q[r].double()).sum(-1) / math.sqrt(D), -1)
        want = (p[..., None] * v).sum(1)
        assert_close(got[r].reshape(H, D).cpu().numpy(), want.cpu().numpy(), what=f"D={D} share={share} length {n}")
