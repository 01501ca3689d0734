"""The streaming append's chunks: 256 16-byte units of one tensor per wave.

A chunk that lies in one arena row, within capacity, stores through one scalar
base; a chunk that crosses to the next row, holds the tensor's last rows, or
reaches the capacity indexes per lane. Codes, scales, flags and every slot that
is not written are compared with the oracle bit for bit. Inputs hold values
next to half-integer quotients, infinities and NaNs of every payload (a NaN of
all ones must not be taken for a finite quotient).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
import ppk
from helpers import SEED, bf16_bits_to_f32, to_bf16_bits

pytestmark = pytest.mark.gpu


def source(rng, shape, dt, device):
    x = rng.standard_normal(shape).astype(np.float32)
    flat = x.reshape(-1, shape[-1])
    # Quotients at and next to half-integers: the row's scale is near 1.
    n = len(flat[::3])
    flat[::3] = rng.integers(-127, 127, (n, shape[-1])) + np.float32(0.5)
    flat[::3] += rng.integers(-6, 7, (n, shape[-1])).astype(np.float32) * np.float32(2.0**-15)
    flat[::3, 0] = 127.0
    special = np.array([0x7FFFFFFF, 0xFFFFFFFF, 0x7F800001, 0x7FC00000, 0x7F800000, 0xFF800000], np.uint32)
    for i, bits in enumerate(special):
        flat[(7 + 101 * i) % len(flat)].view(np.uint32)[(5 + 11 * i) % shape[-1]] = bits
    flat[len(flat) - 1].view(np.uint32)[-1] = 0x7FFFFFFF
    if dt == "f32":
        return torch.from_numpy(x).to(device), x
    if dt == "f16":
        h = x.astype(np.float16)
        return torch.from_numpy(h).to(device), h.astype(np.float32)
    nan = np.isnan(x)
    bits = to_bf16_bits(np.where(nan, np.float32(0), x))
    bits[nan] = 0x7FFF
    return torch.from_numpy(bits.view(np.int16)).to(device).view(torch.bfloat16), bf16_bits_to_f32(bits)


# (batch, heads, tokens): around the 4 to 32 rows of a chunk, and totals that
# leave the tensor's last chunk ragged; 2 * rows stays at or above 12288.
@pytest.mark.parametrize("b,h,t", [(48, 128, 1), (31, 29, 7), (27, 29, 15), (24, 16, 16), (23, 17, 17), (13, 16, 31),
                                   (12, 16, 33), (3, 16, 131), (1, 3, 2049)])
@pytest.mark.parametrize("d,dt", [(64, "bf16"), (64, "f32"), (128, "bf16"), (128, "f16"), (256, "f32")])
def test_append_chunks_match_oracle(device, b, h, t, d, dt):
    rng = np.random.default_rng(SEED + b * 7 + t + d)
    rows, cap = b * h, t + 9
    past = rng.integers(0, 10, b).astype(np.uint32)
    past[b // 2] = min(cap - 1, t // 2 + 10)  # this sequence's last tokens lie past the capacity
    (k, k32), (v, v32) = (source(rng, (b, h, t, d), dt, device) for _ in range(2))
    kc, vc = (torch.full((rows, cap, d), 77, dtype=torch.uint8, device=device) for _ in range(2))
    ks, vs = (torch.full((rows, cap), 3.0, dtype=torch.float32, device=device) for _ in range(2))
    flags = torch.zeros(1, dtype=torch.int32, device=device)
    ppk.append(k, v, torch.from_numpy(past.view(np.int32)).to(device), kc, vc, ks, vs, flags)
    torch.cuda.synchronize()
    fits = (past[:, None].astype(np.int64) + np.arange(t)) < cap  # [b, t]
    for x32, codes, scales in ((k32, kc, ks), (v32, vc, vs)):
        rc, rs, _ = oracle.quantize(x32.reshape(rows, t, d))
        want_c = np.full((rows, cap, d), 77, np.uint8)
        want_s = np.full((rows, cap), 3.0, np.float32)
        for r in range(rows):
            n, p = int(fits[r // h].sum()), int(past[r // h])
            want_c[r, p:p + n] = np.asarray(rc[r, :n]).view(np.uint8)
            want_s[r, p:p + n] = rs[r, :n]
        assert np.array_equal(codes.cpu().numpy(), want_c)
        assert np.array_equal(scales.cpu().numpy().view(np.uint32), want_s.view(np.uint32))
    assert int(flags.item()) == 1 | (0 if fits.all() else 2)
