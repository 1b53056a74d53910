"""Squareplus of every conv output through the conv kernel (taps of zero, the
bias as the output): all values within the input clamp and past it, and the
ends of int32, against the integer root."""

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_squareplus_every_value(cuda):
    import torch
    from mamba_int import ops
    c = np.arange(-60000, 60001, dtype=np.int64)
    c = np.concatenate([c, [-2**31, 2**31 - 1, -2**31 + 1]])
    v = np.clip(c, -51200, 51200)
    root = np.array([math.isqrt(int(x) * int(x) + (1 << 22)) for x in v])
    ref = np.clip((v + root + 64) >> 7, -127, 127).astype(np.int8)
    for shift in (0, 1, 2, 3):      # every value in every byte of the packed result
        cb = np.roll(c, shift)
        d = len(cb) // 4 * 4
        z = torch.zeros((1, 1, d), dtype=torch.int8, device="cuda")
        y = ops.conv_squareplus(z, d, torch.zeros((d, 4), dtype=torch.int8, device="cuda"),
                                torch.from_numpy(cb[:d].astype(np.int32)).cuda())
        assert np.array_equal(y.cpu().numpy().reshape(-1), np.roll(ref, shift)[:d])
