"""The SSD block scan over rows so far apart that a chunk's rows span more than
2^32 bytes (strides of z and of the x_proj rows), against the CPU oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

WIDE = 143_000_000 // 16 * 16     # 32 rows: 4.6e9 bytes


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("wide", ["z", "xp"])
def test_ssd_block_scan_wide_rows(cuda, rng, wide):
    import torch
    from mamba_int import ops
    b, length, heads, p, n = 1, 33, 2, 16, 64
    d, w = heads * p, 2 * heads * n + 16
    xs = rng.integers(-127, 128, size=(b, length, d), dtype=np.int8)
    z = rng.integers(-127, 128, size=(b, length, 2 * d), dtype=np.int8)
    xp = rng.integers(-127, 128, size=(b, length, w), dtype=np.int8)
    tab = rng.integers(24576, 2**15 + 1, size=(heads, 255), dtype=np.int32)
    ref, h_ref = O.ssd_v2_scan(xs, xp, z, d, tab, 12, heads, n)
    far = torch.zeros((b, length, WIDE), dtype=torch.int8, device="cuda")
    src = T(z if wide == "z" else xp)
    far[..., :src.shape[-1]] = src
    zt, xt = (far, T(xp)) if wide == "z" else (T(z), far)
    h = torch.empty((b, d, n), dtype=torch.int32, device="cuda")
    yo = ops.ssd_block_scan(T(xs), xt, zt, d, T(tab), heads, n, 12, h_out=h)
    assert np.array_equal(yo.cpu().numpy(), ref)
    assert np.array_equal(h.cpu().numpy().reshape(h_ref.shape), h_ref)
