"""Short sequences of many blocks, which take the scans with y on the VALU or
16-step chunks, against the CPU oracle bit for bit: the state handed on, every
state count (test_gpu_scan_routes.py has the bounds of the dispatch)."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def i8(rng, *shape):
    return rng.integers(-128, 128, size=shape, dtype=np.int8)


def state(rng, *shape):
    h = rng.integers(-2**31, 2**31, size=shape, dtype=np.int64).astype(np.int32)
    h.reshape(-1)[::7] >>= 16
    return h


@pytest.mark.parametrize("n,length,b,d", [(16, 1, 24, 4096), (16, 5, 24, 4096), (16, 64, 25, 4080), (32, 33, 24, 4096),
                                          (16, 65, 24, 4096), (16, 37, 9, 1552)])
def test_block_scan(cuda, n, length, b, d):
    from mamba_int import ops
    rng = np.random.default_rng(n + length)
    r = 16
    xs, dm, z = i8(rng, b, length, d), i8(rng, b, length, d), i8(rng, b, length, 2 * d)
    xp = i8(rng, b, length, r + 2 * n)
    base = rng.integers(0, 32001, size=(d, n), dtype=np.int32)
    h = state(rng, b, d, n)
    ref, h_ref = O.block_scan(xs, dm, xp, r, z, d, base, 15, 14, h_state=h.copy())
    ht = T(h)
    yo = ops.block_scan(T(xs), T(dm), T(xp), r, T(z), d, T(base), 15, 14, h_in=ht, h_out=ht)
    assert np.array_equal(yo.cpu().numpy(), ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)


@pytest.mark.parametrize("n", [16, 32, 64])
@pytest.mark.parametrize("length,b,heads,p", [(2, 24, 8, 64), (64, 24, 8, 64), (33, 48, 16, 16), (17, 16, 16, 48)])
def test_ssd_block_scan(cuda, n, length, b, heads, p):
    from mamba_int import ops
    rng = np.random.default_rng(n + 10 * length + p)
    d = heads * p
    w = -(-(2 * heads * n + heads) // 16) * 16
    xs, z, xp = i8(rng, b, length, d), i8(rng, b, length, 2 * d), np.maximum(i8(rng, b, length, w), -127)
    xp[:, ::3, :n] = 0
    xp[:, 1::3, :n] = 0
    xp[:, 1::3, 3] = -127
    tab = rng.integers(0, 2**15 + 1, size=(heads, 255), dtype=np.int32)
    h = state(rng, b, d, n)
    ref, h_ref = O.ssd_v2_scan(xs, xp, z, d, tab, 14, heads, n, h_state=h.copy())
    ht = T(h)
    yo = ops.ssd_block_scan(T(xs), T(xp), T(z), d, T(tab), heads, n, 14, h_in=ht, h_out=ht)
    assert np.array_equal(yo.cpu().numpy(), ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)
