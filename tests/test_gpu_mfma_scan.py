"""The scans with their output on the matrix cores against the CPU oracle (bit
for bit) where their splits and chunks can go wrong: every state count, 16-channel
blocks and wider ones, last blocks that are partly empty, lengths around the group
of four steps and the 16-, 32- and 64-step chunks, the whole int32 state range,
decays 0 and 2^15, bytes of -128, and the state handed on.  (The shortest lengths
take the VALU kernels; test_gpu_scan_routes.py has both sides of that bound, the
48-channel blocks of the plain-channel layout and the requant shifts of wide
blocks.)"""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

LENS = [1, 3, 4, 16, 33, 64, 130]


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def i8(rng, *shape):
    return rng.integers(-128, 128, size=shape, dtype=np.int8)


def state(rng, *shape):
    h = rng.integers(-2**31, 2**31, size=shape, dtype=np.int64).astype(np.int32)
    h.reshape(-1)[::7] >>= 16
    return h


@pytest.mark.parametrize("n", [16, 32, 64, 128])
@pytest.mark.parametrize("length", LENS)
def test_channel_scan(cuda, n, length):
    from mamba_int import ops
    import torch
    rng = np.random.default_rng(n * 1000 + length)
    b, d = (2, 80) if length != 33 else (4, 1296)      # 33 steps: more than one round of 16 channels at any N
    x, bb, cc = i8(rng, b, length, d), i8(rng, b, length, n), i8(rng, b, length, n)
    nd = rng.integers(0, 2**15 + 1, size=(d, n), dtype=np.int32)
    nd[0], nd[1] = 0, 2**15
    h = state(rng, b, d, n)
    y_ref, h_ref = O.dyadic_scan(x, bb, cc, nd, 15, h_state=h.copy())
    ht = T(h)
    y = ops.dyadic_scan(T(x), T(bb), T(cc), T(nd), 15, h_in=ht, h_out=ht)
    assert np.array_equal(y.cpu().numpy(), y_ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)
    assert ht.dtype == torch.int32


@pytest.mark.parametrize("n", [16, 32, 64, 128])
@pytest.mark.parametrize("length,heads,p", [(1, 3, 16), (67, 5, 48), (130, 3, 64), (64, 150, 32)])
def test_head_scan(cuda, n, length, heads, p):
    from mamba_int import ops
    import torch
    rng = np.random.default_rng(n * 100 + length + p)
    b, chunk = 2, 64
    x, bb, cc = i8(rng, b, length, heads, p), i8(rng, b, length, heads, n), i8(rng, b, length, heads, n)
    nd = rng.integers(0, 2**15 + 1, size=heads, dtype=np.int32)
    nd[0], nd[-1] = 2**15, 0
    h = state(rng, b, heads, p, n)
    y_ref, st_ref, h_ref = O.ssd_chunked_scan(x, bb, cc, nd, 15, chunk, h_state=h.copy(), want_chunk_states=True)
    ht = T(h)
    st = torch.empty((b, -(-length // chunk), heads, p, n), dtype=torch.int32, device="cuda")
    y = ops.ssd_chunked_scan(T(x), T(bb), T(cc), T(nd), 15, chunk, chunk_states=st, h_in=ht, h_out=ht)
    assert np.array_equal(y.cpu().numpy(), y_ref)
    assert np.array_equal(st.cpu().numpy(), st_ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)


@pytest.mark.parametrize("n", [16, 32, 64])
@pytest.mark.parametrize("length,b,d", [(1, 1, 16), (7, 2, 80), (64, 1, 48), (130, 2, 112), (37, 4, 1040), (33, 4, 2064),
                                        (20, 3, 4112)])
@pytest.mark.parametrize("s_y", [0, 14, 20])
def test_block_scan(cuda, n, length, b, d, s_y):
    """Decays that reach both clamps in some waves only; s_y on both sides of the
    largest shift whose result the gate saturates alike."""
    from mamba_int import ops
    if s_y != 14 and d > 200:
        pytest.skip("the requant shift does not depend on the block width")
    rng = np.random.default_rng(n * 10 + length + d + s_y)
    r = 16
    xs, dm, z = i8(rng, b, length, d), i8(rng, b, length, d), i8(rng, b, length, 2 * d)
    xp = i8(rng, b, length, r + 2 * n)
    base = rng.integers(20, 31981, size=(d, n), dtype=np.int32)
    base[3], base[-1] = rng.integers(0, 20, size=n), rng.integers(31981, 32001, size=n)
    h = state(rng, b, d, n)
    ref, h_ref = O.block_scan(xs, dm, xp, r, z, d, base, 15, s_y, h_state=h.copy())
    ht = T(h)
    yo = ops.block_scan(T(xs), T(dm), T(xp), r, T(z), d, T(base), 15, s_y, h_in=ht, h_out=ht)
    assert np.array_equal(yo.cpu().numpy(), ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)


@pytest.mark.parametrize("n", [16, 32, 64])
@pytest.mark.parametrize("length,heads,p", [(2, 1, 16), (31, 3, 48), (64, 2, 64), (70, 5, 32)])
def test_ssd_block_scan(cuda, n, length, heads, p):
    """Rows of zeros and of one nonzero value among B and C (the unit vectors' ends)."""
    from mamba_int import ops
    rng = np.random.default_rng(n + 10 * length + p)
    b, d = 2, heads * p
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
