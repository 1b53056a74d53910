"""The scans on both sides of their split into the VALU and
MFMA kernels, by steps and by rounds of blocks on 256 CUs, and over rows too
long for the MFMA kernel's offsets, against the CPU oracle (bit for bit)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def i8(rng, *shape):
    return rng.integers(-128, 128, size=shape, dtype=np.int8)


def i32(rng, *shape):
    return rng.integers(-2**31, 2**31, size=shape, dtype=np.int64).astype(np.int32)


# from below one round up (d not a multiple of the block), every lane split of the VALU
# kernel; lengths with every remainder of the MFMA kernel's groups; 48-channel blocks
# (8192 < b * d <= 12288, also with a partly empty last block)
@pytest.mark.parametrize("n,b,d,lengths", [(16, 2, 80, (16, 17, 19, 22, 31, 63, 68)), (16, 3, 2064, (8, 9)), (16, 4, 2064, (8, 33, 70)),
                                           (16, 4, 2080, (33, 70)), (16, 7, 4096, (12, 13)), (16, 34, 4112, (24, 25)), (16, 50, 4096, (100,)),
                                           (32, 2, 80, (12, 13, 18, 23, 35)), (32, 5, 2064, (4, 5)), (32, 7, 2064, (8, 9)),
                                           (32, 6, 4096, (2, 3)), (32, 8, 4096, (4, 5)),
                                           (64, 2, 80, (12, 13, 18, 23, 35)), (64, 3, 2048, (8, 9)), (64, 5, 2064, (1, 2)),
                                           (128, 2, 80, (1, 9, 15, 18, 35)), (128, 6, 2064, (8, 9)),
                                           (16, 1, 4096, (16, 17)), (32, 7, 2064, (22, 23)), (64, 4, 2048, (6, 7)), (128, 6, 2064, (14, 15))])
def test_channel_routes(cuda, n, b, d, lengths):
    from mamba_int import ops
    rng = np.random.default_rng(n + b + d)
    nd = rng.integers(0, 2**15 + 1, size=(d, n), dtype=np.int32)
    for length in lengths:
        x, bb, cc, h = i8(rng, b, length, d), i8(rng, b, length, n), i8(rng, b, length, n), i32(rng, b, d, n)
        y_ref, h_ref = O.dyadic_scan(x, bb, cc, nd, 15, h_state=h.copy())
        ht = T(h)
        y = ops.dyadic_scan(T(x), T(bb), T(cc), T(nd), 15, h_in=ht, h_out=ht)
        assert np.array_equal(y.cpu().numpy(), y_ref) and np.array_equal(ht.cpu().numpy(), h_ref), length


@pytest.mark.parametrize("n,b,heads,p,lengths", [(16, 2, 3, 48, (16, 17, 22, 31, 63)), (16, 8, 24, 64, (12, 13)),
                                                 (16, 12, 24, 64, (16,)), (16, 24, 24, 64, (16, 17)), (16, 44, 24, 64, (16, 17)),
                                                 (32, 2, 3, 48, (16, 17, 22, 35)), (32, 8, 24, 64, (16, 17)), (32, 12, 24, 64, (16,)),
                                                 (32, 24, 24, 64, (16,)), (32, 44, 24, 64, (16, 17)),
                                                 (64, 2, 5, 16, (16, 17, 22, 35)), (64, 12, 24, 64, (10, 11)), (64, 24, 24, 64, (10, 11)),
                                                 (128, 2, 3, 48, (12, 13)), (128, 8, 24, 64, (16, 17)), (128, 32, 24, 64, (32, 33)),
                                                 (16, 12, 24, 64, (17,)), (64, 2, 5, 16, (28, 29)), (128, 6, 16, 48, (64, 65)),
                                                 (128, 8, 24, 64, (28, 29))])
def test_head_routes(cuda, n, b, heads, p, lengths):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(n + b + heads)
    nd = rng.integers(0, 2**15 + 1, size=heads, dtype=np.int32)
    for length in lengths:
        x, bb, cc = i8(rng, b, length, heads, p), i8(rng, b, length, heads, n), i8(rng, b, length, heads, n)
        h = i32(rng, b, heads, p, n)
        y_ref, st_ref, h_ref = O.ssd_chunked_scan(x, bb, cc, nd, 15, 64, h_state=h.copy(), want_chunk_states=True)
        ht, st = T(h), torch.empty((b, -(-length // 64), heads, p, n), dtype=torch.int32, device="cuda")
        y = ops.ssd_chunked_scan(T(x), T(bb), T(cc), T(nd), 15, 64, chunk_states=st, h_in=ht, h_out=ht)
        for got, want in ((y, y_ref), (st, st_ref), (ht, h_ref)):
            assert np.array_equal(got.cpu().numpy(), want), length


def test_head_long_rows(cuda):
    """B and C rows of 2^22 bytes and more, past the VALU kernel's lengths."""
    from mamba_int import ops
    rng = np.random.default_rng(1)
    b, length, heads, p, n = 1, 33, 32800, 16, 128
    x, bb, cc = i8(rng, b, length, heads, p), i8(rng, b, length, heads, n), i8(rng, b, length, heads, n)
    nd = rng.integers(0, 2**15 + 1, size=heads, dtype=np.int32)
    y = ops.ssd_chunked_scan(T(x), T(bb), T(cc), T(nd), 15, 64)
    assert np.array_equal(y.cpu().numpy(), O.ssd_chunked_scan(x, bb, cc, nd, 15, 64))


@pytest.mark.parametrize("n,length", [(16, 33), (64, 40)])
def test_block_scan_long_rows(cuda, n, length):
    """z rows of 2^22 bytes and more."""
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(n)
    b, d, r = 2, 48, 16
    xs, dm, z = i8(rng, b, length, d), i8(rng, b, length, d), i8(rng, b, length, 2 * d)
    xp, base = i8(rng, b, length, r + 2 * n), rng.integers(0, 32001, size=(d, n), dtype=np.int32)
    far = torch.zeros((b, length, 2**22 + 16), dtype=torch.int8, device="cuda")
    far[..., :2 * d] = T(z)
    h = torch.empty((b, d, n), dtype=torch.int32, device="cuda")
    yo = ops.block_scan(T(xs), T(dm), T(xp), r, far, d, T(base), 15, 14, h_out=h)
    ref, h_ref = O.block_scan(xs, dm, xp, r, z, d, base, 15, 14)
    assert np.array_equal(yo.cpu().numpy(), ref) and np.array_equal(h.cpu().numpy(), h_ref)


@pytest.mark.parametrize("n,b,d,lengths", [(16, 2, 80, (4, 5)), (16, 4, 2048, (12, 13)), (16, 6, 2064, (16, 17)), (16, 8, 2048, (8, 9)),
                                           (16, 9, 2064, (16, 17)), (16, 16, 2064, (64, 65)), (32, 2, 80, (4, 5)),
                                           (32, 4, 2048, (112, 113)), (32, 6, 2064, (16, 200)), (32, 9, 2064, (64, 65)),
                                           (64, 2, 80, (24, 25, 28, 29)), (64, 4, 2048, (112, 113, 160, 161)), (64, 5, 2064, (150,)),
                                           (16, 3, 4112, (24, 25)), (16, 14, 2064, (64, 65)), (32, 5, 2048, (24, 25)), (32, 9, 2048, (80, 81))])
def test_block_routes(cuda, n, b, d, lengths):
    from mamba_int import ops
    rng = np.random.default_rng(n + b + d)
    r, base = 16, rng.integers(0, 32001, size=(d, n), dtype=np.int32)
    for length in lengths:
        xs, dm, z = i8(rng, b, length, d), i8(rng, b, length, d), i8(rng, b, length, 2 * d)
        xp, h = i8(rng, b, length, r + 2 * n), i32(rng, b, d, n)
        ref, h_ref = O.block_scan(xs, dm, xp, r, z, d, base, 15, 14, h_state=h.copy())
        ht = T(h)
        yo = ops.block_scan(T(xs), T(dm), T(xp), r, T(z), d, T(base), 15, 14, h_in=ht, h_out=ht)
        assert np.array_equal(yo.cpu().numpy(), ref) and np.array_equal(ht.cpu().numpy(), h_ref), length


@pytest.mark.parametrize("n,b,heads,p,lengths", [(16, 2, 3, 48, (4, 5)), (16, 4, 8, 64, (12, 13)), (16, 20, 24, 64, (56, 57)),
                                                 (32, 2, 3, 48, (2, 3)), (32, 8, 24, 64, (16, 17)), (32, 20, 24, 64, (48, 49)),
                                                 (64, 2, 3, 48, (16, 17)), (64, 4, 24, 64, (48, 49)), (64, 12, 24, 64, (64, 65)),
                                                 (64, 16, 24, 64, (80, 81)), (64, 26, 24, 64, (100, 101)),
                                                 (16, 8, 24, 64, (12, 13)), (32, 8, 24, 64, (28, 29)), (64, 4, 24, 64, (64, 65)),
                                                 (64, 20, 24, 64, (128, 129))])
def test_ssd_routes(cuda, n, b, heads, p, lengths):
    from mamba_int import ops
    rng = np.random.default_rng(n + b + heads)
    d, w = heads * p, -(-(2 * heads * n + heads) // 16) * 16
    tab = rng.integers(0, 2**15 + 1, size=(heads, 255), dtype=np.int32)
    for length in lengths:
        xs, z, xp = i8(rng, b, length, d), i8(rng, b, length, 2 * d), np.maximum(i8(rng, b, length, w), -127)
        h = i32(rng, b, d, n)
        ref, h_ref = O.ssd_v2_scan(xs, xp, z, d, tab, 14, heads, n, h_state=h.copy())
        ht = T(h)
        yo = ops.ssd_block_scan(T(xs), T(xp), T(z), d, T(tab), heads, n, 14, h_in=ht, h_out=ht)
        assert np.array_equal(yo.cpu().numpy(), ref) and np.array_equal(ht.cpu().numpy(), h_ref), length


@pytest.mark.parametrize("s_y", [0, 14, 20, 30])
@pytest.mark.parametrize("b,d", [(2, 4080), (4, 2064), (4, 2080)])
def test_block_shifts_of_wide_blocks(cuda, b, d, s_y):
    """The requant shift in the 32- and 48-channel blocks (last blocks full and partly empty)."""
    from mamba_int import ops
    rng = np.random.default_rng(b + d + s_y)
    n, r, length = 16, 16, 45
    xs, dm, z = i8(rng, b, length, d), i8(rng, b, length, d), i8(rng, b, length, 2 * d)
    xp, base, h = i8(rng, b, length, r + 2 * n), rng.integers(0, 32001, size=(d, n), dtype=np.int32), i32(rng, b, d, n)
    ref, h_ref = O.block_scan(xs, dm, xp, r, z, d, base, 15, s_y, h_state=h.copy())
    ht = T(h)
    yo = ops.block_scan(T(xs), T(dm), T(xp), r, T(z), d, T(base), 15, s_y, h_in=ht, h_out=ht)
    assert np.array_equal(yo.cpu().numpy(), ref) and np.array_equal(ht.cpu().numpy(), h_ref)
