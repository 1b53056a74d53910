"""The elementwise recurrence and its chunked form against the CPU oracle (bit for
bit) at every row split of the kernel (four, two and one steps of rows, chosen by
the channel count and the chunk length), lengths around its groups and its
look-ahead, channel counts that leave lanes and waves idle, decays outside
[0, 2^k] among ones inside, and the state handed on in place."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def inputs(rng, b, length, c, k, wild):
    u = rng.integers(-2**31, 2**31, size=(b, length, c), dtype=np.int64).astype(np.int32)
    u.reshape(-1)[::3] >>= 12
    n = rng.integers(0, 2**k + 1, size=(b, length, c), dtype=np.int64).astype(np.int32)
    if wild:
        n.reshape(-1)[::53] = -12345
        n.reshape(-1)[::71] = 2**31 - 1
    h = rng.integers(-2**31, 2**31, size=(b, c), dtype=np.int64).astype(np.int32)
    return u, n, h


@pytest.mark.parametrize("b,length,c", [(1, 1, 1), (2, 3, 17), (1, 4, 64), (2, 63, 33), (1, 64, 100), (1, 65, 129),
                                        (2, 131, 31), (3, 70, 2800), (1, 33, 20500), (2, 35, 24600)])
@pytest.mark.parametrize("k,wild", [(15, False), (15, True), (1, False), (30, False)])
def test_elementwise(cuda, b, length, c, k, wild):
    from mamba_int import ops
    rng = np.random.default_rng(b * 7 + length + c + k)
    u, n, h = inputs(rng, b, length, c, k, wild)
    ref, h_ref = O.dyadic_scan_elementwise(u, n, k, h_state=h.copy())
    ht = T(h)
    out = ops.dyadic_scan_elementwise(T(u), T(n), k, h_in=ht, h_out=ht)
    assert np.array_equal(out.cpu().numpy(), ref)
    assert np.array_equal(ht.cpu().numpy(), h_ref)


@pytest.mark.parametrize("b,length,c", [(1, 1, 5), (2, 63, 33), (1, 130, 129), (3, 70, 2800), (1, 36, 24600), (2, 20, 24600)])
@pytest.mark.parametrize("chunk", [1, 2, 3, 4, 6, 64, 200])
def test_chunked(cuda, b, length, c, chunk):
    from mamba_int import ops
    rng = np.random.default_rng(b + length + c + chunk)
    u, n, h = inputs(rng, b, length, c, 15, chunk == 3)
    h_ref, f_ref, d_ref, hs_ref = O.dyadic_chunked_scan(u, n, 15, chunk, h_state=h.copy())
    ht = T(h)
    out, f, d = ops.dyadic_chunked_scan(T(u), T(n), 15, chunk, h_in=ht, h_out=ht)
    assert np.array_equal(out.cpu().numpy(), h_ref)
    assert np.array_equal(f.cpu().numpy(), f_ref)
    assert np.array_equal(d.cpu().numpy(), d_ref)
    assert np.array_equal(ht.cpu().numpy(), hs_ref)
