"""The elementwise and chunked recurrences on both sides of their split into rows
of steps and lanes (few steps, many sequences of few channels) against the CPU
oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("b,length,c", [(1, 1, 1), (3, 4, 70), (2, 5, 33), (3, 15, 65), (3, 16, 65), (2, 31, 10300), (2, 32, 10300),
                                        (300, 9, 300), (300, 33, 300), (8200, 17, 1), (4100, 40, 5), (4096, 40, 8), (2048, 17, 8),
                                        (2049, 33, 16), (2048, 155, 1), (2048, 160, 1), (4096, 130, 1), (4096, 136, 1),
                                        (4096, 345, 1), (4096, 355, 1), (6000, 400, 2)])
def test_elementwise_and_chunked(cuda, b, length, c):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(b + length + c)
    u = rng.integers(-2**31, 2**31, size=(b, length, c), dtype=np.int64).astype(np.int32)
    n = rng.integers(0, 2**15 + 1, size=(b, length, c), dtype=np.int32)
    n[0, -1, 0] = 2**31 - 1                       # outside [0, 2^k]: saturates
    h0 = rng.integers(-2**31, 2**31, size=(b, c), dtype=np.int64).astype(np.int32)
    h_ref, s_ref = O.dyadic_scan_elementwise(u, n, 15, h_state=h0.copy())
    ut, st = T(u), T(h0)
    h = ops.dyadic_scan_elementwise(ut, T(n), 15, h_in=st, h_out=st)
    assert np.array_equal(h.cpu().numpy(), h_ref) and np.array_equal(st.cpu().numpy(), s_ref)
    for chunk in (3, 8):
        want = O.dyadic_chunked_scan(u, n, 15, chunk, h_state=h0.copy())
        got = ops.dyadic_chunked_scan(ut, T(n), 15, chunk, h_in=T(h0))
        for a, w in zip(got, want):
            assert np.array_equal(a.cpu().numpy(), w)
