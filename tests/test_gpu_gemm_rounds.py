"""Prefill products whose 128 x 128 tiles are one round of the CUs, on both sides of
the bound between those tiles and the 64 x 64 ones, against the CPU oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(767, 4096, 1024), (769, 4096, 1024), (769, 4096, 896), (1025, 4096, 1024)])
def test_one_round(cuda, rng, m, n, k):
    import torch
    from mamba_int import ops
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    wp = O.pack_ternary(rng.integers(-1, 2, size=(n, k), dtype=np.int8))
    at, wt = torch.from_numpy(a).cuda(), torch.from_numpy(wp).cuda()
    for kind, shift in ((ops.OUT_INT8, 7), (ops.OUT_INT32, 0)):
        got = ops.bitlinear(at, wt, kind, n, shift=shift)
        assert np.array_equal(got.cpu().numpy(), O.bitlinear(a, wp, kind, shift=shift)), kind
