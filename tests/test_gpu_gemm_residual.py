"""The RESIDUAL epilogue of the prefill GEMMs against 64-bit integers: increments
that fit 32 bits and ones that do not (both sides of the host's bound and of the
shift range), saturation at the residual's limits, the accumulator clamp, and the
row statistics."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = 2**23 - 1


@pytest.mark.parametrize("m,n,k", [(65, 36, 64), (130, 128, 192), (16384, 1024, 128)])
@pytest.mark.parametrize("mult,shift", [(1234567, 18), (-1234567, 18), (2**31 - 1, 14), (2**31 - 1, 15), (2**31 - 1, 16),
                                        (3, 0), (3, 1), (2**30, 31), (2**30, 32), (-(2**31), 62)])
@pytest.mark.parametrize("clamp", [0, 100])
def test_residual_epilogue(cuda, m, n, k, mult, shift, clamp):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(m + n + k + shift)
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int64).astype(np.int8)
    a[0], w = 127, rng.integers(-1, 2, size=(n, k), dtype=np.int64).astype(np.int8)
    w[0], w[1] = 1, -1
    r = rng.integers(-LIMIT, LIMIT + 1, size=(m, n), dtype=np.int64).astype(np.int32)
    r[:, ::5] >>= 8
    acc = (torch.from_numpy(a).float() @ torch.from_numpy(w).float().T).numpy().astype(np.int64)  # below 2^24: exact
    c = np.clip(acc, -clamp, clamp) if clamp else acc
    p = c * mult
    ref = np.clip(r + ((p + ((1 << shift) >> 1)) >> shift), -LIMIT, LIMIT).astype(np.int32)
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).cuda()
    wp = ops.pack_ternary(t(w))
    for stats in (None, torch.zeros((m, 2), dtype=torch.int64, device="cuda")):
        out = t(r)
        ops.bitlinear(t(a), wp, ops.OUT_RESIDUAL, n, out=out, res_mult=mult, res_shift=shift, res_clamp=clamp,
                      row_stats=stats, path="gemm")
        assert np.array_equal(out.cpu().numpy(), ref)
        if stats is not None:
            w64 = ref.astype(np.int64)
            assert np.array_equal(stats.cpu().numpy(), np.stack([w64.sum(1), (w64 * w64).sum(1)], 1))
