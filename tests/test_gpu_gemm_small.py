"""The narrow prefill products against an exact one: k of one MFMA (dt_proj) at
every word count, token and feature counts around its tiles; and few outputs
(x_proj) at the row counts where its block of 16, 32 or 64 rows changes."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(m, n, k, kind, shift, lim, pad):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(m * 7 + n + k)
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int64).astype(np.int8)
    w = rng.integers(-1, 2, size=(n, k), dtype=np.int64).astype(np.int8)
    ta, tw = torch.from_numpy(a).cuda(), torch.from_numpy(w).cuda()
    acc = (ta.float() @ tw.float().T).to(torch.int64)   # below 2^24: exact
    out = torch.full((m, n + pad), 99, dtype=torch.int8, device="cuda")
    ops.bitlinear(ta, ops.pack_ternary(tw), kind, n, shift=shift, out=out, path="gemm")
    ref = torch.clamp((acc + ((1 << shift) >> 1)) >> shift, -lim, lim).to(torch.int8)
    assert torch.equal(out[:, :n], ref)
    assert bool((out[:, n:] == 99).all())


@pytest.mark.parametrize("m", [1, 15, 64, 65, 200])
@pytest.mark.parametrize("n", [16, 64, 240, 272, 1536])
@pytest.mark.parametrize("k", [16, 32, 48, 64])
def test_one_mfma_deep(cuda, m, n, k):
    from mamba_int import ops
    check(m, n, k, ops.OUT_DECAY_MOD, 5, 20, 16)
    check(m, n, k, ops.OUT_INT8, 0, 127, 0)


@pytest.mark.parametrize("m", [65, 4096, 4097, 8192, 8193, 16384, 16385])
@pytest.mark.parametrize("n", [36, 80, 96])
@pytest.mark.parametrize("k", [256, 1536])
def test_few_outputs(cuda, m, n, k):
    from mamba_int import ops
    check(m, n, k, ops.OUT_INT8, 6, 127, 4)
