"""Products of one partial stage (k = 64, half of the 128-deep stage of the prefill
GEMM) against the CPU oracle: every output kind, and the dyadic block of 3 x 701
tokens at d_model 1024, whose dt_rank is 64."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("m,n", [(65, 132), (129, 20), (500, 1040)])
def test_short_k_every_kind(cuda, rng, m, n):
    from mamba_int import ops
    k = 64
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    wp = O.pack_ternary(rng.integers(-1, 2, size=(n, k), dtype=np.int8))
    for kind, shift in ((ops.OUT_INT32, 0), (ops.OUT_INT8, 6), (ops.OUT_DECAY_MOD, 7)):
        got = ops.bitlinear(T(a), T(wp), kind, n, shift=shift)
        assert np.array_equal(got.cpu().numpy(), O.bitlinear(a, wp, kind, shift=shift)), kind
    r = rng.integers(-2**20, 2**20, size=(m, n), dtype=np.int32)
    got = T(r)
    ops.bitlinear(T(a), T(wp), ops.OUT_RESIDUAL, n, out=got, res_mult=4719, res_shift=10)
    assert np.array_equal(got.cpu().numpy(), O.bitlinear(a, wp, ops.OUT_RESIDUAL, residual=r, res_mult=4719, res_shift=10))


def test_block_of_dt_rank_64(cuda):
    from mamba_int import ModelDims, init_random_params
    from mamba_int.model import IntegerMambaRunner
    p = init_random_params(ModelDims(d_model=1024, n_layer=1, vocab_size=64, d_state=16, dt_rank=64), 5)
    ids = np.random.default_rng(5).integers(0, 64, size=(3, 701))
    assert np.array_equal(IntegerMambaRunner(p).forward_logits(T(ids)).cpu().numpy(), O.OracleModel(p).forward(ids))
