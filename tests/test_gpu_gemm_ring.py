"""The 64 x 64-tile prefill GEMM against an exact product: token counts around its
tiles, feature counts with half a tile, one to many stages of k, every output
kind; and its conv form against the separate in_proj and conv kernels, with
sequence starts and ends anywhere in its 61-row tiles."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def i8(rng, *shape, lo=-127, hi=127):
    return rng.integers(lo, hi + 1, size=shape, dtype=np.int64).astype(np.int8)


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("m", [1, 63, 64, 65, 200])
@pytest.mark.parametrize("n,k", [(192, 128), (224, 256), (32, 384), (1056, 640)])
@pytest.mark.parametrize("kind", ["INT32", "INT8", "DECAY_MOD", "RESIDUAL", "FLOAT"])
def test_gemm_ring(cuda, m, n, k, kind):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(m * 7 + n + k)
    a, w = i8(rng, m, k), i8(rng, n, k, lo=-1, hi=1)
    a[-1] = 127
    w[0] = 1
    acc = (torch.from_numpy(a).float() @ torch.from_numpy(w).float().T).numpy().astype(np.int64)  # below 2^24: exact
    wp, kw = ops.pack_ternary(T(w)), {}
    if kind == "INT32":
        ref = acc.astype(np.int32)
    elif kind in ("INT8", "DECAY_MOD"):
        lim, kw["shift"] = (127, 5) if kind == "INT8" else (20, 7)
        ref = np.clip((acc + (1 << (kw["shift"] - 1))) >> kw["shift"], -lim, lim).astype(np.int8)
    elif kind == "RESIDUAL":
        r = rng.integers(-2**23 + 1, 2**23, size=(m, n), dtype=np.int64).astype(np.int32)
        kw = dict(out=T(r), res_mult=76543, res_shift=12)
        ref = np.clip(r + ((acc * 76543 + 2048) >> 12), -(2**23) + 1, 2**23 - 1).astype(np.int32)
        kw["row_stats"] = torch.zeros((m, 2), dtype=torch.int64, device="cuda")
    else:
        xs = rng.random(m, dtype=np.float32)
        kw = dict(x_scale=T(xs), w_scale=0.375)
        ref = acc.astype(np.float32) * (np.float32(0.375) * xs)[:, None]
    y = ops.bitlinear(T(a), wp, getattr(ops, "OUT_" + kind), n, path="gemm", **kw)
    assert np.array_equal(y.cpu().numpy(), ref)
    if kind == "RESIDUAL":
        v = ref.astype(np.int64)
        assert np.array_equal(kw["row_stats"].cpu().numpy(), np.stack([v.sum(1), (v * v).sum(1)], 1))


@pytest.mark.parametrize("batch,length", [(1, 1), (1, 2), (3, 2), (1, 61), (1, 62), (2, 64), (5, 61), (2, 183), (7, 29)])
@pytest.mark.parametrize("d_model,d_inner", [(128, 128), (384, 384)])
def test_in_proj_conv_ring(cuda, batch, length, d_model, d_inner):
    import torch
    from mamba_int import ops
    rng = np.random.default_rng(batch * 1000 + length + d_inner)
    m = batch * length
    a, w = T(i8(rng, m, d_model)), ops.pack_ternary(T(i8(rng, 2 * d_inner, d_model, lo=-1, hi=1)))
    cw, cb = T(i8(rng, d_inner, 4)), T(rng.integers(-60000, 60001, size=d_inner, dtype=np.int64).astype(np.int32))
    st = T(i8(rng, batch, 3, d_inner))
    xz = torch.empty((m, 2 * d_inner), dtype=torch.int8, device="cuda")
    ops.bitlinear(a, w, ops.OUT_INT8, 2 * d_inner, shift=4, out=xz, path="gemm")
    ref_st = torch.empty_like(st)
    ref = ops.conv_squareplus(xz, d_inner, cw, cb, state_in=st, state_out=ref_st, batch=batch)
    xz2, out_st = torch.empty_like(xz), torch.empty_like(st)
    xs = ops.in_proj_conv(a, w, 4, d_inner, cw, cb, batch, state_in=st, state_out=out_st, xz=xz2)[0]
    assert torch.equal(xs.view(m, -1), ref.view(m, -1))
    assert torch.equal(out_st, ref_st)
    assert torch.equal(xz2[:, d_inner:], xz[:, d_inner:])
