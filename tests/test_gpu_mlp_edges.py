"""The radiance cache's kernels where their blocks of 16 and rounds of 64
samples end, on samples that start on any float, and past one round per
workgroup (256 workgroups x 64 samples).

Everything is exact, or has one rounding of 1/n on either side (relative 3e-7).
"""
import numpy as np
import pytest

import ptamd
from ptamd import hip
from test_oracle_mlp import BMAX, BMIN, random_params, random_raw

pytestmark = pytest.mark.gpu


def targets(n, seed):
    return np.random.default_rng(seed).uniform(0.0, 2.0, (n, 3)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 17, 63, 64, 65])
def test_gradient_at_round_edges(ctx, n):
    # The batch's end falls inside a round or block: as if the rest of a larger
    # batch were masked (gradients of whole rounds are held against the oracle
    # in test_gpu_cache).
    print(f"[mlp edges] gradient n={n}", flush=True)
    ctx.cache_init(1, BMIN, BMAX)
    ctx.cache_set_params(random_params(4, bias=0.2))
    raw, tgt = random_raw(128, 15), targets(128, 16)
    got = ctx.cache_gradient(raw[:n].copy(), tgt[:n].copy()).astype(np.float64)
    tgt[n:, 0] = np.nan
    padded = ctx.cache_gradient(raw, tgt).astype(np.float64)
    np.testing.assert_allclose(got * (n / 128), padded, rtol=3e-7, atol=1e-30)


@pytest.mark.parametrize("tail", [1, 64, 100])
def test_masked_rounds_leave_the_rest(ctx, tail):
    # Only a second round's samples count: their own gradient, times tail / n.
    n = 16384 + tail
    print(f"[mlp edges] masked n={n}", flush=True)
    ctx.cache_init(1, BMIN, BMAX)
    ctx.cache_set_params(random_params(5, bias=0.2))
    raw, tgt = random_raw(n, 17), targets(n, 18)
    tgt[:16384, 0] = np.nan
    alone = ctx.cache_gradient(raw[16384:].copy(), tgt[16384:].copy()).astype(np.float64)
    got = ctx.cache_gradient(raw, tgt).astype(np.float64)
    np.testing.assert_allclose(got, alone * (tail / n), rtol=3e-7, atol=1e-30)


@pytest.mark.parametrize("n", [1, 63, 65, 300])
@pytest.mark.parametrize("skip", [1, 2, 3])
def test_samples_on_any_float(ctx, n, skip):
    print(f"[mlp edges] unaligned n={n} skip={skip}", flush=True)
    ctx.cache_init(1, BMIN, BMAX)
    ctx.cache_set_params(random_params(6, bias=0.2))
    raw, tgt = random_raw(n, 19), targets(n, 20)
    buf = hip.DeviceArray.from_host(np.concatenate([np.zeros(skip, np.float32), raw.reshape(-1)]))
    t = hip.DeviceArray.from_host(tgt)
    out = hip.DeviceArray.from_host(np.full(3 * n + 8, -1.0, np.float32))
    grad = hip.DeviceArray(ptamd.CACHE_PARAMS, np.float32)
    ctx.cache_infer_device(buf.ptr + 4 * skip, n, out.ptr)
    ctx.cache_gradient_device(buf.ptr + 4 * skip, t.ptr, n, grad.ptr)
    ctx.synchronize()
    got = out.to_host()
    np.testing.assert_array_equal(got[: 3 * n].reshape(n, 3), ctx.cache_infer(raw))
    assert (got[3 * n:] == -1.0).all()
    np.testing.assert_array_equal(grad.to_host(), ctx.cache_gradient(raw, tgt))
