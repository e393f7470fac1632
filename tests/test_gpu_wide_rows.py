"""Row sums over thousands of columns (zk_row_sum_wide) and output layers on
feature-major operands (zk_narrow_f*), at the edges of their blocks; the layers
of short minibatches (zk_narrow_n1_v, zk_narrow_f22)."""

import numpy as np
import pytest
import torch

from conftest import launches
from oracle import zl_oracle as zo
from zealot_amd import DeviceBuffer, ops, synth
from zealot_amd.rl import GpuMlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(3, 2047), (3, 2048), (1, 8191), (2, 8192), (5, 8193), (2, 24_581), (300, 4096),
                                 (512, 2100), (513, 2100), (600, 8191), (600, 8192)])
def test_row_sum_exact_on_integers(ctx, m, n):
    """Whole numbers below 2^24 in every partial sum: any order gives the same."""
    x = np.random.default_rng(n).integers(-300, 300, (m, n)).astype(np.float32)
    out, dx = ctx.alloc(m), ctx.to_device(x)
    names = launches(ctx, lambda: ops.row_sum(ctx, out, dx, m, n))
    assert names == ["zk_row_sum_wide" if n >= 8192 or n >= 2048 and m <= 512 else "zk_row_sum"]
    assert np.array_equal(out.numpy(), x.sum(1, dtype=np.float64).astype(np.float32))


def test_row_sum_of_two_billion_columns(ctx):
    """A row whose last indices plus a block's stride lie past 2^31."""
    n = 2**31 - 1000
    x = torch.zeros(n, device="cuda")
    x[0], x[n // 2], x[n - 1] = 1, 2, 4
    torch.cuda.synchronize()
    dx, out = DeviceBuffer(ctx, x.data_ptr(), 4 * n, (1, n), np.float32), ctx.alloc(1)
    ops.row_sum(ctx, out, dx, 1, n)
    dx.ptr = 0  # torch frees it
    got = out.numpy()[0]
    del x
    torch.cuda.empty_cache()
    assert got == 7


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_row_sum_not_finite(ctx, bad):
    x = np.ones((2, 9000), np.float32)
    x[1, 8999] = bad
    out = ctx.alloc(2)
    ops.row_sum(ctx, out, ctx.to_device(x), 2, 9000)
    assert np.array_equal(out.numpy(), np.array([9000, bad], np.float32), equal_nan=True)


FEATURE_MAJOR = [(m, n, k) for m in (1, 16, 17, 32)
                 for n, k in ((1, 33), (15, 48), (17, 100), (300, 123), (4096, 512), (131, 513), (64, 16 * 8 * 5))]


@pytest.mark.parametrize("m,n,k", FEATURE_MAJOR + [(33, 300, 129), (48, 31, 40), (64, 8192, 512), (512, 512, 513),
                                                   (29, 4097, 512), (12, 24_577, 123)])
def test_feature_major_output_layer(ctx, m, n, k):
    """C[m x n] = W[m x k] X[k x n] + bias, with and without ELU: 16-column blocks
    of 16 or 32 rows (up to 32 rows), 32 x 32 blocks (more rows, or 17 to 32 past
    4,096 columns). Bound: k products and additions in any order, the bias, the
    activation (|slope| <= 1)."""
    g = np.random.default_rng(m * 1000 + n + k)
    w, x, b = (g.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m,)))
    dw, dx, db, out = ctx.to_device(w), ctx.to_device(x), ctx.to_device(b), ctx.alloc((m, n))
    z = w.astype(np.float64) @ x + b[:, None]
    bound = 2.0**-24 * (k + 4) * (np.abs(w).astype(np.float64) @ np.abs(x) + np.abs(b)[:, None] + 1)
    want = "zk_narrow_f1" if m <= 16 else "zk_narrow_f2" if m <= 32 and n <= 4096 else "zk_narrow_f22"
    for act in (False, True):
        names = launches(ctx, lambda: ops.gemm_bias_act(ctx, out, dw, dx, m, n, k, db, 1, act))
        assert names == [want]
        ref = np.where(z > 0, z, np.expm1(np.minimum(z, 0))) if act else z
        assert np.all(np.abs(out.numpy() - ref) <= bound)


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 383, 384, 385, 511, 512, 513])
@pytest.mark.parametrize("dims", [[48, 80, 64, 16], [30, 512, 100, 33, 5]])
def test_short_batches(ctx, rows, dims):
    """Forward strips and data gradients of up to 512 rows and the row after,
    widths off the 16 and 32 column tiles; against the oracle with the bar of
    the layer GEMMs (1e-4 of each tensor's largest value)."""
    g = np.random.default_rng(rows)
    params = synth.kaiming_uniform_net(g, dims, 0.1)
    x = g.standard_normal((rows, dims[0])).astype(np.float32)
    gout = (g.standard_normal((rows, dims[-1])) / rows).astype(np.float32)
    mlp = GpuMlp(ctx, dims, rows)
    mlp.write_weights(params)
    dx, dg = ctx.to_device(x), ctx.to_device(gout)
    names = launches(ctx, lambda: mlp.forward(dx, rows))
    # Strips for the layers wider than 32 that read whole chunks of 16.
    wide = [i for i, o in zip(dims, dims[1:]) if o > 32 and i % 16 == 0]
    if rows <= 512:
        assert names.count("zk_narrow_n1_v") >= len(wide), names
    else:
        assert any(x.startswith("zk_gemm_ak_bk") for x in names), names
    ref = zo.mlp_forward(dims, params, x)[-1]
    assert np.abs(mlp.output(rows) - ref).max() <= 1e-4 * np.abs(ref).max()
    names = launches(ctx, lambda: mlp.backward(dg))
    assert ("zk_narrow_f22" in names) == (rows <= 512 and any(o > 32 for o in dims[2:])), names
    got, (ref, _) = mlp.read_grads(), zo.mlp_backward(dims, params, x, gout)
    o = 0
    for i, j in zip(dims, dims[1:]):
        for sz in (j * i, j):
            a, b = got[o:o + sz], ref[o:o + sz]
            assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max()
            o += sz
