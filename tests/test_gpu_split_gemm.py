"""The three-piece bf16 GEMMs (zk_split_*): tile edges, K tails, split-K, rows
that are not float4-aligned, gathered rows, and operands that the pieces do not
hold (infinities, values near the largest float, tiny ones), against float64
and against the fp32 kernels (ZL_SPLIT_GEMM=0, read at zl_init)."""

import os

import numpy as np
import pytest

from conftest import launches as used
from zealot_amd import ops, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fp32_ctx():
    from zealot_amd import Context

    os.environ["ZL_SPLIT_GEMM"] = "0"
    try:
        c = Context(0)
    finally:
        del os.environ["ZL_SPLIT_GEMM"]
    yield c
    c.close()


def product(ctx, L, R, lt, rt):
    m, k, n = L.shape[0], L.shape[1], R.shape[1]
    out = ctx.alloc((m, n))
    dl = ctx.to_device(np.ascontiguousarray(L.T if lt else L))
    dr = ctx.to_device(np.ascontiguousarray(R.T if rt else R))
    ops.gemm(ctx, out, dl, lt, dr, rt, m, n, k)
    return out.numpy()


# (m, n, k, lhs_t, rhs_t, variant): whole tiles; one past and one short of a tile
# in each extent; K tails of 1, 31 and one k-tile; K not a multiple of 4 (element
# loads); deep K with slices whose last one holds the tail.
CASES = [(32768, 128, 32, False, True, "ak_bk"), (49153, 127, 33, False, True, "ak_bk_s"),
         (8191, 257, 96, False, True, "ak_bk"), (49170, 250, 1, False, True, "ak_bk_s"),
         (6200, 256, 123, False, True, "ak_bk_s"), (256, 300, 8193, False, True, "ak_bk_s"),
         (250, 24577, 516, False, False, "ak_bn"), (384, 11000, 261, False, False, "ak_bn_s"),
         (255, 16500, 200, True, False, "am_bn"), (193, 513, 24577, True, False, "am_bn"),
         (256, 512, 6144, True, False, "am_bn")]


def as_exact_as_fp32(got, fp32, ref, tag):
    """Relative 2-norm error no larger than the fp32 kernels', by more than a
    quarter (another order of the same number of roundings) and 2e-8. A product
    that dropped one of the six terms is 2e-6 off at any K, the fp32 kernels at
    most 7e-7."""
    e = [np.linalg.norm(x - ref) / np.linalg.norm(ref) for x in (got, fp32)]
    print(f"[gpu] split gemm {tag}: relative error {e[0]:.2e}, fp32 kernels {e[1]:.2e}", flush=True)
    assert e[0] <= 1.25 * e[1] + 2e-8, tag


@pytest.mark.parametrize("case", CASES)
def test_split_gemm_edges(ctx, fp32_ctx, case):
    m, n, k, lt, rt, variant = case
    g = np.random.default_rng(m + 3 * n + 7 * k)
    L, R = synth.normal(g, (m, k)), synth.normal(g, (k, n))
    got = []
    names = used(ctx, lambda: got.append(product(ctx, L, R, lt, rt)))
    assert names[0] == f"zk_split_{variant}", names
    ref = L.astype(np.float64) @ R.astype(np.float64)
    # Six products per 16 reduction indices enter the fp32 accumulator, each
    # rounded to 2^-24 of a partial sum below |L| |R|; the split-K slices and
    # the dropped terms (2^-26) add less than 40 more.
    bound = (6 * (-(-k // 16)) + 40) * 2.0 ** -24 * (np.abs(L).astype(np.float64) @ np.abs(R).astype(np.float64))
    assert np.all(np.abs(got[0] - ref) <= bound), case
    as_exact_as_fp32(got[0], product(fp32_ctx, L, R, lt, rt), ref, case)


@pytest.mark.parametrize("what", ["inf", "-inf", "nan", "max", "tiny", "zero"])
@pytest.mark.parametrize("lt,rt", [(False, True), (False, False), (True, False)])
def test_split_gemm_special_values(ctx, fp32_ctx, what, lt, rt):
    """Infinities, NaN, values that round to a bf16 infinity and operands whose
    low pieces leave the bf16 range give what the fp32 kernels give."""
    m, n, k = 1100, 4200, 300
    g = np.random.default_rng(5)
    L, R = synth.normal(g, (m, k)), synth.normal(g, (k, n), 0.05)
    if what == "tiny":
        L = (L * np.float32(1e-36)).astype(np.float32)
    elif what == "zero":
        L[:] = 0.0
    else:
        v = {"inf": np.inf, "-inf": -np.inf, "nan": np.nan, "max": np.finfo(np.float32).max}[what]
        L[700, 17] = v
        R[17, :] = np.where(np.abs(R[17, :]) < 1e-3, 1e-3, R[17, :])
    assert any(x.startswith("zk_split_") for x in used(ctx, lambda: product(ctx, L, R, lt, rt)))
    a, b = product(ctx, L, R, lt, rt), product(fp32_ctx, L, R, lt, rt)
    assert np.array_equal(np.isnan(a), np.isnan(b))
    inf = np.isinf(b)
    assert np.array_equal(inf, np.isinf(a)) and np.array_equal(a[inf], b[inf])
    ok = np.isfinite(b)
    # Both sums lie within K roundings of 2^-24 of |L| |R|.
    with np.errstate(invalid="ignore", over="ignore"):
        bound = 2 * k * 2.0 ** -24 * (np.abs(L).astype(np.float64) @ np.abs(R).astype(np.float64))
    d = np.abs(a[ok].astype(np.float64) - b[ok])
    assert np.all(d <= np.maximum(bound[ok], 0.0) + 1e-45)


@pytest.mark.parametrize("what", ["tiny x huge", "subnormal x huge", "tiny row", "tiny column", "subnormal row"])
@pytest.mark.parametrize("lt,rt", [(False, True), (False, False), (True, False)])
def test_split_gemm_small_operands(ctx, what, lt, rt):
    """Operands whose low pieces lie below the bf16 range, alone or beside
    ordinary rows and columns, with results of ordinary size or not: every row
    and column as close to float64 as those of ordinary operands. Bound: 6 x
    19 random-sign roundings of 2^-24 of the running sum are 4e-7 of the root
    mean square of a row; two pieces alone leave 1e-5."""
    m, n, k = 1100, 4200, 300
    g = np.random.default_rng(7)
    L, R = synth.normal(g, (m, k)), synth.normal(g, (k, n))
    if what == "tiny x huge":
        L, R = L * np.float32(2.0**-119), R * np.float32(2.0**60)
    elif what == "subnormal x huge":
        L, R = L * np.float32(2.0**-132), R * np.float32(2.0**80)
    elif what == "tiny row":
        L[701] *= np.float32(2.0**-119)
    elif what == "tiny column":
        R[:, 1503] *= np.float32(2.0**-119)
    else:  # beside ordinary rows, all sums below 2^80
        L[701] *= np.float32(2.0**-134)
        R[:, 1503] *= np.float32(2.0**60)
    got = []
    assert any(x.startswith("zk_split_") for x in used(ctx, lambda: got.append(product(ctx, L, R, lt, rt))))
    ref = L.astype(np.float64) @ R.astype(np.float64)
    # Element (i, j) in units of |L_i| |R_j| / sqrt(k), its typical size; results
    # below 2^-126 are themselves rounded to 2^-149.
    unit = np.linalg.norm(L.astype(np.float64), axis=1)[:, None] * np.linalg.norm(R.astype(np.float64), axis=0) / np.sqrt(k)
    e = np.maximum(np.abs(got[0] - ref) - 2.0**-149, 0.0) / unit
    rms = [np.sqrt(np.mean(e * e, axis=axis)).max() for axis in (0, 1)]
    print(f"[gpu] split gemm {what} {lt} {rt}: worst rms of a column {rms[0]:.1e}, of a row {rms[1]:.1e}", flush=True)
    assert max(rms) <= 1e-6


@pytest.mark.parametrize("rows", [12288, 12301])
def test_split_gemm_network(ctx, fp32_ctx, rows):
    """Forward (both accumulator forms), data and weight gradients of a
    network at whole and ragged row counts: the output and every gradient
    tensor as close to float64 as on the fp32 kernels."""
    from zealot_amd.rl import GpuMlp, unpack

    dims = [123, 512, 256, 128, 29]
    g = np.random.default_rng(rows)
    packed = synth.kaiming_uniform_net(g, dims, 0.1)
    x, gout = synth.normal(g, (rows, 123)), synth.normal(g, (rows, 29))
    out = []
    for c in (ctx, fp32_ctx):
        mlp = GpuMlp(c, dims, rows + 100)
        mlp.write_weights(packed)
        dx, dg = c.to_device(x), c.to_device(gout)

        def go():
            mlp.forward(dx, rows)
            mlp.backward(dg)

        names = used(c, go)
        if c is ctx:
            want = {"zk_split_ak_bk_s", "zk_split_ak_bk_acc2", "zk_split_ak_bn_dg", "zk_split_am_bn"}
            assert want <= set(names), names
        out.append((mlp.output(rows), mlp.read_grads()))
        mlp.close()
    ws, bs = unpack(dims, packed.astype(np.float64))
    acts = [x.astype(np.float64)]
    for i, (w, b) in enumerate(zip(ws, bs)):
        z = acts[-1] @ w.T + b
        acts.append(np.where(z > 0, z, np.expm1(np.minimum(z, 0))) if i < 3 else z)
    d, parts = gout.astype(np.float64), []
    for i in range(3, -1, -1):
        parts = [(d.T @ acts[i]).ravel(), d.sum(0)] + parts
        if i:
            d = (d @ ws[i]) * np.where(acts[i] > 0, 1.0, acts[i] + 1.0)
    as_exact_as_fp32(out[0][0], out[1][0], acts[-1], f"network output, {rows} rows")
    o = 0
    for i, p in enumerate(parts):
        tag = f"network {rows} rows, layer {i // 2} {'bias' if i % 2 else 'weight'} gradient"
        as_exact_as_fp32(out[0][1][o:o + p.size], out[1][1][o:o + p.size], p, tag)
        o += p.size


@pytest.mark.parametrize("n", [384, 3001, 24576])
def test_minibatch_forward_stays_fp32(ctx, fp32_ctx, n):
    """The surrogate of a minibatch is a mean of signed terms that nearly
    cancel: its forward stays on the fp32 kernels, so every statistic and the
    log_std gradient have the bits of a context without three-piece GEMMs; the
    weight gradients, which may take them, agree to rounding."""
    from zealot_amd.rl import DeviceBatch, GpuActorCritic, PpoConfig

    ad, cd = [123, 512, 256, 128, 29], [123, 512, 256, 128, 1]
    g = np.random.default_rng(n)
    actor, critic = synth.kaiming_uniform_net(g, ad, 0.1), synth.kaiming_uniform_net(g, cd, 0.1)
    obs = synth.obs(g, n, 123)
    args = [obs, obs, synth.normal(g, (n, 29)), synth.normal(g, (n, 29)), synth.normal(g, n) - 60, synth.normal(g, n),
            synth.normal(g, n), synth.normal(g, n)]
    out = []
    for c in (ctx, fp32_ctx):
        gac = GpuActorCritic(c, ad, cd, n)
        gac.set_params(actor, critic, np.full(29, -0.5, np.float32), 1e-4)
        db = DeviceBatch(c, *args)
        names = used(c, lambda: out.append(gac.minibatch_grads(db, PpoConfig(), 0, n)))
        assert not any(x.startswith("zk_split_ak_bk") for x in names), names
        assert any(x.startswith("zk_split_") for x in names) == (c is ctx), names
        gac.close()
    (ga, gc, gl, st), (ra, rc, rl, rst) = out
    assert st == rst and np.array_equal(gl, rl)
    for a, b in ((ga, ra), (gc, rc)):
        assert np.linalg.norm(a - b) <= 2e-6 * np.linalg.norm(b)


def test_split_gemm_gathered_rows(ctx):
    """A shuffled minibatch of a ragged number of rows (the observation gather
    inside the first layer's forward and weight gradient): the same rows in
    another order, so the first Adam moments agree to the rounding of a sum."""
    from zealot_amd.rl import DeviceBatch, GpuActorCritic, PpoConfig

    ad, cd = [64, 512, 256, 128, 12], [64, 512, 256, 128, 1]
    n = 13001
    g = np.random.default_rng(9)
    actor, critic = synth.kaiming_uniform_net(g, ad, 0.1), synth.kaiming_uniform_net(g, cd, 0.1)
    obs = synth.obs(g, n, 64)
    args = [obs, obs, synth.normal(g, (n, 12)), synth.normal(g, (n, 12)), synth.normal(g, n) - 20, synth.normal(g, n),
            synth.normal(g, n), synth.normal(g, n)]
    out = []
    for shuffle in (True, False):
        gac = GpuActorCritic(ctx, ad, cd, n)
        gac.set_params(actor, critic, np.full(12, -0.5, np.float32), 1e-4)
        db = DeviceBatch(ctx, *args)
        gac.update(db, PpoConfig(epochs=1, minibatches=1, shuffle=shuffle, normalize_adv=False))
        out.append(gac.get_moments())
        gac.close()
    for i in (0, 2, 4):
        a, b = out[0][i], out[1][i]
        assert np.any(b != 0)
        assert np.max(np.abs(a - b)) <= 1e-5 * np.max(np.abs(b)), i


# (m, n, k, slices): weight gradients of short batches: no slice, one k-tile more
# than a slice pair, the slice cap, one row past it; 64-, 96- and 128-wide tiles.
@pytest.mark.parametrize("m,n,k,slices", [(512, 128, 96, 1), (512, 128, 129, 2), (256, 288, 384, 6), (512, 64, 385, 5),
                                          (128, 256, 960, 15), (128, 128, 4096, 64), (128, 128, 4097, 43),
                                          (100, 124, 700, 11)])
def test_short_reductions_are_sliced(ctx, fp32_ctx, m, n, k, slices):
    g = np.random.default_rng(m + n + k)
    L, R = synth.normal(g, (m, k)), synth.normal(g, (k, n))
    got, shapes = [], []
    names = used(ctx, lambda: got.append(product(ctx, L, R, True, False)), shapes)
    assert names[1:] == ["zk_splitk_reduce"] * (slices > 1) and shapes[0] == (m, n, k, slices)
    ref = L.astype(np.float64) @ R.astype(np.float64)
    bound = (6 * (-(-k // 16)) + 104) * 2.0 ** -24 * (np.abs(L).astype(np.float64) @ np.abs(R).astype(np.float64))
    bound = np.maximum(bound, k * 2.0 ** -24 * (np.abs(L).astype(np.float64) @ np.abs(R).astype(np.float64)))
    assert np.all(np.abs(got[0] - ref) <= bound)
    as_exact_as_fp32(got[0], product(fp32_ctx, L, R, True, False), ref, (m, n, k))
