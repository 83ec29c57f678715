"""f32 attention and its gradients on the bf16 matrix cores, operands as three bf16 terms: sizes whose launches take that kernel (many rows),
at the edges of its 128-row workgroups and 32-key tiles, and values the split does not carry.

The bound against 64 bits is 1e-6 of the result's 2-norm: an f32 product of these sizes rounds each of up to 384 / 32 tile sums
and each weight once, about 2^-24 sqrt(20) = 2.7e-7; the f32 kernel it stands in for shows up to 4e-7 here."""
import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import dev, with_common_offset
from _util import seeded_normal

pytestmark = pytest.mark.gpu


# on the other side of the rule's line, some of them under one mask only: the f32 matrix cores, to the same bound
BESIDE = [(13, 20, 161, 36), (16, 16, 130, 64), (9, 16, 225, 80)]


def assert_split(b, h, n, d, causal=False, seq_kv=0, with_lse=False):
    """The launch takes the kernels this file is about."""
    assert ra.debug_f32_split_products(ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none(), seq_kv,
                                       with_lse)


def run(q, k, v, causal):
    b, h, n, d = q.shape
    out = ra.HipStorage(q.size * 4)
    out.upload(np.full(q.size, 7.0, dtype=np.float32))
    mask = ra.Mask.causal() if causal else ra.Mask.none()
    ra.flash_forward_f32_dev(ra.AttentionShape.new(b, h, n, d), dev(q.ravel()), dev(k.ravel()), dev(v.ravel()), out, mask)
    ra.synchronize()
    return out.download(np.float32).reshape(q.shape)


def attention64(q, k, v, causal):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    with np.errstate(all="ignore"):
        s = q @ np.swapaxes(k, -1, -2) / np.sqrt(q.shape[-1])
        if causal:
            n = q.shape[2]
            s = np.where(np.tril(np.ones((n, n), dtype=bool)), s, -np.inf)
        p = np.exp(s - s.max(axis=-1, keepdims=True))
        return (p / p.sum(axis=-1, keepdims=True)) @ v


def inputs(b, h, n, d):
    return [seeded_normal((b, h, n, d), i).reshape(b, h, n, d) for i in (1, 2, 3)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,n,d", [
    (8, 16, 256, 64),   # whole tiles
    (8, 16, 225, 60),   # 31 keys of the last tile missing, head dim padded
    (9, 14, 417, 36),   # one row in a workgroup's second wave, head pairs not a multiple of eight
    (8, 32, 384, 32),   # head dim 32: half the threads split
    (8, 16, 386, 64),   # two rows in the last workgroup
    (8, 16, 256, 128),
    (8, 32, 353, 96),   # three blocks of rows, two a workgroup where causal
    (8, 16, 225, 80),
    (8, 32, 353, 68),
    *BESIDE,
])
def test_against_64_bits(b, h, n, d, causal):
    q, k, v = inputs(b, h, n, d)
    got = run(q, k, v, causal)
    want = attention64(q, k, v, causal)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 5e-6


@pytest.mark.parametrize("what", ["key inf", "value inf", "query nan", "value nan", "large"])
def test_values_the_split_does_not_carry(what):
    """Rows they reach are what f32 arithmetic makes of them; the rest are as they were."""
    b, h, n, d = 8, 16, 256, 64
    q, k, v = inputs(b, h, n, d)
    want = attention64(q, k, v, True)
    at = (3, 5)
    if what == "key inf":
        q[at][:, 9] = -np.abs(q[at][:, 9]) - 0.1  # every query's score of key 40 is -inf: its weight is zero
        k[at][40, 9] = np.inf
    elif what == "value inf":
        v[at][200, 1] = np.inf
    elif what == "query nan":
        q[at][17, 3] = np.nan
    elif what == "value nan":
        v[at][255, 63] = np.nan
    else:
        q[at][100] = 1e25
        k[at][100] = 1e25  # row 100 sees its own key only; the products pass the f32 range
        k[at][100, 1::2] = -1e10
    got = run(q, k, v, True)
    other = np.ones((b, h), dtype=bool)
    other[at] = False
    assert np.abs(got[other] - want[other]).max() <= 5e-6
    with np.errstate(all="ignore"):
        slab = got[at]
        if what == "key inf":
            ref = attention64(q[3:4, 5:6], k[3:4, 5:6], v[3:4, 5:6], True)[0, 0]
            assert np.abs(slab - ref).max() <= 5e-6
        elif what == "value inf":
            assert np.isposinf(slab[200:, 1]).all() and np.isfinite(slab[:, 2:]).all()
        elif what == "query nan":
            assert np.isnan(slab[17]).all() and np.isfinite(np.delete(slab, 17, axis=0)).all()
        elif what == "value nan":
            assert np.isnan(slab[255, 63]) and np.isfinite(slab[:255, :63]).all()
        else:
            assert np.isfinite(slab[:100]).all() and np.abs(slab[:100] - want[at][:100]).max() <= 5e-6


@pytest.mark.parametrize("b,h,n,d", [(8, 16, 256, 64), (8, 32, 384, 32), (8, 32, 353, 96), (8, 16, 256, 128)])
@pytest.mark.parametrize("at", [3, -1])
def test_an_infinite_key_seen_at_once_or_at_the_end(b, h, n, d, at):
    """In the first tile or the last, with one block of rows a workgroup or two: every query's score of that key is -inf,
    so its weight is zero and the rows are those of the other keys."""
    q, k, v = inputs(b, h, n, d)
    q[2, 7, :, 9] = -np.abs(q[2, 7, :, 9]) - 0.1
    k[2, 7, at, 9] = np.inf
    for causal in (False, True):
        got, want = run(q, k, v, causal), attention64(q, k, v, causal)
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
        assert np.abs(got - want).max() <= 5e-6


def test_what_such_values_cost():
    """A NaN in every head goes the way of any value; an infinity in every head costs the f32 products beside the others'
    (measured 1.5 and 1.4 times a clean launch where the first tiles show it, 2.3 and 1.7 where the last does)."""
    import time

    b, h, n, d = 4, 16, 1024, 64
    shape = ra.AttentionShape.new(b, h, n, d)
    clean = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    out, lse, ws = ra.HipStorage(b * h * n * d * 4), ra.HipStorage(b * h * n * 4), ra.HipStorage(b * h * n * 4)
    grads = [ra.HipStorage(b * h * n * d * 4) for _ in range(3)]

    def seconds(value, at):
        x = [a.copy() for a in clean]
        if value is not None:
            x[1][:, :, at, 3] = value
        x = [dev(a.ravel()) for a in x]
        best = [1e9, 1e9]
        for _ in range(5):
            for i, call in enumerate((lambda: ra.flash_forward_stats_f32_dev(shape, *x[:3], out, lse),
                                      lambda: ra.flash_backward_saved_f32_dev(shape, *x[:3], out, lse, x[3], *grads, ws, b * h * n * 4))):
                ra.synchronize()
                start = time.perf_counter()
                for _ in range(10):
                    call()
                ra.synchronize()
                best[i] = min(best[i], time.perf_counter() - start)
        return np.asarray(best)

    usual = seconds(None, 0)
    assert (seconds(np.nan, 5) <= 1.3 * usual).all()
    assert (seconds(np.inf, 5) <= 2.2 * usual).all()
    assert (seconds(np.inf, n - 1) <= 3.2 * usual).all()


def test_small_values():
    """V rows of 2^-120: the last of three bf16 terms would be lost."""
    q, k, v = inputs(8, 16, 256, 64)
    v[2, 7] *= np.float32(2.0 ** -120)
    got, want = run(q, k, v, False), attention64(q, k, v, False)
    assert np.linalg.norm(got[2, 7].astype(np.float64) - want[2, 7]) <= 1e-6 * np.linalg.norm(want[2, 7])
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,n,d", [(8, 16, 256, 64), (8, 32, 353, 32), (8, 16, 256, 128), (8, 16, 225, 60), (1, 2, 300, 64), (1, 8, 257, 20)])
def test_a_small_value_of_v_among_others(b, h, n, d, causal):
    """A subnormal in V leaves the split products to every row whose results are not small themselves: the other columns have
    the bits they have with a zero in its place.  Under the causal mask row 0 is V's first, and its workgroup goes the f32 way."""
    q, k, v = inputs(b, h, n, d)
    rows = 128 if ra.debug_f32_split_products(ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none()) else 32
    col = d // 3
    others = np.arange(d) != col
    for key, value in ((0, 2.0 ** -110 * (1 + 2.0 ** -23)), (n // 2, 1e-40), (n - 1, 1e-40)):
        usual = v[0, 1, key, col]
        v[0, 1, key, col] = value
        got, want = run(q, k, v, causal), attention64(q, k, v, causal)
        v[0, 1, key, col] = 0.0
        zero = run(q, k, v, causal)
        v[0, 1, key, col] = usual
        first = rows if causal and key == 0 else 0
        assert np.array_equal(got[0, 1, first:, others], zero[0, 1, first:, others])
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
        if first:
            assert got[0, 1, 0, col] == np.float32(value)


@pytest.mark.parametrize("d", [32, 64, 128])
def test_small_columns_of_v(d):
    """One column small throughout beside others of the usual size: its results keep their precision."""
    q, k, v = inputs(8, 16, 256, d)
    v[2, 7, :, 5] *= np.float32(2.0 ** -115)
    for causal in (False, True):
        got, want = run(q, k, v, causal)[2, 7].astype(np.float64), attention64(q, k, v, causal)[2, 7]
        assert np.linalg.norm((got - want)[:, 5]) <= 1e-6 * np.linalg.norm(want[:, 5])
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


def run_backward(q, k, v, d_out):
    b, h, n, d = q.shape
    shape = ra.AttentionShape.new(b, h, n, d)
    dq_, dk_, dv_, dd = (dev(x.ravel()) for x in (q, k, v, d_out))
    out, lse, ws = ra.HipStorage(q.size * 4), ra.HipStorage(b * h * n * 4), ra.HipStorage(b * h * n * 4)
    grads = [ra.HipStorage(q.size * 4) for _ in range(3)]
    for g in grads:
        g.upload(np.full(q.size, 7.0, dtype=np.float32))
    ra.flash_forward_stats_f32_dev(shape, dq_, dk_, dv_, out, lse)
    ra.flash_backward_saved_f32_dev(shape, dq_, dk_, dv_, out, lse, dd, *grads, ws, b * h * n * 4)
    ra.synchronize()
    return [g.download(np.float32).reshape(q.shape) for g in grads]


def gradients64(q, k, v, d_out):
    q, k, v, d_out = (x.astype(np.float64) for x in (q, k, v, d_out))
    scale = 1 / np.sqrt(q.shape[-1])
    with np.errstate(all="ignore"):
        s = q @ np.swapaxes(k, -1, -2) * scale
        p = np.exp(s - s.max(axis=-1, keepdims=True))
        p /= p.sum(axis=-1, keepdims=True)
        dp = d_out @ np.swapaxes(v, -1, -2)
        ds = p * (dp - (p * dp).sum(axis=-1, keepdims=True)) * scale
        return ds @ k, np.swapaxes(ds, -1, -2) @ q, np.swapaxes(p, -1, -2) @ d_out


@pytest.mark.parametrize("b,h,n,d", [
    (8, 16, 256, 64),
    (8, 16, 225, 60),
    (8, 32, 353, 32),   # one row in the last tile, head dim 32
    (8, 28, 481, 36),   # head pairs not a multiple of the XCDs' share, padded head dim
    (8, 16, 386, 64),   # two rows in the last workgroup
    (16, 16, 130, 64),
])
def test_gradients_against_64_bits(b, h, n, d):
    """The bound is the forward's times two: dS carries the errors of P and of dP - delta."""
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    for name, got, want in zip(("dq", "dk", "dv"), run_backward(*x), gradients64(*x)):
        assert np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want), name


@pytest.mark.parametrize("what", ["key inf", "d_out nan", "query nan", "small"])
def test_gradients_of_values_the_split_does_not_carry(what):
    """Only the head that holds them changes: by the rules of f32 arithmetic, or, for small ones, not in precision."""
    b, h, n, d = 8, 16, 256, 64
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    q, k, v, d_out = x
    at = (3, 5)
    if what == "key inf":
        q[at][:, 9] = -np.abs(q[at][:, 9]) - 0.1
        k[at][40, 9] = np.inf
    elif what == "d_out nan":
        d_out[at][17, 3] = np.nan
    elif what == "query nan":
        q[at][17, 3] = np.nan
    else:
        d_out[at] *= np.float32(2.0 ** -115)
    got, want = run_backward(*x), gradients64(*x)
    other = np.ones((b, h), dtype=bool)
    other[at] = False
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        assert np.linalg.norm(g[other] - w[other]) <= 2e-6 * np.linalg.norm(w[other]), name
        gs, ws = g[at].astype(np.float64), w[at]
        if what == "small":
            assert np.linalg.norm(gs - ws) <= 2e-6 * np.linalg.norm(ws), name
        else:
            fin = np.isfinite(ws)
            assert np.array_equal(np.isnan(gs), np.isnan(ws)), name
            assert not fin.any() or np.linalg.norm((gs - ws)[fin]) <= 2e-6 * np.linalg.norm(ws[fin]), name


def shapes_of(test):
    return next(m.args[1] for m in test.pytestmark if m.name == "parametrize" and m.args[0] == "b,h,n,d")


def test_the_shapes_of_this_file_take_these_kernels():
    for shape in shapes_of(test_against_64_bits):
        if shape not in BESIDE:
            assert_split(*shape)
            assert_split(*shape, causal=True)
    for shape in shapes_of(test_gradients_against_64_bits):
        if shape not in BESIDE:
            assert_split(*shape, with_lse=True)
    for b, h, n, d in BESIDE:
        assert not ra.debug_f32_split_products(ra.AttentionShape.new(b, h, n, d), ra.Mask.causal())


def bnhd(x):
    return np.ascontiguousarray(np.swapaxes(x, 1, 2))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,hkv,n,d", [
    (8, 16, 16, 225, 60),
    (8, 16, 4, 256, 64),
    (9, 14, 7, 417, 36),   # head pairs not a multiple of eight, padded head dim
    (8, 32, 1, 384, 32),   # one kv head for all
    (8, 32, 8, 353, 96),   # two blocks of rows a workgroup where causal
    (8, 16, 8, 225, 128),
])
def test_grouped_heads_and_rows_apart(b, h, hkv, n, d, causal):
    """kv heads that serve groups, and [batch, seq, heads, dim] tensors, against 64 bits; both layouts give the same bits."""
    assert_split(b, h, n, d, causal)
    q = seeded_normal((b, h, n, d), 1).reshape(b, h, n, d)
    k, v = (seeded_normal((b, hkv, n, d), i).reshape(b, hkv, n, d) for i in (2, 3))
    want = attention64(q, np.repeat(k, h // hkv, axis=1), np.repeat(v, h // hkv, axis=1), causal)
    shape, mask = ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none()
    got = []
    for layout, call in ((np.ascontiguousarray, ra.flash_forward_f32_dev), (bnhd, ra.flash_forward_bnhd_f32_dev)):
        out = ra.HipStorage(q.size * 4)
        out.upload(np.full(q.size, 7.0, dtype=np.float32))
        call(shape, dev(layout(q)), dev(layout(k)), dev(layout(v)), out, mask, n_kv_heads=hkv)
        ra.synchronize()
        got.append(layout(out.download(np.float32).reshape(layout(q).shape)))
    assert np.linalg.norm(got[0] - want) <= 1e-6 * np.linalg.norm(want)
    assert np.abs(got[0] - want).max() <= 5e-6
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("b,h,hkv,t_q,t_kv,d", [
    (8, 16, 16, 256, 300, 64),
    (8, 16, 16, 225, 31, 60),    # one ragged tile of keys
    (12, 21, 21, 161, 513, 36),
    (8, 32, 32, 353, 97, 96),
    (8, 16, 4, 225, 257, 128),   # kv heads that serve groups (the grouped entry)
    (8, 32, 8, 384, 33, 32),
])
def test_keys_of_another_length(b, h, hkv, t_q, t_kv, d):
    assert_split(b, h, t_q, d, seq_kv=t_kv)
    q = seeded_normal((b, h, t_q, d), 1).reshape(b, h, t_q, d)
    k, v = (seeded_normal((b, hkv, t_kv, d), i).reshape(b, hkv, t_kv, d) for i in (2, 3))
    want = attention64(q, np.repeat(k, h // hkv, axis=1), np.repeat(v, h // hkv, axis=1), False)
    out = ra.HipStorage(q.size * 4)
    out.upload(np.full(q.size, 7.0, dtype=np.float32))
    if hkv == h:
        ra.mha_forward_masked_f32_dev(dev(bnhd(q)), dev(bnhd(k)), dev(bnhd(v)), out, b, t_q, t_kv, h, d)
        ra.synchronize()
        got = bnhd(out.download(np.float32).reshape(b, t_q, h, d))
    else:
        ra.gqa_forward_f32_dev(dev(q), dev(k), dev(v), out, b, h, hkv, t_q, t_kv, d)
        ra.synchronize()
        got = out.download(np.float32).reshape(q.shape)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 5e-6


def test_the_rule_turns_away_what_the_kernels_do_not_take():
    """Padding masks, head dims that are no multiple of 4 or above 128 (64 with the row statistic), and few rows."""
    big = ra.AttentionShape.new
    assert not ra.debug_f32_split_products(big(8, 16, 256, 64), ra.Mask.padding(np.ones(256, dtype=bool)))
    for d, with_lse in ((62, False), (132, False), (256, False), (68, True), (128, True)):
        assert not ra.debug_f32_split_products(big(8, 16, 1024, d), with_lse=with_lse)
    assert not ra.debug_f32_split_products(big(1, 1, 64, 64))


# ---- few rows: workgroups of 32 whose waves share the keys


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("d", [4, 20, 32, 36, 60, 64])
@pytest.mark.parametrize("b,h,n", [(1, 1, 129), (1, 8, 160), (2, 3, 161), (1, 4, 255), (1, 8, 257), (1, 2, 500), (3, 1, 513)])
def test_few_rows_against_64_bits(b, h, n, d, causal):
    """One to five tiles a wave, the last one with 1, 31 and 32 keys, head dims that fill the 32 or 64 columns and do not."""
    assert not ra.debug_f32_split_products(ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none())
    q, k, v = inputs(b, h, n, d)
    got, want = run(q, k, v, causal), attention64(q, k, v, causal)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
    assert np.abs(got - want).max() <= 5e-6


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,hkv,n,d", [(8, 2, 200, 64), (4, 1, 333, 20), (6, 3, 161, 32)])
def test_few_rows_of_grouped_heads_and_rows_apart(h, hkv, n, d, causal):
    """What lies behind a head's columns in a [batch, seq, heads, dim] row is another head's, here NaN."""
    b = 2
    q = seeded_normal((b, h, n, d), 1).reshape(b, h, n, d)
    k, v = (seeded_normal((b, hkv, n, d), i).reshape(b, hkv, n, d) for i in (2, 3))
    if hkv > 1:
        k[:, 1], v[:, 1] = np.nan, np.nan
    want = attention64(q, np.repeat(k, h // hkv, axis=1), np.repeat(v, h // hkv, axis=1), causal)
    shape, mask = ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none()
    got = []
    for layout, call in ((np.ascontiguousarray, ra.flash_forward_f32_dev), (bnhd, ra.flash_forward_bnhd_f32_dev)):
        out = ra.HipStorage(q.size * 4)
        call(shape, dev(layout(q)), dev(layout(k)), dev(layout(v)), out, mask, n_kv_heads=hkv)
        ra.synchronize()
        got.append(layout(out.download(np.float32).reshape(layout(q).shape)))
    assert np.array_equal(got[0], got[1], equal_nan=True)
    assert np.array_equal(np.isnan(got[0]), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.linalg.norm((got[0] - want)[ok]) <= 1e-6 * np.linalg.norm(want[ok])


@pytest.mark.parametrize("t_q,t_kv,d", [(1, 300, 64), (33, 129, 60), (70, 1000, 32)])
def test_few_rows_keys_of_another_length(t_q, t_kv, d):
    b, h = 2, 3
    q = seeded_normal((b, h, t_q, d), 1).reshape(b, h, t_q, d)
    k, v = (seeded_normal((b, h, t_kv, d), i).reshape(b, h, t_kv, d) for i in (2, 3))
    out = ra.HipStorage(q.size * 4)
    ra.mha_forward_masked_f32_dev(dev(bnhd(q)), dev(bnhd(k)), dev(bnhd(v)), out, b, t_q, t_kv, h, d)
    ra.synchronize()
    got, want = bnhd(out.download(np.float32).reshape(b, t_q, h, d)), attention64(q, k, v, False)
    assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,n,d", [(1, 2, 300, 64), (1, 4, 500, 20), (8, 16, 256, 64), (8, 32, 353, 32), (8, 16, 256, 128)])
@pytest.mark.parametrize("q_times,offset", [(2.5, 0.0), (8.0, 0.0), (1.0, 130.0), (3.5, 130.0)])
def test_scores_of_any_size(b, h, n, d, causal, q_times, offset):
    """Waves whose keys' maxima lie far apart, and scores that all lie near -130.  A scaled score is off by about eight
    roundings at the size of its products' magnitudes together, a weight by that share of itself, and a result by twice
    that (numerator and row sum) of the attention over |V|; 2^-20 for everything else."""
    q, k, v = inputs(b, h, n, d)
    q *= np.float32(q_times)
    if offset:
        q, k = with_common_offset(q, k, d, offset)
    got, want = run(q, k, v, causal), attention64(q, k, v, causal)
    sizes = attention64(q, k, np.abs(v), causal)
    scores = (np.abs(q).astype(np.float64) @ np.swapaxes(np.abs(k), -1, -2).astype(np.float64)).max(axis=-1, keepdims=True) / np.sqrt(d)
    assert (np.abs(got - want) <= (2 * 8 * 2.0 ** -24 * scores + 2.0 ** -20) * sizes).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("what", ["q inf", "k inf", "v inf", "q nan", "k nan", "v nan", "k large", "v small", "v zero"])
def test_few_rows_what_the_split_does_not_carry(what, causal):
    """Infinities, values from 2^30 on and values of V below 2^-100 send the workgroups that read them to the f32 products; NaN
    is carried.  Zeros are neither small nor large."""
    b, h, n, d = 1, 2, 300, 64
    q, k, v = inputs(b, h, n, d)
    x = {"q": q, "k": k, "v": v}[what[0]]
    value = {"inf": np.inf, "nan": np.nan, "large": np.float32(2.0) ** 40, "small": np.float32(1e-33), "zero": 0.0}[what.split()[1]]
    if what[2:] in ("small", "zero"):
        x[0, 0] = value
    else:
        x[0, 1, 37, 5] = value
    got = run(q, k, v, causal)
    want = attention64(q, k, v, causal)
    if what == "v small":
        assert np.linalg.norm(got[0, 0].astype(np.float64) - want[0, 0]) <= 1e-6 * np.linalg.norm(want[0, 0])
    if what in ("v inf", "v nan") and causal:  # rows of the tile that do not see the key: zero times its value, as in every f32 kernel
        assert np.isfinite(got[0, 1, 64:, :5]).all() and not np.isfinite(got[0, 1, 37:, 5]).any()
        return
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = np.isfinite(want)
    assert np.abs(got - want)[ok].max() <= 5e-6


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("b,h,hkv,n,d", [
    (1, 1, 1, 129, 96),    # one key in the second tile of the first wave
    (1, 1, 1, 225, 128),   # one key in the eighth tile
    (1, 8, 8, 161, 96),    # rows of 24 slots in LDS
    (2, 4, 1, 333, 68),    # grouped heads, the least of the padded columns
    (1, 4, 2, 257, 100),
    (1, 8, 8, 545, 80),    # three tiles a wave, then five
    (2, 8, 8, 640, 128),   # more workgroups than CUs
])
def test_few_rows_above_head_dim_64(b, h, hkv, n, d, causal):
    """The edges of tiles and of the padded columns, both layouts (what lies behind a head's columns there is another head's)."""
    assert not ra.debug_f32_split_products(ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none())
    q = seeded_normal((b, h, n, d), 1).reshape(b, h, n, d)
    k, v = (seeded_normal((b, hkv, n, d), i).reshape(b, hkv, n, d) for i in (2, 3))
    want = attention64(q, np.repeat(k, h // hkv, axis=1), np.repeat(v, h // hkv, axis=1), causal)
    shape, mask = ra.AttentionShape.new(b, h, n, d), ra.Mask.causal() if causal else ra.Mask.none()
    got = []
    for layout, call in ((np.ascontiguousarray, ra.flash_forward_f32_dev), (bnhd, ra.flash_forward_bnhd_f32_dev)):
        out = ra.HipStorage(q.size * 4)
        out.upload(np.full(q.size, 7.0, dtype=np.float32))
        call(shape, dev(layout(q)), dev(layout(k)), dev(layout(v)), out, mask, n_kv_heads=hkv)
        ra.synchronize()
        got.append(layout(out.download(np.float32).reshape(layout(q).shape)))
    assert np.array_equal(got[0], got[1])
    assert np.linalg.norm(got[0] - want) <= 1e-6 * np.linalg.norm(want)
    assert np.abs(got[0] - want).max() <= 5e-6


@pytest.mark.parametrize("d", [96, 128])
@pytest.mark.parametrize("what", ["k inf", "v inf", "q nan", "v small"])
def test_few_rows_above_head_dim_64_what_the_split_does_not_carry(what, d):
    """The second pass in f32 out of tiles of these widths: rows that see the value are what 64 bits make of them, the rest as they were."""
    q, k, v = inputs(1, 2, 300, d)
    x = {"q": q, "k": k, "v": v}[what[0]]
    if what == "v small":
        x[0, 0] = np.float32(1e-33)
    else:
        x[0, 1, 0 if what == "v inf" else 37, d - 1] = np.inf if what[2:] == "inf" else np.nan  # (every row sees key 0)
    got, want = run(q, k, v, True), attention64(q, k, v, True)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    for head in range(2):
        ok = np.isfinite(want[0, head])
        err = np.linalg.norm((got[0, head].astype(np.float64) - want[0, head])[ok])
        assert err <= 1e-6 * np.linalg.norm(want[0, head][ok])


# ---- gradients above head dim 64: dK and dV in workgroups of their own

WIDE = [
    (2, 8, 300, 96),    # all three in one launch, the last tile of 12 rows, the last workgroup of 44
    (4, 8, 225, 68),    # one row in the last tile, most of the third column block empty
    (2, 8, 640, 128),   # whole tiles
    (6, 16, 200, 128),  # one launch of more workgroups than CUs
    (4, 16, 453, 80),   # dQ ahead of dK and dV
    (8, 17, 257, 100),  # head pairs not a multiple of eight, one row in the last workgroup
    (8, 16, 128, 96),   # four tiles
    (1, 8, 3, 68),      # a few rows
    (1, 8, 18, 96),     # one tile: no step has a next one
    (4, 8, 32, 80),
    (16, 16, 33, 128),  # two, the last of a row, dQ ahead of dK and dV
    (5, 17, 64, 96),    # two, all three in one launch
    (16, 16, 64, 96),
    (5, 17, 95, 100),   # three
    (16, 16, 96, 128),
]
NOT_WIDE = [(8, 16, 32, 96), (1, 8, 64, 96), (4, 8, 96, 128), (16, 16, 32, 128), (1, 8, 250, 96), (8, 16, 64, 128)]


def test_the_rule_of_the_wide_gradients():
    """On a device of 256 compute units."""
    for shapes, wide in ((WIDE + [(8, 16, 200, 128)], True), (NOT_WIDE, False)):
        for b, h, n, d in shapes:
            assert ra.debug_f32_wide_gradients(ra.AttentionShape.new(b, h, n, d)) == wide, (b, h, n, d)
    for d in (64, 66, 130, 132, 256):
        assert not ra.debug_f32_wide_gradients(ra.AttentionShape.new(4, 16, 1024, d))


@pytest.mark.parametrize("b,h,n,d", NOT_WIDE)
def test_few_tiles_stay_with_the_f32_gradients(b, h, n, d):
    test_wide_gradients_against_64_bits(b, h, n, d)


@pytest.mark.parametrize("b,h,n,d", WIDE)
def test_wide_gradients_against_64_bits(b, h, n, d):
    """The bound of test_gradients_against_64_bits."""
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    got = run_backward(*x)
    for name, g, w in zip(("dq", "dk", "dv"), got, gradients64(*x)):
        assert np.linalg.norm(g - w) <= 2e-6 * np.linalg.norm(w), name
    for g, again in zip(got, run_backward(*x)):
        assert np.array_equal(g, again)


@pytest.mark.parametrize("b,h,n,d", [(2, 8, 300, 96), (8, 16, 200, 128)])
@pytest.mark.parametrize("what", ["key inf", "value inf", "d_out nan", "query nan", "small"])
def test_wide_gradients_of_values_the_split_does_not_carry(b, h, n, d, what):
    """Only the head that holds them changes, and its workgroups that read them do their rows once more in f32."""
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    q, k, v, d_out = x
    at = (1, 5)
    if what == "key inf":
        q[at][:, 9] = -np.abs(q[at][:, 9]) - 0.1
        k[at][n - 1, 9] = np.inf
    elif what == "value inf":
        v[at][40, 9] = np.inf
    elif what == "d_out nan":
        d_out[at][17, 3] = np.nan
    elif what == "query nan":
        q[at][17, 3] = np.nan
    else:
        d_out[at] *= np.float32(2.0 ** -115)
    got, want = run_backward(*x), gradients64(*x)
    other = np.ones((b, h), dtype=bool)
    other[at] = False
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        assert np.linalg.norm(g[other] - w[other]) <= 2e-6 * np.linalg.norm(w[other]), name
        gs, ws = g[at].astype(np.float64), w[at]
        fin = np.isfinite(ws)
        assert np.array_equal(np.isfinite(gs), fin), name
        assert not fin.any() or np.linalg.norm((gs - ws)[fin]) <= 2e-6 * np.linalg.norm(ws[fin]), name


@pytest.mark.parametrize("b,h,n,d", [(2, 8, 300, 96), (8, 16, 200, 128)])
def test_wide_gradients_of_a_key_that_no_query_weighs(b, h, n, d):
    """Every weight of the key is about e^-85 = 2^-123, as f32 has it: its rows of dK and dV hold what f32 makes of them.  The weights' error
    is that of the exponent, a difference of f32 values of 85 (a score that is rounded twice, the statistic, their difference and the
    product with log2 e: 5 x 2^-18 of the weight); three bf16 terms of a weight that small leave out up to 2^-11 of it."""
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    q, k, v, d_out = x
    at, key = (1, 5), 40
    q[at][:, 9], k[at][:, 9] = 4.0, 0.0
    k[at][key] = 0.0
    k[at][key, 9] = np.float32(-79.0 * np.sqrt(d) / 4.0)
    got, want = run_backward(*x), gradients64(*x)
    for name, g, w in zip(("dq", "dk", "dv"), got, want):
        assert np.linalg.norm(g - w) <= 2e-6 * np.linalg.norm(w), name
        if name == "dq":
            continue
        row, wrow = g[at][key].astype(np.float64), w[at][key]
        assert 2.0 ** -126 < np.abs(wrow).max() < 2.0 ** -110
        assert np.linalg.norm(row - wrow) <= 5 * 2.0 ** -18 * np.linalg.norm(wrow), name


@pytest.mark.parametrize("over", ["dk k", "dk v, dv k", "dq out", "dv k"])
def test_wide_gradients_over_what_they_read(over):
    """Tensors that share memory take the f32 kernels, one behind the other."""
    b, h, n, d = 2, 8, 300, 96
    x = inputs(b, h, n, d) + [seeded_normal((b, h, n, d), 4).reshape(b, h, n, d)]
    shape = ra.AttentionShape.new(b, h, n, d)
    t = dict(zip(("q", "k", "v", "d_out"), (dev(y.ravel()) for y in x)))
    t["out"], lse, ws = ra.HipStorage(4 * b * h * n * d), ra.HipStorage(4 * b * h * n), ra.HipStorage(4 * b * h * n)
    g = {y: ra.HipStorage(4 * b * h * n * d) for y in ("dq", "dk", "dv")}
    ra.flash_forward_stats_f32_dev(shape, t["q"], t["k"], t["v"], t["out"], lse)
    for pair in over.split(", "):
        a, z = pair.split()
        g[a] = t[z]
    ra.flash_backward_saved_f32_dev(shape, t["q"], t["k"], t["v"], t["out"], lse, t["d_out"], g["dq"], g["dk"], g["dv"], ws, ws.byte_len)
    ra.synchronize()
    for name, w in zip(("dq", "dk", "dv"), gradients64(*x)):
        got = g[name].download(np.float32).reshape(b, h, n, d)
        assert np.linalg.norm(got - w) <= 2e-6 * np.linalg.norm(w), name
