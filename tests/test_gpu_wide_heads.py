"""Head dims above 128, whose longer walks take tiles of 64 keys straight into LDS and shorter ones tiles of 32 through registers
(takes_tiles_direct, flash_bf16_tile.hip), either side of the line between them and at the edges of tiles, against the CPU
oracle run in f32 on the same bf16-rounded inputs.  Bar: max-abs <= 2e-2 and relative Frobenius error <= 1e-2 per block of 256 rows."""
import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import assert_bf16_parity, bf16_round, dev, flash_bf16
from _util import seeded_normal
from test_gpu_attention_general import run_chunk
from test_gpu_flash_bf16 import run_varlen
from test_gpu_window import window_bnhd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [136, 200, 256])
@pytest.mark.parametrize("n", [95, 96, 97, 127, 128, 129, 160, 191, 257, 450])
def test_masks_at_the_edges_of_tiles(oracle, n, d):
    b, h = 2, 3
    (qb, qf), (kb, kf), (vb, vf) = (bf16_round(seeded_normal((b, h, n, d), n + i)) for i in range(3))
    shape = ra.AttentionShape.new(b, h, n, d)
    keep = np.random.default_rng(n).random(n) < 0.7
    keep[0] = True
    for mask, om in ((ra.Mask.none(), None), (ra.Mask.causal(), "causal"), (ra.Mask.padding(keep), ("padding", keep))):
        got = flash_bf16(shape, qb, kb, vb, mask)
        want = oracle.flash_forward_masked(oracle.AttentionShape(b, h, n, d), qf, kf, vf, om)
        assert_bf16_parity(got, want, d, n, f"n={n} d={d} mask={mask.kind}")
        assert np.array_equal(got, flash_bf16(shape, qb, kb, vb, mask)), "two launches, two results"


@pytest.mark.parametrize("d", [136, 256])
@pytest.mark.parametrize("n", [129, 199, 200, 287, 288, 321])
def test_workgroups_that_fill_the_chip(oracle, n, d):
    """Either side of the lines there.  All heads have the same rows, so that one stands for all."""
    b, h = 14, 16
    one = [bf16_round(seeded_normal((1, 1, n, d), n + i)) for i in range(3)]
    q, k, v = (np.ascontiguousarray(np.broadcast_to(x[0].reshape(1, 1, n, d), (b, h, n, d))) for x in one)
    for mask, om in ((ra.Mask.none(), None), (ra.Mask.causal(), "causal")):
        got = np.asarray(flash_bf16(ra.AttentionShape.new(b, h, n, d), q, k, v, mask)).reshape(b * h, n * d)
        assert (got == got[0]).all()
        want = oracle.flash_forward_masked(oracle.AttentionShape(1, 1, n, d), *(x[1].ravel() for x in one), om)
        assert_bf16_parity(got[0], want, d, n, f"n={n} d={d} {om}")


@pytest.mark.parametrize("b,s,hq,hkv,d,keys", [(25, 8, 8, 8, 136, 299), (25, 8, 8, 8, 136, 300), (25, 8, 8, 8, 256, 300), (13, 66, 16, 16, 256, 249), (17, 66, 16, 16, 256, 999), (17, 66, 16, 16, 256, 1000)])
def test_chunks_that_fill_the_chip(oracle, b, s, hq, hkv, d, keys):
    qb, kb, vb = (bf16_round(seeded_normal(shape, i))[0] for i, shape in enumerate([(1, s, 1, d), (1, 1, keys, d), (1, 1, keys, d)]))
    q = np.ascontiguousarray(np.broadcast_to(qb.reshape(1, s, 1, d), (b, s, hq, d)))
    k, v = (np.ascontiguousarray(np.broadcast_to(x.reshape(1, 1, keys, d), (b, hkv, keys, d))) for x in (kb, vb))
    out = ra.HipStorage(q.size * 2)
    out.upload(np.full(q.size, 0x7B7B, dtype=np.uint16))
    dq, dk, dv = dev(q), dev(k), dev(v)
    ra.LlmKernels().gqa_decode_chunk_bf16(None, dq, dk, dv, out, keys, b, s, hq, hkv, d, keys)
    ra.synchronize()
    got = oracle.bf16_to_f32(out.download(np.uint16)).reshape(b, s, hq, d)
    assert (got == got[:1, :, :1]).all()
    want = oracle.gqa_decode_chunk_bf16(qb, kb, vb, [keys], 1, s, 1, 1, d, keys)
    assert_bf16_parity(got[0, :, 0].ravel(), want, d, None, f"s={s} d={d} keys={keys}")


@pytest.mark.parametrize("d", [152, 256])
@pytest.mark.parametrize("window", [1, 31, 33, 64, 97, 191, 257])
def test_windows(oracle, d, window):
    for n in (95, 96, 450, 513):
        got, want, _ = window_bnhd(oracle, 1, n, 2, 1, d, window, 5 * window + n)
        assert_bf16_parity(got.reshape(1, n, 2 * d), want.reshape(1, n, 2 * d), 2 * d, None, f"n={n} window {window}", block_rows=64)


def test_windows_that_fill_the_chip(oracle):
    for hkv in (16, 8):  # through registers, and straight to LDS
        got, want, _ = window_bnhd(oracle, 7, 193, 16, hkv, 136, 97, hkv)
        assert_bf16_parity(got.reshape(7, 193, 16 * 136), want.reshape(7, 193, 16 * 136), 16 * 136, None, f"kv heads {hkv}", block_rows=64)


@pytest.mark.parametrize("n,d", [(193, 136), (353, 136)])
def test_padded_batches_that_fill_the_chip(oracle, n, d):
    test_padded_batch(oracle, d, 13, 8, n, [n, 0, 1, 64, 65, 129, n - 1] + [n // 2] * 6)


@pytest.mark.parametrize("d", [168, 256])
def test_padded_batch(oracle, d, b=6, h=2, n=200, lens=(200, 0, 1, 64, 65, 129)):
    lens = np.array(lens, dtype=np.int32)
    (qb, qf), (kb, kf), (vb, vf) = (bf16_round(seeded_normal((b, h, n, d), i)) for i in range(3))
    kb, vb = (x.copy().reshape(b, h, n, d) for x in (kb, vb))
    for i, m in enumerate(lens):  # what lies behind a sequence is not read, or weighs nothing
        kb[i, :, m:] = vb[i, :, m:] = 0x7FC0
    got = run_varlen(ra.AttentionShape.new(b, h, n, d), qb, kb.ravel(), vb.ravel(), lens)
    got = np.asarray(got).reshape(b, h, n, d)
    rows = lambda x, i, m: np.ascontiguousarray(np.asarray(x).reshape(b, h, n, d)[i, :, :m]).ravel()
    for i, m in enumerate(lens):
        assert not got[i, :, m:].any()
        if m:
            want = oracle.flash_forward_masked(oracle.AttentionShape(1, h, int(m), d), rows(qf, i, m), rows(kf, i, m), rows(vf, i, m), "causal")
            assert_bf16_parity(got[i, :, :m].ravel(), want, d, None, f"length {m}")


@pytest.mark.parametrize("b,s,hq,hkv,d,max_seq,lens", [
    (2, 130, 4, 1, 256, 500, [500, 131]),   # whole, more rows than a tile
    (4, 40, 16, 16, 200, 200, [200, 41, 96, 40]),
    (1, 100, 16, 2, 256, 2047, [2047]),     # spans of fewer than 256 keys,
    (1, 100, 16, 2, 256, 2049, [2049]),     # and of more; the last of a key
    (1, 200, 16, 2, 160, 4000, [3333]),
])
def test_chunks(oracle, b, s, hq, hkv, d, max_seq, lens):
    run_chunk(oracle, b, s, hq, hkv, d, max_seq, lens)


@pytest.mark.parametrize("b,s,hq,hkv,d,max_seq,lens", [
    (1, 130, 4, 1, 256, 500, [500]),        # whole, more rows than a tile
    (4, 40, 16, 16, 200, 200, [200] * 4),
    (1, 100, 16, 2, 256, 2047, [2047]),     # spans of fewer than 256 keys,
    (1, 100, 16, 2, 256, 2049, [2049]),     # and of more; the last of a key
    (1, 200, 16, 2, 160, 4000, [3333]),
])
def test_chunks_of_a_length_the_launch_knows(oracle, b, s, hq, hkv, d, max_seq, lens):
    run_chunk(oracle, b, s, hq, hkv, d, max_seq, lens, scalar_len=True)


@pytest.mark.parametrize("s,lens", [(255, [700, 300, 255, 400]), (256, [700, 256, 1, 321]), (300, [700, 301, 300, 0])])
def test_chunks_of_many_positions_and_unknown_lengths(oracle, s, lens):
    run_chunk(oracle, 4, s, 16, 16, 136, 700, lens)
