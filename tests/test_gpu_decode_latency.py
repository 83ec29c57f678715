"""The one-launch decode form (decode_latency_kernel): contexts at the edges of its steps, waves and splits, ragged
batches with empty sequences, calls in a row, and workspaces that hold anything (the words its fold goes by lie there)."""
import threading

import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import assert_decode_parity, bf16_round, dev
from _util import seeded_normal

pytestmark = pytest.mark.gpu
K = ra.LlmKernels()


@pytest.mark.parametrize("b,hq,hkv,d,max_seq,lens", [
    (4, 8, 2, 128, 400, [1, 31, 32, 33]),                # one wave's step
    (5, 7, 1, 64, 400, [0, 127, 128, 129, 400]),         # one step per wave and the next; a group of 7; an empty sequence
    (3, 32, 8, 128, 1056, [385, 1055, 1056]),            # the longest context of any batch
    (2, 16, 1, 128, 3100, [3073, 97]),                   # 24 splits, and 24 that hold one step each; a full group of 16
    (1, 4, 4, 256, 1280, [1279]),                        # the widest head dim, one sequence
    (3, 6, 6, 256, 900, [900, 0, 450]),
])
def test_contexts_at_the_edges(oracle, b, hq, hkv, d, max_seq, lens):
    qb, _ = bf16_round(seeded_normal((b, hq, d), 1))
    kb, _ = bf16_round(seeded_normal((b, hkv, max_seq, d), 2))
    vb, _ = bf16_round(seeded_normal((b, hkv, max_seq, d), 3))
    dq, dk, dv = dev(qb), dev(kb), dev(vb)
    ws = ra.HipStorage(max(K.gqa_decode_workspace_bytes(b, hq, hkv, d, max_seq), 256))
    stream = ra.Stream()
    for shift in range(3):  # other lengths: the partials and words of the call before must not show
        now = np.roll(np.asarray(lens, dtype=np.int32), shift)
        dout = ra.HipStorage(b * hq * d * 2)
        dout.upload(np.full(b * hq * d, 0x7B7B, dtype=np.uint16))
        K.gqa_decode_batched_bf16(stream, dq, dk, dv, dout, dev(now), b, hq, hkv, d, max_seq, ws, ws.byte_len)
        stream.synchronize()
        got = oracle.bf16_to_f32(dout.download(np.uint16))
        want = oracle.gqa_decode_batched_bf16(qb, kb, vb, now, b, hq, hkv, d, max_seq)
        assert_decode_parity(got, want, d, f"lens {list(now)}")
        if b == 1:
            break
    stream.destroy()


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (2, 2, 64), (16, 1, 64), (16, 1, 256)])
def test_every_count_of_splits_folds_whole(oracle, hq, hkv, d):
    """Contexts whose splits number 1, 2, 3, ... to the most there are: every head's weights and sum stand, whichever
    waves of the folding workgroup come late (V is one everywhere, so a missing weight, sum or partial moves a row away
    from one; a weight is rounded to bf16, 2^-9, the sum of weights is not)."""
    max_seq = 3200 if d < 256 else 1280
    qb, _ = bf16_round(seeded_normal((1, hq, d), 1))
    kb, _ = bf16_round(seeded_normal((1, hkv, max_seq, d), 2))
    dq, dk = dev(qb), dev(kb)
    dv = dev(np.full(hkv * max_seq * d, 0x3F80, dtype=np.uint16))
    outs, lens = [], list(range(97, max_seq, 128))
    for n in lens:
        outs.append(ra.HipStorage(hq * d * 2))
        outs[-1].upload(np.full(hq * d, 0x7B7B, dtype=np.uint16))
        K.gqa_decode_online_bf16(None, dq, dk, dv, outs[-1], hq, hkv, n, d, max_seq)
    ra.synchronize()
    for n, o in zip(lens, outs):
        got = oracle.bf16_to_f32(o.download(np.uint16))
        assert np.abs(got - 1).max() <= 2 ** -7, n


def test_the_workspace_may_hold_anything(oracle):
    b, hq, hkv, d, max_seq, lens = 2, 32, 8, 128, 2100, [2100, 1333]
    qb, _ = bf16_round(seeded_normal((b, hq, d), 1))
    kb, _ = bf16_round(seeded_normal((b, hkv, max_seq, d), 2))
    vb, _ = bf16_round(seeded_normal((b, hkv, max_seq, d), 3))
    dq, dk, dv, dl = dev(qb), dev(kb), dev(vb), dev(np.asarray(lens, dtype=np.int32))
    want = oracle.gqa_decode_batched_bf16(qb, kb, vb, lens, b, hq, hkv, d, max_seq)
    size = K.gqa_decode_workspace_bytes(b, hq, hkv, d, max_seq)
    rng = np.random.default_rng(5)
    first = None
    for fill in ("zeros", "ones", "random", "words", "as left"):
        if fill == "words":  # of some launch, every count there is
            ws.upload((np.full(size // 8, 0x1234567 << 8, dtype=np.uint64) + np.arange(size // 8, dtype=np.uint64) % 256))
        elif fill != "as left":
            byte = {"zeros": np.zeros, "ones": lambda n, t: np.full(n, 255, t), "random": lambda n, t: rng.integers(0, 256, n, t)}[fill]
            ws = ra.HipStorage.from_numpy(byte(size, np.uint8))
        for again in range(3):
            dout = ra.HipStorage(b * hq * d * 2)
            dout.upload(np.full(b * hq * d, 0x7B7B, dtype=np.uint16))
            K.gqa_decode_batched_bf16(None, dq, dk, dv, dout, dl, b, hq, hkv, d, max_seq, ws, size)
            ra.synchronize()
            bits = dout.download(np.uint16)
            first = bits if first is None else first
            assert np.array_equal(bits, first), (fill, again)
    assert_decode_parity(oracle.bf16_to_f32(first), want, d)


def test_threads_on_the_per_thread_stream(oracle):
    """hipStreamPerThread (handle 2): a stream of its own for every thread, one handle for all."""
    ra.init(0)
    hq, hkv, d, max_seq = 32, 8, 128, 2100
    kb, _ = bf16_round(seeded_normal((hkv, max_seq, d), 2))
    vb, _ = bf16_round(seeded_normal((hkv, max_seq, d), 3))
    dk, dv = dev(kb), dev(vb)
    qs = [bf16_round(seeded_normal((hq, d), 10 + i))[0] for i in range(4)]
    lens = [2100, 2000, 1500, 700]
    outs, errors = [None] * 4, []

    def work(i):
        try:
            dq, dl = dev(qs[i]), dev(np.asarray(lens[i:i + 1], dtype=np.int32))
            ws = ra.HipStorage(K.gqa_decode_workspace_bytes(1, hq, hkv, d, max_seq))
            got = [ra.HipStorage(hq * d * 2) for _ in range(20)]
            ra.synchronize()
            for j, o in enumerate(got):
                if i % 2 and j % 2:
                    K.gqa_decode_batched_bf16(2, dq, dk, dv, o, dl, 1, hq, hkv, d, max_seq, ws, ws.byte_len)
                else:
                    K.gqa_decode_online_bf16(2, dq, dk, dv, o, hq, hkv, lens[i], d, max_seq)
            ra.synchronize(2)
            outs[i] = [o.download(np.uint16) for o in got]
        except Exception as e:  # noqa: BLE001 (reported by the test's thread)
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i in range(4):
        want = oracle.gqa_decode_batched_bf16(qs[i], kb, vb, lens[i:i + 1], 1, hq, hkv, d, max_seq)
        for o in outs[i]:
            assert_decode_parity(oracle.bf16_to_f32(o), want, d, f"thread {i}")
