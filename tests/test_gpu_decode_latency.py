"""The one-launch decode form (decode_latency_kernel): contexts at the edges of its steps, waves and splits, ragged
batches with empty sequences, and calls in a row (the counters its fold goes by are back at rest after each)."""
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
    for shift in range(3):  # other lengths: the partials and counters of the call before must not show
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
