"""Spans of a chunked decode's keys: partials of blocks that are not whole, their fold by one wave and by four, and calls
whose partials do not fit the stream's fixed scratch (a kept buffer; under capture fewer spans)."""
import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import assert_bf16_parity, bf16_round, dev
from _util import seeded_normal
from test_gpu_decode_graph import Hip

pytestmark = pytest.mark.gpu
K = ra.LlmKernels()


def tensors(b, s, hq, hkv, d, max_seq):
    q, k, v = (bf16_round(seeded_normal(shape, i))[0] for i, shape in
               enumerate([(b, s, hq, d), (b, hkv, max_seq, d), (b, hkv, max_seq, d)]))
    out = ra.HipStorage(q.size * 2)
    out.upload(np.full(q.size, 0x7B7B, dtype=np.uint16))
    return (q, k, v), (dev(q), dev(k), dev(v)), out


@pytest.mark.parametrize("b,s,hq,hkv,d,max_seq,lens", [
    (1, 1, 7, 1, 128, 1024, [1000]),          # 7 rows, 16 spans
    (1, 11, 6, 2, 128, 1500, [1500]),         # 33 rows: a block and one row; 24 spans
    (2, 43, 3, 1, 96, 700, [700, 130]),       # 129 rows: a query tile and one row
    (1, 31, 1, 1, 8, 4096, [4096]),           # one piece of eight columns
    (1, 3, 64, 2, 200, 2000, [1990]),         # columns past the head dim
    (1, 100, 16, 2, 256, 2048, [2048]),       # partials past the fixed scratch
])
def test_spans_fold_to_the_whole(oracle, b, s, hq, hkv, d, max_seq, lens):
    (q, k, v), (dq, dk, dv), out = tensors(b, s, hq, hkv, d, max_seq)
    K.gqa_decode_chunk_bf16(None, dq, dk, dv, out, dev(np.asarray(lens, dtype=np.int32)), b, s, hq, hkv, d, max_seq)
    ra.synchronize()
    want = oracle.gqa_decode_chunk_bf16(q, k, v, lens, b, s, hq, hkv, d, max_seq)
    assert_bf16_parity(oracle.bf16_to_f32(out.download(np.uint16)), want, d, None, f"s={s} hq={hq} d={d}")


@pytest.mark.parametrize("b,s,hq,hkv,d,max_seq,lens", [
    (1, 2, 16, 16, 64, 900, [900]),           # as many spans as tiles, the last of four keys
    (1, 4, 8, 2, 64, 1473, [1473]),           # the last of one
    (3, 4, 32, 8, 128, 200, [200, 65, 4]),    # not cut
    (1, 4, 32, 8, 128, 200, [65]),            # four spans, two without keys, one of the last position's key alone
    (1, 8, 16, 2, 256, 300, [300]),           # tiles of 32 keys
    (2, 5, 12, 12, 80, 321, [320, 257]),      # columns past the head dim
    (4, 4, 16, 16, 64, 800, [800, 1, 0, 449]),  # spans of two tiles, the last of one; positions without keys
    (3, 2, 8, 8, 64, 900, [900, 66, 1]),      # most spans of two sequences without keys, a position without
    (2, 4, 16, 16, 64, 800, [800, 449]),      # two workgroups a CU
])
def test_spans_of_a_tile(oracle, b, s, hq, hkv, d, max_seq, lens):
    """(tests/cpp/api_host_test.cpp holds the number of spans of every case here.)"""
    (q, k, v), (dq, dk, dv), out = tensors(b, s, hq, hkv, d, max_seq)
    K.gqa_decode_chunk_bf16(None, dq, dk, dv, out, dev(np.asarray(lens, dtype=np.int32)), b, s, hq, hkv, d, max_seq)
    ra.synchronize()
    want = oracle.gqa_decode_chunk_bf16(q, k, v, lens, b, s, hq, hkv, d, max_seq)
    assert_bf16_parity(oracle.bf16_to_f32(out.download(np.uint16)), want, d, None, f"s={s} hq={hq} d={d}")


def test_a_captured_call_stays_within_the_fixed_scratch(oracle):
    b, s, hq, hkv, d, max_seq = 1, 100, 16, 2, 256, 2048
    (q, k, v), (dq, dk, dv), out = tensors(b, s, hq, hkv, d, max_seq)
    want = oracle.gqa_decode_chunk_bf16(q, k, v, [max_seq], b, s, hq, hkv, d, max_seq)
    hip, stream = Hip(), ra.Stream()
    graph, exe, types = hip.capture(stream.handle, lambda: K.gqa_decode_chunk_bf16(
        stream.handle, dq, dk, dv, out, max_seq, b, s, hq, hkv, d, max_seq))
    assert types == [0, 0], types  # two kernels
    for _ in range(3):
        out.upload(np.full(q.size, 0x7B7B, dtype=np.uint16))
        hip.launch(exe, stream.handle)
        stream.synchronize()
        assert_bf16_parity(oracle.bf16_to_f32(out.download(np.uint16)), want, d, None, "replay")
    hip.destroy(graph, exe)
