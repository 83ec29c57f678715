"""The staging of the host-slice entries: whatever the size of a call and whoever else is calling, its results are those
of the device entry, bit for bit."""
import threading

import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import dev

pytestmark = pytest.mark.gpu


def inputs(n, seed, count=3):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(n, dtype=np.float32) for _ in range(count)]


def on_device(shape, q, k, v, mask):
    out = ra.HipStorage(q.nbytes)
    ra.flash_forward_f32_dev(shape, dev(q), dev(k), dev(v), out, mask, None if mask.keep is None else dev(mask.keep))
    ra.synchronize()
    return out.download(np.float32)


@pytest.mark.parametrize("bhnd", [
    (1, 1, 3, 4),          # one transfer each way, results straight into pinned memory
    (1, 3, 257, 20),       # inputs that end inside a 16-byte unit of their padding
    (2, 4, 300, 66),       # a head dim whose kernel stores single elements
    (1, 4, 1024, 64),      # several chunks that span inputs, results in two
    (8, 16, 500, 64),      # three times the ring's size up, twice the slots' down, copies shared with the helpers
    (3, 16, 1000, 128),    # a block larger than what is kept between calls
])
def test_host_slices_give_the_device_entrys_bits(bhnd):
    shape = ra.AttentionShape.new(*bhnd)
    q, k, v = inputs(shape.buffer_len(), 7)
    keep = np.arange(bhnd[2]) % 5 != 3
    for mask in (ra.Mask.none(), ra.Mask.padding(keep)):
        assert np.array_equal(ra.flash_forward_masked(shape, q, k, v, mask), on_device(shape, q, k, v, mask))


def test_threads_and_shutdown():
    shapes = [ra.AttentionShape.new(2, 8, 700, 64), ra.AttentionShape.new(1, 2, 100, 64)]
    cases = [(s, inputs(s.buffer_len(), i)) for i, s in enumerate(shapes * 2)]
    want = [on_device(s, *x, ra.Mask.causal()) for s, x in cases]
    for _ in range(2):
        got = [None] * len(cases)

        def call(i):
            for _ in range(3):
                got[i] = ra.flash_forward_masked(cases[i][0], *cases[i][1], ra.Mask.causal())

        threads = [threading.Thread(target=call, args=(i,)) for i in range(len(cases))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        ra.shutdown()  # ends the helpers and frees the staging memory; the next call brings them back


def test_backward_through_the_staging():
    shape = ra.AttentionShape.new(2, 4, 600, 64)
    host = inputs(shape.buffer_len(), 3, 4)
    d_in, d_out = [dev(x) for x in host], [ra.HipStorage(host[0].nbytes) for _ in range(3)]
    ws = ra.HipStorage(ra.flash_backward_workspace_bytes(shape))
    ra.flash_backward_f32_dev(shape, *d_in, *d_out, ws, ws.byte_len)
    ra.synchronize()
    for got, want in zip(ra.flash_backward(shape, *host), d_out):
        assert np.array_equal(got, want.download(np.float32))
