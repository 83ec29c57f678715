"""The orders in which the bf16 prefill kernels take their work: jobs dealt by rank (persistent kernel, counts of query
tiles that do not divide its rows of workers), and grid positions as (group, kv head) pairs (tile kernel, GQA)."""
import numpy as np
import pytest

import rustorch_amd as ra
from _gpu import assert_bf16_parity, bf16_round, flash_bf16
from _util import seeded_normal

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def auto_again():
    yield
    ra.debug_force_bf16_prefill_kernel("auto")


@pytest.mark.parametrize("kernel", ["auto", "persistent", "tile"])
@pytest.mark.parametrize("b,hq,hkv,n,mask", [
    (2, 32, 8, 1100, "causal"),  # 5 query tiles, 8 pairs per XCD: 40 jobs for 32 workers
    (2, 32, 32, 600, "none"),    # 3 query tiles, equal jobs
    (3, 12, 3, 700, "causal"),   # pairs that do not divide by 8: dealt over all workers
    (1, 24, 1, 520, "causal"),   # one kv head
    (1, 14, 7, 130, "causal"),   # seven kv heads
])
def test_every_head_gets_its_own_rows_and_keys(oracle, kernel, b, hq, hkv, n, mask):
    d, g = 128, hq // hkv
    qb, qf = bf16_round(seeded_normal((b, hq, n, d), 1))
    kb, kf = bf16_round(seeded_normal((b, hkv, n, d), 2))
    vb, vf = bf16_round(seeded_normal((b, hkv, n, d), 3))
    qf, kf, vf = (x.reshape(b, -1, n, d) for x in (qf, kf, vf))
    ra.debug_force_bf16_prefill_kernel(kernel)
    m = ra.Mask.causal() if mask == "causal" else ra.Mask.none()
    got = flash_bf16(ra.AttentionShape.new(b, hq, n, d), qb, kb, vb, m, n_kv_heads=hkv).reshape(b, hq, n, d)
    slabs = [(i % b, (7 * i + 3) % hq) for i in range(6)] + [(0, 0), (b - 1, hq - 1)]
    for bi, h in slabs:
        want = oracle.flash_forward_masked(oracle.AttentionShape(1, 1, n, d), qf[bi, h].copy(), kf[bi, h // g].copy(),
                                           vf[bi, h // g].copy(), mask)
        assert_bf16_parity(got[bi, h].ravel(), want, d, n, f"{kernel} b={bi} h={h}")
    # the other heads: attention averages values, so each stays within the spread of its own keys' rows
    for bi in range(b):
        for h in range(hq):
            v = vf[bi, h // g]
            assert np.allclose(got[bi, h, 0], v[0] if mask == "causal" else got[bi, h, 0], atol=2e-2), (bi, h)
            assert (got[bi, h] <= v.max(axis=0) + 2e-2).all() and (got[bi, h] >= v.min(axis=0) - 2e-2).all(), (bi, h)
