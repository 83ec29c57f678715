"""Host-side mirror of `rustorch_nn::gqa` (crates/rustorch-nn/src/gqa.rs:94-210) over the HIP library."""
from __future__ import annotations

import numpy as np

from . import _lib as L
from .attention import _f32
from .errors import check


def gqa_forward_f32(q, k, v, out, batch, n_heads, n_kv_heads, seq_q, seq_kv, head_dim):
    """Same argument order as the reference.  q/out [B,Hq,Sq,D], k/v [B,Hkv,Skv,D], flat f32;
    `out` (numpy f32, C-contiguous) is fully overwritten and returned."""
    q, k, v = _f32(q), _f32(k), _f32(v)
    assert out.dtype == np.float32 and out.flags.c_contiguous
    check(L.native.rt_gqa_forward_f32(q, q.size, k, k.size, v, v.size, out, out.size, batch, n_heads, n_kv_heads, seq_q, seq_kv,
                                      head_dim))
    return out


def gqa_forward_f32_dev(q, k, v, out, batch, n_heads, n_kv_heads, seq_q, seq_kv, head_dim, stream=None):
    """The same on device-resident f32 tensors; enqueues on `stream` and returns."""
    check(L.native.rt_gqa_forward_f32_dev(stream, q, k, v, out, batch, n_heads, n_kv_heads, seq_q, seq_kv, head_dim))
