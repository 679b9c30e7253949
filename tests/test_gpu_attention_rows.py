"""Both attention kernels at the line between them (at most 640 workgroups of
16 query rows, 1024 from 512 keys on, or at most 16 queries: attn_rows_kernel;
else attn_fused_kernel), packed heads and heads side by side in rows, against the
oracle on sampled heads. Tolerance as in test_gpu_attention.py."""
import math

import numpy as np
import pytest

from oxidizedmlx_amd import backend as hb
from oxidizedmlx_amd.opkind import OpKind, meta
from parity import assert_allclose
from test_gpu_attention import cpu_attention, qkv

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("hip", "oracle_lib")]

CASES = [
    # (heads, tq, tk, dh, causal): the kernel it takes
    (80, 128, 128, 64, True),     # 640 workgroups: rows
    (81, 128, 128, 64, True),     # 648: fused
    (320, 17, 40, 32, True),      # 640: rows, one row in the second block
    (321, 17, 40, 32, False),     # 642: fused
    (16, 1024, 512, 32, True),    # 1024: rows
    (205, 70, 512, 16, False),    # 1025: fused
    (900, 16, 33, 16, False),     # 16 queries: rows whatever the number of heads
    (900, 15, 257, 64, False),    # nine tiles: one wave takes two
    (2, 300, 31, 64, True),       # fewer keys than a tile, queries past them
    (3, 50, 519, 128, True),      # more keys than causal queries see
    (13, 777, 777, 32, False),
    (160, 100, 70, 128, True),    # fused, partial blocks and tiles
    (200, 257, 257, 16, False),   # fused
]


@pytest.mark.parametrize("heads,tq,tk,dh,causal", CASES)
def test_packed_heads(heads, tq, tk, dh, causal):
    print(f"attention heads={heads} tq={tq} tk={tk} dh={dh} causal={causal}", flush=True)
    q, k, v = qkv(tq, tk, dh, heads + tq, batch=heads)
    scale = 1.0 / math.sqrt(dh)
    d = [hb.DeviceBuffer.from_array(a) for a in (q, k, v)]
    o = hb.DeviceBuffer(q.nbytes)
    hb.attention(*d, o, heads, tq, tk, dh, scale, causal)
    hb.synchronize()
    got = o.download().reshape(q.shape)
    assert np.isfinite(got).all()
    for h in (0, heads // 2, heads - 1):
        ref = cpu_attention(q[h], k[h], v[h], scale, causal)
        assert_allclose(got[h], ref, 2e-6 * float(np.abs(v).max()), 1e-5, f"head {h} of {heads}")


@pytest.mark.parametrize("groups,heads,tq,tk,dh", [(2, 3, 70, 45, 64), (40, 4, 90, 90, 32)])
def test_heads_side_by_side(groups, heads, tq, tk, dh):
    w = heads * dh
    q, k, v = qkv(tq, tk, w, 5 * groups, batch=groups)
    scale = 1.0 / math.sqrt(dh)
    d = [hb.DeviceBuffer.from_array(a) for a in (q, k, v)]
    o = hb.DeviceBuffer(q.nbytes)
    hb.eval_node_dev(OpKind.HeadAttention(scale, True, heads), [(b, a.shape) for b, a in zip(d, (q, k, v))],
                     meta(q.shape), o)
    hb.synchronize()
    got = o.download().reshape(q.shape)
    for g, h in ((0, 0), (groups - 1, heads - 1)):
        c = slice(h * dh, (h + 1) * dh)
        ref = cpu_attention(q[g][:, c].copy(), k[g][:, c].copy(), v[g][:, c].copy(), scale, True)
        assert_allclose(got[g][:, c], ref, 2e-6 * float(np.abs(v).max()), 1e-5, f"group {g} head {h}")
