"""GPU: prefill steps long enough for two row tiles per wave (256 query rows a
unit: 42 tokens at six heads a group, 32 at eight), at the edges of their
tiles, against the oracle's fp32 attention at 2e-3, and their gate within one
ulp of the gate applied to the ungated output."""
import numpy as np
import pytest

from oracle import kvattn_oracle as orc

from gpu_helpers import D, build_cache, max_err, say
from test_gpu_gate import ulps
from test_gpu_multiquery import _ids

pytestmark = pytest.mark.gpu
TOL = 2e-3


# 12 one-tile units of a head over 257 blocks of 64 keys, four heads (12336
# blocks; 48 per workgroup of 256 is 12288), with tiles of 42, 5 and 3 tokens
# and a sequence of 10 rows beside them; then a group of eight heads.
@pytest.mark.parametrize("heads,kv_heads,prefix,chunk", [(24, 4, [16400, 16390, 7], [131, 85, 3]),
                                                         (16, 2, [24600, 0], [257, 33])])
def test_two_tile_prefill(device, heads, kv_heads, prefix, chunk):
    say(f"two-tile prefill heads={heads}/{kv_heads} prefix={prefix} chunk={chunk}")
    rng = np.random.default_rng(heads + sum(chunk))
    total = [p + c for p, c in zip(prefix, chunk)]
    cache, kr, vr = build_cache(total, _ids(rng, [(t + 15) // 16 for t in total]), extra_rows=0, num_heads=heads,
                                num_kv_heads=kv_heads, rng=rng)
    B, T = len(prefix), sum(chunk)
    for b in range(B):
        cache.set_len(b, prefix[b])
    q = rng.standard_normal((T, heads, D), dtype=np.float32).astype(np.float16)
    gate = (2 * rng.standard_normal((T, heads, D), dtype=np.float32)).astype(np.float16)
    dq, dg = device.array(q), device.array(gate)
    plain, gated = device.empty((T, heads, D), np.float16), device.empty((T, heads, D), np.float16)
    cache.begin_step(list(range(B)), chunk)
    assert cache.query_tile() == (2, 256 // (heads // kv_heads))
    cache.prefill(0, dq, plain)
    cache.prefill(0, dq, gated, gate=dg)
    device.synchronize()
    p, g = plain.numpy(), gated.numpy()
    t = 0
    for b in range(B):
        s = slice(t, t + chunk[b])
        assert max_err(p[s], orc.chunk_attention(q[s], kr[0][b], vr[0][b], prefix[b])) <= TOL, b
        t += chunk[b]
    assert ulps(g, orc.sigmoid_gate(p, gate)).max() <= 1
    cache.destroy()
