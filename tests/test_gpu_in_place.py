"""GPU: projections whose output is their own input: kva_out_project with out
= attn, and kva_project_append with q_out = x, in one launch and in several
(a workspace smaller than the step).  The inputs' fp32 sums are exact, so
every output is bit-exact whatever the tile or split."""
import numpy as np
import pytest

from oracle import kvattn_oracle as orc

from gpu_helpers import D, Tables, build_cache, say
from test_gpu_oproj import _inputs

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint16)


# One launch at 24/4 heads; 512 tokens a launch with the smallest workspace.
@pytest.mark.parametrize("heads,n_tok,q_dim,n_out", [((24, 4), 40, 6144, 6144), ((24, 4), 200, 1024, 1024),
                                                     ((24, 4), 700, 1024, 528), ((1, 1), 1100, 512, 512),
                                                     ((1, 1), 1100, 1024, 496)])
def test_out_project_over_attn(device, heads, n_tok, q_dim, n_out):
    rng = np.random.default_rng(n_tok + n_out)
    say(f"out_project over attn heads={heads} n_tok={n_tok} q_dim={q_dim} n_out={n_out}")
    cache, _, _ = build_cache([8], [[0]], extra_rows=[1], num_heads=heads[0], num_kv_heads=heads[1],
                              max_step_tokens=16)
    x, w, r = _inputs(rng, n_tok, q_dim, n_out, True)
    buf = device.array(x)
    cache.out_project(buf, n_tok, q_dim, device.array(w), n_out, buf, residual=device.array(r))
    device.synchronize()
    got = buf.numpy().reshape(-1)[:n_tok * n_out].reshape(n_tok, n_out)
    assert np.array_equal(_bits(got), _bits(orc.out_project(x, w, r)))
    cache.destroy()


# 24/4 heads in one launch; 2/1 heads over a workspace of 1024 tokens.
@pytest.mark.parametrize("heads,hidden,n_new", [((24, 4), 6144, [40]), ((24, 4), 6144, [100, 9]),
                                                ((2, 1), 512, [700, 400])])
def test_project_append_over_x(device, heads, hidden, n_new):
    H, HKV = heads
    rng = np.random.default_rng(hidden + sum(n_new))
    say(f"project_append over x heads={heads} hidden={hidden} n_new={n_new}")
    T, tables = sum(n_new), Tables(device, 1024)
    ids, o = [], 0
    for n in n_new:
        ids.append(list(range(o, o + (n + 15) // 16)))
        o += len(ids[-1])
    cache, _, _ = build_cache([0] * len(n_new), ids, extra_rows=list(n_new), num_heads=H, num_kv_heads=HKV,
                              max_step_tokens=1200, rng=rng)
    x = rng.integers(-3, 4, (T, hidden), dtype=np.int8).astype(np.float16)
    wq = (rng.integers(-2, 3, (2 * H * D, hidden), dtype=np.int8) * 2.0 ** -7).astype(np.float16)
    wkv = (rng.integers(-2, 3, (2 * HKV * D, hidden), dtype=np.int8) * 2.0 ** -7).astype(np.float16)
    qw, kw = [(1 + 0.02 * rng.standard_normal(D, dtype=np.float32)).astype(np.float16) for _ in range(2)]
    buf, gate = device.array(x), device.empty((T, H, D), np.float16)
    cache.begin_step(list(range(len(n_new))), n_new)
    cache.project_append(0, buf, hidden, device.array(wq), device.array(wkv), device.array(qw), device.array(kw),
                         tables.d_cos, tables.d_sin, tables.rows, buf, gate)
    device.synchronize()
    pos = [i for n in n_new for i in range(n)]
    q, g, _, k, v = orc.project_append(x, wq, wkv, qw, kw, tables.cos[pos], tables.sin[pos], H, HKV)
    assert np.array_equal(_bits(buf.numpy().reshape(T, H, D)), _bits(q))
    assert np.array_equal(_bits(gate.numpy()), _bits(g))
    o = 0
    for b, n in enumerate(n_new):
        krow, vrow = cache.gather(0, b, n)
        assert np.array_equal(_bits(krow), _bits(k[o:o + n])) and np.array_equal(_bits(vrow), _bits(v[o:o + n])), b
        o += n
    cache.destroy()
