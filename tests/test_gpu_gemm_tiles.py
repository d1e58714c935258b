"""GPU: the tile GEMMs behind kva_out_project and kva_project_append, each tile
that they are built for (64, 128, 192 and 256 tokens; 128, 256 and 320 rows)
with token and row remainders, with and without a split of hidden, on inputs
whose fp32 sums are exact, so every output is bit-exact whatever the tile,
split or order."""
import numpy as np
import pytest

from oracle import kvattn_oracle as orc

from gpu_helpers import Tables, build_cache, say
from test_gpu_oproj import _inputs
from test_gpu_project import _check_cache_rows, _run

pytestmark = pytest.mark.gpu


def _bits(a):
    return a.view(np.uint16)


# Sizes of layers: token remainders of 1, 8 and 44, 16, 80 and 336 rows of tiles
# of 128, one round and several, one split and several.
@pytest.mark.parametrize("n_tok,q_dim,n_out", [(33, 512, 16), (64, 6144, 336), (65, 1536, 5120), (129, 6144, 80),
                                               (200, 6144, 5120), (700, 6144, 5120), (1300, 512, 5120)])
def test_out_project_tiles_exact(device, n_tok, q_dim, n_out):
    rng = np.random.default_rng(n_tok + n_out)
    say(f"out_project tiles n_tok={n_tok} q_dim={q_dim} n_out={n_out}")
    cache, _, _ = build_cache([8], [[0]], extra_rows=[1])
    x, w, r = _inputs(rng, n_tok, q_dim, n_out, True)
    guard = np.full((1, n_out), 77.0, np.float16)  # a row past the output stays as it was
    out = device.array(np.concatenate([r, guard]))
    cache.out_project(device.array(x), n_tok, q_dim, device.array(w), n_out, out, residual=out)
    device.synchronize()
    got = out.numpy()
    assert np.array_equal(_bits(got[:n_tok]), _bits(orc.out_project(x, w, r)))
    assert np.array_equal(_bits(got[n_tok:]), _bits(guard))
    cache.destroy()


@pytest.mark.parametrize("hidden,n_new", [(512, [33]), (5120, [64]), (5120, [50, 79]), (2560, [300])])
def test_project_tiles_exact(device, hidden, n_new):
    rng = np.random.default_rng(hidden + sum(n_new))
    lengths = [int(x) for x in rng.integers(0, 60, len(n_new))]
    say(f"project_append tiles hidden {hidden}, n_new {n_new}")
    tables = Tables(device, 512)
    cache, kr, vr, exp, got, _, _, _, _ = _run(device, rng, lengths, n_new, hidden, True, tables)
    q, gate, k_raw, k, v = exp
    assert np.array_equal(_bits(got["kv"][:, 0]), _bits(k_raw))
    assert np.array_equal(_bits(got["kv"][:, 1]), _bits(v))
    assert np.array_equal(_bits(got["g"]), _bits(gate))
    assert np.array_equal(_bits(got["q"]), _bits(q))
    _check_cache_rows(cache, kr, vr, lengths, n_new, k, v)
    cache.destroy()


# Head tiles of two heights in one launch: 192 then 128 tokens (1200), 256
# then 192 (2048, and 1990 with a ragged last tile), one height of 192, and
# rows of more tiles than the plan's search spans (21 tall ones at 4090).
@pytest.mark.parametrize("n_new", [[1200], [2048], [1000, 990], [700], [4090]])
def test_project_two_heights_exact(device, n_new):
    rng = np.random.default_rng(sum(n_new))
    lengths = [int(x) for x in rng.integers(0, 60, len(n_new))]
    say(f"project_append two heights n_new {n_new}")
    tables = Tables(device, sum(n_new) + 256)
    cache, kr, vr, exp, got, _, _, _, _ = _run(device, rng, lengths, n_new, 512, True, tables)
    q, gate, k_raw, k, v = exp
    assert np.array_equal(_bits(got["kv"][:, 0]), _bits(k_raw))
    assert np.array_equal(_bits(got["kv"][:, 1]), _bits(v))
    assert np.array_equal(_bits(got["g"]), _bits(gate))
    assert np.array_equal(_bits(got["q"]), _bits(q))
    _check_cache_rows(cache, kr, vr, lengths, n_new, k, v)
    cache.destroy()


# Every tile by its plan, token and row remainders in each: the rows past the
# last whole tile read as zeros and are not stored, tokens likewise.
@pytest.mark.parametrize("n_tok,q_dim,n_out,tile,partial", [
    (78, 512, 528, (64, 128), 0), (2099, 512, 16, (64, 128), 0), (3, 512, 528, (64, 128), 1),
    (1, 512, 7184, (64, 256), 1), (1794, 512, 1040, (128, 128), 0), (65, 6144, 3088, (128, 128), 1),
    (2054, 512, 7184, (128, 256), 0), (780, 8192, 1552, (128, 256), 1), (1027, 512, 7184, (128, 320), 0),
    (1930, 512, 5120, (128, 320), 0), (520, 512, 7184, (192, 128), 0), (130, 6144, 3088, (192, 128), 1),
    (780, 512, 7184, (256, 128), 0), (962, 6144, 1040, (256, 128), 1)])
def test_out_project_each_tile(device, n_tok, q_dim, n_out, tile, partial):
    rng = np.random.default_rng(n_tok + n_out)
    say(f"out_project tile {tile} partial={partial} n_tok={n_tok} q_dim={q_dim} n_out={n_out}")
    cache, _, _ = build_cache([8], [[0]], extra_rows=[1])
    x, w, r = _inputs(rng, n_tok, q_dim, n_out, True)
    guard = np.full((1, n_out), 77.0, np.float16)
    out = device.array(np.concatenate([r, guard]))
    cache.out_project(device.array(x), n_tok, q_dim, device.array(w), n_out, out, residual=out)
    device.synchronize()
    plan = cache.product_plan()
    assert (plan["tile_tokens"], plan["tile_rows"]) == tile and plan["partial"] == partial, plan
    got = out.numpy()
    assert np.array_equal(_bits(got[:n_tok]), _bits(orc.out_project(x, w, r)))
    assert np.array_equal(_bits(got[n_tok:]), _bits(guard))
    cache.destroy()


@pytest.mark.parametrize("hidden,n_tok,tile,partial", [
    (512, 4, (64, 0, 128), 1), (512, 1, (64, 0, 256), 1), (512, 65, (64, 0, 256), 0), (1024, 65, (128, 0, 128), 1),
    (512, 260, (128, 0, 256), 0), (8192, 260, (128, 0, 256), 1), (2048, 130, (192, 0, 128), 1),
    (512, 520, (192, 0, 256), 0), (4096, 195, (256, 0, 128), 1), (512, 780, (256, 0, 256), 0),
    (512, 1157, (192, 128, 256), 0), (512, 1417, (256, 128, 256), 0), (512, 1729, (256, 192, 256), 0)])
def test_project_each_tile(device, hidden, n_tok, tile, partial):
    rng = np.random.default_rng(hidden + n_tok)
    say(f"project_append tile {tile} partial={partial} hidden {hidden}, {n_tok} tokens")
    tables = Tables(device, n_tok + 64)
    cache, kr, vr, exp, got, _, _, _, _ = _run(device, rng, [37], [n_tok], hidden, True, tables)
    plan = cache.product_plan()
    assert (plan["tile_tokens"], plan["low_tokens"], plan["tile_rows"]) == tile, plan
    assert plan["partial"] == partial, plan
    q, gate, k_raw, k, v = exp
    assert np.array_equal(_bits(got["kv"][:, 0]), _bits(k_raw))
    assert np.array_equal(_bits(got["kv"][:, 1]), _bits(v))
    assert np.array_equal(_bits(got["g"]), _bits(gate))
    assert np.array_equal(_bits(got["q"]), _bits(q))
    _check_cache_rows(cache, kr, vr, [37], [n_tok], k, v)
    cache.destroy()
