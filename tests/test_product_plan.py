"""The launch that a projection's sizes and operands lead to
(kva_get_product_plan), on host-only caches: every check and the whole plan
run on the CPU before the call ends for want of a device."""
import pytest

from mi50grad_amd._lib import KvaError
from mi50grad_amd.kv_cache import PagedKVCache

X, W, OUT = 1 << 40, 1 << 41, 1 << 46  # operands and outputs far apart


def make(num_heads=24, num_kv_heads=4, max_step_tokens=4096):
    return PagedKVCache(n_layers=1, max_seqs=4, max_blocks=2048, max_blocks_per_seq=512,
                        max_step_tokens=max_step_tokens, num_heads=num_heads, num_kv_heads=num_kv_heads,
                        host_only=True)


def out_plan(c, n_tok, q_dim, n_out, out=OUT, residual=None):
    with pytest.raises(KvaError) as e:
        c.out_project(X, n_tok, q_dim, W, n_out, out, residual=residual)
    assert e.value.code == -3  # every check passed: only the device is missing
    return c.product_plan()


def project_plan(c, n_new, hidden, q_out=OUT, gate=None, kv=None):
    c.set_len(0, 0)
    c.begin_step([0], [n_new])
    with pytest.raises(KvaError) as e:
        c.project_append(0, X, hidden, W, 2 * W, 8 * W, 8 * W, 8 * W, 8 * W, 8192, q_out, gate, kv)
    assert e.value.code == -3
    return c.product_plan()


@pytest.mark.parametrize("n_tok", [1, 33, 64, 65, 129, 700, 2048, 4097])
def test_output_over_an_operand_goes_through_partials(n_tok):
    """A tile writes its outputs while tiles of other rows still read the same
    tokens, so an output that overlaps attn or W_o must wait in partials."""
    c = make()
    end = X + n_tok * 1024 * 2
    for out in (X, X + 64, X - (n_tok * 1024 - 8) * 2, end - 16, W + 32):
        p = out_plan(c, n_tok, 1024, 1024, out=out)
        assert p["partial"], (out, p)
    for out in (end, X - n_tok * 1024 * 2):  # beside it
        assert out_plan(c, n_tok, 1024, 1024, out=out) == out_plan(c, n_tok, 1024, 1024), out
    assert not out_plan(c, 700, 1024, 1024, out=OUT, residual=OUT)["partial"]  # in place over the residual
    c.destroy()


@pytest.mark.parametrize("n_new", [1, 40, 64, 200, 2048])
def test_project_outputs_over_x_go_through_partials(n_new):
    c = make()
    for kw in (dict(q_out=X), dict(gate=X + n_new * 6144 * 2 - 16), dict(kv=X), dict(q_out=2 * W)):
        p = project_plan(c, n_new, 6144, **kw)
        assert p["partial"], (kw, p)
    beside = project_plan(c, n_new, 6144, q_out=X + n_new * 6144 * 2)
    assert beside == project_plan(c, n_new, 6144)
    c.destroy()


def test_query_tile_of_a_step():
    """Two row tiles per wave from 48 blocks of 64 keys a workgroup in one-tile
    units (256 workgroups: 12288 blocks), causal steps of eight waves only."""
    c = PagedKVCache(n_layers=1, max_seqs=2, max_blocks=8192, max_blocks_per_seq=4096, max_step_tokens=4096,
                     host_only=True)
    # 24 tiles of 21 tokens, four heads: 128 blocks a unit are 12288.
    for rows, tiles in ((127 * 64 - 252, 2), (127 * 64 - 253, 1)):
        c.set_len(0, 0)
        c.reserve(0, rows)
        c.set_len(0, rows)
        c.begin_step([0], [504])
        assert c.query_tile() == (tiles, 42 if tiles == 2 else 21), rows
    c.reserve(0, 60100)
    c.set_len(0, 60000)
    c.begin_step([0], [10], tree_bits=[1 << i for i in range(10)])
    assert c.query_tile() == (1, 10)  # four waves of 16 rows, 6 heads a group
    c.begin_step([0], [63], tree_bits=[1 << i for i in range(63)])
    assert c.query_tile() == (1, 21)
    c.destroy()
