"""GPU: the whole-sequence decode with six and eight query heads per
workgroup, which walks pages with the scores on the matrix unit, at the edges
of a page, of a round of its eight waves (128 rows) and of its range."""
import numpy as np
import pytest

from mi50grad_amd import _lib
from oracle import kvattn_oracle as orc

from gpu_helpers import D, Tables, build_cache, max_err, say
from test_gpu_decode import TOL, run_decode_step

pytestmark = pytest.mark.gpu


def test_paged_edges(device):
    # 40 sequences x 4 kv heads on 256 CUs: six query heads a workgroup.
    edges = [0, 1, 2, 14, 15, 16, 17, 30, 31, 32, 126, 127, 128, 129, 143, 144, 254, 255, 256, 257, 383, 512, 1007,
             1008, 1022, 1023]
    lengths = edges + [int(x) for x in np.random.default_rng(7).integers(0, 600, 40 - len(edges))]
    nblk = [(n + 1 + 15) // 16 for n in lengths]
    rng = np.random.default_rng(8)
    perm = rng.permutation(sum(nblk))
    ids, o = [], 0
    for n in nblk:
        ids.append([int(x) for x in perm[o:o + n]])
        o += n
    say("whole form on pages, paged edges")
    cache, kr, vr = build_cache(lengths, ids, extra_rows=1, rng=rng)
    got, exp, *_ = run_decode_step(device, cache, kr, vr, lengths, rng, Tables(device, 1040))
    assert cache.decode_split() == (0, 160)  # one workgroup per (sequence, kv head)
    assert max_err(got, exp) <= TOL
    cache.destroy()


@pytest.mark.parametrize("h,hkv,B,L", [(32, 4, 40, 1), (32, 4, 40, 17), (24, 4, 40, 129), (8, 1, 130, 250)])
def test_contiguous_edges(device, h, hkv, B, L):
    rng = np.random.default_rng(h + L)
    K = rng.standard_normal((B, L, hkv, D), dtype=np.float32).astype(np.float16)
    V = rng.standard_normal((B, L, hkv, D), dtype=np.float32).astype(np.float16)
    Q = rng.standard_normal((B, h, D), dtype=np.float32).astype(np.float16)
    say(f"whole form on pages, contiguous h={h} hkv={hkv} B={B} L={L}")
    dq, dk, dv = device.array(Q), device.array(K), device.array(V)
    out = device.empty((B, h, D), np.float16)
    _lib.call("kva_legacy_decode_batched", None, dq.ptr, dk.ptr, dv.ptr, out.ptr, L, B, L * hkv * D * 2, h, hkv, None)
    device.synchronize()
    ref = np.stack([orc.attention_fp32(Q[b:b + 1], K[b], V[b])[0] for b in range(B)])
    assert max_err(out.numpy(), ref) <= TOL
