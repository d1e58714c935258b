"""GPU: the stream-K combine at the edges of its forms.

A sequence of 64-token shares has one piece per 64 rows (and one more where
shares and sequences do not line up), so its length sets the number of
pieces: up to 16 one wave merges them; past that 16, 8 or 4 waves of four
pieces per load, chosen from the number of workgroups and of pieces.  Each
is compared with fp32 attention, gated and not, at lengths around a pass of
all waves (256, 128 and 64 pieces) and where the last one is ragged.
"""
import numpy as np
import pytest

from oracle import kvattn_oracle as orc

from gpu_helpers import H, D, Tables, build_cache, max_err, say
from test_gpu_decode import run_decode_step

pytestmark = pytest.mark.gpu
TOL = 2e-3


@pytest.mark.parametrize("lengths", [
    [16300], [16500],  # one sequence: 16 waves, 255 and past 256 pieces
    [1100, 8100],  # 16 waves: few and 127 pieces
    [4200, 8000, 4000],  # 8 waves
    [8100, 60, 1000, 3000],  # 8 waves, with a sequence of one piece
    [1200, 2500, 4100, 700, 1030, 64, 63],  # 4 waves, past 64 pieces
])
def test_combine_forms(device, lengths):
    rng = np.random.default_rng(sum(lengths))
    nblk = [(L + 1 + 15) // 16 for L in lengths]
    perm = rng.permutation(sum(nblk))
    ids, o = [], 0
    for n in nblk:
        ids.append([int(x) for x in perm[o:o + n]])
        o += n
    say(f"combine forms {lengths}")
    cache, kr, vr = build_cache(lengths, ids, extra_rows=1, rng=rng)
    tables = Tables(device, 32768)
    got, exp, qn, _, _ = run_decode_step(device, cache, kr, vr, lengths, rng, tables, split=64)
    assert max_err(got, exp) <= TOL
    gate = (2 * rng.standard_normal((len(lengths), H, D), dtype=np.float32)).astype(np.float16)
    dg, dq, out = device.array(gate), device.array(qn), device.empty((len(lengths), H, D), np.float16)
    cache.decode(0, dq, out, gate=dg, gate_stride=H * D)
    device.synchronize()
    assert max_err(out.numpy(), orc.sigmoid_gate(got, gate)) <= TOL
    cache.destroy()
