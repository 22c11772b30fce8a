"""kvq_decode_launch_noalloc on steps whose padded plan needs more than its
fixed scratch array: they run the unpadded plan.

Parity as in test_gpu_decode: 1e-4 abs + 1e-3 rel elementwise against the oracle.
"""
import numpy as np
import pytest
import torch

from _util import assert_close, make_problem
from _gpu import down, kvq, poisoned, up
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SCRATCH = 16 << 20


# The unpadded plans need no workspace: the general kernel (head dims 48, 112
# and 192; more work units than arrival counters or one full round).
@pytest.mark.parametrize("B,G,Hkv,d", [(700, 16, 8, 48), (64, 16, 32, 112), (200, 12, 8, 192)])
def test_unpadded_plan_when_the_padded_one_does_not_fit(B, G, Hkv, d):
    o = orc.get()
    cap = 130
    rng = np.random.default_rng(B + d)
    lengths = rng.integers(0, 24, B).astype(np.int32)
    lengths[:3] = [cap, 1, 0]
    p = make_problem(rng, B, G * Hkv, Hkv, cap, d, o.quantize_rows, lengths=lengths)
    g = [up(p[n]) for n in ("q", "k", "v", "ks", "vs")]
    gl = up(lengths)
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths)
    out = poisoned((B, G * Hkv, d))
    params = kvq.decode_params(*g, out, gl)
    assert kvq.workspace_size(params) > SCRATCH
    assert kvq.decode_launch_noalloc(params) == 0
    torch.cuda.synchronize()
    assert_close(down(out), want)
