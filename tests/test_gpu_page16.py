"""Matrix-core decode of caches whose rows or pages do not fit its 32-token
tiles: 16-token pages (two per tile; odd page counts, so the last tile's second
page lies past the table row), and odd capacities (scale rows at any 4-byte
alignment, the last scale quad reaching past the row).

Parity as in test_gpu_decode: 1e-4 abs + 1e-3 rel elementwise against the
oracle; appended int8 values and scales bit-exact.
"""
import numpy as np
import pytest

from _util import assert_close, make_problem
import _gpu
from _gpu import kvq
from oracle import oracle as orc
from test_gpu_paged import from_pages, paged_decode, to_pages

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def o():
    return orc.get()


def _problem(o, seed, B, Hkv, G, d, cap):
    rng = np.random.default_rng(seed)
    lengths = rng.integers(1, cap + 1, B).astype(np.int32)
    lengths[:4] = [cap, 1, min(17, cap), min(16, cap)]
    p = make_problem(rng, B, Hkv * G, Hkv, cap, d, o.quantize_rows, lengths=lengths)
    kn, vn = (rng.standard_normal((B, Hkv, d)).astype(np.float32) for _ in range(2))
    return rng, lengths, p, kn, vn


@pytest.mark.parametrize("G,d", [(4, 128), (8, 128), (4, 64), (3, 96), (6, 80)])
@pytest.mark.parametrize("B,cap", [(4, 16), (5, 33), (6, 721), (70, 150), (300, 1041)])
def test_page16(o, G, d, B, cap):
    Hkv = 2
    rng, lengths, p, kn, vn = _problem(o, 10 * G + d + B, B, Hkv, G, d, cap)
    kp, vp, ksp, vsp, table = to_pages(rng, p["k"], p["v"], p["ks"], p["vs"], lengths, 16)
    got = paged_decode(p["q"], kp, vp, ksp, vsp, table, lengths, k_new=kn, v_new=vn)
    assert kvq.paged_decode_plan(got[5].params).kernel == kvq.KERNEL_DECODE_MFMA
    o.append(kn, vn, p["k"], p["v"], p["ks"], p["vs"], positions=lengths - 1)
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths)
    assert_close(got[0], want, what=f"G={G} d={d} B={B} cap={cap}")
    back = from_pages(*got[1:5], table, lengths, p["k"].shape)
    for b in range(B):
        n = int(lengths[b])
        for g, w in zip(back, (p["k"], p["v"], p["ks"], p["vs"])):
            assert g[b, :, :n].tobytes() == w[b, :, :n].tobytes()


@pytest.mark.parametrize("G,d", [(4, 128), (8, 64), (5, 112)])
@pytest.mark.parametrize("cap", [1, 31, 33, 129, 1023, 2050])
@pytest.mark.parametrize("B", [4, 66])
def test_odd_capacity(o, G, d, cap, B):
    Hkv = 3
    rng, lengths, p, kn, vn = _problem(o, 10 * G + d + cap, B, Hkv, G, d, cap)
    prm = kvq.DecodeParams(B, Hkv * G, Hkv, d, cap, cap, 4096, *[4096] * 6, 0.0, 0, 4096, 4096)
    assert kvq.decode_plan(prm).kernel == kvq.KERNEL_DECODE_MFMA
    got, gk, gv, gks, gvs = _gpu.decode(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths, k_new=kn, v_new=vn)
    o.append(kn, vn, p["k"], p["v"], p["ks"], p["vs"], positions=lengths - 1)
    for g, w in zip((gk, gv, gks, gvs), (p["k"], p["v"], p["ks"], p["vs"])):
        assert g.tobytes() == w.tobytes()
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths)
    assert_close(got, want, what=f"G={G} d={d} cap={cap} B={B}")
