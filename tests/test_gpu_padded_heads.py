"""Matrix-core decode of head dims and head groups that do not fill its tiles:
head dims that are multiples of 16 between 48 and 128, and groups of 2 to 17
query heads per kv head, under every split plan (static splits, the tile
stream, the in-kernel and launched schedules), contiguous and paged, with and
without the fused append.  Slots past each length hold NaN scales and garbage
bytes.

Parity as in test_gpu_decode: out[b, hq] = oracle kvq_ref_decode_f32 over the
first length[b] tokens of kv head hq / G, 1e-4 abs + 1e-3 rel elementwise;
appended int8 values and scales bit-exact.
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


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# G: a pair, one short of a tile, one past it, two groups of unequal size, three groups.
@pytest.mark.parametrize("G", [2, 3, 5, 7, 9, 12, 17])
@pytest.mark.parametrize("d", [48, 64, 80, 112, 128])
@pytest.mark.parametrize("B,cap,ragged", [(1, 2052, False), (5, 700, True), (70, 200, True), (130, 1100, True)])
def test_padded_heads(o, G, d, B, cap, ragged):
    rng = np.random.default_rng(1000 * G + d + B)
    Hkv = 1 if B > 5 else 2
    lengths = None
    if ragged:
        lengths = rng.integers(1, cap + 1, B).astype(np.int32)
        lengths[:4] = [cap, 1, 31, 33]
    p = make_problem(rng, B, Hkv * G, Hkv, cap, d, o.quantize_rows, lengths=lengths)
    kn, vn = (rng.standard_normal((B, Hkv, d)).astype(np.float32) for _ in range(2))
    prm = kvq.DecodeParams(B, Hkv * G, Hkv, d, cap, cap, 4096 if ragged else None, *[4096] * 6, 0.0, 0, 4096, 4096)
    assert kvq.decode_plan(prm).kernel == kvq.KERNEL_DECODE_MFMA
    L = lengths if ragged else np.full(B, cap, np.int32)
    got, gk, gv, gks, gvs = _gpu.decode(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths, max_seq_len=cap,
                                         k_new=kn, v_new=vn)
    paged = None
    if ragged:
        kp, vp, ksp, vsp, table = to_pages(rng, p["k"], p["v"], p["ks"], p["vs"], lengths, 32)
        paged = paged_decode(p["q"], kp, vp, ksp, vsp, table, lengths, k_new=kn, v_new=vn)
    o.append(kn, vn, p["k"], p["v"], p["ks"], p["vs"], positions=L - 1)
    assert np.array_equal(gk, p["k"]) and np.array_equal(gv, p["v"])
    assert np.array_equal(_bits(gks), _bits(p["ks"])) and np.array_equal(_bits(gvs), _bits(p["vs"]))
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=L)
    assert_close(got, want, what=f"G={G} d={d} B={B}")
    if paged is not None:
        assert_close(paged[0], want, what=f"paged G={G} d={d} B={B}")
        back = from_pages(*paged[1:5], table, lengths, p["k"].shape)
        for b in range(B):
            n = int(lengths[b])
            for g, w in zip(back, (p["k"], p["v"], p["ks"], p["vs"])):
                assert g[b, :, :n].tobytes() == w[b, :, :n].tobytes()
