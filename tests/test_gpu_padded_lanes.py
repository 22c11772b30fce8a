"""The per-lane FMA decode kernel at head dims its lanes pad (multiples of 16
between 48 and 240 other than 64 and 128): one query head per kv head, or
head dims past the matrix-core kernel's, under every split plan, contiguous
and paged, with and without the fused append, and through the reference's
entry point.  Slots past each length hold NaN scales and garbage bytes.

Parity as in test_gpu_decode: 1e-4 abs + 1e-3 rel elementwise against the
oracle; appended int8 values and scales bit-exact.
"""
import numpy as np
import pytest

from _util import assert_close, make_problem
import _gpu
from _gpu import kvq
from oracle import oracle as orc
from test_gpu_paged import paged_decode, to_pages
from test_gpu_reference_abi import _run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def o():
    return orc.get()


def _bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


@pytest.mark.parametrize("G,d", [(1, 48), (1, 80), (1, 96), (1, 112), (1, 144), (1, 192), (2, 192), (3, 240), (4, 192), (5, 144)])
@pytest.mark.parametrize("B,cap,ragged,page", [(1, 2052, False, 0), (3, 130, False, 0), (5, 1500, True, 32), (70, 300, True, 16),
                                               (300, 90, True, 0)])
def test_padded_lanes(o, G, d, B, cap, ragged, page):
    rng = np.random.default_rng(1000 * G + d + B)
    Hkv = 1 if B > 5 else 2
    lengths = None
    if ragged:
        lengths = rng.integers(1, cap + 1, B).astype(np.int32)
        lengths[:4] = [cap, 1, 31, 33]
    p = make_problem(rng, B, Hkv * G, Hkv, cap, d, o.quantize_rows, lengths=lengths)
    L = lengths if ragged else np.full(B, cap, np.int32)
    prm = kvq.DecodeParams(B, Hkv * G, Hkv, d, cap, cap, 4096 if ragged else None, *[4096] * 6, 0.0, 0, None, None)
    info = kvq.decode_plan(prm)
    assert info.kernel == kvq.KERNEL_DECODE_VALU
    want0 = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=L)
    got = _gpu.decode(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths, max_seq_len=cap)[0]
    assert_close(got, want0, what=f"no append G={G} d={d} B={B}")
    kn, vn = (rng.standard_normal((B, Hkv, d)).astype(np.float32) for _ in range(2))
    got, gk, gv, gks, gvs = _gpu.decode(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths, max_seq_len=cap,
                                         k_new=kn, v_new=vn)
    paged = None
    if page:
        kp, vp, ksp, vsp, table = to_pages(rng, p["k"], p["v"], p["ks"], p["vs"], lengths, page)
        paged = paged_decode(p["q"], kp, vp, ksp, vsp, table, lengths, k_new=kn, v_new=vn)
        whole_tiles = page % (info.tile_tokens // 8) == 0  # a wave tile of 8 waves' tokens lies in one page
        assert kvq.paged_decode_plan(paged[5].params).kernel == (kvq.KERNEL_DECODE_VALU if whole_tiles else
                                                                  kvq.KERNEL_DECODE_GENERIC)
    o.append(kn, vn, p["k"], p["v"], p["ks"], p["vs"], positions=L - 1)
    assert np.array_equal(gk, p["k"]) and np.array_equal(gv, p["v"])
    assert np.array_equal(_bits(gks), _bits(p["ks"])) and np.array_equal(_bits(gvs), _bits(p["vs"]))
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=L)
    assert_close(got, want, what=f"G={G} d={d} B={B}")
    if paged is not None:
        assert_close(paged[0], want, what=f"paged G={G} d={d} B={B}")


@pytest.mark.parametrize("d", [48, 80, 112, 192, 240])
@pytest.mark.parametrize("H,N", [(1, 1), (3, 129), (4, 4099)])
def test_padded_lanes_reference_abi(o, H, N, d):
    rng = np.random.default_rng(N + d)
    Q, K, V, ks, vs = _gpu.reference_problem(H, N, d, rng)
    assert kvq.reference_plan(H, N, d).kernel == kvq.KERNEL_DECODE_VALU
    want = o.head_f32(Q, K, V, ks, vs)
    for entry in ("solve", "split", "simple"):
        assert_close(_run(entry, Q, K, V, ks, vs), want, what=f"{entry} H{H} N{N} d{d}")
