"""Matrix-core decode at the ends of fp32's range, under every layout and split
plan of the padded shapes (head groups and head dims that do not fill a tile,
odd capacities, 16-token pages), and one shape that fills its tile.

References are float64 on the CPU over the dequantised cache.
"""
import numpy as np
import pytest

from _util import assert_close, make_problem, textbook_decode_f64
import _gpu
from _gpu import kvq
from oracle import oracle as orc
from test_gpu_paged import paged_decode, to_pages

pytestmark = pytest.mark.gpu

# name: B, Hkv, G, d, capacity, ragged, page, split plan
SHAPES = {
    "static_splits": (1, 2, 3, 128, 2052, False, 0, kvq.SPLITS_STATIC),
    "in_kernel_plan": (5, 2, 6, 96, 700, True, 0, kvq.SPLITS_IN_KERNEL),
    "tile_stream": (70, 2, 2, 80, 200, True, 0, kvq.SPLITS_TILES),
    "odd_capacity": (4, 3, 4, 64, 129, True, 0, kvq.SPLITS_IN_KERNEL),
    "page16": (6, 2, 4, 128, 721, True, 16, kvq.SPLITS_IN_KERNEL),
    "page16_tile_stream": (70, 2, 5, 112, 150, True, 16, kvq.SPLITS_TILES),
    "full_tiles": (5, 2, 4, 128, 704, True, 0, kvq.SPLITS_IN_KERNEL),
}


@pytest.fixture(scope="module")
def o():
    return orc.get()


def _problem(o, name, seed):
    B, Hkv, G, d, cap, ragged, page, plan = SHAPES[name]
    rng = np.random.default_rng(seed)
    lengths = None
    if ragged:
        lengths = rng.integers(1, cap + 1, B).astype(np.int32)
        lengths[:4] = [cap, 33, 31, min(cap, 70)]
    p = make_problem(rng, B, Hkv * G, Hkv, cap, d, o.quantize_rows, lengths=lengths)
    prm = kvq.DecodeParams(B, Hkv * G, Hkv, d, cap, cap, 4096 if ragged else None, *[4096] * 6, 0.0, 0, None, None)
    info = kvq.decode_plan(prm)
    assert (info.kernel, info.split_plan) == (kvq.KERNEL_DECODE_MFMA, plan), (name, info.kernel, info.split_plan)
    return rng, p, lengths, page


def _decode(rng, p, lengths, page):
    if page == 0:
        return _gpu.decode(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths, max_seq_len=p["k"].shape[2])[0]
    out = paged_decode(p["q"], *to_pages(rng, p["k"], p["v"], p["ks"], p["vs"], lengths, page), lengths)
    assert kvq.paged_decode_plan(out[5].params).kernel == kvq.KERNEL_DECODE_MFMA
    return out[0]


@pytest.mark.parametrize("name", SHAPES)
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_non_finite_queries(o, name, bad):
    """A query row with an element that is not finite gives a row of NaN (its
    scores are NaN, infinite, or all -inf); the other heads of its group and
    the other sequences are untouched."""
    rng, p, lengths, page = _problem(o, name, 3)
    want = o.decode_f32(p["q"], p["k"], p["v"], p["ks"], p["vs"],
                        lengths=lengths if lengths is not None else np.full(len(p["q"]), p["k"].shape[2], np.int32))
    B, Hq, d = p["q"].shape
    rows = np.zeros((B, Hq), bool)
    for b, h, dims in ((0, 0, [d - 1]), (B - 1, Hq - 1, [0]), (B // 2, 1, range(d))):
        p["q"][b, h, list(dims)] = bad
        rows[b, h] = True
    got = _decode(rng, p, lengths, page)
    assert np.isnan(got[rows]).all()
    assert_close(got[~rows], want[~rows], what=name)


def _relative_error(got, p, lengths):
    """Largest error of an output row over the row's norm, against float64."""
    want = textbook_decode_f64(p["q"], p["k"], p["v"], p["ks"], p["vs"], lengths=lengths)
    assert np.isfinite(got).all()
    return (np.linalg.norm(got - want, axis=-1) / np.linalg.norm(want, axis=-1)).max()


# fp32 sums of up to 2052 weighted terms and fp32 scores below 2^5: a few 1e-6
# at most; the scales themselves are exact inputs.
RANGE_BOUND = 1e-5


@pytest.mark.parametrize("name", SHAPES)
def test_tiny_v_scales(o, name):
    """V scales near the low end of the normal range: all of a sequence's, and
    those of its first tile (one of them subnormal) before ordinary ones."""
    rng, p, lengths, page = _problem(o, name, 5)
    vs = p["vs"]
    for top in (2.0 ** -100, 2.0 ** -115):
        p["vs"] = vs * np.float32(top / vs.max())
        assert _relative_error(_decode(rng, p, lengths, page), p, lengths) <= RANGE_BOUND
    p["vs"] = vs.copy()
    p["vs"][:, :, :32] *= np.float32(2.0 ** -115)
    p["vs"][:, :, 9] = np.float32(2.0 ** -140)
    assert _relative_error(_decode(rng, p, lengths, page), p, lengths) <= RANGE_BOUND


PADDED = [n for n in SHAPES if n != "full_tiles"]


@pytest.mark.parametrize("name", PADDED)
def test_huge_v_scales(o, name):
    """A V scale of 1.5 * 2^127 at token 0, which has most of the weight, and of
    2^118 elsewhere, on V rows of -1, 0 and 1 (so that the unnormalised sums of
    any part of the sequence are in fp32's range)."""
    rng, p, lengths, page = _problem(o, name, 6)
    d = p["q"].shape[2]
    p["q"] = np.abs(p["q"]) + np.float32(0.5)
    p["k"][:, :, 0] = 127
    p["ks"][:, :, 0] = 10.0 / (127 * 1.3 * d ** 0.5)
    p["ks"][:, :, 1:] *= np.float32(1e-3)
    p["v"] = np.sign(p["v"]).astype(np.int8)
    p["vs"] = p["vs"] / p["vs"].max() * np.float32(2.0 ** 118)
    p["vs"][:, :, 0] = np.float32(1.5 * 2.0 ** 127)
    assert _relative_error(_decode(rng, p, lengths, page), p, lengths) <= RANGE_BOUND


@pytest.mark.parametrize("name", PADDED)
def test_zero_and_non_finite_v_scales(o, name):
    """Scales of 0 give 0; a NaN scale makes every dim of its sequence and kv
    head NaN, an infinite one infinite with V's sign, or NaN where V is 0 in
    that token."""
    rng, p, lengths, page = _problem(o, name, 7)
    G = p["q"].shape[1] // p["k"].shape[1]
    v = p["v"][1, 0, 9] if len(p["q"]) > 1 else p["v"][0, 0, 9]
    b = 1 if len(p["q"]) > 1 else 0
    p["vs"][b, 0, 9] = np.inf
    p["vs"][b, 1, 5] = np.nan
    if b:
        p["vs"][0, 0] = 0.0
    got = _decode(rng, p, lengths, page)
    heads = got[b, :G]
    assert np.array_equal(np.isnan(heads), np.broadcast_to(v == 0, heads.shape))
    assert np.array_equal(np.isposinf(heads), np.broadcast_to(v > 0, heads.shape))
    assert np.isnan(got[b, G:2 * G]).all()
    if b:
        assert (got[0, :G] == 0.0).all()
        assert np.isfinite(got[2:]).all()


@pytest.mark.parametrize("name", PADDED)
def test_weights_far_below_the_largest_scale(o, name):
    """One token whose V scale is 2^26 times the others' and whose weight is
    nothing: the others' weights keep their bits (their products with the
    scale lie below 2^-26 of the running reference)."""
    rng, p, lengths, page = _problem(o, name, 8)
    p["q"] = np.abs(p["q"]) + np.float32(0.5)
    p["k"][:, :, 7] = -127
    p["ks"][:, :, 7] = 100.0
    p["vs"][:, :, 7] = p["vs"].mean() * np.float32(2.0 ** 26)
    assert _relative_error(_decode(rng, p, lengths, page), p, lengths) <= RANGE_BOUND
