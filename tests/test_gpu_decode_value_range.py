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
