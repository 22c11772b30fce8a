"""Prefill quantiser at row lengths between the powers of two: the smallest and
largest that the padded lanes take (8 and 248 elements), one 16-byte piece to
either side of the 64- and 128-element layouts, and lengths that only fp32 rows
or neither type divides into whole pieces.  Bit-exact as in test_gpu_prefill.
"""
import pytest

import test_gpu_prefill as base
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def o():
    return orc.get()


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("d", [4, 8, 24, 40, 44, 56, 72, 80, 112, 120, 136, 192, 248, 98])
def test_contiguous(o, d, bf16):
    base.test_prefill_contiguous(o, d, bf16)


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("d,page", [(8, 16), (80, 32), (112, 64), (192, 16), (248, 128)])
def test_paged(o, d, page, bf16):
    base.test_prefill_paged(o, d, page, bf16)
