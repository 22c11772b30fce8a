"""attention_limbs (dense attention on bf16 matrix cores, three limbs per fp32
value) at the edges of its tiles and dims, against float64.

Bound: an output is a weighted mean of V rows, so it is at most max|V|; the
limb products drop terms below 2^-24 of a product and the sums run in fp32, so
scores of magnitude s (log2 units, s < 40 here) carry absolute errors of a few
s * 2^-24, which are relative errors of the weights: 40 * 4 * 2^-24 < 1e-5, of
max|V| < 6."""
import ctypes
import math

import numpy as np
import pytest
import torch

import _gpu
from _gpu import down, kvq, up

pytestmark = pytest.mark.gpu
BOUND = 6e-5


def _problem(M, N, d, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((n, d)).astype(np.float32) for n in (M, N, N)]


def _exact(q, k, v):
    s = q.astype(np.float64) @ k.astype(np.float64).T / math.sqrt(q.shape[1])
    p = np.exp(s - s.max(1, keepdims=True))
    return p @ v.astype(np.float64) / p.sum(1, keepdims=True)


def _run(q, k, v, splits=None):
    """attention_online's own splits, or kvq.attention with a request."""
    gq, gk, gv = up(q), up(k), up(v)
    out = _gpu.poisoned(q.shape)
    info = kvq.attention_plan(kvq.attention_params(gq, gk, gv, out, num_splits=splits or 0))
    assert info.kernel == kvq.KERNEL_ATTENTION_MFMA
    if splits is None:
        kvq.attention_online(gq, gk, gv, out)
    else:
        kvq.attention(gq, gk, gv, out, num_splits=splits)
    torch.cuda.synchronize()
    return down(out), info


@pytest.mark.parametrize("d", [1, 17, 30, 33, 80, 96, 99, 112, 130, 160, 192, 255])
@pytest.mark.parametrize("M,N,splits", [(1, 1, None), (17, 33, 0), (64, 31, None), (65, 257, None), (300, 95, 1),
                                        (300, 950, None)])
def test_head_dims(d, M, N, splits):
    """Dims between the padded widths (32, 64, 96, 128, 192, 256), whole
    16-byte columns and not; rows past M, keys past N, split and unsplit."""
    q, k, v = _problem(M, N, d, 7 * d + M + N)
    out, _ = _run(q, k, v, splits)
    assert np.abs(out - _exact(q, k, v)).max() <= BOUND


@pytest.mark.parametrize("M,N,d,qblock", [(65, 28640, 128, 64), (65, 28641, 128, 128), (1100, 14560, 64, 128),
                                          (1089, 14561, 64, 256), (1089, 29121, 96, 256), (700, 9001, 256, 128)])
def test_query_blocks(M, N, d, qblock):
    """Each block size on both sides of the lines between them, with a ragged last split."""
    q, k, v = _problem(M, N, d, M + N)
    out, info = _run(q, k, v)
    assert info.query_block == qblock
    rows = np.random.default_rng(1).permutation(M)[:64]
    assert np.abs(out[rows] - _exact(q[rows], k, v)).max() <= BOUND


@pytest.mark.parametrize("M,N,d", [(70, 200, 96), (150, 9000, 64)])
def test_rescaled_maximum(M, N, d):
    """Scores that climb through the keys: the softmax reference moves again and again."""
    q, k, v = _problem(M, N, d, 3)
    k = (k * np.linspace(0.01, 3.0, N, dtype=np.float32)[:, None]).astype(np.float32)
    out, _ = _run(q, k, v)
    assert np.abs(out - _exact(q, k, v)).max() <= BOUND


@pytest.mark.parametrize("splits", [1, None])
def test_overflow_and_non_finite(splits):
    """Values whose limbs overflow or are not finite take fp32 products: a key
    whose score is -inf has weight 0, an infinite V element stays in its column."""
    q, k, v = _problem(90, 300, 96, 11)
    q = np.abs(q) + np.float32(1.0)
    ref = _exact(q, np.delete(k, 40, 0), np.delete(v, 40, 0))
    for big in (np.float32(-3.4e38), np.float32(-np.inf)):
        kk = k.copy()
        kk[40] = big
        out, _ = _run(q, kk, v, splits)
        assert np.abs(out - ref).max() <= BOUND
    vv = v.copy()
    vv[200, 5] = np.inf
    out, _ = _run(q, k, vv, splits)
    rest = np.arange(96) != 5
    assert np.isposinf(out[:, 5]).all() and np.abs(out - _exact(q, k, v))[:, rest].max() <= BOUND


@pytest.mark.parametrize("d", [1, 31, 32, 50, 64, 96, 127, 128, 160, 192, 255, 256])
@pytest.mark.parametrize("M,N,splits", [(70, 95, 1), (300, 950, None), (1089, 2100, 2), (2100, 2050, None)])
def test_fp32_products_at_tile_edges(d, M, N, splits):
    """Every wave on the fp32 products (an infinite V element and a key of -inf
    scores in the keys of each split): each block size, rows past M, keys past
    N, dims past d."""
    q, k, v = _problem(M, N, d, M + N + d)
    q = np.abs(q) + np.float32(0.5)
    out, info = _run(q, k, v, splits)
    dead = np.arange(info.chunk // 2, N, max(16, info.chunk // 3))
    k[dead] = -np.inf
    v[dead[:-1]] = 0.0
    ref = _exact(q, np.delete(k, dead, 0), np.delete(v, dead, 0))
    out, _ = _run(q, k, v, splits)
    assert np.abs(out - ref).max() <= BOUND
    v[N // 3, d // 2] = -np.inf
    out, _ = _run(q, k, v, splits)
    rest = np.arange(d) != d // 2
    assert (out[:, d // 2] == -np.inf).all() if N // 3 not in dead else np.isnan(out[:, d // 2]).all()
    assert rest.sum() == 0 or np.abs(out - ref)[:, rest].max() <= BOUND


def test_non_finite_values_cost_a_few_times_more_at_most():
    """One infinity in V sends every wave to the fp32 products, which take 2-3
    times as long as the limbs (one query at a time they took 100 times)."""
    q, k, v = (torch.randn((4096, 128), device="cuda") for _ in range(3))
    out = torch.empty_like(q)

    def best(v):
        t = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            kvq.attention_online(q, k, v, out)
            a.record()
            for _ in range(5):
                kvq.attention_online(q, k, v, out)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t)

    finite = best(v)
    v[2048, 3] = np.inf
    assert best(v) < 12 * finite


@pytest.mark.parametrize("M,N,d", [(70, 95, 96), (300, 950, 50), (1089, 2100, 128)])
@pytest.mark.parametrize("splits", [1, None])
def test_values_below_the_limbs_range(M, N, d, splits):
    """Values whose third limb is below bf16's subnormals keep fp32's precision:
    V rows of 2^-118, and tiny q against huge K and the reverse.  Error over the
    output's norm; BOUND's scores, V of one magnitude."""
    q, k, v = _problem(M, N, d, M)

    def check(q, k, v, what):
        out, _ = _run(q, k, v, splits)
        want = _exact(q, k, v)
        err = np.linalg.norm(out - want, axis=1) / np.linalg.norm(want, axis=1)
        assert err.max() <= BOUND, (what, err.max())

    check(q, k, (v * 2.0 ** -118).astype(np.float32), "V")
    check((q * 2.0 ** -118).astype(np.float32), (k * 2.0 ** 118).astype(np.float32), v, "q")
    check((q * 2.0 ** 118).astype(np.float32), (k * 2.0 ** -118).astype(np.float32), v, "K")
    q[M // 2] *= np.float32(2.0 ** -118)  # one row of many
    q[3] = 0.0
    check(q, k, v, "one row")


@pytest.mark.parametrize("M,N,d", [(300, 950, 96), (70, 9000, 50), (32700, 1100, 128)])
def test_capture_without_an_eager_call_before(M, N, d):
    """Calls that ran without memory before they were split can be captured on
    a stream that has none yet (they run unsplit there), with eager calls on
    the same stream between the replays."""
    q, k, v = (up(x) for x in _problem(M, N, d, 21))
    assert kvq.attention_plan(kvq.attention_params(q, k, v, q)).kernel == kvq.KERNEL_ATTENTION_MFMA
    rows = np.random.default_rng(2).permutation(M)[:64]
    out, eager = torch.empty_like(q), torch.empty_like(q)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        kvq.attention_online(q, k, v, out)
    for rep in range(3):
        q.copy_(up(_problem(M, 1, d, 30 + rep)[0]))
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            kvq.attention_online(q, k, v, eager)
        s.synchronize()
        want = _exact(down(q)[rows], down(k), down(v))
        for got in (out, eager):
            assert np.abs(down(got)[rows] - want).max() <= BOUND, rep


@pytest.mark.parametrize("d", [30, 96, 192])
@pytest.mark.parametrize("M,N,splits", [(1, 5000, 40), (70, 1000, 3), (300, 950, 1 << 20), (1089, 2100, 2)])
def test_caller_workspace_splits_and_null(d, M, N, splits):
    """A caller's own workspace (NaN-filled, the size the query gives) at head
    dims without a few-query kernel: a split request, and the same with NULL."""
    q, k, v = _problem(M, N, d, d + M)
    want = _exact(q, k, v)
    g = [up(x) for x in (q, k, v)]
    out = _gpu.poisoned(q.shape)
    p = kvq.attention_params(*g, out, num_splits=splits)
    info = kvq.attention_plan(p)
    assert info.splits > 1 and info.workspace_bytes > 0
    ws = torch.full((info.workspace_bytes,), 0xFF, dtype=torch.uint8, device="cuda")
    kvq.attention(*g, out, num_splits=splits, workspace=ws)
    torch.cuda.synchronize()
    assert np.abs(down(out) - want).max() <= BOUND
    assert (ws != 0xFF).any()  # the records were written
    out.fill_(float("nan"))
    assert kvq.lib().kvq_attention_launch(ctypes.byref(p), None, 0, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert np.abs(down(out) - want).max() <= BOUND
