"""Timed cases: the calls a user of this library makes, over the sizes they make them at.

  listed()             the named cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  device inputs and the launch handle a program keeps
  run(state)           one call through the public entry points, and its outputs
  exact(case, seed)    the same outputs from plain torch in 64 bits
  work(case)           bytes and operations one call cannot do without
  tolerance(case)      how far two correct implementations may differ

A case's "op" names the entry point:
  abi        kv_int8_split_launch, the reference's stream-aware C entry point:
             one query per head over [H, N, d] int8 caches, caller scratch S
  decode     kvq.Decoder: batched (grouped-query) decode over a contiguous cache
  paged      kvq.PagedDecoder: the same over a page pool with block tables
  prefill    kvq.prefill: bulk int8 quantisation of K/V rows into a cache
  attention  attention_online_launch: dense fp32 attention of M queries over N keys
"""
import ctypes
import importlib
import math

import numpy as np
import torch

kvq = importlib.import_module("cuda-operators_amd").kvq

DEV = "cuda"
CHUNK = 1 << 26  # elements drawn at a time


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _abi(name, H, N, d):
    return {"name": name, "op": "abi", "H": H, "N": N, "d": d}


def _decode(name, B, Hq, Hkv, d, lo, hi, append, dist="normal", page=0):
    return {"name": name, "op": "paged" if page else "decode", "B": B, "Hq": Hq, "Hkv": Hkv, "d": d, "lo": lo, "hi": hi,
            "append": append, "dist": dist, "page": page}


def _prefill(name, B, Hkv, L, d, dtype, page):
    return {"name": name, "op": "prefill", "B": B, "Hkv": Hkv, "L": L, "d": d, "dtype": dtype, "page": page}


def _attention(name, M, N, d):
    return {"name": name, "op": "attention", "M": M, "N": N, "d": d}


def listed():
    return [
        # The drop-in caller's smallest decode: one short sequence, where the
        # call's own latency is what counts.
        _abi("abi_h8_n1024_d64", 8, 1024, 64),
        # The same entry point in a single-stream chat loop: one sequence of a
        # 32-head model, at whatever odd length the loop has reached.
        _abi("abi_h32_n4099_d128", 32, 4099, 128),
        # The benchmark step: a multi-head model's decode with the new token's
        # quantise-and-append fused into it.
        _decode("mha_b8_h32_l4096_append", 8, 32, 32, 128, 4096, 4096, True),
        # A grouped-query model serving a small batch of unequal contexts.
        _decode("gqa_b16_h32_8_ragged", 16, 32, 8, 128, 1024, 8192, False),
        # One very long context; K with outlier channels, as trained models have.
        _decode("gqa_b1_h32_8_l131072", 1, 32, 8, 128, 131072, 131072, False, "outlier"),
        # A full serving batch of a large grouped-query model, heavy-tailed
        # activations, append fused.
        _decode("gqa_b256_h64_8_ragged_append", 256, 64, 8, 128, 512, 4096, True, "student_t"),
        # A serving engine's paged cache with 16-token pages scattered over the pool.
        _decode("paged16_b32_h32_8_append", 32, 32, 8, 128, 200, 4000, True, "normal", 16),
        # A head dim between the powers of two and three query heads per kv head.
        _decode("gqa_b8_h24_8_d96_ragged", 8, 24, 8, 96, 500, 3000, False),
        # Prompt ingestion: bf16 K/V rows of a batch of prompts into a paged cache.
        _prefill("prefill_b16_h8_l2047_bf16_page64", 16, 8, 2047, 128, "bf16", 64),
        # Dense attention of a prompt over itself.
        _attention("attention_m4096_n4096_d128", 4096, 4096, 128),
        # Dense attention of one query over a long fp32 cache.
        _attention("attention_m1_n65536_d128", 1, 65536, 128),
        # Dense attention at ragged sizes and a head dim between the powers of two.
        _attention("attention_m1000_n3001_d96", 1000, 3001, 96),
    ]


MAX_BYTES = 1.0e9          # of cache (or rows) a drawn case touches
MAX_MND = 4096 * 4096 * 128  # M * N * d of a drawn dense attention


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    op = rng.choice(["decode"] * 4 + ["paged"] * 2 + ["abi", "prefill"] + ["attention"] * 2)
    d = rng.choice([64, 80, 96, 112, 128, 128, 128, 192, 256])
    if op == "abi":
        H = rng.choice([1, 4, 8, 12, 16, 24, 32, 40, 64, 128])
        N = _log_int(rng, 64, 65536)
        N = max(1, min(N, int(MAX_BYTES / (H * (2 * d + 8)))))
        return {k: v for k, v in _abi("", H, N, d).items() if k != "name"}
    if op == "attention":
        d = rng.choice([32, 64, 64, 80, 96, 128, 128, 128, 256])
        M = _log_int(rng, 1, 8192)
        N = _log_int(rng, 64, 131072)
        N = max(1, min(N, MAX_MND // (M * d)))
        return {k: v for k, v in _attention("", M, N, d).items() if k != "name"}
    if op == "prefill":
        Hkv = rng.choice([1, 2, 4, 8, 8, 16, 32])
        L = _log_int(rng, 1, 8192)
        dtype = rng.choice(["f32", "bf16", "bf16"])
        B = _log_int(rng, 1, 256)
        B = max(1, min(B, int(MAX_BYTES / (2 * Hkv * L * d * (5 if dtype == "f32" else 3)))))
        page = rng.choice([0, 0, 16, 32, 64, 128])
        return {k: v for k, v in _prefill("", B, Hkv, L, d, dtype, page).items() if k != "name"}
    G = rng.choice([1, 1, 2, 3, 4, 4, 5, 6, 7, 8, 8, 12, 16])
    Hkv = rng.choice([8, 16, 32, 40]) if G == 1 else rng.choice([1, 2, 4, 8, 8, 8])
    hi = _log_int(rng, 64, 32768)
    lo = max(1, hi // rng.choice([1, 1, 2, 4, 8]))
    B = _log_int(rng, 1, 256)
    B = max(1, min(B, int(MAX_BYTES / (hi * Hkv * (2 * d + 8)))))
    if B == 1:
        lo = hi
    append = rng.random() < 0.5
    dist = rng.choice(["normal", "normal", "student_t", "outlier"])
    page = rng.choice([16, 16, 32, 64, 128]) if op == "paged" else 0
    return {k: v for k, v in _decode("", B, G * Hkv, Hkv, d, lo, hi, append, dist, page).items() if k != "name"}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _values(gen, shape, dist):
    x = torch.randn(shape, generator=gen, device=DEV)
    if dist == "student_t":  # 4 degrees of freedom
        chi = torch.randn(shape, generator=gen, device=DEV).square_()
        for _ in range(3):
            chi += torch.randn(shape, generator=gen, device=DEV).square_()
        x = x.div_(chi.div_(4.0).sqrt_())
    return x


def _cache(gen, X, H, T, d, dist, gain=None):
    """int8 rows [X, H, T, d] and fp32 scales [X, H, T], as a per-token quantiser leaves them; gain [H, d] scales channels."""
    q = torch.empty((X, H, T, d), dtype=torch.int8, device=DEV)
    s = torch.empty((X, H, T), dtype=torch.float32, device=DEV)
    step = max(1, CHUNK // (H * T * d))
    for i in range(0, X, step):
        x = _values(gen, (min(step, X - i), H, T, d), dist)
        if gain is not None:
            x *= gain[:, None, :]
        s[i:i + step] = x.abs().amax(-1) / 127.0
        q[i:i + step] = (x / s[i:i + step, :, :, None]).round_().clamp_(-127.0, 127.0).to(torch.int8)
    return q, s


def _gain(gen, H, d):
    """One channel in a hundred 20 times the others."""
    g = torch.ones((H, d), device=DEV)
    n = max(1, math.ceil(0.01 * d))
    pick = torch.rand((H, d), generator=gen, device=DEV).argsort(1)[:, :n]
    return g.scatter_(1, pick, 20.0)


def _lengths(case, seed):
    """B lengths evenly spread over [lo, hi], in an order of the seed (their sum is the case's)."""
    n = np.linspace(case["lo"], case["hi"], case["B"]).round().astype(np.int32) if case["B"] > 1 else np.array([case["hi"]], np.int32)
    return np.random.default_rng(seed).permutation(n)


def _table(case, seed, tokens):
    """Block table [B, pages per sequence] over a shuffled pool with a few spare pages, and the pool size."""
    per = -(-tokens // case["page"])
    pool = case["B"] * per + 7
    ids = np.random.default_rng(seed + 1).permutation(pool)[:case["B"] * per]
    return torch.from_numpy(ids.reshape(case["B"], per).astype(np.int32)).to(DEV), pool


def _decode_inputs(case, seed):
    gen = _gen(seed)
    B, Hq, Hkv, d, hi = (case[k] for k in ("B", "Hq", "Hkv", "d", "hi"))
    lens = _lengths(case, seed)
    kdist = vdist = case["dist"]
    gain = None
    if kdist == "outlier":
        kdist = vdist = "normal"
        gain = _gain(gen, Hkv, d)
    i = {"lens": lens, "q": torch.randn((B, Hq, d), generator=gen, device=DEV),
         "lengths": torch.from_numpy(lens).to(DEV) if case["lo"] != hi else None}
    X, T = B, hi
    if case["page"]:
        i["table"], X = _table(case, seed, hi)
        T = case["page"]
    i["k"], i["ks"] = _cache(gen, X, Hkv, T, d, kdist, gain)
    i["v"], i["vs"] = _cache(gen, X, Hkv, T, d, vdist)
    i["kn"] = i["vn"] = None
    if case["append"]:
        i["kn"] = _values(gen, (B, Hkv, d), kdist)
        if gain is not None:
            i["kn"] *= gain
        i["vn"] = _values(gen, (B, Hkv, d), vdist)
    return i


def _abi_inputs(case, seed):
    gen = _gen(seed)
    H, N, d = case["H"], case["N"], case["d"]
    k, ks = _cache(gen, 1, H, N, d, "normal")
    v, vs = _cache(gen, 1, H, N, d, "normal")
    return {"q": torch.randn((H, d), generator=gen, device=DEV), "k": k[0], "v": v[0], "ks": ks[0], "vs": vs[0]}


def _prefill_inputs(case, seed):
    gen = _gen(seed)
    B, Hkv, L, d = case["B"], case["Hkv"], case["L"], case["d"]
    dt = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
    i = {"k": (torch.randn((B, Hkv, L, d), generator=gen, device=DEV) * 3.0).to(dt),
         "v": (torch.randn((B, Hkv, L, d), generator=gen, device=DEV) * 3.0).to(dt)}
    # Prompts that continue a conversation start past its earlier turns.
    i["start"] = np.random.default_rng(seed).integers(0, 33, B).astype(np.int32)
    i["table"] = None
    shape = (B, Hkv, L + 32)
    if case["page"]:
        i["table"], pool = _table(case, seed, L + 32)
        shape = (pool, Hkv, case["page"])
    i["shape"] = shape
    return i


def _attention_inputs(case, seed):
    gen = _gen(seed)
    M, N, d = case["M"], case["N"], case["d"]
    return {"q": torch.randn((M, d), generator=gen, device=DEV), "k": torch.randn((N, d), generator=gen, device=DEV),
            "v": torch.randn((N, d), generator=gen, device=DEV)}


# ---------------------------------------------------------------------------
# one call
# ---------------------------------------------------------------------------
def prepare(case, seed):
    op = case["op"]
    stream = torch.cuda.current_stream().cuda_stream
    if op == "abi":
        i = _abi_inputs(case, seed)
        out = torch.empty_like(i["q"])
        scratch = torch.empty(case["H"] * case["N"], device=DEV)
        args = [ctypes.c_void_p(t.data_ptr()) for t in (i["q"], i["k"], i["v"], i["ks"], i["vs"], out)]
        args += [case["H"], case["N"], case["d"], ctypes.c_void_p(scratch.data_ptr()), stream]
        return {"call": kvq.lib().kv_int8_split_launch, "args": args, "out": out, "keep": (i, scratch)}
    if op == "attention":
        i = _attention_inputs(case, seed)
        out = torch.empty_like(i["q"])
        args = [ctypes.c_void_p(t.data_ptr()) for t in (i["q"], i["k"], i["v"], out)]
        args += [case["M"], case["N"], case["d"], stream]
        return {"call": kvq.lib().attention_online_launch, "args": args, "out": out, "keep": i}
    if op == "prefill":
        i = _prefill_inputs(case, seed)
        shape, d = i["shape"], case["d"]
        cache = {n: torch.zeros(shape + (d,), dtype=torch.int8, device=DEV) for n in ("k", "v")}
        cache.update({n: torch.zeros(shape, device=DEV) for n in ("ks", "vs")})
        return {"prefill": (i["k"], i["v"], cache["k"], cache["v"], cache["ks"], cache["vs"]),
                "start": torch.from_numpy(i["start"]).to(DEV), "table": i["table"], "out": cache, "stream": stream}
    i = _decode_inputs(case, seed)
    out = torch.empty_like(i["q"])
    if op == "paged":
        dec = kvq.PagedDecoder(i["q"], i["k"], i["v"], i["ks"], i["vs"], i["table"], i["lengths"], out,
                               max_seq_len=case["hi"], k_new=i["kn"], v_new=i["vn"])
    else:
        dec = kvq.Decoder(i["q"], i["k"], i["v"], i["ks"], i["vs"], out, lengths=i["lengths"],
                          max_seq_len=case["hi"], k_new=i["kn"], v_new=i["vn"])
    outs = {"out": out}
    if case["append"]:
        outs.update(k=i["k"], v=i["v"], ks=i["ks"], vs=i["vs"])
    return {"decoder": dec, "stream": stream, "out": outs}


def run(state):
    if "decoder" in state:
        state["decoder"](state["stream"])
    elif "prefill" in state:
        kvq.prefill(*state["prefill"], start=state["start"], block_table=state["table"], stream=state["stream"])
    else:
        code = state["call"](*state["args"])
        if code:
            raise RuntimeError(f"hipError {code}")
    return state["out"]


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _attend(q, k, v, ks, vs):
    """q [H, G, d], k/v [H, n, d] int8, scales [H, n] -> [H, G, d]."""
    s = (q.double() @ k.double().transpose(1, 2).contiguous()) * ks.double()[:, None, :] / math.sqrt(q.shape[-1])
    return (s.softmax(-1) * vs.double()[:, None, :]) @ v.double()


def _quantise(x):
    """The append rule on fp32 rows [..., d], on the CPU: int8 rows and scales."""
    x = x.cpu()
    s = x.abs().amax(-1) / 127.0
    return (x / s[..., None]).round().clamp(-127.0, 127.0).to(torch.int8).to(DEV), s.to(DEV)


def _exact_decode(case, seed):
    i = _decode_inputs(case, seed)
    B, Hq, Hkv, d, page = (case[k] for k in ("B", "Hq", "Hkv", "d", "page"))
    if case["append"]:
        last = torch.from_numpy(i["lens"].astype(np.int64)).to(DEV) - 1
        at = torch.arange(B, device=DEV)
        if page:
            at, last = i["table"][at, last // page].long(), last % page
        for c, s, n in (("k", "ks", "kn"), ("v", "vs", "vn")):
            i[c][at, :, last], i[s][at, :, last] = _quantise(i[n])
    out = torch.empty((B, Hkv, Hq // Hkv, d), dtype=torch.float64, device=DEV)
    for b, n in enumerate(int(x) for x in i["lens"]):
        part = [i[c][b] for c in ("k", "v", "ks", "vs")]
        if page:
            ids = i["table"][b, :-(-n // page)].long()
            part = [i[c][ids].transpose(0, 1).reshape((Hkv, -1, d)[:t]) for c, t in (("k", 3), ("v", 3), ("ks", 2), ("vs", 2))]
        k, v, ks, vs = (t[:, :n] for t in part)
        out[b] = _attend(i["q"][b].view(Hkv, -1, d), k, v, ks, vs)
    outs = {"out": out.view(B, Hq, d)}
    if case["append"]:
        outs.update(k=None, v=None, ks=i["ks"].double(), vs=i["vs"].double())
    return outs


def _exact_prefill(case, seed):
    i = _prefill_inputs(case, seed)
    L, page = case["L"], case["page"]
    outs = {"k": None, "v": None}
    for n in ("k", "v"):
        s = torch.zeros(i["shape"], dtype=torch.float64, device=DEV)
        amax = i[n].double().abs().amax(-1) / 127.0
        for b, p in enumerate(int(x) for x in i["start"]):
            if page:
                t = torch.arange(p, p + L, device=DEV)
                s[i["table"][b, t // page].long(), :, t % page] = amax[b].transpose(0, 1)
            else:
                s[b, :, p:p + L] = amax[b]
        outs[n + "s"] = s
    return outs


def _exact_attention(case, seed):
    i = _attention_inputs(case, seed)
    k, v = i["k"].double().transpose(0, 1).contiguous(), i["v"].double()
    rows = max(1, CHUNK // case["N"])
    return torch.cat([(q.double() @ k / math.sqrt(case["d"])).softmax(-1) @ v for q in i["q"].split(rows)])


def exact(case, seed):
    if case["op"] == "abi":
        i = _abi_inputs(case, seed)
        return _attend(i["q"][:, None, :], i["k"], i["v"], i["ks"], i["vs"])[:, 0]
    if case["op"] == "attention":
        return _exact_attention(case, seed)
    return (_exact_prefill if case["op"] == "prefill" else _exact_decode)(case, seed)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def work(case):
    d = case["d"]
    if case["op"] == "abi":
        H, N = case["H"], case["N"]
        return {"bytes": H * N * (2 * d + 8) + 8 * H * d, "flops": 4 * H * N * d}
    if case["op"] == "attention":
        M, N = case["M"], case["N"]
        return {"bytes": 8 * (M + N) * d, "flops": 4 * M * N * d}
    if case["op"] == "prefill":
        rows = 2 * case["B"] * case["Hkv"] * case["L"]
        return {"bytes": rows * (d * (4 if case["dtype"] == "f32" else 2) + d + 4), "flops": 4 * rows * d}
    B, Hq, Hkv = case["B"], case["Hq"], case["Hkv"]
    tokens = int(_lengths(case, 0).sum())
    n = tokens * Hkv * (2 * d + 8) + 8 * B * Hq * d
    if case["append"]:  # the new rows are read as fp32 instead of from the cache, and written
        n += 8 * B * Hkv * d
    return {"bytes": n, "flops": 4 * tokens * Hq * d}


def tolerance(case):
    """Four times the largest error against 64 bits that fp32 sums show over these ranges: dense attention 1.1e-6;
    decode 6.6e-6 over long sequences summed token by token, 4.5e-5 where the values are heavy-tailed.  Quantised
    bytes and scales follow one stated rule and are the same everywhere."""
    if case["op"] == "prefill":
        return "exact"
    if case["op"] == "attention":
        return {"rel": 5e-6}
    return {"rel": 2e-4 if case.get("dist") == "student_t" else 3e-5}
