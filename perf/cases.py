"""Timed cases of the EXL3 expert path and of the dense EXL3 linear, through the entry points a program calls.

Shapes are this repository's own: the 48-layer decoder of bench.py (H 2048, I 512, 512 experts, top-10, 3 bits), the
wider experts of its second configuration (H 4096, I 1536, 128 experts, top-8, 2 to 4 bits) and the dense projections
of one decoder layer (bench.py's LINEAR_GROUPS). Weights are seeded random trellis words (any bit stream is a valid
trellis), suh +-1 and svh +-0.02; routing is Zipf(1.1) for decode and softmax top-k of normal logits for prefill.

Kinds:
  token    one decode step of M rows through `layers` MoE layers, replayed from a HIP graph, as an engine decodes
  cached   the same through the expert cache (ExpertStore.forward_cached), every pick in an HBM slot
  moe      one moe_forward call (decode sizes below 103 rows at top-10, prefill above)
  ltoken   one decode step of M rows through `layers` layers of dense projections, replayed from a HIP graph
  linear   one FusedGroup call
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qwen38-flash-next-b70-offload_amd"))

from exl3xpu.linear import FusedGroup, C as linear_ops          # noqa: E402
from exl3xpu.moe_offload import BlobLayout, ExpertStore, ops    # noqa: E402

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# the fused groups of one decoder layer's dense projections: input size, output widths of the shards
GROUPS = ((2048, (2048, 2048, 4096, 4096)), (4096, (2048,)), (2048, (512, 512)), (512, (2048,)))


def _moe(name, M, H=2048, I=512, K=3, E=512, topk=10, routing="zipf", dtype="bf16", kind="moe", layers=1):  # noqa: E741
    return {"name": name, "kind": kind, "M": M, "H": H, "I": I, "K": K, "E": E, "topk": topk, "routing": routing,
            "dtype": dtype, "layers": layers}


def _wide(name, M, K, routing="softmax", dtype="bf16"):
    return _moe(name, M, H=4096, I=1536, K=K, E=128, topk=8, routing=routing, dtype=dtype)


def _lin(name, M, group, K=3, cb=2, int8=False, dtype="bf16"):
    return {"name": name, "kind": "linear", "M": M, "group": group, "K": K, "cb": cb, "int8": int8, "dtype": dtype}


def listed():
    return [
        # one user decoding: a token through the 48 MoE layers, the framework's headline workload
        _moe("token_bs1", 1, kind="token", layers=48),
        # two users through the expert cache in its steady state (hits), where a server spends most of its calls
        _moe("cached_bs2", 2, E=48, kind="cached", layers=6),
        # a server's decode batch, small and large; Zipf routing, so rows share experts
        _moe("decode_bs16", 16),
        _moe("decode_bs64", 64, dtype="fp16"),
        # the wider experts at 4 bits, a small decode batch
        _wide("decode_wide_bs6", 6, 4),
        # a short ragged prompt: few rows per expert, every expert read
        _moe("prefill_301", 301, routing="softmax"),
        # the wider experts at 2 bits, a ragged chunk
        _wide("prefill_wide_777", 777, 2),
        # a chunk of chunked prefill, and the largest chunk
        _moe("prefill_2048", 2048, routing="softmax"),
        _moe("prefill_8192", 8192, routing="softmax"),
        # the dense projections of one user's token (16 layers, so that the weights do not stay in cache)
        {"name": "linear_token_bs1", "kind": "ltoken", "M": 1, "K": 3, "cb": 2, "dtype": "bf16", "layers": 16},
        # a decode batch above the smallest sizes, and a prefill chunk, through the widest group
        _lin("linear_m40", 40, 0, K=4),
        _lin("linear_m1024", 1024, 0),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["token", "cached", "decode", "decode", "prefill", "prefill", "ltoken", "linear", "linear"])
    dt = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    K = rng.choice([2, 3, 3, 4])
    if kind == "token":
        c = _moe("", rng.randint(1, 5), K=K, kind="token", layers=rng.randint(8, 48), dtype=dt)
    elif kind == "cached":
        c = _moe("", rng.randint(1, 6), K=K, E=48, kind="cached", layers=rng.randint(3, 6), dtype=dt)
    elif kind == "decode":
        c = (_wide("", logint(1, 100), K, routing=rng.choice(["zipf", "softmax"]), dtype=dt) if rng.random() < 0.35 else
             _moe("", logint(1, 102), K=K, routing=rng.choice(["zipf", "zipf", "softmax"]), dtype=dt))
    elif kind == "prefill":
        c = (_wide("", logint(129, 1800), K, dtype=dt) if rng.random() < 0.35 else
             _moe("", logint(103, 8000), K=K, routing=rng.choice(["zipf", "softmax", "softmax"]), dtype=dt))
    elif kind == "ltoken":
        c = {"kind": "ltoken", "M": rng.randint(1, 8), "K": rng.choice([2, 3, 3, 4, 5, 6]), "cb": 2, "dtype": dt,
             "layers": rng.randint(4, 16)}
    else:
        K, cb, int8 = rng.choice([(2, 2, 0), (3, 2, 0), (3, 2, 0), (4, 2, 0), (5, 2, 0), (6, 2, 0), (4, 1, 0), (6, 0, 0),
                                  (4, 2, 1)])
        M = logint(17, 2048) if int8 else logint(1, 2048)
        c = _lin("", M, rng.randrange(4), K=K, cb=cb, int8=bool(int8), dtype=dt)
    c.pop("name", None)
    return c


# ---- inputs -----------------------------------------------------------------------------------------------------------

def _gen(seed, *more):
    s = int(seed) % (1 << 40)
    for m in more:
        s = (s * 1000003 + int(m) + 17) % (1 << 62)
    return torch.Generator(device=DEV).manual_seed(s)


def _words(g, *shape):
    return torch.randint(-(1 << 31), 1 << 31, shape, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)


def _signs(g, *shape):
    return (torch.randint(0, 2, shape, generator=g, device=DEV) * 2 - 1).to(torch.float16)


def _blobs(case, seed, n):
    """uint8 [n, blob] experts on the device: random trellis words, suh +-1, svh +-0.02."""
    H, I, K = case["H"], case["I"], case["K"]       # noqa: E741
    lay = BlobLayout(H, I, K)
    g = _gen(seed, 1)
    out = torch.empty(n, lay.nbytes // 4, dtype=torch.int32, device=DEV)
    for i in range(0, n, 64):
        out[i:i + 64] = _words(g, min(64, n - i), lay.nbytes // 4)
    out = out.view(torch.uint8)
    for name, off, nb in lay.fields:
        if name.startswith("su") or name.startswith("sv"):
            v = _signs(g, n, nb // 2) * (1.0 if name.startswith("su") else 0.02)
            out[:, off:off + nb] = v.to(torch.float16).view(torch.uint8)
    return out


def _routing(case, seed, layer):
    """ids int32 / w fp32 [M, topk]: Zipf(1.1) over a permutation of the experts (Gumbel top-k) with softmax weights
    of normal logits, or the top-k of the softmax of normal logits, renormalised."""
    M, E, topk = case["M"], case["E"], case["topk"]
    g = _gen(seed, 2, layer)
    if case["routing"] == "zipf":
        perm = torch.randperm(E, generator=g, device=DEV)
        u = torch.rand(M, E, generator=g, device=DEV, dtype=torch.float64).clamp_(1e-12, 1 - 1e-12)
        score = -1.1 * torch.log(torch.arange(1, E + 1, device=DEV, dtype=torch.float64)) - torch.log(-torch.log(u))
        ids = perm[torch.topk(score, topk, dim=-1).indices]
        w = torch.softmax(torch.randn(M, topk, generator=g, device=DEV), dim=-1)
    else:
        p = torch.softmax(torch.randn(M, E, generator=g, device=DEV), dim=-1)
        w, ids = torch.topk(p, topk, dim=-1)
        w = w / w.sum(-1, keepdim=True)
    return ids.to(torch.int32).contiguous(), w.float().contiguous()


def _acts(case, seed, cols, layer=0):
    g = _gen(seed, 3, layer)
    return torch.randn(case["M"], cols, generator=g, device=DEV).to(DTYPES[case["dtype"]])


def _pool(case):
    """Distinct experts of a case: a layer's own, and for several layers a pool larger than the 256 MB cache."""
    return case["E"] if case["kind"] != "cached" else case["E"] * case["layers"]


def _expert_of(case, seed, layer):
    """Pool index of every expert of a layer, int64 [E]."""
    E = case["E"]
    if case["kind"] == "cached":
        return torch.arange(layer * E, (layer + 1) * E, device=DEV)
    if case["layers"] == 1:
        return torch.arange(E, device=DEV)
    return torch.randperm(E, generator=_gen(seed, 4, layer), device=DEV)


def _shards(case, seed, group, layer=0):
    """(trellis int16, suh, svh) of every shard of a fused group, on the device."""
    k, widths = GROUPS[group]
    g = _gen(seed, 5, layer, group)
    return [(_words(g, k // 16, n // 16, 8 * case["K"]).view(torch.int16), _signs(g, k),
             (_signs(g, n) * 0.02).to(torch.float16)) for n in widths]


def _capture(fn):
    """A graph of fn() after a call outside it (which sizes the library's buffers) on a side stream."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = fn()
    return graph, outs


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case}
    if kind in ("moe", "token", "cached"):
        L, E, H, I, K = case["layers"], case["E"], case["H"], case["I"], case["K"]     # noqa: E741
        blobs = _blobs(case, seed, _pool(case))
        calls = []
        if kind == "cached":
            store = ExpertStore(H, I, K, E, n_slots=E * L, max_layers=L)
            for li in range(L):
                store.add_layer(li, blobs[li * E:(li + 1) * E].cpu())
            for li in range(L):
                ids, w = _routing(case, seed, li)
                calls.append((li, _acts(case, seed, H, li), ids, w))
            st.update(store=store, calls=calls)
            st["graph"], st["outs"] = _capture(lambda: [store.forward_cached(*c) for c in calls])
            return st
        base = blobs.data_ptr()
        for li in range(L):
            table = base + _expert_of(case, seed, li) * blobs.shape[1]
            ids, w = _routing(case, seed, li)
            calls.append((_acts(case, seed, H, li), ids, w, table.contiguous(), I, K, E))
        st.update(blobs=blobs, calls=calls)
        if kind == "token":
            X = ops()
            st["graph"], st["outs"] = _capture(lambda: [X.moe_forward(*c) for c in calls])
        return st
    groups = range(len(GROUPS)) if kind == "ltoken" else [case["group"]]
    layers = range(case.get("layers", 1))
    calls = [(FusedGroup(_shards(case, seed, gi, li), DEV, cb=case["cb"]), _acts(case, seed, GROUPS[gi][0], li * 8 + gi))
             for li in layers for gi in groups]
    st["calls"] = calls
    if kind == "ltoken":
        st["graph"], st["outs"] = _capture(lambda: [fg(x) for fg, x in calls])
    return st


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    if state["kind"] == "moe":
        return ops().moe_forward(*state["calls"][0])
    fg, x = state["calls"][0]
    if not state["case"]["int8"]:
        return fg(x)
    linear_ops().exl3_set_int8(1)                   # the opt-in W8A8 route, for this call only
    y = fg(x)
    linear_ops().exl3_set_int8(0)
    return y


# ---- work and tolerance -----------------------------------------------------------------------------------------------

def _distinct(case):
    """Expected distinct experts of one call."""
    M, E, topk = case["M"], case["E"], case["topk"]
    if case["routing"] != "zipf":
        return E * (1 - (1 - topk / E) ** M)
    q = np.arange(1, E + 1, dtype=np.float64) ** -1.1
    q /= q.sum()
    lo, hi = 0.0, 1e6                               # inclusion 1 - exp(-t q) with t such that topk are picked
    for _ in range(100):
        t = (lo + hi) / 2
        lo, hi = (t, hi) if (1 - np.exp(-t * q)).sum() < topk else (lo, t)
    return float((1 - np.exp(-t * q * M)).sum())


def work(case):
    esz = 4 if case["dtype"] == "fp32" else 2
    M = case["M"]
    if case["kind"] in ("moe", "token", "cached"):
        H, I, L = case["H"], case["I"], case["layers"]           # noqa: E741
        blob = BlobLayout(H, I, case["K"]).nbytes
        return {"bytes": L * (_distinct(case) * blob + 2 * M * H * esz + M * case["topk"] * 8),
                "flops": L * 2.0 * M * case["topk"] * 3 * H * I}
    groups = GROUPS if case["kind"] == "ltoken" else [GROUPS[case["group"]]]
    L = case.get("layers", 1)
    nbytes = flops = 0.0
    for k, widths in groups:
        n = sum(widths)
        nbytes += k * n * case["K"] / 8 + 2 * k * len(widths) + 2 * n + M * (k + n) * esz
        flops += 2.0 * M * k * n
    return {"bytes": L * nbytes, "flops": L * flops}


def tolerance(case):
    """Errors against 64 bits measure 1.7e-3 to 1.9e-3 with bf16 results (a bf16 rounding alone is 1.7e-3) and 0.4e-3 to
    0.8e-3 with fp16 and fp32 ones (fp16 intermediates); about four times that between two correct paths."""
    if case.get("int8"):
        return {"rel": 2e-2, "max": 0.3}            # int8 products: 1.1 % against 64 bits
    return {"rel": 7e-3, "max": 0.05} if case["dtype"] == "bf16" else {"rel": 3e-3, "max": 0.03}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------

_HAD = {}


def _had(v):
    """Orthonormal 128-point Walsh-Hadamard of each 128-block of the last axis, fp64."""
    h = _HAD.get("h")
    if h is None:
        h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
        for _ in range(7):
            h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
        h = _HAD["h"] = h / math.sqrt(128)
    s = v.shape
    return (v.reshape(-1, 128) @ h).reshape(s)


def _codebook(cb):
    """fp64 [65536]: the codebook's fp16 value of every 16-bit state."""
    if cb not in _HAD:
        s = torch.arange(65536, dtype=torch.int64, device=DEV)
        if cb == 2:
            x = (s * 0x83DCD12D) & 0xFFFFFFFF
            h = 1024 + (x & 255) + ((x >> 8) & 255) + ((x >> 16) & 255) + (x >> 24)
            w = h.double() * 0.00676727294921875 - 10.3828125
        else:
            x = (s * 89226354 + 64248484 if cb == 0 else s * 0xCBAC1FED) & 0xFFFFFFFF
            m = (x & 0x8FFF8FFF) ^ 0x3B603B60

            def half(bits):
                return (bits - ((bits >> 15) << 16)).to(torch.int16).view(torch.float16).double()
            w = half(m & 0xFFFF) + half(m >> 16)
        _HAD[cb] = w.to(torch.float16).double()
    return _HAD[cb]


def _decode(words, K, cb, planar):
    """fp64 weights [16 rows, 16 cols] of trellis words int32 [rows, cols, 8K] (stream order, or the plane order of a
    blob's odd bitrates: groups of 4 tiles stored [plane][tile][period])."""
    r, c, _ = words.shape
    w = words.to(torch.int64) & 0xFFFFFFFF
    if planar and K % 2:
        w = w.reshape(r, c // 4, K, 4, 8).permute(0, 1, 3, 4, 2).reshape(r, c, 8 * K)
    t = torch.arange(256, device=DEV)
    e = (t + 1) * K                                  # the 16-bit window ends at stream bit e
    i1 = (e - 1) // 32
    i0 = (i1 - 1) % (8 * K)
    both = (w[..., i0] & 0xFFFF) << 32 | w[..., i1]  # (only the low 16 bits of the previous word can be reached)
    states = (both >> ((i1 + 1) * 32 - e)) & 0xFFFF
    row = 8 * ((t >> 1) & 1) + 2 * ((t >> 3) & 3) + (t & 1)
    col = (t >> 5) + 8 * ((t >> 2) & 1)
    out = torch.empty(r, c, 256, dtype=torch.float64, device=DEV)
    out[..., row * 16 + col] = _codebook(cb)[states]
    return out.view(r, c, 16, 16).permute(0, 2, 1, 3).reshape(r * 16, c * 16)


def _exact_layer(case, blobs, x, ids, w, expert):
    H, I, K = case["H"], case["I"], case["K"]        # noqa: E741
    lay = BlobLayout(H, I, K)
    off = {n: (o, b) for n, o, b in lay.fields}
    out = torch.zeros(case["M"], H, dtype=torch.float64, device=DEV)
    xd = x.double()
    flat = ids.reshape(-1).long()
    order = torch.argsort(flat, stable=True)
    counts = torch.bincount(flat, minlength=case["E"]).tolist()
    pos = 0
    for e, n in enumerate(counts):
        if not n:
            continue
        pairs = order[pos:pos + n]
        pos += n
        rows = pairs // case["topk"]
        b = blobs[expert[e]]
        vec = {k: b[o:o + nb].view(torch.float16).double() for k, (o, nb) in off.items() if k[0] == "s"}
        wgu = _decode(b[:off["gate_up"][1]].view(torch.int32).view(H // 16, 2 * I // 16, 8 * K), K, 2, True)
        o, nb = off["down"]
        wd = _decode(b[o:o + nb].view(torch.int32).view(I // 16, H // 16, 8 * K), K, 2, True)
        xe = xd[rows]
        g = _had(_had(xe * vec["suh_g"]) @ wgu[:, :I]) * vec["svh_g"]
        u = _had(_had(xe * vec["suh_u"]) @ wgu[:, I:]) * vec["svh_u"]
        a = _had(g * torch.sigmoid(g) * u * vec["suh_d"])
        y = _had(a @ wd) * vec["svh_d"]
        out.index_add_(0, rows, y * w.reshape(-1)[pairs].double()[:, None])
    return out


def exact(case, seed):
    if case["kind"] in ("moe", "token", "cached"):
        blobs = _blobs(case, seed, _pool(case))
        outs = []
        for li in range(case["layers"]):
            ids, w = _routing(case, seed, li)
            outs.append(_exact_layer(case, blobs, _acts(case, seed, case["H"], li), ids, w,
                                     _expert_of(case, seed, li).tolist()))
        return outs[0] if case["kind"] == "moe" else outs
    groups = range(len(GROUPS)) if case["kind"] == "ltoken" else [case["group"]]
    outs = []
    for li in range(case.get("layers", 1)):
        for gi in groups:
            x = _acts(case, seed, GROUPS[gi][0], li * 8 + gi).double()
            parts = []
            for tr, su, sv in _shards(case, seed, gi, li):
                wt = _decode(tr.view(torch.int32), case["K"], case["cb"], False)
                parts.append(_had(_had(x * su.double()) @ wt) * sv.double())
            outs.append(torch.cat(parts, 1))
    return outs if case["kind"] == "ltoken" else outs[0]
