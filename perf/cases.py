"""Performance cases of the tiered KV cache: the calls a serving program makes, at the sizes it makes them.

A case is a dict of plain values.  `prepare` builds what a program holds before the call (quantized caches and pools
filled from seeded K/V, queries, plans, captured step graphs), `run` makes one pass through the public entry points
and returns its outputs, `exact` restates the result in 64 bits with plain torch, `work` counts the bytes and
operations that the path cannot do without.  The kinds:

  decode  dense decode of one token per sequence over the position-ring cache, all layers (kvt_decode_attn)
  topk    top-k sparse decode of one token per request over a slot-indexed pool, all layers (qwen_sparse_decode_attn)
  slots   dense decode over the slot-indexed tiered pool, one layer (decode_attn_slots)
  paged   prefix-chunk attention over the indexer's selection, one layer (sparse_gqa_fwd_interface_paged)
  prefill causal prefill of a chunk, one layer (kvt_prefill_attn)
  append  two consecutive ring-long quantize-appends, the oldest rows requantized into INT4 pages (PosTieredCache)
  store   the decode step's dual write of one token per request, all layers (quant_store_kv_tiered)
  gather  dequantizing gathers into a bf16 scratch, one layer (whole prefix, or the top-k selection)

A decode step of a serving program (decode, topk, store) is captured once as a HIP graph and replayed for every token,
as the integration notes describe, so `prepare` captures it and `run` replays it; the other calls are made eagerly.
K is N(0, 1) with 8 of the 256 channels of a head 8 times larger (the outlier channels of real keys), V is N(0, 1);
queries are N(0, 1), so that scores spread over several units and the softmax is neither flat nor one-hot.
"""
import math

import torch

import kvtier  # noqa: F401  (loads the package directory)
from kvtier import kvt, sparse_attn

D = 256
PAGE = 64
G8, G4 = 64, 32
RING = 8192
FP16_MAX = 65504.0


# ------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # the headline: one long conversation (262,144 tokens) decoding, all 12 attention layers, 16 / 2 heads
        dict(name="decode_262k", kind="decode", hq=16, h=2, layers=12, lens="262144", shared=0),
        # a mixed batch: 8 conversations of log-uniform lengths, the first two share a 4,096-token prefix
        dict(name="decode_ragged8", kind="decode", hq=16, h=2, layers=12,
             lens="63627,5121,1055,30011,12288,2500,9001,43210", shared=4096),
        # a short conversation just past the ring: latency and launches count
        dict(name="decode_10k", kind="decode", hq=16, h=2, layers=12, lens="10001", shared=0),
        # the served model's head count (24 / 2) on a small batch of medium contexts
        dict(name="decode_24q", kind="decode", hq=24, h=2, layers=12, lens="32768,20011,30000,9973", shared=0),
        # the served decode step: the indexer's 2,051 positions of each of 8 requests, 12 layers, tiered pool
        dict(name="topk_8x2051", kind="topk", hq=24, h=2, layers=12, batch=8, ctx=65536, topk=2051, pool="tiered"),
        # the same backend with every position attended (dense layers of the slot-indexed pool)
        dict(name="slots_4x65k", kind="slots", hq=16, h=2, batch=4, ctx=65536),
        # prefix-chunk attention straight from the pool: 60,000-token prefix + 1,024-query chunk, 12 / 1 heads per rank
        dict(name="paged_60k", kind="paged", hq=12, h=1, prefix=60000, chunk=1024, topk=2051, pool="tiered",
             smooth=False),
        # the first chunk of a prompt, over its own bf16 K/V, served model's heads
        dict(name="prefill_first", kind="prefill", hq=24, h=2, start=0, n=4096),
        # the last chunk of the 10,001-token prompt: ragged length, keys in both tiers
        dict(name="prefill_10k", kind="prefill", hq=16, h=2, start=8192, n=1809),
        # steady-state prompt ingestion: ring-long appends, every token evicts one
        dict(name="append_8k", kind="append", h=2, layers=6, ring=8192, dtype="bf16"),
        # the smallest call: the decode step's K/V of 8 requests written to both tiers, 12 layers
        dict(name="store_8", kind="store", h=2, layers=12, n=8, dtype="bf16"),
        # a prompt's prefix dequantized for a dense chunk (4 requests, ragged)
        dict(name="gather_prefix", kind="gather", h=2, which="prefix", lens="40000,9001,20480,2051", topk=0,
             pool="tiered"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "topk", "slots", "paged", "prefill", "prefill", "append", "store",
                       "gather"])
    if kind == "decode":
        n = rng.choice([1, 1, 2, 3, 5, 8])
        lens = [_log_int(rng, 300, 200_000 // n) for _ in range(n)]
        return dict(kind=kind, hq=rng.choice([16, 16, 24, 8]), h=2, layers=rng.choice([4, 12]),
                    lens=",".join(map(str, lens)), shared=0)
    if kind == "topk":
        batch = _log_int(rng, 1, 16)
        return dict(kind=kind, hq=rng.choice([16, 24]), h=2, layers=rng.choice([4, 12]), batch=batch,
                    ctx=_log_int(rng, 2500, 500_000 // batch), topk=rng.choice([512, 1024, 2048, 2051]), pool=rng.choice(["tiered", "int4", "int8"]))
    if kind == "slots":
        batch = rng.randint(1, 6)
        return dict(kind=kind, hq=rng.choice([16, 24]), h=2, batch=batch, ctx=_log_int(rng, 1000, 250_000 // batch))
    if kind == "paged":
        return dict(kind=kind, hq=rng.choice([8, 12]), h=1, prefix=_log_int(rng, 1000, 60000),
                    chunk=_log_int(rng, 64, 1024), topk=rng.choice([512, 1024, 2051]),
                    pool=rng.choice(["tiered", "int4", "int8"]), smooth=rng.random() < 0.25)
    if kind == "prefill":
        hq = rng.choice([16, 24])
        if rng.random() < 0.4:
            return dict(kind=kind, hq=hq, h=2, start=0, n=_log_int(rng, 100, 4096))
        start = _log_int(rng, 1000, 24000)
        return dict(kind=kind, hq=hq, h=2, start=start, n=min(_log_int(rng, 100, 2048), int(2.6e8 / (hq * (start + 1024)))))
    if kind == "append":
        return dict(kind=kind, h=2, layers=6, ring=rng.choice([512, 1024, 2048, 4096, 8192]),
                    dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]))
    if kind == "store":
        return dict(kind=kind, h=2, layers=12, n=_log_int(rng, 1, 2048), dtype=rng.choice(["bf16", "bf16", "fp16"]))
    which = rng.choice(["prefix", "topk"])
    if which == "prefix":
        lens = [_log_int(rng, 500, 40000) for _ in range(rng.randint(1, 4))]
        return dict(kind=kind, h=2, which=which, lens=",".join(map(str, lens)), topk=0,
                    pool=rng.choice(["tiered", "int4", "int8"]))
    lens = [_log_int(rng, 2500, 40000) for _ in range(rng.randint(1, 8))]
    return dict(kind=kind, h=2, which=which, lens=",".join(map(str, lens)), topk=rng.choice([512, 2048, 2051]),
                pool=rng.choice(["tiered", "int4", "int8"]))


# --------------------------------------------------------------------------------------------------- inputs and tools
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def _gen(seed, *parts):
    x = int(seed)
    for p in parts:
        x = (x * 1_000_003 + int(p) + 17) % (1 << 40)
    return torch.Generator(device="cuda").manual_seed(x)


def _kv(seed, tag, n, h, dtype=torch.bfloat16):
    """K and V of n tokens [n, h, D]."""
    g = _gen(seed, 1, tag)
    mul = torch.ones(h, D, device="cuda")
    for i in range(h):
        mul[i, torch.randperm(D, generator=g, device="cuda")[:8]] = 8.0
    k = torch.randn(n, h, D, generator=g, device="cuda", dtype=dtype).mul_(mul.to(dtype))
    return k, torch.randn(n, h, D, generator=g, device="cuda", dtype=dtype)


def _q(seed, tag, *shape):
    return torch.randn(*shape, D, generator=_gen(seed, 2, tag), device="cuda", dtype=torch.bfloat16)


def _randperm(seed, tag, n):
    return torch.randperm(n, generator=_gen(seed, 3, tag), device="cuda")


def _captured(step):
    """A HIP graph of step(), captured after an eager run on a side stream."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return graph


def _quant(x, group, qmax):
    """Codes (float32) and fp16 scales of x [..., D]: the storage format's symmetric group quantization."""
    g = x.float().reshape(*x.shape[:-1], D // group, group)
    a = g.abs().amax(-1)
    q = torch.full_like(a, qmax)   # (a tensor: a division by a Python number is a product with its reciprocal)
    s = torch.where(a > 0, a / q, torch.ones_like(a)).clamp(max=FP16_MAX).half()
    return (g / s.float()[..., None]).round().clamp(-qmax, qmax), s


def _value(codes_scales):
    """code * scale [..., D] in fp32 (exact: at most 8 + 11 significant bits)."""
    c, s = codes_scales
    return (c * s.float()[..., None]).flatten(-2)


def _int8_rows(x):
    return _value(_quant(x, G8, 127.0))


def _int4_rows(x):
    return _value(_quant(x, G4, 7.0))


def _pow2_ring(n):
    return min(RING, 1 << (max(1, n) - 1).bit_length())


def _attend(q, k, v, scale, mask=None):
    """softmax(q k^T scale) v in float64 for one KV head: q [..., g, D], k and v [..., n, D]."""
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * scale
    if mask is not None:
        s = s.masked_fill(~mask, float("-inf"))
    return s.softmax(-1) @ v.double()


# -------------------------------------------------------------------------------- position-ring cache (decode, prefill)
def _pos_cache(case, seed, lens, layers):
    """The cache of sequences of the given lengths after their prompts were appended through the write path; the first
    two sequences share case["shared"] prefix tokens kept in common INT4 pages."""
    h, shared = case["h"], case.get("shared", 0)
    rings = [_pow2_ring(n) for n in lens]
    pages = sum(max(0, n - r) // PAGE + 2 for n, r in zip(lens, rings)) + shared // PAGE
    cache = kvt.PosTieredCache(layers, h, D, n_pages=pages, ring_total=sum(rings), max_seqs=len(lens),
                               max_pages=max(lens) // PAGE + 2, device="cuda", page_seed=seed)
    kv = [[_kv(seed, 100 * layer + s, n, h) for s, n in enumerate(lens)] for layer in range(layers)]
    common = []
    if shared:
        common = [cache.alloc.pop() for _ in range(shared // PAGE)]
        rows = (torch.tensor(common, device="cuda")[:, None] * PAGE + torch.arange(PAGE, device="cuda")).reshape(-1)
        ones = torch.ones(h, D, dtype=torch.float16, device="cuda")
        for layer in range(layers):
            sparse_attn.quant_store_kv_int4(*_kv(seed, 100 * layer + 99, shared, h), rows, cache.k4[layer],
                                            cache.v4[layer], cache.ks4[layer], cache.vs4[layer], ones, ones)
    done = []
    for s, r in enumerate(rings):
        own = shared if s < 2 else 0
        cache.add_seq(r, ring_start=own, shared_pages=common if own else ())
        done.append(own)
    while any(d < n for d, n in zip(done, lens)):
        act = [s for s, n in enumerate(lens) if done[s] < n]
        cnt = [min(rings[s], lens[s] - done[s]) for s in act]
        plan = cache.plan_append(act, cnt)
        for layer in range(layers):
            part = [[t[done[s]:done[s] + c] for t in kv[layer][s]] for s, c in zip(act, cnt)]
            cache.append(layer, plan, torch.cat([p[0] for p in part]), torch.cat([p[1] for p in part]))
        cache.commit(plan)
        for s, c in zip(act, cnt):
            done[s] += c
    return cache


def _pos_rows(case, seed, layer, s, n):
    """What the cache holds for sequence s (length n) of a layer: code * scale of every position, fp32 [n, h, D]."""
    shared = case.get("shared", 0) if s < 2 else 0
    hot = max(shared, n - _pow2_ring(n))
    out = []
    pre = _kv(seed, 100 * layer + 99, shared, case["h"]) if shared else (None, None)
    for t, p in zip(_kv(seed, 100 * layer + s, n, case["h"]), pre):
        rows = torch.empty(t.shape, dtype=torch.float32, device="cuda")
        for a in range(0, n, 32768):
            e8 = _int8_rows(t[a:a + 32768])
            rows[a:a + 32768] = e8
            cold = min(hot, a + 32768) - a
            if cold > 0:
                rows[a:a + cold] = _int4_rows(e8[:cold])
        if shared:
            rows[:shared] = _int4_rows(p)
        out.append(rows)
    return out


def _prepare_decode(case, seed):
    lens = [int(x) for x in case["lens"].split(",")]
    layers, hq = case["layers"], case["hq"]
    cache = _pos_cache(case, seed, lens, layers)
    q = _q(seed, 0, layers, len(lens), hq)
    out = torch.empty(layers, len(lens), hq, D, dtype=torch.float32, device="cuda")
    ws = {}
    planned = hq // case["h"] <= 8   # decode plans serve up to 8 q heads per KV head

    def step():
        plan = kvt.kvt_decode_plan(cache, hq, workspace=ws) if planned else None
        for layer in range(layers):
            kvt.kvt_decode_attn(cache, layer, q[layer], out=out[layer], impl="mfma", workspace=ws, plan=plan,
                                check_q=False)

    return dict(graph=_captured(step), out=out, keep=(cache, q, ws))


def _exact_decode(case, seed):
    lens = [int(x) for x in case["lens"].split(",")]
    q = _q(seed, 0, case["layers"], len(lens), case["hq"])
    gs = case["hq"] // case["h"]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for layer in range(case["layers"]):
        for s, n in enumerate(lens):
            k, v = _pos_rows(case, seed, layer, s, n)
            for i in range(case["h"]):
                out[layer, s, i * gs:(i + 1) * gs] = _attend(q[layer, s, i * gs:(i + 1) * gs], k[:, i], v[:, i], D ** -0.5)
    return out


def _prepare_prefill(case, seed):
    start, n, hq = case["start"], case["n"], case["hq"]
    st = dict(q=_q(seed, 0, n, hq), cu=torch.tensor([0, n], dtype=torch.int32, device="cuda"), n=n)
    st["out"] = torch.empty_like(st["q"])
    st["cache"] = _pos_cache(case, seed, [start + n], 1)
    st["src"] = dict(zip(("k_src", "v_src"), _kv(seed, 0, n, case["h"]))) if start == 0 else {}
    return st


def _run_prefill(st):
    return kvt.kvt_prefill_attn(st["cache"], 0, st["q"], st["cu"], max_q=st["n"], out=st["out"],
                                kv_lens=st["cache"].seq_lens[:1], **st["src"])


def _exact_prefill(case, seed):
    start, n, gs = case["start"], case["n"], case["hq"] // case["h"]
    q = _q(seed, 0, n, case["hq"])
    if start == 0:
        k, v = _kv(seed, 0, n, case["h"])
    else:   # the rows as every reader sees them: bf16 of code * scale
        k, v = [t.bfloat16() for t in _pos_rows(case, seed, 0, 0, start + n)]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    pos = torch.arange(start + n, device="cuda")
    for j in range(case["hq"]):
        kk, vv = k[:, j // gs].double(), v[:, j // gs].double()
        for a in range(0, n, 2048):
            b = min(n, a + 2048)
            mask = pos[None, :] <= (start + torch.arange(a, b, device="cuda"))[:, None]
            out[a:b, j] = _attend(q[a:b, j], kk, vv, D ** -0.5, mask)
    return out


def _prepare_append(case, seed):
    """The cache holds ring-long chunk B; a pass appends chunk A (evicting B into pages) and B again (evicting A), so
    that every pass starts from the same ring."""
    r, h, layers, dt = case["ring"], case["h"], case["layers"], _DTYPES[case["dtype"]]
    cache = kvt.PosTieredCache(layers, h, D, n_pages=2 * r // PAGE, ring_total=r, max_seqs=1, max_pages=2 * r // PAGE + 1,
                               device="cuda", page_seed=seed)
    cache.add_seq(r)
    a = [_kv(seed, 2 * layer, r, h, dt) for layer in range(layers)]
    b = [_kv(seed, 2 * layer + 1, r, h, dt) for layer in range(layers)]
    plan = cache.plan_append([0], [r])
    for layer in range(layers):
        cache.append(layer, plan, *b[layer])
    cache.commit(plan)
    plans = []
    for _ in range(2):
        plans.append(cache.plan_append([0], [r]))
        cache.commit(plans[-1])
    return dict(cache=cache, plans=plans, kv=(a, b), layers=layers)


def _run_append(st):
    cache = st["cache"]
    for plan, kv in zip(st["plans"], st["kv"]):
        for layer in range(st["layers"]):
            cache.append(layer, plan, *kv[layer])
    return [cache.k4, cache.v4, cache.ks4, cache.vs4, cache.rk, cache.rv, cache.rks, cache.rvs]


def _exact_append(case, seed):
    """The scales (a group's largest value / qmax); codes are whole numbers."""
    r, h, layers = case["ring"], case["h"], case["layers"]
    order = torch.randperm(2 * r // PAGE, generator=torch.Generator().manual_seed(seed)).to("cuda")   # page order
    res = [[], [], [], []]
    for layer in range(layers):
        ab = [_kv(seed, 2 * layer + i, r, h, _DTYPES[case["dtype"]]) for i in (0, 1)]
        for t in (0, 1):
            a8, b8 = _int8_rows(ab[0][t]), _int8_rows(ab[1][t])
            amax4 = torch.cat([b8, a8]).double().reshape(2 * r // PAGE, PAGE, h, D // G4, G4).abs().amax(-1)
            s4 = torch.empty_like(amax4)
            s4[order] = amax4 / 7.0
            res[t].append(s4.reshape(2 * r, h, D // G4))
            res[2 + t].append(ab[1][t].double().reshape(r, h, D // G8, G8).abs().amax(-1) / 127.0)
    none = [None] * layers
    return [none, none, res[0], res[1], none, none, res[2], res[3]]


# ---------------------------------------------------------------------------------------------- slot-indexed pools
class _Slots:
    """Placement of the requests of a slot-indexed pool: page-granular slots in a random order, each request's
    positions written oldest first and the requests in turn, so that the ring holds the newest tokens; a ring row
    belongs to the token written to it last."""

    def __init__(self, case, seed, lens):
        self.lens = lens
        pages = [-(-n // PAGE) for n in lens]
        perm = _randperm(seed, 0, sum(pages))
        self.rows = sum(pages) * PAGE
        self.r2t = torch.zeros(len(lens), max(lens), dtype=torch.int32, device="cuda")
        at = 0
        for b, n in enumerate(lens):
            slots = (perm[at:at + pages[b], None] * PAGE + torch.arange(PAGE, device="cuda")).reshape(-1)
            self.r2t[b, :n] = slots[:n].to(torch.int32)
            at += pages[b]
        self.slot = torch.cat([self.r2t[b, :n] for b, n in enumerate(lens)]).long()     # of every token
        age = torch.cat([torch.arange(n, 0, -1, device="cuda") for n in lens])             # distance to its end
        order = age.argsort(descending=True, stable=True)                                   # write order
        self.owner = torch.full((RING,), -1, dtype=torch.int64, device="cuda")
        key = torch.full((RING,), -1, dtype=torch.int64, device="cuda")
        rank = torch.empty_like(order)
        rank[order] = torch.arange(order.numel(), device="cuda")
        key.scatter_reduce_(0, self.slot % RING, rank, "amax")
        held = key >= 0
        self.owner[held] = self.slot[order[key[held]]]
        self.hot = self.owner[self.slot % RING] == self.slot                                # of every token
        self.owner = self.owner.to(torch.int32)
        self.cu = torch.tensor([0] + lens, device="cuda").cumsum(0)


def _smooth(case, seed, h):
    if not case.get("smooth", False):
        return [torch.ones(h, D, dtype=torch.float16, device="cuda")] * 2
    g = _gen(seed, 4)
    return [(0.5 + torch.rand(h, D, generator=g, device="cuda")).half() for _ in range(2)]


def _pool(case, seed, place, layer):
    """One layer's pool filled with the requests' tokens: (k, v, k_scale, v_scale, ring arguments or None)."""
    h, kind = case["h"], case["pool"]
    k, v = _kv(seed, layer, place.slot.numel(), h)
    one = torch.ones(h, D, dtype=torch.float16, device="cuda")

    def buffers(rows, group, dtype, width):
        return ([torch.zeros(rows, h, width, dtype=dtype, device="cuda") for _ in range(2)]
                + [torch.zeros(rows, h, D // group, dtype=torch.float16, device="cuda") for _ in range(2)])

    if kind == "int8":
        p = buffers(place.rows, G8, torch.int8, D)
        sparse_attn.quant_store_kv_int8(k, v, place.slot, *p, one, one)
        return p, {}
    p = buffers(place.rows, G4, torch.uint8, D // 2)
    sparse_attn.quant_store_kv_int4(k, v, place.slot, *p, one, one)
    if kind == "int4":
        return p, {}
    ring = buffers(RING, G8, torch.int8, D)
    at = place.hot.nonzero()[:, 0]
    sparse_attn.quant_store_kv_int8(k[at], v[at], place.slot[at] % RING, *ring, one, one)
    return p, dict(ring_k=ring[0], ring_v=ring[1], ring_ks=ring[2], ring_vs=ring[3], owner=place.owner, ring_mask=RING - 1)


def _pool_rows(case, seed, place, layer, at=None):
    """bf16(code * scale * smoothing) of the tokens `at` (all by default), as every reader of the pool sees them."""
    out = []
    for t, sm in zip(_kv(seed, layer, place.slot.numel(), case["h"]), _smooth(case, seed, case["h"])):
        hot = place.hot
        if at is not None:
            t, hot = t[at], hot[at]
        hot = torch.ones_like(hot) if case["pool"] == "int8" else hot & (case["pool"] == "tiered")
        rows = torch.empty(t.shape, dtype=torch.bfloat16, device="cuda")
        for a in range(0, t.shape[0], 65536):
            c = t[a:a + 65536]
            x = torch.where(hot[a:a + 65536, None, None], _int8_rows(c), _int4_rows(c))
            rows[a:a + 65536] = (x * sm.float()).bfloat16()
        out.append(rows)
    return out


def _selection(seed, tag, n, topk):
    """An indexer's choice among n positions, ascending: the newest 128 and random older ones."""
    if n <= topk:
        return torch.arange(n, device="cuda")
    new = min(128, topk)
    old = _randperm(seed, 1000 + tag, n - new)[:topk - new]
    return torch.cat([old, torch.arange(n - new, n, device="cuda")]).sort().values


def _selections(case, seed, lens):
    idx = torch.full((len(lens), case["topk"]), -1, dtype=torch.int32, device="cuda")
    for b, n in enumerate(lens):
        s = _selection(seed, b, n, case["topk"])
        idx[b, :s.numel()] = s.to(torch.int32)
    return idx


def _prepare_topk(case, seed):
    lens = [case["ctx"]] * case["batch"]
    b, hq, layers, topk = case["batch"], case["hq"], case["layers"], case["topk"]
    place = _Slots(case, seed, lens)
    pools = [_pool(case, seed, place, layer) for layer in range(layers)]
    sk, sv = _smooth(case, seed, case["h"])
    bits = 8 if case["pool"] == "int8" else 4
    idx = _selections(case, seed, lens)
    seq = torch.tensor(lens, dtype=torch.int32, device="cuda")
    req = torch.arange(b, device="cuda")
    counts = torch.empty(b, dtype=torch.int32, device="cuda")
    cu = torch.empty(b + 1, dtype=torch.int32, device="cuda")
    q = _q(seed, 0, layers, b, hq)
    out = torch.empty(layers, b, hq, D, dtype=torch.float32, device="cuda")
    ws = {}

    def step():
        sparse_attn.qwen_sparse_fa2_cu_seqlens_triton(seq, idx, counts, cu, b, topk)
        for layer in range(layers):
            (k, v, ks, vs), ring = pools[layer]
            sparse_attn.qwen_sparse_decode_attn(q[layer], k, v, place.r2t, req, idx, seq, cu, b, topk, ks, vs, sk, sv,
                                                bits, out=out[layer], workspace=ws, **ring)

    return dict(graph=_captured(step), out=out, keep=(place, pools, sk, sv, idx, seq, req, counts, cu, q, ws))


def _exact_topk(case, seed):
    lens = [case["ctx"]] * case["batch"]
    place = _Slots(case, seed, lens)
    idx = _selections(case, seed, lens)
    q = _q(seed, 0, case["layers"], case["batch"], case["hq"])
    gs = case["hq"] // case["h"]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for layer in range(case["layers"]):
        sel = [idx[b][idx[b] >= 0].long() for b in range(case["batch"])]
        k, v = _pool_rows(case, seed, place, layer, torch.cat([s + place.cu[b] for b, s in enumerate(sel)]))
        at = 0
        for b, s in enumerate(sel):
            for i in range(case["h"]):
                out[layer, b, i * gs:(i + 1) * gs] = _attend(q[layer, b, i * gs:(i + 1) * gs], k[at:at + s.numel(), i],
                                                             v[at:at + s.numel(), i], D ** -0.5)
            at += s.numel()
    return out


def _prepare_slots(case, seed):
    case = dict(case, pool="tiered")
    lens = [case["ctx"] - 37 * b for b in range(case["batch"])]   # requests differ a little in length
    place = _Slots(case, seed, lens)
    (k, v, ks, vs), ring = _pool(case, seed, place, 0)
    return dict(args=(_q(seed, 0, case["batch"], case["hq"]), torch.tensor(lens, dtype=torch.int32, device="cuda"),
                      place.r2t, torch.arange(case["batch"], device="cuda"), k, v, ks, vs, ring["ring_k"], ring["ring_v"],
                      ring["ring_ks"], ring["ring_vs"], ring["owner"], ring["ring_mask"]),
                sm=_smooth(case, seed, case["h"]), max_len=max(lens), ws={})


def _run_slots(st):
    return kvt.decode_attn_slots(*st["args"], sm_k=st["sm"][0], sm_v=st["sm"][1], max_len=st["max_len"],
                                 workspace=st["ws"])


def _exact_slots(case, seed):
    case = dict(case, pool="tiered")
    lens = [case["ctx"] - 37 * b for b in range(case["batch"])]
    place = _Slots(case, seed, lens)
    q = _q(seed, 0, case["batch"], case["hq"])
    gs = case["hq"] // case["h"]
    k, v = _pool_rows(case, seed, place, 0)
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b, n in enumerate(lens):
        at = int(place.cu[b])
        for i in range(case["h"]):
            out[b, i * gs:(i + 1) * gs] = _attend(q[b, i * gs:(i + 1) * gs], k[at:at + n, i], v[at:at + n, i], D ** -0.5)
    return out


def _chunk_rows(case, seed):
    """Indexer rows of a chunk: query j sees prefix + j + 1 positions and selects up to topk of them (sorted, -1
    behind); one row in eight selects fewer."""
    prefix, chunk, topk = case["prefix"], case["chunk"], case["topk"]
    g = _gen(seed, 5)
    visible = prefix + 1 + torch.arange(chunk, device="cuda")
    want = torch.full((chunk,), topk, device="cuda")
    short = torch.rand(chunk, generator=g, device="cuda") < 0.125
    few = 1 + (torch.rand(chunk, generator=g, device="cuda") * (topk - 1)).long()
    want = torch.minimum(torch.where(short, few, want), visible)
    idx = torch.full((chunk, topk), -1, dtype=torch.int32, device="cuda")
    for a in range(0, chunk, 128):
        vis, n = visible[a:a + 128], want[a:a + 128]
        score = torch.rand(vis.numel(), prefix + chunk, generator=g, device="cuda")
        score.masked_fill_(torch.arange(prefix + chunk, device="cuda")[None] >= vis[:, None], -1.0)
        best = score.topk(min(topk, prefix + chunk), dim=-1).indices
        best = torch.where(torch.arange(best.shape[1], device="cuda")[None] < n[:, None], best, prefix + chunk)
        best = best.sort(-1).values
        best = torch.where(best < prefix + chunk, best, -1)
        idx[a:a + 128, :best.shape[1]] = best.to(torch.int32)
    return idx


def _prepare_paged(case, seed):
    n = case["prefix"] + case["chunk"]
    place = _Slots(case, seed, [n])
    (k, v, ks, vs), ring = _pool(case, seed, place, 0)
    sk, sv = _smooth(case, seed, case["h"])
    q = _q(seed, 0, case["chunk"], case["hq"])
    return dict(args=(q, _chunk_rows(case, seed), torch.tensor([0, case["chunk"]], dtype=torch.int32, device="cuda"),
                      torch.tensor([n], dtype=torch.int32, device="cuda"), place.r2t, torch.zeros(1, dtype=torch.int64,
                                                                                                 device="cuda"),
                      k, v, ks, vs, sk, sv, D ** -0.5, case["chunk"], 8 if case["pool"] == "int8" else 4), ring=ring)


def _run_paged(st):
    return sparse_attn.sparse_gqa_fwd_interface_paged(*st["args"], **st["ring"])


def _exact_paged(case, seed):
    n = case["prefix"] + case["chunk"]
    place = _Slots(case, seed, [n])
    k, v = [t.double() for t in _pool_rows(case, seed, place, 0)]
    q = _q(seed, 0, case["chunk"], case["hq"])
    idx = _chunk_rows(case, seed).long()
    gs = case["hq"] // case["h"]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for a in range(0, case["chunk"], 128):
        sel = idx[a:a + 128]
        for i in range(case["h"]):
            out[a:a + 128, i * gs:(i + 1) * gs] = _attend(q[a:a + 128, i * gs:(i + 1) * gs], k[sel.clamp(min=0), i],
                                                          v[sel.clamp(min=0), i], D ** -0.5, (sel >= 0)[:, None, :])
    return out


def _prepare_store(case, seed):
    h, layers, n = case["h"], case["layers"], case["n"]
    rows = 65536
    z = dict(device="cuda")
    big = [torch.zeros(layers, rows, h, D // 2, dtype=torch.uint8, **z) for _ in range(2)]
    big += [torch.zeros(layers, rows, h, D // G4, dtype=torch.float16, **z) for _ in range(2)]
    big += [torch.zeros(layers, RING, h, D, dtype=torch.int8, **z) for _ in range(2)]
    big += [torch.zeros(layers, RING, h, D // G8, dtype=torch.float16, **z) for _ in range(2)]
    owner = torch.full((RING,), -1, dtype=torch.int32, **z)
    # one token per request: slots anywhere in the pool, each in a ring row of its own
    loc = _randperm(seed, 0, RING)[:n] + RING * torch.randint(0, rows // RING, (n,), generator=_gen(seed, 6), **z)
    one = torch.ones(h, D, dtype=torch.float16, **z)
    kv = [_kv(seed, layer, n, h, _DTYPES[case["dtype"]]) for layer in range(layers)]

    def step():
        for layer in range(layers):
            sparse_attn.quant_store_kv_tiered(*kv[layer], loc, *[t[layer] for t in big], owner, one, one, RING - 1)

    return dict(graph=_captured(step), out=big + [owner], keep=(kv, loc, one))


def _exact_store(case, seed):
    h, layers, n, rows = case["h"], case["layers"], case["n"], 65536
    loc = _randperm(seed, 0, RING)[:n] + RING * torch.randint(0, rows // RING, (n,), generator=_gen(seed, 6),
                                                              device="cuda")
    z = dict(dtype=torch.float64, device="cuda")
    s4 = [torch.zeros(layers, rows, h, D // G4, **z) for _ in range(2)]
    s8 = [torch.zeros(layers, RING, h, D // G8, **z) for _ in range(2)]
    for layer in range(layers):
        for t, x in enumerate(_kv(seed, layer, n, h, _DTYPES[case["dtype"]])):
            s4[t][layer, loc] = x.double().reshape(n, h, D // G4, G4).abs().amax(-1) / 7.0
            s8[t][layer, loc % RING] = x.double().reshape(n, h, D // G8, G8).abs().amax(-1) / 127.0
    return [None, None, *s4, None, None, *s8, None]


def _prepare_gather(case, seed):
    lens = [int(x) for x in case["lens"].split(",")]
    place = _Slots(case, seed, lens)
    (k, v, ks, vs), ring = _pool(case, seed, place, 0)
    sk, sv = _smooth(case, seed, case["h"])
    b = len(lens)
    seq = torch.tensor(lens, dtype=torch.int32, device="cuda")
    req = torch.arange(b, device="cuda")
    st = dict(pool=(k, v, ks, vs), sm=(sk, sv), ring=ring, place=place, seq=seq, req=req, b=b, which=case["which"],
              kind=case["pool"], max_len=max(lens))
    if case["which"] == "prefix":
        st["cu"] = place.cu.to(torch.int32)
        total = sum(lens)
    else:
        idx = _selections(case, seed, lens)
        counts, cu = torch.empty(b, dtype=torch.int32, device="cuda"), torch.empty(b + 1, dtype=torch.int32, device="cuda")
        sparse_attn.qwen_sparse_fa2_cu_seqlens_triton(seq, idx, counts, cu, b, case["topk"])
        st.update(idx=idx, cu=cu, topk=case["topk"])
        total = sum(min(n, case["topk"]) for n in lens)
    st["out"] = [torch.empty(total, case["h"], D, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    return st


def _run_gather(st):
    (k, v, ks, vs), (sk, sv), ring = st["pool"], st["sm"], st["ring"]
    if st["which"] == "prefix":
        fn = getattr(sparse_attn, "qwen_sparse_prefix_gather_dequant_" + st["kind"])
        fn(k, v, ks, vs, sk, sv, st["place"].r2t, st["req"], st["seq"], st["cu"], *st["out"], st["b"], st["max_len"], **ring)
    else:
        sparse_attn.qwen_sparse_kv_extraction_compact_triton(
            k, v, st["place"].r2t, st["req"], st["idx"], st["seq"], st["cu"], *st["out"], st["b"], st["topk"], ks, vs, sk,
            sv, 8 if st["kind"] == "int8" else 4, **ring)
    return st["out"]


def _exact_gather(case, seed):
    lens = [int(x) for x in case["lens"].split(",")]
    place = _Slots(case, seed, lens)
    at = None
    if case["which"] == "topk":
        idx = _selections(case, seed, lens)
        at = torch.cat([idx[b][idx[b] >= 0].long() + place.cu[b] for b in range(len(lens))])
    return [t.double() for t in _pool_rows(case, seed, place, 0, at)]


# ------------------------------------------------------------------------------------------------------ the interface
_PREPARE = dict(decode=_prepare_decode, topk=_prepare_topk, slots=_prepare_slots, paged=_prepare_paged,
                prefill=_prepare_prefill, append=_prepare_append, store=_prepare_store, gather=_prepare_gather)
_RUN = dict(slots=_run_slots, paged=_run_paged, prefill=_run_prefill, append=_run_append, gather=_run_gather)
_EXACT = dict(decode=_exact_decode, topk=_exact_topk, slots=_exact_slots, paged=_exact_paged, prefill=_exact_prefill,
              append=_exact_append, store=_exact_store, gather=_exact_gather)


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, int(seed))
    st["kind_of_call"] = case["kind"]
    return st


def run(state):
    if "graph" in state:   # a captured step
        state["graph"].replay()
        return state["out"]
    return _RUN[state["kind_of_call"]](state)


def exact(case, seed):
    return _EXACT[case["kind"]](case, int(seed))


def work(case):
    kind, h, hq = case["kind"], case["h"], case.get("hq", 0)
    row8, row4 = h * 2 * (D + 2 * D // G8), h * 2 * (D // 2 + 2 * D // G4)   # K and V of one token, codes + scales
    row = {"tiered": row4, "int4": row4, "int8": row8}   # a tiered pool of any size holds most tokens in INT4
    if kind == "decode":
        lens = [int(x) for x in case["lens"].split(",")]
        shared = case.get("shared", 0)
        nbytes = 0
        for s, n in enumerate(lens):
            hot = n - max(shared if s < 2 else 0, n - _pow2_ring(n))
            nbytes += hot * row8 + (n - hot) * row4 + hq * D * (2 + 4)
        if shared:
            nbytes -= shared * row4   # the common prefix is one copy
        return dict(bytes=case["layers"] * nbytes, flops=case["layers"] * 4 * hq * D * sum(lens))
    if kind == "topk":
        n = case["batch"] * min(case["topk"], case["ctx"])
        nbytes = n * (row[case["pool"]] + 12) + case["batch"] * hq * D * (2 + 4)
        return dict(bytes=case["layers"] * nbytes, flops=case["layers"] * 4 * hq * D * n)
    if kind == "slots":
        n = sum(case["ctx"] - 37 * b for b in range(case["batch"]))
        return dict(bytes=n * (row4 + 8) + case["batch"] * hq * D * 6, flops=4 * hq * D * n)
    if kind == "paged":
        prefix, chunk, topk = case["prefix"], case["chunk"], case["topk"]
        sel = chunk * min(topk, prefix) * (1 - 0.125 / 2)   # one query in eight selects half as many on average
        return dict(bytes=(prefix + chunk) * (row[case["pool"]] + 8) + sel * 4 + chunk * hq * D * 4, flops=4 * hq * D * sel)
    if kind == "prefill":
        start, n = case["start"], case["n"]
        pairs = n * start + n * (n + 1) // 2
        hot = min(RING, start + n)
        keys = n * h * D * 4 if start == 0 else hot * row8 + (start + n - hot) * row4
        return dict(bytes=keys + n * hq * D * 4, flops=4 * hq * D * pairs)
    width = {"bf16": 2, "fp16": 2, "fp32": 4}
    if kind == "append":
        token = h * 2 * D * width[case["dtype"]] + 2 * row8 + row4 + 12   # read, write the ring; read the old row, write INT4
        return dict(bytes=2 * case["layers"] * case["ring"] * token, flops=0)
    if kind == "store":
        return dict(bytes=case["layers"] * case["n"] * (h * 2 * D * width[case["dtype"]] + row8 + row4 + 12), flops=0)
    n = sum(min(int(x), case["topk"]) if case["which"] == "topk" else int(x) for x in case["lens"].split(","))
    return dict(bytes=n * (row[case["pool"]] + h * 2 * D * 2 + 8), flops=0)


def tolerance(case):
    """About four times the distance from `exact` measured over these ranges."""
    kind = case["kind"]
    if kind in ("append", "store", "gather"):
        return "exact"   # codes, scales and dequantized rows are fixed bit for bit
    if kind == "decode":   # fp16 weights over raw codes, fp32 sums: 5e-5 at 10,000 positions, 3.2e-4 at 262,144
        return {"rel": 1.3e-3, "max": 6e-3}
    if kind in ("paged", "prefill"):   # bf16 outputs: 1.7e-3, largest 6.2e-3
        return {"rel": 6.6e-3, "max": 2.5e-2}
    return {"rel": 4e-6, "max": 6e-5}   # topk, slots: fp32 outputs of 16-bit weights, 1e-6, largest 1.4e-5
