"""The 16-column tiles of the sparse attention kernel at the edges of its column table and of its row pairs: selections
of 1 to 65 columns and just past one table pass, with identity smoothing (bodies without the products) and without,
whole tiles in one tier, mixed tiles, and decode blocks of one and of several tiles per wavefront, for every pool kind.

The queries are peaked: each q head puts about half of its weight on two columns at such an edge (the last column, the
first, columns 15 to 17, 31 to 33, 63 to 65, 1,023 to 1,025, 4,095 and 4,096 where the selection has them), the second at 0.8 of the
first's score, so that a lost or doubled edge row changes its outputs by far more than the tolerance, and so does a P
rounded to bf16 without its remainder (both checked on the CPU, planted in the oracle).

Tolerance, against the oracle's fp32 attention over the gather's bf16 rows (K and V are those rows exactly): P's
remainder leaves 2^-17 of a weight, a score of up to 16 log2 units in fp32 2^-18 of one (2 ulps), a chain of 65 tiles 2^-18 of a sum;
times the largest |V|, 4.2 (code 8, scale 0.35, factor 1.5): 2^-16 * 4.2 = 6.4e-5 at most, and a mean of 1 / 8 of it."""
import math

import pytest
import torch

from kvt_testutil import close, pool_args, slot_pools, slot_rows
from oracle import ref

dev = "cuda"
H, D, HQ = 2, 256, 24
GS = HQ // H
MAX_ABS, MEAN_ABS = 6.4e-5, 8e-6
KINDS = [("tiered", "mixed", True), ("tiered", "mixed", False), ("tiered", "ring", True), ("tiered", "pool", True),
         ("int4", "", True), ("int8", "", True), ("int8", "", False)]
COUNTS = [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 1025, 4097]
R, LEN, TOPK = 8192, 5000, 4100


def _owner(p, R, tiers, slots):
    if tiers == "ring":        # the selected slots (below R) all own their ring rows
        p["owner"] = torch.arange(R, dtype=torch.int32)
    elif tiers == "pool":
        p["owner"] = torch.full((R,), -1, dtype=torch.int32)


def _edges(c):
    """Columns at an edge of a selection of c, the last one first, in pairs for the 12 heads of a group."""
    cols = [x for x in (c - 1, 4095, 1024, 1023, 64, 63, 32, 31, 16, 15, 0, 4096, 17, 33, 65, 1025) if 0 <= x < c]
    cols = list(dict.fromkeys(cols))[:GS]
    return [(cols[i % len(cols)], cols[(i + 1) % len(cols)]) for i in range(GS)]


def _case(kind, tiers, identity):
    """Pool, index rows, queries and the selected rows of one request per count."""
    gen = torch.Generator().manual_seed(71)
    slots = R if tiers == "ring" else 2 * R
    p = slot_pools(slots, R, 64, gen)
    _owner(p, R, tiers, slots)
    if identity:
        p["sm_k"], p["sm_v"] = (torch.ones(H, D, dtype=torch.float16) for _ in range(2))
    n = len(COUNTS)
    r2t = torch.stack([torch.randperm(slots, generator=gen)[:LEN] for _ in range(n)]).to(torch.int32)
    idx = torch.full((n, TOPK), -1, dtype=torch.int32)
    q = torch.empty(n, HQ, D)
    rows = []
    for b, c in enumerate(COUNTS):
        idx[b, :c] = torch.randperm(LEN, generator=gen)[:c].to(torch.int32)
        kk, vv = slot_rows(kind, p, r2t[b, idx[b, :c].long()].long(), R, 64)
        rows.append((kk, vv))
        for h in range(H):
            for i, (x, y) in enumerate(_edges(c)):
                k = kk[x, h].float() + (0.8 * kk[y, h].float() if x != y else 0.0)
                q[b, h * GS + i] = k * (16.0 * (math.log(c) + 1.0) / float(kk[x, h].float().square().sum()))
    return p, r2t, idx, q.to(torch.bfloat16), rows


def _oracle(q, rows, drop=None, bf16_weights=False):
    """The oracle's attention per request; drop: leaves column drop(b) out; bf16_weights: rounds P / max P to bf16."""
    out = torch.empty(len(COUNTS), HQ, D)
    for b, (kk, vv) in enumerate(rows):
        keep = torch.arange(kk.shape[0]) != (-1 if drop is None else drop(b))
        for h in range(H):
            qh, kh, vh = q[b, h * GS:(h + 1) * GS], kk[keep, h], vv[keep, h]
            if bf16_weights:
                s = qh.float() @ kh.float().T * D ** -0.5
                e = (s - s.amax(-1, keepdim=True)).exp()
                out[b, h * GS:(h + 1) * GS] = e.to(torch.bfloat16).float() @ vh.float() / e.sum(-1, keepdim=True)
            else:
                out[b, h * GS:(h + 1) * GS] = ref.attention_rows(qh, kh[:, None], vh[:, None], D ** -0.5)
    return out


@pytest.mark.parametrize("kind,tiers,identity", KINDS)
def test_edges_carry_weight(kind, tiers, identity):
    """On the CPU: the oracle with one edge column left out (the last, 1,023, 1,024, 4,095 or 4,096) differs from the oracle
    by more than a thousand times the tolerance, with P rounded to bf16 by more than five times."""
    p, r2t, idx, q, rows = _case(kind, tiers, identity)
    exp = _oracle(q, rows)
    off = (_oracle(q, rows, bf16_weights=True) - exp).abs().amax((1, 2))
    assert (off[1:] > 5 * MAX_ABS).all(), off   # (a single column's weight is 1 exactly)
    for drop in (lambda b: COUNTS[b] - 1, lambda b: 1023, lambda b: 1024, lambda b: 4095, lambda b: 4096):
        moved = [b for b in range(1, len(COUNTS)) if drop(b) < COUNTS[b]]
        off = (_oracle(q, rows, drop) - exp).abs().amax((1, 2))
        assert moved and (off[moved] > 1000 * MAX_ABS).all(), off


@pytest.mark.gpu
@pytest.mark.parametrize("kind,tiers,identity", KINDS)
def test_tile_edges(kvt_pkg, kind, tiers, identity):
    from kvtier import sparse_attn as sa
    p, r2t, idx, q, rows = _case(kind, tiers, identity)
    exp = _oracle(q, rows)
    n = len(COUNTS)
    lens = torch.full((n,), LEN, dtype=torch.int32)
    a = pool_args(kind, p, R, dev)
    req = torch.arange(n, device=dev)
    # prefill rows: one chunk of one query per request
    cu = torch.arange(n + 1, dtype=torch.int32, device=dev)
    out = torch.empty(n, HQ, D, device=dev)
    sa.sparse_gqa_fwd_interface_paged(q.to(dev), idx.to(dev), cu, lens.to(dev), r2t.to(dev), req, scale=D ** -0.5,
                                      max_q=1, out=out, **a)
    close(out.cpu(), exp, MAX_ABS, MEAN_ABS)
    # decode: one tile per wavefront, several (one and two table passes)
    cu_k = torch.nn.functional.pad(torch.tensor(COUNTS).cumsum(0), (1, 0)).to(torch.int32).to(dev)
    for splits in (-(-TOPK // 64), 5, 1):
        got = sa.qwen_sparse_decode_attn(
            q.to(dev), a["k_buf"], a["v_buf"], r2t.to(dev), req, idx.to(dev), lens.to(dev), cu_k, n, TOPK, a["k_scale"],
            a["v_scale"], a["sm_k"], a["sm_v"], a["kv_bits"], **{k: a[k] for k in a if k.startswith(("ring_", "owner"))},
            splits=splits, out=torch.empty(n, HQ, D, device=dev))
        close(got.cpu(), exp, MAX_ABS, MEAN_ABS)


@pytest.mark.gpu
def test_unaligned_smoothing(kvt_pkg):
    """Smoothing factors at an odd element offset (2-byte aligned only) give the outputs of aligned ones, bit for bit:
    prefill rows and decode."""
    from kvtier import sparse_attn as sa
    p, r2t, idx, q, rows = _case("tiered", "mixed", False)
    n = len(COUNTS)
    lens = torch.full((n,), LEN, dtype=torch.int32, device=dev)
    req, cu = torch.arange(n, device=dev), torch.arange(n + 1, dtype=torch.int32, device=dev)
    a = pool_args("tiered", p, R, dev)
    outs = []
    for shift in (0, 1):
        for name in ("sm_k", "sm_v"):
            buf = torch.zeros(H * D + 1, dtype=torch.float16, device=dev)
            a[name] = buf[shift:shift + H * D].view(H, D)
            a[name].copy_(p[name])
        pre = torch.empty(n, HQ, D, device=dev)
        sa.sparse_gqa_fwd_interface_paged(q.to(dev), idx.to(dev), cu, lens, r2t.to(dev), req, scale=D ** -0.5, max_q=1,
                                          out=pre, **a)
        dec = sa.qwen_sparse_decode_attn(
            q.to(dev), a["k_buf"], a["v_buf"], r2t.to(dev), req, idx.to(dev), lens, sa.ALL_COLUMNS, n, TOPK, a["k_scale"],
            a["v_scale"], a["sm_k"], a["sm_v"], 4, **{k: a[k] for k in a if k.startswith(("ring_", "owner"))})
        outs.append((pre.cpu(), dec.cpu()))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    close(outs[0][1], _oracle(q, rows), MAX_ABS, MEAN_ABS)


@pytest.mark.gpu
def test_all_columns_equals_counted(kvt_pkg):
    """ALL_COLUMNS in place of the valid counts (every position selected) gives the counted call's output bit for bit:
    lengths 0 (NaN), 1, at and beside a tile's end, and beyond the selection's width."""
    from kvtier import sparse_attn as sa
    gen = torch.Generator().manual_seed(72)
    R, slots, width = 1024, 4096, 700
    p = slot_pools(slots, R, 64, gen)
    lens = torch.tensor([0, 1, 16, 17, 640, 699, 700, 900], dtype=torch.int32)
    n = lens.numel()
    r2t = torch.stack([torch.randperm(slots, generator=gen)[:1000] for _ in range(n)]).to(torch.int32).to(dev)
    idx = torch.arange(width, dtype=torch.int32, device=dev)[None].expand(n, width)
    cu = torch.nn.functional.pad(lens.clamp(max=width).cumsum(0), (1, 0)).to(torch.int32).to(dev)
    q = (torch.randn(n, HQ, D, generator=gen) / 4).to(torch.bfloat16).to(dev)
    a = pool_args("tiered", p, R, dev)
    ring = {k: a[k] for k in a if k.startswith(("ring_", "owner"))}
    for splits in (None, 2):   # one tile per wavefront; several
        out = [sa.qwen_sparse_decode_attn(q, a["k_buf"], a["v_buf"], r2t, torch.arange(n, device=dev), idx, lens.to(dev), c,
                                          n, width, a["k_scale"], a["v_scale"], a["sm_k"], a["sm_v"], 4, splits=splits,
                                          **ring).cpu() for c in (cu, sa.ALL_COLUMNS)]
        assert torch.isnan(out[0][0]).all() and not torch.isnan(out[0][1:]).any()
        assert torch.equal(out[0].view(torch.int32), out[1].view(torch.int32))


@pytest.mark.gpu
def test_all_columns_takes_every_column(kvt_pkg):
    """ALL_COLUMNS attends a valid entry wherever it stands: rows whose valid entries come last, behind -1 padding, and
    in between, at columns beyond the request's length (lengths 3 to 100 against 512 columns), equal the call whose
    counts say all 512 columns, bit for bit, and the oracle; one tile per wavefront and several, merged in the launch
    and by the combine."""
    from kvtier import sparse_attn as sa
    gen = torch.Generator().manual_seed(74)
    R, slots, topk = 1024, 4096, 512
    p = slot_pools(slots, R, 64, gen)
    lens = torch.tensor([3, 40, 100, 100], dtype=torch.int32)
    n = lens.numel()
    idx = torch.full((n, topk), -1, dtype=torch.int32)
    for b in range(n):
        valid = torch.randperm(int(lens[b]), generator=gen).to(torch.int32)
        at = torch.arange(topk - valid.numel(), topk) if b % 2 == 0 else torch.randperm(topk, generator=gen)[:valid.numel()]
        idx[b, at] = valid
    idx[3, idx[3] < 0] = 100   # (at the length: not attended)
    r2t = torch.stack([torch.randperm(slots, generator=gen)[:100] for _ in range(n)]).to(torch.int32)
    q = (torch.randn(n, HQ, D, generator=gen) / 4).to(torch.bfloat16)
    exp = torch.empty(n, HQ, D)
    gs = HQ // H
    for b in range(n):
        kk, vv = slot_rows("tiered", p, r2t[b, :int(lens[b])].long(), R, 64)
        for h in range(H):
            exp[b, h * gs:(h + 1) * gs] = ref.attention_rows(q[b, h * gs:(h + 1) * gs], kk[:, h:h + 1], vv[:, h:h + 1],
                                                             D ** -0.5)
    cu = (torch.arange(n + 1) * topk).to(torch.int32).to(dev)
    a = pool_args("tiered", p, R, dev)
    ring = {k: a[k] for k in a if k.startswith(("ring_", "owner"))}
    for splits in (8, 3, 1):
        for merge in ("launch", "combine"):
            out = [sa.qwen_sparse_decode_attn(
                q.to(dev), a["k_buf"], a["v_buf"], r2t.to(dev), torch.arange(n, device=dev), idx.to(dev), lens.to(dev), c, n,
                topk, a["k_scale"], a["v_scale"], a["sm_k"], a["sm_v"], 4, splits=splits, merge=merge, **ring).cpu()
                for c in (cu, sa.ALL_COLUMNS)]
            assert torch.equal(out[0], out[1]), (splits, merge)
            close(out[1], exp)
