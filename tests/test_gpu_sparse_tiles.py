"""The 16-column tiles of the sparse attention kernel at the edges of its column table and of its row pairs: selections
of 1 to 65 columns and just past one table pass, with identity smoothing (bodies without the products) and without,
whole tiles in one tier, mixed tiles, and decode blocks of one and of several tiles per wavefront, for every pool kind.
Against the oracle's fp32 attention over the gather's bf16 rows within 2e-3 max-abs / 1e-3 mean-abs (P keeps 16
significant bits, K and V are the oracle's rows exactly, sums are fp32: the difference is far below, 1e-5)."""
import pytest
import torch

from kvt_testutil import close, pool_args, slot_pools, slot_rows
from oracle import ref

pytestmark = pytest.mark.gpu
dev = "cuda"
H, D, HQ = 2, 256, 24


def _owner(p, R, tiers, slots):
    if tiers == "ring":        # the selected slots (below R) all own their ring rows
        p["owner"] = torch.arange(R, dtype=torch.int32)
    elif tiers == "pool":
        p["owner"] = torch.full((R,), -1, dtype=torch.int32)


@pytest.mark.parametrize("kind,tiers,identity", [("tiered", "mixed", True), ("tiered", "mixed", False),
                                                 ("tiered", "ring", True), ("tiered", "pool", True),
                                                 ("int4", "", True), ("int8", "", True), ("int8", "", False)])
def test_tile_edges(kvt_pkg, kind, tiers, identity):
    from kvtier import sparse_attn as sa
    gen = torch.Generator().manual_seed(71)
    R = 8192
    slots = R if tiers == "ring" else 2 * R
    p = slot_pools(slots, R, 64, gen)
    _owner(p, R, tiers, slots)
    if identity:
        p["sm_k"], p["sm_v"] = (torch.ones(H, D, dtype=torch.float16) for _ in range(2))
    counts = [1, 2, 15, 16, 17, 31, 33, 63, 64, 65, 1025, 4097]
    n = len(counts)
    L, topk = 5000, 4100
    r2t = torch.stack([torch.randperm(slots, generator=gen)[:L] for _ in range(n)]).to(torch.int32)
    idx = torch.full((n, topk), -1, dtype=torch.int32)
    for b, c in enumerate(counts):
        idx[b, :c] = torch.randperm(L, generator=gen)[:c].to(torch.int32)
    q = (torch.randn(n, HQ, D, generator=gen) / 4).to(torch.bfloat16)
    lens = torch.full((n,), L, dtype=torch.int32)
    exp = torch.empty(n, HQ, D)
    gs = HQ // H
    for b, c in enumerate(counts):
        kk, vv = slot_rows(kind, p, r2t[b, idx[b, :c].long()].long(), R, 64)
        for h in range(H):
            exp[b, h * gs:(h + 1) * gs] = ref.attention_rows(q[b, h * gs:(h + 1) * gs], kk[:, h:h + 1], vv[:, h:h + 1],
                                                             D ** -0.5)
    a = pool_args(kind, p, R, dev)
    req = torch.arange(n, device=dev)
    # prefill rows: one chunk of one query per request
    cu = torch.arange(n + 1, dtype=torch.int32, device=dev)
    out = torch.empty(n, HQ, D, device=dev)
    sa.sparse_gqa_fwd_interface_paged(q.to(dev), idx.to(dev), cu, lens.to(dev), r2t.to(dev), req, scale=D ** -0.5,
                                      max_q=1, out=out, **a)
    close(out.cpu(), exp)
    # decode: one tile per wavefront, several (one and two table passes)
    cu_k = torch.nn.functional.pad(torch.tensor(counts).cumsum(0), (1, 0)).to(torch.int32).to(dev)
    for splits in (-(-topk // 64), 5, 1):
        got = sa.qwen_sparse_decode_attn(
            q.to(dev), a["k_buf"], a["v_buf"], r2t.to(dev), req, idx.to(dev), lens.to(dev), cu_k, n, topk, a["k_scale"],
            a["v_scale"], a["sm_k"], a["sm_v"], a["kv_bits"], **{k: a[k] for k in a if k.startswith(("ring_", "owner"))},
            splits=splits, out=torch.empty(n, HQ, D, device=dev))
        close(got.cpu(), exp)


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
