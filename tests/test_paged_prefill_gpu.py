"""Paged block-sparse prefill (srswa.unlimited_dash_ops.dash_sparse_attn, the
drop-in for the SGLang backend's K10 dash_sparse_attn) vs the CPU oracle
(``srswa_oracle.paged_prefill_attend``, K10's two passes query by query).

Bar: bf16 / fp16 outputs max-abs <= 2e-2 beyond the output format's half-ulp
(tests/tolerance.py) against fp64 on the same rounded inputs.  Inputs follow
the router's contract: per-kv-head ids packed at the front (ascending,
unique, -1 after), optional fp32 slot biases.  fp8 caches of the four torch
fp8 formats are compared against the oracle on their exact values."""

import math

import pytest
import torch

from oracle import srswa_oracle as O
from srswa import unlimited_dash_ops as U
from tolerance import assert_close_lowp

pytestmark = pytest.mark.gpu


def _case(seed, q_lens, ctx, page, Hkv, G, D, S, dtype, nb_extra=3, bias=True, kv=None):
    g = torch.Generator().manual_seed(seed)
    R = len(q_lens)
    seq = [c + q for c, q in zip(ctx, q_lens)]
    nb = max(-(-s // page) for s in seq) + nb_extra
    npages = R * nb + 4
    kc = torch.randn(npages, page, Hkv, D, generator=g).to(kv or dtype)
    vc = torch.randn(npages, page, Hkv, D, generator=g).to(kv or dtype)
    bt = torch.randperm(npages, generator=g)[:R * nb].view(R, nb).to(torch.int32)
    cu = [0]
    for ql in q_lens:
        cu.append(cu[-1] + ql)
    total = cu[-1]
    H = Hkv * G
    q = torch.randn(total, H, D, generator=g).to(dtype)
    topk = torch.full((Hkv, total, S), -1, dtype=torch.int32)
    for r in range(R):
        for n in range(cu[r], cu[r + 1]):
            qp = ctx[r] + n - cu[r]
            live = -(-seq[r] // page)
            for kh in range(Hkv):
                k = int(torch.randint(0, S + 1, (1,), generator=g))
                ids = torch.randperm(max(live, 1), generator=g)[:k].sort().values
                topk[kh, n, :len(ids)] = ids.to(torch.int32)
            _ = qp
    bsl = torch.randn(Hkv, total, S, generator=g) if bias else None
    return dict(q=q, kc=kc, vc=vc, bt=bt, cu=torch.tensor(cu, dtype=torch.int32),
                seq=torch.tensor(seq, dtype=torch.int32), ctx=torch.tensor(ctx, dtype=torch.int32),
                topk=topk, bias=bsl, max_q=max(q_lens), Hkv=Hkv, page=page)


CASES = {
    "bf16_p64_lb8": dict(q_lens=[70, 1, 130], ctx=[900, 40, 0], page=64, Hkv=2, G=2, D=128, S=8,
                         dtype=torch.bfloat16, lb=8),
    "bf16_p32_lb4_nobias": dict(q_lens=[64, 33], ctx=[500, 1200], page=32, Hkv=1, G=3, D=128, S=6,
                                dtype=torch.bfloat16, lb=4, bias=False),
    "fp16_p16_d64": dict(q_lens=[90, 17, 5], ctx=[300, 0, 77], page=16, Hkv=2, G=1, D=64, S=5,
                         dtype=torch.float16, lb=6),
    "bf16_p128_no_window": dict(q_lens=[40, 65], ctx=[600, 200], page=128, Hkv=2, G=2, D=128, S=4,
                                dtype=torch.bfloat16, lb=0),
    "fp8_e4m3fn_p64": dict(q_lens=[70, 1, 130], ctx=[900, 40, 0], page=64, Hkv=2, G=2, D=128, S=8,
                           dtype=torch.bfloat16, lb=8, kv=torch.float8_e4m3fn),
    "fp8_e5m2_p32_nobias": dict(q_lens=[64, 33], ctx=[500, 1200], page=32, Hkv=1, G=3, D=128, S=6,
                                dtype=torch.bfloat16, lb=4, bias=False, kv=torch.float8_e5m2),
    "fp8_e4m3fnuz_fp16_d64": dict(q_lens=[90, 17, 5], ctx=[300, 0, 77], page=16, Hkv=2, G=1, D=64, S=5,
                                  dtype=torch.float16, lb=6, kv=torch.float8_e4m3fnuz),
    "fp8_e5m2fnuz_p128": dict(q_lens=[40, 65], ctx=[600, 200], page=128, Hkv=2, G=2, D=128, S=4,
                              dtype=torch.bfloat16, lb=2, kv=torch.float8_e5m2fnuz),
}


@pytest.mark.parametrize("name", list(CASES))
def test_dash_sparse_attn_matches_oracle(dev, name):
    kw = dict(CASES[name])
    lb = kw.pop("lb")
    c = _case(list(CASES).index(name) + 40, **kw)
    scale = 1 / math.sqrt(kw["D"])
    out = torch.full(c["q"].shape, float("nan"), dtype=c["q"].dtype, device=dev)
    print(f"dash_sparse_attn {name}", flush=True)
    U.dash_sparse_attn(c["q"].to(dev), c["kc"].to(dev), c["vc"].to(dev), c["topk"].to(dev),
                       None if c["bias"] is None else c["bias"].to(dev), c["bt"].to(dev), c["cu"].to(dev),
                       c["seq"].to(dev), c["ctx"].to(dev), c["max_q"], c["Hkv"], scale, out, local_blocks=lb,
                       sparse_block_size=c["page"])
    ref = O.paged_prefill_attend(c["q"].double(), c["kc"].double(), c["vc"].double(), c["topk"].long(),
                                 None if c["bias"] is None else c["bias"].double(), c["bt"].long(), c["cu"].tolist(),
                                 c["seq"].tolist(), c["ctx"].tolist(), lb, scale)
    assert_close_lowp(out.cpu(), ref, kw["dtype"], 2e-2, f"dash_sparse_attn {name}")


def test_dash_sparse_attn_head_expanded_ids(dev):
    """The backend's call: one router row expanded over the kv heads with
    stride 0 (unlimited_ocr_v2_backend.py:1421-1422), read in place."""
    c = _case(77, [50, 20], [300, 64], 64, 1, 2, 128, 8, torch.bfloat16)
    Hkv = 4
    g = torch.Generator().manual_seed(5)
    kc = torch.randn(c["kc"].shape[0], 64, Hkv, 128, generator=g).to(torch.bfloat16)
    vc = torch.randn(c["vc"].shape[0], 64, Hkv, 128, generator=g).to(torch.bfloat16)
    q = torch.randn(c["q"].shape[0], Hkv * 2, 128, generator=g).to(torch.bfloat16)
    ids = c["topk"][0].to(dev)
    bias = c["bias"][0].to(dev)
    di = ids.unsqueeze(0).expand(Hkv, -1, -1)
    db = bias.unsqueeze(0).expand(Hkv, -1, -1)
    out = torch.empty(q.shape, dtype=q.dtype, device=dev)
    U.dash_sparse_attn(q.to(dev), kc.to(dev), vc.to(dev), di, db, c["bt"].to(dev), c["cu"].to(dev), c["seq"].to(dev),
                       c["ctx"].to(dev), c["max_q"], Hkv, 0.088, out, local_blocks=8, sparse_block_size=64)
    ref = O.paged_prefill_attend(q.double(), kc.double(), vc.double(), di.cpu().long(), db.cpu().double(),
                                 c["bt"].long(), c["cu"].tolist(), c["seq"].tolist(), c["ctx"].tolist(), 8, 0.088)
    assert_close_lowp(out.cpu(), ref, torch.bfloat16, 2e-2, "dash_sparse_attn head-expanded ids")


@pytest.mark.parametrize("max_q,parts", [(64, 8), (190, 4), (640, 2), (1100, 1)])
@pytest.mark.parametrize("kv", [None, torch.float8_e4m3fn])
def test_split_launch_matches_whole_tiles(dev, monkeypatch, max_q, parts, kv):
    """A launch of few tiles runs each as 8, 4 or 2 workgroups over parts of its
    chunks (16 heads x 3 requests of ceil(max_q / 64) tiles, most of them past
    their request's rows; a request of one key leaves parts without a chunk)
    against every tile whole.  Each probability is rounded to bf16 (2^-9 of it)
    relative to its part's own reference maximum, so the two forms round it
    differently: they are at most 2 * 2^-9 * sum(p |v|) <= 2^-8 max|v| apart
    before the output's own rounding (one unit in the last place)."""
    import ctypes
    from srswa import _lib
    lib, H, D, page, K = _lib.lib(), 16, 128, 64, 8
    g = torch.Generator().manual_seed(max_q)
    q_lens, ctx = [max_q, 1, min(65, max_q)], [700, 0, 64 * 9 - 1]
    seq = [a + b for a, b in zip(q_lens, ctx)]
    nb = -(-max(seq) // page)
    total = sum(q_lens)
    rnd = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, kc, vc = rnd(total, H, D).to(dev), rnd(3 * nb, page, H, D), rnd(3 * nb, page, H, D)
    kc, vc = (x.to(kv or torch.bfloat16).to(dev) for x in (kc, vc))
    bt = torch.randperm(3 * nb, generator=g).view(3, nb).to(torch.int32).to(dev)
    ids = torch.randint(-1, nb, (H, total, K), generator=g).to(torch.int32).to(dev)
    bias = torch.randn(H, total, K, generator=g).to(dev)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    cu = i32([0, q_lens[0], q_lens[0] + 1, total])
    asked = []
    real = lib.srswa_gather_fwd_paged_workspace

    def run(split):
        def workspace(a):
            asked.append(real(a))
            return asked[-1] if split else 0
        monkeypatch.setattr(lib, "srswa_gather_fwd_paged_workspace", workspace)
        out = torch.zeros(total, H, D, dtype=torch.bfloat16, device=dev)
        U.dash_sparse_attn(q, kc, vc, ids, bias, bt, cu, i32(seq), i32(ctx), max_q, H, D ** -0.5, out, local_blocks=2,
                           sparse_block_size=page)
        return out.float()

    whole, split = run(False), run(True)
    tiles = 3 * H * -(-max_q // 64)
    assert asked[0] == (0 if parts == 1 else tiles * parts * (64 * D + 128) * 4), (asked, tiles)
    assert torch.isfinite(split).all()
    ulp = torch.exp2(torch.floor(torch.log2(whole.abs().clamp(min=1e-3))) - 7)
    assert ((split - whole).abs() <= 2.0 ** -8 * vc.float().abs().max() + ulp).all()
    if parts == 1:
        assert torch.equal(split, whole)


def _request_case(dev, seed, q_lens, ctx, *, H, HKV, D, page, K, dtype, kv=None, bias=True):
    """Requests over pages dealt in random order, every row its own selection."""
    g = torch.Generator(device=dev).manual_seed(seed)
    seq = [a + b for a, b in zip(q_lens, ctx)]
    nb, total = -(-max(seq) // page), sum(q_lens)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)
    kc, vc = (rnd(len(seq) * nb, page, HKV, D).to(kv or dtype) for _ in range(2))
    return dict(q=rnd(total, H, D), k=kc, v=vc, page=page, HKV=HKV, q_lens=q_lens, ctx=ctx,
                bt=torch.randperm(len(seq) * nb, generator=g, device=dev).view(len(seq), nb).to(torch.int32),
                ids=torch.randint(-1, nb, (HKV, total, K), generator=g, device=dev).to(torch.int32),
                bias=torch.randn(HKV, total, K, generator=g, device=dev) if bias else None)


def _attend(c, pieces=None):
    """The requests' rows in one launch, or ``pieces`` [(request, first row, rows)] as its requests."""
    dev, starts = c["q"].device, [sum(c["q_lens"][:i]) for i in range(len(c["q_lens"]))]
    pieces = pieces or [(r, 0, n) for r, n in enumerate(c["q_lens"])]
    rows = torch.cat([torch.arange(starts[r] + t, starts[r] + t + n) for r, t, n in pieces]).to(dev)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)
    q = c["q"][rows]
    out = torch.zeros_like(q)
    U.dash_sparse_attn(q, c["k"], c["v"], c["ids"][:, rows].contiguous(),
                       None if c["bias"] is None else c["bias"][:, rows].contiguous(),
                       c["bt"][[r for r, _, _ in pieces]].contiguous(),
                       i32([0] + [n for _, _, n in pieces]).cumsum(0).to(torch.int32),
                       i32([c["ctx"][r] + c["q_lens"][r] for r, _, _ in pieces]), i32([c["ctx"][r] + t for r, t, _ in pieces]),
                       max(n for _, _, n in pieces), c["HKV"], q.shape[-1] ** -0.5, out, local_blocks=2,
                       sparse_block_size=c["page"])
    return out


@pytest.mark.parametrize("D,K,page,ctx,kv", [(128, 8, 64, 20000, None), (128, 8, 64, 20000, torch.float8_e4m3fn),
                                             (128, 12, 16, 5000, None), (64, 39, 64, 29000, None),
                                             (64, 39, 64, 29000, torch.float8_e5m2)])
def test_more_rounds_than_one_match_short_launches(dev, monkeypatch, D, K, page, ctx, kv):
    """784 tiles of one request, more than three workgroups per CU: a layout that
    holds four takes the narrower V pitch.  Launches of 400 and 384 of the same
    tiles take the other; both visit the same chunks in the same order, so
    their rows agree to the last bit.  (Without the split, which rounds otherwise.)"""
    from srswa import _lib
    monkeypatch.setattr(_lib.lib(), "srswa_gather_fwd_paged_workspace", lambda a: 0)
    c = _request_case(dev, D + K, [49 * 64 - 5], [ctx], H=16, HKV=16, D=D, page=page, K=K, dtype=torch.bfloat16, kv=kv)
    whole = _attend(c)
    first = _attend(c, [(0, 0, 25 * 64)])
    second = _attend(c, [(0, 25 * 64, 24 * 64 - 5)])
    assert torch.isfinite(whole.float()).all()
    assert torch.equal(whole, torch.cat([first, second]))


@pytest.mark.parametrize("H,rows", [(1, 1), (1, 700), (3, 64), (3, 321), (10, 65), (10, 1000), (4, 700), (8, 321)])
def test_one_request_matches_itself_beside_another(dev, monkeypatch, H, rows):
    """The tiles of one request are dealt to the XCDs in eighths, those of
    several in turn (tile counts that are no multiple of eight, fewer than
    eight, one; requests times heads 8 and 16, where a head's tiles stay on one
    XCD): the same rows to the last bit.  (Without the split.)"""
    from srswa import _lib
    monkeypatch.setattr(_lib.lib(), "srswa_gather_fwd_paged_workspace", lambda a: 0)
    c = _request_case(dev, rows, [rows, 1], [900, 70], H=H, HKV=H, D=128, page=64, K=5, dtype=torch.bfloat16)
    alone, beside = _attend(c, [(0, 0, rows)]), _attend(c)
    assert torch.isfinite(beside.float()).all() and alone.abs().amax(-1).min() > 0
    assert torch.equal(alone, beside[:rows])


BF, HF = torch.bfloat16, torch.float16


@pytest.mark.parametrize("H,HKV,D,page,K,dtype,kv,bias,q_lens,ctx,parts", [
    (8, 2, 64, 16, 6, HF, None, False, [320, 1, 65], [700, 0, 300], 8),
    (8, 8, 128, 32, 4, BF, None, False, [320, 1, 65], [700, 0, 300], 8),
    (6, 3, 64, 64, 5, BF, torch.float8_e5m2, True, [130], [640], 8),
    (16, 4, 64, 32, 5, HF, None, False, [400, 3], [300, 900], 4),
    (16, 4, 128, 16, 5, HF, None, True, [640, 3], [100, 2000], 2),
    (10, 10, 128, 64, 8, BF, None, True, [250], [0], 4),          # a table of four chunks
    (16, 16, 128, 64, 8, BF, None, True, [250], [0], 2),
    (10, 10, 128, 64, 8, BF, None, True, [60], [0], 1),           # of one: nothing to split
    (10, 10, 128, 64, 8, BF, None, True, [168, 12], [64, 30], 4),
    (10, 10, 128, 64, 8, BF, None, True, [250, 60, 100], [64, 0, 64], 2),
    (10, 10, 128, 64, 8, BF, None, True, [120, 20, 12, 60, 90, 30, 15, 100], [150] * 8, 1),
    (10, 10, 128, 64, 8, BF, None, True, [64, 1, 20, 33] * 3, [64] * 12, 1),
])
def test_split_forms_match_whole_tiles(dev, monkeypatch, H, HKV, D, page, K, dtype, kv, bias, q_lens, ctx, parts):
    """The split over head dims, types, head groups, page sizes and the number of
    parts (256 CUs), with and without bias, against every tile whole.  Bar as
    in test_split_launch_matches_whole_tiles: 2 u max|v| and one unit in the
    output's last place, u the 16-bit type's rounding of a probability."""
    from srswa import _lib
    real, asked = _lib.lib().srswa_gather_fwd_paged_workspace, []
    c = _request_case(dev, sum(q_lens), q_lens, ctx, H=H, HKV=HKV, D=D, page=page, K=K, dtype=dtype, kv=kv, bias=bias)
    monkeypatch.setattr(_lib.lib(), "srswa_gather_fwd_paged_workspace", lambda a: asked.append(real(a)) or asked[-1])
    split = _attend(c)
    monkeypatch.setattr(_lib.lib(), "srswa_gather_fwd_paged_workspace", lambda a: 0)
    whole = _attend(c)
    tiles = len(q_lens) * H * -(-max(q_lens) // 64)
    assert asked == [0 if parts == 1 else tiles * parts * (64 * D + 128) * 4]
    if parts == 1:
        assert torch.equal(split, whole)
        return
    split, whole, vmax = split.float(), whole.float(), c["v"].float().abs().max()
    digits = 8 if dtype == BF else 11
    ulp = torch.exp2(torch.floor(torch.log2(whole.abs().clamp(min=1e-3))) - (digits - 1))
    assert torch.isfinite(split).all() and ((split - whole).abs() <= 2.0 ** -digits * vmax + ulp).all()
    assert not torch.equal(split, whole)          # the split did run
