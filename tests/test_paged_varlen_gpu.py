"""Packed prompts over a paged cache, read in place by the paged tile kernel, against the same call
with a gradient asked for (which gathers the pages and runs the packed forward) and, where that is
also the same tile walk, against it bit for bit. The cases cover GQA groups packed into the rows,
tiles around 256 rows, pages of 16 to 256 rows, lengths that end inside a page, sequences without
queries or keys, seqused, windows on both sides, a chunk, softcap and alibi, the kernel widths, and
caches whose pages, rows and heads are strided."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.helpers import TOL

pytestmark = pytest.mark.gpu

# name, D, Hq, Hk, page, q lengths, k lengths, options
CASES = [
    ("gqa4 p16", 128, 8, 2, 16, [37, 64, 100], [90, 64, 230], {}),
    ("mha p32", 128, 2, 2, 32, [256, 257, 1], [256, 300, 700], {}),
    ("gqa8 p256 long", 128, 8, 1, 256, [65, 30], [2500, 31], {}),
    ("empty sequences", 128, 4, 2, 16, [0, 5, 20, 0], [33, 0, 20, 0], {}),
    ("more queries than keys", 128, 4, 2, 16, [90, 40], [50, 40], {}),
    ("full mask", 128, 4, 1, 16, [50, 3], [500, 129], {"causal": False}),
    ("window", 128, 4, 2, 16, [200, 77], [600, 77], {"window_size": (100, 0)}),
    ("two-sided window", 128, 4, 2, 16, [200, 77], [600, 90], {"causal": False, "window_size": (64, 33)}),
    ("chunk", 128, 4, 2, 16, [200, 77], [600, 90], {"attention_chunk": 128}),
    ("softcap", 128, 4, 2, 64, [200, 77], [300, 77], {"softcap": 20.0}),
    ("alibi", 128, 4, 2, 64, [200, 77], [300, 77], {"alibi": True}),
    ("D64", 64, 8, 2, 16, [150, 300], [900, 300], {}),
    ("D40", 40, 4, 2, 16, [150, 30], [200, 30], {}),
    ("D256", 256, 4, 2, 16, [70, 130], [400, 130], {}),
    ("D256 window softcap", 256, 4, 2, 16, [70, 130], [400, 130], {"window_size": (96, 0), "softcap": 30.0}),
    ("D96 gathers", 96, 4, 2, 16, [70], [100], {}),
]


def _call(case, dt, strided=False, used=False):
    import torch

    from fable_attn import flash_attn_varlen_func
    name, D, Hq, Hk, page, lq, lk, opt = case
    opt = dict(opt)
    opt.setdefault("causal", True)
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=dt)
    if opt.pop("alibi", False):
        opt["alibi_slopes"] = torch.linspace(0.02, 0.3, Hq, device="cuda")
    nb = max(1, max(-(-n // page) for n in lk))
    q = rnd(sum(lq), Hq, D)
    pool = len(lk) * nb + 2
    if strided:   # (heads outside rows, and K and V interleaved per page)
        kv = rnd(pool, 2, Hk, page, D)
        kc, vc = kv[:, 0].transpose(1, 2), kv[:, 1].transpose(1, 2)
    else:
        kc, vc = rnd(pool, page, Hk, D), rnd(pool, page, Hk, D)
    bt = torch.randperm(pool, generator=torch.Generator().manual_seed(5))[:len(lk) * nb].view(len(lk), nb).int()
    for z, n in enumerate(lk):
        bt[z, -(-n // page):] = 10 ** 6 + z      # never read
    bt = bt.cuda()
    cu = lambda n: torch.tensor([0] + list(np.cumsum(n)), dtype=torch.int32, device="cuda")
    if used:
        opt["seqused_q"] = torch.tensor([max(n - 3, 0) for n in lq], dtype=torch.int32, device="cuda")
        opt["seqused_k"] = torch.tensor([max(n - 5, 0) for n in lk], dtype=torch.int32, device="cuda")
    f = lambda qq: flash_attn_varlen_func(qq, kc, vc, cu(lq), cu(lk), max(lq), max(lk), block_table=bt, **opt)
    with torch.no_grad():
        got = f(q)
    qg = q.clone()
    if "attention_chunk" in opt:    # (no gradient with a chunk: the packed call itself)
        from fable_attn import flash_attn_interface as fai
        k, v, ck, uk, mk = fai._pages_as_packed(kc, vc, bt, cu(lk), opt.pop("seqused_k", None))
        want = flash_attn_varlen_func(q, k, v, cu(lq), ck, max(lq), mk, seqused_k=uk, **opt)
    else:
        want = f(qg.requires_grad_(True)).detach()
    torch.cuda.synchronize()
    return got, want


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_paged_equals_gathered(case, dt):
    import torch
    print(f"[paged] {case[0]} {dt}", flush=True)
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dt]
    for kw in ({}, {"strided": True}, {"used": True}):
        got, want = _call(case, t, **kw)
        a, b = got.float().cpu().numpy(), want.float().cpu().numpy()
        assert np.isfinite(a).all()
        # both are within TOL of the exact result
        assert orc.rel_rms(a, b) <= 2 * TOL[dt], kw
        assert np.array_equal(a == 0, b == 0), kw   # rows without a key


@pytest.mark.parametrize("D,page,window", [(128, 16, 100), (64, 64, 77), (256, 16, 33), (40, 32, 5)])
def test_pages_before_the_window_are_not_read(D, page, window):
    """NaN in the rows that no query's window reaches, and in the page that their table entries name."""
    import torch

    from fable_attn import flash_attn_varlen_func
    lq, lk, Hk = [70, 9, 130], [700, 300, 130], 2
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    nb = -(-max(lk) // page)
    kc, vc = rnd(3 * nb + 1, page, Hk, D), rnd(3 * nb + 1, page, Hk, D)
    bt = torch.randperm(3 * nb, generator=torch.Generator().manual_seed(5)).view(3, nb).int()
    q = rnd(sum(lq), 4, D)
    cu = lambda n: torch.tensor([0] + list(np.cumsum(n)), dtype=torch.int32, device="cuda")
    f = lambda table: flash_attn_varlen_func(q, kc, vc, cu(lq), cu(lk), max(lq), max(lk), block_table=table.cuda(),
                                             causal=True, window_size=(window, 0))
    want = f(bt)
    kc[-1], vc[-1] = float("nan"), float("nan")
    hidden = bt.clone()
    for z in range(3):
        lo = max(lk[z] - lq[z] - window, 0)
        kc[bt[z, lo // page].item(), :lo % page] = float("nan")
        vc[bt[z, lo // page].item(), :lo % page] = float("nan")
        hidden[z, :lo // page] = 3 * nb
    assert torch.equal(f(hidden), want)


@pytest.mark.parametrize("batch,Hk,gqa", [(8, 2, 4), (8, 4, 2), (8, 8, 1), (12, 2, 4), (9, 3, 2), (3, 1, 4)])
def test_paged_work_order(batch, Hk, gqa):
    """The order of the work items (the groups of an XCD turned step by step): every tile of every prompt,
    whatever the count of K/V groups per XCD (2, 4, 8, 3, 3 and some left over, none full), their lengths
    unequal."""
    import torch
    r = np.random.default_rng(batch * Hk)
    lq = [int(x) for x in r.integers(1, 700, batch)]
    lk = [n + int(x) for n, x in zip(lq, r.integers(0, 500, batch))]
    lq[batch // 2], lk[0] = 900, 1900
    lk[batch // 2] = 1000
    got, want = _call(("order", 64, Hk * gqa, Hk, 16, lq, lk, {}), torch.bfloat16)
    assert orc.rel_rms(got.float().cpu().numpy(), want.float().cpu().numpy()) <= 2 * TOL["bf16"]


@pytest.mark.parametrize("max_sk", [1500, None, 12000])
def test_wide_prompts_on_both_sides_of_the_gather(max_sk, monkeypatch):
    """Head dim 256 read in place or gathered, as max_seqlen_k (a bound, or None for the table's) says: the
    same result to the rounding of both."""
    import torch

    from fable_attn import _C, flash_attn_varlen_func
    seen = []
    fwd_paged = _C.fwd_paged
    monkeypatch.setattr(_C, "fwd_paged", lambda *a, **k: seen.append(1) or fwd_paged(*a, **k))
    g = torch.Generator(device="cuda").manual_seed(4)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    lq, lk, H, Hk, page, cols = [1030, 40], [1500, 900], 8, 1, 64, 192
    kc, vc, q = rnd(48, page, Hk, 256), rnd(48, page, Hk, 256), rnd(sum(lq), H, 256)
    bt = torch.randperm(48, generator=torch.Generator().manual_seed(5)).view(2, 24).int()
    bt = torch.cat([bt, bt[:, :1].expand(2, cols - 24)], 1).contiguous().cuda()
    cu = lambda n: torch.tensor([0] + list(np.cumsum(n)), dtype=torch.int32, device="cuda")
    f = lambda mk: flash_attn_varlen_func(q, kc, vc, cu(lq), cu(lk), max(lq), mk, block_table=bt, causal=True)
    got = f(max_sk)
    assert len(seen) == (max_sk == 1500)   # 24.7M pairs; the table's 12288 keys or 12000: 200M
    assert orc.rel_rms(got.float().cpu().numpy(), f(1500).float().cpu().numpy()) <= 2 * TOL["bf16"]
