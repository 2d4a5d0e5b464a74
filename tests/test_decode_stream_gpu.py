"""Decode calls whose keys are shared out by the kernels from the lengths on the device (a table that
can hold many keys), and the same calls with equal splits per sequence (a narrow table), against
the fp64 decode oracle with the bounds of the decode tests: batches of unequal lengths whose sequences
end inside a workgroup's share, span several of them, or are empty; more sequences than a wave has
lanes; several tokens and heads packed into groups of 16 rows (with the last group partly filled);
K/V head counts that do not divide the CUs; every kernel width; the append written by the
workgroups that read the new keys, with a left pad past them and both rotary forms; a dense cache read
without a block table. Which path a call takes is asserted from the workspace it asks for
(test_shared_path). Replays of a captured shared call are in test_graph_gpu.py."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.helpers import to_np
from tests.test_decode_gpu import check, make_case, run_kernel, run_oracle

pytestmark = pytest.mark.gpu
RAGGED = [3000, 1, 0, 700, 64, 65, 2047]   # (7: divides no power of two)

# name, HD, NH, gqa, ctx(list per batch), window, rotary, append, leftpad, nq, softcap, alibi, page
CASES = [
    ("ragged", 128, 8, 4, RAGGED, -1, 0, False, 0, 1, 0.0, False, 16),
    ("ragged append rotary", 128, 8, 4, RAGGED, -1, 1, True, 0, 1, 0.0, False, 16),
    ("ragged mha 5 heads", 64, 5, 1, RAGGED, -1, 2, True, 0, 1, 0.0, False, 64),
    ("96 kv heads", 64, 96, 1, [500, 3, 200], -1, 0, True, 0, 1, 0.0, False, 16),
    ("300 kv heads", 64, 300, 1, [130, 3, 64], -1, 0, False, 0, 1, 0.0, False, 16),
    ("130 sequences", 64, 4, 4, [(37 * i) % 400 for i in range(130)], -1, 1, True, 0, 1, 0.0, False, 16),
    ("4 tokens x 4 heads", 128, 8, 4, RAGGED, -1, 1, True, 0, 4, 0.0, False, 16),
    ("5 tokens x 4 heads", 128, 8, 4, RAGGED, -1, 1, True, 0, 5, 0.0, False, 16),
    ("3 tokens x 8 heads no append", 128, 16, 8, RAGGED, -1, 0, False, 0, 3, 0.0, False, 16),
    ("21 tokens x 3 heads window", 128, 6, 3, [900, 40, 0], 50, 1, True, 0, 21, 0.0, False, 16),
    ("20 heads in a group", 128, 40, 20, [900, 40], -1, 0, True, 0, 2, 0.0, False, 16),
    ("window", 128, 8, 4, RAGGED, 100, 0, True, 0, 2, 0.0, False, 16),
    ("leftpad past the new keys", 128, 8, 4, [300, 5, 0], -1, 1, True, 40, 2, 0.0, False, 16),
    ("softcap", 128, 8, 4, RAGGED, -1, 1, True, 0, 3, 20.0, False, 16),
    ("alibi", 128, 8, 4, RAGGED, -1, 0, True, 0, 3, 0.0, True, 16),
    ("page 1", 128, 8, 4, [90, 1, 0, 130], -1, 1, True, 0, 2, 0.0, False, 1),
    ("page 8", 64, 8, 4, [90, 1, 0, 1300], -1, 1, True, 0, 2, 0.0, False, 8),
    ("D40", 40, 8, 4, RAGGED, -1, 1, True, 0, 2, 0.0, False, 16),
    ("D96", 96, 8, 4, RAGGED, -1, 1, True, 0, 2, 0.0, False, 16),
    ("D160 alibi", 160, 4, 2, RAGGED, -1, 0, True, 0, 2, 0.0, True, 16),
    ("D192", 192, 4, 2, RAGGED, -1, 2, True, 0, 2, 0.0, False, 16),
    ("D224 softcap", 224, 4, 2, RAGGED, -1, 1, True, 0, 2, 15.0, False, 16),
    ("D256", 256, 4, 2, RAGGED, -1, 1, True, 0, 2, 0.0, False, 32),
    ("D256 alibi", 256, 4, 2, RAGGED, -1, 0, False, 0, 2, 0.0, True, 32),
]


def widen(c, bytes_held=1 << 28):
    """The case with block-table columns (out-of-range entries, never read) up to a table that can
    hold `bytes_held` of keys and values."""
    nblk, page, Hk, D = c["kc"].shape
    B, nb = c["bt"].shape
    cols = -(-bytes_held // (B * page * Hk * D * 4))
    c["bt"] = np.concatenate([c["bt"], np.full((B, max(cols - nb, 0)), 10 ** 6, np.int32)], 1)
    return c


# (the rule also leaves four of CASES on equal splits under the wide table: batches of 3 and 2 that divide the
# parts, and pages under 16 rows; SHARED holds such heads and groups on the shared path)
@pytest.mark.parametrize("wide", [True, False], ids=["wide", "narrow"])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_stream_parity(case, dt, wide):
    print(f"[stream] {case[0]} {dt} {'wide' if wide else 'narrow'}", flush=True)
    c = make_case(case, dt)
    c = widen(c) if wide else c
    o, l, kc, vc = run_kernel(c, dt)
    o_ref, l_ref = run_oracle(c, dt)
    check(o, l, o_ref, l_ref, dt, case[0])
    if c["nk"] is not None:
        kcn, vcn, page = to_np(kc), to_np(vc), c["kc"].shape[1]
        for b, cx in enumerate(c["ctx"]):
            for t in range(c["q"].shape[1]):
                blk, row = c["bt"][b, (cx + t) // page], (cx + t) % page
                assert np.array_equal(vcn[blk, row], c["nv"][b, t])
                if not c["rotary"]:
                    assert np.array_equal(kcn[blk, row], c["nk"][b, t])


def test_stream_equals_fixed_splits():
    """The split count of the caller's choice takes the grid of fixed splits: same result to the
    rounding of the output (both paths round the same probabilities relative to maxima of their
    own: see test_decode_tiles_gpu.test_tiles_partial_rotary for the bound)."""
    c = widen(make_case(("fixed", 128, 8, 4, RAGGED, -1, 1, True, 0, 3, 0.0, False, 16), "bf16"))
    a, la, _, _ = run_kernel(c, "bf16")
    for n in (1, 3):
        b, lb, _, _ = run_kernel(c, "bf16", num_splits=n)
        assert orc.rel_rms(a, b) <= 2.0 ** -8
        fin = np.isfinite(la)
        assert np.array_equal(fin, np.isfinite(lb)) and np.abs(la[fin] - lb[fin]).max() <= 1e-4


@pytest.mark.parametrize("nq", [1, 3, 40])
def test_dense_cache_without_table(nq):
    """A dense cache read and appended to without a block table (the kernels form sequence b's page
    as b) against the same cache with the table spelt out, bit for bit; nq 40 runs on the tiles."""
    import torch

    from fable_attn import _lib
    L = _lib.load()
    B, H, Hk, D, cap = 5, 8, 2, 128, 1024
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    q, nk, nv, kc0, vc0 = rnd(B, nq, H, D), rnd(B, nq, Hk, D), rnd(B, nq, Hk, D), rnd(B, cap, Hk, D), rnd(B, cap, Hk, D)
    lens = torch.tensor([900, 0, 1, 64, 333], dtype=torch.int32, device="cuda")
    res = []
    for table in (None, torch.arange(B, dtype=torch.int32, device="cuda").view(B, 1)):
        kc, vc, out = kc0.clone(), vc0.clone(), torch.empty_like(q)
        p = _lib.FableDecParams()
        p.q, p.Kc, p.Vc, p.o, p.ctx_len = q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), lens.data_ptr()
        p.block_table = table.data_ptr() if table is not None else None
        p.batch, p.NH, p.gqa, p.HD, p.page, p.max_blocks, p.nq, p.window, p.scale = B, H, H // Hk, D, cap, 1, nq, -1, D ** -0.5
        n = L.fable_attn_dec_ws_bytes(p, _lib.FA_BF16, 1)
        ws = torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        _lib.check(L.fable_attn_dec_ws(p, _lib.FA_BF16, ws.data_ptr(), n, st, nk.data_ptr(), nv.data_ptr()), "dec")
        torch.cuda.synchronize()
        res.append((out, kc, vc))
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rotary", [False, True])
@pytest.mark.parametrize("paged", [True, False], ids=["paged", "dense"])
def test_appends_to_a_shared_cache_row(paged, rotary):
    """Tokens of one sequence laid out as batch rows of successive lengths (one block table, or one
    cache row by cache_batch_idx): each row sees the keys that the rows before it append in the same
    call, as the same tokens of one batch row do. Called twice, as a serving loop does."""
    import torch

    from fable_attn import flash_attn_with_kvcache
    n, H, Hk, D, L, cap, page = 8, 8, 2, 128, 1500, 4096, 16
    g = torch.Generator(device="cuda").manual_seed(2)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    q, k, v = rnd(1, n, H, D), rnd(1, n, Hk, D), rnd(1, n, Hk, D)
    kc0, vc0 = (rnd(cap // page, page, Hk, D) if paged else rnd(2, cap, Hk, D) for _ in range(2))
    table = torch.randperm(cap // page, generator=torch.Generator().manual_seed(3)).view(1, -1).int().cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    ang = torch.rand(cap, D // 2, generator=g, device="cuda") * 6.28
    opt = dict(rotary_cos=ang.cos(), rotary_sin=ang.sin()) if rotary else {}
    where = lambda b: dict(block_table=table.expand(b, -1).contiguous()) if paged else dict(cache_batch_idx=i32([1] * b))
    rows = lambda t: t.view(n, 1, *t.shape[2:]).contiguous()
    res = []
    for b, args in ((1, (q, k, v)), (n, tuple(rows(t) for t in (q, k, v)))):
        lens = i32([L] if b == 1 else [L + i for i in range(n)])
        for _ in range(2):
            kc, vc = kc0.clone(), vc0.clone()
            out = flash_attn_with_kvcache(args[0], kc, vc, args[1], args[2], cache_seqlens=lens, **where(b), **opt)
        res.append((out.reshape(n, H, D).float(), kc, vc))
    torch.cuda.synchronize()
    (a, ka, va), (b, kb, vb) = res
    assert torch.equal(ka, kb) and torch.equal(va, vb)
    # both round their probabilities (to running maxima of their own) and results to bf16, as in
    # test_decode_tiles_gpu.test_tiles_partial_rotary
    assert orc.rel_rms(a.cpu().numpy(), b.cpu().numpy()) <= 2.0 ** -8


def test_append_of_a_misaligned_new_token():
    """new_v needs no alignment at the C-ABI entry points of the decode kernel."""
    import torch

    from fable_attn import _lib
    L = _lib.load()
    B, H, Hk, D, cap = 1, 8, 2, 128, 256
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    q, nk, kc, vc = rnd(B, 1, H, D), rnd(B, 1, Hk, D), rnd(B, cap, Hk, D), rnd(B, cap, Hk, D)
    nv = rnd(B * Hk * D + 1)[1:].view(B, 1, Hk, D)
    lens, table = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([100], [[0]]))
    out = torch.empty_like(q)
    p = _lib.FableDecParams()
    p.q, p.Kc, p.Vc, p.o, p.ctx_len = q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), lens.data_ptr()
    p.block_table, p.nsplit = table.data_ptr(), 1
    p.batch, p.NH, p.gqa, p.HD, p.page, p.max_blocks, p.nq, p.window, p.scale = B, H, H // Hk, D, cap, 1, 1, -1, D ** -0.5
    _lib.check(L.fable_attn_dec(p, _lib.FA_BF16, torch.cuda.current_stream().cuda_stream, nk.data_ptr(), nv.data_ptr()), "dec")
    torch.cuda.synchronize()
    assert torch.equal(vc[0, 100], nv[0, 0]) and torch.equal(kc[0, 100], nk[0, 0])


def shared(batch, nq, NH, Hk, D, page, max_blocks, append):
    """Whether such a call is shared out on the device: its workspace is then two ints per sequence and two
    records of 16 rows for each workgroup of a grid of one per part (two if there are more sequences than
    parts), not a partial per row and split."""
    from fable_attn import _lib
    L = _lib.load()
    p = _lib.FableDecParams()
    p.batch, p.NH, p.gqa, p.HD, p.page, p.max_blocks, p.nq, p.window, p.scale = batch, NH, NH // Hk, D, page, max_blocks, nq, -1, 1.0
    X = Hk * -(-nq * (NH // Hk) // 16)
    parts = 256 // X
    if parts * X < 224:
        parts = -(-512 // X)
    parts = max(min(parts, batch * (-(-max_blocks * page // 64) + 1)), 1)
    wgs = parts if batch <= parts else 2 * parts
    want = ((2 * batch + 63) // 64 * 64 + wgs * 2 * X * 16 * (D + 2)) * 4
    return L.fable_attn_dec_ws_bytes(p, _lib.FA_BF16, int(append)) == want


# name, HD, NH, gqa, ctx(list per batch), window, rotary, append, leftpad, nq, softcap, alibi, page
SHARED = [
    ("96 kv heads", 64, 96, 1, [500, 3, 200, 0, 77], -1, 0, True, 0, 1, 0.0, False, 16),
    ("20 heads in a group", 128, 40, 20, [900, 40, 0, 300, 1000], -1, 0, True, 0, 2, 0.0, False, 16),
    ("17 heads in a group, one token", 128, 34, 17, [900, 40, 0, 300, 1000], -1, 1, True, 0, 1, 0.0, False, 16),
    ("short, many parts", 128, 2, 2, [1, 63, 64, 65, 0, 300, 128], -1, 0, False, 0, 1, 0.0, False, 16),
    ("alike, 24 sequences", 128, 8, 1, [500] * 24, -1, 0, False, 0, 1, 0.0, False, 16),
]


@pytest.mark.parametrize("case", SHARED, ids=[c[0] for c in SHARED])
def test_shared_path(case):
    name, HD, NH, gqa, ctx, _, _, append, _, nq, _, _, page = case
    c = widen(make_case(case, "bf16"))
    assert shared(len(ctx), nq, NH, NH // gqa, HD, page, c["bt"].shape[1], append)
    o, l, _, _ = run_kernel(c, "bf16")
    o_ref, l_ref = run_oracle(c, "bf16")
    check(o, l, o_ref, l_ref, "bf16", "shared " + name)


def test_append_by_several_row_groups():
    """One token of 20 heads per K/V head, a single sequence: two row groups write the one new key."""
    c = make_case(("20 heads, one token", 128, 40, 20, [700], -1, 1, True, 0, 1, 0.0, False, 16), "bf16")
    o, l, _, vc = run_kernel(c, "bf16")
    o_ref, l_ref = run_oracle(c, "bf16")
    check(o, l, o_ref, l_ref, "bf16", "append by two row groups")
    assert np.array_equal(to_np(vc)[c["bt"][0, 700 // 16], 700 % 16], c["nv"][0, 0])


@pytest.mark.parametrize("gqa", [4, 20])
def test_shared_dense_cache_without_table(gqa):
    """A dense cache large enough to be shared out, read and appended to without a block table, against the
    table spelt out (whose append runs ahead in a kernel of its own), bit for bit."""
    import torch

    from fable_attn import _lib
    L = _lib.load()
    B, Hk, D, cap = 5, 2, 128, 65536
    H = gqa * Hk
    assert shared(B, 1, H, Hk, D, cap, 1, True)
    g = torch.Generator(device="cuda").manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda", dtype=torch.bfloat16)
    q, nk, nv, kc0, vc0 = rnd(B, 1, H, D), rnd(B, 1, Hk, D), rnd(B, 1, Hk, D), rnd(B, cap, Hk, D), rnd(B, cap, Hk, D)
    lens = torch.tensor([9000, 0, 1, 640, 65535], dtype=torch.int32, device="cuda")
    res = []
    for table in (None, torch.arange(B, dtype=torch.int32, device="cuda").view(B, 1)):
        kc, vc, out = kc0.clone(), vc0.clone(), torch.empty_like(q)
        p = _lib.FableDecParams()
        p.q, p.Kc, p.Vc, p.o, p.ctx_len = q.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), lens.data_ptr()
        p.block_table = table.data_ptr() if table is not None else None
        p.batch, p.NH, p.gqa, p.HD, p.page, p.max_blocks, p.nq, p.window, p.scale = B, H, gqa, D, cap, 1, 1, -1, D ** -0.5
        n = L.fable_attn_dec_ws_bytes(p, _lib.FA_BF16, 1)
        ws = torch.empty(n, dtype=torch.uint8, device="cuda")
        st = torch.cuda.current_stream().cuda_stream
        _lib.check(L.fable_attn_dec_ws(p, _lib.FA_BF16, ws.data_ptr(), n, st, nk.data_ptr(), nv.data_ptr()), "dec")
        torch.cuda.synchronize()
        res.append((out, kc, vc))
    for a, b in zip(*res):
        assert torch.equal(a, b)
    z = torch.arange(B, device="cuda")
    assert torch.equal(res[0][1][z, lens.long()], nk[:, 0]) and torch.equal(res[0][2][z, lens.long()], nv[:, 0])
