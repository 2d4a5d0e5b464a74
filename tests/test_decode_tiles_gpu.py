"""Many new tokens per call on the paged tile kernel (tokens x heads of a K/V head's group are the
rows of a query tile), through the C-ABI binding, against the fp64 decode oracle with the bounds of
the decode tests. The cases cover both sides of the row count at which the path starts, row counts
around the tiles of 128 and 256, key splits with shares that hold no key, contexts of 0 and 1, pages
of 16 to 256 rows, every kernel width with zero columns, and each option (window, left pad,
softcap, alibi, both rotary forms, a partial rotary width) with and without appending."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.helpers import to_np
from tests.test_decode_gpu import check, make_case, run_kernel, run_oracle

pytestmark = pytest.mark.gpu

# (make_case gives 16 rotary rows past the last key: without an append the new tokens, which are
# rotated at the positions after it, must be no more)
# name, HD, NH, gqa, ctx(list per batch), window, rotary, append, leftpad, nq, softcap, alibi, page
CASES = [
    ("63 rows", 128, 8, 1, [300, 41], -1, 0, True, 0, 63, 0.0, False, 16),
    ("64 rows", 128, 8, 4, [300, 41], -1, 0, True, 0, 16, 0.0, False, 16),
    ("odd rows rotary", 128, 6, 3, [1000, 0, 1], -1, 1, True, 0, 43, 0.0, False, 16),
    ("128 rows rotary", 128, 8, 8, [700], -1, 1, True, 0, 16, 0.0, False, 64),
    ("129 rows rotary interleaved", 128, 3, 3, [700, 65], -1, 2, True, 0, 43, 0.0, False, 256),
    ("257 rows", 128, 1, 1, [500, 64], -1, 0, True, 0, 257, 0.0, False, 32),
    ("no append", 128, 8, 4, [900, 0, 17], -1, 0, False, 0, 40, 0.0, False, 16),
    ("no append rotary", 128, 8, 8, [900, 33], -1, 1, False, 0, 12, 0.0, False, 16),
    ("window", 128, 4, 2, [1200, 90], 100, 0, True, 0, 70, 0.0, False, 16),
    ("window no append rotary", 128, 8, 8, [1200, 90], 100, 1, False, 0, 12, 0.0, False, 16),
    ("leftpad", 128, 4, 2, [600, 80], -1, 0, True, 37, 70, 0.0, False, 16),
    ("leftpad past the keys", 128, 4, 2, [600, 20], -1, 0, False, 37, 70, 0.0, False, 16),
    ("softcap", 128, 4, 2, [400, 80], -1, 1, True, 0, 70, 20.0, False, 16),
    ("alibi", 128, 4, 2, [400, 80], -1, 0, True, 0, 70, 0.0, True, 16),
    ("alibi no append", 128, 4, 2, [400, 80], -1, 0, False, 0, 70, 0.0, True, 16),
    ("D64 rotary", 64, 8, 4, [777, 5], -1, 1, True, 0, 33, 0.0, False, 16),
    ("D64 window softcap", 64, 8, 4, [777, 5], 200, 0, True, 0, 33, 25.0, False, 64),
    ("D40 rotary", 40, 4, 2, [300], -1, 1, True, 0, 50, 0.0, False, 16),
    ("D96 rotary", 96, 4, 2, [300, 64], -1, 2, True, 0, 50, 0.0, False, 16),
    ("D192 alibi", 192, 4, 2, [300, 64], -1, 0, True, 0, 50, 0.0, True, 32),
    ("D256 rotary", 256, 4, 4, [520, 64], -1, 1, True, 0, 40, 0.0, False, 16),
    ("D256", 256, 4, 4, [520, 64], -1, 0, True, 0, 40, 0.0, False, 16),
    ("D256 window softcap", 256, 4, 4, [520, 64], 128, 0, True, 5, 40, 30.0, False, 16),
    ("split long", 128, 8, 8, [6000], -1, 1, True, 0, 17, 0.0, False, 16),
    ("split ragged", 64, 8, 8, [5000, 3, 900], -1, 0, True, 0, 9, 0.0, False, 16),
]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("case", CASES, ids=[c[0] for c in CASES])
def test_tiles_parity(case, dt):
    print(f"[tiles] {case[0]} {dt}", flush=True)
    c = make_case(case, dt)
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


def test_tiles_partial_rotary():
    """A rotary width of 48 in a head dim of 128: the columns past it are copied as they are."""
    import torch

    from fable_attn import _C
    c = make_case(("partial", 128, 4, 2, [300, 31], -1, 1, True, 0, 40, 0.0, False, 16), "bf16")
    rd = 48
    c["cos"], c["sin"] = (np.ascontiguousarray(t[:, :rd // 2]) for t in (c["cos"], c["sin"]))
    dev = lambda a: torch.from_numpy(a).cuda().bfloat16()
    f32 = lambda a: torch.from_numpy(a).cuda()
    args = lambda q, k, v, kc, vc: (q, kc, vc, f32(c["bt"]), f32(c["ctx"]), k, v, f32(c["cos"]),
                                    f32(c["sin"]), False, c["scale"], -1, 0, None, True, 0.0, None, rd, None)
    outs = []
    for chunk in (40, 8):     # one call on the tile kernel, and in steps below its row count
        kc, vc = dev(c["kc"]), dev(c["vc"])
        ctx0, parts = c["ctx"].copy(), []
        for t in range(0, 40, chunk):
            c["ctx"] = ctx0 + t
            sl = [dev(np.ascontiguousarray(c[n][:, t:t + chunk])) for n in ("q", "nk", "nv")]
            parts.append(_C.dec(*args(*sl, kc, vc))[0])
        c["ctx"] = ctx0
        outs.append((torch.cat(parts, 1).float(), kc.float(), vc.float()))
    torch.cuda.synchronize()
    for a, b in zip(*outs):
        # each path rounds its probabilities (relative to running maxima of its own) and its result
        # to bf16: four independent roundings of at most 2^-9, rms 2^-9 / sqrt(3) each, so
        # 2.3e-3 is expected; the bound is 2^-8
        assert orc.rel_rms(a.cpu().numpy(), b.cpu().numpy()) <= 2.0 ** -8


def hide(c):
    """The case with NaN in every K and V row below the first key a token sees, and with the table entries
    of whole pages below it naming one page of NaN (a read there shows as a wrong value)."""
    kc, vc = (np.concatenate([c[n], np.full_like(c[n][:1], np.nan)]) for n in ("kc", "vc"))
    bt, page = c["bt"].copy(), c["kc"].shape[1]
    for b, cx in enumerate(c["ctx"]):
        lo = max(c["lp"][b] if c["lp"] is not None else 0, cx - c["window"] + 1 if c["window"] >= 0 else 0)
        lo = min(lo, cx)             # (the new keys are written, whatever the pad)
        for x in (kc, vc):
            if lo // page < bt.shape[1]:
                x[bt[b, lo // page], :lo % page] = np.nan
        bt[b, :lo // page] = len(kc) - 1
    return dict(c, kc=kc, vc=vc, bt=bt)


# name, HD, NH, gqa, ctx(list per batch), window, rotary, append, leftpad, nq, softcap, alibi, page
HIDDEN = [
    ("window", 128, 4, 2, [1200, 90, 333], 100, 0, True, 0, 70, 0.0, False, 16),
    ("window no append rotary", 128, 8, 8, [1200, 90], 101, 1, False, 0, 12, 0.0, False, 16),
    ("window split", 128, 8, 8, [5003], 2000, 0, True, 0, 12, 0.0, False, 16),
    ("leftpad", 128, 4, 2, [600, 80], -1, 0, True, 37, 70, 0.0, False, 16),
    ("leftpad one page", 128, 4, 2, [600, 80], -1, 1, True, 37, 70, 0.0, False, 1024),
    ("leftpad past the keys", 128, 4, 2, [600, 20], -1, 0, False, 63, 70, 0.0, False, 16),
    ("D64 window", 64, 8, 4, [777, 5], 201, 0, True, 0, 33, 25.0, False, 64),
    ("D40 leftpad", 40, 4, 2, [300], -1, 1, True, 49, 50, 0.0, False, 16),
    ("D256 window leftpad", 256, 4, 4, [520, 64], 128, 0, True, 33, 40, 0.0, False, 16),
    ("D256 alibi leftpad", 256, 4, 4, [520, 64], -1, 0, True, 31, 40, 0.0, True, 32),
    ("below the tiles", 128, 4, 2, [600, 80], 99, 1, True, 37, 5, 0.0, False, 16),
]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("case", HIDDEN, ids=[c[0] for c in HIDDEN])
def test_nothing_below_the_first_visible_key_is_read(case, dt):
    print(f"[tiles] hidden {case[0]} {dt}", flush=True)
    c = make_case(case, dt)
    o, l, _, _ = run_kernel(hide(c), dt)
    o_ref, l_ref = run_oracle(c, dt)
    check(o, l, o_ref, l_ref, dt, "hidden " + case[0])


@pytest.mark.parametrize("append", [False, True])
@pytest.mark.parametrize("nq", [3, 31, 32, 70])
def test_window_of_no_keys(nq, append):
    """window 0 hides every key (a token sees keys from its position + 1 on) on both sides of the row count
    at which the tile kernel starts (64: 32 tokens of 2 heads)."""
    c = make_case(("window 0", 128, 4, 2, [300, 0], 0, 0, append, 0, nq, 0.0, False, 16), "bf16")
    o, l, _, _ = run_kernel(c, "bf16")
    assert not o.any() and np.isneginf(l).all()


@pytest.mark.parametrize("splits", [1, 2, 5, 32, 100])
def test_split_counts(splits):
    c = make_case(("splits", 128, 16, 8, [3000, 70, 0], -1, 1, True, 0, 17, 0.0, False, 16), "f16")   # (54 groups of 16 rows)
    o, l, _, _ = run_kernel(c, "f16", num_splits=splits)
    o_ref, l_ref = run_oracle(c, "f16")
    check(o, l, o_ref, l_ref, "f16", f"tiles in {splits} splits")


@pytest.mark.parametrize("softcap", [0.0, 30.0])
@pytest.mark.parametrize("dt", ["f16", "bf16"])
def test_largest_probability_is_not_rounded(dt, softcap):
    """One key of logit b > 0 behind 70 keys of logit 0, values 1 and 0: the result is the probability of the
    one, whose numerator is exactly 1 in 16 bits when the row's own maximum is its exponent's base. Then
    only the result is rounded, by half a unit in its last place (of 8 significant bits in bf16, 11 in
    fp16: at most 2^-8 and 2^-11 of the value; 1e-5 for the fp32 sums); against an older maximum the
    numerator e^b is rounded as well."""
    import torch

    from fable_attn import _C
    B, nq, D, page, n = 40, 64, 64, 128, 70
    t = {"f16": torch.float16, "bf16": torch.bfloat16}[dt]
    b = torch.arange(B, device="cuda") / 64 + 3.0            # exact in both types
    q, kc, vc = torch.zeros(B, nq, 1, D, device="cuda", dtype=t), *(torch.zeros(B, page, 1, D, device="cuda", dtype=t) for _ in range(2))
    q[..., 0] = 1
    kc[:, n, 0, 0], vc[:, n] = b.to(t), 1
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out, _ = _C.dec(q, kc, vc, torch.arange(B, dtype=torch.int32, device="cuda").view(B, 1), i32([n + 1] * B), None, None, None,
                    None, False, 1.0, -1, 0, None, False, softcap)
    x = b.double() if not softcap else softcap * torch.tanh(b.double() / softcap)
    want = (x.exp() / (x.exp() + n)).view(B, 1, 1, 1)
    assert ((out.double() - want).abs() / want).max() <= {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}[dt] + 1e-5


# Calls of few sequences and K/V heads stay on the decode kernel (up to 16 groups of 16 rows: some of CASES and
# HIDDEN): the same shapes with more K/V heads, on the tiles.
# name, HD, NH, gqa, ctx(list per batch), window, rotary, append, leftpad, nq, softcap, alibi, page
MORE_HEADS = [
    ("128 rows rotary", 128, 24, 8, [700], -1, 1, True, 0, 16, 0.0, False, 64),
    ("no append rotary", 128, 24, 8, [900, 33], -1, 1, False, 0, 12, 0.0, False, 16),
    ("window no append rotary", 128, 24, 8, [1200, 90], 100, 1, False, 0, 12, 0.0, False, 16),
    ("window split", 128, 24, 8, [5003], 2000, 0, True, 0, 12, 0.0, False, 16),
    ("split long", 128, 24, 8, [6000], -1, 1, True, 0, 17, 0.0, False, 16),
    ("split ragged", 64, 16, 8, [5000, 3, 900], -1, 0, True, 0, 9, 0.0, False, 16),
    ("64 heads, one token", 128, 64, 64, [3000, 0, 7, 900, 64], -1, 1, True, 0, 1, 0.0, False, 16),
    ("16 groups: decode kernel", 128, 64, 64, [3000, 0, 7, 900], -1, 1, True, 0, 1, 0.0, False, 16),
]


@pytest.mark.parametrize("dt", ["f16", "bf16"])
@pytest.mark.parametrize("case", MORE_HEADS, ids=[c[0] for c in MORE_HEADS])
def test_tiles_parity_more_heads(case, dt):
    test_tiles_parity(case, dt)


@pytest.mark.parametrize("case", MORE_HEADS[2:4], ids=[c[0] for c in MORE_HEADS[2:4]])
def test_hidden_more_heads(case):
    test_nothing_below_the_first_visible_key_is_read(case, "bf16")
