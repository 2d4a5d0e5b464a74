"""The attention calls whose speed and accuracy are measured, through the public API.

Four kinds of call, as a serving or a training program makes them:

  kvcache  flash_attn_with_kvcache over a paged or dense K/V cache: token-by-token decode,
           several tokens at once (drafted tokens to verify), a chunk of a prompt; with or
           without appending the new keys (rotary applied) to the cache;
  paged    flash_attn_varlen_func over packed queries and a paged K/V cache (block_table): the
           prompt phase of a batch of requests, some of whose keys are cached already;
  dense    flash_attn_func / flash_attn_qkvpacked_func on (batch, seqlen, heads, dim);
  varlen   flash_attn_varlen_func on packed sequences.

`dense` and `varlen` run forward alone (inference) or forward and backward (`grad`, a training
step's attention layer: the output and the gradients of q, k and v come back).
Inputs are N(0, 1), as this repository's benchmark and tests draw them.
"""
import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(ROOT, "flash-attention-rdna2_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from fable_attn import (  # noqa: E402
    flash_attn_func,
    flash_attn_qkvpacked_func,
    flash_attn_varlen_func,
    flash_attn_with_kvcache,
)

_DT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _case(name, kind, dtype, **kw):
    """A case with every field of its kind present."""
    c = {"kind": kind, "dtype": dtype, "causal": True, "window": -1, "softcap": 0.0,
         "alibi": False, "dropout": 0.0, "grad": False}
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # One request being answered token by token: the new key goes into a dense cache of 4096
        # rows with rotary, then one query token reads some 2000 cached keys. Latency and the
        # count of launches are what a user feels here.
        _case("decode_step", "kvcache", "bf16", batch=1, nq=1, lo=2000, hi=2000, cap=4096, page=0,
              hq=32, hk=8, d=128, append=True),
        # A serving batch in flight: 48 requests with contexts of very different lengths in a
        # cache of 16-row pages, one new token each (the new keys were written before).
        _case("decode_ragged", "kvcache", "bf16", batch=48, nq=1, lo=64, hi=8192, cap=8192, page=16,
              hq=64, hk=8, d=128, append=False),
        # Long contexts: the benchmark's paged decode (HBM bound).
        _case("decode_long", "kvcache", "fp16", batch=16, nq=1, lo=32768, hi=32768, cap=32768, page=256,
              hq=32, hk=8, d=128, append=False),
        # A prompt taken in chunks: 512 new tokens of two requests are appended to a paged cache
        # (rotary) that holds up to 7000 earlier keys, and attend to all of them.
        _case("prefill_chunk", "kvcache", "bf16", batch=2, nq=512, lo=1000, hi=7000, cap=8192, page=256,
              hq=32, hk=8, d=128, append=True),
        # The prompt phase of a batch of requests over a paged cache, part of whose prefix is
        # shared and cached already.
        _case("prefill_paged", "paged", "bf16", batch=8, qlo=16, qhi=2048, clo=0, chi=4096, page=16,
              hq=32, hk=8, d=128),
        # A small layer: the benchmark's C1 (64 query tiles for 256 CUs).
        _case("fwd_small", "dense", "fp16", batch=1, sq=1024, sk=1024, hq=8, hk=8, d=64, causal=False,
              packed=False),
        # A long prompt in one call: the benchmark's headline (matrix-core bound).
        _case("fwd_long", "dense", "fp16", batch=1, sq=16384, sk=16384, hq=32, hk=32, d=128, packed=False),
        # Sliding-window layers with capped logits on packed prompts: the benchmark's varlen case.
        _case("fwd_window", "varlen", "bf16", batch=8, lo=512, hi=8192, hq=16, hk=16, d=256, window=512,
              softcap=30.0),
        # A causal training step: the benchmark's backward shape, forward included.
        _case("train_causal", "dense", "bf16", batch=2, sq=4096, sk=4096, hq=32, hk=32, d=128, packed=False,
              grad=True),
        # Fine-tuning on packed samples of uneven lengths, grouped heads.
        _case("train_packed", "varlen", "bf16", batch=24, lo=64, hi=2048, hq=32, hk=8, d=128, grad=True),
        # A bidirectional encoder's layer: packed projections, dropout on the probabilities.
        _case("train_encoder", "dense", "fp16", batch=32, sq=509, sk=509, hq=16, hk=16, d=64, causal=False,
              dropout=0.1, packed=True, grad=True),
        # A small model trained or checked in single precision, with position slopes.
        _case("train_fp32", "dense", "fp32", batch=2, sq=1000, sk=1000, hq=12, hk=12, d=64, packed=False,
              alibi=True, grad=True),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges above: the kinds in the proportion in which they are listed,
    sizes over the logarithm of their range."""
    kind = rng.choice(["kvcache"] * 4 + ["paged"] + ["infer"] * 3 + ["train"] * 4)
    hk = rng.choice([1, 2, 4, 8])
    hq = hk * rng.choice([1, 4, 8])
    if kind == "kvcache":
        nq = rng.choice([1, 1, rng.randint(2, 16), _log_int(rng, 17, 1024)])
        hi = _log_int(rng, 128, 32768)
        d = rng.choice([64, 96, 128, 128, 256])
        # (at most 2 GiB of keys and values, and half the operations of the longest prompt)
        nq = min(nq, max(1, int(2.5e11 / (hi * hq * d))))
        batch = _log_int(rng, 1, max(1, min(64, (1 << 29) // (hi * hk * d), int(2.5e11 / (nq * hi * hq * d)))))
        cap = 1 << max(8, (hi + nq - 1).bit_length())
        page = rng.choice([0, 16, 16, 64, 256])
        pool = 2 * 2 * batch * cap * hk * d
        return _case(None, "kvcache", rng.choice(["bf16", "fp16"]), batch=batch, nq=nq,
                     lo=rng.choice([hi, max(1, hi // 16)]), hi=hi, cap=cap, page=page, hq=hq, hk=hk, d=d,
                     append=pool <= (1 << 27) and rng.random() < 0.7)
    if kind == "paged":
        d = rng.choice([64, 128, 128, 256])
        qhi, chi = _log_int(rng, 64, 4096), rng.choice([0, _log_int(rng, 64, 8192)])
        batch = _log_int(rng, 1, max(1, min(16, int(2.5e11 / (qhi * (qhi + chi) * hq * d)))))
        return _case(None, "paged", rng.choice(["bf16", "fp16"]), batch=batch, qlo=rng.randint(1, 64), qhi=qhi,
                     clo=0, chi=chi, page=rng.choice([16, 32, 64, 256]), hq=hq, hk=hk, d=d)
    grad = kind == "train"
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"])
    d = rng.choice([64, 64, 80, 96, 128, 128, 128, 192, 256])
    seq = _log_int(rng, 100, 2000 if dtype == "fp32" else 8192)
    # (at most about the operations of the largest listed training step or prompt)
    most = (1.5e8 if dtype == "fp32" else 6e8 if grad else 2.5e9) * 128 / (d * hq)
    seq = min(seq, int(most ** 0.5))
    batch = _log_int(rng, 1, max(1, min(64, int(most / (float(seq) * seq)))))
    opt = rng.choice(["", "", "", "", "window", "softcap", "alibi", "dropout"])
    kw = {"window": _log_int(rng, 64, 4096) if opt == "window" else -1,
          "softcap": 30.0 if opt == "softcap" else 0.0, "alibi": opt == "alibi",
          "dropout": 0.1 if opt == "dropout" and grad else 0.0}
    kw["causal"] = opt == "window" or rng.random() < 0.7
    if rng.random() < 0.4:
        return _case(None, "varlen", dtype, batch=batch + 1, lo=rng.randint(1, max(1, seq // 8)), hi=seq,
                     hq=hq, hk=hk, d=d, grad=grad, **kw)
    packed = hq == hk and rng.random() < 0.5
    sk = seq if packed or grad or rng.random() < 0.7 else seq + rng.randint(1, seq)
    return _case(None, "dense", dtype, batch=batch, sq=seq, sk=sk, hq=hq, hk=hk, d=d, packed=packed,
                 grad=grad, **kw)


# ----------------------------------------------------------------------------- sizes of a case
def _spread(seed, n, lo, hi):
    """n lengths of [lo, hi], even over their range; the longest is hi."""
    r = random.Random(seed)
    v = [r.randint(lo, hi) for _ in range(n)]
    v[r.randrange(n)] = hi
    return v


def _lengths(case, seed):
    """(query lengths, key lengths) of the sequences of a case. The lengths of a batch are part
    of the case, drawn once from its sizes, so that every seed has the same work."""
    del seed
    kind = case["kind"]
    if kind == "kvcache":
        ctx = _spread(7, case["batch"], case["lo"], case["hi"])
        return [case["nq"]] * case["batch"], [c + (case["nq"] if case["append"] else 0) for c in ctx]
    if kind == "paged":
        q = _spread(11, case["batch"], min(case["qlo"], case["qhi"]), case["qhi"])
        c = _spread(13, case["batch"], case["clo"], case["chi"])
        return q, [a + b for a, b in zip(q, c)]
    if kind == "varlen":
        n = _spread(17, case["batch"], case["lo"], case["hi"])
        return n, n
    return [case["sq"]] * case["batch"], [case["sk"]] * case["batch"]


def _pairs(case, sq, sk):
    """Visible (query, key) pairs of one head of one sequence."""
    if case["kind"] == "kvcache":
        return sq * sk - (sq * (sq - 1) // 2 if case["append"] else 0)
    if not case["causal"]:
        return sq * sk
    n = 0
    left = case["window"] if case["window"] >= 0 else sk + sq
    for i in range(sq):
        hi = i + sk - sq
        n += max(0, min(hi, sk - 1) - max(0, hi - left) + 1)
    return n


def work(case):
    """Operations: two products per visible pair forward (4 d), five backward (10 d). Bytes: each
    input read once and each output written once."""
    sqs, sks = _lengths(case, 0)
    el = 4 if case["dtype"] == "fp32" else 2
    hq, hk, d = case["hq"], case["hk"], case["d"]
    flops = sum(4 * d * hq * _pairs(case, a, b) for a, b in zip(sqs, sks))
    nq, nk = sum(sqs) * hq * d * el, sum(sks) * hk * d * el
    nbytes = 2 * nq + 2 * nk
    if case["kind"] == "kvcache" and case["append"]:
        nbytes += 2 * sum(sqs) * hk * d * el       # the new keys and values are written to the cache
    if case["grad"]:
        flops = flops * 7 // 2
        nbytes += 2 * nq + 2 * nk                  # dout in; dq, dk, dv out
    return {"bytes": nbytes, "flops": flops}


# ----------------------------------------------------------------------------- inputs
def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda", dtype=dtype)


def _cu(lens):
    return torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device="cuda")


def _table(seed, batch, blocks):
    """Block table of `batch` sequences of `blocks` pages each over a shuffled pool."""
    perm = torch.randperm(batch * blocks, generator=torch.Generator().manual_seed(seed))
    return perm.view(batch, blocks).to(torch.int32).cuda()


def prepare(case, seed):
    """Inputs of one call, on the GPU; of the caches, tables and lengths, what a serving program
    keeps between calls."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DT[case["dtype"]]
    hq, hk, d = case["hq"], case["hk"], case["d"]
    sqs, sks = _lengths(case, seed)
    s = {"case": case, "seed": seed}
    if case["alibi"]:
        s["alibi"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / hq) for h in range(hq)], device="cuda")
    if case["kind"] == "kvcache":
        b, nq, cap, page = case["batch"], case["nq"], case["cap"], case["page"]
        s["q"] = _randn(gen, (b, nq, hq, d), dt)
        rows = (b * cap // page, page) if page else (b, cap)
        s["kc"], s["vc"] = (_randn(gen, rows + (hk, d), dt) for _ in range(2))
        s["table"] = _table(seed, b, cap // page) if page else None
        new = nq if case["append"] else 0
        s["lens"] = torch.tensor([n - new for n in sks], dtype=torch.int32, device="cuda")
        if new:
            s["k"], s["v"] = (_randn(gen, (b, nq, hk, d), dt) for _ in range(2))
            pos = torch.arange(cap, device="cuda", dtype=torch.float32)[:, None]
            freq = 10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float32) / d)
            s["cos"], s["sin"] = torch.cos(pos * freq), torch.sin(pos * freq)
    elif case["kind"] == "paged":
        page = case["page"]
        blocks = -(-max(sks) // page)
        b = case["batch"]
        s["q"] = _randn(gen, (sum(sqs), hq, d), dt)
        s["kc"], s["vc"] = (_randn(gen, (b * blocks, page, hk, d), dt) for _ in range(2))
        s["table"] = _table(seed, b, blocks)
        s["cu_q"], s["cu_k"], s["mq"], s["mk"] = _cu(sqs), _cu(sks), max(sqs), max(sks)
    else:
        if case["kind"] == "dense":
            qs, ks = (case["batch"], case["sq"]), (case["batch"], case["sk"])
        else:
            qs, ks = (sum(sqs),), (sum(sks),)
            s["cu_q"] = s["cu_k"] = _cu(sqs)
            s["mq"] = s["mk"] = max(sqs)
        if case.get("packed"):
            s["qkv"] = _randn(gen, qs + (3, hq, d), dt)
            s["leaf"] = (s["qkv"],)
        else:
            s["q"] = _randn(gen, qs + (hq, d), dt)
            s["k"], s["v"] = (_randn(gen, ks + (hk, d), dt) for _ in range(2))
            s["leaf"] = (s["q"], s["k"], s["v"])
        if case["grad"]:
            s["dout"] = _randn(gen, qs + (hq, d), dt)
            for t in s["leaf"]:
                t.requires_grad_(True)
    return s


# ----------------------------------------------------------------------------- one pass
def run(state):
    """One call of the public API (with `grad`, forward and backward)."""
    s, case = state, state["case"]
    if case["kind"] == "kvcache":
        if not case["append"]:
            return flash_attn_with_kvcache(s["q"], s["kc"], s["vc"], cache_seqlens=s["lens"],
                                           block_table=s["table"], causal=True)
        out = flash_attn_with_kvcache(s["q"], s["kc"], s["vc"], k=s["k"], v=s["v"], rotary_cos=s["cos"],
                                      rotary_sin=s["sin"], cache_seqlens=s["lens"],
                                      block_table=s["table"], causal=True, rotary_interleaved=False)
        return {"out": out, "k_cache": s["kc"], "v_cache": s["vc"]}
    if case["kind"] == "paged":
        return flash_attn_varlen_func(s["q"], s["kc"], s["vc"], s["cu_q"], s["cu_k"], s["mq"], s["mk"],
                                      causal=True, block_table=s["table"])
    if case["dropout"]:
        random.seed(s["seed"])        # the dropout stream of a step is drawn from Python's generator
    window = (case["window"], 0) if case["window"] >= 0 else (-1, -1)
    kw = dict(causal=case["causal"], window_size=window, softcap=case["softcap"])
    if case["dropout"]:
        kw["dropout_p"] = case["dropout"]
    if case["alibi"]:
        kw["alibi_slopes"] = s["alibi"]
    if case["kind"] == "varlen":
        out = flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], s["mq"], s["mk"], **kw)
    elif case["packed"]:
        out = flash_attn_qkvpacked_func(s["qkv"], **kw)
    else:
        out = flash_attn_func(s["q"], s["k"], s["v"], **kw)
    if not case["grad"]:
        return out
    return (out.detach(),) + torch.autograd.grad(out, s["leaf"], s["dout"])


# ----------------------------------------------------------------------------- the same in 64 bits
def _philox_keep(seed, h, sq, sk, p):
    """Keep mask (sq, sk) of head h: word 0 of Philox4x32-10 (Salmon et al., SC 2011) on the
    counter (h*sq + i)*sk + j under the key `seed`, kept where its top 24 bits are at least p."""
    m32 = 0xFFFFFFFF
    idx = torch.arange(sq * sk, device="cuda", dtype=torch.int64) + h * sq * sk
    c = [idx & m32, idx >> 32, torch.zeros_like(idx), torch.zeros_like(idx)]
    k0, k1 = seed & m32, seed >> 32

    def mul(a, x):               # (high, low) 32 bits of a * x without passing 63 bits
        lo, hi = a * (x & 0xFFFF), a * (x >> 16)
        t = hi + (lo >> 16)
        return t >> 16, ((t & 0xFFFF) << 16) | (lo & 0xFFFF)

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & m32, (k1 + 0xBB67AE85) & m32
    u = (c[0] >> 8).to(torch.float32) * (1.0 / 16777216.0)
    return (u >= torch.tensor(p, dtype=torch.float32, device="cuda")).view(sq, sk)


def _attend(case, q, k, v, h, delta, slope=None, dout=None, drop=None):
    """Attention of one head of one sequence in float64 (q (sq, d), k and v (sk, d)); row i sees
    the keys up to i + delta where it is causal. With dout also dq, dk, dv."""
    sq, sk, scale = q.shape[0], k.shape[0], q.shape[1] ** -0.5
    s = (q @ k.t()).mul_(scale)
    cap = case["softcap"]
    if cap:
        s = s.div_(cap).tanh_().mul_(cap)
    t = s.clone() if cap and dout is not None else None
    i = torch.arange(sq, device="cuda")[:, None]
    j = torch.arange(sk, device="cuda")[None, :]
    if slope is not None:
        s += slope.double() * (j - i).double()
    if case["causal"] and delta is not None:
        s.masked_fill_(j > i + delta, -math.inf)
        if case["window"] >= 0:
            s.masked_fill_(j < i + delta - case["window"], -math.inf)
    p = s.sub_(s.amax(1, keepdim=True).clamp_min_(-1e300)).exp_()
    p.div_(p.sum(1, keepdim=True).clamp_min_(1e-300))
    z = None
    if drop is not None:
        z = _philox_keep(drop, h, sq, sk, case["dropout"]).double().div_(1.0 - case["dropout"])
    pz = p if z is None else p * z
    out = pz @ v
    if dout is None:
        return out
    dv = pz.t() @ dout
    dp = dout @ v.t()
    if z is not None:
        dp.mul_(z)
    ds = dp.sub_((dp * p).sum(1, keepdim=True)).mul_(p)
    if cap:
        ds.mul_(1.0 - (t / cap) ** 2)
    return out, (ds @ k).mul_(scale), (ds.t() @ q).mul_(scale), dv


def _rotate(x, cos, sin, pos):
    """Rotary embedding of x (n, h, d), halves (not interleaved), at rows pos."""
    c, s = cos[pos].double()[:, None], sin[pos].double()[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def exact(case, seed):
    """What run() returns for these inputs, in float64 by plain torch."""
    s = prepare(case, seed)
    hq, hk = case["hq"], case["hk"]
    g = hq // hk
    sqs, sks = _lengths(case, seed)
    with torch.no_grad():
        if case["kind"] in ("kvcache", "paged"):
            return _exact_cached(case, s, sqs, sks, g)
        if case.get("packed"):
            q, k, v = (x.detach() for x in s["qkv"].unbind(2))
        else:
            q, k, v = (s[n].detach() for n in ("q", "k", "v"))
        drop = random.Random(seed).getrandbits(63) if case["dropout"] else None
        grad = case["grad"]
        res = [torch.zeros(x.shape, dtype=torch.float64, device="cuda") for x in ((q, q, k, v) if grad else (q,))]
        at = (0, 0)
        for z, (a, b) in enumerate(zip(sqs, sks)):
            rq = slice(at[0], at[0] + a) if case["kind"] == "varlen" else slice(None)
            rk = slice(at[1], at[1] + b) if case["kind"] == "varlen" else slice(None)
            at = (at[0] + a, at[1] + b)
            view = (lambda t: t) if case["kind"] == "varlen" else (lambda t: t[z])
            for h in range(hq):
                head = [view(t)[r, n].double() for t, r, n in ((q, rq, h), (k, rk, h // g), (v, rk, h // g))]
                dout = view(s["dout"])[rq, h].double() if grad else None
                # (the dropout counter of a packed batch runs over each sequence's own lengths)
                r = _attend(case, *head, h, b - a, s["alibi"][h] if case["alibi"] else None, dout, drop)
                if not grad:
                    view(res[0])[rq, h] = r
                    continue
                view(res[0])[rq, h] = r[0]
                view(res[1])[rq, h] = r[1]
                view(res[2])[rk, h // g] += r[2]
                view(res[3])[rk, h // g] += r[3]
        if not grad:
            return res[0]
        if case.get("packed"):
            return res[0], torch.stack(res[1:], 2)
        return tuple(res)


def _exact_cached(case, s, sqs, sks, g):
    hq, hk, d = case["hq"], case["hk"], case["d"]
    q = s["q"]
    out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    new = case["kind"] == "kvcache" and case["append"]
    page = s["kc"].shape[1]
    if new:
        kc, vc = s["kc"].double(), s["vc"].double()
    at = 0
    for z, (a, b) in enumerate(zip(sqs, sks)):
        pages = (s["table"][z].long() if s["table"] is not None else torch.tensor([z], device="cuda"))
        pages = pages[:-(-b // page)]
        k = s["kc"][pages].reshape(-1, hk, d)[:b].double()
        v = s["vc"][pages].reshape(-1, hk, d)[:b].double()
        qz = (q[at:at + a] if case["kind"] == "paged" else q[z]).double()
        at += a
        if new:
            pos = torch.arange(b - a, b, device="cuda")
            qz = _rotate(qz, s["cos"], s["sin"], pos)
            k[b - a:] = _rotate(s["k"][z].double(), s["cos"], s["sin"], pos)
            v[b - a:] = s["v"][z].double()
            kc[pages[pos // page], pos % page] = k[b - a:]
            vc[pages[pos // page], pos % page] = v[b - a:]
        delta = b - a if case["kind"] == "paged" or new else None
        for h in range(hq):
            r = _attend(case, qz[:, h], k[:, h // g], v[:, h // g], h, delta)
            if case["kind"] == "paged":
                out[at - a:at, h] = r
            else:
                out[z, :, h] = r
    return {"out": out, "k_cache": kc, "v_cache": vc} if new else out


# ----------------------------------------------------------------------------- tolerance
def tolerance(case):
    """Relative 2-norm, about four times the distance of the path from exact(), which measured
    over the listed and drawn cases 2.0e-3 to 2.5e-3 in bf16 and 2.5e-4 to 3.0e-4 in fp16 (the
    operands of the second product, P and dS, and the results are rounded to the dtype), and up
    to 4.8e-7 in fp32 for 1000 keys (a few times that for longer sums and for capped logits)."""
    return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 5e-6}[case["dtype"]]}
