"""flash_attn_with_kvcache keeps the launch parameters of a signature it has served: calls that repeat
it (new tensors, new lengths, new addresses, another stream, another thread, an append that moves on)
give what the first, fully checked call gives, and anything that changes the signature or an address
that cannot be read in place goes through the checks again."""
import threading

import pytest

pytestmark = pytest.mark.gpu


def _inputs(seed, dense=False, append=True, off=0):
    import torch
    B, H, Hk, D, page, nb = 3, 8, 2, 128, 16, 16
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*s):
        n = 1
        for x in s:
            n *= x
        return torch.randn(n + off, generator=g, device="cuda", dtype=torch.bfloat16)[off:].view(*s)
    c = dict(q=rnd(B, 1, H, D))
    shape = (B, page * nb) if dense else (B * nb, page)
    c["k_cache"], c["v_cache"] = rnd(*shape, Hk, D), rnd(*shape, Hk, D)
    if not dense:
        c["block_table"] = torch.randperm(B * nb, generator=torch.Generator().manual_seed(seed)).view(B, nb).int().cuda()
    c["cache_seqlens"] = torch.tensor([100 + seed, 7, 3 * seed], dtype=torch.int32, device="cuda")
    if append:
        c["k"], c["v"] = rnd(B, 1, Hk, D), rnd(B, 1, Hk, D)
    return c


def _both(c, **kw):
    """(planned or not as it comes, the general path) on copies of the same inputs."""
    import torch

    from fable_attn import flash_attn_interface as fai
    res = []
    for f in (fai.flash_attn_with_kvcache, fai._with_kvcache):
        a = {n: t.clone() if n.endswith("cache") else t for n, t in c.items()}
        res.append((f(**a, **kw), a["k_cache"], a["v_cache"]))
    torch.cuda.synchronize()
    for x, y in zip(*res):
        assert torch.equal(x, y)
    return res[0][0]


@pytest.mark.parametrize("dense", [False, True], ids=["paged", "dense"])
@pytest.mark.parametrize("append", [False, True], ids=["read", "append"])
def test_repeated_signature(dense, append):
    import torch
    outs = [_both(_inputs(s, dense, append)) for s in (1, 2, 3)]
    assert not torch.equal(outs[1], outs[2])
    _both(_inputs(4, dense, append), window_size=(31, 0), softcap=20.0)
    _both(_inputs(5, dense, append), window_size=(31, 0), softcap=20.0)
    _both(_inputs(6, dense, append, off=1))          # addresses off by two bytes
    c = _inputs(7, dense, append)
    c["cache_seqlens"] = c["cache_seqlens"].long()   # converted by the general path
    _both(c)
    _both(c)
    c["cache_seqlens"] = None                         # the whole cache
    if not append:
        _both(c)
        _both(c)
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        _both(_inputs(8, dense, append))
    torch.cuda.current_stream().wait_stream(st)
    err = []

    def work(seed):
        try:
            for i in range(3):
                _both(_inputs(seed + i, dense, append))
        except Exception as e:   # noqa: BLE001  (reported by the main thread)
            err.append(e)
    ts = [threading.Thread(target=work, args=(10 * i,)) for i in (1, 2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not err, err


def test_checks_still_raise():
    """A signature that was served does not let a wrong one through."""
    from fable_attn import flash_attn_with_kvcache
    c = _inputs(1)
    flash_attn_with_kvcache(**c)
    flash_attn_with_kvcache(**c)
    with pytest.raises(RuntimeError):
        flash_attn_with_kvcache(**dict(c, cache_seqlens=c["cache_seqlens"][:2].contiguous()))
    with pytest.raises(RuntimeError):
        flash_attn_with_kvcache(**dict(c, v_cache=c["v_cache"].half()))
    with pytest.raises(ValueError):
        flash_attn_with_kvcache(**dict(c, v=None))
    with pytest.raises(TypeError):
        flash_attn_with_kvcache(**c, num_splits=1.5)


def test_packed_inference_equals_separate():
    """qkv- and kv-packed inference on views of the packed tensor, as flash_attn_func on them."""
    import torch

    from fable_attn import flash_attn_func, flash_attn_kvpacked_func, flash_attn_qkvpacked_func
    qkv = torch.randn(2, 77, 3, 4, 64, device="cuda", dtype=torch.float16)
    for kw in ({}, {"causal": True}, {"window_size": (20, 5)}, {"softcap": 10.0}):
        want = flash_attn_func(*(t.contiguous() for t in qkv.unbind(2)), **kw)
        for _ in range(2):
            assert torch.equal(flash_attn_qkvpacked_func(qkv, **kw), want)
            assert torch.equal(flash_attn_kvpacked_func(qkv[:, :, 0], qkv[:, :, 1:], **kw), want)


def test_tensor_options_by_value():
    """A scale, cap or window given as a tensor counts by the value it has at the call."""
    import torch

    from fable_attn import flash_attn_kvpacked_func
    c = _inputs(1, append=False)
    qkv = torch.randn(2, 77, 3, 4, 64, device="cuda", dtype=torch.float16)
    x = torch.tensor(2.0)
    for opt in ({"softmax_scale": x}, {"softcap": x}, {"window_size": (x, 0)}):
        for value in (2.0, 5.0):
            x.fill_(value)
            plain = {n: value if t is x else (int(value), 0) for n, t in opt.items()}
            for _ in range(2):
                assert torch.equal(_both(c, **opt), _both(c, **plain))
                assert torch.equal(flash_attn_kvpacked_func(qkv[:, :, 0], qkv[:, :, 1:], **opt),
                                   flash_attn_kvpacked_func(qkv[:, :, 0], qkv[:, :, 1:], **plain))


def test_packed_inference_mixed_dtypes_refused():
    """A served (fp16, fp16) signature does not let (fp16 q, bf16 kv) of the same shapes through."""
    import torch

    from fable_attn import flash_attn_func, flash_attn_kvpacked_func
    q = torch.randn(1, 32, 4, 64, device="cuda", dtype=torch.float16)
    kv = torch.randn(1, 32, 2, 4, 64, device="cuda", dtype=torch.float16)
    flash_attn_kvpacked_func(q, kv)
    with pytest.raises(RuntimeError):
        flash_attn_kvpacked_func(q, kv.bfloat16())
    k, v = kv.unbind(2)
    for a, b in ((k.bfloat16(), v), (k, v.bfloat16())):
        with pytest.raises(RuntimeError):
            flash_attn_func(q, a, b)
