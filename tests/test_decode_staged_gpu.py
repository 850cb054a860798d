"""Decode attention over keys and values that go through LDS, against caches that start off 16 bytes,
which go straight to registers: the same sums in the same order."""

import pytest
import torch

from neuronx_distributed_inference_amd import ops

pytestmark = pytest.mark.gpu


def _off(t):
    """A copy that starts 8 bytes behind 16."""
    n = 8 // t.element_size()
    flat = torch.empty(t.numel() + 2 * n, dtype=t.dtype, device=t.device)
    at = n if flat.data_ptr() % 16 == 0 else 0
    copy = flat[at:at + t.numel()].view(t.shape)
    copy.copy_(t)
    assert copy.data_ptr() % 16 == 8
    return copy


# a wave's step is 32 keys, a workgroup's 128, splits keep 128 or 256; 768 sets go a wave a set
@pytest.mark.parametrize("B,Hkv,gq,cap", [(1, 1, 1, 1), (2, 2, 4, 31), (3, 2, 8, 32), (2, 8, 1, 33), (1, 2, 16, 129),
                                          (5, 3, 4, 257), (1, 8, 4, 4097), (64, 8, 2, 700), (97, 8, 4, 200)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("dtype,f8", [(torch.bfloat16, False), (torch.float16, False), (torch.bfloat16, True)])
@pytest.mark.parametrize("window", [0, 40])
def test_staged_as_straight(B, Hkv, gq, cap, D, dtype, f8, window):
    g = torch.Generator(device="cuda").manual_seed(cap)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(dtype)  # noqa: E731
    q, k, v = rnd(B, Hkv * gq, 1, D), rnd(B, Hkv, cap, D), rnd(B, Hkv, cap, D)
    if f8:
        k, v = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
    else:
        v[0, 0, cap // 2, 3] = float("nan")
    pos = torch.randint(0, cap, (B, 1), generator=g, device="cuda")
    pos[-1] = cap - 1
    if B > 2:
        pos[1] = -1
    call = lambda k, v: ops.attention_decode(q, k, v, pos, sliding_window=window)  # noqa: E731
    a, b = call(k, v), call(_off(k), _off(v))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("B,Hkv,gq,pages,size", [(1, 2, 4, 1, 16), (3, 2, 8, 5, 7), (2, 8, 4, 33, 64), (100, 8, 1, 4, 32)])
@pytest.mark.parametrize("D", [64, 128])
def test_staged_pages_as_straight(B, Hkv, gq, pages, size, D):
    g = torch.Generator(device="cuda").manual_seed(pages)
    rnd = lambda *s: torch.empty(*s, device="cuda").normal_(0, 1, generator=g).to(torch.bfloat16)  # noqa: E731
    n = B * pages + 1
    q, k, v = rnd(B, Hkv * gq, 1, D), rnd(n, size, Hkv, D), rnd(n, size, Hkv, D)
    v[0] = float("nan")                                # what stands in for a missing page
    table = (torch.randperm(n - 1, generator=g, device="cuda") + 1).view(B, pages).int()
    if pages > 2:
        table[0, 1] = -1
    pos = torch.randint(0, pages * size, (B, 1), generator=g, device="cuda")
    call = lambda k, v: ops.attention_decode_paged(q, k, v, pos, table)  # noqa: E731
    a, b = call(k, v), call(_off(k), _off(v))
    assert a.isfinite().all() and torch.equal(a.view(torch.int16), b.view(torch.int16))


def _kernels(call):
    """The result, and the names of the kernels that made it."""
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as p:
        y = call()
        torch.cuda.synchronize()
    return y, " ".join(e.key for e in p.key_averages())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,D,N,L,pos,f8,by", [
    (32, 8, 64, 2048, 1024, 700, False, "product"), (32, 8, 128, 4096, 1024, 1023, False, "product"),
    (8, 8, 64, 516, 512, 0, False, "product"), (4, 1, 64, 64, 2048, 900, True, "product"),
    (16, 2, 128, 2048, 4096, 4000, True, "product"), (64, 8, 128, 8192, 8192, 8000, False, "kernel"),
    (9, 3, 128, 1000, 300, 200, False, "product"), (8, 2, 64, 20000, 1500, 1400, False, "product"),
    (4, 4, 64, 100, 4096, 17, False, "product"), (4, 2, 64, 256, 128, 100, False, "none"),
    (8, 1, 128, 512, 120, 119, True, "none")])
def test_decode_and_its_product(Hq, Hkv, D, N, L, pos, f8, by, dtype):
    """One token's attention and output product in one call against one after the other, with shares
    added up by the product, by a kernel of their own, and with none."""
    g = torch.Generator(device="cuda").manual_seed(L + N)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)  # noqa: E731
    q, w = rnd(1, Hq, 1, D), rnd(N, Hq * D) * 0.05
    kc, vc = (rnd(3, Hkv, L, D) for _ in range(2))
    if f8:
        kc, vc = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
    p = torch.tensor([[pos]], device="cuda", dtype=torch.int32)
    sid = torch.tensor([2], device="cuda", dtype=torch.int32)
    for window in (0, 130):
        y, names = _kernels(
            lambda: ops.attention_decode_product(q, kc, vc, p, sid, D ** -0.5, window, w))
        assert ("shares_gemm" in names, "decode_attn_pass2" in names) == \
            {"product": (True, False), "kernel": (False, True), "none": (False, False)}[by]
        o = ops.attention_decode(q, kc, vc, p, seq_ids=sid, scale=D ** -0.5, sliding_window=window)
        want = ops.linear_parts(o.transpose(1, 2).reshape(1, 1, Hq * D), w)
        assert y.shape == want.shape and y.dtype == want.dtype
        if by != "product":
            assert torch.equal(y, want)
            continue
        # The product adds shares up one after the other, the kernel in a tree: sums that differ by
        # some 2^-20, of which a rounding to 16 bits now and then falls the other way (2^-7, 2^-10
        # at most). Of one value in 16 at the most.
        both = [t.double().sum(0) if t.dim() == 4 else t.double() for t in (y, want)]
        slack = (2.0 ** -11 if dtype == torch.bfloat16 else 2.0 ** -14) \
            * (o.flatten().double().abs() @ w.double().abs().t())
        if want.dim() < 4:                             # the result's own rounding
            slack = slack + (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) * both[1].view(-1).abs()
        assert ((both[0] - both[1]).abs().view(-1) <= slack).all()
    vc[2, :, min(pos, 5)] = float("nan")
    y = ops.attention_decode_product(q, kc, vc, p, sid, D ** -0.5, 0, w)
    assert y.float().isnan().any()
    assert ops.attention_decode_product(q.float(), kc, vc, p, sid, 1.0, 0, w) is None
    # (1,) is a length and not a position
    assert ops.attention_decode_product(q, kc, vc, p.view(1), sid, 1.0, 0, w) is None
