"""The prompt kernels (rotary + cache write, causal attention) against a float64 statement of the same sums, at the edges of
their tiles: 16 queries a wave, 64 a workgroup, 32 keys a step."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 32), (8, 2, 64), (4, 1, 128), (2, 2, 256)]      # heads, key/value heads, head size


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


@pytest.mark.parametrize("nh,nkv,hd", SHAPES)
@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 33, 64, 65, 97, 130])
def test_prompt_rope_and_attention(nh, nkv, hd, T):
    from any_precision_amd import _capi
    max_len = 131
    gen = torch.Generator().manual_seed(1000 * T + hd)
    qkv = torch.randn((T, nh + 2 * nkv, hd), generator=gen).half()
    ang = torch.rand((max_len, hd // 2), generator=gen) * 6.28
    cos, sin = ang.cos(), ang.sin()
    stale = float("nan")                                          # cache rows past the prompt are not read
    kc = torch.full((nkv, max_len, hd), stale).half().cuda()
    vc = torch.full((nkv, max_len, hd), stale).half().cuda()
    x, c, s = qkv.cuda(), cos.cuda(), sin.cuda()
    scale = 1.0 / math.sqrt(hd)
    stream = torch.cuda.current_stream().cuda_stream
    _capi.check(_capi.lib.ap_prompt_rope(x.data_ptr(), c.data_ptr(), s.data_ptr(), kc.data_ptr(), vc.data_ptr(), T, nh, nkv, hd,
                                         max_len, stream), "ap_prompt_rope")
    want = _rotate(qkv[:, :nh + nkv].double(), cos[:T, None].double(), sin[:T, None].double())
    got = torch.cat((x[:, :nh].cpu(), kc[:, :T].cpu().transpose(0, 1)), dim=1).double()
    # one rounding to fp16 of a sum of two products of values below about 5: half a unit at 8 is 2^-9
    assert (got - want).abs().max().item() <= 2.0 ** -9 + 1e-4
    assert torch.equal(vc[:, :T].cpu(), qkv[:, nh + nkv:].transpose(0, 1))
    assert torch.isnan(kc[:, T:]).all() and torch.isnan(vc[:, T:]).all()

    q, k, v = x[:, :nh].cpu().double(), kc[:, :T].cpu().double(), vc[:, :T].cpu().double()
    k, v = k.repeat_interleave(nh // nkv, 0), v.repeat_interleave(nh // nkv, 0)
    scores = torch.einsum("thd,hjd->htj", q, k) * scale
    scores.masked_fill_(torch.arange(T)[None, :] > torch.arange(T)[:, None], float("-inf"))
    ctx = torch.einsum("htj,hjd->thd", scores.softmax(-1), v)
    for first in sorted({0, T // 2, T - 1}):
        out = torch.full((T - first, nh * hd), stale).half().cuda()
        _capi.check(_capi.lib.ap_prompt_attention(x.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), first, T, nh, nkv,
                                                  hd, max_len, scale, stream), "ap_prompt_attention")
        err = (out.cpu().double().view(T - first, nh, hd) - ctx[first:]).abs().max().item()
        # a convex combination of values below about 5: weights in fp16 and a result in fp16 are off by 2^-11 each,
        # relative; exponentials of fp32 scores by less
        assert err <= 5 * (2 * 2.0 ** -11) + 1e-3, f"first={first}: {err}"


def test_prompt_argument_errors():
    from any_precision_amd import _capi
    L, fake = _capi.lib, 4096
    assert L.ap_prompt_rope(None, fake, fake, fake, fake, 4, 2, 2, 64, 16, None) == _capi.AP_ENULL
    assert L.ap_prompt_rope(fake, fake, fake, fake, fake, 17, 2, 2, 64, 16, None) == _capi.AP_ESHAPE
    assert L.ap_prompt_rope(fake, fake, fake, fake, fake, 4, 2, 2, 48, 16, None) == _capi.AP_ESHAPE
    assert L.ap_prompt_attention(fake, fake, fake, fake, 4, 4, 2, 2, 64, 16, 1.0, None) == _capi.AP_ESHAPE
    assert L.ap_prompt_attention(fake, fake, fake, fake + 8, 0, 4, 2, 2, 64, 16, 1.0, None) == _capi.AP_EALIGN


@pytest.mark.parametrize("nh,nkv,hd", SHAPES)
def test_prompt_attention_with_scores_of_minus_infinity(nh, nkv, hd):
    """A key whose score is -inf weighs nothing, also where a query meets only such keys in its first tile of 32; a query that
    sees nothing else has no result (NaN, as softmax has it)."""
    from any_precision_amd import _capi
    T, hidden, scale = 100, 40, 0.5
    gen = torch.Generator().manual_seed(hd)
    qkv = torch.randn((T, nh + 2 * nkv, hd), generator=gen).half()
    qkv[:, :nh, 0] = qkv[:, :nh, 0].abs() + 1
    k, v = (torch.randn((nkv, T, hd), generator=gen).half() for _ in range(2))
    k[:, :hidden, 0] = float("-inf")
    x, kc, vc = qkv.cuda(), k.cuda(), v.cuda()
    out = torch.zeros((T, nh * hd)).half().cuda()
    _capi.check(_capi.lib.ap_prompt_attention(x.data_ptr(), kc.data_ptr(), vc.data_ptr(), out.data_ptr(), 0, T, nh, nkv, hd, T, scale,
                                              torch.cuda.current_stream().cuda_stream), "ap_prompt_attention")
    k, v = (t.double().repeat_interleave(nh // nkv, 0) for t in (k, v))
    scores = torch.einsum("thd,hjd->htj", qkv[:, :nh].double(), k) * scale
    scores.masked_fill_(torch.arange(T)[None, :] > torch.arange(T)[:, None], float("-inf"))
    want = torch.einsum("htj,hjd->thd", scores[:, hidden:].softmax(-1), v)
    got = out.cpu().double().view(T, nh, hd)
    assert torch.isnan(got[:hidden]).all()
    # as above: fp16 weights and results over values below about 5
    assert (got[hidden:] - want).abs().max().item() <= 5 * (2 * 2.0 ** -11) + 1e-3
