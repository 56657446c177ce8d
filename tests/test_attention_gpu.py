"""GPU parity of the one-launch decode attention (nm_attention_decode) against
attention in 64 bits: both element types and head dimensions, 1 to 16 query
heads per key/value head, positions at the edges of the splits (first, last
of a split, first of the next, last of the cache), every span, padded key
rows, and cached values past the position that are not finite."""
import math

import pytest
import torch

from spmv_decode_amd import hip_spmv

pytestmark = pytest.mark.gpu


def case(nh, kvh, hd, S, dtype, pad, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randn(nh, hd + pad, device="cuda", generator=gen).to(dtype)
    k = torch.randn(kvh, hd + pad, S, device="cuda", generator=gen).to(dtype)
    v = torch.randn(kvh, hd, S, device="cuda", generator=gen).to(dtype)
    return q, k, v


def exact(q, k, v, hd, n):
    kvh = k.shape[0]
    qd = q[:, :hd].double().view(kvh, -1, hd)
    p = torch.softmax(torch.bmm(qd, k[:, :hd, :n].double().contiguous()) / math.sqrt(hd), dim=-1)
    return torch.bmm(p, v[:, :, :n].double().transpose(1, 2).contiguous()).reshape(1, -1)


# (query heads, key/value heads, head_dim, cache length, padding)
SHAPES = [(32, 8, 128, 640, 32), (40, 8, 128, 4096, 32), (16, 8, 128, 128, 0), (64, 8, 128, 1032, 32),
          (16, 1, 64, 264, 8), (4, 2, 64, 8, 32), (5, 5, 128, 9000, 0)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_attention_decode_matches_exact(gpu, shape, dtype):
    nh, kvh, hd, S, pad = shape
    q, k, v = case(nh, kvh, hd, S, dtype, pad, seed=S + nh)
    # one rounding of each probability and of each output: two half-ulps, relative to the outputs' norm
    bar = 2 * torch.finfo(dtype).eps
    for pos in sorted({0, 1, 7, 63, 64, 127, 255, 256, S // 2, S - 2, S - 1, S + 5}):
        if pos >= S and pos != S + 5:
            continue
        n = min(pos + 1, S)
        ref = exact(q, k, v, hd, n)
        kd, vd = k.clone(), v.clone()
        vd[:, :, n:] = float("nan")  # stale cache contents must not reach the result
        kd[:, :, n:] = float("nan")
        at = torch.tensor([pos], device="cuda")
        for span in (0, 64, 128, 256):
            if span and 8 * -(-S // span) * (nh // kvh) + 4112 > 2 * hd * span:
                continue
            y = hip_spmv.nmsparse_attention_decode(q, kd, vd, at, hd, span=span)
            again = hip_spmv.nmsparse_attention_decode(q, kd, vd, at, hd, span=span)
            assert torch.equal(y, again), (shape, pos, span)
            rel = float((y.double() - ref).norm() / ref.norm())
            assert rel <= bar, (shape, dtype, pos, span, rel)


def test_attention_decode_edges(gpu):
    q, k, v = case(8, 2, 128, 64, torch.float16, 0, seed=3)
    none = hip_spmv.nmsparse_attention_decode(q, k, v, torch.tensor([-1], device="cuda"), 128)
    assert torch.isnan(none).all()
    k[0, :, 5] = float("nan")  # a NaN score makes its heads' rows NaN, and no others
    y = hip_spmv.nmsparse_attention_decode(q, k, v, torch.tensor([9], device="cuda"), 128).view(8, 128)
    assert torch.isnan(y[:4]).all() and torch.isfinite(y[4:]).all()
    for bad in ((q.float(), k.float(), v.float()), (q, k[:, :, :60], v[:, :, :60]), (q[:, :64], k, v), (q[:7], k, v)):
        assert not hip_spmv.attention_supported(*bad, 128)
        with pytest.raises(ValueError):
            hip_spmv.nmsparse_attention_decode(*bad, torch.tensor([3], device="cuda"), 128)


# (positions, query heads, key/value heads, head_dim, cache length, padded key rows, norms, row padding)
PROMPTS = [(1, 4, 2, 64, 8, 32, False, 0), (63, 32, 8, 128, 640, 32, False, 0), (64, 16, 8, 128, 128, 0, True, 0),
           (65, 6, 2, 128, 72, 32, True, 64), (200, 40, 8, 128, 256, 32, True, 0), (333, 4, 4, 64, 336, 0, False, 8),
           (520, 16, 1, 128, 1024, 32, False, 0)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", PROMPTS, ids=str)
def test_prompt_attention_matches_exact(gpu, case, dtype):
    P, nh, kvh, hd, S, pad, norms, rowpad = case
    gen = torch.Generator(device="cuda").manual_seed(P + nh)

    def rows(heads):
        return torch.randn(P, heads * hd + rowpad, device="cuda", generator=gen).to(dtype)[:, :heads * hd]

    q, k, v = rows(nh), rows(kvh), rows(kvh)
    qn, kn = ((1 + 0.1 * torch.randn(2, hd, device="cuda", generator=gen)).to(dtype).unbind(0) if norms
              else (None, None))
    ang = torch.rand(S, hd // 2, device="cuda", generator=gen, dtype=torch.float64) * 6.28
    table = torch.view_as_real(torch.polar(torch.ones_like(ang), ang).to(torch.complex64)).contiguous()
    kc = torch.full((kvh, hd + pad, S), float("nan"), device="cuda", dtype=dtype)  # stale contents stay out
    vc = torch.full((kvh, hd, S), float("nan"), device="cuda", dtype=dtype)
    y = hip_spmv.nmsparse_prefill_attention(q, k, v, kc, vc, table, hd, q_norm=qn, k_norm=kn, norm_eps=1e-6)

    def turned(t, heads, norm):
        t = t.double().view(P, heads, hd)
        if norm is not None:
            t = t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-6) * norm.double()
        c, s = table[:P, None, :, 0].double(), table[:P, None, :, 1].double()
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack((a * c - b * s, a * s + b * c), dim=-1).flatten(-2)

    eps = torch.finfo(dtype).eps
    kr = turned(k, kvh, kn)
    assert float((kc[:, :hd, :P].double() - kr.permute(1, 2, 0)).norm() / kr.norm()) <= eps  # one rounding
    assert torch.equal(vc[:, :, :P], v.reshape(P, kvh, hd).permute(1, 2, 0))
    assert bool(torch.isnan(kc[:, hd:]).all()) and bool(torch.isnan(kc[:, :, P:]).all())
    assert bool(torch.isnan(vc[:, :, P:]).all())
    # attention of the rounded queries and keys in 64 bits
    qr, kr = turned(q, nh, qn).to(dtype).double(), kc[:, :hd, :P].double()
    s = torch.bmm(qr.transpose(0, 1).contiguous(), kr.repeat_interleave(nh // kvh, 0).contiguous()) / math.sqrt(hd)
    s = s.masked_fill(torch.ones(P, P, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    ref = torch.bmm(torch.softmax(s, -1), vc[:, :, :P].double().transpose(1, 2).repeat_interleave(nh // kvh, 0)
                    .contiguous()).transpose(0, 1).reshape(P, nh * hd)
    rel = float((y.double() - ref).norm() / ref.norm())
    assert rel <= 2 * eps, rel


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=str)
def test_attention_decode_over_splits_of_infinite_scores(gpu, dtype):
    """Whole splits whose every score is -inf weigh nothing and leave the rest
    its softmax; a row of nothing else is NaN, as a softmax of it is."""
    hd, S = 128, 640
    q, k, v = case(8, 2, hd, S, dtype, 0, seed=5)
    q[:, 0] = 1
    k[0, 0, :256] = -math.inf
    bar = 2 * torch.finfo(dtype).eps
    for span in (0, 64, 128, 256):
        for pos in (256, 300, 511, 639):
            y = hip_spmv.nmsparse_attention_decode(q, k, v, torch.tensor([pos], device="cuda"), hd, span=span)
            ref = exact(q, k, v, hd, pos + 1)
            assert float((y.double() - ref).norm() / ref.norm()) <= bar, (span, pos)
        for pos in (63, 255):
            y = hip_spmv.nmsparse_attention_decode(q, k, v, torch.tensor([pos], device="cuda"), hd, span=span)
            assert torch.isnan(y[0, :4 * hd]).all() and torch.isfinite(y[0, 4 * hd:]).all(), (span, pos)


def test_prompt_attention_over_blocks_of_infinite_scores(gpu):
    """The same of a row's leading blocks in a prompt: in bf16, scores of
    -1e60 are -inf in fp32."""
    P, nh, kvh, hd, S, first = 200, 4, 2, 128, 256, 70
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(P, h * hd, device="cuda", generator=gen).bfloat16() for h in (nh, kvh, kvh))
    q[:, ::hd], k[:, ::hd] = 1e30, 0
    k[:first, ::hd] = -1e30
    table = torch.zeros(S, hd // 2, 2, device="cuda")
    table[..., 0] = 1  # no rotation
    kc, vc = (torch.zeros(kvh, hd, S, device="cuda").bfloat16() for _ in range(2))
    y = hip_spmv.nmsparse_prefill_attention(q, k, v, kc, vc, table, hd).view(P, nh, hd)
    qd, kd, vd = (t.double().view(P, -1, hd).transpose(0, 1).contiguous() for t in (q, k, v))
    kd, vd = kd.repeat_interleave(nh // kvh, 0), vd.repeat_interleave(nh // kvh, 0)
    s = torch.bmm(qd, kd.transpose(1, 2).contiguous()) / math.sqrt(hd)
    s = s.masked_fill(torch.ones(P, P, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    ref = torch.bmm(torch.softmax(s, -1), vd).transpose(0, 1)[first:]
    assert float((y[first:].double() - ref).norm() / ref.norm()) <= 2 * torch.finfo(torch.bfloat16).eps
    assert torch.isnan(y[:first]).all()
