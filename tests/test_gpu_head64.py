"""Heads of 64 on the matrix cores, against float64 and against the general kernels, which the same call takes when a tensor
does not start on a 16-byte boundary."""
import numpy as np
import pytest
import torch

from diopi_amd import functions as F
from diopi_amd import runtime as rt

pytestmark = pytest.mark.gpu
DEV = "cuda"
# unit roundoff of the element type, and half its smallest step (what a rounding is off by where the type runs out of exponents)
ROUND = {torch.float16: (2.0 ** -11, 2.0 ** -25), torch.bfloat16: (2.0 ** -8, 0.0)}


def _unaligned(t):
    """The same values one element behind a 16-byte boundary."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


def _decode(lens, H, Hkv, dt, idt, seed, D=64):
    g = torch.Generator().manual_seed(seed)
    B, longest, total = len(lens), max(lens) + 5, sum(lens)
    slots = total + 3
    order = torch.randperm(slots, generator=g)
    b_loc, start = torch.zeros(B, longest, dtype=idt), np.concatenate(([0], np.cumsum(lens)))[:-1]
    for i, n in enumerate(lens):
        b_loc[i, longest - n:] = order[start[i]:start[i] + n].to(idt)
    rand = lambda *shape: torch.randn(*shape, generator=g).to(dt).to(DEV)
    return dict(B=B, longest=longest, total=total, start=start, b_loc=b_loc.to(DEV), b_start=torch.from_numpy(start).to(idt).to(DEV),
                b_len=torch.tensor(lens, dtype=idt, device=DEV), q=rand(B, H, D), k=rand(slots, Hkv, D), v=rand(slots, Hkv, D), logits=rand(H, total) * 3)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,Hkv,idt", [(1, 1, torch.int32), (4, 4, torch.int32), (9, 3, torch.int64), (32, 8, torch.int32), (16, 2, torch.int64),
                                       (27, 3, torch.int32), (16, 1, torch.int32)])
def test_softmax_reducev(dt, H, Hkv, idt):
    lens = [1, 31, 32, 33, 0, 127, 128, 129, 511, 513, 2048, 2049, 8193]
    w = _decode(lens, H, Hkv, dt, idt, 64 + H)
    if H > 1:
        w["logits"][0, int(w["start"][7]):int(w["start"][7]) + 129] = -float("inf")  # a head that sees nothing
    w["logits"][H - 1, int(w["start"][8]):int(w["start"][8]) + 400] = -float("inf")
    rest = (w["b_loc"], w["b_start"], w["b_len"], w["longest"], 0)
    out, general = (torch.full((w["B"], H, 64), 5.0, dtype=dt, device=DEV) for _ in range(2))
    F.token_softmax_reducev(w["logits"], w["v"], out, *rest)
    F.token_softmax_reducev(w["logits"], _unaligned(w["v"]), general, *rest)
    u, tiny = ROUND[dt]
    for i, n in enumerate(lens):
        if n == 0:
            assert not out[i].any()
            continue
        at = int(w["start"][i])
        v = w["v"][w["b_loc"][i, w["longest"] - n:].long()].double().repeat_interleave(H // Hkv, 1).transpose(0, 1).contiguous()
        p = torch.softmax(w["logits"][:, at:at + n].double(), -1).nan_to_num(0.0)
        want = (p[:, None] @ v)[:, 0]
        # one rounding of every probability, at worst n roundings of an fp32 sum, one rounding of the result
        sizes = (p[:, None] @ v.abs())[:, 0]
        bound = (u + n * 2.0 ** -23) * sizes + n * tiny * v.abs().amax(1) + u * want.abs() + tiny + 1e-6
        assert ((out[i].double() - want).abs() <= 1.01 * bound).all(), (i, n)
        assert ((out[i].double() - general[i].double()).abs() <= 2.02 * bound).all(), (i, n)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("H,Hkv,lens", [(16, 2, [1, 128, 129, 507]), (16, 2, [1, 384, 385, 508]), (9, 3, [508]), (32, 32, [700, 3, 699, 0, 513, 129, 1, 600, 64])])
def test_softmax_reducev_waves_and_order(H, Hkv, lens, D):
    """Few work-groups over windows of 512 and of 513 columns, which four and sixteen waves take, and more work-groups than compute
    units over sequences of unequal length, which are taken longest first."""
    w = _decode(lens, H, Hkv, torch.float16, torch.int32, 264 + H, D)
    out = torch.full((w["B"], H, D), 5.0, dtype=torch.float16, device=DEV)
    F.token_softmax_reducev(w["logits"], w["v"], out, w["b_loc"], w["b_start"], w["b_len"], w["longest"], 0)
    u, tiny = ROUND[torch.float16]
    for i, n in enumerate(lens):
        at = int(w["start"][i])
        v = w["v"][w["b_loc"][i, w["longest"] - n:].long()].double().repeat_interleave(H // Hkv, 1).transpose(0, 1).contiguous() if n else torch.zeros(H, 1, D, device=DEV).double()
        p = torch.softmax(w["logits"][:, at:at + n].double(), -1) if n else torch.zeros(H, 1, device=DEV).double()
        want, sizes = (p[:, None] @ v)[:, 0], (p[:, None] @ v.abs())[:, 0]
        bound = (u + n * 2.0 ** -23) * sizes + n * tiny * v.abs().amax(1) + u * want.abs() + tiny + 1e-6  # as above
        assert ((out[i].double() - want).abs() <= 1.01 * bound).all(), (i, n)


def test_softmax_reducev_infinite_values():
    """An infinite value in a sequence's last row, which a step of 32 tokens reads more than once."""
    w = _decode([1, 30, 33, 129], 8, 4, torch.float16, torch.int32, 3)
    for i, n in enumerate([1, 30, 33, 129]):
        w["v"][int(w["b_loc"][i, -1]), 1, 7] = float("inf")
    out, general = (torch.zeros(4, 8, 64, dtype=torch.float16, device=DEV) for _ in range(2))
    rest = (w["b_loc"], w["b_start"], w["b_len"], w["longest"], 0)
    F.token_softmax_reducev(w["logits"], w["v"], out, *rest)
    F.token_softmax_reducev(w["logits"], _unaligned(w["v"]), general, *rest)
    assert torch.equal(out.isinf(), general.isinf()) and int(out.isinf().sum()) == 8 and not out.isnan().any()


@pytest.mark.parametrize("n", [100, 3000])
def test_softmax_reducev_infinite_values_that_nothing_weighs(n):
    """A head whose logits are all -inf over rows with an infinite value and a NaN: zeros, and NaN where those stand."""
    w = _decode([n], 4, 2, torch.float16, torch.int32, 4)
    w["logits"][1] = -float("inf")
    w["v"][int(w["b_loc"][0, -1]), 0, 7] = float("inf")
    w["v"][int(w["b_loc"][0, -n]), 0, 9] = float("nan")
    out, general = (torch.zeros(1, 4, 64, dtype=torch.float16, device=DEV) for _ in range(2))
    rest = (w["b_loc"], w["b_start"], w["b_len"], w["longest"], 0)
    F.token_softmax_reducev(w["logits"], w["v"], out, *rest)
    F.token_softmax_reducev(w["logits"], _unaligned(w["v"]), general, *rest)
    assert out[0, 1].isnan().nonzero().flatten().tolist() == [7, 9] and int((out[0, 1] == 0).sum()) == 62
    assert torch.equal(out[0, 1].isnan(), general[0, 1].isnan())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,Hkv,idt", [(1, 1, torch.int32), (9, 3, torch.int64), (32, 8, torch.int32), (27, 3, torch.int32), (16, 1, torch.int32)])
def test_token_attention(dt, H, Hkv, idt):
    lens = [1, 15, 16, 17, 0, 63, 64, 65, 255, 257, 1030]
    w = _decode(lens, H, Hkv, dt, idt, 164 + H)
    w["k"][int(w["b_loc"][9, -1]), 0, 5] = float("inf")  # one head's infinity is no other head's business
    rest = (w["b_loc"], w["b_start"], w["b_len"], w["longest"])
    out, general = (torch.full((H, w["total"]), 5.0, dtype=dt, device=DEV) for _ in range(2))
    F.token_attention(w["q"], w["k"], out, *rest)
    F.token_attention(w["q"], _unaligned(w["k"]), general, *rest)
    assert torch.equal(out.isfinite(), general.isfinite())
    u, tiny = ROUND[dt]
    for i, n in enumerate(lens):
        at = int(w["start"][i])
        k = w["k"][w["b_loc"][i, w["longest"] - n:].long()].double().repeat_interleave(H // Hkv, 1).permute(1, 2, 0).contiguous()
        want = (w["q"][i].double()[:, None] @ k)[:, 0] / 8
        # an fp32 sum of 64 products, a rounding, a division by 8, a rounding
        bound = 2 * u * want.abs() + 64 * 2.0 ** -23 * (w["q"][i].double().abs()[:, None] @ k.abs())[:, 0] + tiny + 1e-9
        got = [t[:, at:at + n].double() for t in (out, general)]
        fine = want.isfinite()
        assert ((got[0] - want).abs() <= 1.01 * bound)[fine].all() and ((got[0] - got[1]).abs() <= 2.02 * bound)[fine].all(), (i, n)


def _in_window(w, window):
    table = torch.zeros(w["B"], window, dtype=torch.int32, device=DEV)
    table[:, -w["longest"]:] = w["b_loc"]
    return table, w["b_start"], w["b_len"], window


@pytest.mark.parametrize("H,Hkv,window", [(2, 2, 65535 * 64 + 1), (4, 1, 65535 * 128)])
def test_token_attention_long_windows(H, Hkv, window):
    """Windows of more tiles of 64 tokens than a launch can have: only their last columns are in use."""
    w = _decode([70, 200], H, Hkv, torch.float16, torch.int32, 31)
    out, short = (torch.zeros(H, w["total"], dtype=torch.float16, device=DEV) for _ in range(2))
    F.token_attention(w["q"], w["k"], out, *_in_window(w, window))
    F.token_attention(w["q"], w["k"], short, w["b_loc"], w["b_start"], w["b_len"], w["longest"])
    assert torch.equal(out, short)


def test_token_attention_long_window_of_grouped_heads():
    """Heads of 128 in groups had tiles of 256 tokens whatever the number of cached tokens."""
    H, Hkv, D, window, n = 8, 2, 128, 65535 * 64 + 1, 100
    g = torch.Generator().manual_seed(32)
    q, k = (torch.randn(s, generator=g).half().to(DEV) for s in ((1, H, D), (n, Hkv, D)))
    table = torch.zeros(1, window, dtype=torch.int32, device=DEV)
    table[0, -n:] = torch.arange(n)
    start, length = (torch.tensor([x], dtype=torch.int32, device=DEV) for x in (0, n))
    out, short = (torch.zeros(H, n, dtype=torch.float16, device=DEV) for _ in range(2))
    F.token_attention(q, k, out, table, start, length, window)
    F.token_attention(q, k, short, table[:, -n:].contiguous(), start, length, n)
    assert torch.equal(out, short)


def test_softmax_reducev_long_window():
    """A window of more ranges of 512 tokens than a launch can have."""
    w = _decode([70, 200], 2, 1, torch.float16, torch.int32, 31)
    out, general = (torch.zeros(2, 2, 64, dtype=torch.float16, device=DEV) for _ in range(2))
    F.token_softmax_reducev(w["logits"], w["v"], out, *_in_window(w, 65535 * 512 + 1), 0)
    F.token_softmax_reducev(w["logits"], _unaligned(w["v"]), general, w["b_loc"], w["b_start"], w["b_len"], w["longest"], 0)
    assert torch.equal(out, general)


def _packed(lens, H, Hkv, dt, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(sum(lens), h, 64, generator=g).to(dt).to(DEV) for h in (H, Hkv, Hkv))
    return q * 2, k, v, np.concatenate(([0], np.cumsum(lens)))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("H,Hkv,scale", [(1, 1, None), (6, 2, 0.3), (8, 1, None)])
def test_attention(dt, causal, H, Hkv, scale):
    lens = [1, 31, 32, 33, 0, 63, 64, 65, 127, 128, 129, 257, 700]
    q, k, v, start = _packed(lens, H, Hkv, dt, 11 + H)
    k[int(start[12]) + 300:int(start[12]) + 330] *= 9  # scores that rise late move the softmax reference
    cu = torch.from_numpy(start.astype(np.int32)).to(DEV)
    call = lambda vv: (F.flash_attention_varlen(q, k, vv, cu, cu, None, 700, 700, 0.0, scale, causal), F.GLOBAL_STATE["flash_attention_varlen_softmax_lse"])
    (out, lse), (general, general_lse) = call(v), call(_unaligned(v))
    lightllm = None
    if causal and H == Hkv:
        lightllm = F.context_attention(q, k, v, torch.zeros_like(q), cu[:-1], torch.tensor(lens, dtype=torch.int32, device=DEV), 700)
    u, tiny = ROUND[dt]
    for i, n in enumerate(lens):
        if n == 0:
            continue
        rows = slice(int(start[i]), int(start[i]) + n)
        qs, ks, vs = (t[rows].double().transpose(0, 1).contiguous() for t in (q, k, v))
        ks, vs = ks.repeat_interleave(H // Hkv, 0), vs.repeat_interleave(H // Hkv, 0)
        c = scale or 0.125
        s = qs @ ks.transpose(1, 2).contiguous() * c
        # an fp32 sum of 64 products, in any order, and its scaling: an absolute error of the score, a relative one of exp(score)
        e = (66 * 2.0 ** -24 * c * (qs.abs() @ ks.abs().transpose(1, 2).contiguous())).amax(-1, keepdim=True)
        if causal:
            s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -float("inf"))
        p = s.softmax(-1)
        want = (p @ vs).transpose(0, 1)
        sizes = (p @ vs.abs()).transpose(0, 1)
        # twice the scores' error, n roundings of a sum, two 16-bit halves of a probability (2^-16), and the result's rounding
        bound = (2 * e.transpose(0, 1) + n * 2.0 ** -23 + 2.0 ** -15) * sizes + n * tiny * 8 + u * want.abs() + tiny + 1e-6
        assert ((out[rows].double() - want).abs() <= 1.01 * bound).all(), (i, n)
        assert ((out[rows].double() - general[rows].double()).abs() <= 2.02 * bound).all(), (i, n)
        if lightllm is not None:
            assert ((lightllm[rows].double() - want).abs() <= 1.01 * bound).all(), (i, n)
        ref, at = s.logsumexp(-1), (i, slice(None), slice(0, n))
        assert ((lse[at].double() - ref).abs() <= e[..., 0] + 1e-5 + 1e-6 * ref.abs()).all(), (i, n)
        assert ((lse[at] - general_lse[at]).double().abs() <= 2 * e[..., 0] + 2e-5 + 2e-6 * ref.abs()).all(), (i, n)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,gap", [(16384, 10), (16384, 14), (32768, 20)])
def test_attention_one_key_over_many(dt, n, gap):
    """A key far above all others, whose own value is zero: what comes out is the sum of many small probabilities."""
    g = torch.Generator().manual_seed(gap)
    q, k, v = torch.zeros(n, 1, 64), torch.zeros(n, 1, 64), torch.rand(n, 1, 64, generator=g) + 0.5
    q[:, 0, 0] = 8
    k[:, 0, 0] = torch.randn(n, generator=g).clamp(-3, 3) * np.log(2)
    k[5, 0, 0] = gap * np.log(2)
    v[:, 0, :32] = 1
    v[5] = 0
    q, k, v = (t.to(dt).to(DEV) for t in (q, k, v))
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    out = F.flash_attention_varlen(q, k, v, cu, cu, None, n, n, 0.0, None, False)[:, 0].double()
    p = k[:, 0, 0].double().softmax(0)  # q . k / 8
    want = p @ v[:, 0].double()
    u, tiny = ROUND[dt]
    # the exponent of a score of at most 16 powers of two, scaled, shifted and taken in fp32; a rounding for each half of 16 keys, within
    # and after a tile; the halves of a probability (2^-17, and in fp16 2^-36 of the largest); the result's rounding
    rel = 64 * 2.0 ** -24 + (n / 8 + 64) * 2.0 ** -24 + 2.0 ** -17
    bound = rel * want + (n * 2.0 ** -36 * p.max() * 1.5 if dt == torch.float16 else 0.0) + u * want + tiny
    assert ((out - want).abs() <= 1.01 * bound).all(), float(((out - want) / want).abs().max())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_attention_values_that_are_no_numbers(dt):
    """What a row does not see leaves it alone: infinities and NaN among later rows' values, wherever the row stands in its tile."""
    lens = [200, 64, 33]
    q, k, v, start = _packed(lens, 4, 4, dt, 5)
    inf, nan = float("inf"), float("nan")
    for row, head, d, x in ((150, 0, 3, inf), (155, 0, 3, -inf), (140, 1, 40, -inf), (10, 2, 7, nan), (100, 2, 8, nan), (199, 3, 63, inf), (220, 0, 0, inf), (240, 0, 0, inf),
                            (296, 1, 33, nan)):
        v[row, head, d] = x
    k[199, 1] = nan
    start_loc, length = torch.tensor(start[:-1], dtype=torch.int32, device=DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)
    out = F.context_attention(q, k, v, torch.zeros_like(q), start_loc, length, 200)
    general = F.context_attention(q, k, _unaligned(v), torch.zeros_like(q), start_loc, length, 200)
    assert not general.isfinite().all()
    for kind in (torch.isnan, torch.isposinf, torch.isneginf):
        differ = (kind(out) != kind(general)).nonzero()[:8].tolist()
        assert not differ, [(at, float(out[tuple(at)]), float(general[tuple(at)])) for at in differ]
    fine = general.isfinite()
    assert ((out - general).abs()[fine].float() <= 3 * ROUND[dt][0] * general.abs()[fine].float() + 1e-3).all()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 2, 5])
def test_attention_log_sum_exp_near_zero(dt, n):
    """Rows of a few keys with small scores, which are exact in fp32: the log-sum-exp keeps the relative precision of its terms."""
    B = 200
    g = torch.Generator().manual_seed(n)
    q, k = torch.zeros(B * n, 1, 64), torch.zeros(B * n, 1, 64)
    q[:, 0, 0] = 8
    k[:, 0, 0] = torch.randn(B * n, generator=g) * 0.05
    q, k = (t.to(dt).to(DEV) for t in (q, k))
    cu = torch.arange(B + 1, dtype=torch.int32, device=DEV) * n
    F.flash_attention_varlen(q, k, k, cu, cu, None, n, n, 0.0, None, False)
    lse = F.GLOBAL_STATE["flash_attention_varlen_softmax_lse"][:, 0].double()
    s = k[:, 0, 0].double().view(B, n)
    want = s.logsumexp(1, keepdim=True)
    # the reference rounded, and the result; with more than one key their exponents, exponentials, sum and logarithm
    bound = 2.02 * 2.0 ** -24 * (s.abs().amax(1, keepdim=True) + want.abs()) + (6 * 2.0 ** -24 if n > 1 else 0)
    assert ((lse - want).abs() <= bound).all(), float(((lse - want).abs() / bound).max())


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("late", [False, True])
def test_attention_infinite_values_of_keys_that_weigh_little(dt, late):
    """2^-135 of another key's weight, below the normal numbers of fp32, is still something: infinite values stay infinite, whichever key
    comes first."""
    n = 200
    q, k = torch.zeros(n, 1, 64), torch.zeros(n, 1, 64)
    q[:, 0, 0] = 8
    light, heavy = (3, 150) if late else (150, 3)
    k[heavy, 0, 0] = 135 * np.log(2)
    v = torch.randn(n, 1, 64, generator=torch.Generator().manual_seed(12))
    v[light, 0, 5], v[light, 0, 6], v[heavy, 0, 9], v[light + 1, 0, 9] = float("inf"), -float("inf"), float("inf"), -float("inf")
    q, k, v = (t.to(dt).to(DEV) for t in (q, k, v))
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    out = F.flash_attention_varlen(q, k, v, cu, cu, None, n, n, 0.0, None, False)[:, 0]
    assert out[:, 5].isposinf().all() and out[:, 6].isneginf().all() and out[:, 9].isnan().all()
    rest = [d for d in range(64) if d not in (5, 6, 9)]
    assert torch.equal(out[:, rest], v[heavy, 0, rest].expand(n, -1))


@pytest.mark.parametrize("scale", [-0.125, 1e-20])
def test_attention_odd_scales(scale):
    q, k, v, start = _packed([70, 130], 2, 2, torch.float16, 6)
    cu = torch.from_numpy(start.astype(np.int32)).to(DEV)
    out, general = (F.flash_attention_varlen(q, k, t, cu, cu, None, 130, 130, 0.0, scale, True) for t in (v, _unaligned(v)))
    assert ((out - general).abs() <= 3 * 2.0 ** -11 * general.abs() + 1e-3).all()


def test_attention_scale_that_fp32_holds_as_zero():
    """All keys weigh the same, and masked ones nothing."""
    q, k, v, _ = _packed([130], 2, 2, torch.float16, 8)
    q, k, v = (t.view(1, 130, 2, 64) for t in (q, k, v))
    out, general = (F.multihead_attention(q, k, t, 0.0, True, False, 1e-50) for t in (v, _unaligned(v)))
    want = v.double().cumsum(1) / torch.arange(1, 131, device=DEV, dtype=torch.float64).view(1, -1, 1, 1)
    assert ((out.double() - want).abs() <= 2.0 ** -11 * want.abs() + 130 * 2.0 ** -23 * 4 + 2.0 ** -25).all()
    assert ((out - general).abs() <= 2 * 2.0 ** -11 * general.abs() + 1e-4).all()


def test_attention_where_no_plan_can_be_had():
    """The allocation-free entry point with more query tiles than its static plan holds: refused for heads of 128, for heads of 64
    the general kernel takes the call, as it did every one.  From a context the same call takes its plan and the tile kernel."""
    lens = [10490 + i % 3 for i in range(100)]  # 8203 tiles of 128 rows and 100 sequences, against 8192
    total = sum(lens)
    assert (total + 127) // 128 + len(lens) > 8192
    assert (4 * len(lens) + total // 128 + 1) * 4 <= 65536  # what a plan takes in LDS: the tile kernel is not ruled out before
    start = np.concatenate(([0], np.cumsum(lens)))[:-1]
    loc, length = (torch.tensor(t, dtype=torch.int32, device=DEV) for t in (start.tolist(), lens))
    g = torch.Generator(device=DEV).manual_seed(7)
    q, k, v = (torch.randn(total, 1, 64, generator=g, device=DEV).half() for _ in range(3))
    out = F.context_attention_no_alloc(q, k, v, torch.zeros_like(q), loc, length, max(lens))
    want = F.context_attention(q, k, v, torch.zeros_like(q), loc, length, max(lens))
    # both round a result once; before that the scores' fp32 sums, taken in other orders, move it by 2^-14 of values of up to 5
    assert ((out - want).abs() <= 2 * 2.0 ** -11 * want.abs() + 10 * 2.0 ** -14).all()
    assert not torch.equal(out, want)  # two kernels
    wide = torch.zeros(2500 * 304, 1, 128, dtype=torch.float16, device=DEV)
    many = torch.arange(2500, dtype=torch.int32, device=DEV) * 304
    with pytest.raises(rt.DiopiException, match="at most 8192"):
        F.context_attention_no_alloc(wide, wide, wide, torch.zeros_like(wide), many, torch.full_like(many, 304), 304)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("batch,longest", [(33, 300), (64, 300), (64, 20), (100, 300), (40, 1100), (1, 33000)])
def test_attention_over_many_tiles(batch, longest, causal, D):
    """Tiles that the work-groups find (up to 64 sequences, of which the later ones stand in the upper half of a ballot, and 256 tiles)
    and tiles from a table, of lengths in no order, some of them zero or the same."""
    H = 1 if batch == 1 else 3
    lens = [longest] if batch == 1 else [(i * 37) % longest + 1 if i % 7 else (0 if i % 2 else longest) for i in range(batch)]
    g = torch.Generator().manual_seed(batch + D)
    q, k, v = (torch.randn(sum(lens), H, D, generator=g).half().to(DEV) for _ in range(3))
    cu = torch.tensor(np.concatenate(([0], np.cumsum(lens))), dtype=torch.int32, device=DEV)
    call = lambda vv: (F.flash_attention_varlen(q, k, vv, cu, cu, None, longest, longest, 0.0, None, causal), F.GLOBAL_STATE["flash_attention_varlen_softmax_lse"])
    (out, lse), (general, general_lse) = call(v), call(_unaligned(v))
    # heads of 128 round the scaled query and the probabilities to 16 bits: scores of up to 6, values of up to 5
    slack = 2.0 ** -11 * (6 + 1) * 5 if D == 128 else 10 * 2.0 ** -14
    assert ((out - general).abs() <= 2 * 2.0 ** -11 * general.abs() + slack).all()
    assert ((lse - general_lse).abs() <= (6 * 2.0 ** -10 if D == 128 else 1e-5) + 1e-6 * general_lse.abs()).all()
