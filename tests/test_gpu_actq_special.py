"""The activation quantisers on values that their integer maxima and short roundings have to get right: NaNs of either sign,
infinities, zeros of either sign, rows without a positive element and rounding ties, at every lane and piece, alone and on
the way into the int8 product of few tokens; against the tensor operations they stand for."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def _negative_nan():
    return torch.tensor([0xFFC1 - 0x10000], dtype=torch.int16).view(torch.bfloat16)


def _x(M, K, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    x[0, : K // 2] = torch.arange(K // 2).sub(K // 4).to(torch.bfloat16) / 2  # ties
    return x


def _per_tensor(x):
    """x8 and clamp value of lq_act_quant_i8_dynamic"""
    c = x.max()
    q = ((x * 127.0) / c).round()
    q = torch.where(torch.isnan(q), torch.zeros_like(q), q).clamp(-128, 127)
    return q.to(torch.int8), c


def _per_token(x):
    xf = x.float()
    am = xf.abs().amax(1)  # NaN if one element is
    inv = torch.where(am == 0, torch.zeros_like(am), torch.full_like(am, 127.0) / am)  # (a number / a tensor is a product)
    q = (xf * inv[:, None]).round()
    return torch.where(torch.isnan(q), torch.zeros_like(q), q).clamp(-128, 127).to(torch.int8), am / 127.0


SPECIALS = ["none", "nan", "negative nan", "inf", "-inf", "all negative", "all zero", "one zero among negatives", "tiny"]


def _special(x, name, at):
    x = x.clone()
    flat = x.view(-1)
    if name == "nan":
        flat[at] = NAN
    elif name == "negative nan":
        flat[at] = _negative_nan()[0]
    elif name in ("inf", "-inf"):
        flat[at] = float(name)
    elif name == "all negative":
        x = -x.abs().clamp(min=2.0 ** -6)
    elif name == "all zero":
        x = torch.zeros_like(x)
    elif name == "one zero among negatives":
        x = -x.abs().clamp(min=2.0 ** -6)
        x.view(-1)[at] = 0.0
    elif name == "tiny":
        x = x * 2.0 ** -130
    return x


@pytest.mark.parametrize("M,K", [(1, 128), (5, 1024), (16, 3968), (3, 8192)])
@pytest.mark.parametrize("name", SPECIALS)
def test_quantisers(hip_lib, M, K, name):
    from latentq_llm_amd import ops
    base = _x(M, K, M + K)
    w = torch.randint(-127, 128, (32, K), generator=torch.Generator().manual_seed(1)).to(torch.int8)
    qs = torch.full((32, 1), 2.0 ** -7, dtype=torch.bfloat16)
    for at in (0, 1, M * K - 1, M * K // 2 + 3):
        x = _special(base, name, at)
        want8, c = _per_tensor(x)
        x8, _, work = ops.act_quant_i8_dynamic(x.cuda())
        cv = work[0].cpu()
        assert (torch.isnan(c) and torch.isnan(cv)) or cv == c.float(), (name, at)
        assert torch.equal(x8.cpu(), want8), (name, at)
        want8t, sxt = _per_token(x)
        x8t, sx = ops.act_quant_i8_per_token(x.cuda())
        assert torch.equal(x8t.cpu(), want8t), (name, at)
        assert torch.equal(torch.nan_to_num(sx.cpu(), nan=-1.0), torch.nan_to_num(sxt, nan=-1.0)), (name, at)
        # on the way into the product: the same codes and scales (bit patterns, except a NaN's)
        for per_token, q, s in ((False, want8, (c.float() * torch.tensor(1.0 / 127.0)).expand(M)), (True, want8t, sxt)):
            y = ops.infer8(x.cuda(), w.cuda(), qs.cuda(), per_token=per_token).cpu()
            acc = (q.double() @ w.double().t()).float()
            ref = ((acc * s[:, None]) * qs.float().view(1, -1)).to(torch.bfloat16)
            assert torch.equal(torch.nan_to_num(y.float(), nan=7.25), torch.nan_to_num(ref.float(), nan=7.25)), (name, at, per_token)


@pytest.mark.parametrize("M,K", [(1, 1), (3, 7), (5, 1021), (10, 8192), (10, 8193), (13, 7867), (60, 7001)])
@pytest.mark.parametrize("name", SPECIALS)
def test_maximum_in_one_launch_and_two(hip_lib, M, K, name):
    """Sizes on both sides of the number of elements up to which every workgroup finds the maximum itself, remainders of eight."""
    from latentq_llm_amd import ops
    base = _x(M, K, M + K) if K > 8 else torch.randn(M, K, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16)
    for at in sorted({0, M * K - 1, M * K // 2}):
        x = _special(base, name, at)
        want8, c = _per_tensor(x)
        x8, sx, work = ops.act_quant_i8_dynamic(x.cuda())
        cv = work[0].cpu()
        assert (torch.isnan(c) and torch.isnan(cv)) or cv == c.float(), (name, at)
        assert torch.equal(x8.cpu(), want8), (name, at)
        alpha = c.float() * torch.tensor(1.0 / 127.0)
        assert torch.equal(torch.nan_to_num(sx.cpu(), nan=-1.0), torch.nan_to_num(alpha.expand(M), nan=-1.0)), (name, at)
