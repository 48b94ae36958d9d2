"""The arithmetic behind the fp32 kernels' bf16 planes (csrc/tt_planes.h): the
split x = h + m + l and the six plane products, restated on the CPU."""
import pytest
import torch


def _split(x):
    h = x.bfloat16().float()
    m = (x - h).bfloat16().float()
    return h, m, (x - h - m).bfloat16().float()


def _random(n, lo, hi, seed):
    """n random floats with magnitudes of 2^lo .. 2^hi, either sign."""
    g = torch.Generator().manual_seed(seed)
    e = torch.randint(lo, hi, (n,), generator=g)
    s = torch.randint(0, 2, (n,), generator=g) * 2 - 1
    return torch.ldexp(1.0 + torch.rand(n, generator=g), e) * s


def test_split_is_exact():
    """All 24 bits from 2^-110 up to bf16's rounding to infinity (3.389e38);
    below, what the planes miss is at most half of bf16's smallest step, 2^-134."""
    x = torch.cat([_random(1 << 20, -110, 127, 0), torch.tensor([3.3895e38 * 0.9999, -3.38e38, 2.0 ** -110, 0.0])])
    assert torch.equal(sum(p.double() for p in _split(x)), x.double())
    tiny = _random(1 << 16, -140, -110, 1)
    assert (sum(p.double() for p in _split(tiny)) - tiny.double()).abs().max() <= 2.0 ** -134
    for v in (float("inf"), -float("inf"), float("nan"), 3.4e38):
        assert not torch.isfinite(sum(_split(torch.tensor([v])))).any()


@pytest.mark.parametrize("seed", [0, 1])
def test_six_products(seed):
    """The dropped m l + l m + l l stay below 2^-24 (1 + 2^-9) of the product,
    one unit roundoff of fp32, and near 2^-27.5 of it in the root mean square;
    the bound is reached to within 1 % by 1 + 2^-8 - 2^-17 squared."""
    x, y = _random(1 << 21, 0, 1, 2 * seed), _random(1 << 21, 0, 1, 2 * seed + 1)
    edge = torch.tensor([1.0 + 2.0 ** -8 - 2.0 ** -17])
    x, y = torch.cat([x, edge]), torch.cat([y, edge])
    (xh, xm, xl), (yh, ym, yl) = ([p.double() for p in _split(t)] for t in (x, y))
    six = xh * yh + (xh * ym + xm * yh) + (xm * ym + xh * yl + xl * yh)
    rel = ((x.double() * y.double() - six) / (x.double() * y.double())).abs()
    assert rel.max() <= 2.0 ** -24 * (1 + 2.0 ** -9)
    assert rel[-1] >= 0.99 * 2.0 ** -24
    assert 2.0 ** -28 < rel.square().mean().sqrt() < 2.0 ** -27
