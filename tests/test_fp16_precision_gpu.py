"""fp16 storage where every product and sum is fp32: the result is off by its own rounding and
by fp32 sums, not by a rounded comb(CF, SF).

Bound, per element: half a unit of the stored result, 2^-11 of it (2^-25 below fp16's normal
range), and for ``terms`` fp32 products and additions 2^-23 of the sum of the terms' magnitudes
each (a product rounds once, an addition once).  A combination rounded to fp16 is off by 2^-11
of its term: with terms that cancel it misses the bound by far."""
import pytest
import torch

from ddfnet_amd import _lib
from ddf_testlib import random_case, run_ddf
from test_net_gpu import Norm, call

import oracle

pytestmark = pytest.mark.gpu


def _ids(v):
    return str(v).replace('torch.', '')


def within(got, want, magnitude, terms, stored=0.):
    """stored: magnitudes of intermediate values that are fp16 by design."""
    want, got = want.double(), got.double().cpu()
    bound = 2.0 ** -11 * (want.abs() + stored) + 2.0 ** -25 + terms * 2.0 ** -23 * magnitude.double()
    worst = ((got - want).abs() / bound).max().item()
    assert worst <= 1, worst


def magnitudes(x, cf, sf, go, k, d, s, combine):
    """The sums with every term's magnitude in its place (CF and SF of 'add' apart)."""
    a = [t.abs() for t in (x, cf, sf, go)]
    return (oracle.forward(a[0], a[1], a[2], k, d, s, combine),
            oracle.backward(a[3], a[0], a[1], a[2], k, d, s, combine)[0])


def check(case, k, d, s, combine, need):
    x, cf, sf, go = case
    sum_out, sum_dx = magnitudes(x, cf, sf, go, k, d, s, combine)
    out, dx, _, _ = run_ddf(x, cf, sf, go, k, d, s, combine, need=need)
    within(out, oracle.forward(x, cf, sf, k, d, s, combine), sum_out, 2 * k * k)
    if need[0]:
        within(dx, oracle.backward(go, x, cf, sf, k, d, s, combine)[0], sum_dx, 2 * k * k)


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,k,d,s', [
    ((4, 256, 50, 75), 3, 1, 1),       # odd rows in vectors of four
    ((4, 66, 113, 133), 3, 1, 1),
    ((4, 64, 113, 265), 3, 1, 1),     # ... and cut into segments
    ((2, 64, 49, 75), 3, 1, 2),        # stride 2 over odd planes
    ((2, 64, 50, 78), 3, 1, 2)], ids=_ids)
def test_forward_and_feature_gradient_alone(shape, k, d, s, combine):
    if s == 1:
        assert 'ragged' in _lib.describe(shape, k, d, s, combine, torch.float16)
    check(random_case(*shape, k, s, torch.float16, seed=sum(shape)), k, d, s, combine, (True, False, False))


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,d', [
    ((4, 256, 50, 75), 1),             # odd rows
    ((16, 64, 57, 58), 1),             # even ones of an odd number of pairs, an odd number of them
    ((4, 66, 113, 134), 1),            # ... cut into segments
    ((2, 16, 60, 131), 2),             # dilated
    ((2, 16, 60, 130), 2)], ids=_ids)
def test_feature_gradient_with_the_filters(shape, d, combine):
    assert 'ragged' in _lib.describe(shape, 3, d, 1, combine, torch.float16, need=7)
    case = random_case(*shape, 3, 1, torch.float16, seed=sum(shape))
    _, magnitude = magnitudes(*case, 3, d, 1, combine)
    x, cf, sf, go = case
    _, dx, _, _ = run_ddf(x, cf, sf, go, 3, d, 1, combine)
    within(dx, oracle.backward(go, x, cf, sf, 3, d, 1, combine)[0], magnitude, 18)


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('n,c,h,w,s', [(8, 512, 7, 7, 1), (8, 512, 14, 14, 2), (2, 64, 5, 9, 1), (3, 128, 11, 3, 1),
                                       (2, 256, 6, 10, 2)], ids=_ids)
def test_channels_last_filter_over_odd_rows(n, c, h, w, s, combine):
    """The network's own kernel of the operator, nothing behind it but its ReLU."""
    x, cf, sf, _ = random_case(n, c, h, w, 3, s, torch.float16, seed=c + w)
    ho, wo = h // s, w // s
    taps = torch.zeros(n, ho * wo, 12, dtype=torch.float16)
    taps[:, :, :9] = sf.reshape(n, 9, ho * wo).permute(0, 2, 1)
    out = torch.empty(n, ho, wo, c, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_filter', x.permute(0, 2, 3, 1).contiguous().cuda(), cf.cuda(), taps.cuda(), None, out, n, h, w,
         c, s, _lib.COMBINE[combine])
    a = [t.abs() for t in (x, cf, sf)]
    want, magnitude = oracle.forward(x, cf, sf, 3, 1, s, combine), oracle.forward(*a, 3, 1, s, combine)
    within(out.permute(0, 3, 1, 2), want.clamp_min(0), magnitude, 18)


@pytest.mark.parametrize('n,c,o,residual', [
    (1, 64, 10, False), (3, 128, 33, True),              # few pixels: 16 x 16 results per workgroup
    (300, 64, 136, False), (300, 128, 64, True), (6000, 64, 200, False)], ids=_ids)   # tiles
def test_bias_without_a_norm_is_part_of_the_sum(n, c, o, residual):
    """The classifier's product: sums that its bias takes back to small values."""
    g = torch.Generator().manual_seed(n)
    x, w = torch.rand(n, c, generator=g).half() + 1, torch.rand(o, c, generator=g).half() + 1
    sums = x.double() @ w.double().t()
    bias = -sums.mean(0).half()
    res = torch.randn(n, o, generator=g).half() if residual else None
    keep = bias.cuda()
    out = torch.empty(n, o, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv', x.cuda(), w.cuda(), Norm(conv_bias=keep.data_ptr()), None if res is None else res.cuda(),
         out, n, 1, 1, c, o, 1, 0)
    want = sums + bias.double() + (0 if res is None else res.double())
    # (with a residual the tiles hand the sum on as fp16: one more rounding, of the sum)
    within(out, want, (sums + bias.double().abs()), c + 1, (sums + bias.double()).abs() * bool(residual))


def test_bias_without_a_norm_beside_a_projection():
    g = torch.Generator().manual_seed(9)
    n, c, side, o = 300, 64, 128, 256
    x, w = torch.rand(n, c, generator=g).half() + 1, torch.rand(o, c, generator=g).half() + 1
    xs, ws = torch.rand(n, side, generator=g).half() + 1, torch.rand(o, side, generator=g).half() + 1
    sums, sides = x.double() @ w.double().t(), xs.double() @ ws.double().t()
    b, bs = -sums.mean(0).half(), -sides.mean(0).half()
    db, dbs = b.cuda(), bs.cuda()
    out = torch.empty(n, o, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv_pair', x.cuda(), w.cuda(), Norm(conv_bias=db.data_ptr()), c, xs.cuda(), ws.cuda(),
         Norm(conv_bias=dbs.data_ptr()), 1, 1, side, 1, out, n, o, 0)
    want, want_side = sums + b.double(), sides + bs.double()
    # (both sums are fp16 before their biases, as two convolutions' results are, and the projection's
    # result is)
    within(out, want + want_side, sums + sides + b.double().abs() + bs.double().abs(), c + side + 2,
           sums + sides + want_side.abs())
