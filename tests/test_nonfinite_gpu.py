"""NaN and infinities go where the modules have them."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

import ddfnet_amd
import oracle
from ddf_testlib import random_case, run_ddf
from test_net_gpu import Norm, call
from test_plans_gpu import by_modules

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,c', [(2, 16), (3, 64), (20, 256), (2, 512)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_hidden_nan_reaches_the_channel_filter_and_the_gradients(n, c, dtype):
    """A NaN of one sample's features, and of a hidden bias."""
    torch.manual_seed(c)
    layer = ddfnet_amd.DDFPack(c).cuda().to(dtype)
    x = torch.randn(n, c, 6, 4, device='cuda').to(dtype)
    x[1, 3, 2, 2] = float('nan')
    with torch.no_grad():
        out = layer(x)
        assert torch.equal(out.isnan(), by_modules(layer, x).isnan())
        assert out[1].isnan().all() and not out[0].isnan().any()
    leaves = [x.requires_grad_(True)] + list(layer.parameters())
    for poison in (False, True):
        if poison:
            x.data[1, 3, 2, 2] = 0.
            layer.channel_branch[1].bias.data[0] = float('nan')
        outs = [f(x) for f in (layer, lambda y: by_modules(layer, y))]
        assert 'PackAutograd' in outs[0].grad_fn.name()
        go = torch.randn_like(outs[0])
        grads = [torch.autograd.grad(o, leaves, go) for o in outs]
        assert torch.equal(outs[0].isnan(), outs[1].isnan())
        for name, got, want in zip(['x'] + [k for k, _ in layer.named_parameters()], *grads):
            assert torch.equal(got.isnan(), want.isnan()), (poison, name)


@pytest.mark.parametrize('value', [float('inf'), float('-inf'), float('nan')])
def test_stem_keeps_nonfinite_pixels_inside_their_windows(value):
    """The network's 7 x 7 stem against the same in fp64, one such pixel per image."""
    torch.manual_seed(1)
    x = torch.randn(9, 3, 64, 64).half()
    at = [(0, 0), (0, 63), (63, 0), (31, 30), (30, 31), (33, 40), (40, 33), (22, 21), (63, 63)]
    for i, (r, c) in enumerate(at):
        x[i, i % 3, r, c] = value
    w = torch.randn(64, 3, 7, 7).half()
    keep = [torch.rand(64).half().cuda() + 0.5 for _ in range(4)]
    norm = Norm(**dict(zip(('weight', 'bias', 'mean', 'var'), [t.data_ptr() for t in keep])), eps=1e-5)
    out = torch.empty(9, 16, 16, 64, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_stem', x.cuda(), w.cuda(), norm, out, 9, 64, 64)
    y = F.batch_norm(F.conv2d(x.double(), w.double(), stride=2, padding=3), keep[2].cpu().double(),
                     keep[3].cpu().double(), keep[0].cpu().double(), keep[1].cpu().double(), eps=1e-5)
    want = F.max_pool2d(F.relu(y), 3, 2, 1).permute(0, 2, 3, 1)
    got = out.cpu()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,k,d,s', [((8, 66, 61, 85), 3, 1, 1), ((4, 66, 113, 134), 3, 1, 1),
                                         ((2, 16, 60, 131), 3, 2, 1), ((2, 16, 23, 71), 5, 2, 1),
                                         ((3, 37, 11, 131), 3, 1, 2), ((3, 37, 10, 13), 3, 1, 2)])
def test_nonfinite_pixels_over_ragged_rows(shape, k, d, s, combine, dtype):
    """At the ends of rows and planes, where lanes hold what is not theirs: the forward and the
    feature gradient, alone and beside the filters' (whose sums over a plane meet the zeros
    around it, zero times NaN included, in every kernel)."""
    x, cf, sf, go = random_case(*shape, k, s, dtype, seed=k)
    n, c, h, w = shape
    for t in (x, go):
        th, tw = t.shape[2:]
        for i, (y, z) in enumerate([(0, 0), (0, tw - 1), (th - 1, 0), (th - 1, tw - 1), (th // 2, tw - 2), (2, 1)]):
            t[i % n, (3 * i) % c, y, z] = (float('nan'), float('inf'))[i % 2]
    want = (oracle.forward(x, cf, sf, k, d, s, combine),) + tuple(oracle.backward(go, x, cf, sf, k, d, s, combine))
    for need in ((True, False, False), (True, True, True)):
        for name, got, ref in zip(('out', 'dX'), run_ddf(x, cf, sf, go, k, d, s, combine, need=need), want):
            assert torch.equal(got.cpu().isfinite(), ref.isfinite()), (name, need)


@pytest.mark.parametrize('n,c,h,w,s', [(8, 512, 7, 7, 1), (2, 512, 14, 14, 2), (5, 128, 9, 13, 1), (2, 64, 56, 56, 1)])
def test_nonfinite_pixels_in_the_networks_kernels(n, c, h, w, s):
    x, cf, sf, _ = random_case(n, c, h, w, 3, s, torch.float16, seed=c)
    at = [(0, 0), (h - 1, w - 1), (h // 2, w - 1), (1, 0)]
    for i, (y, z) in enumerate(at):
        x[i % n, 5 * i, y, z] = (float('nan'), float('inf'))[i % 2]
    ho, wo = h // s, w // s
    taps = torch.zeros(n, ho * wo, 12, dtype=torch.float16)
    taps[:, :, :9] = sf.reshape(n, 9, ho * wo).permute(0, 2, 1)
    xl = x.permute(0, 2, 3, 1).contiguous().cuda()
    out = torch.empty(n, ho, wo, c, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_filter', xl, cf.cuda(), taps.cuda(), None, out, n, h, w, c, s, 0)
    want = oracle.forward(x, cf, sf, 3, 1, s, 'mul').clamp_min(0)      # (minus infinity: zero)
    assert torch.equal(out.permute(0, 3, 1, 2).cpu().isfinite(), want.isfinite())
    # the spatial branch: a pixel's taps, and the sums of its plane
    ws = torch.randn(9, c).half()
    got, parts, count = torch.empty(n, ho * wo, 12, device='cuda').half(), torch.empty(n * c * 8, device='cuda'), ctypes.c_int()
    call('ddf_hip_net_spatial', xl, ws.cuda(), None, got, parts, ctypes.byref(count), n, h, w, c, s, 0.6)
    sampled = x[:, :, ::s, ::s].isfinite().all(1).reshape(n, 1, -1).expand(n, 9, ho * wo)
    assert torch.equal(got[:, :, :9].permute(0, 2, 1).cpu().isfinite(), sampled)
    sums = parts[:n * count.value * c].view(n, count.value, c).sum(1).cpu()
    assert torch.equal(sums.isfinite(), x.isfinite().all(3).all(2))
    # a product: its pixel's results
    wt = torch.randn(64, c).half().cuda()
    prod = torch.empty(n, h, w, 64, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv', xl, wt, None, None, prod, n, h, w, c, 64, 1, 0)
    assert torch.equal(prod.cpu().isfinite().all(3), x.isfinite().all(1))
