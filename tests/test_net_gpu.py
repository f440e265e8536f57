"""The channels-last fp16 kernels of the DDF-ResNets' inference, each against plain PyTorch in
fp32 on the same fp16 values, and the whole network against its modules."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

import ddfnet_amd
from ddfnet_amd import _lib, ddf_resnet

pytestmark = pytest.mark.gpu


class Norm(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ('weight', 'bias', 'mean', 'var', 'conv_bias')] + [('eps', ctypes.c_float)]


def make_norm(c, bn, bias):
    t = {}
    if bn:
        t = {'weight': torch.rand(c) + 0.5, 'bias': torch.randn(c) * 0.2, 'mean': torch.randn(c) * 0.2,
             'var': torch.rand(c) + 0.5}
    if bias:
        t['conv_bias'] = torch.randn(c)
    t = {k: v.half().cuda() for k, v in t.items()}
    norm = Norm(**{k: v.data_ptr() for k, v in t.items()}, eps=1e-5)

    def apply(y):   # y (..., c) fp32
        if bias:
            y = y + t['conv_bias'].float()
        if bn:
            y = (y - t['mean'].float()) / torch.sqrt(t['var'].float() + 1e-5) * t['weight'].float() + t['bias'].float()
        return y
    return norm, apply, t


def call(name, *args):
    conv = [ctypes.c_void_p(a.data_ptr()) if torch.is_tensor(a) else ctypes.byref(a) if isinstance(a, Norm) else a
            for a in args]
    _lib.check(getattr(_lib.lib(), name)(*conv, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))


def close(got, want, tol):
    err = (got.float() - want.float()).abs().max().item() / want.float().abs().max().item()
    assert torch.isfinite(got).all() and err <= tol, err


@pytest.mark.parametrize('n,h,w,c,o,stride,bn,bias,res,relu', [
    (1, 1, 1, 64, 10, 1, 0, 1, 0, 0),          # the classifier: one row, channels no multiple of 8
    (3, 5, 7, 64, 64, 1, 1, 0, 0, 1),          # one step of K, rows past the end of a tile
    (2, 7, 7, 2048, 512, 1, 1, 0, 0, 1),       # few pixels, long rows: waves split K
    (1, 14, 14, 256, 1024, 1, 1, 1, 1, 1),
    (9, 56, 56, 64, 256, 1, 1, 0, 1, 1),       # tiles of 128 x 128
    (33, 28, 28, 256, 64, 1, 1, 0, 0, 1),      # 64 channels
    (21, 28, 28, 128, 72, 1, 1, 0, 1, 0),      # channels past a tile
    (8, 28, 28, 192, 136, 1, 0, 1, 0, 1),      # three steps of K
    (5, 28, 30, 256, 512, 2, 1, 0, 0, 0),      # projection under stride 2
    (40, 56, 56, 256, 512, 2, 1, 0, 0, 0),
    (16, 28, 28, 128, 264, 1, 1, 0, 1, 1),     # tiles of 128 x 64, channels past the last
    (42, 56, 56, 64, 136, 1, 1, 1, 0, 1),      # 2058 tiles of 128 x 128 in short stages
    (3, 7, 7, 2112, 520, 1, 1, 0, 1, 1),       # 330 tiles of 16 x 16, 33 blocks of K
    (10, 8, 8, 2112, 520, 1, 1, 0, 1, 1), (20, 8, 8, 2112, 1000, 1, 1, 0, 1, 1),    # tiles of 64, 33 stages of K: 90 of them; 320
    (1, 5, 7, 576, 200, 1, 1, 1, 1, 1),        # K split over the waves: 9 blocks, rows and channels past a tile
    (17, 1, 1, 64, 33, 1, 0, 1, 0, 1),         # one block of K
    (1, 13, 9, 1088, 31, 2, 1, 0, 0, 0),       # 17 blocks, under stride 2
    (1, 16, 16, 192, 4096, 1, 1, 0, 0, 1), (1, 1, 257, 320, 4096, 1, 1, 0, 1, 1),    # 256 tiles of 64, three stages; 320, five
    (20, 4, 8, 1024, 256, 1, 1, 0, 1, 1), (10, 8, 8, 2048, 1000, 1, 0, 1, 0, 0),     # 160 of 32 x 32; 160 of 64, a workgroup per unit
    (1, 16, 32, 128, 256, 1, 1, 0, 1, 1), (1, 27, 19, 128, 256, 1, 1, 0, 1, 1),      # 512 tiles of 16 x 16; 528, and K short: of 64
    (1, 16, 16, 64, 256, 1, 1, 1, 0, 0), (1, 16, 17, 64, 256, 1, 1, 1, 0, 0),        # 256 of a K of 64; 272
    (1, 16, 16, 320, 1024, 1, 1, 0, 1, 1), (1, 1, 257, 320, 1024, 1, 1, 0, 1, 1),    # 256 tiles of 32 x 32, five blocks of K; 288: of 64
    (3, 25, 26, 576, 264, 2, 1, 1, 1, 1), (10, 8, 8, 2048, 520, 1, 0, 1, 0, 0),      # 32 x 32 under stride 2, channels past a tile; no BatchNorm
    (1, 64, 65, 64, 33, 1, 1, 0, 1, 1),        # 780 tiles of 16 x 16, channels no multiple of 8
    # 128 x 128 in three stages, a workgroup per unit: one, two, three and seventeen stages of K, rows and channels past a tile; 592: 128 x 64
    (1, 129, 163, 64, 128, 1, 1, 0, 1, 1), (1, 129, 163, 128, 128, 1, 0, 1, 0, 0), (1, 90, 120, 192, 136, 1, 1, 0, 1, 1),
    (1, 65, 128, 1088, 256, 1, 1, 0, 0, 1), (1, 172, 220, 192, 256, 1, 1, 0, 1, 1),
    # 1536 tiles of 128 x 128: a short K in short stages, a long one or a residual by eight waves
    (1, 256, 256, 704, 264, 1, 1, 0, 0, 1), (1, 241, 272, 832, 264, 1, 1, 0, 0, 1), (1, 241, 272, 320, 264, 1, 1, 0, 1, 1),
])
def test_conv(n, h, w, c, o, stride, bn, bias, res, relu):
    torch.manual_seed(c + o)
    x = torch.randn(n, h, w, c, device='cuda').half()
    wt = (torch.randn(o, c, device='cuda') * c ** -0.5).half()
    norm, apply, keep = make_norm(o, bn, bias)
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    r = torch.randn(n, ho, wo, o, device='cuda').half() if res else None
    want = apply(x[:, ::stride, ::stride].reshape(-1, c).float() @ wt.float().t()).reshape(n, ho, wo, o)
    want = want + r.float() if res else want
    want = want.clamp_min(0) if relu else want
    out = r if res else torch.empty(n, ho, wo, o, device='cuda', dtype=torch.float16)   # (in place where it may be)
    call('ddf_hip_net_conv', x, wt, norm, r, out, n, h, w, c, o, stride, relu)
    close(out, want, 3e-3)


@pytest.mark.parametrize('n,h,w,c,side,o,stride,relu', [
    (3, 5, 7, 64, 64, 64, 1, 1),               # a stage of K each, one tile
    (5, 9, 13, 64, 192, 136, 2, 0),            # tiles of 16 x 16, rows and channels past one
    (1, 14, 14, 512, 1024, 2048, 2, 1),        # few pixels, long rows: 512 tiles of 16 x 16
    (8, 28, 28, 256, 512, 1024, 2, 1),         # tiles of 64
    (16, 28, 28, 128, 256, 264, 1, 1),         # 128 x 64
    (42, 56, 56, 64, 64, 136, 1, 1),           # 128 x 128, 2058: short stages
    (27, 56, 56, 128, 256, 512, 2, 1),         # 128 x 128, 664 tiles
    (7, 45, 44, 64, 64, 264, 1, 1),            # 327 tiles, rows and channels past the last: a stage of K each
    (64, 16, 16, 64, 192, 2048, 2, 0),         # 512, one stage and three
    (26, 56, 55, 192, 128, 520, 2, 1),         # 800, three and two
    (21, 31, 33, 320, 256, 640, 1, 1),         # 840, five and four
    (42, 56, 56, 128, 64, 64, 1, 1),           # 128 x 64, 1029: short stages
    (5, 9, 13, 192, 64, 133, 2, 0),            # channels no multiple of 8
    (3, 25, 26, 128, 320, 264, 2, 1), (2, 17, 16, 64, 256, 520, 1, 0),    # tiles of 32 x 32, a wave with both products; of 64, channels past a tile
    (1, 520, 516, 64, 64, 64, 2, 1),           # 128 x 64, 67080 pixels: too many for a division by multiplying
    # 128 x 128 in three stages: one and one of K, two and three, fourteen and three; 596 tiles: 128 x 64
    (7, 45, 44, 64, 64, 256, 1, 1), (28, 45, 44, 128, 192, 136, 2, 0), (5, 40, 42, 896, 192, 256, 1, 1), (16, 68, 70, 128, 64, 512, 2, 1),
])
def test_conv_pair(n, h, w, c, side, o, stride, relu):
    torch.manual_seed(c + o)
    ho, wo = (h - 1) // stride + 1, (w - 1) // stride + 1
    xs = torch.randn(n, h, w, side, device='cuda').half()
    x = torch.randn(n, ho, wo, c, device='cuda').half()
    wt, ws = ((torch.randn(o, k, device='cuda') * k ** -0.5).half() for k in (c, side))
    norm, apply, keep = make_norm(o, 1, 1)
    norm_s, apply_s, keep_s = make_norm(o, 1, 0)
    want = apply(x.reshape(-1, c).float() @ wt.float().t()) + \
        apply_s(xs[:, ::stride, ::stride].reshape(-1, side).float() @ ws.float().t())
    want = (want.clamp_min(0) if relu else want).reshape(n, ho, wo, o)
    out = torch.empty(n, ho, wo, o, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv_pair', x, wt, norm, c, xs, ws, norm_s, h, w, side, stride, out, n, o, relu)
    close(out, want, 3e-3)


@pytest.mark.parametrize('n,c,side,o,once', [
    (40, 64, 192, 96, 1), (600, 128, 320, 264, 1),                              # tiles of 16 x 16, of 32 x 32
    (1200, 64, 256, 520, 0), (5000, 128, 64, 1000, 0), (3000, 512, 512, 1000, 0),      # of 64, of 128 x 128, in three stages
    (9600, 64, 128, 1000, 0), (33000, 64, 64, 1000, 0), (132000, 64, 128, 64, 0),      # of 128 x 64, of 128 x 128 in short stages, of 128 x 64 in those
])
def test_conv_pair_without_batchnorm(n, c, side, o, once):
    """In small tiles a bias joins the fp32 sum: each product is rounded once, and their sum once (2^-11 of it each).  Larger ones
    round a product's sum in front of its bias as well."""
    torch.manual_seed(c + o)
    x, xs = (torch.randn(n, 1, 1, k, device='cuda').half() for k in (c, side))
    wt, ws = ((torch.randn(o, k, device='cuda') * k ** -0.5).half() for k in (c, side))
    (norm, _, keep), (norm_s, _, keep_s) = (make_norm(o, 0, 1) for _ in range(2))
    sum_a, sum_b = x.view(n, c).double() @ wt.double().t(), xs.view(n, side).double() @ ws.double().t()
    a, b = sum_a + keep['conv_bias'].double(), sum_b + keep_s['conv_bias'].double()
    out = torch.empty(n, o, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv_pair', x, wt, norm, c, xs, ws, norm_s, 1, 1, side, 1, out, n, o, 0)
    rounded = a.abs() + b.abs() if once else sum_a.abs() + sum_b.abs() + b.abs()
    bound = (rounded + (a + b).abs()) * 2.0 ** -11 + 1e-4    # (and the fp32 sums)
    assert ((out.double() - a - b).abs() <= bound).all()


@pytest.mark.parametrize('n,h,w', [(1, 32, 32), (2, 64, 96), (3, 40, 36), (70, 64, 64)])
def test_stem(n, h, w):
    torch.manual_seed(h)
    x = torch.randn(n, 3, h, w, device='cuda').half()
    wt = (torch.randn(64, 3, 7, 7, device='cuda') * 0.1).half()
    norm, apply, keep = make_norm(64, 1, 1)
    y = apply(F.conv2d(x.float(), wt.float(), stride=2, padding=3).permute(0, 2, 3, 1)).clamp_min(0)
    want = F.max_pool2d(y.permute(0, 3, 1, 2), 3, 2, 1).permute(0, 2, 3, 1)
    out = torch.empty(want.shape, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_stem', x, wt, norm, out, n, h, w)
    close(out, want, 3e-3)


def test_stem_takes_images_at_any_address_and_keeps_what_is_not_finite_local():
    """Pairs of columns from an odd element on; the window's idle column holds an infinity."""
    torch.manual_seed(0)
    x = torch.randn(2, 3, 36, 44, device='cuda').half()
    wt = (torch.randn(64, 3, 7, 7, device='cuda') * 0.1).half()
    norm, apply, keep = make_norm(64, 1, 1)
    out, odd_out = (torch.empty(2, 9, 11, 64, device='cuda', dtype=torch.float16) for _ in range(2))
    call('ddf_hip_net_stem', x, wt, norm, out, 2, 36, 44)
    odd = torch.empty(x.numel() + 1, device='cuda', dtype=torch.float16)[1:].view(x.shape).copy_(x)
    call('ddf_hip_net_stem', odd, wt, norm, odd_out, 2, 36, 44)
    assert torch.equal(odd_out, out)
    x[0, 1, 17, 20] = float('inf')     # under the convolution results of columns 9 .. 11
    reached = torch.zeros(2, 1, 36, 44)
    reached[0, 0, 17, 20] = 1
    reached = F.max_pool2d(F.max_pool2d(F.pad(reached, (3, 3, 3, 3)), 7, 2), 3, 2, 1)[:, 0] > 0
    call('ddf_hip_net_stem', x, wt, norm, odd_out, 2, 36, 44)
    same = (odd_out == out).all(-1).cpu()
    assert same[~reached].all() and not same[reached].any()


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('n,h,w,c,s', [(2, 56, 56, 64, 1), (1, 2, 2, 512, 1), (3, 7, 7, 512, 1), (5, 9, 13, 128, 1),
                                       (2, 14, 14, 256, 1), (2, 4, 6, 256, 2), (1, 28, 28, 128, 2), (3, 14, 14, 512, 2),
                                       (2, 12, 10, 64, 2), (70, 14, 14, 256, 1)])
def test_filter_and_spatial_branch(n, h, w, c, s, combine):
    torch.manual_seed(h * w + c)
    x = torch.randn(n, c, h, w, device='cuda').half()
    ws = (torch.randn(9, c, device='cuda') * c ** -0.5).half()
    bs = torch.randn(9, device='cuda').half()
    ho, wo = h // s, w // s
    xl = x.permute(0, 2, 3, 1).contiguous()
    sf = torch.empty(n, ho * wo, 12, device='cuda', dtype=torch.float16)
    parts = torch.empty(n * c * 8, device='cuda')
    count = ctypes.c_int(0)
    call('ddf_hip_net_spatial', xl, ws, bs, sf, parts, ctypes.byref(count), n, h, w, c, s, 0.6)
    raw = F.conv2d(x.float(), ws.float().view(9, c, 1, 1), bs.float(), stride=s)
    want = (raw - raw.mean(1, keepdim=True)) / (raw.std(1, keepdim=True) + 1e-10) * 0.6
    taps = sf[:, :, :9].permute(0, 2, 1).reshape(n, 9, ho, wo)
    close(taps, want, 4e-3)
    total = parts[:n * count.value * c].view(n, count.value, c).double().sum(1)
    assert (total - x.double().sum((2, 3))).abs().max() <= 1e-5 * x.double().abs().sum((2, 3)).max()
    cf = torch.randn(n, c, 3, 3, device='cuda').half()
    norm, apply, keep = make_norm(c, 1, 0)
    out = torch.empty(n, ho, wo, c, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_filter', xl, cf, sf, norm, out, n, h, w, c, s, _lib.COMBINE[combine])
    y = ddfnet_amd.ddf(x.double(), cf.double(), taps.double().contiguous(), 3, 1, s, combine)
    close(out, apply(y.permute(0, 2, 3, 1).float()).clamp_min(0), 4e-3)


@pytest.mark.parametrize('build,n,size,classes', [('ddf_mul_resnet50', 2, 64, 10), ('ddf_add_resnet50', 3, 96, 1000),
                                                  ('ddf_mul_resnet101', 1, 128, 1000), ('ddf_mul_resnet50', 40, 224, 1000)])
def test_network_matches_its_modules(build, n, size, classes):
    torch.manual_seed(n)
    model = getattr(ddf_resnet, build)(num_classes=classes, zero_init_last_bn=False).cuda()
    for m in model.modules():
        if isinstance(m, torch.nn.BatchNorm2d):
            torch.nn.init.uniform_(m.weight, 0.5, 1.5)
            torch.nn.init.uniform_(m.bias, -0.2, 0.2)
            m.running_mean.uniform_(-0.1, 0.1)
            m.running_var.uniform_(0.5, 1.5)
    model = model.half().eval()
    x = torch.randn(n, 3, size, size, device='cuda').half()
    with torch.no_grad():
        assert ddfnet_amd.functional.extension().net_forward(
            model._native_plan(ddfnet_amd.functional.extension()), x) is not None
        out = model(x)
        modules = lambda net, y: net.fc(net.global_pool(net.forward_features(y)).flatten(1))
        by_modules = modules(model, x).float()
        want = modules(model.float(), x.float())
        assert out.shape == (n, classes)
        off = lambda y: ((y.float() - want).norm() / want.norm()).item()
        # (fp16 over so many layers is as far off as it is: not farther than the modules are)
        most = max(4e-3, 1.3 * off(by_modules))
        assert off(out) <= most
        folded = ddf_resnet.fold_batchnorm(model).half()
        assert folded._native_plan(ddfnet_amd.functional.extension()) is not None
        assert off(folded(x)) <= 1.5 * most
        # a change of any kind is seen: a parameter's values, a hook, train mode
        model = model.half()
        model.fc.weight.zero_()
        assert torch.equal(model(x), model.fc.bias.expand(n, -1))
        calls = []
        handle = model.layer2[0].act1.register_forward_hook(lambda *a: calls.append(1))
        model(x)
        handle.remove()
        assert calls == [1]


@pytest.mark.parametrize('n,h,w,c,o', [
    (1, 1, 1, 64, 64),                          # one pixel
    (5, 7, 7, 64, 64), (3, 5, 7, 512, 512),     # samples that end inside tiles of 16 rows
    (1, 14, 14, 1024, 256), (2, 14, 14, 1024, 256),
    (9, 28, 28, 64, 128), (33, 28, 28, 256, 64), (16, 28, 28, 128, 264), (42, 56, 56, 64, 136),
    (200, 14, 14, 256, 520), (1, 56, 56, 256, 72), (42, 56, 56, 64, 64), (20, 4, 8, 1024, 256),
    (5, 11, 11, 320, 264), (50, 3, 4, 576, 264), (3, 16, 16, 2048, 264), (7, 13, 9, 128, 65),    # 32 x 32, samples ending inside; 16 x 16
    (1, 260, 258, 64, 64),                      # 67080 pixels: too many for a division by multiplying
    (110, 14, 14, 192, 128), (45, 14, 14, 1024, 264), (7, 41, 43, 64, 136),    # 128 x 128 in three stages
    (99, 14, 14, 256, 520),                     # 760 of them in two
])
def test_conv_pool(n, h, w, c, o):
    """The results of conv, and their sums over the pixels, slot by slot of the tiles."""
    torch.manual_seed(c + o)
    x = torch.randn(n, h, w, c, device='cuda').half()
    wt = (torch.randn(o, c, device='cuda') * c ** -0.5).half()
    norm, apply, keep = make_norm(o, 1, 1)
    want, out = (torch.empty(n, h, w, o, device='cuda', dtype=torch.float16) for _ in range(2))
    call('ddf_hip_net_conv', x, wt, norm, None, want, n, h, w, c, o, 1, 1)
    count = _lib.lib().ddf_hip_net_conv_pool_parts(n, h, w, c, o)
    parts = torch.full((n, count + 1, o), float('nan'), device='cuda')
    call('ddf_hip_net_conv_pool', x, wt, norm, out, parts, n, h, w, c, o, 1)
    assert torch.equal(out, want) and parts.view(-1)[n * count * o:].isnan().all()
    total = parts.view(-1)[:n * count * o].view(n, count, o).double().sum(1)
    # (fp32 sums of at most h * w terms of one sign)
    assert (total - want.double().sum((1, 2))).abs().max() <= 1e-6 * want.double().abs().sum((1, 2)).max() + 1e-30


@pytest.mark.parametrize('n,h,w,c,side,o,next_o,bn', [
    (8, 56, 56, 64, 0, 256, 64, 1), (29, 47, 49, 64, 0, 256, 64, 1),       # samples that end inside tiles
    (21, 56, 56, 64, 64, 256, 64, 1), (3, 151, 149, 64, 64, 64, 64, 1),    # a projection; one chunk
    (70, 31, 31, 64, 0, 192, 128, 1), (84, 28, 28, 128, 0, 512, 128, 1),
    (60, 28, 28, 128, 0, 512, 256, 1), (1, 199, 199, 128, 0, 128, 256, 1),
    (1100, 8, 8, 64, 0, 256, 64, 0), (70000, 1, 1, 128, 0, 128, 128, 0),   # folded BatchNorm; samples of a tile, of a pixel
    (700, 6, 6, 64, 64, 128, 64, 0),
    (8, 56, 56, 64, 0, 1088, 64, 1), (29, 21, 23, 64, 64, 2048, 64, 1), (27, 28, 28, 128, 0, 2048, 256, 0),    # wide ones past 1024
])
def test_conv_chain(n, h, w, c, side, o, next_o, bn):
    """The two convolutions of one launch: what the two calls leave, and the sums over the pixels."""
    torch.manual_seed(c + o + next_o)
    x = torch.randn(n, h, w, c, device='cuda').half()
    wt, ws, wn = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((o, c), (o, side or 1), (next_o, o)))
    norm, _, keep = make_norm(o, bn, 1)
    norm_s, _, keep_s = make_norm(o, bn, 1)
    norm_n, _, keep_n = make_norm(next_o, bn, 1)
    xs = torch.randn(n, h, w, side, device='cuda').half() if side else None
    res = None if side else torch.randn(n, h, w, o, device='cuda').half()
    want = torch.empty(n, h, w, o, device='cuda', dtype=torch.float16)
    if side:
        call('ddf_hip_net_conv_pair', x, wt, norm, c, xs, ws, norm_s, h, w, side, 1, want, n, o, 1)
    else:
        call('ddf_hip_net_conv', x, wt, norm, res, want, n, h, w, c, o, 1, 1)
    want_next = torch.empty(n, h, w, next_o, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_conv', want, wn, norm_n, None, want_next, n, h, w, o, next_o, 1, 1)
    count = _lib.lib().ddf_hip_net_conv_chain_parts(n, h, w, c, side, o, next_o)
    assert count > 0
    parts = torch.full((n, count + 1, next_o), float('nan'), device='cuda')
    out = torch.empty_like(want) if side else res     # (in place where it may be)
    got_next = torch.empty_like(want_next)
    call('ddf_hip_net_conv_chain', x, wt, norm, res, xs, ws if side else None, norm_s if side else None, side, out, wn, norm_n,
         got_next, parts, n, h, w, c, o, next_o)
    assert torch.equal(out, want)
    # (a bias without a BatchNorm joins the sum last instead of first: a rounding of fp32 below one of fp16)
    close(got_next, want_next, 0 if bn else 1e-3)
    assert parts.view(-1)[n * count * next_o:].isnan().all()
    total = parts.view(-1)[:n * count * next_o].view(n, count, next_o).double().sum(1)
    # (fp32 sums of at most h * w terms of one sign)
    assert (total - got_next.double().sum((1, 2))).abs().max() <= 1e-6 * got_next.double().abs().sum((1, 2)).max() + 1e-30


@pytest.mark.parametrize('n,h,w,c,side,o,next_o,combine,bn', [
    (8, 56, 56, 64, 0, 256, 64, 0, 1), (9, 55, 52, 64, 0, 256, 64, 1, 1),          # samples that end inside tiles
    (21, 56, 56, 64, 64, 256, 64, 0, 1), (70, 33, 28, 64, 0, 192, 128, 1, 0),      # a projection; no BatchNorm
    (84, 28, 28, 128, 0, 512, 128, 0, 1), (32, 28, 28, 128, 0, 128, 256, 1, 1),
    (4, 56, 56, 64, 64, 64, 64, 0, 1),                                              # fewest tiles
    (1, 1, 24804, 64, 0, 64, 64, 0, 1), (2, 4100, 4, 64, 64, 64, 64, 0, 1),        # one row (no fused launch: None), rows of one run
    (3100, 2, 4, 128, 0, 64, 128, 0, 1), (1, 7, 4096, 64, 0, 64, 128, 1, 1),       # samples of a lane's pixels; the widest rows
    (5, 53, 52, 64, 64, 1088, 64, 0, 1), (27, 28, 28, 128, 0, 2048, 256, 1, 0),    # wide channels past 1024
])
def test_filter_chain(n, h, w, c, side, o, next_o, combine, bn):
    """The spatial branch and the filter in front of the chain's launch: what the three calls leave, to the bit."""
    torch.manual_seed(c + o + next_o + w)
    x = torch.randn(n, h, w, c, device='cuda').half()
    cf = torch.randn(n, c, 9, device='cuda').half()
    tap_w, tap_b = (torch.randn(9, c, device='cuda') * c ** -0.5).half(), torch.randn(9, device='cuda').half() if bn else None
    wt, ws, wn = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((o, c), (o, side or 1), (next_o, o)))
    (norm_f, _, keep_f), (norm, _, keep), (norm_s, _, keep_s), (norm_n, _, keep_n) = (make_norm(k, bn, 1) for k in (c, o, o, next_o))
    xs = torch.randn(n, h, w, side, device='cuda').half() if side else None
    res = None if side else torch.randn(n, h, w, o, device='cuda').half()
    count = _lib.lib().ddf_hip_net_filter_chain_parts(n, h, w, c, side, o, next_o)
    assert (count > 0) == (w <= 4096) and _lib.lib().ddf_hip_net_filter_chain_parts(n, h, w + 2, c, side, o, next_o) == 0
    if not count:
        return
    filtered, sf = torch.empty_like(x), torch.empty(n, h * w, 12, device='cuda', dtype=torch.float16)
    sums, n_sums = torch.empty(n, 1, c, device='cuda'), ctypes.c_int(0)
    call('ddf_hip_net_spatial', x, tap_w, tap_b, sf, sums, ctypes.byref(n_sums), n, h, w, c, 1, 0.7)
    call('ddf_hip_net_filter', x, cf, sf, norm_f, filtered, n, h, w, c, 1, combine)

    def outputs():
        return (res.clone() if res is not None else torch.empty(n, h, w, o, device='cuda', dtype=torch.float16),
                torch.empty(n, h, w, next_o, device='cuda', dtype=torch.float16),
                torch.full((n, count + 1, next_o), float('nan'), device='cuda'))
    want, got = outputs(), outputs()
    for (out, nxt, parts), filters in ((want, None), (got, (cf, tap_w, tap_b, 0.7, norm_f, combine))):
        call('ddf_hip_net_filter_chain' if filters else 'ddf_hip_net_conv_chain', x if filters else filtered, *(filters or ()), wt,
             norm, None if side else out, xs, ws if side else None, norm_s if side else None, side, out, wn, norm_n, nxt, parts,
             n, h, w, c, o, next_o)
    for g, v in zip(got, want):
        assert torch.equal(g.nan_to_num(nan=-7.), v.nan_to_num(nan=-7.))


@pytest.mark.parametrize('n,h,w,c,side,o,next_o,filtered', [
    (1, 1, 12289, 64, 0, 256, 64, 0), (5, 47, 53, 64, 64, 256, 64, 0),        # a last tile of one pixel, of 39
    (3, 79, 52, 64, 0, 64, 128, 0), (1, 1, 18305, 128, 0, 512, 128, 0), (9, 47, 49, 128, 0, 128, 256, 0),     # 36, 1, 119
    (9, 55, 52, 64, 0, 256, 64, 1), (1, 53, 236, 64, 64, 256, 64, 1),         # 12, 92
    (1, 1, 4100 * 3, 64, 0, 64, 128, 0), (1, 3073, 4, 64, 0, 256, 128, 1),    # 12, 4
    (1, 4577, 4, 128, 0, 512, 128, 1), (23, 33, 28, 128, 0, 512, 256, 1),     # 4, 4
])
def test_chains_store_nothing_behind_the_last_pixel(n, h, w, c, side, o, next_o, filtered):
    """Tiles that end early: rows of another value behind both results stay, also where the residual is the output."""
    torch.manual_seed(c + o + next_o + w)
    m, behind = n * h * w, 128
    assert m % 128
    x = torch.randn(m, c, device='cuda').half()
    wt, ws, wn = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((o, c), (o, side or 1), (next_o, o)))
    (norm_f, _, keep_f), (norm, _, keep), (norm_s, _, keep_s), (norm_n, _, keep_n) = (make_norm(k, 1, 1) for k in (c, o, o, next_o))
    front = (torch.randn(n, c, 9, device='cuda').half(), (torch.randn(9, c, device='cuda') * c ** -0.5).half(), None, 0.7, norm_f, 0)
    xs = torch.randn(m, side, device='cuda').half() if side else None
    name = 'filter' if filtered else 'conv'
    count = getattr(_lib.lib(), 'ddf_hip_net_%s_chain_parts' % name)(n, h, w, c, side, o, next_o)
    assert count > 0
    parts = torch.full((n * count + 1, next_o), 7., device='cuda')
    out, nxt = (torch.full((m + behind, k), 7., device='cuda', dtype=torch.float16) for k in (o, next_o))
    if not side:
        out[:m].normal_()
    call('ddf_hip_net_%s_chain' % name, x, *(front if filtered else ()), wt, norm, None if side else out, xs,
         ws if side else None, norm_s if side else None, side, out, wn, norm_n, nxt, parts, n, h, w, c, o, next_o)
    assert (out[m:] == 7).all() and (nxt[m:] == 7).all() and (parts[-1] == 7).all()
    assert torch.isfinite(out).all() and not (out[:m] == 7).all(1).any() and not (nxt[:m] == 7).all(1).any()


@pytest.mark.parametrize('n,h,w,c,s,mid,n_parts', [
    (1, 56, 56, 64, 1, 12, 49), (70, 6, 10, 64, 2, 12, 3), (300, 4, 4, 64, 1, 12, 1),     # samples past one per compute unit
    (3, 9, 13, 128, 1, 25, 8), (2, 4, 6, 128, 2, 25, 9),
    (1, 14, 14, 256, 1, 51, 13), (17, 3, 5, 256, 1, 51, 2), (3, 28, 28, 256, 2, 51, 7),
    (5, 7, 7, 512, 1, 102, 2), (1, 14, 14, 512, 2, 102, 4),
    (2, 5, 5, 64, 1, 40, 2), (2, 5, 5, 256, 1, 20, 3), (1, 1, 1, 512, 1, 512, 1),         # channel branch of its own
])
def test_both_branches(n, h, w, c, s, mid, n_parts):
    from test_branches_gpu import channel_reference
    torch.manual_seed(h * w + c)
    x = torch.randn(n, h, w, c, device='cuda').half()
    ws, bs = (torch.randn(9, c, device='cuda') * c ** -0.5).half(), torch.randn(9, device='cuda').half()
    parts = torch.randn(n, n_parts, c, device='cuda')
    w1, w2 = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((mid, c), (9 * c, mid)))
    b1, b2, gv, ov = (torch.randn(k, device='cuda').half() for k in (mid, 9 * c, 9 * c, 9 * c))
    ho, wo = h // s, w // s
    sf = torch.empty(n, ho * wo, 12, device='cuda', dtype=torch.float16)
    cf = torch.empty(n, c, 9, device='cuda', dtype=torch.float16)
    call('ddf_hip_net_branches', x, ws, bs, sf, 0.6, parts, n_parts, w1, b1, w2, b2, cf, mid, 0.7, gv, ov, n, h, w, c, s)
    raw = F.conv2d(x.float().permute(0, 3, 1, 2), ws.float().view(9, c, 1, 1), bs.float(), stride=s)
    want = (raw - raw.mean(1, keepdim=True)) / (raw.std(1, keepdim=True) + 1e-10) * 0.6
    close(sf[:, :, :9].permute(0, 2, 1).reshape(n, 9, ho, wo), want, 4e-3)
    ref = channel_reference(parts.double().sum(1).cpu() / (h * w), *(t.cpu() for t in (w1, b1, w2, b2)), 3, 0.7, gv.cpu(), ov.cpu())
    close(cf.cpu(), ref.view(n, c, 9), 6e-3)


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('n,h,w,c,s,mid,n_parts', [
    (1, 56, 56, 64, 1, 12, 49), (3, 56, 56, 64, 1, 12, 25), (8, 56, 56, 64, 1, 12, 25),    # a row, 2 rows, two launches
    (1, 1, 1, 64, 1, 12, 1), (3, 5, 9, 64, 1, 12, 2), (2, 10, 18, 64, 2, 12, 3),
    (1, 28, 28, 128, 1, 25, 13), (3, 56, 30, 128, 2, 25, 9), (1, 3, 200, 128, 1, 25, 5),
    (1, 14, 14, 256, 1, 51, 13), (8, 14, 14, 256, 1, 51, 2), (1, 28, 28, 256, 2, 51, 13), (5, 13, 11, 256, 1, 51, 3),
    (1, 7, 7, 512, 1, 102, 4), (8, 7, 7, 512, 1, 102, 2), (3, 14, 14, 512, 2, 102, 3), (2, 4, 70, 512, 1, 102, 2),
    (1, 6, 6, 512, 1, 300, 2),                                                              # w1 and w2 in parts
    (2, 5, 5, 256, 1, 20, 3),                                                               # not covered
])
def test_ddf_layer(n, h, w, c, s, mid, n_parts, combine):
    """Branches and filter of one call: what the two calls leave."""
    torch.manual_seed(h * w + c)
    x = torch.randn(n, h, w, c, device='cuda').half()
    ws, bs = (torch.randn(9, c, device='cuda') * c ** -0.5).half(), torch.randn(9, device='cuda').half()
    parts = torch.randn(n, n_parts, c, device='cuda')
    w1, w2 = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((mid, c), (9 * c, mid)))
    b1, b2, gv, ov = (torch.randn(k, device='cuda').half() for k in (mid, 9 * c, 9 * c, 9 * c))
    ho, wo = h // s, w // s
    sf = torch.empty(n, ho * wo, 12, device='cuda', dtype=torch.float16)
    cf = torch.empty(n, c, 9, device='cuda', dtype=torch.float16)
    want, got = (torch.full((n, ho, wo, c), float('nan'), device='cuda').half() for _ in range(2))
    norm, apply, keep = make_norm(c, 1, 0)
    branches = (x, ws, bs, sf, 0.6, parts, n_parts, w1, b1, w2, b2, cf, mid, 0.7, gv, ov)
    call('ddf_hip_net_branches', *branches, n, h, w, c, s)
    call('ddf_hip_net_filter', x, cf, sf, norm, want, n, h, w, c, s, _lib.COMBINE[combine])
    call('ddf_hip_net_ddf', *branches, norm, got, n, h, w, c, s, _lib.COMBINE[combine])
    assert torch.isfinite(want).all()
    close(got, want, 2e-3)      # (order of the sums over the partial sums)


@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('n,h,w,c,s,mid,n_parts', [
    (1, 56, 56, 64, 1, 12, 49), (2, 10, 18, 64, 2, 12, 3), (8, 56, 56, 64, 1, 12, 25), (1, 28, 28, 128, 1, 25, 13),
    (3, 56, 30, 128, 2, 25, 200), (1, 14, 14, 256, 1, 51, 13), (5, 13, 11, 256, 1, 51, 60), (1, 7, 7, 512, 1, 102, 4),
    (3, 14, 14, 512, 2, 102, 30), (1, 6, 6, 512, 1, 300, 2), (2, 5, 5, 256, 1, 20, 3),
])
def test_ddf_layer_matches_pytorch(n, h, w, c, s, mid, n_parts, combine):
    """The same against plain PyTorch on the same fp16 values, many partial sums among them."""
    from test_branches_gpu import channel_reference
    torch.manual_seed(h * w + c)
    x = torch.randn(n, h, w, c, device='cuda').half()
    ws, bs = (torch.randn(9, c, device='cuda') * c ** -0.5).half(), torch.randn(9, device='cuda').half()
    parts = torch.randn(n, n_parts, c, device='cuda') * (h * w / n_parts ** 0.5)
    w1, w2 = ((torch.randn(a, b, device='cuda') * b ** -0.5).half() for a, b in ((mid, c), (9 * c, mid)))
    b1, b2, gv, ov = (torch.randn(k, device='cuda').half() for k in (mid, 9 * c, 9 * c, 9 * c))
    ho, wo = h // s, w // s
    sf = torch.empty(n, ho * wo, 12, device='cuda', dtype=torch.float16)
    cf = torch.empty(n, c, 9, device='cuda', dtype=torch.float16)
    got = torch.full((n, ho, wo, c), float('nan'), device='cuda').half()
    norm, apply, keep = make_norm(c, 1, 0)
    call('ddf_hip_net_ddf', x, ws, bs, sf, 0.6, parts, n_parts, w1, b1, w2, b2, cf, mid, 0.7, gv, ov, norm, got, n, h, w, c, s,
         _lib.COMBINE[combine])
    xc = x.float().permute(0, 3, 1, 2)
    raw = F.conv2d(xc, ws.float().view(9, c, 1, 1), bs.float(), stride=s)
    sf_want = (raw - raw.mean(1, keepdim=True)) / (raw.std(1, keepdim=True) + 1e-10) * 0.6
    cf_want = channel_reference(parts.double().sum(1).cpu() / (h * w), *(t.cpu() for t in (w1, b1, w2, b2)), 3, 0.7, gv.cpu(),
                                ov.cpu()).float().cuda().view(n, c, 9, 1, 1)
    taps = sf_want.view(n, 1, 9, ho, wo)
    comb = cf_want * taps if combine == 'mul' else cf_want + taps
    window = F.unfold(xc, 3, padding=1, stride=s).view(n, c, 9, (h - 1) // s + 1, (w - 1) // s + 1)[..., :ho, :wo]
    want = apply((window * comb).sum(2).permute(0, 2, 3, 1)).clamp_min(0)
    close(got, want, 4e-3 + 4e-3 + 6e-3)     # (what the filter, its spatial and its channel taps may be off)


@pytest.mark.parametrize('n,c,mid,n_parts', [(1, 64, 12, 512), (2, 128, 25, 513), (1, 512, 102, 33), (33, 256, 51, 9),
                                             (3, 20, 4, 1030), (2, 70, 14, 17), (70, 64, 12, 1)])
def test_sum_parts(n, c, mid, n_parts):
    parts = torch.randn(n, n_parts, c, device='cuda')
    totals = torch.empty(n, c, device='cuda')
    call('ddf_hip_net_sum_parts', parts, n_parts, totals, n, c)
    want = parts.double().sum(1)
    # (fp32 sums of n_parts values: at most n_parts roundings of the values' absolute sum, a tree's few)
    assert (totals - want).abs().max() <= 1e-6 * parts.double().abs().sum(1).max()
    assert 8 <= _lib.lib().ddf_hip_net_parts_left(n, c, mid) <= 1024


@pytest.mark.parametrize('n,h,w', [(1, 1024, 1024), (3, 1024, 768), (1, 2048, 512)])
def test_network_of_large_images(n, h, w):
    """Hundreds of partial sums per pooled value: some are left to the channel branch, some become
    totals first."""
    lib, left = _lib.lib(), []
    for k, (c, width) in enumerate(((256, 64), (256, 128), (512, 256), (1024, 512))):
        hw = [v >> (2 + max(k - 1, 0)) for v in (h, w)]
        left.append(lib.ddf_hip_net_conv_pool_parts(n, *hw, c, width) <= lib.ddf_hip_net_parts_left(n, width, int(.2 * width)))
    assert True in left and False in left
    torch.manual_seed(n)
    model = ddf_resnet.ddf_mul_resnet50(num_classes=10, zero_init_last_bn=False).cuda().half().eval()
    x = torch.randn(n, 3, h, w, device='cuda').half()
    with torch.no_grad():
        out = ddfnet_amd.functional.extension().net_forward(
            model._native_plan(ddfnet_amd.functional.extension()), x)
        modules = lambda net, y: net.fc(net.global_pool(net.forward_features(y)).flatten(1))
        by_modules = modules(model, x).float()
        want = modules(model.float(), x.float())
    off = lambda y: ((y.float() - want).norm() / want.norm()).item()
    assert off(out) <= max(4e-3, 1.3 * off(by_modules))


def test_network_of_images_wider_than_the_filter_takes():
    """Rows of more than 4096 pixels behind the stem: a block's last convolution and the next one's first are one launch,
    its branches and filter others."""
    n, h, w = 1, 32, 16416
    lib = _lib.lib()
    for side, next_o in ((64, 64), (0, 64), (0, 128)):
        assert lib.ddf_hip_net_conv_chain_parts(n, h // 4, w // 4, 64, side, 256, next_o) > 0
        assert lib.ddf_hip_net_filter_chain_parts(n, h // 4, w // 4, 64, side, 256, next_o) == 0
    torch.manual_seed(n)
    model = ddf_resnet.ddf_mul_resnet50(num_classes=10, zero_init_last_bn=False).cuda().half().eval()
    x = torch.randn(n, 3, h, w, device='cuda').half()
    with torch.no_grad():
        out = ddfnet_amd.functional.extension().net_forward(
            model._native_plan(ddfnet_amd.functional.extension()), x)
        modules = lambda net, y: net.fc(net.global_pool(net.forward_features(y)).flatten(1))
        by_modules = modules(model, x).float()
        want = modules(model.float(), x.float())
    off = lambda y: ((y.float() - want).norm() / want.norm()).item()
    assert off(out) <= max(4e-3, 1.3 * off(by_modules))
