"""NaN and infinities go where the modules have them."""
import pytest
import torch
import torch.nn.functional as F

import ddfnet_amd
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
