"""NaN and infinities go where the modules have them."""
import pytest
import torch

import ddfnet_amd
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
