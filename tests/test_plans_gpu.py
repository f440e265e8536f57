"""Layers and networks around their native plans: what runs is always the module that was
called, as it is at the time of the call."""
import copy

import pytest
import torch
import torch.utils._python_dispatch

import ddfnet_amd
from test_plans import replica_of, small_net

pytestmark = pytest.mark.gpu


def by_modules(layer, x):
    """The layer from its branches, run as modules, and the operator."""
    b, c, h, w = x.shape
    g, k, s = layer.head, layer.kernel_size, layer.stride
    cf = layer.channel_branch(x).reshape(b * g, c // g, k, k)
    sf = layer.spatial_branch(x).reshape(b * g, k * k, h // s, w // s)
    out = ddfnet_amd.ddf(x.reshape(b * g, c // g, h, w), cf, sf, k, layer.dilation, s, layer.kernel_combine)
    return out.reshape(b, c, h // s, w // s)


def close(got, want, tol=1e-4):
    assert got.shape == want.shape
    assert (got - want).abs().max() <= tol * want.abs().max()


@pytest.mark.parametrize('grad', [False, True])
def test_shallow_copy_runs_as_configured(grad):
    torch.manual_seed(0)
    layer = ddfnet_amd.DDFPack(16).cuda()
    x = torch.randn(2, 16, 8, 8, device='cuda')
    with torch.set_grad_enabled(grad):
        layer(x)
        other = copy.copy(layer)
        other.kernel_combine = 'add'
        for m in (other, layer, other):
            close(m(x), by_modules(m, x))


@pytest.mark.parametrize('grad', [False, True])
def test_replicas_run_with_their_own_weights(grad):
    torch.manual_seed(1)
    layer = ddfnet_amd.DDFPack(16).cuda()
    x = torch.randn(2, 16, 8, 8, device='cuda')
    with torch.set_grad_enabled(grad):
        layer(x)
        for scale in (2., 3.):
            replica = replica_of(layer)
            replica.channel_branch[4].std.mul_(scale)
            close(replica(x), scale * by_modules(layer, x))
            close(layer(x), by_modules(layer, x))


def test_replicas_of_a_network_run_with_their_own_weights():
    torch.manual_seed(2)
    net = small_net().cuda()
    x = torch.randn(2, 3, 64, 64, device='cuda').half()
    with torch.no_grad():
        want = net(x)
        for value in (1., 2.):
            replica = replica_of(net)
            replica.fc.weight.zero_()
            replica.fc.bias.fill_(value)
            assert torch.equal(replica(x), torch.full_like(want, value))
        assert torch.equal(net(x), want)


def test_appended_modules_and_replaced_methods_take_part():
    torch.manual_seed(3)
    layer = ddfnet_amd.DDFPack(16).cuda()
    x = torch.randn(2, 16, 8, 8, device='cuda')
    net = small_net().cuda()
    image = torch.randn(2, 3, 64, 64, device='cuda').half()
    with torch.no_grad():
        layer(x)
        layer.spatial_branch.append(torch.nn.Tanh())
        close(layer(x), by_modules(layer, x))
        want = net(image)
        net.layer1[0].forward = lambda y: torch.zeros(2, 256, 16, 16, device='cuda', dtype=torch.float16)
        zeroed = net(image)
        assert not torch.equal(zeroed, want)
        del net.layer1[0].forward
        assert torch.equal(net(image), want)
        net.layer1[0].act3.forward = lambda y: y * 0
        close(net(image), zeroed, 2e-2)


def test_what_inference_refused_it_refuses():
    x = torch.randn(2, 64, 8, 8, device='cuda')
    with torch.no_grad():
        with pytest.raises(RuntimeError, match='heads'):
            ddfnet_amd.DDFPack(64, head=3).cuda()(x)
        layer = ddfnet_amd.DDFPack(64).cuda()
        layer(x)
        layer.kernel_combine = 'max'
        with pytest.raises(AssertionError, match='only support mul or add'):
            layer(x)
        layer = ddfnet_amd.DDFPack(64).cuda()
        layer(x)
        weight = layer.channel_branch[1].weight
        weight.data = torch.stack([weight.data, weight.data], -1)[..., 0]
        with pytest.raises(RuntimeError, match='contiguous'):
            layer(x)
        layer = ddfnet_amd.DDFPack(64).cuda()
        layer(x)
        layer.spatial_branch[0].weight.data = torch.randn(9, 32, 1, 1, device='cuda')
        with pytest.raises(RuntimeError, match='fit'):
            layer(x)
        layer = ddfnet_amd.DDFPack(64).cuda()
        layer(x)
        layer.channel_branch[3].bias.data = torch.randn(9 * 63, device='cuda')
        with pytest.raises(RuntimeError, match='fit'):
            layer(x)
    layer = ddfnet_amd.DDFPack(64).cuda()
    layer(x)
    layer.kernel_combine = 'max'
    with pytest.raises(AssertionError, match='only support mul or add'):
        layer(x)


def test_resized_parameters_of_a_network_are_refused_by_their_modules():
    net = small_net().cuda()
    x = torch.randn(1, 3, 64, 64, device='cuda').half()
    with torch.no_grad():
        net(x)
        net.layer1[0].conv3.weight.data = torch.ones(256, 32, 1, 1, device='cuda').half()
        with pytest.raises(RuntimeError):
            net(x)
        net = small_net().cuda()
        net(x)
        net.layer1[0].conv2.kernel_combine = 'max'
        with pytest.raises(AssertionError, match='only support mul or add'):
            net(x)


@pytest.mark.parametrize('k', [7, 9])
@pytest.mark.parametrize('dtype,tol', [(torch.float32, 1e-4), (torch.float16, 1e-2)])
def test_filter_sizes_past_the_branch_kernels_in_inference(k, dtype, tol):
    torch.manual_seed(4)
    layer = ddfnet_amd.DDFPack(16, kernel_size=k).cuda().to(dtype)
    x = torch.randn(2, 16, 12, 10, device='cuda').to(dtype)
    with torch.no_grad():
        close(layer(x), by_modules(layer, x), tol)


def test_a_network_whose_hidden_layer_no_kernel_takes_runs_by_modules():
    torch.manual_seed(5)
    net = small_net().cuda()
    branch = net.layer1[0].conv2.channel_branch
    branch[1] = torch.nn.Conv2d(64, 16384, 1).cuda().half()
    branch[3] = torch.nn.Conv2d(16384, 9 * 64, 1).cuda().half()
    x = torch.randn(1, 3, 64, 64, device='cuda').half()
    ext = ddfnet_amd.functional.extension()
    with torch.no_grad():
        assert net._native_plan(ext) is not None and ext.net_forward(net._native_plan(ext), x) is None


@pytest.mark.parametrize('grad', [False, True])
def test_forward_mode_is_refused_and_not_dropped(grad):
    x, cf, sf = (torch.randn(*s, device='cuda') for s in ((2, 16, 6, 6), (2, 16, 3, 3), (2, 9, 6, 6)))
    layer = ddfnet_amd.DDFPack(16).cuda().requires_grad_(False)
    net = small_net().cuda().requires_grad_(False)
    image = torch.randn(1, 3, 64, 64, device='cuda').half()
    fw = torch.autograd.forward_ad
    with fw.dual_level(), torch.set_grad_enabled(grad):
        for i in range(3):
            ops = [fw.make_dual(t, torch.ones_like(t)) if i == j else t for j, t in enumerate((x, cf, sf))]
            with pytest.raises(RuntimeError):
                ddfnet_amd.ddf(*ops)
        for module, data in ((layer, x), (net, image)):
            module(data)
            with pytest.raises(RuntimeError):
                module(fw.make_dual(data, torch.ones_like(data)))


def test_transforms_of_functions_are_refused():
    x, cf, sf = (torch.randn(*s, device='cuda') for s in ((2, 16, 6, 6), (2, 16, 3, 3), (2, 9, 6, 6)))
    with pytest.raises(RuntimeError):
        torch.vmap(lambda t: ddfnet_amd.ddf(t, cf, sf))(x[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: ddfnet_amd.ddf(t, cf, sf).sum())(x)


def test_a_dispatch_mode_sees_a_networks_operators():
    class Count(torch.utils._python_dispatch.TorchDispatchMode):
        convolutions = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.convolutions += 'convolution' in func.name()
            return func(*args, **(kwargs or {}))

    net = small_net().cuda()
    image = torch.randn(1, 3, 64, 64, device='cuda').half()
    with torch.no_grad():
        want = net(image)
        with Count() as seen:
            out = net(image)
    assert seen.convolutions >= 13
    close(out, want, 2e-2)
