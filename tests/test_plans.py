"""When the native plan of a layer or network may be used: everything that needs no GPU
(a plan is made of tensors wherever they live; only running it needs the device)."""
import copy
import gc
import weakref

import pytest
import torch

import ddfnet_amd
from ddfnet_amd import ddf_resnet, functional


@pytest.fixture
def ext():
    e = functional.extension()
    if e is None:
        pytest.skip('torch extension not built')
    return e


def small_net():
    return ddf_resnet.DDFResNet([1, 1, 1, 1], num_classes=16).half().eval()


def kinds():
    return [lambda: ddfnet_amd.DDFPack(16), small_net]


def replica_of(module, **tensors):
    """What nn.DataParallel makes of one module: tables copied, parameters as plain attributes."""
    r = module._replicate_for_data_parallel()
    for key, value in module._parameters.items():
        setattr(r, key, None if value is None else value.detach().clone())
    for key, child in module._modules.items():
        r._modules[key] = None if child is None else replica_of(child)
    return r


@pytest.mark.parametrize('make', kinds(), ids=['layer', 'network'])
def test_a_plan_belongs_to_one_module(make, ext):
    module = make()
    plan = module._native_plan(ext)
    assert plan is not None and module._native_plan(ext) is plan
    for other in (copy.copy(module), copy.deepcopy(module)):
        theirs = other._native_plan(ext)
        assert theirs is not None and theirs is not plan
        assert other._native_plan(ext) is theirs and module._native_plan(ext) is plan
    # (a copy of a copy whose original is gone)
    second = copy.copy(copy.copy(module))
    assert second._native_plan(ext) not in (None, plan)


@pytest.mark.parametrize('make', kinds(), ids=['layer', 'network'])
@pytest.mark.parametrize('planned', [True, False])
def test_replicas_have_no_plan(make, planned, ext):
    module = make()
    plan = module._native_plan(ext) if planned else None
    first, second = replica_of(module), replica_of(module)
    assert first._native_plan(ext) is None and second._native_plan(ext) is None
    assert module._native_plan(ext) is not None and (plan is None or module._native_plan(ext) is plan)


def _replace_class(m, monkeypatch):
    m.channel_branch[2].__class__ = torch.nn.LeakyReLU


def _class_method(m, monkeypatch):
    monkeypatch.setattr(torch.nn.Conv2d, 'forward', lambda self, x: x)


def _call_of_every_module(m, monkeypatch):
    monkeypatch.setattr(torch.nn.Module, '__call__', lambda self, *a: None)


LAYER_CHANGES = {
    # (stock: whether a new plan may be made of the changed layer)
    'module appended': (False, lambda m, mp: m.spatial_branch.append(torch.nn.Tanh())),
    'module added': (False, lambda m, mp: m.channel_branch.add_module('5', torch.nn.Tanh())),
    'module replaced': (True, lambda m, mp: m.channel_branch.__setitem__(1, torch.nn.Conv2d(16, 3, 1))),
    'modules reordered': (False, lambda m, mp: m.channel_branch._modules.__setitem__(
        '2', m.channel_branch._modules.pop('2'))),
    'other table': (True, lambda m, mp: setattr(m.spatial_branch, '_modules', dict(m.spatial_branch._modules))),
    'unused parameter': (True, lambda m, mp: m.spatial_branch.register_parameter(
        'extra', torch.nn.Parameter(torch.ones(1)))),
    'parameter replaced': (True, lambda m, mp: setattr(m.spatial_branch[0], 'weight', torch.nn.Parameter(
        torch.ones(9, 16, 1, 1)))),
    'parameter hidden': (False, lambda m, mp: m.spatial_branch[0].__dict__.__setitem__('weight', torch.ones(9, 16, 1, 1))),
    'instance forward': (False, lambda m, mp: setattr(m.spatial_branch[0], 'forward', lambda x: x)),
    'forward of a branch': (False, lambda m, mp: setattr(m.spatial_branch, 'forward', lambda x: x)),
    'method of the layer': (False, lambda m, mp: setattr(m, '_channel_filter', lambda x: x)),
    'class replaced': (False, _replace_class),
    'class method': (False, _class_method),
    'calls of all modules': (False, _call_of_every_module),
    'attribute': (True, lambda m, mp: setattr(m, 'kernel_combine', 'add')),
    'attribute of a module': (False, lambda m, mp: setattr(m.spatial_branch[0], 'stride', (2, 2))),
    'hook': (False, lambda m, mp: m.channel_branch[2].register_forward_hook(lambda *a: None)),
    'hooks of its own dictionary': (False, lambda m, mp: setattr(m.channel_branch[2], '_forward_hooks', {0: lambda *a: None})),
    'operator': (False, lambda m, mp: mp.setattr(ddfnet_amd.modules, 'ddf', lambda *a: None)),
}


@pytest.mark.parametrize('change', LAYER_CHANGES)
def test_a_changed_layer_loses_its_plan(change, ext, monkeypatch):
    m = ddfnet_amd.DDFPack(16)
    plan = m._native_plan(ext)
    still_stock, apply = LAYER_CHANGES[change]
    apply(m, monkeypatch)
    assert not plan.valid()
    assert (m._native_plan(ext) is not None) == still_stock


def test_what_does_not_matter_keeps_a_plan(ext):
    m = ddfnet_amd.DDFPack(16)
    plan = m._native_plan(ext)
    m.calls = 1                                   # attributes that nothing of a plan reads
    m.spatial_branch[0].note = torch.ones(1)
    m.forward = m.forward                         # wrapped: whoever calls this one wants it
    m.register_forward_hook(lambda *a: None)      # the layer's own hooks run around its forward
    m.eval()
    with torch.no_grad():
        m.spatial_branch[0].weight.mul_(2.)
    m.half()
    assert plan.valid() and m._native_plan(ext) is plan


class _Widened(ddfnet_amd.DDFPack):
    def _channel_filter(self, x):
        return super()._channel_filter(x) * 2


def test_subclasses_with_methods_of_their_own_have_no_plan(ext):
    assert _Widened(16)._native_plan(ext) is None
    assert type('Named', (ddfnet_amd.DDFPack,), {})(16)._native_plan(ext) is not None


NET_CHANGES = {
    'block appended': lambda m, mp: m.layer1.append(copy.deepcopy(m.layer1[0])),
    'forward of a block': lambda m, mp: setattr(m.layer1[0], 'forward', lambda x: x),
    'forward of a layer': lambda m, mp: setattr(m.layer2[0].conv2, 'forward', lambda x: x),
    'features': lambda m, mp: setattr(m, 'forward_features', lambda x: x),
    'class of a block': lambda m, mp: setattr(m.layer1[0], '__class__', torch.nn.Identity),
    'method of a class': lambda m, mp: mp.setattr(torch.nn.BatchNorm2d, 'forward', lambda self, x: x),
    'class of a norm': lambda m, mp: setattr(m.bn1, '__class__', torch.nn.SyncBatchNorm),
    'norm in training': lambda m, mp: m.layer3[0].bn2.train(),
    'hook': lambda m, mp: m.layer4[0].act3.register_forward_pre_hook(lambda *a: None),
}


@pytest.mark.parametrize('before', [False, True])
@pytest.mark.parametrize('change', NET_CHANGES)
def test_a_changed_network_has_no_plan(change, before, ext, monkeypatch):
    """before: the change is there when a plan is first asked for."""
    m = small_net()
    plan = None if before else m._native_plan(ext)
    if not before:
        assert plan is not None
    NET_CHANGES[change](m, monkeypatch)
    assert before or not plan.valid()
    assert m._native_plan(ext) is None


def _strided(t):
    """The same values, every second element of a larger tensor."""
    wide = torch.zeros(t.shape + (2,), dtype=t.dtype, device=t.device)
    wide[..., 0] = t.detach()
    return wide[..., 0]


def _set(module, name, value):
    setattr(module, name, torch.nn.Parameter(value))


LAYER_MISFITS = {
    'heads': (lambda: ddfnet_amd.DDFPack(16, head=3), lambda m: None),
    'strided weight': (None, lambda m: _set(m.channel_branch[1], 'weight', _strided(m.channel_branch[1].weight))),
    'strided in place': (None, lambda m: setattr(m.channel_branch[3].weight, 'data', _strided(m.channel_branch[3].weight))),
    'spatial width': (None, lambda m: _set(m.spatial_branch[0], 'weight', torch.ones(9, 8, 1, 1))),
    'hidden width': (None, lambda m: _set(m.channel_branch[1], 'weight', torch.ones(5, 16, 1, 1))),
    'taps': (None, lambda m: _set(m.channel_branch[3], 'weight', torch.ones(9 * 8, 3, 1, 1))),
    'spatial bias': (None, lambda m: _set(m.spatial_branch[0], 'bias', torch.ones(8))),
    'hidden bias': (None, lambda m: _set(m.channel_branch[1], 'bias', torch.ones(2))),
    'taps bias': (None, lambda m: setattr(m.channel_branch[3].bias, 'data', torch.ones(9 * 15))),
    'gain': (None, lambda m: _set(m.channel_branch[4], 'std', torch.ones(9 * 15))),
    'normalised channels': (None, lambda m: setattr(m.channel_branch[4], 'in_channels', 8)),
    'type': (None, lambda m: m.channel_branch[1].half()),
}


@pytest.mark.parametrize('what', LAYER_MISFITS)
def test_a_plan_does_not_run_what_does_not_fit(what, ext):
    make, change = LAYER_MISFITS[what]
    m = make() if make else ddfnet_amd.DDFPack(16)
    x = torch.ones(2, 16, 6, 6)
    if make is None:
        assert m._native_plan(ext).misfit(x) is None
        assert m._native_plan(ext).misfit(x[:, :8]) is not None
        assert m._native_plan(ext).misfit(x.double()) is not None
    change(m)
    assert m._native_plan(ext).misfit(x) is not None


def test_an_unknown_combination_has_no_plan(ext):
    m = ddfnet_amd.DDFPack(16)
    m._native_plan(ext)
    m.kernel_combine = 'max'
    assert m._native_plan(ext) is None
    with pytest.raises(AssertionError, match='only support mul or add'):
        m._pack_plan(ext)
    net = small_net()
    net._native_plan(ext)
    net.layer3[0].conv2.kernel_combine = 'max'
    assert net._native_plan(ext) is None


NET_MISFITS = {
    'resized in place': lambda m: setattr(m.layer1[0].conv3.weight, 'data', torch.ones(256, 32, 1, 1).half()),
    'norm': lambda m: _set(m.layer2[0].bn2, 'weight', torch.ones(64).half()),
    'statistics': lambda m: setattr(m.bn1, 'running_mean', torch.ones(32).half()),
    'taps': lambda m: _set(m.layer1[0].conv2.spatial_branch[0], 'weight', torch.ones(8, 64, 1, 1).half()),
    'strided': lambda m: _set(m.layer4[0].conv1, 'weight', _strided(m.layer4[0].conv1.weight)),
    'classifier': lambda m: _set(m.fc, 'weight', torch.ones(15, 2048).half()),
    'type': lambda m: m.fc.float(),
}


@pytest.mark.parametrize('what', NET_MISFITS)
def test_a_network_plan_does_not_run_what_does_not_fit(what, ext):
    m = small_net()
    x = torch.ones(1, 3, 64, 64).half()
    with torch.no_grad():
        assert m._native_plan(ext).misfit(x) is None
        for other in (x.float(), x[:, :2], x[:, :, :60], x[:0]):
            assert m._native_plan(ext).misfit(other) is not None
        NET_MISFITS[what](m)
        assert m._native_plan(ext).misfit(x) is not None
    assert m._native_plan(ext).misfit(x) is not None


@pytest.mark.parametrize('k', [3, 5, 7, 9])
def test_a_plan_only_for_filter_sizes_of_the_branch_kernels(k, ext):
    assert (ddfnet_amd.DDFPack(16, kernel_size=k)._native_plan(ext) is not None) == (k in (3, 5))


def test_images_past_the_kernels_limit_do_not_fit(ext):
    net = small_net()
    one = torch.zeros(1, dtype=torch.float16)
    with torch.no_grad():
        assert net._native_plan(ext).misfit(one.expand(1, 3, 8192, 16384)) is not None
        assert net._native_plan(ext).misfit(one.expand(1, 3, 8192, 16352)) is None


@pytest.mark.parametrize('make', kinds(), ids=['layer', 'network'])
def test_a_planned_module_goes_with_its_last_user(make, ext):
    """... at once, as any module does; and at a collection where its parts lead back to it."""
    gc.collect()
    gc.disable()
    try:
        module = make()
        assert module._native_plan(ext).valid()
        for m in module.modules():
            if isinstance(m, ddfnet_amd.DDFPack):
                assert m._native_plan(ext).valid()
        gone = [weakref.ref(t) for t in list(module.modules()) + list(module.parameters())]
        m = None
        del module
        assert not any(ref() is not None for ref in gone)
        module = make()
        plan = module._native_plan(ext)
        del module
        assert not plan.valid()
    finally:
        gc.enable()
    module = make()
    first = next(m for m in module.modules() if isinstance(m, torch.nn.Conv2d))
    first.owner = module
    first.weight.owner = module
    assert module._native_plan(ext).valid()
    gone = [weakref.ref(t) for t in list(module.modules()) + list(module.parameters())]
    del module, first
    gc.collect()
    assert not any(ref() is not None for ref in gone)


def _dual(t):
    return torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))


@pytest.mark.parametrize('make,shape', [(kinds()[0], (1, 16, 6, 6)), (kinds()[1], (1, 3, 64, 64))],
                         ids=['layer', 'network'])
@torch.no_grad()
def test_a_plan_leaves_forward_mode_alone(make, shape, ext):
    module = make()
    x = torch.ones(shape, dtype=next(module.parameters()).dtype)
    with torch.autograd.forward_ad.dual_level():
        plan = module._native_plan(ext)
        assert plan.misfit(x) is None
        assert plan.misfit(_dual(x)) is not None
        conv = next(m for m in module.modules() if isinstance(m, torch.nn.Conv2d))
        weight = _dual(conv.weight)
        conv._parameters['weight'] = weight
        plan = module._native_plan(ext)
        assert plan is None or plan.misfit(x) is not None


@pytest.mark.parametrize('make', kinds(), ids=['layer', 'network'])
def test_a_refusal_stands_until_something_changes(make, ext):
    module = make()
    conv = next(m for m in module.modules() if isinstance(m, torch.nn.Conv2d) and m.kernel_size == (1, 1))
    handle = conv.register_forward_hook(lambda *a: None)
    assert module._native_plan(ext) is None
    refused = module.__dict__['_plan'].refused
    assert refused.holds()
    with torch.no_grad():
        conv.weight.mul_(2.)
    assert module._native_plan(ext) is None and module.__dict__['_plan'].refused is refused
    conv.note = 1
    assert not refused.holds() and module._native_plan(ext) is None
    refused = module.__dict__['_plan'].refused
    handle.remove()
    assert not refused.holds() and module._native_plan(ext) is not None
    assert module.__dict__['_plan'].refused is None
    # (neither outlives its module)
    conv.register_forward_hook(lambda *a: None)
    assert module._native_plan(ext) is None
    refused, gone = module.__dict__['_plan'].refused, weakref.ref(module)
    del module
    assert gone() is None and not refused.holds()


@pytest.mark.parametrize('make', kinds(), ids=['layer', 'network'])
def test_no_plan_holds_on_to_the_graph_of_weights_put_in_for_a_call(make, ext):
    module = make()
    assert module._native_plan(ext) is not None
    conv = next(m for m in module.modules() if isinstance(m, torch.nn.Conv2d))
    own = conv.weight
    conv._parameters['weight'] = fast = own * 2
    gone = weakref.ref(fast)
    assert module._native_plan(ext) is None
    conv._parameters['weight'] = own
    del fast
    assert gone() is None
    assert module._native_plan(ext) is not None


def test_a_network_that_trains_lets_replaced_parts_go(ext):
    net = small_net().float()
    assert net._native_plan(ext) is not None
    gone = weakref.ref(net.fc)
    net.fc = torch.nn.Linear(2048, 4)
    with pytest.raises((AssertionError, RuntimeError)):      # (no device: the operator refuses)
        net.train()(torch.zeros(2, 3, 64, 64))
    assert gone() is None
