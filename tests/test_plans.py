"""When the native plan of a layer or network may be used: everything that needs no GPU
(a plan is made of tensors wherever they live; only running it needs the device)."""
import copy

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
