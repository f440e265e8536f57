"""Row-register kernels over rows that are no whole number of vectors: every length of the last
vector, both lane layouts, planes whose last row ends a tensor, each gradient on its own."""
import pytest
import torch

import ddfnet_amd
from ddfnet_amd import _lib
from ddf_testlib import TOL, check_against_oracle, random_case, rel_err, run_ddf

import oracle

pytestmark = pytest.mark.gpu


def _ids(v):
    return str(v).replace('torch.', '')


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('k,d', [(3, 1), (3, 2), (5, 1), (5, 2)])
@pytest.mark.parametrize('W', [9, 10, 11, 33, 61, 63, 71, 129, 131, 263, 265])
def test_every_tail(W, k, d, combine, dtype):
    """Rows of one vector and a tail up to rows cut into segments; enough channels that the
    filter gradients go through partial sums."""
    N, C, H = (5, 67, 23) if W < 100 else (3, 24, 131 if k == 3 and d == 1 and W == 131 else 9)
    shape = (N, C, H, W)
    names = _lib.describe(shape, k, d, 1, combine, dtype), _lib.describe(shape, k, d, 1, combine, dtype, need=7)
    if W % 2 and (d == 2 or k == 5):     # (nothing else covers these)
        assert all('ragged' in n for n in names), names
    case = random_case(N, C, H, W, k, 1, dtype, seed=W + k + d)
    check_against_oracle(*case, k, d, 1, combine, '', what='ragged rows')


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape', [(16, 70, 47, 57), (8, 66, 61, 85), (4, 66, 113, 133)], ids=_ids)
def test_wide_vectors_instead_of_single_pixels(shape, combine, dtype):
    """Sizes that single-pixel vectors cover too and the wide ones take over; each gradient
    on its own."""
    for need in (0, _lib.NEED_DX, 6, 7):
        name = _lib.describe(shape, 3, 1, 1, combine, dtype, need) if need else \
            _lib.describe(shape, 3, 1, 1, combine, dtype)
        assert 'ragged' in name, name
    x, cf, sf, go = random_case(*shape, 3, 1, dtype, seed=3)
    want = (oracle.forward(x, cf, sf, 3, 1, 1, combine),) + tuple(oracle.backward(go, x, cf, sf, 3, 1, 1, combine))
    for need in ((True, False, False), (False, True, True), (True, True, True)):
        got = run_ddf(x, cf, sf, go, 3, 1, 1, combine, need=need)
        for g, w in zip(got, want):
            if g is not None:
                assert rel_err(g, w) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,k,d', [((4, 40, 113, 150), 3, 1), ((4, 33, 50, 263), 3, 1), ((2, 33, 140, 301), 3, 1),
                                       ((5, 36, 200, 296), 3, 1), ((4, 40, 113, 150), 3, 2), ((2, 33, 140, 301), 3, 2),
                                       ((2, 33, 140, 301), 5, 1), ((4, 66, 113, 133), 5, 1), ((2, 33, 140, 301), 5, 2),
                                       ((4, 66, 113, 133), 5, 2)], ids=_ids)
def test_planes_as_one_run_of_lanes(shape, k, d, combine, dtype):
    """Strips that end inside an image row: every vector width, with and without a tail; the
    result, each gradient on its own and all of them."""
    for need in (0, _lib.NEED_DX):
        name = _lib.describe(shape, k, d, 1, combine, dtype, need) if need else \
            _lib.describe(shape, k, d, 1, combine, dtype)
        assert 'run>' in name, name
    x, cf, sf, go = random_case(*shape, k, 1, dtype, seed=k + d)
    want = (oracle.forward(x, cf, sf, k, d, 1, combine),) + tuple(oracle.backward(go, x, cf, sf, k, d, 1, combine))
    for need in ((True, False, False), (False, True, True), (True, True, True)):
        got = run_ddf(x, cf, sf, go, k, d, 1, combine, need=need)
        for g, w in zip(got, want):
            if g is not None:
                assert rel_err(g, w) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,k,d', [((2, 100, 130, 140), 3, 1), ((8, 33, 100, 150), 3, 1), ((4, 70, 45, 90), 3, 1),
                                       ((2, 33, 140, 301), 3, 1), ((3, 37, 90, 130), 3, 2), ((2, 33, 140, 301), 3, 2),
                                       ((3, 66, 60, 100), 5, 1), ((8, 70, 40, 44), 5, 1), ((4, 66, 113, 133), 5, 1),
                                       ((2, 40, 200, 304), 5, 1), ((3, 66, 60, 100), 5, 2), ((2, 33, 140, 301), 5, 2)],
                         ids=_ids)
def test_filter_gradients_in_one_run_of_lanes(shape, k, d, combine, dtype):
    """The same for the filter gradients, whose read-only lanes must stay out of the sums: with
    the feature gradient and without, with and without a channel split, each filter alone."""
    for need in (6, 7):
        name = _lib.describe(shape, k, d, 1, combine, dtype, need).split('filters')[-1]
        assert 'run>' in name, name
    x, cf, sf, go = random_case(*shape, k, 1, dtype, seed=k + d)
    want = (oracle.forward(x, cf, sf, k, d, 1, combine),) + tuple(oracle.backward(go, x, cf, sf, k, d, 1, combine))
    for need in ((False, True, False), (False, False, True), (False, True, True), (True, True, True)):
        got = run_ddf(x, cf, sf, go, k, d, 1, combine, need=need)
        for g, w in zip(got, want):
            if g is not None:
                assert rel_err(g, w) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('H,W', [(9, 10), (8, 11), (7, 12), (10, 13), (31, 15), (24, 18), (13, 30), (12, 63), (11, 131),
                                 (9, 261), (6, 262), (7, 263), (4, 286), (3, 257), (2, 135)])
def test_stride_two_of_any_size(H, W, combine, dtype):
    """Odd heights and widths, every tail, segments: all gradients in one launch, the features'
    alone, the filters' alone."""
    shape = (3, 37, H, W)
    if W % 2:      # (vectors that divide the rows need even ones)
        assert 'ragged' in _lib.describe(shape, 3, 1, 2, combine, dtype)
        for need in (_lib.NEED_DX, 6, 7):
            assert 'ragged' in _lib.describe(shape, 3, 1, 2, combine, dtype, need)
    x, cf, sf, go = random_case(*shape, 3, 2, dtype, seed=H + W)
    want = (oracle.forward(x, cf, sf, 3, 1, 2, combine),) + tuple(oracle.backward(go, x, cf, sf, 3, 1, 2, combine))
    for need in ((True, False, False), (False, True, True), (True, True, True)):
        got = run_ddf(x, cf, sf, go, 3, 1, 2, combine, need=need)
        for g, w in zip(got, want):
            if g is not None:
                assert rel_err(g, w) <= TOL[dtype]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16], ids=_ids)
@pytest.mark.parametrize('combine', ['mul', 'add'])
@pytest.mark.parametrize('shape,k,d,s', [((8, 66, 61, 85), 3, 1, 1), ((4, 66, 113, 134), 3, 1, 1),
                                         ((2, 16, 60, 131), 3, 2, 1), ((2, 16, 23, 71), 5, 2, 1),
                                         ((3, 37, 11, 131), 3, 1, 2), ((3, 37, 10, 13), 3, 1, 2)], ids=_ids)
def test_operands_at_odd_element_addresses(shape, k, d, s, combine, dtype):
    """Every operand and result one element into its buffer: these launches take any address."""
    def odd(t):
        view = torch.empty(t.numel() + 1, dtype=t.dtype, device='cuda')[1:].view(t.shape)
        return view.copy_(t)
    assert 'ragged' in _lib.describe(shape, k, d, s, combine, dtype)
    x, cf, sf, go = random_case(*shape, k, s, dtype, seed=k + s)
    xd, cfd, sfd, god = (odd(t) for t in (x, cf, sf, go))
    out, dx = odd(torch.zeros_like(go)), odd(torch.zeros_like(x))
    _lib.forward(xd, cfd, sfd, out, k, d, s, combine)
    assert rel_err(out, oracle.forward(x, cf, sf, k, d, s, combine)) <= TOL[dtype]
    need = _lib.NEED_DX
    ws = torch.empty(max(1, _lib.backward_workspace_bytes(shape, k, d, s, combine, dtype, need)), dtype=torch.uint8,
                     device='cuda')
    _lib.backward(god, xd, cfd, sfd, dx, None, None, k, d, s, combine, need, ws)
    want = oracle.backward(go, x, cf, sf, k, d, s, combine)
    assert rel_err(dx, want[0]) <= TOL[dtype]
    # (all gradients, by the public operator; its results are fresh tensors)
    leaves = [t.requires_grad_(True) for t in (xd, cfd, sfd)]
    got = torch.autograd.grad(ddfnet_amd.ddf(*leaves, k, d, s, combine), leaves, god)
    for g, w in zip(got, want):
        assert rel_err(g, w) <= TOL[dtype]
