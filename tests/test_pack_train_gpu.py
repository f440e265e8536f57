"""A DDFPack training step through the native node (one autograd function for the branches
and the operator) against the same layer on the CPU in fp64 with the oracle as operator."""
import pytest
import torch

import ddfnet_amd
from test_modules_gpu import cpu_reference

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, stride, head, combine
    (2, 64, 14, 14, 1, 1, 'mul'),
    (1, 16, 1, 1, 1, 1, 'add'),        # a single pixel: one step, all of it remainder
    (33, 20, 7, 7, 1, 1, 'mul'),       # odd planes, mid = 4
    (3, 136, 9, 11, 1, 2, 'mul'),      # channels past a tile of 16, two heads
    (2, 64, 12, 16, 1, 4, 'add'),
    (2, 340, 8, 6, 1, 1, 'mul'),       # mid = 68: past one chunk of 64 hidden values
    (5, 32, 18, 10, 2, 1, 'mul'),      # stride 2
    (2, 48, 20, 28, 2, 2, 'mul'),
    (1, 64, 61, 50, 1, 1, 'mul'),      # several pixel ranges per sample
    (70, 24, 3, 5, 1, 1, 'mul'),       # samples past a chunk of 64 where a workgroup has one channel,
    (65, 300, 4, 2, 1, 1, 'add'),      # two,
    (131, 344, 2, 3, 1, 1, 'mul'),     # and four
    (30000, 64, 1, 1, 1, 1, 'mul'),    # so many that two keep the partial sums within their bound
]


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 1e-4), (torch.float16, 2e-2)])
@pytest.mark.parametrize('case', CASES, ids=lambda c: 'x'.join(map(str, c)))
def test_native_training_step(case, dtype, tol, monkeypatch):
    n, c, h, w, s, head, combine = case
    torch.manual_seed(n + c + h)
    pack = ddfnet_amd.DDFPack(c, stride=s, head=head, kernel_combine=combine).cuda().to(dtype)
    x = torch.randn(n, c, h, w, device='cuda').to(dtype).requires_grad_(True)
    out = pack(x)
    assert 'PackAutograd' in type(out.grad_fn).__name__ or 'PackAutograd' in out.grad_fn.name()
    go = torch.randn_like(out)
    params = dict(pack.named_parameters())
    got = torch.autograd.grad(out, [x] + list(params.values()), go)
    ref, (xr,), out_r = cpu_reference(pack, monkeypatch, x)
    want = torch.autograd.grad(out_r, [xr] + list(ref.parameters()), go.cpu().double())
    for name, g, r in zip(['out', 'x'] + list(params), (out.detach(),) + got, (out_r.detach(),) + want):
        assert g.dtype == dtype and g.shape == r.shape, name
        err = (g.cpu().double() - r).abs().max().item() / max(r.abs().max().item(), 1e-3)
        assert err <= tol, (name, err)
    # (frozen features: other operator kernels, the same parameter gradients)
    again = torch.autograd.grad(pack(x.detach()), list(params.values()), go)
    for name, g, r in zip(params, again, got[1:]):
        assert (g - r).abs().max().item() <= tol * max(r.abs().max().item(), 1e-3), name


def test_native_training_step_has_no_second_derivative_and_follows_changes():
    pack = ddfnet_amd.DDFPack(16).cuda()
    x = torch.randn(2, 16, 6, 6, device='cuda', requires_grad=True)
    gx, = torch.autograd.grad(pack(x).square().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(gx.sum(), x)
    with torch.no_grad():
        pack.spatial_branch[0].weight.mul_(2.)      # seen without renewing anything
        pack.channel_branch[1] = torch.nn.Conv2d(16, 5, 1).cuda()   # another hidden width
        pack.channel_branch[3] = torch.nn.Conv2d(5, 144, 1).cuda()
        want = pack.channel_branch(x).reshape(2, 16, 3, 3), pack.spatial_branch(x)
        ref = ddfnet_amd.ddf(x, *want)
        assert (pack(x) - ref).abs().max() <= 1e-4 * ref.abs().max()
    assert (pack(x) - ref).abs().max() <= 1e-4 * ref.abs().max()
    pack.channel_branch[1].weight.requires_grad_(False)             # partly frozen: op by op
    pack(x).sum().backward()
    assert pack.channel_branch[1].weight.grad is None and pack.channel_branch[3].weight.grad is not None


@pytest.mark.parametrize('n,levels', [(16, 4), (33, 6)])
def test_sums_over_samples_are_added_in_pairs(n, levels):
    """A sample's gradient of 2^24 and the others' of one, added up by sixteen threads: each level of pairs loses one at most (half of
    2^24's last place), where one after another all of them would be lost."""
    from ctypes import c_void_p
    from ddfnet_amd import _lib
    c, h, w, mid = 16, 4, 4, 3
    lib = _lib.lib()

    def zeros(*shape):
        return torch.zeros(*shape, device='cuda')
    x, dcf, draw, pooled, hidden, taps = zeros(n, c, h, w), zeros(n, c, 9), zeros(n, 9, h, w), zeros(n, c), zeros(n, mid), torch.randn(n, c * 9, device='cuda')
    w1, w2, ws = zeros(mid, c), zeros(9 * c, mid), zeros(9, c)
    draw[:, :, 1, 2] = 1.
    draw[0, :, 1, 2] = 2. ** 24
    grads = [zeros(9, c), zeros(9), zeros(mid, c), zeros(mid), zeros(9 * c, mid), zeros(9 * c), zeros(9 * c)]
    size = lib.ddf_hip_pack_backward_workspace_bytes(n, c, h, w, mid, 1, 3, 1, _lib.DTYPE[torch.float32])
    space = torch.empty(size, dtype=torch.uint8, device='cuda')
    pointers = [c_void_p(t.data_ptr()) for t in (x, dcf, draw, pooled, hidden, taps, ws, w1, w2)]
    _lib.check(lib.ddf_hip_pack_backward(*pointers, None, 1.0, None, *(c_void_p(g.data_ptr()) for g in grads), c_void_p(space.data_ptr()), size,
                                         n, c, h, w, mid, 1, 3, 1, _lib.DTYPE[torch.float32],
                                         c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert (grads[1].double() - (2 ** 24 + n - 1)).abs().max() <= levels
