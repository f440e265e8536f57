"""The one-launch filter branches of DDFPack through the C ABI
(ddf_hip_spatial_branch, ddf_hip_channel_branch) against fp64 restatements of
the reference modules they replace: the 1x1 convolution with the operator's
stride followed by FilterNorm('spatial') (ddf/ddf.py:176-180, :145-157), and
the bottleneck MLP on the pooled features followed by FilterNorm('channel')
(ddf/ddf.py:183-192, :158-170)."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from ddfnet_amd import _lib  # noqa: E402


def spatial_reference(x, w, b, head, k, s, gain, gain_vec, offset_vec):
    kk = k * k
    n, c, h, wd = x.shape
    ho, wo = h // s, wd // s
    xs = x.double()[:, :, :ho * s:s, :wo * s:s]
    u = torch.einsum('oc,nchw->nohw', w.double().view(head * kk, c), xs)
    if b is not None:
        u = u + b.double().view(1, -1, 1, 1)
    u = u.view(n, head, kk, ho, wo)
    m = u.mean(2, keepdim=True)
    r = (u - m) / ((u - m).std(2, keepdim=True) + 1e-10)
    r = r * (gain if gain_vec is None else gain_vec.double().view(1, head, kk, 1, 1))
    if offset_vec is not None:
        r = r + offset_vec.double().view(1, head, kk, 1, 1)
    return r.view(n, head * kk, ho, wo)


def channel_reference(pooled, w1, b1, w2, b2, k, gain, gain_vec, offset_vec):
    kk = k * k
    n, c = pooled.shape
    hdn = torch.relu(pooled.double() @ w1.double().t() + b1.double())
    u = (hdn @ w2.double().t() + b2.double()).view(n, c, kk)
    m = u.mean(2, keepdim=True)
    r = (u - m) / ((u - m).std(2, keepdim=True) + 1e-10)
    r = r * (gain if gain_vec is None else gain_vec.double().view(1, c, kk))
    if offset_vec is not None:
        r = r + offset_vec.double().view(1, c, kk)
    return r.view(n, c, k, k)


# (N, C, H, W, stride, head): the ResNet-50 layer shapes at a small batch, planes
# whose size rules out one vector width after the other, odd sizes under stride 2,
# several heads, channel counts that are no multiple of the kernel's channel group
SPATIAL_CASES = [
    (3, 16, 12, 14, 1, 1), (3, 16, 12, 14, 2, 1), (3, 16, 9, 11, 1, 4), (2, 300, 7, 7, 1, 1),
    (3, 64, 30, 32, 1, 2), (2, 64, 56, 56, 1, 1), (2, 128, 56, 56, 2, 1), (2, 128, 28, 28, 1, 1),
    (2, 256, 28, 28, 2, 1), (2, 256, 14, 14, 1, 1), (2, 512, 14, 14, 2, 1), (2, 512, 7, 7, 1, 1),
    (1, 8, 5, 3, 1, 1), (1, 6, 5, 3, 2, 1), (2, 36, 13, 17, 2, 3), (1, 4, 64, 64, 1, 1),
    (5, 1024, 7, 9, 1, 1), (2, 20, 40, 24, 2, 2), (2, 7, 10, 12, 1, 1), (40, 32, 28, 28, 1, 1),
    (7, 44, 30, 24, 1, 2), (1, 40, 40, 43, 1, 2), (2, 184, 17, 15, 1, 2), (3, 40, 38, 40, 2, 1),    # a round of channels per wave
]


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 4e-3)])
@pytest.mark.parametrize('case', SPATIAL_CASES, ids=lambda c: 'x'.join(map(str, c)))
@pytest.mark.parametrize('vectors', [False, True])
def test_spatial_branch_matches_fp64(case, vectors, dtype, tol):
    n, c, h, w_, s, head = case
    torch.manual_seed(hash(case) % 1000)
    x = torch.randn(n, c, h, w_, device='cuda').to(dtype)
    w = (torch.randn(head * 9, c, device='cuda') * 0.2).to(dtype)
    b = torch.randn(head * 9, device='cuda').to(dtype) if vectors else None
    gv = (torch.rand(head * 9, device='cuda') + 0.5).to(dtype) if vectors else None
    ov = torch.randn(head * 9, device='cuda').to(dtype) if vectors else None
    out = _lib.spatial_branch(x, w, b, head, 3, s, 0.7, gv, ov)
    ref = spatial_reference(*(None if t is None else t.cpu() for t in (x, w, b)), head, 3, s, 0.7,
                            None if gv is None else gv.cpu(), None if ov is None else ov.cpu())
    assert out.shape == ref.shape
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 4e-3)])
def test_spatial_branch_unaligned_views(dtype, tol):
    """Tensors that start at odd element offsets: the vector widths fall back."""
    torch.manual_seed(5)
    for shift in (1, 2, 3):
        n, c, h, w_ = 2, 24, 12, 16
        store = torch.randn(n * c * h * w_ + shift, device='cuda').to(dtype)
        x = store[shift:].view(n, c, h, w_)
        w = (torch.randn(9, c, device='cuda') * 0.2).to(dtype)
        out = _lib.spatial_branch(x, w, None, 1, 3, 1, 1.0, None, None)
        ref = spatial_reference(x.cpu(), w.cpu(), None, 1, 3, 1, 1.0, None, None)
        err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
        assert err < tol, (shift, err)


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,k', [(3, 16, 3), (128, 64, 3), (5, 128, 3), (4, 256, 3), (3, 512, 3),
                                   (2, 70, 5), (7, 300, 3), (2, 1024, 3), (3, 64, 5), (6, 96, 3),
                                   (130, 512, 3), (9, 256, 5),
                                   # fp16 on the matrix cores: hidden layers of exactly one step, of a
                                   # step and a few values, of several steps; batches that end inside a tile
                                   (16, 160, 3), (4, 192, 3), (20, 320, 3), (2, 448, 5), (33, 1024, 3),
                                   (17, 1280, 3),
                                   (32, 512, 3), (40, 512, 3), (56, 456, 3), (70, 250, 3), (300, 130, 3), (9, 99, 5)])
def test_channel_branch_matches_fp64(n, c, k, dtype, tol):
    torch.manual_seed(n + c)
    mid = int(c * 0.2)
    pooled = torch.randn(n, c, device='cuda').to(dtype)
    w1 = (torch.randn(mid, c, device='cuda') * 0.2).to(dtype)
    b1 = torch.randn(mid, device='cuda').to(dtype)
    w2 = (torch.randn(c * k * k, mid, device='cuda') * 0.3).to(dtype)
    b2 = torch.randn(c * k * k, device='cuda').to(dtype)
    gv = (torch.rand(c * k * k, device='cuda') + 0.5).to(dtype)
    ov = torch.randn(c * k * k, device='cuda').to(dtype)
    out = _lib.channel_branch(pooled, w1, b1, w2, b2, k, 1.0, gv, ov)
    ref = channel_reference(*(t.cpu() for t in (pooled, w1, b1, w2, b2)), k, 1.0, gv.cpu(), ov.cpu())
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err


@pytest.mark.parametrize('n,c,k', [(5, 256, 3), (18, 512, 3), (3, 160, 5), (4, 64, 3)])
def test_channel_branch_without_biases_and_vectors(n, c, k):
    """Scalar gain, no offset, no biases (fp16: the matrix-core kernel where the shape allows it)."""
    torch.manual_seed(c)
    mid = int(c * 0.2)
    pooled = torch.randn(n, c, device='cuda').half()
    w1 = (torch.randn(mid, c, device='cuda') * 0.2).half()
    w2 = (torch.randn(c * k * k, mid, device='cuda') * 0.3).half()
    out = _lib.channel_branch(pooled, w1, None, w2, None, k, 0.7, None, None)
    zeros1, zeros2 = torch.zeros(mid), torch.zeros(c * k * k)
    ref = channel_reference(pooled.cpu(), w1.cpu(), zeros1, w2.cpu(), zeros2, k, 0.7, None, None)
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < 6e-3, err


def test_channel_branch_operands_at_odd_addresses():
    """Weights, biases and vectors that start 2 bytes into their allocations (views of
    larger tensors): whichever kernel takes the call, the taps are the same as from
    aligned copies."""
    torch.manual_seed(3)
    n, c, k = 20, 256, 3
    mid = int(c * 0.2)

    def shifted(t):
        store = torch.empty(t.numel() + 1, device='cuda', dtype=t.dtype)
        view = store[1:].view(t.shape)
        view.copy_(t)
        return view

    pooled = torch.randn(n, c, device='cuda').half()
    w1 = (torch.randn(mid, c, device='cuda') * 0.2).half()
    b1 = torch.randn(mid, device='cuda').half()
    w2 = (torch.randn(c * k * k, mid, device='cuda') * 0.3).half()
    b2 = torch.randn(c * k * k, device='cuda').half()
    gv = (torch.rand(c * k * k, device='cuda') + 0.5).half()
    ov = torch.randn(c * k * k, device='cuda').half()
    want = _lib.channel_branch(pooled, w1, b1, w2, b2, k, 1.0, gv, ov)
    ref = channel_reference(*(t.cpu() for t in (pooled, w1, b1, w2, b2)), k, 1.0, gv.cpu(), ov.cpu())
    scale = ref.abs().max()
    for which in range(7):
        args = [pooled, w1, b1, w2, b2, gv, ov]
        args[which] = shifted(args[which])
        out = _lib.channel_branch(args[0], args[1], args[2], args[3], args[4], k, 1.0, args[5], args[6])
        assert ((out.double().cpu() - ref).abs().max() / scale).item() < 6e-3, which
        assert ((out.float() - want.float()).abs().max() / scale).item() < 2e-3, which


POOL_CASES = [(2, 64, 56, 56, 1, 1), (2, 128, 56, 56, 2, 1), (2, 128, 28, 28, 1, 1), (2, 256, 28, 28, 2, 1),
              (2, 256, 14, 14, 1, 1), (2, 512, 14, 14, 2, 1), (2, 512, 7, 7, 1, 1), (3, 16, 12, 14, 1, 1),
              (3, 16, 12, 14, 2, 1), (3, 16, 9, 11, 1, 4), (2, 36, 10, 18, 2, 3), (1, 8, 5, 3, 1, 1),
              (2, 20, 40, 24, 2, 2), (40, 32, 28, 28, 1, 1), (2, 64, 30, 32, 1, 2), (2, 24, 6, 20, 2, 1)]


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('case', POOL_CASES, ids=lambda c: 'x'.join(map(str, c)))
def test_spatial_branch_pool(case, dtype):
    """ddf_hip_spatial_branch_pool: the same taps as ddf_hip_spatial_branch, bit for
    bit, and partial sums that add up to the feature planes' sums (the global
    average pool of ddf/ddf.py:184 times H * W)."""
    n, c, h, w_, s, head = case
    torch.manual_seed(7)
    x = torch.randn(n, c, h, w_, device='cuda').to(dtype)
    w = (torch.randn(head * 9, c, device='cuda') * 0.2).to(dtype)
    b = torch.randn(head * 9, device='cuda').to(dtype)
    both = _lib.spatial_branch_pool(x, w, b, head, 3, s, 0.7, None, None)
    assert both is not None
    sf, parts = both
    assert parts.dtype == torch.float32 and parts.shape[0] == n and parts.shape[2] == c
    assert torch.equal(sf, _lib.spatial_branch(x, w, b, head, 3, s, 0.7, None, None))
    sums = x.double().sum((2, 3)).cpu()
    scale = x.double().abs().sum((2, 3)).cpu().max()
    assert ((parts.double().sum(1).cpu() - sums).abs().max() / scale).item() < 1e-6


# vectors of four and of eight pixels, whole and partly filled tiles, odd and even numbers of
# 16-channel groups, several heads
MMA_CASES = [(11, 32, 40, 44, 1), (11, 16, 40, 44, 1), (9, 48, 64, 36, 2), (70, 64, 8, 13, 1), (3, 96, 60, 100, 3), (40, 320, 36, 52, 1), (34, 256, 33, 64, 1),
             (2, 64, 240, 300, 1), (1, 64, 200, 300, 1)]


@pytest.mark.parametrize('vectors', [False, True])
@pytest.mark.parametrize('case', MMA_CASES, ids=lambda c: 'x'.join(map(str, c)))
def test_spatial_branch_on_the_matrix_cores(case, vectors):
    n, c, h, w_, head = case
    torch.manual_seed(c + h)
    x = torch.randn(n, c, h, w_, device='cuda').half()
    w = (torch.randn(head * 9, c, device='cuda') * 0.2).half()
    b, gv, ov = (torch.randn(3, head * 9, device='cuda').half() if vectors else (None, None, None))
    sf, parts = _lib.spatial_branch_pool(x, w, b, head, 3, 1, 0.7, gv, ov)
    assert torch.equal(sf, _lib.spatial_branch(x, w, b, head, 3, 1, 0.7, gv, ov))
    ref = spatial_reference(*(None if t is None else t.cpu() for t in (x, w, b)), head, 3, 1, 0.7,
                            None if gv is None else gv.cpu(), None if ov is None else ov.cpu())
    assert ((sf.double().cpu() - ref).abs().max() / ref.abs().max()).item() < 4e-3
    sums, scale = x.double().sum((2, 3)), x.double().abs().sum((2, 3)).max()
    assert ((parts.double().sum(1) - sums).abs().max() / scale).item() < 1e-6
    # what is not finite stays with its pixel and its channel
    x[0, 5, h - 1, w_ - 1] = float('inf')
    sf2, parts2 = _lib.spatial_branch_pool(x, w, b, head, 3, 1, 0.7, gv, ov)
    last = sf2.reshape(n, head * 9, -1)[0, :, -1]
    assert torch.isnan(last).all()
    sf2.reshape(n, head * 9, -1)[0, :, -1] = sf.reshape(n, head * 9, -1)[0, :, -1]
    assert torch.equal(sf2, sf)
    assert torch.isinf(parts2[0, :, 5].sum()) and torch.isfinite(parts2.sum(1)).sum().item() == n * c - 1


# runs (stride 2: rows) that end inside a vector, by 1 to VP - 1 pixels: of four and two pixels in fp32, of eight, four
# and two in fp16, under stride 2, on the matrix cores (16-channel groups); a run one pixel longer than a vector
RAGGED_CASES = [
    (80, 12, 17, 55, 1, 2, 'f', 2), (26, 48, 27, 43, 1, 2, 'f', 2), (22, 100, 51, 13, 1, 2, 'f', 2), (9, 200, 45, 23, 1, 2, 'f', 2),
    (46, 12, 63, 53, 1, 2, 'f', 4), (53, 48, 31, 37, 1, 2, 'f', 4), (45, 100, 15, 41, 1, 2, 'f', 4), (80, 12, 90, 38, 2, 2, 'f', 2),
    (64, 48, 110, 14, 2, 2, 'f', 2), (68, 100, 110, 6, 2, 2, 'f', 2), (16, 200, 90, 22, 2, 2, 'f', 2),
    (74, 12, 19, 55, 1, 2, 'h', 2), (64, 100, 7, 61, 1, 2, 'h', 2), (26, 200, 9, 57, 1, 2, 'h', 2), (80, 12, 65, 29, 1, 2, 'h', 4),
    (54, 100, 41, 25, 1, 2, 'h', 4), (46, 200, 41, 15, 1, 2, 'h', 4), (65, 12, 75, 63, 1, 2, 'h', 8), (65, 100, 75, 22, 1, 2, 'h', 8),
    (80, 12, 38, 94, 2, 2, 'h', 2), (64, 200, 106, 6, 2, 2, 'h', 2), (59, 12, 118, 82, 2, 2, 'h', 4),
    (32, 64, 7, 6, 1, 2, 'h', 4), (40, 48, 51, 53, 1, 1, 'h', 4), (12, 64, 151, 149, 1, 2, 'h', 8), (40, 256, 45, 47, 1, 1, 'h', 8),
    (65000, 16, 1, 9, 1, 1, 'h', 8), (300, 64, 11, 11, 1, 1, 'h', 4), (500, 160, 9, 9, 1, 1, 'h', 4),     # a third of the lanes
]


@pytest.mark.parametrize('shift', [0, 1])
@pytest.mark.parametrize('case', RAGGED_CASES, ids=lambda c: 'x'.join(map(str, c)))
def test_spatial_branch_whose_runs_end_inside_a_vector(case, shift):
    """Every pixel once in the sums, all taps; what is not finite stays with its pixel and its channel, also
    where it is one that two vectors hold; tensors at odd element addresses."""
    n, c, h, w_, s, head, kind, vp = case
    dtype = {'f': torch.float32, 'h': torch.float16}[kind]
    torch.manual_seed(c + h)
    store = torch.randn(n * c * h * w_ + shift, device='cuda').to(dtype)
    x = store[shift:].view(n, c, h, w_)
    w = (torch.randn(head * 9, c, device='cuda') * 0.2).to(dtype)
    b = torch.randn(head * 9, device='cuda').to(dtype)
    sf, parts = _lib.spatial_branch_pool(x, w, b, head, 3, s, 0.7, None, None)
    run, lines = (h // s * (w_ // s), 1) if s == 1 else (w_ // s, h // s)
    assert run % vp and parts.shape[1] in (1, -(-(lines * -(-run // vp)) // 64)), parts.shape
    again = _lib.spatial_branch_pool(x, w, b, head, 3, s, 0.7, None, None)
    assert torch.equal(sf, again[0]) and torch.equal(parts, again[1])
    assert torch.equal(sf, _lib.spatial_branch(x, w, b, head, 3, s, 0.7, None, None))
    few = slice(0, min(n, 64))
    ref = spatial_reference(x[few].cpu(), w.cpu(), b.cpu(), head, 3, s, 0.7, None, None)
    # (as the other tests of this kernel: a tap's spread of nine values divides its rounding)
    assert ((sf[few].double().cpu() - ref).abs().max() / ref.abs().max()).item() < {'f': 2e-5, 'h': 4e-3}[kind]
    sums, scale = x.double().sum((2, 3)), x.double().abs().sum((2, 3)).max()
    assert ((parts.double().sum(1) - sums).abs().max() / scale).item() < 1e-6
    yl, xl = (h // s - 1) * s, (w_ // s - 1) * s
    x[n - 1, 5, yl, xl - s] = float('inf')       # (held by the last vector and the one before it, or the last only)
    sf2, parts2 = _lib.spatial_branch_pool(x, w, b, head, 3, s, 0.7, None, None)
    at = torch.zeros(h // s, w_ // s, dtype=torch.bool, device='cuda')
    at[-1, -2] = True
    assert torch.isnan(sf2[n - 1][:, at]).all()
    sf2[n - 1][:, at] = sf[n - 1][:, at]
    assert torch.equal(sf2, sf)
    total = parts2.sum(1)
    assert torch.isposinf(total[n - 1, 5]) and torch.isfinite(total).sum().item() == n * c - 1


def test_spatial_branch_pool_turns_down_what_it_cannot_cover():
    x = torch.randn(2, 16, 9, 8, device='cuda')
    w5 = torch.randn(25, 16, device='cuda')
    w3 = torch.randn(9, 16, device='cuda')
    assert _lib.spatial_branch_pool(x, w5, None, 1, 5, 1, 1.0) is None      # 5 x 5 taps
    assert _lib.spatial_branch_pool(x, w3, None, 1, 3, 2, 1.0) is None      # odd height under stride 2
    assert _lib.spatial_branch_pool(x[:, :, :8].contiguous(), w3, None, 1, 3, 2, 1.0) is not None
    assert _lib.spatial_branch_pool(x[:, :15].contiguous(), w3[:, :15].contiguous(), None, 1, 3, 1, 1.0) is None   # odd channel count


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,k,tiles', [(3, 16, 3, 1), (128, 64, 3, 13), (5, 128, 3, 4), (4, 256, 3, 2),
                                         (3, 512, 3, 7), (2, 70, 5, 3), (19, 160, 3, 1), (128, 512, 3, 4),
                                         (33, 256, 3, 16), (5, 192, 5, 6), (40, 1024, 3, 28)])
def test_channel_branch_parts_matches_fp64(n, c, k, tiles, dtype, tol):
    torch.manual_seed(n + c)
    mid = int(c * 0.2)
    parts = torch.randn(n, tiles, c, device='cuda')
    scale = 1.0 / 37
    w1 = (torch.randn(mid, c, device='cuda') * 0.2).to(dtype)
    b1 = torch.randn(mid, device='cuda').to(dtype)
    w2 = (torch.randn(c * k * k, mid, device='cuda') * 0.3).to(dtype)
    b2 = torch.randn(c * k * k, device='cuda').to(dtype)
    gv = (torch.rand(c * k * k, device='cuda') + 0.5).to(dtype)
    ov = torch.randn(c * k * k, device='cuda').to(dtype)
    out = _lib.channel_branch_parts(parts, scale, w1, b1, w2, b2, k, 1.0, gv, ov)
    assert out.dtype == dtype
    pooled = parts.double().sum(1).cpu() * scale
    ref = channel_reference(pooled, *(t.cpu() for t in (w1, b1, w2, b2)), k, 1.0, gv.cpu(), ov.cpu())
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,mid,k', [
    (100, 200, 39, 3), (100, 200, 40, 3), (101, 201, 47, 3),     # one sample a workgroup: rows of w2 as elements, as vectors
    (250, 200, 39, 3), (251, 200, 41, 3), (137, 300, 130, 3),    # two samples
    (500, 200, 40, 3), (503, 200, 41, 3),                        # four
    (5, 70, 39, 5), (5, 70, 40, 5), (3, 90, 167, 5),
])
def test_channel_branch_rows_of_the_second_product(n, c, mid, k, dtype, tol):
    """Hidden layers around the length from which rows come in as vectors: what is left of a row, rows at odd addresses;
    an infinite weight at the end of a row reaches its own channel's taps only."""
    torch.manual_seed(n + mid)
    pooled = torch.randn(n, c, device='cuda').to(dtype)
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).to(dtype)
    b1 = torch.rand(mid, device='cuda').to(dtype) + 1     # (the last hidden value is not zero for every sample)
    w2 = (torch.randn(c * k * k, mid, device='cuda') * mid ** -0.5).to(dtype)
    b2 = torch.randn(c * k * k, device='cuda').to(dtype)
    out = _lib.channel_branch(pooled, w1, b1, w2, b2, k, 0.7)
    ref = channel_reference(*(t.cpu() for t in (pooled, w1, b1, w2, b2)), k, 0.7, None, None)
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err
    w2[(c // 2) * k * k, mid - 1] = float('inf')
    got = _lib.channel_branch(pooled, w1, b1, w2, b2, k, 0.7)
    same = (got == out).flatten(2).all(-1)
    assert same[:, :c // 2].all() and same[:, c // 2 + 1:].all() and not same[:, c // 2].all()


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('n,c,mid,tiles', [(1, 256, 51, 1), (2, 256, 51, 9), (3, 160, 32, 13), (17, 320, 64, 11),
                                           (5, 64, 12, 3), (300, 96, 19, 2)])
def test_channel_branch_reads_no_partial_sums_but_its_own(n, c, mid, tiles, dtype):
    """Partial sums are asked for eight at a time: NaN in front of and behind them stays out of every filter."""
    torch.manual_seed(c + mid)
    around = torch.full((n * tiles * c + 2 * 64 * c,), float('nan'), device='cuda')
    parts = around[64 * c:-64 * c].view(n, tiles, c).normal_()
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).to(dtype)
    w2 = (torch.randn(c * 9, mid, device='cuda') * mid ** -0.5).to(dtype)
    out = _lib.channel_branch_parts(parts, 0.25, w1, None, w2, None, 3, 0.7)
    assert torch.equal(out, _lib.channel_branch_parts(parts.clone(), 0.25, w1, None, w2, None, 3, 0.7))
    assert torch.isfinite(out).all()


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,mid,tiles', [(1, 64, 16, 1), (3, 64, 17, 8), (2, 65, 16, 9), (3, 128, 31, 8), (2, 129, 32, 3),
                                           (2, 257, 20, 2), (3, 300, 65, 8), (1, 511, 3, 9), (2, 1, 1, 1)])
def test_channel_branch_one_sample_per_workgroup(n, c, mid, tiles, dtype, tol):
    """Few samples: weights requested ahead, to the edges of what is and past them."""
    torch.manual_seed(c + mid)
    k = 3
    parts = torch.randn(n, tiles, c, device='cuda')
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).to(dtype)
    w2 = (torch.randn(c * k * k, mid, device='cuda') * mid ** -0.5).to(dtype)
    b1, b2 = torch.randn(mid, device='cuda').to(dtype), torch.randn(c * k * k, device='cuda').to(dtype)
    out = _lib.channel_branch_parts(parts, 1.0, w1, b1, w2, b2, k, 0.7, None, None)
    ref = channel_reference(parts.double().sum(1).cpu(), *(t.cpu() for t in (w1, b1, w2, b2)), k, 0.7, None, None)
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err


@pytest.mark.parametrize('n,c,mid,tiles,k', [
    (1, 256, 51, 13, 3), (2, 256, 64, 9, 3), (3, 192, 33, 17, 3),   # a sample's partial sums over four waves, two, one
    (1, 32, 32, 33, 3), (1, 32, 129, 5, 3),                         # one step of channels; more tiles than waves
    (2, 288, 57, 3, 3), (17, 544, 108, 4, 3),                       # rows of w1 in one piece of 1 KB, in two
    (1, 1024, 204, 2, 3), (1, 1664, 332, 1, 3),                     # w1 in parts, then w2 in its place
    (1, 512, 512, 2, 3), (2, 1024, 204, 2, 5),                      # w2 from memory
    (18, 64, 96, 9, 5), (1, 32, 32, 1, 5),                          # taps where rows of w2 were
])
def test_channel_branch_weights_through_lds(n, c, mid, tiles, k):
    """fp16 on the matrix cores: every way the weights take into LDS; and an infinite weight
    reaches the taps of its own channel only (rows end inside a step)."""
    torch.manual_seed(c + mid)
    parts = torch.randn(n, tiles, c, device='cuda')
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).half()
    w2 = (torch.randn(c * k * k, mid, device='cuda') * mid ** -0.5).half()
    b1, b2 = torch.randn(mid, device='cuda').half(), torch.randn(c * k * k, device='cuda').half()
    out = _lib.channel_branch_parts(parts, 1.0, w1, b1, w2, b2, k, 0.7, None, None)
    ref = channel_reference(parts.double().sum(1).cpu(), *(t.cpu() for t in (w1, b1, w2, b2)), k, 0.7, None, None)
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < 6e-3, err      # (pooled and hidden values rounded to 11 bits, see above)
    w2[(c // 2) * k * k, 0] = float('inf')
    got = _lib.channel_branch_parts(parts, 1.0, w1, b1, w2, b2, k, 0.7, None, None).view(n, c, -1)
    rest = [i for i in range(c) if i != c // 2]
    assert torch.equal(got[:, rest], out.view(n, c, -1)[:, rest])


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,mid,tiles', [
    (1, 64, 12, 118), (4, 65, 13, 64), (2, 129, 25, 33), (1, 200, 31, 17),    # partial sums shared by 8, 4, 2 waves
    (31, 16, 3, 9), (1, 1, 1, 40), (256, 16, 16, 2),                          # blocks of 16, up to 256 workgroups
    (33, 100, 20, 3), (100, 70, 17, 2),                                       # blocks of 32 and 64, the last one short
    (64, 256, 51, 4), (9, 300, 129, 3),                                       # rows of w2 that come in late
    (3, 513, 30, 2), (1, 1030, 206, 5), (2, 20, 300, 1),                      # w1 in parts (fp32), long and short rows
])
def test_channel_branch_rows_through_lds(n, c, mid, tiles, dtype, tol):
    """One sample per workgroup on the vector ALU: every split of the weights over LDS.  (fp16 with
    whole steps of channels and values goes to the matrix cores.)"""
    torch.manual_seed(c + mid)
    k = 3
    parts = torch.randn(n, tiles, c, device='cuda')
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).to(dtype)
    w2 = (torch.randn(c * k * k, mid, device='cuda') * mid ** -0.5).to(dtype)
    b1, b2 = torch.randn(mid, device='cuda').to(dtype), torch.randn(c * k * k, device='cuda').to(dtype)
    gv, ov = (torch.rand(c * k * k, device='cuda') + 0.5).to(dtype), torch.randn(c * k * k, device='cuda').to(dtype)
    out = _lib.channel_branch_parts(parts, 1.0, w1, b1, w2, b2, k, 0.7, gv, ov)
    ref = channel_reference(parts.double().sum(1).cpu(), *(t.cpu() for t in (w1, b1, w2, b2)), k, 0.7, gv.cpu(), ov.cpu())
    err = ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item()
    assert err < tol, err
    w2[(c // 2) * k * k, mid - 1] = float('inf')     # (reaches its own channel only)
    got = _lib.channel_branch_parts(parts, 1.0, w1, b1, w2, b2, k, 0.7, gv, ov).view(n, c, -1)
    rest = [i for i in range(c) if i != c // 2]
    assert torch.equal(got[:, rest], out.view(n, c, -1)[:, rest])


@pytest.mark.parametrize('case,tiles', [
    # few workgroups, or not full of pixels: k_spatial_stream's vectors of two, a pixel
    ((128, 256, 14, 14), 2), ((64, 256, 14, 14), 2), ((32, 256, 28, 28), 7), ((24, 512, 28, 28), 7), ((8, 256, 50, 76), 30),
    # the matrix cores, in vectors of eight and of four; of eight where those of four leave too many sums
    ((128, 128, 28, 28), 2), ((21, 320, 48, 68), 7), ((1, 64, 200, 300), 235), ((16, 64, 56, 56), 13), ((64, 128, 28, 28), 4),
    ((10, 128, 64, 152), 19), ((2, 256, 120, 144), 68), ((3, 256, 120, 120), 29),
], ids=lambda c: str(c).replace(' ', ''))
def test_spatial_branch_takes_the_faster_kernel(case, tiles):
    """Which kernel ran, by the pixels its tiles cover: each as it was measured to be faster."""
    n, c, h, w_ = case
    x = torch.randn(n, c, h, w_, device='cuda').half()
    w = (torch.randn(9, c, device='cuda') * 0.2).half()
    sf, parts = _lib.spatial_branch_pool(x, w, None, 1, 3, 1, 0.7)
    assert parts.shape[1] == tiles
    assert torch.equal(sf, _lib.spatial_branch(x, w, None, 1, 3, 1, 0.7))
    sums, scale = x.double().sum((2, 3)), x.double().abs().sum((2, 3)).max()
    assert ((parts.double().sum(1) - sums).abs().max() / scale).item() < 1e-6


@pytest.mark.parametrize('dtype,tol', [(torch.float32, 2e-5), (torch.float16, 6e-3)])
@pytest.mark.parametrize('n,c,h,w_,tiles', [
    (1, 64, 480, 520, None), (2, 36, 480, 520, None), (3, 132, 250, 250, None), (20, 512, 130, 140, None),   # totals of many sums
    (2, 34, 480, 520, None),                                                                                # channel by channel
    (1, 64, 200, 300, 235), (8, 32, 100, 100, 40),                                                          # left as they are
])
def test_partial_sums_that_the_channel_branch_is_left(n, c, h, w_, tiles, dtype, tol):
    """Few enough rounds for the kernel that will add them up, else totals in a launch of their own."""
    if dtype == torch.float16 and c % 4:
        return      # (pooled by a launch of its own)
    torch.manual_seed(c + h)
    x = torch.randn(n, c, h, w_, device='cuda').relu_().to(dtype)
    w = (torch.randn(9, c, device='cuda') * 0.2).to(dtype)
    sf, parts = _lib.spatial_branch_pool(x, w, None, 1, 3, 1, 0.7)
    if tiles is None:
        assert parts.shape[1] == 1
    elif dtype == torch.float16:
        assert parts.shape[1] == tiles
    sums = x.double().sum((2, 3))
    assert ((parts.double().sum(1) - sums).abs().max() / sums.abs().max()).item() < 1e-6
    mid, k = max(c // 5, 1), 3
    w1 = (torch.randn(mid, c, device='cuda') * c ** -0.5).to(dtype)
    w2 = (torch.randn(c * 9, mid, device='cuda') * mid ** -0.5).to(dtype)
    b1, b2 = torch.randn(mid, device='cuda').to(dtype), torch.randn(c * 9, device='cuda').to(dtype)
    got = _lib.channel_branch_parts(parts, 1 / (h * w_), w1, b1, w2, b2, k, 0.7, None, None)
    ref = channel_reference(sums.cpu() / (h * w_), *(t.cpu() for t in (w1, b1, w2, b2)), k, 0.7, None, None)
    assert ((got.double().cpu() - ref).abs().max() / ref.abs().max()).item() < tol


@pytest.mark.parametrize('n,c,mid,tiles', [(1, 64, 12, 237), (3, 100, 20, 33), (300, 64, 12, 9), (600, 32, 6, 12), (2, 1000, 30, 9),
                                           (1, 1, 1, 1000), (1, 1024, 20, 10)])
def test_channel_branch_of_unaligned_weights_and_many_sums(n, c, mid, tiles):
    """k_channel_branch: the threads of a workgroup share a value's partial sums, one sample or several."""
    torch.manual_seed(c + mid)
    parts = torch.randn(n, tiles, c, device='cuda')
    odd = lambda *size: torch.randn(math.prod(size) + 1, device='cuda')[1:].view(size)
    w1, w2 = odd(mid, c).mul_(c ** -0.5), odd(c * 9, mid).mul_(mid ** -0.5)
    assert w1.data_ptr() % 16 and w2.data_ptr() % 16
    b1, b2 = torch.randn(mid, device='cuda'), torch.randn(c * 9, device='cuda')
    out = _lib.channel_branch_parts(parts, 0.25, w1, b1, w2, b2, 3, 0.7, None, None)
    ref = channel_reference(parts.double().sum(1).cpu() * 0.25, *(t.cpu() for t in (w1, b1, w2, b2)), 3, 0.7, None, None)
    assert ((out.double().cpu() - ref).abs().max() / ref.abs().max()).item() < 2e-5
