"""The work users of this package give it, as cases to be timed.

Four kinds of call, each through its public entry point:

  op    ``ddf`` alone, forward or forward + backward (all three gradients)
  pack  a ``DDFPack`` layer, inference or a training step's forward + backward
  up    ``ddf_up`` (the operator of ``DDFUpPack``), forward + backward
  net   inference of a DDF-ResNet, images to logits

The shapes of the named cases are the benchmark configurations of this
repository (ResNet-50 stages at batch 64, the strided and the dilated 5 x 5
variants, the 256-channel table of its micro-benchmark, batch-128 inference),
detection-sized feature maps whose rows no vector width divides, and the
smallest calls of either end.
"""
import math

import torch

from ddfnet_amd import DDFPack, ddf, ddf_resnet, ddf_up

DTYPES = {'fp16': torch.float16, 'fp32': torch.float32}


def _op(name, n, c, h, w, k=3, d=1, s=1, combine='mul', dtype='fp32', grad=True):
    return {'name': name, 'kind': 'op', 'n': n, 'c': c, 'h': h, 'w': w, 'k': k, 'd': d, 's': s,
            'combine': combine, 'dtype': dtype, 'grad': grad}


def _pack(name, n, c, h, w, s=1, head=1, combine='mul', dtype='fp16', grad=False):
    return {'name': name, 'kind': 'pack', 'n': n, 'c': c, 'h': h, 'w': w, 's': s, 'head': head,
            'combine': combine, 'dtype': dtype, 'grad': grad}


def _up(name, n, c, h, w, scale=2, combine='mul', dtype='fp32'):
    return {'name': name, 'kind': 'up', 'n': n, 'c': c, 'h': h, 'w': w, 'scale': scale,
            'combine': combine, 'dtype': dtype}


def _net(name, n, size, depth=50, combine='mul', dtype='fp16'):
    return {'name': name, 'kind': 'net', 'n': n, 'size': size, 'depth': depth, 'combine': combine,
            'dtype': dtype}


def listed():
    return [
        # one image's small feature map, inference: a single launch, nothing but latency
        _op('op_one_image_14', 1, 64, 14, 14, grad=False),
        # training step of the operator at the ResNet-50 stages it is trained in: the
        # stage-3 shape in fp32, the stage-1 shape in fp16 with the additive combination
        _op('op_stage3_fp32', 64, 256, 14, 14),
        _op('op_stage1_add_fp16', 64, 64, 56, 56, combine='add', dtype='fp16'),
        # first layer of a stage: stride 2
        _op('op_stride2_fp32', 32, 128, 56, 56, s=2),
        # segmentation-style filters: 5 x 5 taps two pixels apart
        _op('op_k5_dilated_fp32', 32, 128, 56, 56, k=5, d=2),
        # 800 x 1200 images at 1/16: rows of 75 pixels
        _op('op_detection_odd_fp16', 4, 256, 50, 75, dtype='fp16'),
        # a layer of a served fp32 model (256-channel micro-benchmark shape)
        _pack('pack_infer_fp32', 32, 256, 28, 28, dtype='fp32'),
        # a layer at 1/4 of 800 x 1200 images, fp16
        _pack('pack_infer_large_fp16', 8, 64, 200, 300),
        # a layer's share of a training step
        _pack('pack_train_fp16', 64, 128, 28, 28, grad=True),
        # training step of the up-sampling operator
        _up('up_train_fp32', 8, 64, 64, 64),
        # batch-128 inference of the whole network, and a single image
        _net('net50_batch128_fp16', 128, 224),
        _net('net50_one_image_fp16', 1, 224),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (pixels * channels * samples of the largest drawn operator or layer call)
_MOST_ELEMENTS = 64 * 64 * 56 * 56


def draw(rng):
    kind = rng.choice(('op', 'op', 'op', 'op', 'op', 'op', 'pack', 'pack', 'pack', 'pack', 'up', 'net'))
    dtype = rng.choice(('fp16', 'fp32'))
    combine = rng.choice(('mul', 'mul', 'mul', 'add'))
    if kind == 'net':
        # (images a multiple of 32 pixels: every stage halves its feature map)
        size = 32 * rng.randint(4, 8)
        n = min(_log(rng, 1, 128), 128 * 224 * 224 // (size * size))
        case = _net('', n, size, combine=combine)
    else:
        h = _log(rng, 7, 200)
        w = max(7, int(h * rng.uniform(0.7, 1.5)))
        c = 8 * _log(rng, 4, 64) if rng.random() < 0.8 else _log(rng, 17, 512)
        most = _MOST_ELEMENTS // (4 if kind == 'up' else 1)
        n = max(1, min(_log(rng, 1, 64), most // (c * h * w)))
        c = max(1, min(c, most // (n * h * w)))
        if kind == 'op':
            k, d, s = rng.choice(((3, 1, 1), (3, 1, 1), (3, 1, 1), (3, 1, 2), (3, 2, 1), (5, 1, 1), (5, 2, 1)))
            if k == 5:   # (25 taps per pixel: a third of the pixels)
                n = max(1, n // 3)
                c = max(1, min(c, most // (3 * n * h * w)))
            case = _op('', n, c, h, w, k, d, s, combine, dtype, rng.random() < 0.6)
        elif kind == 'pack':
            s = rng.choice((1, 1, 1, 2))
            h, w = h // s * s, w // s * s          # (the layer wants sizes its stride divides)
            c = max(16, c // 4 * 4)
            case = _pack('', n, c, h, w, s, rng.choice((1, 1, 1, 2)), combine, dtype,
                         rng.random() < 0.4)
        else:
            case = _up('', n, c, h, w, 2, combine, dtype)
    del case['name']
    return case


def _standardised(f, dim):
    """What FilterNorm makes of a predicted filter: zero mean, unit deviation over its taps."""
    var, mean = torch.var_mean(f, dim=dim, keepdim=True)
    return (f - mean) / (var.sqrt() + 1e-10)


def prepare(case, seed):
    dtype = DTYPES[case['dtype']]
    g = torch.Generator(device='cuda').manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device='cuda')

    def uniform(t, lo, hi):
        t.data.uniform_(lo, hi, generator=g)

    state = {'case': case}
    if case['kind'] == 'net':
        build = getattr(ddf_resnet, 'ddf_%s_resnet%d' % (case['combine'], case['depth']))
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            with torch.device('cuda'):
                model = build(zero_init_last_bn=False)
        for m in model.modules():
            if isinstance(m, torch.nn.BatchNorm2d):
                # a trained network's normalisation: nothing at its initial value
                uniform(m.weight, 0.5, 1.5)
                uniform(m.bias, -0.2, 0.2)
                uniform(m.running_mean, -0.1, 0.1)
                uniform(m.running_var, 0.5, 1.5)
        state['model'] = model.to(dtype).eval()
        state['x'] = normal(case['n'], 3, case['size'], case['size']).to(dtype)
        return state

    n, c, h, w = case['n'], case['c'], case['h'], case['w']
    if case['kind'] == 'pack':
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            with torch.device('cuda'):
                layer = DDFPack(c, stride=case['s'], head=case['head'], kernel_combine=case['combine'])
        state['layer'] = layer.to(dtype).train(case['grad'])
        state['x'] = normal(n, c, h, w).relu_().to(dtype)   # (a layer behind a ReLU)
        if case['grad']:
            state['x'].requires_grad_(True)
            state['leaves'] = [state['x']] + list(layer.parameters())
            state['go'] = normal(n, c, h // case['s'], w // case['s']).to(dtype)
        return state

    if case['kind'] == 'up':
        branches, r = case['scale'] ** 2, case['scale']
        state['x'] = normal(n, c, h, w).to(dtype)
        state['cfs'] = [_standardised(normal(n, c, 9), 2).reshape(n, c, 3, 3).to(dtype) for _ in range(branches)]
        state['sfs'] = [_standardised(normal(n, 9, h, w), 1).to(dtype) for _ in range(branches)]
        state['go'] = normal(n, c, h * r, w * r).to(dtype)
        state['leaves'] = [state['x']] + state['cfs'] + state['sfs']
        for t in state['leaves']:
            t.requires_grad_(True)
        return state

    k, s = case['k'], case['s']
    x = normal(n, c, h, w).to(dtype)
    cf = _standardised(normal(n, c, k * k), 2).reshape(n, c, k, k).to(dtype)
    sf = _standardised(normal(n, k * k, h // s, w // s), 1).to(dtype)
    state['leaves'] = [x, cf, sf]
    if case['grad']:
        for t in state['leaves']:
            t.requires_grad_(True)
        state['go'] = normal(n, c, h // s, w // s).to(dtype)
    return state


def run(state):
    case = state['case']
    if case['kind'] == 'net':
        with torch.no_grad():
            return state['model'](state['x'])
    if case['kind'] == 'pack':
        if not case['grad']:
            with torch.no_grad():
                return state['layer'](state['x'])
        out = state['layer'](state['x'])
    elif case['kind'] == 'up':
        out = ddf_up(state['x'], state['cfs'], state['sfs'], 3, 1, case['scale'], case['combine'])
    else:
        x, cf, sf = state['leaves']
        out = ddf(x, cf, sf, case['k'], case['d'], case['s'], case['combine'])
        if not case['grad']:
            return out
    return [out] + list(torch.autograd.grad(out, state['leaves'], state['go']))


def _net_work(case):
    """Weights, the image and the logits once; two operations per multiply-add."""
    layers = {50: (3, 4, 6, 3), 101: (3, 4, 23, 3)}[case['depth']]
    n, hw = case['n'], case['size'] // 2
    params, macs = 64 * 147 + 128, n * hw * hw * 64 * 147
    hw //= 2
    cin = 64
    for stage, blocks in enumerate(layers):
        width = 64 << stage
        for b in range(blocks):
            s = 2 if b == 0 and stage > 0 else 1
            mid, out = int(0.2 * width), hw // s
            params += cin * width + width * 4 * width + 9 * width + 9 + width * mid + mid + mid * 9 * width + 18 * width
            params += 2 * (2 * width + 4 * width)
            macs += n * (hw * hw * cin * width + out * out * width * (9 + 18 + 4 * width) + width * mid * 10)
            if b == 0:
                params += cin * 4 * width + 8 * width
                macs += n * out * out * cin * 4 * width
            cin, hw = 4 * width, out
    params += cin * 1000 + 1000
    macs += n * cin * 1000
    return params, 2 * macs


def work(case):
    esz = 2 if case['dtype'] == 'fp16' else 4
    n = case['n']
    if case['kind'] == 'net':
        params, flops = _net_work(case)
        return {'bytes': esz * (params + n * 3 * case['size'] ** 2 + n * 1000), 'flops': flops}
    c, h, w = case['c'], case['h'], case['w']
    s, kk = case.get('s', 1), case.get('k', 3) ** 2
    X, P = n * c * h * w, n * (h // s) * (w // s)
    O = P * c
    if case['kind'] == 'up':
        r2 = case['scale'] ** 2
        filters = r2 * (n * c * 9 + n * 9 * h * w)
        # forward: x and filters in, r2 results out; backward: dO (r2), x, filters in, all gradients out
        return {'bytes': esz * (X + filters + r2 * X) + esz * (r2 * X + 2 * X + 2 * filters),
                'flops': 9 * r2 * X * (3 + 7)}
    if case['kind'] == 'pack':
        mid, head = int(0.2 * c), case['head']
        params = head * 9 * (c + 1) + c * mid + mid + mid * 9 * c + 18 * c
        fwd_flops = P * c * (27 + 18 * head) + 20 * n * c * mid
        if not case['grad']:
            return {'bytes': esz * (X + O + params), 'flops': fwd_flops}
        # training: x in and out for the forward; x, dO and the parameters in, their gradients out
        return {'bytes': esz * (X + O + params) + esz * (2 * X + O + 2 * params), 'flops': 3 * fwd_flops}
    filters = n * c * kk + P * kk
    if not case['grad']:
        return {'bytes': esz * (X + O + filters), 'flops': 3 * kk * O}
    return {'bytes': esz * (X + O + filters) + esz * (2 * X + O + 2 * filters), 'flops': 10 * kk * O}


def tolerance(case):
    # fp32: sums of 9 to a few thousand fp32 products.  fp16: operands and results
    # rounded to 11 bits with fp32 sums; a layer rounds half a dozen times on the way and
    # its normalisation divides by the spread of nine values; a network does so 50 layers deep.
    if case['dtype'] == 'fp32':
        return {'rel': 1e-5} if case['kind'] != 'pack' else {'rel': 3e-5}
    if case['kind'] == 'net':
        return {'rel': 8e-3}
    if case['kind'] == 'pack':
        return {'rel': 5e-3}
    return {'rel': 1e-3}
