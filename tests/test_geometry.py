"""Host-side bounds model of the HIP kernels: no kernel is launched.

tests/geometry_model.cpp includes the library's geometry code and replays the
kernels' address arithmetic on the CPU for many shapes (the benchmark shapes,
ragged ones, 1-pixel planes, wide images; every kernel size / dilation / stride
the tuned families are built for; aligned and scalar-access plans; the chunked
kernels for tiny planes and for the up-sampling forward at every plane size,
kernel size and scale they take).  A launch
geometry that would make a kernel read or write out of bounds - the kind of
mistake that faults a GPU - shows up here as a VIOLATION line instead."""
import os
import random
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _hipcc():
    for cand in (os.environ.get('HIPCC'), '/opt/rocm/bin/hipcc', shutil.which('hipcc')):
        if cand and os.path.exists(cand):
            return cand
    return None


@pytest.mark.skipif(_hipcc() is None, reason='hipcc not available')
def test_every_launch_geometry_stays_in_bounds(tmp_path):
    exe = str(tmp_path / 'geometry_model')
    cmd = [_hipcc(), '-O1', '-x', 'hip', '--cuda-host-only', '-w', '-DDDF_TUNING',
           '-I' + os.path.join(ROOT, 'include'), '-I' + os.path.join(ROOT, 'ddfnet_amd', 'csrc'),
           os.path.join(ROOT, 'tests', 'geometry_model.cpp'), '-o', exe]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert build.returncode == 0, build.stdout + build.stderr
    env = dict(os.environ)
    for key in list(env):
        if key.startswith('DDF_TUNE_'):
            del env[key]
    # (the model is built with the geometry knobs switched on, so that other cuts of the
    # same problems are replayed as well; the shipped library compiles them to defaults)
    for extra in ({}, {'DDF_TUNE_WPB': '4'}, {'DDF_TUNE_WIDE': '0'}, {'DDF_TUNE_WAVES': '512'},
                  {'DDF_TUNE_CPW': '3', 'DDF_TUNE_CPW_FILTERS': '3'}, {'DDF_TUNE_VEC': '1'},
                  {'DDF_TUNE_ROWS_R': '2'}, {'DDF_TUNE_ROWS_R': '1', 'DDF_TUNE_ROWS_PAD': '0'},
                  {'DDF_TUNE_ROWS_WAVES': '512', 'DDF_TUNE_ROWS_WPB': '4', 'DDF_TUNE_ROWS_LPR': '64'},
                  {'DDF_TUNE_TAPROW_K3': '1', 'DDF_TUNE_TAPROW_WAVES': '8192'}):
        run = subprocess.run([exe], capture_output=True, text=True, timeout=600,
                             env=dict(env, **extra))
        assert run.returncode == 0
        lines = run.stdout.splitlines()
        assert sum(l.startswith('kind') and 'unsupported' not in l for l in lines) > 500
        bad = [l for l in lines if 'VIOLATION' in l]
        assert not bad, '\n'.join(bad[:10])


@pytest.mark.parametrize('dtype,shape,k,run', [
    # launches that wait for memory: whole rows, in full vectors
    ('float32', (32, 256, 112, 112), 3, False), ('float32', (32, 256, 224, 224), 3, False),
    ('float32', (64, 64, 112, 112), 3, False), ('float32', (32, 192, 139, 145), 3, False),
    ('float16', (51, 170, 108, 162), 3, False), ('float16', (8, 64, 100, 150), 3, False),
    # rows cut into segments, results that fit L2, 25 taps, lanes of one row
    ('float16', (8, 64, 200, 300), 3, True), ('float32', (12, 112, 238, 331), 3, True),
    ('float32', (3, 56, 221, 133), 3, True), ('float16', (26, 64, 65, 85), 5, True),
    ('float32', (8, 64, 90, 100), 5, True), ('float32', (12, 144, 80, 87), 3, True),
])
def test_a_plane_is_a_run_of_lanes_where_that_pays(dtype, shape, k, run):
    """Strips of whole rows against one run of lanes: each as it was measured to be faster."""
    import torch
    from ddfnet_amd import _lib
    dtype = getattr(torch, dtype)
    for need in (0, _lib.NEED_DX):
        name = _lib.describe(shape, k, 1, 1, 'mul', dtype, need)
        assert ('run>' in name) == run, name
        if not run:
            assert 'VX=%d,R=2' % (16 // dtype.itemsize) in name, name


@pytest.mark.parametrize('dtype,shape,run', [
    ('float32', (32, 256, 224, 224), False), ('float32', (4, 128, 445, 448), False),
    ('float32', (16, 192, 156, 208), False), ('float32', (8, 96, 72, 96), True),
    ('float32', (16, 64, 88, 176), True),
    ('float32', (8, 64, 200, 300), True), ('float32', (32, 64, 240, 320), True),
    ('float16', (16, 192, 221, 224), True), ('float16', (8, 64, 200, 300), True),
])
def test_filter_gradients_of_whole_lines_stay_rows(dtype, shape, run):
    """Strips that end with a line are left for a run of lanes where it takes a quarter of them away, or in cache."""
    import torch
    from ddfnet_amd import _lib
    for need in (_lib.NEED_DCF | _lib.NEED_DSF, _lib.NEED_DX | _lib.NEED_DCF | _lib.NEED_DSF):
        name = _lib.describe(shape, 3, 1, 1, 'mul', getattr(torch, dtype), need)
        assert ('run>' in name) == run, name


@pytest.mark.skipif(shutil.which('nm') is None, reason='nm not available')
def test_every_plan_of_all_five_by_five_gradients_has_its_kernel():
    """What describe names as one launch is one: the library holds the kernel that the plan asks for."""
    import torch
    from ddfnet_amd import LIB_PATH, _lib
    names = subprocess.run(['nm', '-C', LIB_PATH], capture_output=True, text=True, check=True).stdout
    built = set(re.findall(r'k_rows_taprow_backward<(float|__half), (\d), (true|false), (\d), (\d), (true|false), \d+, \d+, (\d)>', names))
    rng = random.Random(5)
    shapes = [(13, 120, 34, 34, 2), (6, 76, 9, 66, 1), (3, 40, 31, 30, 2), (4, 256, 50, 74, 1), (2, 64, 100, 150, 1)]
    shapes += [(rng.randint(1, 40), rng.randint(1, 200), rng.randint(3, 200), rng.randint(4, 260), rng.choice((1, 2))) for _ in range(1500)]
    met = set()
    for n, c, h, w, d in shapes:
        for dtype, element in ((torch.float32, 'float'), (torch.float16, '__half')):
            for combine in ('mul', 'add'):
                plan = re.match(r'k_rows_taprow_backward<VXF=(\d),VX=(\d),(.*?)>', _lib.describe((n, c, h, w), 5, d, 1, combine, dtype, need=7))
                if not plan:
                    continue
                vxf, vx, layout = plan.groups()
                ragged = 'ragged' in layout    # (odd fp16 tails: the lane loads from one element further left)
                tail = 0 if not ragged else 2 if dtype == torch.float16 and w % int(vx) % 2 else 1
                pads = ('true', 'false') if layout == 'run' else ('false',) if layout == 'plain' else ('true',)
                wanted = {(element, str(d), 'true' if combine == 'mul' else 'false', vxf, vx, pad, str(tail)) for pad in pads}
                assert wanted & built, ((n, c, h, w), d, dtype, plan.group(0))
                met |= wanted & built
    assert len(met) > 40    # (the sweep meets most of them)
