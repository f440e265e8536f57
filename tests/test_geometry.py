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
