"""CPU check of the deposit's LDS box layouts and node orders (tests/emul/ma_box_emul.cpp).
Needs hipcc (host compile only); no GPU is touched."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = next((p for p in (shutil.which('hipcc'), '/opt/rocm/bin/hipcc') if p and os.path.exists(p)), None)


@pytest.mark.skipif(HIPCC is None, reason='hipcc not found')
def test_box_layouts_and_node_orders(tmp_path):
    exe = str(tmp_path / 'ma_box_emul')
    csrc = os.path.join(ROOT, 'pylians3_amd', 'csrc')
    cmd = [HIPCC, '-x', 'hip', '-O2', '-std=c++17', '--offload-arch=gfx950',
           '-Xarch_device', '-O0', '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops', '-I', csrc, '-I', os.path.join(ROOT, 'include'),
           os.path.join(ROOT, 'tests', 'emul', 'ma_box_emul.cpp'), os.path.join(csrc, 'ctx.hip'), '-o', exe,
           '-lrocfft', '-lrocprofiler-sdk-roctx']
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and 'all ok' in r.stdout, r.stdout[-4000:] + r.stderr[-2000:]
