"""The radix plans of the runtime-shaped FFT passes (host compile of the layout header, CPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, 'tests', 'cpp', 'axis_plan_check.cpp')


@pytest.mark.skipif(shutil.which('g++') is None, reason='g++ not available')
def test_axis_plans_cover_their_lines(tmp_path):
    exe = tmp_path / 'check'
    subprocess.run(['g++', '-O1', '-std=c++17', SRC, '-o', str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and 'OK' in out.stdout, out.stdout + out.stderr
