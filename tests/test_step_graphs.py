"""Host test of which recorded steps run as graphs (lmdeploy_amd/csrc/step_graphs.h), with a stand-in for a graph: the second step of as many rows captures, a capture that fails costs
neither the step nor another try."""
import os
import shutil
import subprocess

import pytest


def test_steps_as_graphs(tmp_path):
    if shutil.which('g++') is None:
        pytest.skip('g++ not available')
    exe = str(tmp_path / 'step_graphs')
    build = subprocess.run(['g++', '-std=c++17', '-O1', '-g', '-fsanitize=address,undefined', '-fno-sanitize-recover=all', '-o', exe,
                            os.path.join(os.path.dirname(__file__), 'cpp', 'step_graphs.cpp')], capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout == 'ok\n', run.stdout + run.stderr
