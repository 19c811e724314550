"""Copies of large results to host memory (csrc/host_copy.cpp) against a
stand-in for the HIP runtime that runs on the CPU: several devices, failing
runtime calls and failing allocations, which a one-GPU machine cannot show."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
HERE = ROOT / 'tests' / 'host_copy'


@pytest.fixture(scope='module')
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp('host_copy') / 'host_copy'
    subprocess.run(['g++', '-std=c++17', '-O1', '-g', '-Wall', '-pthread', f'-I{HERE}', f'-I{ROOT / "lbflow_amd" / "csrc"}',
                    str(HERE / 'main.cpp'), str(ROOT / 'lbflow_amd' / 'csrc' / 'host_copy.cpp'), '-o', str(exe)], check=True)
    return exe


@pytest.mark.parametrize('scenario', ['other_device', 'no_memory', 'no_event', 'no_record', 'small', 'known_memory'])
def test_scenario(program, scenario):
    r = subprocess.run([str(program), scenario], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
