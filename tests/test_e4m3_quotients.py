"""The division-free quotients of the FP8 quantizer's 16-bit inputs: a small host program compares their e4m3 codes with those of IEEE
division for every pair of a maximum and an element."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_codes_as_divided(tmp_path):
    cxx = shutil.which('g++')
    if cxx is None:
        pytest.skip('g++ not available')
    exe = str(tmp_path / 'e4m3_quotients')
    r = subprocess.run([cxx, '-O2', '-ffp-contract=off', os.path.join(ROOT, 'tests', 'host', 'e4m3_quotients.cpp'), '-o', exe],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout[-2000:]
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith('ok'), r.stdout[-2000:]
