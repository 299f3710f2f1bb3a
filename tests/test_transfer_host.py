"""The host side of the copies (transfer.hip) and of the device memory pool
(common.hpp) on a model of two devices (hipstub): a stream's device counts, not
the one that is current; what the pool keeps is given back."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), 'solvcon_amd', 'csrc')


def _build(tmp_path, main, *sources):
    exe = str(tmp_path / 'stub')
    cmd = ['g++', '-std=c++17', '-O1', '-I', os.path.join(HERE, 'hipstub'),
           '-I', CSRC, '-x', 'c++']
    cmd += [os.path.join(CSRC, s) for s in sources]
    cmd += [os.path.join(HERE, 'hipstub', main), '-o', exe, '-pthread']
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


def test_copies_on_another_device(tmp_path):
    r = subprocess.run([_build(tmp_path, 'transfer_main.cpp', 'transfer.hip')],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_copies_short_of_memory(tmp_path):
    # Any one allocation of the first copy fails: nothing terminates.
    exe = _build(tmp_path, 'short_main.cpp', 'transfer.hip')
    for k in range(1, 40):
        r = subprocess.run([exe, str(k)], capture_output=True, text=True,
                           timeout=60)
        assert r.returncode == 0, (k, r.stdout, r.stderr)


def test_pool(tmp_path):
    r = subprocess.run([_build(tmp_path, 'pool_main.cpp')],
                       capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
