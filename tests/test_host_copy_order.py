"""Copies of host arrays on the CPU: csrc/host_copy.hip against stand-ins for the HIP calls (fake_hip.cpp)."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, '..', 'mobulaop_amd', 'csrc')


@pytest.fixture(scope='module')
def copies(tmp_path_factory):
    path = str(tmp_path_factory.mktemp('host_copy') / 'copies.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', '-w', '-pthread', '-D__HIP_PLATFORM_AMD__=1', '-I' + CSRC,
                    '-I/opt/rocm/include', '-o', path, '-x', 'c++', os.path.join(CSRC, 'host_copy.hip'),
                    os.path.join(HERE, 'fake_hip.cpp')], check=True)
    return ctypes.CDLL(path).run_copies


@pytest.mark.parametrize('mib', [1, 2, 5, 6, 7, 60])   # one copy; the caller's stream; two lanes; rounds of the ring
def test_transfers_wait_for_what_the_callers_stream_holds(copies, mib):
    """A transfer in either direction starts behind the work that the caller's stream was given before (it may read what the
    transfer to the device overwrites), and every byte arrives."""
    bytes_ = (mib << 20) + 12345
    before = copies(ctypes.c_size_t(1))   # (below two megabytes: hipMemcpy, no transfers; what was counted so far)
    got = copies(ctypes.c_size_t(bytes_))
    early, transfers = divmod(got - before, 1000)
    assert early == 0
    assert transfers == (0 if mib == 1 else 3 * 2 * -(-bytes_ // ((4 if mib < 7 else 2) << 20)))
