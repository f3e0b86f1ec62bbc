"""Ahead-of-time build of the HIP launcher library for gfx950.

    python -m mobulaop_amd.build          # compile csrc/*.hip + opzoo/*/*.hip

One shared object, `csrc/libmobula_hip.so`, holds the runtime and every
operator's entry points.  It stays in the source tree (next to the code that
loads it).  Replaces the per-call JIT of the reference
(mobula/building/build.py:64-146) with one explicit hipcc invocation.  A second
one, `csrc/_torch_direct.<key>.so` (host code only), is the bundled operators' way from
torch tensors into that library; it is built where torch is installed.
"""
import glob
import hashlib
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

from .config import config

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, 'csrc')
LIB_PATH = os.path.join(CSRC, 'libmobula_hip.so')
TORCH_SOURCES = (os.path.join(CSRC, 'torch_direct.cpp'), os.path.join(_HERE, '..', 'include', 'mobula_roialign.h'))


def sources():
    return sorted(glob.glob(os.path.join(CSRC, '*.hip')) +
                  glob.glob(os.path.join(_HERE, 'opzoo', '*', '*.hip')))


def hipcc_flags():
    flags = [
        '--offload-arch=' + config.OFFLOAD_ARCH, '-std=c++17', '-O3', '-fPIC', '-shared',
        # fp32 expressions are evaluated as written: no fused multiply-add unless
        # the source asks for one, IEEE division and square root.
        '-ffp-contract=off', '-fhip-fp32-correctly-rounded-divide-sqrt',
        # hardware fp32 atomic add on global and LDS memory
        '-munsafe-fp-atomics',
        # keep scalar fp32 code scalar (no packed-fp32 instruction selection)
        '-Xclang', '-target-feature', '-Xclang', '-packed-fp32-ops',
        '-Wall', '-Wno-unused-function', '-Wno-unknown-warning-option',
        '-I' + CSRC,
        # modules compiled on load name the library by this, wherever the tree lies
        '-Wl,-soname,libmobula_hip.so',
    ]
    if config.DEBUG:
        flags.append('-g')
    return flags


def build_library(verbose=False):
    hipcc = shutil.which(config.HIPCC) or '/opt/rocm/bin/hipcc'
    if not os.path.exists(hipcc):
        raise RuntimeError('hipcc not found: the HIP launcher library cannot be built here')
    tmp = LIB_PATH + '.tmp.{}'.format(os.getpid())
    cmd = [hipcc] + hipcc_flags() + ['-o', tmp] + sources()
    if verbose or config.SHOW_BUILDING_COMMAND:
        print(' '.join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # the host pass does not know the packed-fp32 target feature: harmless
    noise = ("is not a recognized feature for this target", )
    log = '\n'.join(l for l in proc.stdout.splitlines() if not any(n in l for n in noise))
    if proc.returncode != 0:
        if os.path.exists(tmp):
            os.remove(tmp)
        raise RuntimeError('hipcc failed:\n' + log)
    if verbose and log.strip():
        print(log)
    os.replace(tmp, LIB_PATH)  # atomic: concurrent loaders never see a partial file
    return LIB_PATH


def torch_lib_path():
    """Where the torch side lies, named by all that it was compiled against -- its sources, this torch
    and this Python: a file left by another torch, whose C++ types may differ, is not found."""
    import torch
    digest = hashlib.sha256(repr((torch.__version__, torch.version.git_version, torch.compiled_with_cxx11_abi(),
                                  sysconfig.get_config_var('SOABI'))).encode())
    for path in TORCH_SOURCES:
        with open(path, 'rb') as f:
            digest.update(f.read())
    return os.path.join(CSRC, '_torch_direct.{}.so'.format(digest.hexdigest()[:12]))


def build_torch_direct(verbose=False):
    """The torch side (csrc/torch_direct.cpp) against the launcher library; None where
    torch is not installed.  (One file per torch_lib_path(): environments that share a tree keep theirs.)"""
    if importlib.util.find_spec('torch') is None:
        return None
    torch_dir = os.path.dirname(importlib.util.find_spec('torch').origin)
    path = torch_lib_path()
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(shutil.which(config.HIPCC) or '/opt/rocm/bin/hipcc')))
    tmp = path + '.tmp.{}'.format(os.getpid())
    cmd = (['g++', '-O2', '-std=c++17', '-fPIC', '-shared', '-Wall',
            # how torch's own headers ask for the ROCm build they are part of
            '-D__HIP_PLATFORM_AMD__=1', '-DUSE_ROCM=1',
            '-I' + os.path.join(_HERE, '..', 'include'), '-I' + sysconfig.get_paths()['include'],
            '-I' + os.path.join(torch_dir, 'include'),
            '-I' + os.path.join(torch_dir, 'include', 'torch', 'csrc', 'api', 'include'),
            '-I' + os.path.join(rocm, 'include'), '-o', tmp, TORCH_SOURCES[0],
            '-L' + CSRC, '-lmobula_hip', '-L' + os.path.join(torch_dir, 'lib'), '-lc10', '-lc10_hip', '-ltorch_cpu',
            '-ltorch_python', '-Wl,-rpath,$ORIGIN'])
    if verbose or config.SHOW_BUILDING_COMMAND:
        print(' '.join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        if os.path.exists(tmp):
            os.remove(tmp)
        raise RuntimeError('g++ failed:\n' + proc.stdout)
    os.replace(tmp, path)
    return path


if __name__ == '__main__':
    print(build_library(verbose=True))
    print(build_torch_direct(verbose=True))
    sys.exit(0)
