"""Loads that write LDS past the registers (buffer_load ... lds) are ordered against the reads of what they
overwrite by a barrier alone, and s_barrier waits for nothing: every LDS read a wavefront has issued must have
returned when it gets there.  Shown on the library's own machine code, without a GPU."""
import os
import re
import shutil
import subprocess

import pytest

from mobulaop_amd import build, native

OBJDUMP = os.path.join(os.environ.get('ROCM_PATH', '/opt/rocm'), 'llvm', 'bin', 'llvm-objdump')


def _kernels(tmp_path):
    """Name -> instructions [(address, text, address branched to or None)] of the library's device code."""
    native.library()   # (built if it is not there)
    lib = shutil.copy(build.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, '--offloading', lib], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    kernels = {}
    for part in sorted(os.listdir(tmp_path)):
        if 'gfx950' not in part:
            continue
        out = subprocess.run([OBJDUMP, '-d', os.path.join(tmp_path, part)], check=True, stdout=subprocess.PIPE, text=True)
        base, code = 0, None
        for line in out.stdout.splitlines():
            head = re.match(r'([0-9a-f]+) <(\S+)>:', line)
            if head:
                base, code = int(head.group(1), 16), kernels.setdefault(head.group(2), [])
                continue
            at = re.match(r'\t(.*?)\s*// ([0-9A-F]+):(.*)', line)
            if at and code is not None:
                to = re.search(r'<[^+>]*(?:\+0x([0-9a-f]+))?>', at.group(3))
                code.append((int(at.group(2), 16), at.group(1), base + int(to.group(1) or '0', 16) if to else None))
    return kernels


def _reads_in_flight_at_barriers(code):
    """The most LDS reads that can be on their way at any s_barrier, over all paths through the code."""
    index = {address: i for i, (address, _, _) in enumerate(code)}
    most = [-1] * len(code)     # reads in flight before an instruction, -1: not reached
    worst, work = 0, [(0, 0)]
    while work:
        i, n = work.pop()
        while i < len(code) and n > most[i]:
            most[i] = n
            _, text, to = code[i]
            op = text.split()[0]
            if op.startswith('ds_read') or op.startswith('ds_bpermute'):
                n = min(n + 1, 64)
            elif op == 's_waitcnt':
                left = re.search(r'lgkmcnt\((\d+)\)', text)
                n = min(n, int(left.group(1))) if left else n
            elif op == 's_barrier':
                worst = max(worst, n)
            elif op == 's_endpgm':
                break
            if to is not None and op.startswith('s_cbranch'):
                work.append((index[to], n))
            i = index[to] if to is not None and op == 's_branch' else i + 1
    return worst


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason='no llvm-objdump')
def test_lds_reads_have_returned_at_barriers_that_free_what_they_read(tmp_path):
    kernels = {name: code for name, code in _kernels(str(tmp_path)).items()
               if any(re.match(r'buffer_load\S* .*\blds\b', text) for _, text, _ in code)}
    assert sum('igemm_b16_kernel' in name for name in kernels) >= 30   # (three products, 1 to 3 parts, heights of tiles)
    late = {name: n for name, code in kernels.items() for n in [_reads_in_flight_at_barriers(code)] if n > 0}
    assert not late, late
