"""The native module over the library, and what the library allocates: Python's lock is not held inside the library, whose launches may
wait, and the callers that do without allocations get none."""
import os
import shutil
import subprocess
import sys
import sysconfig

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

PROGRAM = """
import importlib.util, sys
import torch
spec = importlib.util.spec_from_file_location('_fast', sys.argv[1])
fast = importlib.util.module_from_spec(spec)
spec.loader.exec_module(fast)
counts = {}
def fails(rc):
    raise SystemExit('a call was made with the lock held')
fast.init(counts, fails)
half = lambda *shape: torch.zeros(shape, dtype=torch.float16, device='cuda')
full = lambda *shape: torch.zeros(shape, device='cuda')
assert fast.b2b_gemm(half(1, 32, 64), half(1, 64, 64), half(1, 64, 64), None) is not None
for make, is_half in ((half, True), (full, False)):
    q = make(1, 1, 32, 64)
    for split in (True, False):
        assert fast.flash_attention(is_half, q, q, q, None, None, None, split) is not None
    for small in (True, False):
        assert fast.stacked_lstm(is_half, make(2, 4, 32), make(1, 64, 128), None, None, None, None, -1, None, small) is not None
assert sum(counts.values()) >= 9, counts
print('released in', sum(counts.values()), 'calls')
"""


def test_python_lock_is_released_in_the_library(tmp_path):
    """With the library replaced by one that asks for the lock, in a process of its own."""
    include = sysconfig.get_paths()['include']
    subprocess.run(['g++', '-shared', '-fPIC', '-O1', '-I', include, os.path.join(HERE, 'fast_stub.cpp'), '-Wl,-soname,libftkernels.so',
                    '-o', str(tmp_path / 'libftkernels.so')], check=True)
    shutil.copy(os.path.join(HERE, '..', 'fractaltensor_amd', '_fast.so'), tmp_path / '_fast.so')
    done = subprocess.run([sys.executable, '-c', PROGRAM, str(tmp_path / '_fast.so')], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and 'released in' in done.stdout, done.stdout + done.stderr


COUNTED = """
import ctypes, sys
counter = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import torch
import fractaltensor_amd._core as core
L, T, B, H = 1, 2, 32, 256
xs, WU = torch.zeros((T, B, H), device='cuda'), torch.zeros((L, 2 * H, 4 * H), device='cuda')
out = torch.empty((L, T, B, H), device='cuda'), torch.empty((L, T, B, H), device='cuda')
core.stacked_lstm_noalloc(xs, WU, None, out)
before = counter.host_allocations()
core.stacked_lstm_check(None)
core.stacked_lstm_check(None)
print('without a workspace', counter.host_allocations() - before)
ws = torch.empty(core.stacked_lstm_workspace_bytes(L, T, B, H), dtype=torch.uint8, device='cuda')
core.stacked_lstm(xs, WU, workspace=ws)
core.stacked_lstm_check(ws)
core.stacked_lstm_check(ws)
print('with one', counter.host_allocations() - before)
"""


def test_status_of_the_built_in_scratch_allocates_nothing(tmp_path):
    """The callers of the entry point that allocates nothing read its status without an allocation too; with a workspace the
    first status call keeps one block of pinned host memory."""
    lib = str(tmp_path / 'count_host_alloc.so')
    subprocess.run(['g++', '-shared', '-fPIC', '-O1', os.path.join(HERE, 'count_host_alloc.cpp'), '-o', lib, '-ldl'], check=True)
    done = subprocess.run([sys.executable, '-c', COUNTED, lib], capture_output=True, text=True, timeout=100, cwd=os.path.dirname(HERE))
    assert done.returncode == 0 and 'without a workspace 0' in done.stdout and 'with one 1' in done.stdout, done.stdout + done.stderr
