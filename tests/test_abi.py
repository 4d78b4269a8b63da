"""CPU checks of the C-ABI boundary: libqfx.so loads and exports every
function include/qfx.h declares, the ctypes table covers exactly those, and
error codes map onto the reference's exception types.  No kernel runs."""
import ctypes
import os
import subprocess
import sys

import pytest

from quantumflow_amd import _native


def test_library_built():
    assert os.path.exists(_native.LIB_PATH), "run python -m quantumflow_amd._build"


def test_exports_every_declared_symbol():
    declared = _native.header_symbols()
    assert len(declared) >= 15
    lib = ctypes.CDLL(_native.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name), name
    # the ctypes binding declares exactly the header's functions
    assert sorted(_native.SIGNATURES) == declared


def test_exported_symbols_are_c_linkage():
    out = subprocess.run(['nm', '-D', '--defined-only', _native.LIB_PATH],
                         capture_output=True, text=True).stdout
    syms = {line.split()[-1] for line in out.splitlines() if ' T ' in line}
    for name in _native.header_symbols():
        assert name in syms, name        # unmangled


def test_version_and_errors_without_gpu():
    lib = _native.load()
    assert b'gfx950' in lib.qfx_version()
    # argument validation happens on the host before any HIP call
    rc = lib.qfx_apply_matrix(None, None, None, 4, 1, None, None)
    assert rc == _native.QFX_EINVAL or rc == _native.QFX_ERANGE
    rc = lib.qfx_apply_matrix(None, ctypes.c_void_p(16), ctypes.c_void_p(16), 40, 1,
                              _native.int_array([0]), _native.c128_array([1, 0, 0, 1]))
    assert rc == _native.QFX_ERANGE
    rc = lib.qfx_apply_diagonal(None, ctypes.c_void_p(16), ctypes.c_void_p(16), 4, 2,
                                _native.int_array([1, 1]), _native.c128_array([1] * 4))
    assert rc == _native.QFX_EINVAL
    assert 'repeated' in _native.last_error()
    rc = lib.qfx_apply_monomial(None, ctypes.c_void_p(16), ctypes.c_void_p(16), 4, 1,
                                _native.int_array([0]), _native.int_array([0, 0]), None)
    assert rc == _native.QFX_EINVAL
    with pytest.raises(ValueError):
        _native.check(_native.QFX_EINVAL, 'x')
    with pytest.raises(RuntimeError):
        _native.check(_native.QFX_EHIP, 'x')


def test_workspace_size_formula():
    lib = _native.load()
    assert lib.qfx_reduce_workspace_bytes(1 << 28) >= (1 << 12) * 17 * 8
    assert lib.qfx_reduce_workspace_bytes(4) >= 1024 * 16


@pytest.mark.parametrize("n", [1, 10, 11, 20, 25, 26, 28, 30, 31, 34])
def test_sample_workspace_by_draws(n):
    lib = _native.load()
    chunks = 2 ** max(n - 10, 0)
    few = 8 * (2 * chunks + 1 + (chunks + 1023) // 1024)
    many = few + (8 * 64 * chunks if n <= 30 else 0)
    first = 2 ** (n - 15) if n > 25 else 1024
    for trials in (-1, 0, 1, first - 1):
        assert lib.qfx_sample_workspace_bytes_for(n, trials) == few
    for trials in (first, 2 ** 40):
        assert lib.qfx_sample_workspace_bytes_for(n, trials) == many
    assert lib.qfx_sample_workspace_bytes(n) == many
    assert lib.qfx_sample_workspace_bytes_for(0, 1) == 0
    assert lib.qfx_sample_workspace_bytes_for(35, 1) == 0


def test_gate_list_without_memory_for_it_is_an_error():
    """Host memory that runs out in qfx_apply_gates comes back as an error
    code, not as an exception out of a C function."""
    code = '''
import ctypes, resource
from quantumflow_amd import _native
lib = _native.load()
z = (ctypes.c_double * 8)(0, 0, 1, 0, 1, 0, 0, 0)
gate = _native.QfxGate(0, 1, ctypes.addressof(z), None)
count = 1 << 23
gates = (ctypes.c_void_p * count)(*([ctypes.addressof(gate)] * count))
bits = (ctypes.c_int * count)()
pages = int(open('/proc/self/statm').read().split()[0])
limit = pages * resource.getpagesize() + (16 << 20)
resource.setrlimit(resource.RLIMIT_AS, (limit, limit))
p = ctypes.c_void_p(16)
rc = lib.qfx_apply_gates(None, p, p, 14, count, gates, bits)
assert rc == _native.QFX_EHIP, rc
assert 'memory' in _native.last_error(), _native.last_error()
print('refused')
'''
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, '-c', code], cwd=root, capture_output=True, text=True)
    assert run.returncode == 0 and 'refused' in run.stdout, (run.returncode, run.stderr)
