"""The C-ABI library loads, exports every function include/kernel_matmul_amd.h declares, and
its argument validation works without touching a GPU (no compute calls here)."""
import ctypes
import os
import re

import numpy as np
import pytest

from kernel_matmul_amd import _native

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "kernel_matmul_amd.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(km_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    for required in ("km_matmul", "km_param_grad", "km_param_grad_workspace_size", "km_param_grad_static", "km_index",
                     "km_make_ranges", "km_make_ranges_symmetric", "km_transpose_ranges",
                     "km_make_ranges_device", "km_make_ranges_symmetric_device", "km_last_error",
                     "km_version", "km_num_params"):
        assert required in names


def test_library_exports_every_declared_symbol():
    lib = _native.load_library()
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} declared in the header but not exported"


def test_version_and_num_params():
    lib = _native.load_library()
    assert lib.km_version() >= 100
    assert [lib.km_num_params(i) for i in range(4)] == [2, 3, 4, -1]


def test_host_argument_validation():
    lib = _native.load_library()
    x = np.zeros(4, dtype=np.float32)
    out = np.zeros(4, dtype=np.int32)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    status = lib.km_make_ranges_symmetric(p(x), 1, 4, 1.0, 0, p(out), p(out))
    assert status == -1 and b"block_size" in lib.km_last_error()
    status = lib.km_make_ranges(None, None, 1, 4, 4, 1.0, 2, 0, p(out), p(out))
    assert status == -1 and b"NULL" in lib.km_last_error()
    status = lib.km_transpose_ranges(p(out), p(out), 1, 3, 4, 4, 2, p(out), p(out))
    assert status == -1 and b"rows" in lib.km_last_error()


def test_device_entry_points_reject_bad_arguments_before_launching():
    lib = _native.load_library()
    sizes = (ctypes.c_int64 * 1)(2)
    # unknown kernel type
    status = lib.km_matmul(9, 1, sizes, 4, 4, 1, None, None, None, None, None, None, None, None,
                           None, None, None, None, None, None, None)
    assert status == -2 and b"kernel type" in lib.km_last_error()
    # too many batch dimensions
    status = lib.km_matmul(0, 7, sizes, 4, 4, 1, None, None, None, None, None, None, None, None,
                           None, None, None, None, None, None, None)
    assert status == -2 and b"batch rank" in lib.km_last_error()
    # NULL data pointer
    status = lib.km_matmul(0, 1, sizes, 4, 4, 1, None, None, None, None, None, None, None, None,
                           None, None, None, None, None, None, None)
    assert status == -1 and b"NULL" in lib.km_last_error()
    # empty problems are accepted and do nothing
    assert lib.km_matmul(0, 1, sizes, 0, 4, 1, None, None, None, None, None, None, None, None,
                         None, None, None, None, None, None, None) == 0
    assert lib.km_param_grad_workspace_size(1, 1, sizes, 1000, 1000, 4) > 0
    assert lib.km_param_grad_workspace_size(1, 1, sizes, 0, 1000, 4) == 0
    # the allocation-free variant refuses problems beyond its static scratch before anything else
    many = (ctypes.c_int64 * 1)(64)
    assert lib.km_param_grad_workspace_size(0, 1, many, 1_000_000, 1_000_000, 2) > 4 << 20
    status = lib.km_param_grad_static(0, 1, many, 1_000_000, 1_000_000, 2, *([None] * 14), None, None)
    assert status == -4 and b"static buffer" in lib.km_last_error()


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(_native, "_lib", None)
    monkeypatch.setattr(_native, "LIB_PATH", "/nonexistent/libkernel_matmul_amd.so")
    with pytest.raises(RuntimeError, match="native library not found"):
        _native.load_library()


def test_launch_descriptions_without_a_gpu():
    """km_matmul_describe / km_param_grad_describe report the launch tables' choices (host only)."""
    matmul, grad = _native.describe_matmul, _native.describe_param_grad
    # rbf and spectral kernels: the grid form from 48 row blocks on, and nothing else in the text
    text = matmul("spectral", 8, 100_000, 100_000, 16, None)
    assert "fwd_grid_grouped<spectral, G=1>" in text and "last 32 row blocks" in text and "fwd_table" not in text
    assert "fwd_grid<spectral, G=2, W=1>" in matmul("spectral", 8, 1_000_000, 1_000_000, 32, None)
    assert "fwd_grid<spectral, G=4, W=1>" in matmul("spectral", 8, 1_000_000, 1_000_000, 64, None)
    assert "fwd_grid<rbf, G=2, W=1>" in matmul("rbf", 8, 1_000_000, 1_000_000, 32, None)
    assert "fwd_grid<rbf, G=1, W=4>" in matmul("rbf", 1, 65_536, 65_536, 16, None)
    assert "fwd_table_f16<rbf, G=1" in matmul("rbf", 1, 4096, 4096, 1, None)
    assert "fwd_block<locally_periodic" in matmul("locally_periodic", 8, 1_000_000, 1_000_000, 16, None)
    # two workgroups for 64 spectral columns: as many wavefronts as asked for where a launch can have them
    wavefronts = _native.LaunchOptions(variant=7, rows_per_wave=16)
    assert "fwd_grid<spectral, G=4, W=8>" in matmul("spectral", 1, 100_000_000, 100_000, 64, wavefronts)
    assert "fwd_grid<spectral, G=4, W=4>" in matmul("spectral", 1, 600_000_000, 100_000, 64, wavefronts)
    assert "fwd_grid<spectral, G=4, W=2>" in matmul("spectral", 1, 1_500_000_000, 100_000, 64, wavefronts)
    assert "fwd_grid<spectral, G=2, W=8>" in matmul("spectral", 1, 600_000_000, 100_000, 32, wavefronts)
    # the kernels evaluated entry by entry, where they are asked for
    entries = _native.LaunchOptions(variant=3)
    text = matmul("spectral", 8, 100_000, 100_000, 16, entries)
    assert "fwd_table_f16_grouped<spectral>" in text and "128 rows per wavefront" in text
    assert "fwd_table_f16<spectral, G=2" in matmul("spectral", 8, 1_000_000, 1_000_000, 32, entries)
    assert "fwd_mfma_f16<spectral, G=4" in matmul("spectral", 8, 1_000_000, 1_000_000, 64, entries)
    assert "fwd_mfma_f16<rbf, G=2" in matmul("rbf", 8, 1_000_000, 1_000_000, 32, entries)
    assert "fwd_table_f16_grouped<rbf>" in matmul("rbf", 8, 1_000_000, 1_000_000, 16, entries)
    # narrow vectors, and wide ones in small launches: grid form; else pairwise
    assert "param_grad_grid<spectral, packed, TL=1>" in grad("spectral", 16, 100_000, 4)
    assert "param_grad_features" not in grad("spectral", 16, 100_000, 4)
    assert "param_grad_partial<spectral, TL=2>" in grad("spectral", 2, 50_000, 8)
    assert "param_grad_grid<spectral, TL=4>" in grad("spectral", 1, 7200, 11)
    assert "param_grad_grid<rbf, TL=4>" in grad("rbf", 2, 50_000, 10)
    assert "param_grad_partial<locally_periodic" in grad("locally_periodic", 2, 5_000, 3)
    # a decomposition that the asked-for kernel does not have is refused
    options = _native.LaunchOptions(variant=7, col_splits=2)
    with pytest.raises(RuntimeError, match="col_splits"):
        _native.describe_matmul("rbf", 8, 100_000, 100_000, 16, options)
    lib = _native.load_library()
    buf = ctypes.create_string_buffer(16)
    assert lib.km_param_grad_describe(7, 1, 128, 4, buf, len(buf)) == -2
    assert lib.km_param_grad_describe(1, 1, 128, 4, None, 0) == -1
    # a failed status reaches Python as RuntimeError with the library's message
    with pytest.raises(RuntimeError, match="km_param_grad_describe: invalid argument"):
        _native.describe_param_grad("spectral", 1, -5, 4)
    with pytest.raises(RuntimeError, match="km_matmul_describe: invalid argument"):
        _native.describe_matmul("spectral", 1, -5, 10, 4)


@pytest.mark.parametrize("kernel", ["rbf", "spectral", "locally_periodic"])
@pytest.mark.parametrize("variant", [0, 1, 2, 3, 5])
@pytest.mark.parametrize("batches,m,n,k", [(0, 300, 9000, 4), (1, 0, 0, 1), (2, 0, 9000, 4), (1, 300, 0, 4), (1, 300, 9000, 0)])
def test_descriptions_of_empty_problems(kernel, variant, batches, m, n, k):
    """No rows, columns, right-hand sides or batch items: described, with nothing divided by their number."""
    for options in (None, _native.LaunchOptions(variant=variant)):
        assert "<" + kernel in _native.describe_matmul(kernel, batches, m, n, k, options)
