"""The C-ABI library loads on a host without a GPU, exports every symbol that
include/fuel_rocm.h declares, and its host-only logic answers without a device
(no compute calls here)."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "fuel_rocm.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(frq_\w+)\s*\(", text)))


def test_header_declares_the_seams():
    syms = declared_symbols()
    for s in ("frq_qstorage_load", "frq_qstorage_zeros", "frq_qstorage_fwd", "frq_qstorage_dequantize",
              "frq_qstorage_data", "frq_qstorage_device_ptr", "frq_qmatmul", "frq_quantize_q8k",
              "frq_block_isums"):
        assert s in syms


def test_library_exports_every_declared_symbol():
    import fuel_amd

    lib = fuel_amd.lib()
    syms = declared_symbols()
    missing = [s for s in syms if not hasattr(lib, s)]
    assert not missing, missing
    # the Python binding types every declared entry point
    assert sorted(fuel_amd.SIGNATURES) == syms


def test_block_geometry_without_device():
    import fuel_amd

    assert [fuel_amd.type_size(t) for t in (8, 12, 14, 15)] == [34, 144, 210, 292]
    assert [fuel_amd.block_size(t) for t in (8, 12, 14, 15)] == [32, 256, 256, 256]
    assert fuel_amd.type_size(2) == 0  # Q4_0 is not handled by this backend


def test_errors_are_status_codes_not_crashes():
    import fuel_amd

    if fuel_amd.device_count() > 0:
        pytest.skip("a GPU is present; the no-device path is not reachable")
    with pytest.raises(fuel_amd.FuelRocmError) as ei:
        fuel_amd.RocmDevice(0)
    assert ei.value.status == 2
    lib = fuel_amd.lib()
    assert lib.frq_qmatmul(None, 12, 1, 1, 1, 256, None, 1024, None, 144, None, 4) == 2
    assert b"null device" in lib.frq_last_error()


class _ActView(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("qs", "d", "bsums", "bsh")]


class _MmqGroup(C.Structure):
    _fields_ = [("tile_expert", C.c_void_p), ("tile_row0", C.c_void_p), ("ntiles", C.c_void_p),
                ("expert_offsets", C.c_void_p), ("x_row", C.c_void_p), ("expert_bytes", C.c_size_t),
                ("w2", C.c_void_p), ("n_split", C.c_int)]


def test_grouped_launcher_refuses_what_its_wide_tiles_cannot_read():
    """launch_mmq_grouped with 64-row tiles, which read Q4_K blocks in 16-byte
    pieces over 128 columns on one side of the W | W2 split: any other operand is
    hipErrorInvalidValue before anything is launched.  (Without a GPU a call that
    passes the checks ends in another error, so nothing runs either way.)"""
    import fuel_amd

    if fuel_amd.device_count() > 0:
        pytest.skip("a GPU is present; only the no-device path may pass made-up pointers")
    fn = fuel_amd.lib()["_ZN3frq18launch_mmq_groupedEiPKhNS_7ActViewEPfiiiiiRKNS_8MmqGroupEP12ihipStream_t"]
    fn.restype = C.c_int
    fn.argtypes = [C.c_int, C.c_void_p, _ActView, C.c_void_p] + [C.c_int] * 5 + [C.POINTER(_MmqGroup), C.c_void_p]

    def call(dt=fuel_amd.Q4K, w=1 << 20, w2=1 << 21, n_split=256, expert_bytes=144 * 512, bm=64):
        g = _MmqGroup(expert_bytes=expert_bytes, w2=w2, n_split=n_split)
        return fn(dt, w, _ActView(), None, bm, 1, 2 * n_split, 256, 2 * n_split, C.byref(g), None)

    invalid = 1  # hipErrorInvalidValue
    assert call() != invalid and call(n_split=384) != invalid
    assert call(n_split=192) == invalid      # a tile would straddle W | W2
    assert call(w=(1 << 20) + 4) == invalid  # off 16-byte alignment
    assert call(w2=(1 << 21) + 8) == invalid
    assert call(expert_bytes=144 * 512 + 8) == invalid
    assert call(dt=fuel_amd.Q6K) == invalid
    # the 16- and 32-row tiles: 64 columns, any alignment, both formats
    assert call(bm=16, n_split=192, w=(1 << 20) + 4) != invalid and call(bm=32, dt=fuel_amd.Q6K) != invalid
    assert call(bm=16, n_split=96) == invalid
