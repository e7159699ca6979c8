"""flyvec_amd/csrc/fv_window_scan.h on the host: every number of chunks that the window scan accepts gives launches that
the runtime takes (fewer than 2^32 threads in a dimension, at most 65535 blocks in the second), and the limit is where
the device's memory for the offsets ends anyway."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("window_scan") / "libscan.so"
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flyvec_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "window_scan_shim.c"), "-o", str(out)], check=True)
    lib = C.CDLL(str(out))
    for name in ("fvt_scan_tiles", "fvt_scan_max_tiles"):
        getattr(lib, name).restype = C.c_uint64
    lib.fvt_scan_tiles.argtypes = [C.c_uint64]
    for name in ("fvt_scan_tile", "fvt_scan_threads", "fvt_scan_parts"):
        getattr(lib, name).restype = C.c_uint32
    lib.fvt_scan_grids.argtypes = [C.c_uint64, C.POINTER(C.c_uint32)]
    return lib


@pytest.mark.parametrize("n_chunks", [1, 2047, 2048, 2049, 320_000, (1 << 32) - 1, 1 << 32, (1 << 32) + 1, 1 << 34,
                                      (1 << 35) - 4096])
def test_accepted_chunk_counts_give_launches_the_runtime_takes(shim, n_chunks):
    tiles = shim.fvt_scan_tiles(n_chunks)
    assert (tiles - 1) * shim.fvt_scan_tile() < n_chunks <= tiles * shim.fvt_scan_tile()
    assert tiles <= shim.fvt_scan_max_tiles()
    g = (C.c_uint32 * 4)()
    shim.fvt_scan_grids(tiles, g)
    assert g[0] * g[1] == tiles and g[2] * g[3] == tiles * shim.fvt_scan_parts()
    for x, y in ((g[0], g[1]), (g[2], g[3])):
        assert x * shim.fvt_scan_threads() < 1 << 32 and 1 <= y <= 65535


def test_the_limit(shim):
    assert shim.fvt_scan_tiles((1 << 35) - 4096 + 2048) <= shim.fvt_scan_max_tiles()
    assert shim.fvt_scan_tiles(1 << 35) > shim.fvt_scan_max_tiles()
    assert shim.fvt_scan_tiles((1 << 64) - 1) > shim.fvt_scan_max_tiles()
    g = (C.c_uint32 * 4)()
    shim.fvt_scan_grids(shim.fvt_scan_max_tiles(), g)
    assert max(g[0], g[2]) * shim.fvt_scan_threads() < 1 << 32
