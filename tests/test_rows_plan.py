"""flyvec_amd/csrc/fv_rows_plan.h on the host: at which sizes the dense launch visits rows as they are needed, and how many
clear launches a sequence of such steps asks for."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MIB = 1 << 20


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("rows_plan") / "librows.so"
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flyvec_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "rows_plan_shim.c"), "-o", str(out)], check=True)
    lib = C.CDLL(str(out))
    lib.fvt_rows_pay.argtypes = [C.c_uint64, C.c_uint32, C.c_uint64]
    lib.fvt_rows_clear_after.argtypes = [C.c_uint32]
    return lib


@pytest.mark.parametrize("mib,K,most", [
    (3, 128, None), (4, 128, 8), (8, 300, 8), (9, 300, 2), (12, 212, 2), (13, 72, 2), (14, 72, 0.25), (14, 128, 0.75), (16, 400, 0.75),
    (25, 1000, 0.75), (26, 1000, 24), (26, 72, 0.25), (39, 96, 0.25), (40, 96, 24), (64, 400, 24), (400, 1000, 24), (64, 28, None),
])
def test_sizes_where_visiting_rows_pays(shim, mib, K, most):
    """`most` window positions per row and no more (None: not at all)."""
    n_rows = -(-mib * MIB // (4 * K))
    if most is None:
        assert not shim.fvt_rows_pay(n_rows, K, 1)
    else:
        limit = int(most * n_rows)
        assert shim.fvt_rows_pay(n_rows, K, limit) and not shim.fvt_rows_pay(n_rows, K, limit + 1)
        assert bool(shim.fvt_rows_pay(n_rows, K, 8 * n_rows)) == (most >= 8 or (K >= 100 and 20 <= mib < 26))
        assert not shim.fvt_rows_pay(n_rows, K, 24 * n_rows + 1)


def test_clear_launches_asked_for_never_exceed_the_most(shim):
    asked = [shim.fvt_rows_clear_first()]
    for _ in range(12):
        asked.append(shim.fvt_rows_clear_after(asked[-1]))
    assert asked[:4] == [3, 6, 12, 24] and asked[8:] == [768, 1024, 1024, 1024, 1024] and shim.fvt_rows_clear_most() == 1024
