"""flyvec_amd/csrc/fv_host_plan.h on the host: which transfers go through the page-locked slots, and that their pieces
cover what they carry once, each inside a slot."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MB = 1 << 20


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_plan") / "libplan.so"
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", "-I", os.path.join(ROOT, "flyvec_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "host_plan_shim.c"), "-o", str(out)], check=True)
    lib = C.CDLL(str(out))
    u64, u32 = C.c_uint64, C.c_uint32
    for name, args in (("fvt_slot_bytes", []), ("fvt_copy_pieces", [u64]), ("fvt_copy_slots", [u64]), ("fvt_copy_piece_bytes", [u64, u64]),
                       ("fvt_matrix_pieces", [u32, u64])):
        getattr(lib, name).restype = u64
        getattr(lib, name).argtypes = args
    for name in ("fvt_upload_staged", "fvt_download_staged", "fvt_matrix_upload_staged"):
        getattr(lib, name).argtypes = [u64]
    lib.fvt_plan_hash.argtypes = [u64, u32, u64, u64, C.c_int, C.c_int, C.POINTER(u64)]
    lib.fvt_hash_stage.argtypes = [u64, u64, u64, u64, u64, u32, C.POINTER(u64)]
    lib.fvt_matrix_piece.argtypes = [u32, u64, u64, C.POINTER(u64)]
    return lib


def test_small_and_middling_transfers_stay_with_the_runtime(shim):
    """Where the slots were measured to be no faster: uploads below 24 MB, downloads below 5 MB, matrices between one
    slot and 8 MB upwards."""
    for up, down, matrix, size in ((0, 0, 1, 1), (0, 0, 1, 4 * MB), (0, 0, 0, 4 * MB + 4), (0, 0, 0, 5 * MB - 1), (0, 1, 0, 5 * MB),
                                   (0, 1, 0, 8 * MB - 4), (0, 1, 1, 8 * MB), (0, 1, 1, 24 * MB - 1), (1, 1, 1, 24 * MB),
                                   (1, 1, 1, 1 << 40)):
        got = shim.fvt_upload_staged(size), shim.fvt_download_staged(size), shim.fvt_matrix_upload_staged(size)
        assert tuple(map(bool, got)) == (bool(up), bool(down), bool(matrix)), size


@pytest.mark.parametrize("size", [5 * MB, 8 * MB, 8 * MB + 1, 16 * MB, 16 * MB + 1, 20 * MB - 1, 33 * MB + 24])
def test_pieces_of_a_plain_copy(shim, size):
    n = shim.fvt_copy_pieces(size)
    sizes = [shim.fvt_copy_piece_bytes(size, t) for t in range(n)]
    assert sum(sizes) == size and min(sizes) > 0 and max(sizes) <= shim.fvt_slot_bytes()
    assert all(s == shim.fvt_slot_bytes() for s in sizes[:-1])
    assert shim.fvt_copy_slots(size) == min(n, 4)


@pytest.mark.parametrize("K,N", [(1, 2), (2048, 2), (400, 1874), (400, 2620), (400, 2622), (64, 16384), (64, 16386),
                                 (63, 16644), (63, 16646), (65, 16130), (65, 32770), (2048, 512), (2048, 514),
                                 (130, 81926), (1, 1048576), (1, 1048578)])
def test_pieces_of_a_matrix_cover_it_once(shim, K, N):
    seen = np.zeros((K, N), np.uint8)
    n = shim.fvt_matrix_pieces(K, N)
    assert (n == 1) == (K * N * 4 <= shim.fvt_slot_bytes())  # what fits a slot goes in one piece
    m = (C.c_uint64 * 5)()
    for t in range(n):
        shim.fvt_matrix_piece(K, N, t, m)
        h, rows, i, cols, pitch = m
        assert rows and cols and h + rows <= K and i + cols <= N and pitch >= cols
        assert ((rows - 1) * pitch + cols) * 4 <= shim.fvt_slot_bytes()
        seen[h:h + rows, i:i + cols] += 1
    assert (seen == 1).all()


def plan(shim, n, w, K, bits=False, codes=False, pageable=True):
    out = (C.c_uint64 * 3)()
    shim.fvt_plan_hash(n, w, -(-K // 64) * 8 if bits else 0, K if codes else 0, pageable, pageable, out)
    return bool(out[0]), bool(out[1]), out[2]


@pytest.mark.parametrize("K,w,bits,codes,largest", [(400, 1, False, True, 648), (400, 1, True, True, 569), (70, 11, False, True, 2299),
                                                    (70, 11, True, True, 2016), (2, 1, True, False, 21845), (2048, 64, True, True, 102)])
def test_largest_batch_of_the_one_buffer(shim, K, w, bits, codes, largest):
    """2^18 bytes of indices and codes."""
    for pageable in (True, False):
        assert plan(shim, largest, w, K, bits, codes, pageable) == (True, False, largest)
        assert plan(shim, largest + 1, w, K, bits, codes, pageable) == (False, False, largest + 1)


def test_batches_that_get_host_threads(shim):
    """Large results for ordinary memory, and any of more windows than a chunk: two streams' chunks overlap only if the
    host does not wait for each copy. Page-locked arrays need neither."""
    chunk = 1 << 17
    for n, K, kw in ((200000, 64, dict(bits=True)), (500000, 64, dict(bits=True)), (chunk + 1, 2, dict(bits=True)),
                     (200000, 20, dict(codes=True)), (10486, 400, dict(codes=True)), (1 << 20, 400, dict(bits=True, codes=True))):
        direct, crew, size = plan(shim, n, 11, K, **kw)
        assert not direct and crew and 0 < size <= chunk and size < n, (n, K)
        assert plan(shim, n, 11, K, pageable=False, **kw) == (False, False, min(n, chunk))
    for n, K, kw in ((chunk, 64, dict(bits=True)), (10485, 400, dict(codes=True)), (50000, 400, dict(bits=True)),
                     (1 << 20, 400, {})):
        assert plan(shim, n, 11, K, **kw) == (False, False, min(n, chunk)), (n, K)


@pytest.mark.parametrize("K,w,bits,codes", [(400, 1, False, True), (400, 11, True, False), (1000, 15, True, True), (2, 1, True, False),
                                            (2048, 64, False, True)])
def test_chunks_of_a_batch(shim, K, w, bits, codes):
    row = (-(-K // 64) * 8 if bits else 0) + (K if codes else 0)
    for n in (1, 655, 10486, 20000, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, 1 << 20, 10_000_019):
        direct, crew, size = plan(shim, n, w, K, bits, codes)
        assert 1 <= size <= min(n, 1 << 17)
        if crew:
            assert size * row >= 3 << 19 or size == 1 << 17  # a chunk is worth its launch and its copies


@pytest.mark.parametrize("n,K,w,bits,codes", [(20000, 400, 1, False, True), (10486, 400, 11, False, True), (100003, 400, 11, True, False),
                                              (100003, 400, 11, True, True), (1 << 20, 400, 11, True, False),
                                              (5000, 2048, 64, True, True), (200000, 2, 64, True, False)])
@pytest.mark.parametrize("got", [0, 1, 2, 3])
@pytest.mark.parametrize("indices", [False, True])
def test_staging_of_a_batch_fits_its_slots(shim, n, K, w, bits, codes, got, indices):
    """The chunks in flight take up to four slots, whatever the pool gives; what they write lies inside the slots and
    nowhere twice."""
    bits_row, codes_row = -(-K // 64) * 8 if bits else 0, K if codes else 0
    in_row, out_row = 4 * w if indices else 0, bits_row + codes_row
    out = (C.c_uint64 * 20)()
    shim.fvt_hash_stage(n, bits_row, codes_row, in_row, out_row, got, out)
    want, slots, chunk, lanes = out[:4]
    assert 1 <= want <= 4 and slots == (min(got, want) if got else want) and 1 <= chunk < n
    assert lanes == (4 if 4 * in_row <= out_row else 2)
    parts = []
    for lane in range(lanes):
        slot, at, in_slot, in_at = out[4 + 4 * lane:8 + 4 * lane]
        parts += [(slot, at, chunk * out_row), (in_slot, in_at, chunk * in_row)]
    for slot, at, size in parts:
        assert slot < slots and at + size <= shim.fvt_slot_bytes()
    for i, (slot, at, size) in enumerate(parts):
        for other, o_at, o_size in parts[i + 1:]:
            assert slot != other or at + size <= o_at or o_at + o_size <= at or not size or not o_size
