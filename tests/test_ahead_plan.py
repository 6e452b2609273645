"""Which source rows a layout reads ahead for the dispatch behind it: every index and the amount, on the host (the arithmetic is the
kernel's own), and where the library reads ahead at all."""

import ctypes
import shutil
import subprocess

import numpy as np
import pytest

import cabi

MIB = 1 << 20


@pytest.fixture(scope="module")
def ahead(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no C++ compiler")
    library = tmp_path_factory.mktemp("ahead") / "ahead_plan.so"
    subprocess.run(
        ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-I/opt/rocm/include",
         f"-I{cabi.ROOT / 'nanoep_amd' / 'csrc'}", str(cabi.ROOT / "tests" / "ahead_plan.cpp"), "-o", str(library)],
        check=True, capture_output=True, text=True,
    )
    handle = ctypes.CDLL(str(library))
    i64, p = ctypes.c_int64, ctypes.c_void_p
    handle.plan.argtypes = [i64] * 6 + [ctypes.POINTER(i64)]
    handle.bytes_of.argtypes, handle.bytes_of.restype = [i64] * 6, i64
    handle.walk.argtypes, handle.walk.restype = [i64] * 6 + [p, p, i64], i64
    return handle


# One row and rows of one vector, shares that end inside a wavefront's vectors, the last XCDs' empty, as many rows as are read and
# one more, workgroups of 2, 7 and 16 wavefronts, forced XCD counts.
@pytest.mark.parametrize("xcds", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("block_waves", [2, 7, 16])
@pytest.mark.parametrize(
    "tokens,row_vectors,window",
    [(1, 1, 256), (33, 32, 256), (256, 896, 256), (257, 129, 64), (1024, 256, 128), (1025, 256, 128), (1537, 352, 128), (4096, 896, 256),
     (32767, 32, 1024)],
)
def test_every_vector_read_ahead_is_a_source_row_and_within_the_limit(ahead, tokens, row_vectors, window, block_waves, xcds):
    out = (ctypes.c_int64 * 3)()
    for limit in (MIB, 2 * MIB, 8 * MIB):
        ahead.plan(tokens, row_vectors, window, xcds, block_waves, limit, out)
        blocks, vectors, share = out
        assert vectors == tokens * row_vectors and blocks % xcds == 0
        assert (blocks > 0) == (xcds * block_waves * 8192 <= limit)  # a workgroup for every XCD, 8 KiB a wavefront
        for work_blocks in (1, 26, 251):
            reader, xcd_of = np.zeros(vectors, np.uint8), np.full(vectors, -1, np.int8)
            largest = ahead.walk(blocks, vectors, share, work_blocks, xcds, block_waves, reader.ctypes.data, xcd_of.ctypes.data, vectors)
            assert largest < vectors
            assert reader.max() <= 1  # nothing twice
            total = int(reader.sum()) * 16
            assert total <= limit and total == ahead.bytes_of(blocks, vectors, share, work_blocks, xcds, block_waves)
            whole = block_waves * 512 * (blocks // xcds)  # vectors an XCD may read
            for xcd in range(xcds):
                read = np.flatnonzero(xcd_of == xcd)
                first, end = xcd * share, min((xcd + 1) * share, vectors)
                assert len(read) == max(0, min(end - first, whole))  # the start of the XCD's share, without a gap
                assert len(read) == 0 or (read[0] == first and read[-1] == first + len(read) - 1)


def test_rows_beyond_the_index_range_are_not_read_ahead(ahead):
    out = (ctypes.c_int64 * 3)()
    ahead.plan(1 << 20, 2048, 256, 8, 8, 2 * MIB, out)
    assert list(out) == [0, 0, 0]


def bytes_ahead(tokens, topk, experts, hidden):
    return cabi.lib().nanoep_layout_ahead_bytes(tokens, topk, experts, hidden)


def test_how_much_a_layout_reads_ahead():
    with cabi.forced_tuning({"XCDS": 8}):
        assert bytes_ahead(16, 2, 2, 256) == 16 * 512  # all of a small batch
        assert 3 * MIB < bytes_ahead(1537, 6, 60, 2816) <= 4 * MIB
        assert 3 * MIB < bytes_ahead(4096, 8, 256, 7168) <= 4 * MIB
        assert 4 * MIB < bytes_ahead(32768, 8, 64, 512) <= 8 * MIB
        for refused in ((0, 2, 2, 256), (16, 0, 2, 256), (16, 33, 64, 256), (16, 2, 0, 256), (16, 2, 3840, 256), (16, 2, 2, 0), (16, 2, 2, 252)):
            assert bytes_ahead(*refused) == 0


def test_nothing_is_read_ahead_where_no_list_is_walked():
    with cabi.forced_tuning({"XCDS": 8}):
        assert bytes_ahead(300, 8, 64, 32768) > 0 and bytes_ahead(300, 8, 64, 32776) == 0  # rows beyond 64 KiB
        assert bytes_ahead(1 << 26, 8, 64, 8) == 0  # lists of 2^29 entries
        for switch in ("DISPATCH_PREFETCH", "DISPATCH_ORDER"):
            with cabi.forced_tuning({switch: 0}):
                for batch in ((16, 2, 2, 256), (256, 8, 64, 4096), (1537, 6, 60, 2816), (32768, 8, 64, 512)):
                    assert bytes_ahead(*batch) == 0
        with cabi.forced_tuning({"DISPATCH_PREFETCH": 1}):
            assert bytes_ahead(256, 8, 64, 4096) > 0


# 4 MiB are 64 workgroups of eight wavefronts or 32 of sixteen: with 128 or 160 of the assignment's own three quarters of the compute units
# have one.  2 MiB are half as many: with 224 or 240 all have one.
@pytest.mark.parametrize("topk,hidden,most,some", [(8, 2048, 8128, 14272), (8, 512, 20352, 30592)])
def test_less_is_read_beside_an_assignment_that_leaves_less_room(topk, hidden, most, some):
    with cabi.forced_tuning({"XCDS": 8}):
        assert cabi.device_topology()[0] == 256
        assert bytes_ahead(most, topk, 64, hidden) == 4 * MIB and bytes_ahead(most + 1, topk, 64, hidden) == 2 * MIB
        assert bytes_ahead(some, topk, 64, hidden) == 2 * MIB and bytes_ahead(some + 1, topk, 64, hidden) == 0
        assert bytes_ahead(32767, topk, 64, hidden) == 0
