"""Which gate calls of several positions read the rows once for all of them (gemv_batch_take, gemv.hip): the lines
of the rule, on both sides, for the MI355X's 256 compute units.  Also what the GPU tests of that kernel rely on: that
their shapes reach it."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def shared():
    with open(os.path.join(ROOT, "larql_amd", "csrc", "kernels.h")) as f:
        text = f.read()
    kind = {n: int(re.search(rf"KIND_{n} = (\d+)", text).group(1)) for n in ("BF16", "F16", "F32")}
    take = C.CDLL(os.path.join(ROOT, "larql_amd", "liblarql_hip.so"))["_ZN5larql15gemv_batch_takeEimmmmjj"]  # gemv_batch_take(int, 4 x uint64_t, 2 x uint32_t)
    take.restype, take.argtypes = C.c_uint32, [C.c_int] + [C.c_uint64] * 4 + [C.c_uint32] * 2
    return lambda fmt, rows, k, batch, layers=1: take(kind[fmt], rows, k, batch, layers, 256, 2) > 1


@pytest.mark.parametrize("fmt,rows,k,batch,want", [
    # jobs that end with a workgroup's share meet in the L2: read together, two positions never share
    ("F16", 10240, 2560, 2, False), ("F32", 16384, 2048, 2, False), ("BF16", 16384, 3584, 2, False), ("F32", 16000, 3584, 2, True),
    ("F32", 8192, 8192, 2, True), ("F16", 16384, 8192, 2, True),
    # four: 16-bit rows late, f32 rows and those with two blocks of 256 threads a CU from 100 MB on
    ("F16", 10240, 2560, 4, False), ("F16", 8192, 2560, 4, False), ("F16", 8200, 2560, 4, True), ("F16", 8192, 2048, 4, True), ("BF16", 10240, 4096, 4, True),
    ("BF16", 12288, 3584, 4, False), ("F32", 10240, 2560, 4, True), ("F32", 16384, 640, 4, False), ("F16", 16384, 1280, 4, False),
    # eight
    ("F16", 16384, 640, 8, False), ("F16", 10240, 2560, 8, True), ("F32", 4096, 1024, 8, True), ("F16", 2048, 1280, 8, False),
    # positions that read apart: by size alone
    ("F16", 9000, 2560, 4, True), ("F32", 2300, 1280, 3, False), ("F32", 3700, 1280, 3, True), ("BF16", 12000, 528, 5, False), ("BF16", 3500, 2064, 5, True),
    # several jobs
    ("F32", 2048, 640, 12, False), ("F32", 1500, 1536, 9, False), ("F32", 5000, 2560, 9, True), ("F16", 8192, 1280, 16, False), ("F16", 6144, 1280, 16, True),
    ("F16", 14336, 768, 12, False), ("F16", 13000, 768, 12, True), ("F16", 1700, 2560, 9, False), ("F16", 1500, 2560, 11, True), ("F32", 1304, 1536, 11, True), ("BF16", 4096, 1552, 12, True),
])
def test_lines(shared, fmt, rows, k, batch, want):
    assert shared(fmt, rows, k, batch) == want


def test_positions_that_meet_share_over_several_layers(shared):
    assert not shared("F16", 8192, 2560, 2) and shared("F16", 8192, 2560, 2, 8) and shared("F32", 10240, 1024, 2, 16)


def test_shapes_of_the_gpu_tests(shared):
    for fmt in ("BF16", "F16", "F32"):
        for rows, k, batch in ((400009, 16, 8), (50021, 208, 8), (30011, 656, 5), (5003, 4352, 12), (1500, 5136, 7), (4001, 4608, 8)):
            assert shared(fmt, rows, k, batch), (fmt, rows, k, batch)
    for fmt, k in (("BF16", 2064), ("F16", 2560), ("F32", 1040)):
        for batch in (3, 8):
            assert shared(fmt, 2003, k, batch, 11), (fmt, k, batch)


def test_never_for_rows_the_kernel_does_not_take(shared):
    assert not shared("F32", 16000, 8208, 4) and not shared("F16", 16000, 8200, 4)   # longer than 512 slices of 16
