"""Which tiles sb_dsd runs, compiled for the CPU from the launch's own rule: row
blocks of 64 go in pairs only where the caller says that they are a routing
layout's, whose neighbours share their block columns."""

import ctypes

import pytest

from sparsebench_amd import _lib

CUS = 256


@pytest.fixture(scope="module")
def form():
    path = _lib.LIB_PATH.with_name("libsparsebench_probe.so")
    if not path.exists():
        from sparsebench_amd.build import build

        build()
    _lib.lib()  # torch's HIP runtime first
    fn = ctypes.CDLL(str(path)).sbt_dsd_form
    fn.argtypes = [ctypes.c_int64] * 5 + [ctypes.c_int] * 2
    return fn


# (row blocks, block columns, D, share of the blocks held)
RANDOM = [(300, 64, 1024, 0.5), (96, 64, 4096, 0.5), (150, 64, 2048, 0.25), (640, 128, 512, 0.1), (40, 16, 8192, 0.5),
          (1024, 8, 512, 16)]


@pytest.mark.parametrize(("rb", "cols", "d", "share"), RANDOM)
def test_pairs_only_for_routing_layouts(form, rb: int, cols: int, d: int, share: float) -> None:
    nnz, w_rows = int(rb * cols * share), cols * 64
    assert form(64, nnz, w_rows, rb, d, 1, CUS) & 1  # by size alone they would take pairs
    assert not form(64, nnz, w_rows, rb, d, 0, CUS) & 1
    assert not form(128, nnz, w_rows * 2, rb, d, 1, CUS) & 1


@pytest.mark.parametrize(("e", "d", "rows", "paired"), [
    # rows: row blocks that hold rows; one expert's odd one out and the worst case add up to E more
    (16, 1024, 63, True), (2, 768, 104, True), (1, 512, 158, True),     # the pairs leave CUs enough
    (2, 768, 146, True), (4, 768, 122, True), (8, 768, 120, False),     # the fewer, the more experts
    (4, 1536, 66, False), (2, 768, 158, False), (16, 512, 400, False),  # one round, nearly full
    (16, 1024, 122, False),                                             # one by one may be one round
    (20, 1024, 80, False),                                              # many row blocks alone
    (2, 512, 510, False), (16, 512, 545, True), (16, 1024, 290, True),  # just over one round, or surely more
])
def test_pairs_leave_room_for_row_blocks_alone(form, e: int, d: int, rows: int, paired: bool) -> None:
    ffn, rb = 2048, rows + e
    assert bool(form(64, rb * (ffn // 64), e * ffn, rb, d, 1, CUS) & 1) == paired


@pytest.mark.parametrize("rb", [1, 7, 64, 1000])
def test_fewer_blocks_than_rows(form, rb: int) -> None:
    assert not form(64, rb - 1, 512, rb, 512, 1, CUS) & 1
