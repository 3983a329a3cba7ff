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
RANDOM = [(256, 64, 1024, 0.5), (64, 64, 4096, 0.5), (128, 64, 2048, 0.25), (512, 128, 512, 0.1), (40, 16, 8192, 0.5),
          (1024, 8, 512, 16)]


@pytest.mark.parametrize(("rb", "cols", "d", "share"), RANDOM)
def test_pairs_only_for_routing_layouts(form, rb: int, cols: int, d: int, share: float) -> None:
    nnz, w_rows = int(rb * cols * share), cols * 64
    assert form(64, nnz, w_rows, rb, d, 1, CUS) & 1  # by size alone they would take pairs
    assert not form(64, nnz, w_rows, rb, d, 0, CUS) & 1
    assert not form(128, nnz, w_rows * 2, rb, d, 1, CUS) & 1


@pytest.mark.parametrize("rb", [1, 7, 64, 1000])
def test_fewer_blocks_than_rows(form, rb: int) -> None:
    assert not form(64, rb - 1, 512, rb, 512, 1, CUS) & 1
