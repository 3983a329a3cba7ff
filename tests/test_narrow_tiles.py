"""The narrow tiles of the layer's SDD and DSD (64, 128 or 256 columns, for
layouts of few live row blocks).

On the CPU: their width rule and tile order, compiled from the kernels' own
functions, give every (row block, column slice) to exactly one of the CUs'
workgroups. On the GPU: every real row of H and y equals, bit for bit, what
the per-row-block kernels write for it (test_sdd_gpu.py and test_dsd_gpu.py pin
those to the oracle), at each width, tile height (1 to 4 groups of 32 rows)
and wave count, with experts of several row blocks under both of the stage's
choices.
"""
from __future__ import annotations

import ctypes

import pytest
import torch

from sparsebench_amd import _lib

CUS = 256


@pytest.fixture(scope="module")
def sched():
    path = _lib.LIB_PATH.with_name("libsparsebench_probe.so")
    if not path.exists():
        from sparsebench_amd.build import build

        build()
    _lib.lib()  # torch's HIP runtime first
    return ctypes.CDLL(str(path))


@pytest.mark.parametrize("columns", [256, 768, 1024, 1536, 2048, 4096, 14336, 16384])
@pytest.mark.parametrize("widest", [128, 256])
def test_width_rule_and_tile_order(sched, columns: int, widest: int) -> None:
    rb, sl = ctypes.c_int(), ctypes.c_int()
    for live in [0, 1, 2, 3, 4, 5, 7, 8, 9, 16, 17, 31, 32, 33, 64, 100, 128, 255, 256, 257, 5000]:
        width = sched.sbt_narrow_width(live, columns, widest, CUS)
        fits = [w for w in (64, 128, 256) if w <= widest and live * (columns // w) <= CUS]
        assert width == (fits[0] if live and fits else 0)
        if not width:
            continue
        slices = columns // width
        seen = []
        for bid in range(CUS):  # the launched grid holds at least one workgroup per CU
            sched.sbt_narrow_tile_for(bid, live, slices, ctypes.byref(rb), ctypes.byref(sl))
            if rb.value < live:
                assert 0 <= sl.value < slices
                seen.append((rb.value, sl.value))
        assert sorted(seen) == [(r, s) for r in range(live) for s in range(slices)]


@pytest.mark.parametrize("columns", [256, 768, 2048, 4352, 14336])
@pytest.mark.parametrize("widest", [128, 256])
def test_instances_without_narrow_tiles(sched, columns: int, widest: int) -> None:
    # Launched only when no layout of at least min_rows rows would take a narrow tile; always launched then.
    sched.sbt_may_be_narrow.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int, ctypes.c_int]
    for min_rows in [-5, 0, 1, 128, 129, 1000, 2047, 2048, 2049, 32768, 32769, 10**6, 2**40]:
        live = max(0, -(-min_rows // 128))
        widths = [sched.sbt_narrow_width(n, columns, widest, CUS) for n in range(live, CUS + 2)]
        assert bool(sched.sbt_may_be_narrow(min_rows, columns, widest, CUS)) == (live == 0 or any(widths))


SINGLE = [1, 33, 0, 70, 127]  # one row block each: 1, 2, 3 and 4 row groups
CASES = {
    # name: (rows per expert, D, F); the stages' widths follow from row blocks x columns
    "sdd64_dsd64": (SINGLE, 256, 512),
    "sdd128_dsd64_deep": (SINGLE, 256, 8192),  # F >= 8192: the DSD's 8 waves
    "sdd256_dsd64_deep": (SINGLE, 256, 16384),
    "sdd64_dsd128": (SINGLE, 8192, 256),
    "sdd128_dsd128_deep": (SINGLE, 8192, 8192),
    "sdd64_f768": (SINGLE, 256, 768),  # F % 512 != 0
    "sdd256_f8448": (SINGLE, 256, 8448),
    "one_copy": ([0, 1], 256, 512),
    "shortest": ([3, 31, 32], 256, 256),
    # Several row blocks an expert: whole under skew, cut when the expert tiles are the choice.
    "blocks_skewed": ([300, 129, 5, 128], 512, 2048),
    "blocks_balanced": ([200, 170, 257], 512, 2048),
    "blocks_f768": ([300, 129, 5, 128], 512, 768),
}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_rows_equal_the_row_block_kernels(case: str) -> None:
    from sparsebench_amd import _C
    from sparsebench_amd.routing import route_device
    from sparsebench_amd.spmm import dsd, sdd

    counts, d, f = CASES[case]
    e, t = len(counts), sum(counts)
    g = torch.Generator().manual_seed(7)
    idx = torch.repeat_interleave(torch.arange(e), torch.tensor(counts))
    idx = idx[torch.randperm(t, generator=g)].reshape(-1, 1).contiguous().cuda()
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(t, d, generator=g, device="cuda").bfloat16()
    w1 = (torch.randn(e, d, f, generator=g, device="cuda") / d**0.5).bfloat16()
    w2 = (torch.randn(e, f, d, generator=g, device="cuda") / f**0.5).bfloat16().view(e * f, d)
    topo = route_device(idx, e, f, 128)
    rows = (topo.row_token >= 0).nonzero().squeeze(1)

    def real(blocks: torch.Tensor) -> torch.Tensor:
        return blocks.view(-1, f // 128, 128, 128).permute(0, 2, 1, 3).reshape(-1, f)[rows]

    h = sdd(x, w1, topo)
    assert torch.equal(real(_C.sdd_experts_cuda(x, w1, topo, True)), real(h))
    assert torch.equal(_C.dsd_experts_cuda(h, w2, topo)[rows], dsd(h, w2, topo, version=5)[rows])
