"""Every tile form the SDD / DSD drop-ins pick, against the oracle.

sb_sdd / sb_dsd pick one tile form per shape and grid (sdd_form in
sdd_tile.hpp, dsd_form in dsd_tile.hpp, for 256 CUs). These tests reach each of
them through a call that selects it, which they check with the launch's own
rule compiled for the CPU, and hold it to the bf16 tolerance of the defaults
(1.6e-2). The DSD's pairs of 64-row blocks are in test_dsd_pairs_gpu.py.

  SDD  128 x 512, 3 stages (wide)         more tiles than CUs, D < 4096, F % 512 == 0
       128 x 512, 4 stages (deep)         the same, D >= 4096
       128 x 256 (narrow)                 more tiles than CUs and F % 512 != 0, or they fit 256 wide
       128 x 128 (half)                   they fit 128 wide
  DSD  512 wide, 4 waves (wide)           more tiles than CUs, D % 512 == 0, K < 8192
       512 wide, 8 waves (deep)           the same, K = F per expert >= 8192
       256 wide (mid), 128 wide (narrow)  they fit, or D % 512 != 0, D % 256 != 0
"""

import ctypes
import math

import numpy as np
import pytest
import torch

from oracle.moe_ref import dsd_rows, sdd_blocks
from oracle.topology_ref import build_layout
from sparsebench_amd import _lib
from sparsebench_amd.workloads import routing_case

pytestmark = pytest.mark.gpu

TOL = {"rtol": 1.6e-2, "atol": 1.6e-2}
CUS = 256
SDD_FORMS = ["wide", "deep", "narrow", "half"]  # SddTile


@pytest.fixture(scope="module")
def shims():
    _lib.lib()  # torch's HIP runtime first
    so = ctypes.CDLL(str(_lib.LIB_PATH.with_name("libsparsebench_probe.so")))
    so.sbt_sdd_form.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int]
    so.sbt_dsd_form.argtypes = [ctypes.c_int64] * 5 + [ctypes.c_int] * 2
    return so


@pytest.mark.parametrize(("form", "t", "e", "d_model", "ffn_dim"), [
    ("wide", 600, 8, 256, 8192), ("deep", 900, 4, 4096, 4096), ("narrow", 2500, 8, 256, 768),
    ("narrow", 450, 4, 256, 4096), ("half", 600, 8, 256, 512), ("half", 600, 8, 4096, 512), ("half", 600, 8, 256, 768),
])
@pytest.mark.parametrize("case", ["zipf", "empty_middle"])
def test_sdd_tile_forms(shims, form: str, t: int, e: int, d_model: int, ffn_dim: int, case: str) -> None:
    from sparsebench_amd.routing import route_device
    from sparsebench_amd.spmm import sdd

    g = torch.Generator().manual_seed(d_model + ffn_dim)
    idx = routing_case(case, t, e, seed=3)
    x = torch.randn(t, d_model, generator=g).bfloat16()
    w1 = (torch.randn(e, d_model, ffn_dim, generator=g) / d_model**0.5).bfloat16()
    dev = route_device(idx.cuda(), e, ffn_dim, 128)
    assert SDD_FORMS[shims.sbt_sdd_form(dev.row_block_expert.numel(), d_model, ffn_dim, CUS)] == form
    out = sdd(x.cuda(), w1.cuda(), dev)
    lay = build_layout(idx.numpy(), e, ffn_dim, 128)
    torch.testing.assert_close(out[: lay.col_indices.size].float().cpu(), sdd_blocks(x.float(), w1.float(), lay),
                               **TOL)


DSD_FORMS = {"wide": 512, "deep": 512 + 2, "mid": 256, "narrow": 128}


@pytest.mark.parametrize(("form", "rows", "d_model", "ffn_dim"), [
    # rows of each expert, in row blocks of bs (the middle one has none, and is not there in the deep case)
    ("wide", (10.2, 0, 9.4), 4096, 256), ("deep", (19.5,), 4096, 9216), ("mid", (10.2, 0, 9.4), 2048, 256),
    ("mid", (30.5, 0, 31.2), 768, 256), ("narrow", (10.2, 0, 9.4), 512, 256), ("narrow", (3.1, 0, 2.4), 768, 256),
    ("narrow", (10.2, 0, 9.4), 384, 256), ("narrow", (60.2, 0, 59.4), 640, 128),
])
@pytest.mark.parametrize("bs", [64, 128])
@pytest.mark.parametrize("version", [1, 4])
def test_dsd_tile_forms(shims, form: str, rows: tuple, d_model: int, ffn_dim: int, bs: int, version: int) -> None:
    from sparsebench_amd import _C

    g = torch.Generator().manual_seed(100 + d_model + bs)
    e = len(rows)
    idx = np.repeat(np.arange(e), [int(r * bs) for r in rows])
    lay = build_layout(np.random.default_rng(5).permutation(idx).reshape(-1, 1), e, ffn_dim, bs)
    blocks = (torch.randn(lay.col_indices.size, bs, bs, generator=g) / math.sqrt(ffn_dim)).bfloat16()
    w = torch.randn(e * ffn_dim, d_model, generator=g).bfloat16()
    # Worst-case buffers: two dead row blocks after the live ones.
    row_offsets = torch.cat([torch.as_tensor(lay.row_offsets), torch.full((2,), int(lay.row_offsets[-1]))]).int()
    picked = shims.sbt_dsd_form(bs, blocks.shape[0], w.shape[0], row_offsets.numel() - 1, d_model, 0, CUS)
    assert picked == DSD_FORMS[form]
    out = _C.dsd_cuda(blocks.cuda(), w.cuda(), row_offsets.cuda(), torch.as_tensor(lay.col_indices).cuda(), version)
    torch.testing.assert_close(out[: lay.num_rows].float().cpu(), dsd_rows(blocks.float(), w.float(), lay), **TOL)
    if version == 1:  # versions 1-3 write dead row blocks as zeros
        assert torch.all(out[lay.num_rows:] == 0)
