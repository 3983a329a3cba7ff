"""DSD and SDD of the drop-in kernels at each tile width that the grid's size
selects (128, 256, 512 columns), and the DSD's pairs of 64-row blocks: pairs
with the same columns, neighbours with other columns or another block count,
an odd last row block and dead ones, against the oracle."""

import ctypes
import math

import numpy as np
import pytest
import torch

from oracle.moe_ref import dsd_rows, sdd_blocks
from oracle.topology_ref import build_layout
from sparsebench_amd import _lib

pytestmark = pytest.mark.gpu

TOL = {"rtol": 1.6e-2, "atol": 1.6e-2}


def routed(counts: list[int], seed: int) -> np.ndarray:
    idx = np.repeat(np.arange(len(counts)), counts)
    return np.random.default_rng(seed).permutation(idx).reshape(-1, 1)


@pytest.fixture(scope="module")
def form():
    """The launch's own rule, for 256 CUs: width + 1 in pairs + 2 deep."""
    _lib.lib()  # torch's HIP runtime first
    fn = ctypes.CDLL(str(_lib.LIB_PATH.with_name("libsparsebench_probe.so"))).sbt_dsd_form
    fn.argtypes = [ctypes.c_int64] * 5 + [ctypes.c_int] * 2
    return fn


PAIRED, DEEP = 1, 2


@pytest.mark.parametrize(("counts", "d", "f", "want"), [
    # rows per expert; the row blocks and D choose the form
    ([520], 8192, 256, 256 + PAIRED),               # 512 wide they leave CUs idle, in pairs 256 wide fit
    ([2000, 2100], 1024, 256, 256 + PAIRED),        # the same, an odd row block of one expert
    ([4000, 1, 3900], 1536, 128, 512),              # one round of pairs would be nearly full
    ([4200, 250, 4300], 1024, 256, 512 + PAIRED),   # pairs leave room
    ([8700, 130, 9000], 1024, 256, 512 + PAIRED),   # pairs are more than one round
    ([2000, 2100, 2000], 768, 1024, 256 + PAIRED),  # D % 512 != 0
    ([1050], 8192, 9216, 512 + PAIRED + DEEP),
    ([700, 650], 512, 256, 128), ([70, 1, 64], 512, 256, 128), ([2600], 1536, 64, 256),
])
def test_block_64_against_oracle(form, counts: list[int], d: int, f: int, want: int) -> None:
    from sparsebench_amd import _C

    e = len(counts)
    lay = build_layout(routed(counts, d), e, f, 64)
    g = torch.Generator().manual_seed(f)
    blocks = (torch.randn(lay.col_indices.size, 64, 64, generator=g) / math.sqrt(f)).bfloat16()
    w = torch.randn(e * f, d, generator=g).bfloat16()
    dead = 1
    offsets = torch.cat([torch.as_tensor(lay.row_offsets), torch.full((dead,), int(lay.row_offsets[-1]))]).int()
    assert form(64, blocks.shape[0], w.shape[0], offsets.numel() - 1, d, 1, 256) == want
    out = _C.dsd_cuda(blocks.cuda(), w.cuda(), offsets.cuda(), torch.as_tensor(lay.col_indices).cuda(), 1, routed=True)
    torch.testing.assert_close(out[: lay.num_rows].float().cpu(), dsd_rows(blocks.float(), w.float(), lay), **TOL)
    assert torch.all(out[lay.num_rows:] == 0)


@pytest.mark.parametrize("routed", [False, True])
@pytest.mark.parametrize("version", [1, 4])
def test_block_64_any_bsr(version: int, routed: bool) -> None:
    # Not a routing layout: block counts and columns differ from row to row, in an order of their own, some repeated,
    # some out of w's range (they add nothing); 41 row blocks over one "expert" take the pairs
    # when they are said to be a routing layout's.
    from sparsebench_amd import _C

    rng = np.random.default_rng(5)
    d, col_blocks, rows = 8192, 8, 41
    cols: list[list[int]] = []
    for r in range(rows):
        if r % 4 == 1:
            cols.append(list(cols[-1]))  # the pair's columns, the same
        elif r % 4 == 3:
            cols.append(list(cols[-1][::-1]) if r % 8 == 3 else cols[-1][:-1])  # other order, or fewer
        else:
            n = 0 if r == 20 else int(rng.integers(6, 9))
            cols.append([int(c) for c in rng.integers(0, col_blocks + (1 if r > 30 else 0), size=n)])
    offsets = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    flat = np.concatenate([np.asarray(c, dtype=np.int32) for c in cols])
    g = torch.Generator().manual_seed(2)
    blocks = (torch.randn(flat.size, 64, 64, generator=g) / 20).bfloat16()
    w = torch.randn(col_blocks * 64, d, generator=g).bfloat16()
    out = _C.dsd_cuda(blocks.cuda(), w.cuda(), torch.as_tensor(offsets).cuda(), torch.as_tensor(flat).cuda(), version,
                      routed=routed)
    wide = torch.cat([w.float(), torch.zeros(64, d)])  # the block past w
    for r in range(rows):
        if not cols[r] and version == 4:
            continue
        want = torch.zeros(64, d)
        for i, c in enumerate(cols[r]):
            want += blocks[offsets[r] + i].float() @ wide[c * 64:(c + 1) * 64]
        torch.testing.assert_close(out[r * 64:(r + 1) * 64].float().cpu(), want, **TOL)


@pytest.mark.parametrize("version", [1, 4])
def test_block_64_long_rows_among_short_ones(version: int) -> None:
    # Row blocks of 65536 blocks (columns repeated), more than a pair takes, as the first and the second of theirs,
    # in a layout that takes pairs. Small whole numbers: every sum is exact, up to the rounding of the result.
    from sparsebench_amd import _C

    d, col_blocks, rows, long = 512, 8, 1024, {0, 3}
    counts = torch.tensor([65536 if r in long else 8 for r in range(rows)])
    offsets = torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)])
    nnz = int(offsets[-1])
    g = torch.Generator(device="cuda").manual_seed(4)
    blocks = torch.randint(-1, 2, (nnz, 64, 64), generator=g, device="cuda", dtype=torch.int8).bfloat16()
    w = torch.randint(-1, 2, (col_blocks * 64, d), generator=g, device="cuda", dtype=torch.int8).bfloat16()
    cols = (torch.arange(nnz, device="cuda") % col_blocks).int()
    out = _C.dsd_cuda(blocks, w, offsets.int().cuda(), cols, version, routed=True)
    for r in (0, 1, 2, 3, 4, 5, rows - 1):
        own = blocks[offsets[r]: offsets[r + 1]].view(-1, col_blocks, 64, 64).sum(0, dtype=torch.float32)
        want = own.permute(1, 0, 2).reshape(64, -1).double() @ w.double()
        assert torch.equal(out[r * 64: (r + 1) * 64], want.bfloat16()), r


@pytest.mark.parametrize(("counts", "d", "f"), [
    ([100, 300], 256, 512), ([100, 300], 128, 8192), ([100, 300], 64, 16384), ([200, 5], 64, 33024), ([130], 64, 768),
])
def test_sdd_widths(counts: list[int], d: int, f: int) -> None:
    from sparsebench_amd.routing import route_device
    from sparsebench_amd.spmm import sdd

    e = len(counts)
    idx = routed(counts, f)
    g = torch.Generator().manual_seed(d)
    x = torch.randn(idx.shape[0], d, generator=g).bfloat16()
    w1 = (torch.randn(e, d, f, generator=g) / d**0.5).bfloat16()
    lay = build_layout(idx, e, f, 128)
    out = sdd(x.cuda(), w1.cuda(), route_device(torch.as_tensor(idx).cuda(), e, f, 128))
    torch.testing.assert_close(out[: lay.col_indices.size].float().cpu(), sdd_blocks(x.float(), w1.float(), lay), **TOL)


@pytest.mark.parametrize(("counts", "d", "f", "want"), [
    ([100, 300], 256, 256, 128), ([100, 300], 8192, 256, 128), ([400, 300], 8192, 256, 256),
    ([300, 200], 32768, 128, 512),
])
def test_dsd_widths_block_128(form, counts: list[int], d: int, f: int, want: int) -> None:
    from sparsebench_amd import _C

    e = len(counts)
    lay = build_layout(routed(counts, d), e, f, 128)
    g = torch.Generator().manual_seed(f + d)
    blocks = (torch.randn(lay.col_indices.size, 128, 128, generator=g) / math.sqrt(f)).bfloat16()
    w = torch.randn(e * f, d, generator=g).bfloat16()
    assert form(128, blocks.shape[0], w.shape[0], len(lay.row_offsets) - 1, d, 0, 256) == want
    out = _C.dsd_cuda(blocks.cuda(), w.cuda(), torch.as_tensor(lay.row_offsets).int().cuda(),
                      torch.as_tensor(lay.col_indices).cuda(), 1)
    torch.testing.assert_close(out.float().cpu(), dsd_rows(blocks.float(), w.float(), lay), **TOL)
