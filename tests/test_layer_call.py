"""The layer as one native call (sb_layer and its variants): what it refuses, on
the CPU; on the GPU, the same bits as the stages called one by one, for every
operand form that it takes or leaves to them, and the stages' errors."""

import ctypes

import pytest
import torch

from sparsebench_amd import _lib


@pytest.fixture(scope="module")
def lib():
    if not _lib.LIB_PATH.exists():
        from sparsebench_amd.build import build

        build()
    return _lib.lib()


@pytest.mark.parametrize(("tokens", "copies", "e", "d", "f"), [
    (0, 0, 8, 256, 512), (0, 16, 0, 256, 512), (0, 16, 1025, 256, 512), (0, 16, 8, 128, 512), (0, 16, 8, 256, 384),
    (0, 16, 8, 0, 512), (0, 16, 8, 256, 0), (0, 2**33, 8, 256, 512),
    (0, 2**20, 8, 256, 1024),  # H of 2 GiB
    (0, 16, 8, 2**15, 2**15),  # one expert's W1 of 2 GiB
])
def test_sizes_refuse(lib, tokens, copies, e, d, f) -> None:
    size = ctypes.c_int64(-1)
    assert lib.sb_layer_sizes(tokens, copies, e, d, f, ctypes.byref(size)) == 1
    assert size.value == -1 and lib.sb_last_error()


def test_sizes_and_workspace_check(lib) -> None:
    size, listed = ctypes.c_int64(), ctypes.c_int64()
    assert lib.sb_layer_sizes(0, 512, 8, 256, 512, ctypes.byref(size)) == 0
    rows = (512 + 8 * 127) // 128 * 128
    assert size.value >= rows * (512 + 256) * 2 and size.value % 256 == 0
    assert lib.sb_layer_sizes(256, 512, 8, 256, 512, ctypes.byref(listed)) == 0
    assert listed.value >= size.value + (256 + 1 + 512) * 4
    args = [None, None, 0, None, 0, None, None, None, 4096, size.value - 1, 256, 2, 8, 256, 512, None, None]
    assert lib.sb_layer(*args) == 1 and b"workspace" in lib.sb_last_error()
    args[8] = 4096 + 16
    assert lib.sb_layer(*args) == 1 and b"aligned" in lib.sb_last_error()


def layer(t=300, e=8, d=256, f=512, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(t, d, generator=g, device="cuda").bfloat16()
    w1 = (torch.randn(e, d, f, generator=g, device="cuda") / d**0.5).bfloat16()
    w2 = (torch.randn(e, f, d, generator=g, device="cuda") / f**0.5).bfloat16()
    idx = torch.rand(t, e, generator=g, device="cuda").topk(2, dim=-1).indices
    gates = torch.softmax(torch.randn(t, 2, generator=g, device="cuda"), dim=-1)
    return x, idx, gates, w1, w2


def staged(stage: str) -> None:
    """A mark, so that the layer runs stage by stage."""


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "int32", "bf16", "fp16", "fp64 gates", "transposed gates", "valid_tokens",
                                  "bad ids", "one token", "not 16-byte aligned"])
def test_same_bits_as_the_stages(form: str) -> None:
    from sparsebench_amd.moe import moe_forward

    x, idx, gates, w1, w2 = layer(1 if form == "one token" else 300)
    valid, rows = None, x.shape[0]
    if form == "int32":
        idx = idx.int()
    elif form in ("bf16", "fp16", "fp64 gates"):
        gates = gates.to({"bf16": torch.bfloat16, "fp16": torch.float16, "fp64 gates": torch.float64}[form])
    elif form == "transposed gates":
        gates = gates.t().contiguous().t()
    elif form == "valid_tokens":
        valid, rows = torch.tensor([77], dtype=torch.int32, device="cuda"), 77
    elif form == "bad ids":
        idx[3, 0], idx[5] = 8, -1
    elif form == "not 16-byte aligned":
        flat = torch.empty(x.numel() + 1, dtype=x.dtype, device="cuda")
        flat[1:] = x.reshape(-1)
        x = flat[1:].view(x.shape)
        for mark in ({}, {"mark": staged}):
            with pytest.raises(RuntimeError, match="16-byte aligned"):
                moe_forward(x, idx, gates, w1, w2, **mark)
        return
    got = moe_forward(x, idx, gates, w1, w2, valid_tokens=valid)
    want = moe_forward(x, idx, gates, w1, w2, mark=staged, valid_tokens=valid)
    assert torch.equal(got[:rows], want[:rows])


@pytest.mark.gpu
@pytest.mark.parametrize("routed", ["all", "few"])
@pytest.mark.parametrize(("t", "e", "d", "f"), [
    (2048, 8, 1280, 4096),  # neither stage can be narrow
    (2048, 8, 512, 4096), (512, 2, 8192, 512),  # the SDD cannot; the DSD cannot
    (1024, 4, 2304, 8192), (512, 2, 8192, 8192),  # the same with the DSD's 8 waves: neither; the DSD
    (2048, 8, 1280, 4352),  # F % 512 != 0
])
def test_instances_without_narrow_tiles_same_bits(t: int, e: int, d: int, f: int, routed: str) -> None:
    # The one call launches its stages without narrow tiles where 2 T routed copies rule them out; stage by stage
    # they are always there. With most ids out of range few row blocks live after all: the same rows still.
    from sparsebench_amd.moe import moe_forward

    x, idx, gates, w1, w2 = layer(t, e, d, f)
    if routed == "few":
        idx[3:] = e
    got = moe_forward(x, idx, gates, w1, w2)
    assert torch.equal(got, moe_forward(x, idx, gates, w1, w2, mark=staged))


@pytest.mark.gpu
@pytest.mark.parametrize("index", [torch.int32, torch.int64])
def test_assigned_and_rounded_same_bits(index: torch.dtype) -> None:
    from sparsebench_amd.moe import moe_forward_assigned, moe_forward_rounded

    x, idx, gates, w1, w2 = layer()
    order = torch.argsort(idx.reshape(-1), stable=True)
    token, expert = (order // 2).to(index), idx.reshape(-1)[order].to(index)
    weight = gates.reshape(-1)[order]
    for tok, exp, wt in ((token, expert, weight), (token.view(-1, 1), expert, weight.bfloat16()),
                         (token, expert, weight.double())):
        got = moe_forward_assigned(x, tok, exp, wt, w1, w2)
        assert torch.equal(got, moe_forward_assigned(x, tok, exp, wt, w1, w2, mark=staged))
    g = torch.Generator(device="cuda").manual_seed(1)
    scores = torch.softmax(torch.randn(300, 8, generator=g, device="cuda"), dim=-1)
    for tile in (16, 128):
        got = moe_forward_rounded(x, scores, 2, w1, w2, tile)
        assert torch.equal(got, moe_forward_rounded(x, scores, 2, w1, w2, tile, mark=staged))


@pytest.mark.gpu
@pytest.mark.parametrize("break_it", ["cpu idx", "float idx", "fp32 x", "odd D", "too many experts"])
def test_refused_as_by_the_stages(break_it: str) -> None:
    from sparsebench_amd.moe import moe_forward

    x, idx, gates, w1, w2 = layer(20, 1025 if break_it == "too many experts" else 8, 128 if break_it == "odd D" else 256,
                                  256)
    if break_it == "cpu idx":
        idx = idx.cpu()
    elif break_it == "float idx":
        idx = idx.float()
    elif break_it == "fp32 x":
        x = x.float()
    seen = []
    for mark in ({}, {"mark": staged}):
        with pytest.raises(RuntimeError) as e:
            moe_forward(x, idx, gates, w1, w2, **mark)
        seen.append(str(e.value))
    assert seen[0] == seen[1]
