"""Routing of up to 1024 copies, in one launch: copy counts around its waves and
around the bound to the two-launch form, bad ids and valid_tokens, bit for bit
against the layout oracle."""

import numpy as np
import pytest
import torch

from oracle.topology_ref import device_layout

pytestmark = pytest.mark.gpu

FIELDS = ("tokens_per_expert", "padded_offsets", "row_token", "copy_row", "row_block_expert", "row_offsets",
          "col_indices")


@pytest.mark.parametrize("num_experts", [1, 5, 64, 1024])
@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 511, 512, 513])
@pytest.mark.parametrize("form", ["plain", "bad ids", "valid tokens"])
def test_matches_oracle(num_experts: int, tokens: int, form: str) -> None:
    from sparsebench_amd.routing import route_device

    g = torch.Generator().manual_seed(tokens + num_experts)
    idx = torch.randint(0, num_experts, (tokens, 2), generator=g)
    valid, live = None, tokens
    if form == "bad ids":
        idx[tokens // 2, 1], idx[tokens - 1, 0] = num_experts, -1
    elif form == "valid tokens":
        live = (tokens + 1) // 2
        valid = torch.tensor([live], dtype=torch.int32, device="cuda")
    dev = route_device(idx.cuda(), num_experts, 256, 128, valid)
    want = device_layout(idx.numpy(), num_experts, 256, 128, **({"valid_tokens": live} if valid is not None else {}))
    for f in FIELDS:
        np.testing.assert_array_equal(getattr(dev, f).cpu().numpy(), getattr(want, f), err_msg=f)
    assert int(dev.error.item()) == want.error
