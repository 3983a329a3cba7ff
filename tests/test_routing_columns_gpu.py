"""Routing beyond 32 chunks of 1024 copies, where a columns kernel sums the
per-chunk counts: expert counts on both sides of its 8 columns a workgroup,
chunk counts on both sides of its 128 runs a column, bit for bit against the
layout oracle."""

import numpy as np
import pytest
import torch

from oracle.topology_ref import device_layout

pytestmark = pytest.mark.gpu

FIELDS = ("tokens_per_expert", "padded_offsets", "row_token", "copy_row", "row_block_expert", "row_offsets",
          "col_indices")


@pytest.mark.parametrize("num_experts", [1, 7, 8, 15, 16, 1023])
@pytest.mark.parametrize("copies", [32 * 1024 + 1, 128 * 1024, 128 * 1024 + 1])
def test_matches_oracle(num_experts: int, copies: int) -> None:
    from sparsebench_amd.routing import route_device

    g = torch.Generator().manual_seed(copies + num_experts)
    # A few ids out of range: column E and the error flag.
    idx = torch.randint(0, num_experts, (copies, 1), generator=g)
    idx[torch.randint(0, copies, (5,), generator=g)] = num_experts
    dev = route_device(idx.cuda(), num_experts, 32, 16)
    want = device_layout(idx.numpy(), num_experts, 32, 16)
    for f in FIELDS:
        np.testing.assert_array_equal(getattr(dev, f).cpu().numpy(), getattr(want, f), err_msg=f)
    assert int(dev.error.item()) == want.error == 1
