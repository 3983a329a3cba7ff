"""Token grouping at the edges of its workgroups (128 tokens each), of the
lists it ranks in LDS (64 copies a token) and of the copies that LDS holds
(8192 a workgroup), of the lists it holds in registers (256 to 8192 copies) and
of those it takes in passes (524288 on): every way of placing a copy, against a
stable sort."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["sorted", "sorted, all routed", "shuffled"])
@pytest.mark.parametrize(("num_tokens", "n", "hot"), [
    (127, 400, 0), (128, 1024, 0), (129, 1025, 0), (32768, 40000, 0), (40000, 30000, 0),
    (1, 65, 0), (1, 64, 0),  # one token's list just past, and at, what is ranked
    (1, 9000, 0), (300, 9000, 8500),  # a token with most of the copies
    (64, 64 * 140, 0),  # many copies a token: fewer tokens a workgroup
    (1, 1, 0), (1000, 3, 0), (200, 256, 0), (200, 257, 0), (700, 1024, 100), (700, 2048, 0), (2000, 2049, 0),
    (5, 4097, 0), (4096, 8192, 0), (4096, 8193, 0),
    # in passes: short lists, one past what a lane sorts, one at and one past what LDS sorts, and a token alone
    (1 << 19, (1 << 19) - 1, 0), (150000, 1 << 19, 0), (150000, (1 << 19) + 77, 65), (20000, (1 << 19) + 77, 0),
    (128, 1 << 19, 0), (3000, (1 << 19) + 1, 30000), (1, 1 << 19, 0),
])
@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_matches_stable_sort(order: str, num_tokens: int, n: int, hot: int, dtype: torch.dtype) -> None:
    from sparsebench_amd import _C

    rng = np.random.default_rng(n + num_tokens)
    token = rng.integers(0, num_tokens, size=n)
    token[:hot] = num_tokens // 2
    if order == "shuffled":
        rng.shuffle(token)
    else:
        token = np.sort(token)
    copy_row = np.where((rng.random(n) > 0.05) | (order == "sorted, all routed"), np.arange(n), -1).astype(np.int32)
    listed = np.nonzero((copy_row >= 0))[0]
    want = listed[np.argsort(token[listed], kind="stable")]
    offs, copies = _C.token_csr_cuda(torch.from_numpy(token).to(dtype).cuda(), torch.from_numpy(copy_row).cuda(),
                                     num_tokens)
    counts = np.bincount(token[listed], minlength=num_tokens)
    assert np.array_equal(offs.cpu().numpy(), np.concatenate([[0], np.cumsum(counts)]))
    got = copies.cpu().numpy()
    assert np.array_equal(got[: want.size], want) and np.all(got[want.size:] == -1)
