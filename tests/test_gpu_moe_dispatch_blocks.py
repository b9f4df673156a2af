"""MoE dispatch around the choice of its workgroup (1024 threads where blocks x
experts reach 3072, up to 1024 experts) and around the chunks and rounds of its
four or sixteen wavefronts; exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("tokens,k,n_experts", [(512, 1, 128), (513, 1, 128), (129, 4, 1024), (129, 4, 1025), (2048, 1, 3),
                                                (2049, 1, 1024), (4099, 3, 7), (5000, 8, 1024), (9000, 8, 1025)])
def test_dispatch_blocks(tokens, k, n_experts):
    from fellm_amd import ops

    rng = np.random.default_rng(tokens + n_experts)
    ids = rng.integers(0, n_experts, size=(tokens, k)).astype(np.uint32)
    d = ops.moe_dispatch(torch.from_numpy(ids.view(np.int32)).cuda(), n_experts)
    for got, want in zip(d, oracle.moe_dispatch(ids, n_experts)):
        assert np.array_equal(got.cpu().numpy().view(np.uint32), want)


@pytest.mark.parametrize("tokens,k,n_experts", [(4096, 1, 1024), (4097, 1, 1024), (6145, 1, 1025), (47104, 1, 128),
                                                (47105, 1, 128), (6000, 8, 127), (24700, 8, 16)])
def test_dispatch_workgroup_choice(tokens, k, n_experts):
    test_dispatch_blocks(tokens, k, n_experts)
