"""MoE gather and combine above the size from which their rows are streamed
(128 or 256 MiB of grouped rows by their length, 192 MiB of expert rows) and below it, at row lengths and
token counts around the combine's 512- and 1024-thread workgroups; bit-exact against torch on the same
rows (the combine's adds in order, each product rounded before its sum)."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    from fellm_amd import ops as _ops

    return _ops


def _ids(gen, tokens, k, n_experts):
    return torch.argsort(torch.rand(tokens, n_experts, generator=gen, device="cuda"), 1)[:, :k].to(torch.int32).contiguous()


# expert rows: 139 MB, 135 MB, 134.2 MB, 134.2 MB less a row, 4 MB; 204 MB, 202 MB, 201.3 MB (the limit itself),
# 201.3 MB less a row; more than 512 vectors or elements a row for 512 tokens and 513
@pytest.mark.parametrize("tokens,k,hidden", [(1500, 8, 2892), (16500, 8, 256), (8192, 2, 2048), (8191, 2, 2048),
                                             (65, 8, 2048), (2200, 8, 2892), (24600, 8, 256), (12288, 2, 2048),
                                             (12287, 2, 2048), (512, 4, 2052), (513, 4, 2052), (512, 2, 1001),
                                             (513, 2, 1001)])
def test_combine_streamed(ops, tokens, k, hidden):
    gen = torch.Generator(device="cuda").manual_seed(tokens)
    ids = _ids(gen, tokens, k, 32)
    d = ops.moe_dispatch(ids, 32)
    eo = torch.randn(tokens * k, hidden, generator=gen, device="cuda")
    w = torch.rand(tokens, k, generator=gen, device="cuda")
    y0 = torch.randn(tokens, hidden, generator=gen, device="cuda")
    rank = torch.argsort(ids, 1)  # distinct experts: ascending id order of a token's slots
    want_e, want_s = y0.clone(), torch.zeros_like(y0)
    for s in range(k):
        slot = rank[:, s:s + 1]
        rows = d.inv.view(tokens, k).gather(1, slot).view(-1).long()
        want_e += torch.mul(w.gather(1, slot), eo[rows])
        want_s += torch.mul(w[:, s:s + 1], eo[torch.arange(tokens, device="cuda") * k + s])
    assert torch.equal(ops.moe_combine(eo, w, ids=ids, inv=d.inv, y0=y0), want_e)
    assert torch.equal(ops.moe_combine(eo, w), want_s)
    in_place = y0.clone()
    ops.moe_combine(eo, w, ids=ids, inv=d.inv, y0=in_place, out=in_place)
    assert torch.equal(in_place, want_e)


# grouped rows: 135 MB in one and in several segments per thread, 2 MB; 270 MB in one segment, 135 MB and 269 MB in
# rows that end inside a cache line
@pytest.mark.parametrize("tokens,k,hidden", [(16500, 2, 2048), (2000, 8, 4224), (65, 8, 2048), (16500, 4, 2048),
                                             (2000, 8, 4232), (16500, 4, 2040)])
def test_gather_streamed(ops, tokens, k, hidden):
    gen = torch.Generator(device="cuda").manual_seed(hidden)
    ids = _ids(gen, tokens, k, 16)
    ids[0, 0] = 16  # left out: its grouped row at the tail is zero
    d = ops.moe_dispatch(ids, 16)
    x = torch.randn(tokens, hidden, generator=gen, device="cuda").to(torch.bfloat16)
    out = torch.full((tokens * k, hidden), float("nan"), dtype=torch.bfloat16, device="cuda")
    ops.moe_gather(x, d.order, k, inv=d.inv, out=out)
    assert torch.equal(out[:-1], x[(d.order[:-1] // k).long()])
    assert not out[-1].any()
