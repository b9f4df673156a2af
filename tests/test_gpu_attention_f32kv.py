"""Matrix-core attention over contiguous f32 K/V at the edges of its tiles:
head dims below, at and between the compiled ones, slot counts around 16, key
counts around a tile and a workgroup's round of tiles, both output splits (a
quarter of the dims per workgroup, and all of them), non-finite V rows that
only some query rows attend, an output in place of q and one aligned to 4 bytes.

Tolerance as in the other attention tests: 2e-5 of the largest |V| (f32 sums
of at most 1200 products in another order, exp within an ulp) plus an ulp."""
from __future__ import annotations

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _rows(q, k, v, nh, nkv, hd, ql, kvl, causal, window):
    from fellm_amd import _lib

    qd, kd, vd = (torch.from_numpy(a).cuda() for a in (q, k, v))
    out = torch.full_like(qd, float("nan"))
    rc = _lib.lib().fellm_rocm_attention_f32kv_rows(qd.data_ptr(), out.data_ptr(), ql, nh, nkv, hd, kd.data_ptr(),
                                                    vd.data_ptr(), kvl, 0.0, int(causal), window,
                                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    return out.cpu().numpy()


def _inputs(rng, nh, nkv, hd, ql, kvl):
    return (rng.normal(size=nh * ql * hd).astype(np.float32), rng.normal(size=(kvl, nkv * hd)).astype(np.float32),
            rng.normal(size=(kvl, nkv * hd)).astype(np.float32))


@pytest.mark.parametrize("hd", [4, 60, 64, 68, 128, 132, 256])
@pytest.mark.parametrize("nh,nkv,ql,kvl", [(7, 1, 1, 129), (8, 8, 3, 16), (8, 2, 300, 301), (16, 16, 70, 1100),
                                           (8, 1, 600, 640)])
def test_rows_edges(hd, nh, nkv, ql, kvl):
    rng = np.random.default_rng(hd * 7 + ql)
    q, k, v = _inputs(rng, nh, nkv, hd, ql, kvl)
    got = _rows(q, k, v, nh, nkv, hd, ql, kvl, True, 0)
    ref = oracle.fa2_attention(q, k, v, nh, nkv, hd, ql, kvl, float(np.float32(1 / np.sqrt(hd))), True, 0)
    assert np.abs(got - ref).max() <= 2e-5 * np.abs(v).max() + np.abs(ref).max() * 2.0 ** -23


@pytest.mark.parametrize("causal,window", [(True, 0), (True, 5), (False, 9)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_rows_nonfinite_value_stays_with_its_rows(causal, window, bad):
    """Rows that do not attend a key with a non-finite V get the result they
    would have without it; rows that do get a non-finite one."""
    nh, nkv, hd, ql, kvl = 8, 2, 64, 150, 170
    rng = np.random.default_rng(3)
    q, k, v = _inputs(rng, nh, nkv, hd, ql, kvl)
    at = 100
    v2 = v.copy()
    v2[at, 5] = bad  # dim 5 of KV head 0
    clean = _rows(q, k, v, nh, nkv, hd, ql, kvl, causal, window).reshape(nh, ql, hd)
    got = _rows(q, k, v2, nh, nkv, hd, ql, kvl, causal, window).reshape(nh, ql, hd)
    row = np.arange(ql)
    last = kvl - ql + row
    sees = ((at <= last) & ((window == 0) | (at > last - window))) if causal else np.abs(row - at) < window
    hit = np.zeros((nh, ql, hd), bool)
    hit[:nh // nkv, :, 5] = sees[None, :]
    assert np.all(~np.isfinite(got[hit]))
    assert np.abs(got[~hit] - clean[~hit]).max() <= 2e-5 * np.abs(v).max()


@pytest.mark.parametrize("hd", [60, 64, 68, 128, 132, 256])
@pytest.mark.parametrize("ql", [6, 150])
@pytest.mark.parametrize("causal,window", [(True, 0), (False, 9)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_nonfinite_key_of_some_rows_in_every_kernel(hd, ql, causal, window, bad):
    """The key-by-key walk in both output splits and every padding of the head
    dim: bad V dims in each quarter of the output, and a bad K row, all of one
    key that half of the rows attend."""
    nh, nkv, kvl = 8, 2, 170
    rng = np.random.default_rng(hd + ql)
    q, k, v = _inputs(rng, nh, nkv, hd, ql, kvl)
    at = kvl - ql // 2 - 1 if causal else ql // 2 + 8
    dims = [1, hd // 3, hd // 2 + 1, hd - 2]
    k2, v2 = k.copy(), v.copy()
    k2[at, 3] = bad  # KV head 0
    v2[at, [hd + d for d in dims]] = bad  # KV head 1
    clean = _rows(q, k, v, nh, nkv, hd, ql, kvl, causal, window).reshape(nh, ql, hd)
    got = _rows(q, k2, v2, nh, nkv, hd, ql, kvl, causal, window).reshape(nh, ql, hd)
    row = np.arange(ql)
    sees = at <= kvl - ql + row if causal else np.abs(row - at) < window
    assert sees.any() and not sees.all()
    hit = np.zeros((nh, ql, hd), bool)
    hit[np.ix_(np.arange(nh // nkv, nh), sees, dims)] = True
    assert np.all(~np.isfinite(got[hit]))
    hit[:nh // nkv, sees] = True  # a bad score: whatever its row then holds
    assert np.abs(got[~hit] - clean[~hit]).max() <= 2e-5 * np.abs(v).max()


@pytest.mark.parametrize("rows,past", [(16, 1), (33, 47), (80, 1000)])
def test_canvas_edges(rows, past):
    from fellm_amd import _lib

    nh, nkv, hd = 16, 4, 128
    rng = np.random.default_rng(rows + past)
    q = rng.normal(size=(rows, nh * hd)).astype(np.float32)
    k, v = (rng.normal(size=(past, nkv * hd)).astype(np.float32) for _ in range(2))
    ck, cv = (rng.normal(size=(rows, nkv * hd)).astype(np.float32) for _ in range(2))
    d = [torch.from_numpy(a).cuda() for a in (q, k, v, ck, cv)]
    out = torch.full_like(d[0], float("nan"))
    rc = _lib.lib().fellm_rocm_attention_f32kv(d[0].data_ptr(), out.data_ptr(), rows, nh, nkv, hd, d[1].data_ptr(),
                                               d[2].data_ptr(), 0, past, d[3].data_ptr(), d[4].data_ptr(), rows, 0.0,
                                               torch.cuda.current_stream().cuda_stream)
    assert rc == 0, rc
    ref = oracle.attention_f32kv(q, nh, nkv, hd, k, v, 0, past, ck, cv, rows)
    assert np.abs(out.cpu().numpy() - ref).max() <= 2e-5 * max(np.abs(v).max(), np.abs(cv).max()) + \
        np.abs(ref).max() * 2.0 ** -23


@pytest.mark.parametrize("hd", [60, 64, 128, 256])
@pytest.mark.parametrize("rows", [1, 7, 200])
def test_out_in_place_and_at_4_bytes(rows, hd):
    """The same bits whether out stands apart, in place of q or one f32 past a
    16-byte boundary.  In place takes the kernel with all dims in a workgroup,
    whose sums run over other tiles: there the tolerance of this file."""
    from fellm_amd import _lib

    nh, nkv, keys = 8, 2, 500
    rng = np.random.default_rng(rows + hd)
    q, k, v = _inputs(rng, nh, nkv, hd, rows, keys)
    ref = oracle.attention_f32kv(q.reshape(rows, nh * hd), nh, nkv, hd, k, v, 0, keys).reshape(-1)
    kd, vd = torch.from_numpy(k).cuda(), torch.from_numpy(v).cuda()

    def run(qd, out):
        rc = _lib.lib().fellm_rocm_attention_f32kv(qd.data_ptr(), out.data_ptr(), rows, nh, nkv, hd, kd.data_ptr(),
                                                   vd.data_ptr(), 0, keys, None, None, 0, 0.0,
                                                   torch.cuda.current_stream().cuda_stream)
        assert rc == 0, rc
        return out.cpu().numpy()

    qd = torch.from_numpy(q).cuda()
    apart = run(qd, torch.empty_like(qd))
    wide = torch.full((q.size + 2,), 7.0, device="cuda")
    assert np.array_equal(run(qd, wide[1:-1]), apart)
    assert wide[0].item() == 7.0 and wide[-1].item() == 7.0
    for got in (apart, run(qd, qd)):
        assert np.abs(got - ref).max() <= 2e-5 * np.abs(v).max() + np.abs(ref).max() * 2.0 ** -23
