"""f32 ops in 4-element vectors and bf16 gathers rounded in pairs: lengths
around a vector and a workgroup, buffers aligned to 16 but not 32 bytes and to 4
bytes only, rows of every register layout of RMSNorm and of the fused f32 gather, NaN payloads.  Bit-exact
against the oracle; RMSNorm within 1e-5 (its sum runs in another order)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from fellm_amd import synth

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    from fellm_amd import ops as _ops

    return _ops


def _at(a, skip):
    """a on the device, `skip` elements past a 256-byte boundary."""
    t = torch.empty(a.size + skip, dtype=torch.float32, device="cuda")
    t[skip:] = torch.from_numpy(a.reshape(-1))
    return t[skip:].view(a.shape)


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("skip", [0, 1, 4])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 511, 512, 2049, 4100, 1 << 20])
def test_silu_and_add_f32(ops, n, skip):
    rng = np.random.default_rng(n + skip)
    a, b = (rng.normal(size=n).astype(np.float32) * 4 for _ in range(2))
    a[: n // 7] *= 40
    da, db, out = _at(a, skip), _at(b, skip), _at(np.zeros(n, np.float32), skip)
    assert np.array_equal(_bits(ops.silu_gate(da, db, out=out)), oracle.silu_gate(a, b).view(np.uint32))
    assert np.array_equal(_bits(ops.add(da, db, out=out)), oracle.add(a, b).view(np.uint32))


@pytest.mark.parametrize("skip", [0, 1, 4])
@pytest.mark.parametrize("rows,group", [(1, 4), (3, 252), (2, 4096), (5, 8192), (3, 16384), (1030, 2052), (1024, 2560),
                                        (1025, 4096), (1024, 4100), (1030, 8192), (1024, 16384)])
def test_rmsnorm_f32(ops, rows, group, skip):
    rng = np.random.default_rng(rows + group)
    x, r = (rng.normal(size=(rows, group)).astype(np.float32) for _ in range(2))
    w = rng.normal(1.0, 0.1, size=group).astype(np.float32)
    dx, dr, dw = _at(x, skip), _at(r, skip), _at(w, skip)
    h, y = ops.add_rmsnorm(dx, dr, dw, 1e-5)
    s = (x + r).astype(np.float32)
    assert np.array_equal(_bits(h), s.view(np.uint32))
    for got, v in ((y, s), (ops.rmsnorm(dx, dw, 1e-5), x)):
        d = v.astype(np.float64)
        ref = d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-5) * w
        assert np.abs(got.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("qt,code", [("q4k", 12), ("q5k", 13), ("q6k", 14)])
@pytest.mark.parametrize("n,blocks", [(1, 1), (70, 14), (33, 17)])
def test_kquant_gather_rows(ops, qt, code, n, blocks, kind):
    rng = np.random.default_rng(n * blocks + code)
    table = synth.KQUANT_TABLES[code](rng, 50, blocks * 256)
    ids = rng.integers(0, 50, size=n, dtype=np.uint32)
    ref = oracle.embedding(table, code, 50, blocks * 256, ids)
    dt = {"f32": torch.float32, "bf16": torch.bfloat16}[kind]
    tab, idd = torch.from_numpy(table).cuda(), torch.from_numpy(ids.view(np.int32)).cuda()
    w = torch.ones(blocks * 256, device="cuda")
    got = ops.embedding(tab, idd, dim=blocks * 256, qtype=qt, out_dtype=dt)
    h, y = ops.embedding_rmsnorm(tab, idd, w, 1e-6, dim=blocks * 256, qtype=qt, out_dtype=dt)
    want = oracle.narrow(ref, kind)
    for t in (got, h):
        b = t.cpu().view(torch.int16 if kind == "bf16" else torch.int32).numpy()
        assert np.array_equal(b.view(want.dtype) if kind == "bf16" else b.view(np.float32), want)
    d = ref.astype(np.float64)
    yr = d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-6)
    assert np.abs(y.double().cpu().numpy() - yr).max() <= (1e-5 if kind == "f32" else 2.0 ** -8) * np.abs(yr).max()


@pytest.mark.parametrize("n", [3, 700])
@pytest.mark.parametrize("dim", [1000, 4096, 8192, 8200, 8448, 16384])
def test_dense_f32_gather_and_norm(ops, dim, n):
    """Rows up to the longest that the fused f32 norm takes, few and many."""
    rng = np.random.default_rng(dim + n)
    table = rng.normal(size=(40, dim)).astype(np.float32)
    ids = rng.integers(0, 40, size=n, dtype=np.uint32)
    w = rng.normal(1.0, 0.1, size=dim).astype(np.float32)
    tab, idd, wd = torch.from_numpy(table).cuda(), torch.from_numpy(ids.view(np.int32)).cuda(), torch.from_numpy(w).cuda()
    got = ops.embedding(tab, idd, out_dtype=torch.float32)
    h, y = ops.embedding_rmsnorm(tab, idd, wd, 1e-6, out_dtype=torch.float32)
    assert np.array_equal(_bits(got), table[ids].view(np.uint32)) and np.array_equal(_bits(h), _bits(got))
    d = table.astype(np.float64)
    ref = (d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-6) * w)[ids]
    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("n", [3, 512, 513])
@pytest.mark.parametrize("dim", [4096, 4100, 8196, 16380])
def test_dense_f32_gather_parts(ops, dim, n):
    """Rows of an odd number of 4-element parts beside even ones, on both sides
    of the row count that chooses between parts of 8 and of 4."""
    test_dense_f32_gather_and_norm(ops, dim, n)


def test_bf16_gather_keeps_nan_payloads(ops):
    rng = np.random.default_rng(9)
    table = rng.integers(0, 1 << 16, size=(64, 512), dtype=np.uint32).astype(np.uint16)  # every kind of bf16
    ids = np.arange(64, dtype=np.uint32)
    tab = torch.from_numpy(table.view(np.int16)).cuda().view(torch.bfloat16)
    idd = torch.from_numpy(ids.view(np.int32)).cuda()
    want = oracle.narrow(oracle.widen(table.reshape(-1), "bf16"), "bf16").reshape(table.shape)
    w = torch.ones(512, device="cuda")
    for got in (ops.embedding(tab, idd, out_dtype=torch.bfloat16),
                ops.embedding_rmsnorm(tab, idd, w, 1e-6, out_dtype=torch.bfloat16)[0]):
        assert np.array_equal(got.cpu().view(torch.int16).numpy().view(np.uint16), want)
