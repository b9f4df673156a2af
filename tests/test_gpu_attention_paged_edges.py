"""Paged decode attention at the edges of its work split: lengths around a
block, a pair of blocks, a round of the four wavefronts' pairs and a split;
rows that finish in one split beside rows that need several; walks long enough
to reload the block-table lanes; windows across splits; non-finite stale bytes
past a row's length and absent blocks; infinite values in attended keys; the
choice between one and four wavefronts.

Tolerance as in test_gpu_attention.py: 2e-5 of the row's largest |V| plus an
ulp of the output."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from test_gpu_attention import check, make_case, run_gpu

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ops():
    from fellm_amd import ops as _ops

    return _ops


def _ref(q, nh, nkv, hd, lengths, arena, table, n_logical, bb, kind, window=0):
    return oracle.paged_attention(q, nh, nkv, hd, np.array(lengths), float(np.float32(1 / np.sqrt(hd))), arena, table,
                                  n_logical, 1, 0, 16, bb, kind=kind, window=window)


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 64), (14, 2, 128), (4, 1, 256)])
@pytest.mark.parametrize("lengths", [[31, 32, 33, 127, 128, 129, 144, 0], [513, 1, 640, 527, 528], [4100, 40]])
def test_lengths_around_the_split(ops, dev, lengths, nh, nkv, hd, kind):
    rng = np.random.default_rng(sum(lengths) + hd)
    q, arena, table, n_logical, bb, v16 = make_case(rng, lengths, nh, nkv, hd, kind)
    got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, table, n_logical, bb, lengths, nh, nkv, hd, kind)
    check(got, _ref(q, nh, nkv, hd, lengths, arena, table, n_logical, bb, kind), v16, "f32", f"{lengths}")


@pytest.mark.parametrize("window", [17, 600, 2048])
def test_window_across_splits_and_table_reload(ops, dev, window):
    """5000 keys with and without split-key scratch: one workgroup then walks
    40 pairs per wavefront, past the 32 its table lanes hold."""
    rng = np.random.default_rng(window)
    nh, nkv, hd, lengths = 8, 2, 64, [5000, 700]
    q, arena, table, n_logical, bb, v16 = make_case(rng, lengths, nh, nkv, hd, "f16")
    for win in (window, 0):
        ref = _ref(q, nh, nkv, hd, lengths, arena, table, n_logical, bb, "f16", window=win)
        for workspace in ("auto", None):
            got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, table, n_logical, bb, lengths, nh, nkv, hd, "f16",
                             window=win, workspace=workspace)
            check(got, ref, v16, "f32", f"window {win} workspace {workspace}")


@pytest.mark.parametrize("kind,bad", [("f16", 0x7E01), ("f16", 0x7C00), ("bf16", 0x7FC1), ("bf16", 0xFF80)])
@pytest.mark.parametrize("length", [1, 20, 37, 600])
def test_stale_bytes_and_absent_blocks(ops, dev, kind, bad, length):
    """NaN or inf in every slot past the row's length changes nothing; a block
    whose table entry is out of range contributes nothing."""
    rng = np.random.default_rng(length)
    nh, nkv, hd, stride = 8, 2, 128, 256
    q, arena, table, n_logical, bb, v16 = make_case(rng, [length], nh, nkv, hd, kind)
    ref = _ref(q, nh, nkv, hd, [length], arena, table, n_logical, bb, kind)
    stale = arena.copy().view(np.uint16).reshape(-1, bb // 2)
    live = np.zeros_like(stale, bool)
    for t in range(length):
        for v in (0, 1):
            at = (v * 16 + t % 16) * stride
            live[table[t // 16], at:at + stride] = True
    stale[~live] = bad
    got, _ = run_gpu(ops, dev, q, "f32", "f32", stale.reshape(-1).view(np.uint8), table, n_logical, bb, [length], nh, nkv,
                     hd, kind)
    check(got, ref, v16, "f32", "stale")
    if length > 32:  # drop the second block: the same as attending the others
        gone = table.copy()
        gone[1] = 10 ** 6
        got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, gone, n_logical, bb, [length], nh, nkv, hd, kind)
        keep = [t for t in range(length) if t // 16 != 1]
        k16 = arena.view(np.uint16).reshape(-1, bb // 2)

        def rows(v):
            bits = np.stack([k16[table[t // 16], (v * 16 + t % 16) * stride:(v * 16 + t % 16 + 1) * stride] for t in keep])
            return oracle.widen(np.ascontiguousarray(bits), kind).reshape(len(keep), stride)

        ref = oracle.attention_f32kv(q, nh, nkv, hd, rows(0), rows(1), 0, len(keep))
        check(got, ref, v16, "f32", "absent block")


@pytest.mark.parametrize("workspace", ["auto", None])
@pytest.mark.parametrize("kind,inf", [("f16", 0x7C00), ("bf16", 0x7F80)])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 64), (32, 2, 128), (4, 1, 256)])
def test_infinite_value_of_an_attended_key(ops, dev, nh, nkv, hd, kind, inf, workspace):
    """+inf and -inf in V reach the dims they stand in with their sign, both in
    one dim make NaN, and every other dim is what it is without them."""
    rng = np.random.default_rng(hd + nkv)
    lengths, stride = [1, 20, 600, 1300], nkv * hd
    q, arena, table, n_logical, bb, v16 = make_case(rng, lengths, nh, nkv, hd, kind)
    a16 = arena.view(np.uint16).reshape(-1, bb // 2)
    table2 = table.reshape(len(lengths), n_logical)
    for r, n in enumerate(lengths):
        def put(t, dim, bits):
            a16[table2[r, t // 16], (16 + t % 16) * stride + dim] = bits

        put(0, 3, inf)
        put(n - 1, hd - 1, inf | 0x8000)
        put(n // 2, stride - 2, inf)  # the last KV head
        if n > 1:
            put(0, hd // 2, inf)
            put(n - 1, hd // 2, inf | 0x8000)
    got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, table, n_logical, bb, lengths, nh, nkv, hd, kind,
                     workspace=workspace)
    ref = _ref(q, nh, nkv, hd, lengths, arena, table, n_logical, bb, kind)
    off = ~np.isfinite(ref)
    assert np.isinf(ref).any() and np.isnan(ref).any()
    assert np.array_equal(np.where(off, got, 0.0), np.where(off, ref, 0.0), equal_nan=True)
    check(np.where(off, 0.0, got), np.where(off, 0.0, ref), v16, "f32", "finite dims")


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("hd", [64, 128, 256])
def test_small_probabilities_keep_their_bits(ops, dev, hd, kind):
    """Two keys a row: one of score 0 and V = 0, one of score -x with every V.
    The output is then p v / (1 + p) with p = exp(-x) down to 2^-29, and shows
    the bits that p is held to.

    Tolerance, relative: exp takes x log2(e) rounded, an error of |x| 2^-23 in
    p, and four more roundings of 2^-23 at most (exp itself, the sum, the
    reciprocal, the products)."""
    rng = np.random.default_rng(hd)
    x = np.arange(0, 20.5, 0.25, dtype=np.float32)  # exact in both types
    rows = x.size
    k = np.zeros((rows, 2, hd), np.float32)
    k[:, 1, 0] = -x
    v = np.zeros((rows, 2, hd), np.float32)
    v[:, 1] = rng.normal(size=(rows, hd))
    from test_oracle_attention import build_cache

    arena, table, n_logical, bb, _, v16 = build_cache(rng, list(k), list(v), kind=kind)
    q = np.zeros((rows, hd), np.float32)
    q[:, 0] = 1.0
    got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, table, n_logical, bb, [2] * rows, 1, 1, hd, kind, scale=1.0)
    p = np.exp(-x.astype(np.float64))[:, None]
    ref = p / (1.0 + p) * np.stack([r[1] for r in v16])
    err = np.abs(got - ref) / np.maximum(np.abs(ref), 1e-30)
    assert np.all(err <= ((x + 4) * 2.0 ** -23)[:, None]), (err.max(1) / ((x + 4) * 2.0 ** -23)).max()


@pytest.mark.parametrize("kind", ["f16", "bf16"])
@pytest.mark.parametrize("rows,nh,nkv,hd,top", [
    (3, 8, 2, 64, 32), (3, 4, 1, 256, 33),  # one pair of blocks or more
    (8, 64, 64, 64, 64), (8, 64, 64, 64, 65), (8, 128, 64, 128, 128), (8, 64, 64, 128, 129),  # 512 (row, KV head) pairs
    (16, 128, 64, 64, 256), (16, 64, 64, 64, 257), (16, 64, 64, 128, 300), (7, 64, 64, 256, 40), (8, 64, 64, 256, 200)])
def test_one_or_four_wavefronts(ops, dev, rows, nh, nkv, hd, top, kind):
    """Both sides of each line of the choice, with rows of 0 to `top` keys and an
    infinite V in the longest."""
    rng = np.random.default_rng(top + hd)
    lengths = [top, 0, 1] + [int(n) for n in rng.integers(1, top + 1, size=rows - 3)]
    q, arena, table, n_logical, bb, v16 = make_case(rng, lengths, nh, nkv, hd, kind)
    a16 = arena.view(np.uint16).reshape(-1, bb // 2)
    a16[table[0], 16 * nkv * hd + 5] = 0xFF80 if kind == "bf16" else 0xFC00  # key 0 of row 0, dim 5: -inf
    got, _ = run_gpu(ops, dev, q, "f32", "f32", arena, table, n_logical, bb, lengths, nh, nkv, hd, kind)
    ref = _ref(q, nh, nkv, hd, lengths, arena, table, n_logical, bb, kind)
    off = ~np.isfinite(ref)
    assert off.any() and np.array_equal(got[off], ref[off])
    check(np.where(off, 0.0, got), np.where(off, 0.0, ref), v16, "f32", f"top {top}")
