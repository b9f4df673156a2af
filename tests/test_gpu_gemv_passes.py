"""K-quant GEMVs of rows longer than 32 blocks, whose blocks are divided over
the wavefronts of a workgroup: block counts around the 32, 64, ... limits and
the largest, row counts around one step of the grid (and of the fold's batches
of four), every format and format pair.  Bit-exact against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from fellm_amd import synth

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

CODE = {"q4k": 12, "q5k": 13, "q6k": 14}


@pytest.fixture(scope="module")
def ops():
    from fellm_amd import ops as _ops

    return _ops


def _bits(t):
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("qt", ["q4k", "q5k", "q6k"])
@pytest.mark.parametrize("rows,nb", [(1, 33), (9, 64), (2050, 33), (300, 65), (4100, 40), (77, 112), (64, 129), (40, 192)])
def test_matvec_passes(ops, qt, rows, nb):
    rng = np.random.default_rng(rows * 200 + nb)
    w = synth.KQUANT_TABLES[CODE[qt]](rng, rows, nb * 256)
    x = rng.normal(size=nb * 256).astype(np.float32)
    wd, xd = torch.from_numpy(w).cuda(), torch.from_numpy(x).cuda()
    ref = oracle.matvec_kquant(CODE[qt], w, rows, nb * 256, x).view(np.uint32)
    assert np.array_equal(_bits(ops.matvec_kquant(wd, xd, qtype=qt)), ref)
    assert np.array_equal(_bits(ops.matvec_kquant_q8k(wd, ops.quantize_q8k(xd), qtype=qt)), ref)


@pytest.mark.parametrize("gq,uq", [("q4k", "q4k"), ("q5k", "q6k"), ("q6k", "q6k"), ("q6k", "q4k")])
@pytest.mark.parametrize("rows,nb", [(3, 33), (1030, 36), (50, 96), (33, 128), (16, 192)])
def test_gate_up_passes(ops, gq, uq, rows, nb):
    rng = np.random.default_rng(rows * 200 + nb)
    g, u = (synth.KQUANT_TABLES[CODE[q]](rng, rows, nb * 256) for q in (gq, uq))
    x = rng.normal(size=nb * 256).astype(np.float32) * 0.01
    gd, ud, xd = (torch.from_numpy(a).cuda() for a in (g, u, x))
    ref = oracle.gate_up_swiglu(CODE[gq], g, CODE[uq], u, rows, nb * 256, x).view(np.uint32)
    assert np.array_equal(_bits(ops.gate_up_swiglu(gd, ud, xd, qtype=gq, up_qtype=uq)), ref)
    assert np.array_equal(_bits(ops.gate_up_swiglu_q8k(gd, ud, ops.quantize_q8k(xd), qtype=gq, up_qtype=uq)), ref)


@pytest.mark.parametrize("qt", ["q4k", "q5k", "q6k"])
@pytest.mark.parametrize("rows,nb", [(256, 64), (257, 40), (1024, 64), (1025, 64), (1536, 33), (2047, 64), (2049, 64),
                                     (1280, 80), (768, 129), (512, 192)])
def test_wavefronts_for_x_and_two_steps(ops, qt, rows, nb):
    """Launches whose workgroups hold wavefronts that only prepare x, on both
    sides of the choice between one step and two, the last rows uneven."""
    test_matvec_passes(ops, qt, rows, nb)


@pytest.mark.parametrize("rows,nb", [(200, 40), (256, 64), (257, 80), (300, 112)])
def test_gate_up_wavefronts_for_x(ops, rows, nb):
    test_gate_up_passes(ops, "q4k", "q6k", rows, nb)
