"""SpMM without options (lane groups of every width, spmm_row_group) and the
row tile on any k and alignment: k around each vector width, one and several
column tiles, means on both sides of each rule, empty rows, rows past the
group's own steps (taken by the whole wave), operands off their alignment
and an inf that must reach exactly the rows that read it.  Bars: 1e-5 sum
|a b|, plus one rounding in bf16."""
import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from sparsewavecomp_amd import workloads as W
from tests import gpu_util as G
from tests._check import assert_within_bound

pytestmark = pytest.mark.gpu

TILE = ("spmm-mapping=wave-per-row-tile spmm-tile-size=32 "
        "spmm-lanes-per-row=64 spmm-block-size=64")


def _csr(mean, seed):
    rng = np.random.default_rng(seed)
    lens = rng.poisson(mean, 701)
    lens[rng.random(701) < 0.1] = 0
    lens[[5, 6, 350]] = [1100, 33, 700]
    lens[-2:] = [129, 0]
    return W.csr_from_lengths(rng, lens, 1201)


def _at(a, dt, offset):
    x = torch.zeros(a.size + offset, dtype=dt, device=G.DEV)
    x[offset:] = G.t(a.reshape(-1)).to(dt)
    return x[offset:].view(a.shape)


def _run(csr, val, rhs, dt, opts, offset):
    out = _at(np.full((csr.rows, rhs.shape[1]), np.nan, np.float32), dt,
              offset)
    G.say(f"spmm k={rhs.shape[1]} nnz={csr.nnz} {dt} offset={offset} "
          f"opts='{opts}'")
    sw.spmm(G.t(csr.row_offsets), G.t(csr.column_indices),
            _at(val, dt, offset), _at(rhs, dt, offset), out, options=opts)
    torch.cuda.synchronize()
    return out.float().cpu().numpy()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("opts", [None, "spmm-block-size=100", TILE])
@pytest.mark.parametrize("mean", [6, 40, 60])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 7, 8, 9, 17, 31, 33, 50, 64,
                               65, 100, 129, 260])
def test_widths(dev, orc, k, mean, opts, offset, dt):
    csr = _csr(mean, k)
    rhs = np.random.default_rng(k).uniform(-1, 1, (csr.cols, k)).astype(
        np.float32)
    val = csr.values
    if dt == torch.bfloat16:
        val, rhs = G.bf16_round(val), G.bf16_round(rhs)
    got = _run(csr, val, rhs, dt, opts, offset)
    ref = orc.spmm(csr.row_offsets, csr.column_indices, val, rhs)
    bound = orc.spmm_abs_bound(csr.row_offsets, csr.column_indices, val, rhs)
    if dt == torch.bfloat16:
        bound = bound * (1 + 2.0 ** -8) + 2.0 ** -8 * np.abs(ref) / 1e-5
    assert_within_bound(got, ref, bound)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mean", [0.4, 2, 4, 9, 20, 150])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 6, 7, 8, 9, 17, 33, 63, 100, 129])
def test_entries_at_a_time(dev, orc, k, mean, dt):
    """Mean rows on every side of the rule that sets how many entries a row's
    lanes take at a time, with one row past the group's own steps.  The rows
    fill 2,048 waves, as fewer take more lanes."""
    rng = np.random.default_rng(k)
    v = 8 if k >= 8 and dt == torch.bfloat16 else min(4, 1 << (k.bit_length()
                                                                - 1))
    lanes = 1
    while lanes < min(16, -(-k // v)):
        lanes *= 2
    at_a_time = 1 if mean < 3 else 2 if mean < 12 else 4 if mean < 48 else 16
    lens = rng.poisson(mean, 2048 * 64 // min(64, lanes * at_a_time) + 5)
    lens[450] = max(200, lens[450])
    csr = W.csr_from_lengths(rng, lens, 1201)
    rhs = rng.uniform(-1, 1, (csr.cols, k)).astype(np.float32)
    val = csr.values
    if dt == torch.bfloat16:
        val, rhs = G.bf16_round(val), G.bf16_round(rhs)
    got = _run(csr, val, rhs, dt, None, 0)
    ref = orc.spmm(csr.row_offsets, csr.column_indices, val, rhs)
    bound = orc.spmm_abs_bound(csr.row_offsets, csr.column_indices, val, rhs)
    if dt == torch.bfloat16:
        bound = bound * (1 + 2.0 ** -8) + 2.0 ** -8 * np.abs(ref) / 1e-5
    assert_within_bound(got, ref, bound)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("opts", [None, TILE])
@pytest.mark.parametrize("k", [3, 30, 70])
def test_inf_reaches_its_rows(dev, orc, k, opts, dt):
    csr = _csr(20, 2)
    val = np.abs(csr.values) + np.float32(0.5)
    rhs = np.ones((csr.cols, k), np.float32)
    rhs[csr.column_indices[csr.row_offsets[7] - 1], k - 1] = np.inf
    got = _run(csr, val, rhs, dt, opts, 0)
    ref = orc.spmm(csr.row_offsets, csr.column_indices, val, rhs)
    assert np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.isfinite(got[~np.isposinf(ref)]).all()
