"""BSR SpMM on the matrix cores for any block size that is a multiple of 4
(bsr_mfma): block sizes below, at and past 16, whose blocks share a 16-wide
step, fill it or take several; odd and partial column strips, aligned and
element-aligned operands; block rows of 0 to 9 blocks, the last block column
among them (a lane whose columns pass k must not read past the end of rhs).

Bars: the fp32 bound 1e-5 sum |a x| against the oracle on the same (bf16-
rounded) inputs; a bf16 output one rounding more."""
import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from sparsewavecomp_amd import workloads as W
from tests import gpu_util as G
from tests._check import assert_within_bound

pytestmark = pytest.mark.gpu


def _bsr(seed, b):
    rng = np.random.default_rng(seed)
    counts = np.array([0, 1, 2, 3, 5, 9, 0, 4, 8, 1, 6, 7])
    nbr = counts.size
    cols = [np.sort(rng.choice(nbr, c, replace=False)) for c in counts]
    cols[-1] = np.sort(np.append(rng.choice(nbr - 1, 6, replace=False),
                                 nbr - 1))
    bro = np.zeros(nbr + 1, np.int32)
    np.cumsum(counts, out=bro[1:])
    bcol = np.concatenate(cols).astype(np.int32)
    vals = rng.standard_normal(bcol.size * b * b).astype(np.float32)
    return W.BSR(nbr * b, nbr * b, b, bro, bcol, vals)


def _at(a, dtype, offset):
    """a on the device, starting `offset` elements off its allocation."""
    x = torch.zeros(a.size + offset, dtype=dtype, device=G.DEV)
    x[offset:] = G.t(a.reshape(-1)).to(dtype)
    return x[offset:].view(a.shape)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("b,k", [(4, 1), (4, 33), (4, 64), (4, 130), (8, 7),
                                 (8, 200), (12, 5),
                                 (12, 61), (16, 64), (16, 65), (16, 30),
                                 (16, 200), (20, 8), (32, 3), (32, 100),
                                 (32, 264), (40, 129), (48, 64), (64, 200),
                                 (64, 9)])
@pytest.mark.parametrize("kind", ["f32", "bf16", "bf16_f32out"])
def test_any_block_size(dev, orc, kind, b, k, offset):
    bsr = _bsr(b + k, b)
    rhs = np.random.default_rng(k).standard_normal((bsr.cols, k)).astype(
        np.float32)
    dt = torch.float32 if kind == "f32" else torch.bfloat16
    odt = torch.bfloat16 if kind == "bf16" else torch.float32
    vals = bsr.block_values
    if dt == torch.bfloat16:
        vals, rhs = G.bf16_round(vals), G.bf16_round(rhs)
    out = _at(np.full((bsr.rows, k), np.nan, np.float32), odt, offset)
    G.say(f"bsr b={b} k={k} {kind} offset={offset}")
    sw.bsr_spmm(G.t(bsr.block_row_offsets), G.t(bsr.block_column_indices),
                _at(vals, dt, offset), _at(rhs, dt, offset), out, b)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = orc.bsr_spmm(bsr.block_row_offsets, bsr.block_column_indices, vals,
                       rhs, b)
    bound = orc.bsr_abs_bound(bsr.block_row_offsets,
                              bsr.block_column_indices, vals, rhs, b)
    if kind == "bf16":  # one rounding to 8 significant bits
        bound = bound * (1 + 2.0 ** -8) + 2.0 ** -8 * np.abs(ref) / 1e-5
    assert_within_bound(got, ref, bound)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,k", [(8, 40), (32, 65)])
def test_non_finite_rows_stay_apart(dev, orc, dt, b, k):
    """An inf in a row of rhs reaches exactly the rows whose blocks read it:
    steps past a block row's end and neighbouring blocks add nothing."""
    bsr = _bsr(b, b)
    vals = np.abs(bsr.block_values) + np.float32(0.5)
    rhs = np.ones((bsr.cols, k), np.float32)
    rhs[5 * b + 1] = np.inf
    out = torch.full((bsr.rows, k), float("nan"), dtype=dt, device=G.DEV)
    G.say(f"bsr inf b={b} k={k} {dt}")
    sw.bsr_spmm(G.t(bsr.block_row_offsets), G.t(bsr.block_column_indices),
                G.t(vals).to(dt), G.t(rhs).to(dt), out, b)
    torch.cuda.synchronize()
    got = out.float().cpu().numpy()
    ref = orc.bsr_spmm(bsr.block_row_offsets, bsr.block_column_indices, vals,
                       rhs, b)
    assert np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.isposinf(ref).any() and np.isfinite(ref).any()
