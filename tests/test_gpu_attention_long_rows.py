"""The fused attention and SDDMM tiles on rows past the 512 entries that the
register path holds (attention_long_tile), and the calls without options that
take the fused form.

The mask's 16-row tiles: last rows of 513 to 1,600 entries (one to twelve
chunks a wave, whole and partial chunks) with ragged prefix rows, empty
leading rows, a tile whose columns are not shared, a tile of short rows and a
partial last tile that ends at the arrays' end.  Bars: the derived attention
bounds (tests/_attention_check.py), the bf16 chain's and the SDDMM's own."""
import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from sparsewavecomp_amd import workloads as W
from tests import gpu_util as G
from tests._attention_check import check_attention_f32
from tests.test_gpu_bf16 import (_attention_bf16, _check_attention_bf16,
                                 _sddmm, _sddmm_check)
from tests.test_gpu_bsr_attention import FUSED, _attention_case

pytestmark = pytest.mark.gpu

COLS = 1700


def _mask(seed=0):
    rng = np.random.default_rng(seed)
    rows_cols = []
    for last, kind in ((513, "ragged"), (1600, "ragged"), (1024, "full"),
                       (700, "empty"), (900, "mixed"), (40, "ragged"),
                       (1025, "ragged"), (771, "partial")):
        nt = 7 if kind == "partial" else 16
        base = np.sort(rng.choice(COLS, last, replace=False))
        lens = np.sort(rng.integers(1, last + 1, nt))
        if kind == "full":
            lens[:] = last
        if kind == "empty":
            lens[:5] = 0
        lens[-1] = last
        tile = [base[:n].copy() for n in lens]
        if kind == "mixed":  # one late column differs: not a prefix tile
            other = np.setdiff1d(np.arange(COLS), base)
            tile[14][-1] = other[-1]
            tile[14] = np.sort(tile[14])
        rows_cols += tile
    lengths = np.array([c.size for c in rows_cols])
    ro = np.zeros(lengths.size + 1, np.int32)
    np.cumsum(lengths, out=ro[1:])
    col = np.concatenate(rows_cols).astype(np.int32)
    csr = W.CSR(lengths.size, COLS, ro, col,
                rng.uniform(-1, 1, col.size).astype(np.float32))
    # the host's rule for rows past 512 entries in fp32
    assert csr.nnz > 401 * csr.rows
    return csr


@pytest.mark.parametrize("opts", [FUSED, ""])
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (64, 80), (128, 192)])
def test_long_rows_f32(dev, orc, opts, d, dv):
    csr = _mask(d)
    G.say(f"long rows f32 nnz={csr.nnz} d={d} dv={dv} opts='{opts}'")
    scores, rmax, rsum, out, refs, v, (mv, q, kt, alpha, beta) = \
        _attention_case(orc, csr, d, dv, opts)
    check_attention_f32(orc, csr, mv, q, kt, v, alpha, beta,
                        scores.cpu().numpy(), rmax.cpu().numpy(),
                        rsum.cpu().numpy(), out.cpu().numpy(), refs)


@pytest.mark.parametrize("opts", [FUSED, ""])
@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (128, 192)])
def test_long_rows_bf16(dev, orc, opts, d, dv):
    csr = _mask(dv)
    rng = np.random.default_rng(d)
    q = rng.standard_normal((csr.rows, d)).astype(np.float32)
    kt = rng.standard_normal((d, COLS)).astype(np.float32)
    v = rng.standard_normal((COLS, dv)).astype(np.float32)
    alpha = 1.0 / np.sqrt(d)
    got = _attention_bf16(csr, csr.values, q, kt, v, alpha, 0.5, opts)
    # (the tile without shared columns and the roundings of its row sums)
    _check_attention_bf16(orc, csr, csr.values, q, kt, v, alpha, 0.5, got,
                          exact_frac=0.90)


@pytest.mark.parametrize("kind", ["f32", "bf16"])
@pytest.mark.parametrize("d", [64, 128])
def test_long_rows_sddmm(dev, orc, kind, d):
    csr = _mask(d + 1)
    rng = np.random.default_rng(d)
    lhs = rng.standard_normal((csr.rows, d)).astype(np.float32)
    rhs = rng.standard_normal((d, COLS)).astype(np.float32)
    opts = "sddmm-mapping=row-tile-mfma"
    for combine in (sw.SDDMM_MUL, sw.SDDMM_AFFINE, sw.SDDMM_DOT):
        if kind == "bf16":
            got = _sddmm(csr, csr.values, lhs, rhs, combine, 0.5, 0.25, opts)
            _sddmm_check(orc, csr, csr.values, lhs, rhs, combine, 0.5, 0.25,
                         got)
            continue
        out = torch.full((csr.nnz,), float("nan"), device=G.DEV)
        G.say(f"long rows sddmm d={d} combine={combine}")
        sw.sddmm(G.t(csr.row_offsets), G.t(csr.column_indices),
                 G.t(csr.values), G.t(lhs), G.t(rhs), out, combine, 0.5,
                 0.25, options=opts)
        torch.cuda.synchronize()
        ref = orc.sddmm(csr.row_offsets, csr.column_indices, csr.values, lhs,
                        rhs, combine, 0.5, 0.25)
        dot = orc.sddmm(csr.row_offsets, csr.column_indices, csr.values,
                        np.abs(lhs), np.abs(rhs), orc.SDDMM_DOT)
        bound = (np.abs(csr.values) * dot if combine == sw.SDDMM_MUL else
                 dot if combine == sw.SDDMM_DOT else
                 0.25 * np.abs(csr.values) + 0.5 * dot)
        err = np.abs(out.cpu().numpy() - ref)
        assert np.all(err <= 1e-5 * bound), float((err / bound).max())


def test_long_rows_non_finite_value(dev, orc):
    """A V row of inf reaches exactly the rows that read it."""
    csr = _mask(5)
    d = dv = 64
    rng = np.random.default_rng(7)
    q = rng.standard_normal((csr.rows, d)).astype(np.float32)
    kt = rng.standard_normal((d, COLS)).astype(np.float32)
    v = rng.standard_normal((COLS, dv)).astype(np.float32)
    # the last row of the second tile alone holds its final column
    last = csr.column_indices[csr.row_offsets[32] - 1]
    v[last] = np.inf
    bufs = [torch.empty(n, device=G.DEV) for n in (csr.nnz, csr.rows,
                                                   csr.rows)]
    out = torch.full((csr.rows, dv), float("nan"), device=G.DEV)
    G.say("long rows inf value row")
    sw.sparse_attention(G.t(csr.row_offsets), G.t(csr.column_indices),
                        G.t(csr.values), G.t(q), G.t(kt), G.t(v), *bufs, out,
                        0.125, 0.5, options=FUSED)
    torch.cuda.synchronize()
    reads = np.array([last in csr.column_indices[a:b] for a, b in
                      zip(csr.row_offsets[:-1], csr.row_offsets[1:])])
    assert np.array_equal(~np.isfinite(out.cpu().numpy()).all(1), reads)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_defaults_with_shared_buffers(dev, dt):
    """Without options, a score buffer that is the mask buffer, an output that
    is the query buffer, and an output that is the key buffer (which one
    kernel would overwrite under tiles still reading it) give what separate
    buffers give: such calls keep the six kernels.  (Compared within the chain's rounding: the six
    kernels sum in another order than the fused one.)"""
    mask = W.attention_mask(seq=512, block=64, window=3, random_blocks=1,
                            seed=1)
    g = torch.Generator(device=G.DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(s, generator=g, device=G.DEV).to(dt)
    ro, col = G.t(mask.row_offsets), G.t(mask.column_indices)
    mv, q, kt, v = (rnd(mask.nnz), rnd(512, 64), rnd(64, 512), rnd(512, 64))
    new = lambda *s: torch.full(s, float("nan"), device=G.DEV, dtype=dt)

    def run(mask_values, query, scores, out, keys=kt):
        rmax, rsum = new(512), new(512)
        sw.sparse_attention(ro, col, mask_values, query, keys, v, scores,
                            rmax, rsum, out, 0.125, 1.0)
        torch.cuda.synchronize()
        return [t.double() for t in (scores, rmax, rsum, out)]

    G.say(f"shared buffers {dt}")
    want = run(mv, q, new(mask.nnz), new(512, 64))
    same = mv.clone()
    onto = q.clone()
    # fp32: a few rounding errors of sums of up to 256 terms; bf16: the
    # scores' rounding (2^-9 of scores up to 8) moved by the order
    tol = 2e-5 if dt == torch.float32 else 0.05
    keys = kt.clone()
    for got in (run(same, q, same, new(512, 64)),
                run(mv, onto, new(mask.nnz), onto),
                run(mv, q, new(mask.nnz), keys.view(512, 64), keys)):
        for a, b in zip(got, want):
            assert float((a - b).norm() / b.norm()) <= tol
