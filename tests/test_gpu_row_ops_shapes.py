"""CSR row reductions (a group of lanes per row, long rows by the wave) and
row-wise maps (cut by positions, up to 512 rows staged per wave) at the
shapes where their splits change.

Row lengths around 8 entries times the group's lanes and four times that,
for every group size; runs of more than 512 empty and one-entry rows (spans
that are not staged); a row across many waves; arrays ending in the middle of
a 16-byte window and starting off one; in place.  Reductions: the maximum
exact, sums within (n + 1) 2^-24 sum |v| of the float64 sum (any order), one
rounding more in bf16.  Maps: exact for sub and mul, division within 1 ulp,
exp within 2 ulp of float64, before bf16's one rounding."""
import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def _lengths(kind, seed):
    rng = np.random.default_rng(seed)
    if kind == "tiny":  # means of 0 to 2: many rows to a window
        return rng.choice([0, 0, 0, 1, 1, 2], 70001)
    if kind == "few tiny":  # fewer rows than fill the chip: 64 lanes a row
        return rng.choice([0, 0, 0, 1, 1, 2], 1501)
    if kind == "one long":
        a = np.ones(20001, np.int64)
        a[700] = 70001
        return a
    mean = int(kind)  # a group of G lanes: mean about 6 G
    near = [0, 1, mean, 8 * mean // 6, 8 * mean // 6 + 1, 32 * mean // 6,
            32 * mean // 6 + 1, 7 * mean]
    a = np.concatenate([np.full(600, mean), rng.permutation(np.repeat(
        near, 12))])
    # rows enough for 2,048 waves of G lanes a row, fewer take more lanes
    g = 2
    while 8 * g < a.mean():
        g *= 2
    return np.tile(a, -(-2048 * 64 // (g * a.size)))


def _data(kind, dt, offset):
    lens = _lengths(kind, 3)
    ro = np.zeros(lens.size + 1, np.int32)
    np.cumsum(lens, out=ro[1:])
    rng = np.random.default_rng(5)
    v = rng.standard_normal(ro[-1]).astype(np.float32) * 3
    rv = (np.abs(rng.standard_normal(lens.size)) + 0.5).astype(np.float32)
    if dt == torch.bfloat16:
        v, rv = G.bf16_round(v), G.bf16_round(rv)
    val = torch.zeros(v.size + offset, dtype=dt, device=G.DEV)[offset:]
    val.copy_(G.t(v))
    return lens, ro, v.astype(np.float64), rv.astype(np.float64), val, G.t(
        rv).to(dt)


KINDS = ["tiny", "few tiny", "one long", "12", "24", "48", "96", "190", "380", "700"]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("opts", [None, "row-reduction-block-size=100",
                                  "sddmm-lanes-per-row=64"])
@pytest.mark.parametrize("kind", KINDS)
def test_reduce(dev, kind, opts, offset, dt):
    lens, ro, v, _, val, _ = _data(kind, dt, offset)
    G.say(f"row reduce {kind} {dt} offset={offset} opts={opts}")
    out = torch.full((lens.size,), float("nan"), dtype=dt, device=G.DEV)
    sw.csr_row_reduce(G.t(ro), None, val, out, "max", options=opts)
    torch.cuda.synchronize()
    # (reduceat gives an empty row the entry at its offset)
    full = lens > 0
    want = np.full(lens.size, -np.inf)
    want[full] = np.maximum.reduceat(v, ro[:-1][full])
    np.testing.assert_array_equal(out.double().cpu().numpy(), want)
    sw.csr_row_reduce(G.t(ro), None, val, out, "sum", options=opts)
    torch.cuda.synchronize()
    want, mag = np.zeros(lens.size), np.zeros(lens.size)
    want[full] = np.add.reduceat(v, ro[:-1][full])
    mag[full] = np.add.reduceat(np.abs(v), ro[:-1][full])
    tol = (lens + 1) * 2.0 ** -24 * mag
    if dt == torch.bfloat16:
        tol += 2.0 ** -8 * np.abs(want)
    assert np.all(np.abs(out.double().cpu().numpy() - want) <= tol)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("offset,in_place", [(0, False), (0, True),
                                             (3, True)])
@pytest.mark.parametrize("copies", [1, 60])
@pytest.mark.parametrize("kind", KINDS)
def test_map(dev, kind, copies, offset, in_place, dt):
    """copies = 60 repeats the rows past 2,000,000 entries (16 a lane)."""
    lens, ro, v, rv, val, rowv = _data(kind, dt, offset)
    if copies > 1:
        n = v.size
        copies = max(2, 4100000 // n) if n > 40000 else 1
        if copies == 1:
            pytest.skip("too few entries to repeat")
        ro = np.concatenate([[0]] + [ro[1:].astype(np.int64) + i * n
                                     for i in range(copies)]).astype(np.int32)
        v, rv = np.tile(v, copies), np.tile(rv, copies)
        big = torch.zeros(v.size + offset, dtype=dt, device=G.DEV)[offset:]
        big.copy_(val.repeat(copies))
        val, rowv = big, rowv.repeat(copies)
    row = np.repeat(np.arange(ro.size - 1), np.diff(ro))
    r = rv[row]
    src = val.clone()
    for name, want, rel in ((sw.MAP_SUB, v - r, 2.0 ** -24),
                            (sw.MAP_MUL, v * r, 2.0 ** -24),
                            (sw.MAP_DIV, v / r, 2.0 ** -23),
                            (sw.MAP_EXP_SUB, None, 2.0 ** -22)):
        if want is None:  # exp of the fp32 difference
            want = np.exp((v - r).astype(np.float32).astype(np.float64))
        val.copy_(src)
        out = val if in_place else torch.full_like(val, float("nan"))
        G.say(f"row map {kind} x{copies} {dt} offset={offset} "
              f"in_place={in_place} kind={name}")
        sw.csr_rowwise_map(G.t(ro), None, val, rowv, out, name)
        torch.cuda.synchronize()
        tol = rel * np.abs(want) + 2.0 ** -149
        if dt == torch.bfloat16:
            tol = tol + 2.0 ** -8 * np.abs(want)
        assert np.all(np.abs(out.double().cpu().numpy() - want) <= tol)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,mean", [(3001, 5), (200003, 24)])
@pytest.mark.parametrize("first,last", [(0, 1.0), (0.4, 0.4), (0.3, 0.7),
                                        (0.999, 1.0)])
def test_rows_that_are_a_slice(dev, first, last, rows, mean, dt):
    """Row offsets that begin past position 0 or end before the arrays do (a
    slice of a matrix's rows, arrays with room): entries outside the rows
    stay as they are, the others are those of the whole matrix, bit for
    bit."""
    g = torch.Generator(device=G.DEV).manual_seed(rows)
    lens = torch.randint(0, 2 * mean + 1, (rows,), generator=g, device=G.DEV)
    ro = torch.zeros(rows + 1, dtype=torch.int32, device=G.DEV)
    ro[1:] = torch.cumsum(lens, 0)
    nnz = int(ro[-1])
    val = torch.randn(nnz + 1000, generator=g, device=G.DEV).to(dt)
    rowv = (torch.rand(rows, generator=g, device=G.DEV) + 0.5).to(dt)
    whole = torch.empty_like(val[:nnz])
    sw.csr_rowwise_map(ro, None, val[:nnz].clone(), rowv, whole, sw.MAP_SUB)
    a, b = int(first * rows), max(int(last * rows), int(first * rows) + 1)
    lo, hi = int(ro[a]), int(ro[b])
    G.say(f"row map over rows {a}..{b} of {rows} {dt}")
    out = torch.full_like(val, 7.0)
    sw.csr_rowwise_map(ro[a:b + 1], None, val, rowv[a:b], out, sw.MAP_SUB)
    red = torch.empty(b - a, dtype=dt, device=G.DEV)
    sw.csr_row_reduce(ro[a:b + 1], None, val, red, "max")
    torch.cuda.synchronize()
    want = torch.full_like(val, 7.0)
    want[lo:hi] = whole[lo:hi]
    assert torch.equal(out, want)
    rmax = torch.full((rows,), -float("inf"), device=G.DEV).index_reduce(
        0, torch.repeat_interleave(lens), val[:nnz].float(), "amax")
    assert torch.equal(red.float(), rmax[a:b])
