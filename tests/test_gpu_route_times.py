"""Calls whose shape decides between kernels, or what a kernel walks, are not
slower than the plain alternative: each test times two public calls on the
same operands (or on operands of the same size) and checks both results.

The bars are wide (the faults they were written for were 1.5 to 1,000 times
over them) and times are the best of several batches, so that neighbours on
the host do not decide."""
import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def us(fn, batches=9):
    """Microseconds per call: the best batch, each a few calls long."""
    for _ in range(2):
        fn()
    torch.cuda.synchronize()
    best = float("inf")
    for _ in range(batches):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(5):
            fn()
        b.record()
        torch.cuda.synchronize()
        best = min(best, a.elapsed_time(b) * 200.0)
    return best


def offsets(lens):
    ro = torch.zeros(lens.numel() + 1, dtype=torch.int64)
    ro[1:] = torch.cumsum(lens, 0)
    return ro.int().to(G.DEV)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [100, 20000])
def test_row_map_over_a_run_of_empty_rows(dev, rows, dt):
    """100,000 empty rows between the entries of one lane's window cost a
    search, not a walk."""
    full = torch.full((5000,), 10, dtype=torch.int64)
    full[-1] = 11  # the run begins inside a 16-byte window
    lens = torch.cat([full, torch.zeros(100000, dtype=torch.int64),
                      torch.full((rows,), 1 + 9 * (rows < 5000))])
    ro, near = offsets(lens), offsets(lens[lens > 0])
    val = torch.randn(int(ro[-1]), device=G.DEV).to(dt)
    rv = torch.randn(lens.numel(), device=G.DEV).to(dt)
    some = rv[lens.to(G.DEV) > 0]
    out, want = torch.empty_like(val), torch.empty_like(val)
    G.say(f"row map, run of empty rows, {rows} after it, {dt}")
    sw.csr_rowwise_map(ro, None, val, rv, out, sw.MAP_SUB)
    sw.csr_rowwise_map(near, None, val, some, want, sw.MAP_SUB)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
    gap = us(lambda: sw.csr_rowwise_map(ro, None, val, rv, out, sw.MAP_SUB))
    plain = us(lambda: sw.csr_rowwise_map(near, None, val, some, want,
                                          sw.MAP_SUB))
    print(f"run {gap:.1f} us, none {plain:.1f} us")
    assert gap <= 6 * plain


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_row_map_of_a_slice_of_rows(dev, dt):
    """2,000 of 2,000,000 rows cost far less than all of them."""
    rows, mean = 2000000, 20
    ro = (torch.arange(rows + 1, device=G.DEV) * mean).int()
    val = torch.randn(rows * mean, device=G.DEV).to(dt)
    rv = torch.randn(rows, device=G.DEV).to(dt)
    out = torch.zeros_like(val)
    a, b = 1000000, 1002000
    G.say(f"row map of a slice {dt}")
    part = us(lambda: sw.csr_rowwise_map(ro[a:b + 1], None, val, rv[a:b],
                                         out, sw.MAP_SUB))
    whole = torch.empty_like(val)
    full = us(lambda: sw.csr_rowwise_map(ro, None, val, rv, whole,
                                         sw.MAP_SUB))
    lo, hi = a * mean, b * mean
    assert torch.equal(out[lo:hi], whole[lo:hi])
    assert not out[:lo].any() and not out[hi:].any()
    print(f"slice {part:.1f} us, all {full:.1f} us")
    assert part <= 0.25 * full


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_sddmm_of_a_slice_of_rows(dev, dt):
    """A slice costs its share of the entries (and the transposition of rhs),
    not those before it too."""
    rows, mean, kdim, cols = 320000, 16, 96, 20000
    g = torch.Generator(device=G.DEV).manual_seed(1)
    ro = (torch.arange(rows + 1, device=G.DEV) * mean).int()
    col = torch.randint(0, cols, (rows * mean,), generator=g,
                        device=G.DEV).int()
    val = torch.randn(rows * mean, generator=g, device=G.DEV).to(dt)
    lhs = torch.randn((rows, kdim), generator=g, device=G.DEV).to(dt)
    rhs = torch.randn((kdim, cols), generator=g, device=G.DEV).to(dt)
    out, whole = torch.zeros_like(val), torch.empty_like(val)
    a, b = 100000, 160000
    # (the arrays end where the rows' mean is still a graph's)
    n = ro[b].item()
    part_ro = ro[a:b + 1]
    some = lhs[a:b].contiguous()
    G.say(f"sddmm of a slice {dt}")
    part = us(lambda: sw.sddmm(part_ro, col[:n], val[:n], some, rhs, out[:n]))
    full = us(lambda: sw.sddmm(ro, col, val, lhs, rhs, whole))
    lo = a * mean
    assert torch.equal(out[lo:n], whole[lo:n])
    assert not out[:lo].any() and not out[n:].any()
    rate = (n - lo) / whole.numel()
    print(f"slice {part:.1f} us, all {full:.1f} us, entries {rate:.3f}")
    assert part <= (rate + 0.2) * full


def _sddmm_without_scratch(ro, col, val, lhs, rhs, out, options):
    o = sw.Options.parse(options) if options else sw.Options()
    fn = getattr(sw.load_library(), "sw_sddmm_csr_" + (
        "f32" if val.dtype == torch.float32 else "bf16"))
    args = [x.data_ptr() for x in (ro, col, val, lhs, rhs, out)] + [
        ro.numel() - 1, rhs.shape[1], col.numel(), lhs.shape[1], sw.SDDMM_MUL,
        1.0, 0.0, o.ref, torch.cuda.current_stream().cuda_stream]

    def run():
        assert fn(*args) == 0
    return run


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,mean,kdim", [(1000000, 1, 4), (500000, 2, 7),
                                            (300000, 3, 8), (2000000, 0, 8)])
def test_sddmm_of_many_short_rows(dev, rows, mean, kdim, dt):
    """Many rows of few products are not given a wave each: half the time of
    that mapping at most, with scratch memory and without.  (mean 0: one
    entry in every tenth row.)"""
    g = torch.Generator(device=G.DEV).manual_seed(1)
    cols = 50000
    ro = torch.arange(rows + 1, device=G.DEV)
    ro = (ro * mean if mean else (ro + 9) // 10).int()
    n = int(ro[-1])
    col = torch.randint(0, cols, (n,), generator=g, device=G.DEV).int()
    val = torch.randn(n, generator=g, device=G.DEV).to(dt)
    lhs = torch.randn((rows, kdim), generator=g, device=G.DEV).to(dt)
    rhs = torch.randn((kdim, cols), generator=g, device=G.DEV).to(dt)
    out, plain, want = (torch.empty_like(val) for _ in range(3))
    G.say(f"sddmm of many short rows {rows} x {mean} kdim={kdim} {dt}")
    wave = us(_sddmm_without_scratch(ro, col, val, lhs, rhs, want,
                                     "sddmm-mapping=wave-per-row"))
    call = us(lambda: sw.sddmm(ro, col, val, lhs, rhs, out))
    alone = us(_sddmm_without_scratch(ro, col, val, lhs, rhs, plain, ""))
    # (sums of up to eight products in another order)
    for got in (out, plain):
        assert float((got.float() - want.float()).norm()) <= (
            2e-6 if dt == torch.float32 else 8e-3) * float(want.float().norm())
    print(f"default {call:.1f} us, without scratch {alone:.1f} us, "
          f"wave {wave:.1f} us")
    assert max(call, alone) <= 0.6 * wave


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("options", ["sddmm-mapping=wave-per-row",
                                     "sddmm-lanes-per-row=64"])
def test_sddmm_wave_per_row_of_long_rows(dev, options, dt):
    """A wave per row that is asked for is one, where rows long enough for the
    16-row tiles share no columns."""
    g = torch.Generator(device=G.DEV).manual_seed(1)
    rows, cols, mean, kdim = 100, 2000, 1000, 64
    ro = (torch.arange(rows + 1, device=G.DEV) * mean).int()
    col = torch.rand((rows, cols), generator=g, device=G.DEV).argsort(
        1)[:, :mean].sort(1).values.int().reshape(-1)
    val = torch.randn(rows * mean, generator=g, device=G.DEV).to(dt)
    lhs = torch.randn((rows, kdim), generator=g, device=G.DEV).to(dt)
    rhs = torch.randn((kdim, cols), generator=g, device=G.DEV).to(dt)
    out, want = torch.empty_like(val), torch.empty_like(val)
    G.say(f"sddmm wave per row {dt} {options}")
    o = sw.Options.parse(options)
    wave = us(lambda: sw.sddmm(ro, col, val, lhs, rhs, out, options=o))
    tiles = us(lambda: sw.sddmm(ro, col, val, lhs, rhs, want))
    # (both sum 64 products in fp32)
    assert float((out.float() - want.float()).norm()) <= (
        2e-6 if dt == torch.float32 else 8e-3) * float(want.float().norm())
    print(f"asked {wave:.1f} us, default {tiles:.1f} us")
    assert wave <= 0.7 * tiles


def _csr(lens, cols, dt, seed=1):
    """Row offsets, random columns and values of rows of these lengths."""
    g = torch.Generator(device=G.DEV).manual_seed(seed)
    ro = offsets(lens)
    n = int(ro[-1])
    col = torch.randint(0, cols, (n,), generator=g, device=G.DEV).int()
    return ro, col, torch.rand(n, generator=g, device=G.DEV).to(dt)


def _spmm_call(lens, k, dt, options=None, cols=100000):
    ro, col, val = _csr(lens, cols, dt)
    g = torch.Generator(device=G.DEV).manual_seed(2)
    rhs = torch.rand((cols, k), generator=g, device=G.DEV).to(dt)
    out = torch.empty((lens.numel(), k), dtype=dt, device=G.DEV)
    o = sw.Options.parse(options) if options else None
    return lambda: sw.spmm(ro, col, val, rhs, out, options=o)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_spmm_of_rows_sorted_by_length(dev, dt):
    """Rows sorted by their lengths are spread over the chip as shuffled ones
    are."""
    g = torch.Generator().manual_seed(3)
    lens = torch.exp(1.5 * torch.randn(200000, generator=g) + 1.9)
    lens = lens.round().clamp(1, 4096).long()
    G.say(f"spmm of sorted rows {dt}")
    mixed = us(_spmm_call(lens, 100, dt))
    up = us(_spmm_call(lens.sort().values, 100, dt))
    down = us(_spmm_call(lens.sort(descending=True).values, 100, dt))
    print(f"ascending {up:.1f} us, descending {down:.1f} us, "
          f"shuffled {mixed:.1f} us")
    assert max(up, down) <= 1.8 * mixed


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [3, 33, 64])
def test_spmm_of_nearly_empty_rows(dev, k, dt):
    """A product of rows of which one in twenty holds an entry takes a few
    times what writing its output does (two launches' floors, and rows of
    k = 33 that share their lines with neighbours)."""
    lens = (torch.arange(1000000) % 20 == 0).long()
    out = torch.empty((1000000, k), device=G.DEV, dtype=dt)
    G.say(f"spmm of nearly empty rows k={k} {dt}")
    fill = us(lambda: out.fill_(1.0))
    call = us(_spmm_call(lens, k, dt))
    print(f"product {call:.1f} us, fill {fill:.1f} us")
    assert call <= 3 * fill + 6


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [16, 64, 100])
def test_spmm_of_short_rows(dev, k, dt):
    """The same entries in rows of 4 take little longer than in rows of 16
    (four times the output)."""
    G.say(f"spmm of short rows k={k} {dt}")
    short = us(_spmm_call(torch.full((1000000,), 4), k, dt))
    long = us(_spmm_call(torch.full((250000,), 16), k, dt))
    print(f"rows of 4 {short:.1f} us, of 16 {long:.1f} us")
    assert short <= 1.9 * long


@pytest.mark.parametrize("k", [4, 64, 200])
def test_spmm_of_few_long_rows(dev, k):
    """20 rows of 20,000 entries fill the chip in bf16 as fp32's row tiles of
    four columns do (bf16's row tiles are the kernel of calls without
    options)."""
    lens = torch.full((20,), 20000)
    tile = "spmm-mapping=wave-per-row-tile"
    G.say(f"spmm of few long rows k={k}")
    want = us(_spmm_call(lens, k, torch.float32, tile))
    call = us(_spmm_call(lens, k, torch.bfloat16, tile))
    plain = us(_spmm_call(lens, k, torch.float32))
    print(f"bf16 {call:.1f} us, fp32 {plain:.1f} us, fp32 tiles {want:.1f}")
    assert max(call, plain) <= 1.8 * want


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,mean,k", [(3, 1500, 1), (3, 1500, 6),
                                         (3, 1500, 130), (40, 200, 33),
                                         (1, 5000, 8), (700, 140, 100)])
def test_spmm_of_few_long_rows_values(dev, orc, rows, mean, k, dt):
    """Every shape that few long rows choose, against the oracle's bound."""
    cols = 3000
    ro, col, val = _csr(torch.full((rows,), mean), cols, dt)
    g = torch.Generator(device=G.DEV).manual_seed(4)
    rhs = torch.randn((cols, k), generator=g, device=G.DEV).to(dt)
    out = torch.full((rows, k), float("nan"), dtype=dt, device=G.DEV)
    G.say(f"spmm of few long rows {rows} x {mean} k={k} {dt}")
    sw.spmm(ro, col, val, rhs, out)
    torch.cuda.synchronize()
    host = [x.cpu().numpy() for x in (ro, col, val.float(), rhs.float())]
    ref, bound = orc.spmm(*host), 1e-5 * orc.spmm_abs_bound(*host)
    if dt == torch.bfloat16:  # one rounding more
        bound = bound + 2.0 ** -8 * np.abs(ref)
    assert np.all(np.abs(out.float().cpu().numpy() - ref) <= bound)


@pytest.mark.parametrize("mean", [0, 4])
def test_spmm_row_tile_of_short_rows_at_odd_widths(dev, mean):
    """Narrow tiles of k = 7 keep one column a lane where rows are short: less
    than the four columns a lane of k = 8 take.  (mean 0: an entry in one row
    of twenty.)"""
    lens = (torch.full((1000000,), mean) if mean else
            (torch.arange(1000000) % 20 == 0).long())
    tile = "spmm-mapping=wave-per-row-tile spmm-lanes-per-row=64"
    G.say(f"spmm row tile of short rows mean={mean}")
    odd = us(_spmm_call(lens, 7, torch.float32, tile))
    even = us(_spmm_call(lens, 8, torch.float32, tile))
    print(f"k = 7 {odd:.1f} us, k = 8 {even:.1f} us")
    assert odd <= 0.85 * even


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,mean", [(100000, 4), (200000, 0), (24000, -8)])
def test_attention_of_many_short_rows(dev, rows, mean, dt):
    """Without options, many rows of a few unshared columns cost what the six
    separate ops cost (mean 0: one entry in every tenth row; -8: rows of
    unequal length, 8 on average, sorted by it, where the separate ops wait
    for the longest rows and one kernel does better)."""
    if mean < 0:
        g = torch.Generator().manual_seed(3)
        lens = torch.exp(0.7 * torch.randn(rows, generator=g) + 1.78)
        lens = lens.round().clamp(1, 4096).long().sort().values
    else:
        lens = (torch.full((rows,), mean) if mean else
                (torch.arange(rows) % 10 == 0).long())
    ro, col, mask = _csr(lens, rows, dt)
    g = torch.Generator(device=G.DEV).manual_seed(4)
    q, v = (torch.randn((rows, 64), generator=g, device=G.DEV).to(dt)
            for _ in range(2))
    kt = torch.randn((64, rows), generator=g, device=G.DEV).to(dt)

    def call(options):
        s, m, r = (torch.empty(n, device=G.DEV, dtype=dt)
                   for n in (col.numel(), rows, rows))
        out = torch.empty((rows, 64), device=G.DEV, dtype=dt)
        o = sw.Options.parse(options) if options else None
        return lambda: sw.sparse_attention(ro, col, mask, q, kt, v, s, m, r,
                                           out, 0.125, 1.0, options=o)

    G.say(f"attention of many short rows {rows} x {mean} {dt}")
    # (any block size that is not the default asks for the separate ops)
    six = us(call("rowwise-map-block-size=128"))
    plain = us(call(None))
    print(f"default {plain:.1f} us, six ops {six:.1f} us")
    assert plain <= (0.75 if mean < 0 else 1.2) * six


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,k,blocks", [(4, 1, 1), (4, 4, 6), (8, 4, 1),
                                        (12, 2, 1), (20, 1, 1), (4, 16, 1)])
def test_bsr_of_few_products(dev, b, k, blocks, dt):
    """Narrow products of small blocks are not slower than one thread per
    output."""
    nbr = 524288 // b
    g = torch.Generator(device=G.DEV).manual_seed(5)
    ro = (torch.arange(nbr + 1, device=G.DEV) * blocks).int()
    col = torch.randint(0, nbr, (nbr * blocks,), generator=g,
                        device=G.DEV).int()
    val = torch.randn((nbr * blocks, b, b), generator=g, device=G.DEV).to(dt)
    rhs = torch.randn((nbr * b, k), generator=g, device=G.DEV).to(dt)
    out, want = (torch.empty((nbr * b, k), device=G.DEV, dtype=dt)
                 for _ in range(2))
    o = sw.Options.parse("bsr-use-mfma=0")
    G.say(f"bsr of few products b={b} k={k} blocks={blocks} {dt}")
    call = us(lambda: sw.bsr_spmm(ro, col, val, rhs, out, b))
    plain = us(lambda: sw.bsr_spmm(ro, col, val, rhs, want, b, options=o))
    # (sums of up to 24 products in another order)
    assert float((out.float() - want.float()).norm()) <= (
        2e-6 if dt == torch.float32 else 8e-3) * float(want.float().norm())
    print(f"default {call:.1f} us, thread per output {plain:.1f} us")
    assert call <= 1.25 * plain


def test_coo_of_one_entry_a_row(dev):
    """Aligned arrays of sorted entries, one a row, are not slower than the
    same off their alignment (one entry a lane)."""
    n = 1000000
    g = torch.Generator(device=G.DEV).manual_seed(6)
    ri = torch.arange(n + 4, device=G.DEV).int()
    col = torch.randint(0, n, (n + 4,), generator=g, device=G.DEV).int()
    val = torch.rand(n + 4, generator=g, device=G.DEV)
    x = torch.rand(n, generator=g, device=G.DEV)
    y = torch.empty(n + 4, device=G.DEV)
    G.say("coo, one entry a row")

    def call(a, z):
        return lambda: sw.coo_spmv(ri[a:z], col[a:z], val[a:z], x, y)

    even = us(call(0, n))
    sums = y.clone()
    odd = us(call(1, n + 1))
    # one product a row either way
    assert torch.equal(sums[1:n], y[1:n])
    assert torch.equal(sums[:n], val[:n] * x[col[:n].long()])
    print(f"aligned {even:.1f} us, off by one {odd:.1f} us")
    assert even <= 1.25 * odd


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,sigma", [(450000, 0.7), (8500, 1.5)])
def test_row_reduction_of_rows_sorted_by_length(dev, rows, sigma, dt):
    """A wave whose rows are all long reads them side by side, and few rows
    are spread over the chip."""
    g = torch.Generator().manual_seed(3)
    lens = torch.exp(sigma * torch.randn(rows, generator=g) + 2.7
                     - (sigma - 0.7))
    lens = lens.round().clamp(1, 4096).long()

    def call(lens):
        ro = offsets(lens)
        val = torch.rand(int(ro[-1]), device=G.DEV).to(dt)
        out = torch.empty(lens.numel(), device=G.DEV, dtype=dt)
        return lambda: sw.csr_row_reduce(ro, None, val, out, "max")

    G.say(f"row reduction of sorted rows {dt}")
    mixed, up = us(call(lens)), us(call(lens.sort().values))
    print(f"sorted {up:.1f} us, shuffled {mixed:.1f} us")
    assert up <= 1.5 * mixed


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_row_map_finds_its_rows(dev, dt):
    """A map over rows of which one in ten holds an entry takes a few more
    trips than the same entries in a few rows, whose search is short."""
    rows = 200000
    lens = (torch.arange(rows) % 10 == 0).long()
    n = int(lens.sum())
    few = torch.full((n // 1000,), 1000)

    def call(lens):
        ro = offsets(lens)
        val = torch.rand(int(ro[-1]), device=G.DEV).to(dt)
        rv = torch.rand(lens.numel(), device=G.DEV).to(dt)
        out = torch.empty_like(val)
        return lambda: sw.csr_rowwise_map(ro, None, val, rv, out, sw.MAP_SUB)

    G.say(f"row map of {rows} rows {dt}")
    many, short = us(call(lens)), us(call(few))
    print(f"many rows {many:.1f} us, few {short:.1f} us")
    assert many <= 2.5 * short


@pytest.mark.parametrize("rows,log_mean,k", [(11000, 2.45, 14), (1000, 1, 60)])
def test_spmm_of_few_sorted_rows(dev, rows, log_mean, k):
    """A few thousand rows of unequal length are spread over the chip, so that
    the longest, side by side, are not one wave's."""
    g = torch.Generator().manual_seed(3)
    lens = torch.exp(1.5 * torch.randn(rows, generator=g) + log_mean)
    lens = lens.round().clamp(1, 4096).long()
    G.say(f"spmm of {rows} sorted rows k={k}")
    mixed = us(_spmm_call(lens, k, torch.bfloat16, cols=20000))
    up = us(_spmm_call(lens.sort().values, k, torch.bfloat16, cols=20000))
    print(f"ascending {up:.1f} us, shuffled {mixed:.1f} us")
    assert up <= 1.6 * mixed
