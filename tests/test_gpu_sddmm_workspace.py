"""SDDMM over a transposed rhs (calls with scratch memory) and the routes of
the mappings beside it.

kdim around the vector widths and lane-group sizes (odd, below one step,
steps of 2 to 16 lanes, more than one step), ragged rows with empty ones and
one of thousands of entries, more than 64 rows to a wave, in place, aligned
and element-aligned operands, with and without samples.  Bar: the SDDMM's
1e-5 (|sample| sum |lhs rhs|), plus one rounding in bf16."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import sparsewavecomp_amd as sw
from sparsewavecomp_amd import workloads as W
from tests import gpu_util as G

pytestmark = pytest.mark.gpu


def _csr(rows, cols, seed):
    rng = np.random.default_rng(seed)
    lens = rng.poisson(6, rows)
    lens[rng.random(rows) < 0.3] = 0
    lens[100:200] = 0
    lens[rows // 2] = min(cols, 2500)
    lens[-3:] = 0
    return W.csr_from_lengths(rng, lens, cols)


def _run(csr, kdim, dt, kind, offset=0, in_place=False, workspace=True,
         opts=None, stream=0):
    """The C entry point with the scratch memory it asks for, or none."""
    rng = np.random.default_rng(kdim)
    lhs = rng.standard_normal((csr.rows, kdim)).astype(np.float32)
    rhs = rng.standard_normal((kdim, csr.cols)).astype(np.float32)
    val = csr.values

    def dev(a):
        x = torch.zeros(a.size + offset, dtype=dt, device=G.DEV)
        x[offset:] = G.t(a.reshape(-1)).to(dt)
        return x[offset:]

    lib = sw.load_library()
    vals, l_, r_ = dev(val), dev(lhs), dev(rhs)
    out = vals if in_place else torch.full_like(vals, float("nan"))
    ro, col = G.t(csr.row_offsets), G.t(csr.column_indices)
    o = sw.Options.parse(opts) if opts else sw.Options()
    elem = vals.element_size()
    need = lib.sw_sddmm_workspace_bytes(csr.rows, csr.cols, csr.nnz, kdim,
                                        elem, o.ref)
    ws = torch.full((max(need, 16),), 255, dtype=torch.uint8, device=G.DEV)
    fn = (lib.sw_sddmm_csr_f32_ws if dt == torch.float32
          else lib.sw_sddmm_csr_bf16_ws)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    G.say(f"sddmm_ws rows={csr.rows} nnz={csr.nnz} kdim={kdim} {dt} "
          f"kind={kind} offset={offset} in_place={in_place} need={need}")
    rc = fn(ptr(ro), ptr(col), ptr(vals), ptr(l_), ptr(r_), ptr(out),
            csr.rows, csr.cols, csr.nnz, kdim, kind, 0.75, 0.5, o.ref,
            ptr(ws) if workspace else None, need if workspace else 0, None)
    torch.cuda.synchronize()
    assert rc == 0, lib.sw_last_error()
    if dt == torch.bfloat16:
        val, lhs, rhs = (G.bf16_round(a) for a in (val, lhs, rhs))
    return out.float().cpu().numpy(), need, (val, lhs, rhs)


def _check(orc, csr, got, kind, dt, operands):
    val, lhs, rhs = operands
    ref = orc.sddmm(csr.row_offsets, csr.column_indices, val, lhs, rhs, kind,
                    0.75, 0.5).astype(np.float64)
    dot = orc.sddmm(csr.row_offsets, csr.column_indices, val, np.abs(lhs),
                    np.abs(rhs), orc.SDDMM_DOT).astype(np.float64)
    bound = {sw.SDDMM_MUL: np.abs(val) * dot, sw.SDDMM_DOT: dot,
             sw.SDDMM_AFFINE: 0.5 * np.abs(val) + 0.75 * dot}[kind]
    tol = 1e-5 * bound
    if dt == torch.bfloat16:
        tol = tol * (1 + 2.0 ** -8) + 2.0 ** -8 * np.abs(ref)
    assert np.all(np.abs(got - ref) <= tol)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kdim,rows", [(2, 1200000), (5, 500000), (8, 300000),
                                       (16, 150000), (31, 80000),
                                       (33, 80000), (64, 40000),
                                       (100, 25000), (130, 20000),
                                       (256, 9000), (300, 9000)])
def test_transposed(dev, orc, kdim, rows, dt):
    csr = _csr(rows, 3001, kdim)
    got, need, ops = _run(csr, kdim, dt, sw.SDDMM_MUL)
    assert need > 0
    _check(orc, csr, got, sw.SDDMM_MUL, dt, ops)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", [sw.SDDMM_MUL, sw.SDDMM_AFFINE,
                                  sw.SDDMM_DOT])
@pytest.mark.parametrize("offset,in_place", [(0, True), (1, False),
                                             (3, True)])
def test_kinds_and_alignment(dev, orc, kind, offset, in_place, dt):
    csr = _csr(40001, 2999, 9)
    got, need, ops = _run(csr, 62, dt, kind, offset, in_place)
    assert need > 0
    _check(orc, csr, got, kind, dt, ops)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("opts", [None, "sddmm-block-size=64",
                                  "sddmm-block-size=512",
                                  "sddmm-block-size=1024",
                                  "sddmm-mapping=wave-per-row",
                                  "sddmm-mapping=row-tile-mfma"])
@pytest.mark.parametrize("kdim", [64, 96])
@pytest.mark.parametrize("rows", [700, 40000])
def test_without_workspace(dev, orc, rows, kdim, opts, dt):
    """No scratch memory: small calls one wave per row, larger ones by their
    mapping (one row per work-item in workgroups of the block size)."""
    csr = _csr(rows, 3001, 4)
    got, _, ops = _run(csr, kdim, dt, sw.SDDMM_AFFINE, workspace=False,
                       opts=opts)
    _check(orc, csr, got, sw.SDDMM_AFFINE, dt, ops)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kdim", [64, 128, 96])
@pytest.mark.parametrize("in_place", [False, True])
def test_block_mask_without_options(dev, orc, kdim, in_place, dt):
    """Rows of more than 96 entries in the mean: the 16-row tiles at kdim 64
    and 128, one wave per row otherwise and in place; 1,003 rows leave a
    partial last tile whose last row's length is no multiple of 4."""
    mask = W.attention_mask(seq=1024, block=64, window=3, random_blocks=1,
                            seed=2)
    n = int(mask.row_offsets[1003])
    csr = W.CSR(1003, 1024, mask.row_offsets[:1004].copy(),
                mask.column_indices[:n].copy(),
                np.random.default_rng(1).uniform(-1, 1, n).astype(np.float32))
    got, need, ops = _run(csr, kdim, dt, sw.SDDMM_AFFINE, in_place=in_place)
    assert need == 0 and csr.nnz > 96 * csr.rows
    _check(orc, csr, got, sw.SDDMM_AFFINE, dt, ops)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("a,b", [(0, 40001), (9000, 40001), (9001, 31003)])
def test_rows_that_are_a_slice(dev, a, b, dt):
    """Row offsets that begin past position 0 or end before the arrays do:
    entries outside the rows stay as they are, the others are those of the
    whole matrix, bit for bit."""
    csr = _csr(40001, 2999, 9)
    g = torch.Generator(device=G.DEV).manual_seed(2)
    lhs = torch.randn((csr.rows, 62), generator=g, device=G.DEV).to(dt)
    rhs = torch.randn((62, csr.cols), generator=g, device=G.DEV).to(dt)
    ro = G.t(csr.row_offsets)
    # room past the rows (with columns of the matrix)
    col = torch.cat([G.t(csr.column_indices), torch.zeros(
        1001, dtype=torch.int32, device=G.DEV)])
    val = torch.randn(col.numel(), generator=g, device=G.DEV).to(dt)
    n = csr.nnz
    lib, o = sw.load_library(), sw.Options()
    assert lib.sw_sddmm_workspace_bytes(b - a, csr.cols, col.numel(), 62,
                                        val.element_size(), o.ref) > 0
    G.say(f"sddmm over rows {a}..{b} {dt}")
    whole = sw.sddmm(ro, col[:n], val[:n], lhs, rhs, torch.empty_like(val[:n]))
    out = torch.full_like(val, 7.0)
    sw.sddmm(ro[a:b + 1], col, val, lhs[a:b].contiguous(), rhs, out)
    torch.cuda.synchronize()
    lo, hi = int(ro[a]), int(ro[b])
    want = torch.full_like(val, 7.0)
    want[lo:hi] = whole[lo:hi]
    assert torch.equal(out, want)


def test_python_call_on_another_stream_and_captured(dev, orc):
    """sw.sddmm on a side stream takes its scratch memory there; a captured
    call takes none.  Both equal the plain call's values."""
    csr = _csr(40000, 3001, 12)
    g = torch.Generator(device=G.DEV).manual_seed(1)
    lhs = torch.randn((csr.rows, 64), generator=g, device=G.DEV)
    rhs = torch.randn((64, csr.cols), generator=g, device=G.DEV)
    ro, col, val = G.t(csr.row_offsets), G.t(csr.column_indices), G.t(
        csr.values)
    G.say("sddmm plain, side stream, captured")
    want = sw.sddmm(ro, col, val, lhs, rhs, torch.empty_like(val))
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    outs = [torch.empty_like(val) for _ in range(4)]
    for o in outs:
        sw.sddmm(ro, col, val, lhs, rhs, o, stream=side)
        junk = torch.full((1 << 22,), 7.0, device=G.DEV)  # other stream
    torch.cuda.synchronize()
    for o in outs:
        assert torch.equal(o, want)
    captured = torch.empty_like(val)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        sw.sddmm(ro, col, val, lhs, rhs, captured)
    for _ in range(3):
        captured.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        err = (captured - want).abs()
        # two orders of a 64-term dot product
        scale = val.abs() * 64 * lhs.abs().max() * rhs.abs().max()
        assert bool((err <= 1e-5 * scale).all())


@pytest.mark.parametrize("rows,asks", [(1000, False), (40000, True)])
def test_small_calls_do_not_ask_for_scratch(dev, monkeypatch, rows, asks):
    """The question costs a call of its own; its answer for small calls is
    0."""
    csr = _csr(rows, 3001, 5)
    ro, col, val = G.t(csr.row_offsets), G.t(csr.column_indices), G.t(
        csr.values)
    lhs = torch.zeros((csr.rows, 62), device=G.DEV)
    rhs = torch.zeros((62, csr.cols), device=G.DEV)
    lib = sw.load_library()
    asked = []

    class Counting:
        def __getattr__(self, name):
            if name == "sw_sddmm_workspace_bytes":
                asked.append(name)
            return getattr(lib, name)

    need = lib.sw_sddmm_workspace_bytes(csr.rows, csr.cols, csr.nnz, 62, 4,
                                        None)
    assert (need > 0) == asks
    monkeypatch.setattr(sw, "load_library", lambda: Counting())
    G.say(f"sddmm asks for scratch, rows={rows}")
    sw.sddmm(ro, col, val, lhs, rhs, torch.empty_like(val))
    torch.cuda.synchronize()
    assert bool(asked) == asks


def test_scratch_while_another_thread_captures(dev):
    """A call on one thread's stream takes its scratch memory also when the
    allocator has to ask the driver for it while another thread captures a
    graph, and leaves that capture alone."""
    csr = _csr(40000, 3001, 7)
    g = torch.Generator(device=G.DEV).manual_seed(1)
    lhs = torch.randn((csr.rows, 64), generator=g, device=G.DEV)
    rhs = torch.randn((64, csr.cols), generator=g, device=G.DEV)
    ro, col, val = G.t(csr.row_offsets), G.t(csr.column_indices), G.t(
        csr.values)
    want = sw.sddmm(ro, col, val, lhs, rhs, torch.empty_like(val))
    out = torch.empty_like(val)
    a, b = torch.ones(1000, device=G.DEV), torch.empty(1000, device=G.DEV)
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()  # the next scratch memory is a new allocation
    failed = []

    def other():
        try:
            with torch.cuda.stream(side):
                sw.sddmm(ro, col, val, lhs, rhs, out)
        except Exception as e:  # noqa: BLE001 (reported below)
            failed.append(e)

    G.say("sddmm while another thread captures")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        torch.mul(a, 3.0, out=b)
        thread = threading.Thread(target=other)
        thread.start()
        thread.join(30)
    assert not thread.is_alive() and not failed, failed
    b.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(b, torch.full_like(b, 3.0))
    assert torch.equal(out, want)
