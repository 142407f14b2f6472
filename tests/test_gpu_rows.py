"""GPU parity of the rows kernel (gemm_rows.hip) against the CPU oracle:
several activation rows multiplied with weights streamed once, the products
formed from the weight codes.

Dense: 2..8 rows at the GEMV bar (f32 activations as two f16 planes), 9..32
rows at the MFMA GEMM bar, over the sizes where its tiling changes: one
block, ragged last waves, one and several K ranges, weight rows that end
inside a tile, one and two passes of rows, groups of matrices in one launch.
Routed: the f16 expert layer over every bank type it takes.
"""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import GEMM_TOL, GEMV_TOL, build_moe, dev, f16_ulps, host, make_weights, rel, say

pytestmark = pytest.mark.gpu
TYPES = [O.Q4_K, O.Q5_K, O.Q6_K, O.Q8_0, O.Q4_0]


def row_inputs(krk, rows, n_in, seed):
    """Rows of very different magnitude, a zero row, and one value that dwarfs
    the rest of its row."""
    x = krk.synth_normal(rows * n_in, seed=seed).reshape(rows, n_in)
    x[0] *= 1e-3
    x[1] *= 300.0
    if rows > 2:
        x[2] = 0.0
    if rows > 3:
        x[3, n_in // 2] = 1000.0
    return x


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("rows,n_out,n_in", [(6, 1, 256), (8, 77, 512), (7, 517, 2304), (8, 4096, 4096), (6, 130, 4352),
                                             (8, 1000, 14336), (5, 33, 16384)])
def test_rows_exact(krk, torch_cuda, be32, be16, dt, rows, n_out, n_in):
    torch = torch_cuda
    w = make_weights(krk, dt, n_out, n_in, seed=n_out + n_in)
    x = row_inputs(krk, rows, n_in, seed=rows + n_in)
    say("rows", dt, rows, n_out, n_in)
    out = torch.full((rows, n_out), float("nan"), dtype=torch.float32, device="cuda")
    be32.gemm(out, dev(torch, x), dev(torch, w), dt, n_out, n_in, rows)
    be32.sync()
    ref = O.gemm(dt, w, x, n_out, nthreads=16)
    for r in range(rows):
        if r == 2:
            assert not host(out)[r].any()
            continue
        # the oracle's one f32 chain of n_in products is itself off by about
        # 2^-24 sqrt(n_in) relative to the sum of their magnitudes, which one
        # output can cancel away; over a row it stays below the bar
        assert rel(host(out)[r], ref[r]) <= (GEMV_TOL if n_out > 1 else 1e-4), r
    xh = x.astype(np.float16)
    out16 = torch.full((rows, n_out), float("nan"), dtype=torch.float16, device="cuda")
    be16.gemm(out16, dev(torch, xh), dev(torch, w), dt, n_out, n_in, rows)
    be16.sync()
    ref16 = O.gemm(dt, w, xh.astype(np.float32), n_out, nthreads=16)
    for r in range(rows):
        # one f16 rounding of the f32 result (values under f16's normal range,
        # row 0's, round to multiples of 2^-24)
        tol = 2.0 ** -11 + (GEMV_TOL if n_out > 1 else 1e-4)
        floor = np.sqrt(n_out) * 2.0 ** -25
        d = np.linalg.norm(host(out16)[r].astype(np.float32) - ref16[r])
        assert d <= tol * np.linalg.norm(ref16[r]) + floor, r


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("rows,n_out,n_in", [(9, 520, 1024), (16, 4097, 2048), (17, 65, 4096), (32, 777, 2048),
                                             (13, 300, 11008)])
def test_rows_f16_products(krk, torch_cuda, be32, be16, dt, rows, n_out, n_in):
    torch = torch_cuda
    w = make_weights(krk, dt, n_out, n_in, seed=n_out)
    x = krk.synth_normal(rows * n_in, seed=rows).reshape(rows, n_in)
    for be, xs, t in ((be32, x, torch.float32), (be16, x.astype(np.float16), torch.float16)):
        out = torch.full((rows, n_out), float("nan"), dtype=t, device="cuda")
        be.gemm(out, dev(torch, xs), dev(torch, w), dt, n_out, n_in, rows)
        be.sync()
        ref = O.gemm(dt, w, xs.astype(np.float32), n_out, nthreads=16)
        assert rel(host(out).astype(np.float32), ref) <= GEMM_TOL


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("n_in", [4096, 5120])
def test_rows_group(krk, torch_cuda, be32, dt, n_in):
    """Matrices of different heights in one launch (one and two K ranges) equal
    one gemm each, bit for bit; the group reports itself unfused, as before."""
    torch = torch_cuda
    rows, shapes = 8, [100, 2048, 33]
    ws = [dev(torch, make_weights(krk, dt, n, n_in, seed=70 + i)) for i, n in enumerate(shapes)]
    x = dev(torch, krk.synth_normal(rows * n_in, seed=74).reshape(rows, n_in))
    outs = [torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda") for n in shapes]
    assert be32.gemm_group(outs, x, ws, dt, shapes, n_in, rows) == (False, False)
    for o, w, n in zip(outs, ws, shapes):
        one = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
        be32.gemm(one, x, w, dt, n, n_in, rows)
        be32.sync()
        assert rel(host(o), O.gemm(dt, host(w), host(x), n)) <= GEMV_TOL
        assert rel(host(o), host(one)) <= 1e-6      # (the tiling may differ, and with it the order of the sums)


@pytest.mark.parametrize("dt", [O.Q4_K, O.Q8_0])
def test_rows_nonfinite(krk, torch_cuda, be32, dt):
    """A row with an infinity or a NaN comes out non-finite, the others do not
    notice."""
    torch = torch_cuda
    rows, n_out, n_in = 8, 64, 1024
    w = make_weights(krk, dt, n_out, n_in, seed=3)
    x = krk.synth_normal(rows * n_in, seed=4).reshape(rows, n_in)
    ref = O.gemm(dt, w, x, n_out)
    x[1, 700] = np.inf
    x[5, 3] = np.nan
    out = torch.zeros((rows, n_out), dtype=torch.float32, device="cuda")
    be32.gemm(out, dev(torch, x), dev(torch, w), dt, n_out, n_in, rows)
    be32.sync()
    got = host(out)
    assert not np.isfinite(got[[1, 5]]).any()
    for r in (0, 2, 3, 4, 6, 7):
        assert rel(got[r], ref[r]) <= GEMV_TOL


def test_rows_graph_replay(krk, torch_cuda, be32):
    """K ranges summed through the handle's counters, replayed from a graph with
    eager calls between: every replay equals the eager result."""
    torch = torch_cuda
    rows, n_out, n_in = 8, 300, 14336
    w = dev(torch, make_weights(krk, O.Q4_K, n_out, n_in, seed=5))
    x = dev(torch, krk.synth_normal(rows * n_in, seed=6).reshape(rows, n_in))
    want = torch.zeros((rows, n_out), dtype=torch.float32, device="cuda")
    be32.gemm_noalloc(want, x, w, O.Q4_K, n_out, n_in, rows)
    be32.sync()
    out = torch.zeros_like(want)
    g, s, old = torch.cuda.CUDAGraph(), torch.cuda.Stream(), be32.stream
    torch.cuda.synchronize()
    try:
        with torch.cuda.graph(g, stream=s):
            be32.set_stream(torch.cuda.current_stream())
            be32.gemm_noalloc(out, x, w, O.Q4_K, n_out, n_in, rows)
    finally:
        be32.set_stream(old)
    for _ in range(4):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        be32.gemm(out, x, w, O.Q4_K, n_out, n_in, rows)
        be32.sync()
        assert torch.equal(out, want)


@pytest.mark.parametrize("dt", [(O.Q4_K, O.Q4_K, O.Q6_K), O.Q5_K, O.Q8_0, O.Q4_0, (O.Q6_K, O.Q6_K, O.Q4_K)])
@pytest.mark.parametrize("n_tok,n_embd,n_ff", [(1, 256, 512), (9, 4096, 256), (90, 768, 2304)])
def test_rows_moe_f16(krk, torch_cuda, be16, dt, n_tok, n_embd, n_ff):
    """Few and many tokens per expert (up to three passes of sixteen), dropped
    slots, one to sixteen waves on either projection: the f16 rounding points
    of orc_moe_ffn_f16 (most outputs bit-equal; a dot's f32 order moves a
    rounding now and then)."""
    torch = torch_cuda
    ne, k = 6, 3
    mats, table, keep = build_moe(krk, torch, dt, ne, n_embd, n_ff, seed=1900)
    ids, wts = O.router_topk(O.router_softmax(krk.synth_normal(n_tok * ne, seed=177).reshape(n_tok, ne)), k)
    if n_tok > 1:
        ids[0, 1] = -1
        ids[n_tok - 1, k - 1] = -1
    x = krk.synth_normal(n_tok * n_embd, seed=178).reshape(n_tok, n_embd).astype(np.float16)
    say("rows moe f16", dt, n_tok, n_embd, n_ff)
    out = torch.full((n_tok, n_embd), float("nan"), dtype=torch.float16, device="cuda")
    be16.moe_dispatch(table, 0, ne, dev(torch, ids), dev(torch, wts), dev(torch, x), out, n_tok, n_embd, n_ff, k)
    be16.sync()
    ref = O.moe_ffn_f16(x.astype(np.float32), [mats[0, e] for e in range(ne)], [mats[1, e] for e in range(ne)],
                        [mats[2, e] for e in range(ne)], dt, ids, wts, n_ff)
    got = host(out)
    assert rel(got.astype(np.float32), ref.astype(np.float32)) <= 3e-4
    assert (f16_ulps(got, ref) == 0).mean() >= 0.8
    be16.moe_table_forget(table)


@pytest.mark.parametrize("dt", TYPES)
def test_tile_gemm_f32_rows(krk, torch_cuda, be32, dt):
    """The tile GEMM's f32 rows, rounded to f16 before it (krk_gemm) or while
    staged (a fixed scratch that does not hold them): the same f16 operands in
    the same order, so bit-equal, and within the MFMA bar of the oracle."""
    torch = torch_cuda
    rows, n_out, n_in = 2050, 260, 16384     # 2050 x 16384 f16 rows: 64.1 MiB
    assert rows * n_in * 2 > krk.lib().krk_gemm_noalloc_scratch_bytes()
    w = make_weights(krk, dt, n_out, n_in, seed=9)
    x = krk.synth_normal(rows * n_in, seed=10).reshape(rows, n_in)
    xd, wd = dev(torch, x), dev(torch, w)
    a = torch.full((rows, n_out), float("nan"), dtype=torch.float32, device="cuda")
    b = torch.full_like(a, float("nan"))
    be32.gemm(a, xd, wd, dt, n_out, n_in, rows)
    be32.gemm_noalloc(b, xd, wd, dt, n_out, n_in, rows)
    be32.sync()
    assert torch.equal(a, b)
    pick = [0, 1, 255, 256, 1000, 2049]
    assert rel(host(a)[pick], O.gemm(dt, w, x[pick], n_out, nthreads=16)) <= GEMM_TOL


@pytest.mark.parametrize("dt", [O.Q8_0, (O.Q5_K, O.Q5_K, O.Q6_K), O.Q4_0, O.Q4_K])
@pytest.mark.parametrize("n_tok", [1, 5, 40])
def test_rows_moe_f32(krk, torch_cuda, be32, dt, n_tok):
    """f32 rows as two planes, one and several passes of eight rows (40 tokens
    under KRK_PATH_EXACT), dropped slots: the GEMV bar."""
    torch = torch_cuda
    ne, n_embd, n_ff, k = 6, 768, 1024, 3
    mats, table, keep = build_moe(krk, torch, dt, ne, n_embd, n_ff, seed=1950)
    ids, wts = O.router_topk(O.router_softmax(krk.synth_normal(n_tok * ne, seed=187).reshape(n_tok, ne)), k)
    if n_tok > 1:
        ids[0, 1] = -1
    x = krk.synth_normal(n_tok * n_embd, seed=188).reshape(n_tok, n_embd)
    x[n_tok // 2] *= 1e4
    say("rows moe f32", dt, n_tok)
    out = torch.full((n_tok, n_embd), float("nan"), dtype=torch.float32, device="cuda")
    be32.set_gemm_path(krk.PATH_EXACT)
    try:
        be32.moe_dispatch(table, 0, ne, dev(torch, ids), dev(torch, wts), dev(torch, x), out, n_tok, n_embd, n_ff, k)
        be32.sync()
    finally:
        be32.set_gemm_path(krk.PATH_AUTO)
        be32.moe_table_forget(table)
    ref = O.moe_ffn(x, [mats[0, e] for e in range(ne)], [mats[1, e] for e in range(ne)],
                    [mats[2, e] for e in range(ne)], dt, ids, wts, n_ff)
    for t in range(n_tok):
        assert rel(host(out)[t], ref[t]) <= GEMV_TOL, t


@pytest.mark.parametrize("act", ["f32", "f16"])
@pytest.mark.parametrize("n_tok", [1, 3, 700])
def test_moe_plan_reduce_edges(krk, torch_cuda, be32, be16, act, n_tok):
    """The plan over 300 experts (threads past the experts, 700 tokens: ids past
    the ones kept in LDS) and the reduces: each token's row where the output
    starts off a vector boundary is the aligned call's, bit for bit."""
    torch = torch_cuda
    be = be32 if act == "f32" else be16
    td = torch.float32 if act == "f32" else torch.float16
    ne, n_embd, n_ff, k = 300, 256, 256, 6
    mats, table, keep = build_moe(krk, torch, O.Q4_K, ne, n_embd, n_ff, seed=2100)
    ids, wts = O.router_topk(O.router_softmax(krk.synth_normal(n_tok * ne, seed=191).reshape(n_tok, ne)), k)
    x = torch.from_numpy(krk.synth_normal(n_tok * n_embd, seed=192).reshape(n_tok, n_embd)).to("cuda", td)
    d_ids, d_wts = dev(torch, ids), dev(torch, wts)
    outs = []
    say("moe plan", act, n_tok)
    be.set_gemm_path(krk.PATH_EXACT)
    try:
        for off in (0, 1):
            buf = torch.full((n_tok * n_embd + 8,), float("nan"), dtype=td, device="cuda")
            out = buf[off:off + n_tok * n_embd]
            be.moe_dispatch(table, 0, ne, d_ids, d_wts, x, out, n_tok, n_embd, n_ff, k)
            be.sync()
            assert torch.isnan(buf[:off]).all() and torch.isnan(buf[off + n_tok * n_embd:]).all()
            outs.append(host(out).reshape(n_tok, n_embd))
    finally:
        be.set_gemm_path(krk.PATH_AUTO)
        be.moe_table_forget(table)
    assert np.array_equal(outs[0], outs[1])
    sel = sorted({0, n_tok // 2, n_tok - 1})
    ref = O.moe_ffn(host(x).astype(np.float32)[sel], [mats[0, e] for e in range(ne)], [mats[1, e] for e in range(ne)],
                    [mats[2, e] for e in range(ne)], O.Q4_K, ids[sel], wts[sel], n_ff)
    for i, t in enumerate(sel):
        # f16: the slots' running sum is rounded to f16 k times (2^-11 each)
        bar = GEMV_TOL if act == "f32" else GEMV_TOL + (k + 2) * 2.0**-11
        assert rel(outs[0][t], ref[i]) <= bar, t


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("rows,act,n_in", [(33, "f32", 256), (41, "f16", 4096), (128, "f32", 2304)])
def test_mfma_group(krk, torch_cuda, be32, be16, dt, rows, act, n_in):
    """A group of 9..128 rows in one launch, one and several K ranges, matrices
    that end inside a tile and of one row: the MFMA GEMM bar, and one gemm each."""
    torch = torch_cuda
    be, td = (be32, torch.float32) if act == "f32" else (be16, torch.float16)
    shapes = [300, 1, 1025]
    ws = [dev(torch, make_weights(krk, dt, n, n_in, seed=2200 + i)) for i, n in enumerate(shapes)]
    x = torch.from_numpy(krk.synth_normal(rows * n_in, seed=2204).reshape(rows, n_in)).to("cuda", td)
    say("mfma group", dt, rows, act, n_in)
    outs = [torch.full((rows, n), float("nan"), dtype=td, device="cuda") for n in shapes]
    assert be.gemm_group(outs, x, ws, dt, shapes, n_in, rows) == (False, False)
    be.sync()
    first = [host(o).copy() for o in outs]
    for o, w, n in zip(first, ws, shapes):
        assert rel(o, O.gemm(dt, host(w), host(x).astype(np.float32), n)) <= GEMM_TOL
        one = torch.full((rows, n), float("nan"), dtype=td, device="cuda")
        be.gemm(one, x, w, dt, n, n_in, rows)
        be.sync()
        # the same products; K in other ranges, summed in f32
        assert rel(o, host(one)) <= (1e-6 if act == "f32" else 2.0**-10)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("rows,n_out,n_in", [(33, 300, 2816), (160, 300, 2816), (257, 520, 3328), (512, 4096, 11008)])
def test_uneven_k_ranges(krk, torch_cuda, be32, dt, rows, n_out, n_in):
    """K ranges of unequal length (block counts of 11, 13 and 43, prime), on
    the weight-streaming and the tile GEMM, replayed into the same workspace,
    and with the fixed scratch, bit for bit (it does not hold the last shape's
    ranges beside the rounded rows)."""
    torch = torch_cuda
    w = dev(torch, make_weights(krk, dt, n_out, n_in, seed=2300))
    x = dev(torch, krk.synth_normal(rows * n_in, seed=2301).reshape(rows, n_in))
    say("uneven ranges", dt, rows, n_out, n_in)
    outs = []
    for call in (be32.gemm, be32.gemm, be32.gemm_noalloc):
        out = torch.full((rows, n_out), float("nan"), dtype=torch.float32, device="cuda")
        call(out, x, w, dt, n_out, n_in, rows)
        be32.sync()
        outs.append(host(out).copy())
    sel = [0, rows // 2, rows - 1]
    ref = O.gemm(dt, host(w), host(x)[sel], n_out)
    assert rel(outs[0][sel], ref) <= GEMM_TOL
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
