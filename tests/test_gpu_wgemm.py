"""GPU parity of the BF16 / F16 GEMM on the 16-bit matrix cores (vgx_qgemm with a workspace, used by
ops.qlinear from 8 activation rows on) against the fp64 oracle.

Bar: the fp32 accumulation bound at the one-row GEMV's relative term (2e-6).  The pieces hold the whole
significand of every activation under its own exponent."""
import numpy as np
import pytest
import torch

from oracle import codec, linalg
from vault_amd import _lib as L
from vault_amd import ops, vlt3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
@pytest.mark.parametrize("rows,cols,batch,epi", [
    (13, 32, 8, "store"), (2, 64, 65, "swiglu"), (257, 96, 63, "accum"), (1030, 1536, 129, "store"),
    (1536, 8960, 64, "accum"), (640, 2048, 1000, "swiglu"), (256, 256, 9, "edge"), (70, 512, 40, "strided"),
    (2100, 32, 2000, "store"), (2048, 32, 2048, "accum"), (1100, 256, 1030, "accum"), (2100, 480, 1030, "swiglu"),
    (70, 544, 9, "edge"), (1024, 544, 1000, "store")])
def test_wgemm_matches_oracle(dev, dt, rows, cols, batch, epi):
    """Tile edges (256 weight rows, 64 activation rows), one K block, K splits with a short last one, every
    epilogue, both sides of the line to the fp32 MFMA (few columns); "edge": weights and rows of extreme
    magnitudes (fp16 subnormals, rows of 1e-30 .. 1e30) and non-finite activations; "strided": rows at an odd
    float offset and stride."""
    rng = np.random.default_rng(rows + cols + batch)
    mk = lambda seed: vlt3.quantize(dt, np.random.default_rng(seed).standard_normal((rows, cols)).astype(np.float32)
                                    * (1e-5 if epi == "edge" else 0.05))  # noqa: E731
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    if epi == "edge":
        x *= (10.0 ** np.linspace(-30, 30, batch)).astype(np.float32)[:, None]
        x[4, 7], x[5, 9] = np.inf, np.nan
    if epi == "strided":
        buf = torch.zeros(batch * (cols + 3) + 1, device=dev)
        xt = buf[1:].view(batch, cols + 3)[:, :cols]
        xt.copy_(torch.from_numpy(x))
    else:
        xt = torch.from_numpy(x).to(dev)
    if epi == "swiglu":
        g, u = mk(1), mk(2)
        w = ops.QWeight.gateup_from_blocks(dt, rows, cols, g, u, dev)
        h = ops.qlinear_swiglu(w, xt).cpu().numpy().astype(np.float64)
        gf, uf = codec.decode(dt, g, rows, cols), codec.decode(dt, u, rows, cols)
        gg, uu = linalg.gemv(gf, x), linalg.gemv(uf, x)
        ref = linalg.swiglu(gg, uu)
        tol = 1.1 * np.abs(uu) * linalg.gemv_bound(gf, x, dt) + np.abs(gg) * linalg.gemv_bound(uf, x, dt) + \
            1e-6 * np.abs(ref) + 1e-30
        assert np.all(np.abs(h - ref) <= tol), float((np.abs(h - ref) / tol).max())
        return
    raw = mk(3)
    w, wf = ops.QWeight.from_blocks(dt, rows, cols, raw, dev), codec.decode(dt, raw, rows, cols)
    bias = rng.standard_normal(rows).astype(np.float32) if epi != "edge" else None
    y0 = rng.standard_normal((batch, rows)).astype(np.float32)
    y = ops.qlinear(w, xt, bias=torch.from_numpy(bias).to(dev) if bias is not None else None,
                    out=torch.from_numpy(y0).to(dev) if epi == "accum" else None, accumulate=epi == "accum")
    y = y.cpu().numpy().astype(np.float64)
    keep = np.isfinite(x).all(axis=1)
    ref = linalg.gemv(wf, x[keep], bias) + (y0[keep] if epi == "accum" else 0.0)
    tol = linalg.gemv_bound(wf, x[keep], dt) + np.abs(ref) * 2e-7
    err = np.abs(y[keep] - ref)
    assert np.all(err <= tol), float((err / tol).max())
    if epi == "edge":
        nz = wf[:, 7] != 0
        assert np.all(np.isinf(y[4][nz])) and np.all(np.isnan(y[4][~nz])) and np.all(np.isnan(y[5]))


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
def test_wgemm_leaves_the_tile_counters(dev, dt):
    """One zero-filled workspace for a 16-bit GEMM and then a Q4_0 decode batch whose workgroups take tickets from
    its counters (the down projection of a batch of 16)."""
    lib, rng = L.load(), np.random.default_rng(3)
    B, d, ff = 16, 1536, 8960
    raw = vlt3.synthetic_blocks(codec.Q4_0, d, ff, rng)
    w4, wf = ops.QWeight.from_blocks(codec.Q4_0, d, ff, raw, dev), codec.decode(codec.Q4_0, raw, d, ff)
    wb = ops.QWeight.from_blocks(dt, d, ff, vlt3.quantize(dt, np.ones((d, ff), np.float32)), dev)
    x = rng.standard_normal((B, ff)).astype(np.float32)
    xt, y = torch.from_numpy(x).to(dev), torch.full((B, d), 7.0, device=dev)
    ws = torch.zeros(int(lib.vgx_qgemm_workspace_bytes(B, d, ff, L.EPI_STORE)), dtype=torch.uint8, device=dev)
    for w in (wb, w4):
        L.check(lib.vgx_qgemm(w.dtype, w.packed.data_ptr(), d, ff, xt.data_ptr(), ff, B, None, 0.0, None, y.data_ptr(), d,
                              L.EPI_STORE, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream), "vgx_qgemm")
    assert int(ws[:65536].max()) == 0
    err = np.abs(y.cpu().numpy() - linalg.gemv(wf, x))
    assert np.all(err <= linalg.gemv_bound(wf, x, codec.Q4_0))


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
@pytest.mark.parametrize("rows,cols,batch", [(70, 96, 9), (258, 1536, 70), (33000, 480, 9)])
@pytest.mark.parametrize("swiglu", [False, True])
def test_wgemm_infinities(dev, dt, rows, cols, batch, swiglu):
    """Infinite and NaN weights and activations (the fp32 MFMA, several K ranges, one): against activations of few
    bits, whose lower pieces are zero, against zeros, each other and ordinary elements.  An output is infinite or NaN
    where the float64 product is, and within the usual bound elsewhere."""
    rng = np.random.default_rng(rows)
    td = torch.bfloat16 if dt == codec.BF16 else torch.float16

    def mk():
        w = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float32)
        w[3, 7], w[4, 7], w[5, 9], w[6, 7], w[6, 8], w[rows - 1, cols - 1] = np.inf, -np.inf, np.nan, np.inf, -np.inf, np.inf
        w[7:9, 7], w[9, 11] = 0.5, 0.0
        return torch.from_numpy(w).to(td)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[1, 7], x[2, 7], x[3, 7], x[4, 11], x[5, 3], x[6, 8] = 1.0, np.inf, 0.0, -np.inf, np.nan, -np.inf
    x[batch - 1, cols - 1] = -2.0
    blocks = lambda t: t.view(torch.uint8).reshape(-1)  # noqa: E731
    ws = [mk() for _ in range(2 if swiglu else 1)]
    xd = torch.from_numpy(x).to(dev)
    if swiglu:
        y = ops.qlinear_swiglu(ops.QWeight.gateup_from_blocks(dt, rows, cols, blocks(ws[0]), blocks(ws[1]), dev), xd)
    else:
        y = ops.qlinear(ops.QWeight.from_blocks(dt, rows, cols, blocks(ws[0]), dev), xd)
    y = y.double().cpu().numpy()
    wf = [w.double().numpy() for w in ws]
    with np.errstate(invalid="ignore", over="ignore"):
        ref = [np.stack([(w * xb.astype(np.float64)).sum(1) for xb in x]) for w in wf]
        out = linalg.swiglu(*ref) if swiglu else ref[0]
    inf, fin = np.isinf(out), np.isfinite(out)
    assert np.array_equal(np.isnan(y), np.isnan(out)) and np.array_equal(y[inf], out[inf])
    bound = [linalg.gemv_bound(np.nan_to_num(w, nan=0.0, posinf=0.0, neginf=0.0).astype(np.float32),
                               np.nan_to_num(x, nan=0.0, posinf=0.0, neginf=0.0), dt) for w in wf]
    with np.errstate(invalid="ignore"):
        tol = 1.1 * np.abs(ref[1]) * bound[0] + np.abs(ref[0]) * bound[1] + 1e-6 * np.abs(out) if swiglu else bound[0]
    assert np.all(np.abs(y[fin] - out[fin]) <= tol[fin] + 1e-30)


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
@pytest.mark.parametrize("big", [1e4, 1e10, 1e30])
def test_wgemm_elements_keep_their_own_exponent(dev, dt, big):
    """A large activation that meets zero weights costs the rest of its row nothing (the bound counts only what the
    weights multiply), whether it stands in one row or in all."""
    rng = np.random.default_rng(1)
    rows, cols, batch = 70, 544, 40
    w = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float32)
    w[:, 5] = 0.0
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[::2, 5] = big
    raw = vlt3.quantize(dt, w)
    wf = codec.decode(dt, raw, rows, cols)
    y = ops.qlinear(ops.QWeight.from_blocks(dt, rows, cols, raw, dev), torch.from_numpy(x).to(dev)).cpu().numpy()
    assert np.all(np.abs(y - linalg.gemv(wf, x)) <= linalg.gemv_bound(wf, x, dt))


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
@pytest.mark.parametrize("how", ["none", "short", "weights at 8 bytes"])
@pytest.mark.parametrize("epi", [L.EPI_STORE, L.EPI_ACCUM, L.EPI_SWIGLU])
def test_qgemm_16bit_weights_without_the_planes(dev, dt, how, epi):
    """vgx_qgemm of 16-bit weights where the DMA tiles cannot run (no workspace, one without room for the partials,
    weights that are not 16-byte aligned) runs on the fp32 MFMA: odd row counts, more rows and activations than a tile."""
    lib, rng = L.load(), np.random.default_rng(4)
    rows, cols, batch = (106 if epi == L.EPI_SWIGLU else 205), 1056, 70
    mk = lambda: vlt3.quantize(dt, (rng.standard_normal((rows, cols)) * 0.05).astype(np.float32))  # noqa: E731
    raws = [mk() for _ in range(2 if epi == L.EPI_SWIGLU else 1)]
    w = ops.QWeight.gateup_from_blocks(dt, rows, cols, *raws, dev) if epi == L.EPI_SWIGLU else \
        ops.QWeight.from_blocks(dt, rows, cols, raws[0], dev)
    shift = torch.empty(w.packed.numel() + 8, dtype=torch.uint8, device=dev)
    shift[8:] = w.packed
    x, y0 = (rng.standard_normal((batch, n)).astype(np.float32) for n in (cols, rows))
    xt, y = torch.from_numpy(x).to(dev), torch.from_numpy(y0).to(dev)
    need = int(lib.vgx_qgemm_workspace_bytes(batch, rows, cols, epi))
    ws = torch.zeros(need, dtype=torch.uint8, device=dev)
    size = {"none": 0, "short": 65536 + 3 * batch * cols * 2, "weights at 8 bytes": need}[how]
    L.check(lib.vgx_qgemm(dt, shift.data_ptr() + 8 if size == need else w.packed.data_ptr(), rows, cols, xt.data_ptr(), cols,
                          batch, None, 0.0, None, y.data_ptr(), rows, epi, ws.data_ptr() if size else None, size,
                          torch.cuda.current_stream().cuda_stream), "vgx_qgemm")
    assert int(ws.max()) == 0                                   # untouched
    wf = [codec.decode(dt, r, rows, cols) for r in raws]
    ref, bound = [linalg.gemv(f, x) for f in wf], [linalg.gemv_bound(f, x, dt) for f in wf]
    if epi == L.EPI_SWIGLU:
        out = linalg.swiglu(*ref)
        tol = 1.1 * np.abs(ref[1]) * bound[0] + np.abs(ref[0]) * bound[1] + 1e-6 * np.abs(out) + 1e-30
    else:
        out = ref[0] + (y0 if epi == L.EPI_ACCUM else 0.0)
        tol = bound[0] + np.abs(out) * 2e-7
    assert np.all(np.abs(y.double().cpu().numpy() - out) <= tol)


@pytest.mark.parametrize("dt", [codec.BF16, codec.F16])
@pytest.mark.parametrize("rows,cols,batch", [(1536, 8960, 16), (70, 800, 600)])
def test_wgemm_in_a_captured_graph(dev, dt, rows, cols, batch):
    """A captured call (down projection of a decode batch with K splits; one K range or few): its scratch belongs to the
    graph, so replays with eager calls of other activations between them give the eager bits."""
    rng = np.random.default_rng(rows)
    w = ops.QWeight.from_blocks(dt, rows, cols, vlt3.quantize(dt, (rng.standard_normal((rows, cols)) * 0.05)
                                                              .astype(np.float32)), dev)
    xs = [torch.from_numpy(rng.standard_normal((batch, cols)).astype(np.float32)).to(dev) for _ in range(3)]
    eager = [ops.qlinear(w, x) for x in xs]
    x, out = xs[0].clone(), torch.zeros(batch, rows, device=dev)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.qlinear(w, x, out=out)
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.qlinear(w, x, out=out)
    for i in (0, 1, 2, 0):
        x.copy_(xs[i])
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        other = ops.qlinear(w, xs[(i + 1) % 3])
        torch.cuda.synchronize()
        assert torch.equal(out, eager[i]) and torch.equal(other, eager[(i + 1) % 3]), f"replay of {i}"
