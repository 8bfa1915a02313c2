"""GPU parity of the prefill attention over fp32 K / V held as bf16 planes (vgx_attn_prefill_planes,
ops.attn_prefill without a Workspace) and of the bf16 tiles at one and two heads per group, against the
float64 oracle.  Bars: those of test_gpu_attn_prefill.py (1e-5 fp32, 2e-3 bf16, values of order 1), times the
magnitude of V where V is scaled."""
import numpy as np
import pytest
import torch

from oracle import attention as oatt
from vault_amd import _lib as L
from vault_amd import ops

pytestmark = pytest.mark.gpu
TOL, TOL32 = 2e-3, 1e-5


def _t(a, dt=torch.float32):
    return torch.from_numpy(np.asarray(a, dtype=np.float32)).to(dt).cuda()


def _ref(q, runs):
    f = lambda t: t.double().cpu().numpy()  # noqa: E731
    return oatt.chunk(f(q), [(f(k), f(v)) for k, v in runs[:-1]], f(runs[-1][0]), f(runs[-1][1]))


@pytest.mark.parametrize("H,G", [(4, 4), (4, 2), (8, 2), (12, 2), (16, 2)])
@pytest.mark.parametrize("T,lens,ws", [(1, (319,), True), (17, (63, 65, 260), True), (129, (64, 1, 128), False),
                                       (333, (257, 512), True), (65, (257, 62), False), (700, (), False), (1300, (64,), False),
                                       (700, (900,), True)])
@pytest.mark.parametrize("kvdt", [torch.float32, torch.bfloat16])
def test_prefill_tiles_match_oracle(dev, H, G, T, lens, ws, kvdt):
    """Tile edges of 64 and 128 keys, 1 .. 1300 queries (narrow, wide, key ranges with a Workspace over few and many keys),
    every group size, both query types; K and V rows at a stride of their own."""
    rng = np.random.default_rng(H + 7 * T + sum(lens))
    runs = [tuple(_t(rng.standard_normal((G, n, 136)), kvdt)[:, :, :128] for _ in range(2)) for n in lens + (T,)]
    w = ops.Workspace(dev) if ws else None
    for qdt in (torch.float32, torch.bfloat16):
        q = _t(rng.standard_normal((T, H, 128)), qdt)
        out = torch.full((T, H, 128), 7.0, device=dev)
        ops.attn_prefill([{"q": q, "out": out, "runs": runs, "causal_base": 0}], H, G, ws=w)
        assert np.abs(out.double().cpu().numpy() - _ref(q, runs)).max() <= (TOL32 if kvdt == torch.float32 else TOL)


@pytest.mark.parametrize("ws", [False, True])
def test_prefill_planes_scales(dev, ws):
    """Magnitudes far apart between key runs: V of 2^-40 and zero in the first run (whose keys carry the weight of half of the
    queries), 2^20 in the last; queries and keys of reciprocal magnitudes 2^+-30.  Bar: 1e-5 of the largest V that a
    query gives a weight of 2^-24 or more."""
    rng = np.random.default_rng(5)
    H, G, T = 12, 2, 200
    mk = lambda n: rng.standard_normal((G, n, 128))  # noqa: E731
    k0, v0, k1, v1 = mk(128), mk(128) * 2.0 ** -40, mk(T), mk(T) * 2.0 ** 20
    v0[:, 64:] = 0.0
    q = rng.standard_normal((T, H, 128))
    k0[:, :, 0], k1[:, :, 0] = 60.0, -60.0
    q[:, :, 0] = np.where(np.arange(T) % 2 == 0, 12.0, -12.0)[:, None]      # even queries: the first run only
    runs = [(_t(k0 * 2.0 ** -30), _t(v0)), (_t(k1 * 2.0 ** -30), _t(v1))]
    qt = _t(q * 2.0 ** 30)
    out = torch.empty(T, H, 128, device=dev)
    ops.attn_prefill([{"q": qt, "out": out, "runs": runs, "causal_base": 0}], H, G, ws=ops.Workspace(dev) if ws else None)
    err = np.abs(out.double().cpu().numpy() - _ref(qt, runs))
    assert err[0::2].max() <= 1e-5 * 4 * 2.0 ** -40 and err[1::2].max() <= 1e-5 * 4 * 2.0 ** 20


def test_prefill_planes_share_runs(dev):
    """Blocks over prefixes of one run (causal attention by query blocks) and a non-finite V element: its dim is not
    finite (infinity or NaN) for the queries that see its key, and nothing else changes."""
    rng = np.random.default_rng(6)
    H, G, L = 8, 2, 500
    k, v = _t(rng.standard_normal((G, L, 128))), _t(rng.standard_normal((G, L, 128)))
    q, out = _t(rng.standard_normal((L, H, 128))), torch.empty(L, H, 128, device=dev)

    def go():
        ops.attn_prefill([{"q": q[a:b], "out": out[a:b], "runs": [(k[:, :b], v[:, :b])], "causal_base": a}
                          for a, b in ((0, 130), (130, 131), (131, 400), (400, 500))], H, G)
        return out.double().cpu().numpy()
    ref = _ref(q, [(k, v)])
    assert np.abs(go() - ref).max() <= TOL32
    v[0, 450, 3] = float("inf")
    got = go()
    assert not np.isfinite(got[460:, :4, 3]).any() and np.abs(got[:400] - ref[:400]).max() <= TOL32
    assert np.abs(got[400:, :, 4:] - ref[400:, :, 4:]).max() <= TOL32


def _bits(q, runs, H, G, dev):
    """vgx_attn_prefill itself: fp32 K / V split by every workgroup, no planes."""
    out = torch.empty(q.shape, device=dev)
    ra = (L.KVRun * 4)(*[L.KVRun(k.data_ptr(), v.data_ptr(), k.shape[1], k.stride(1), k.stride(0)) for k, v in runs])
    arr = (L.AttnBlock * 1)(L.AttnBlock(q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0),
                                        out.stride(1), q.shape[0], 0, len(runs), ra))
    L.check(L.load().vgx_attn_prefill(L.F32, L.BF16 if q.dtype == torch.bfloat16 else L.F32, L.F32, arr, 1, H, G, 128,
                                      128 ** -0.5, torch.cuda.current_stream().cuda_stream), "vgx_attn_prefill")
    return out


@pytest.mark.parametrize("H,G", [(4, 4), (4, 2), (8, 2), (12, 2), (16, 2)])
@pytest.mark.parametrize("qdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,lens", [(129, (64, 1, 128)), (2300, (65,)), (33, (500,)), (1, (200, 31, 95))])
def test_prefill_planes_keep_the_bits(dev, H, G, qdt, T, lens):
    """Planes or not, the same bits: K and V elements over twelve orders of magnitude, every launch shape."""
    rng = np.random.default_rng(H + T)
    runs = [tuple(_t(rng.standard_normal((G, n, 136)) * 10.0 ** rng.uniform(-6, 6, (G, n, 136)))[:, :, :128]
                  for _ in range(2)) for n in lens + (T,)]
    q, out = _t(rng.standard_normal((T, H, 128)), qdt), torch.empty(T, H, 128, device=dev)
    ops.attn_prefill([{"q": q, "out": out, "runs": runs, "causal_base": 0}], H, G)
    assert torch.equal(out, _bits(q, runs, H, G, dev))


def test_prefill_planes_without_memory(dev, monkeypatch):
    rng = np.random.default_rng(12)
    q, k, v = (_t(rng.standard_normal(s)) for s in ((200, 8, 128), (2, 200, 128), (2, 200, 128)))
    out, empty = torch.empty(200, 8, 128, device=dev), torch.empty

    def full(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return empty(*a, **kw)
    monkeypatch.setattr(torch, "empty", full)
    ops.attn_prefill([{"q": q, "out": out, "runs": [(k, v)], "causal_base": 0}], 8, 2)
    monkeypatch.undo()
    assert torch.equal(out, _bits(q, [(k, v)], 8, 2, dev))


@pytest.mark.parametrize("x", [1e10, 1e30])
@pytest.mark.parametrize("where", ["k", "v"])
def test_prefill_future_keys_change_nothing(dev, x, where):
    """A large element of a later key: queries before it keep their values (their bits, but for those whose wave of 16
    queries reaches it, where the running max may move at another key)."""
    rng = np.random.default_rng(8)
    H, G, T, at = 8, 2, 300, 170
    q, k, v = (_t(rng.standard_normal(s)) for s in ((T, H, 128), (G, T, 128), (G, T, 128)))

    def go():
        out = torch.empty(T, H, 128, device=dev)
        ops.attn_prefill([{"q": q, "out": out, "runs": [(k, v)], "causal_base": 0}], H, G)
        return out
    before = go()
    (k if where == "k" else v)[:, at, 5] = x
    after = go()
    assert torch.equal(before[:at // 16 * 16], after[:at // 16 * 16])
    assert float((before - after)[:at].abs().max()) <= TOL32


def test_prefill_unweighted_key_changes_nothing(dev):
    """A key whose weight is zero, with V of 1e30 beside V of order 1 in the same 32 keys."""
    rng = np.random.default_rng(9)
    H, G, T = 12, 2, 200
    q, k, v = (rng.standard_normal(s) for s in ((T, H, 128), (G, T, 128), (G, T, 128)))
    q[:, :, 0], k[:, :, 0] = 20.0, 0.0
    k[:, 3, 0], v[:, 3] = -1e4, 1e30
    qt, kt, vt = _t(q), _t(k), _t(v)
    out = torch.empty(T, H, 128, device=dev)
    ops.attn_prefill([{"q": qt, "out": out, "runs": [(kt, vt)], "causal_base": 0}], H, G)
    assert np.abs(out.double().cpu().numpy() - _ref(qt, [(kt, vt)]))[4:].max() <= TOL32


def test_prefill_elements_keep_their_own_exponent(dev):
    """Dims of a key, a value and a query of magnitudes far apart: V of 1e10 in one dim beside 1 in the others, and a
    score made of one large query element on a small key element beside a large key element on none.  Bar: 1e-5 of
    each dim's own magnitude."""
    rng = np.random.default_rng(11)
    H, G, T = 8, 2, 200
    q, k, v = (rng.standard_normal(s) for s in ((T, H, 128), (G, T, 128), (G, T, 128)))
    v[:, :, 7] *= 1e10
    q[:, :, 3], k[:, :, 3] = q[:, :, 3] * 1e10, k[:, :, 3] * 1e-10
    q[:, :, 4], k[:, :, 4] = 0.0, k[:, :, 4] * 1e10
    qt, kt, vt = _t(q), _t(k), _t(v)
    out = torch.empty(T, H, 128, device=dev)
    ops.attn_prefill([{"q": qt, "out": out, "runs": [(kt, vt)], "causal_base": 0}], H, G)
    err = np.abs(out.double().cpu().numpy() - _ref(qt, [(kt, vt)]))
    assert err[:, :, 7].max() <= TOL32 * 1e10 and np.delete(err, 7, axis=2).max() <= TOL32


@pytest.mark.parametrize("big", [2.0 ** 20, 2.0 ** 60, 2.0 ** 100])
def test_prefill_zero_values_keep_their_weight(dev, big):
    """Equal scores over 64 keys of zero V and keys of large V: the zeros hold their share of the softmax sum."""
    rng = np.random.default_rng(10)
    H, G, T = 4, 4, 150
    q = torch.zeros(T, H, 128, device=dev)
    runs = [(_t(rng.standard_normal((G, 64, 128))), torch.zeros(G, 64, 128, device=dev)),
            (_t(rng.standard_normal((G, T, 128))), _t(rng.uniform(0.5, 1.0, (G, T, 128)) * big))]
    out = torch.empty(T, H, 128, device=dev)
    ops.attn_prefill([{"q": q, "out": out, "runs": runs, "causal_base": 0}], H, G)
    assert np.abs(out.double().cpu().numpy() - _ref(q, runs)).max() <= TOL32 * big


@pytest.mark.parametrize("kvdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [100, 1024])
def test_prefill_workspace_sizes_one_head_per_group(dev, kvdt, T):
    """One head per group: the workspace of vgx_attn_prefill_workspace_bytes and half of it serve the call, less is
    refused (a launch of 256 workgroups or more runs unsplit)."""
    rng, lib, H = np.random.default_rng(T), L.load(), 8
    runs = [tuple(_t(rng.standard_normal((H, n, 128)), kvdt) for _ in range(2)) for n in (77, T)]
    q, out = _t(rng.standard_normal((T, H, 128))), torch.empty(T, H, 128, device=dev)
    ref = _ref(q, runs)
    ra = (L.KVRun * 4)(*[L.KVRun(k.data_ptr(), v.data_ptr(), k.shape[1], k.stride(1), k.stride(0)) for k, v in runs])
    arr = (L.AttnBlock * 1)(L.AttnBlock(q.data_ptr(), q.stride(0), q.stride(1), out.data_ptr(), out.stride(0),
                                        out.stride(1), T, 0, 2, ra))
    full = int(lib.vgx_attn_prefill_workspace_bytes(H, H))
    for size in (full, full // 2, full // 2 - 1):
        ws = torch.full((size + 4096,), 7, dtype=torch.uint8, device=dev)
        out.fill_(7.0)
        rc = lib.vgx_attn_prefill_ws(L.BF16 if kvdt == torch.bfloat16 else L.F32, L.F32, L.F32, arr, 1, H, H, 128, 128 ** -0.5,
                                     ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
        assert (rc == 0) == (size >= full // 2 or T == 1024) and int((ws[size:] != 7).sum()) == 0
        if rc == 0:
            assert np.abs(out.double().cpu().numpy() - ref).max() <= (TOL32 if kvdt == torch.float32 else TOL)


def test_prefill_planes_in_a_captured_graph(dev):
    """A captured call with planes: replays, with eager calls over other keys between them, give the eager bits."""
    rng = np.random.default_rng(13)
    H, G, T = 12, 2, 300
    sets = [tuple(_t(rng.standard_normal(s)) for s in ((T, H, 128), (G, T, 128), (G, T, 128))) for _ in range(3)]

    def run(q, k, v, out):
        ops.attn_prefill([{"q": q, "out": out, "runs": [(k, v)], "causal_base": 0}], H, G)
        return out
    eager = [run(*s, torch.empty(T, H, 128, device=dev)) for s in sets]
    held, out = tuple(t.clone() for t in sets[0]), torch.zeros(T, H, 128, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(*held, out)
    for i in (0, 1, 2, 0):
        for t, src in zip(held, sets[i]):
            t.copy_(src)
        out.zero_()
        torch.cuda.synchronize()
        graph.replay()
        other = run(*sets[(i + 1) % 3], torch.empty(T, H, 128, device=dev))
        torch.cuda.synchronize()
        assert torch.equal(out, eager[i]) and torch.equal(other, eager[(i + 1) % 3]), f"replay of {i}"
