"""GPU parity of the prefill attention over fp32 K / V held as scaled fp16 planes (vgx_attn_prefill_planes,
ops.attn_prefill without a Workspace) and of the bf16 tiles at one and two heads per group, against the
float64 oracle.  Bars: those of test_gpu_attn_prefill.py (1e-5 fp32, 2e-3 bf16, values of order 1), times the
magnitude of V where V is scaled."""
import numpy as np
import pytest
import torch

from oracle import attention as oatt
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
                                       (333, (257, 512), True), (65, (257, 62), False), (700, (), False), (1300, (64,), False)])
@pytest.mark.parametrize("kvdt", [torch.float32, torch.bfloat16])
def test_prefill_tiles_match_oracle(dev, H, G, T, lens, ws, kvdt):
    """Tile edges of 64 and 128 keys, 1 .. 1300 queries (narrow, wide, key ranges with a Workspace), every group size, both query
    types; K and V rows at a stride of their own."""
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
    """Powers of two per 64 keys: V of 2^-40 and zero in the first run (whose keys carry the weight of half of the
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
