"""The fp32 and mixed-cache prefill's split products (prefill_f32.hip) where
they can go wrong: operands of very different magnitudes, magnitudes and
infinities past the split's limit (2^60; those tiles run on the fp32 matrix
cores), and the tile and chunk edges of its KV split.  Reference: float64
attention over the cache's own rows, within the fp32 bar's 5e-6 of the row's
RMS (24-bit operands, fp32 accumulation)."""
import numpy as np
import pytest
import torch

from qx_amd import abi
from qx_amd import runtime as rt
from tests.helpers import TOL_F32, attend64, log, rel_err

pytestmark = pytest.mark.gpu

TORCH = {abi.F32: torch.float32, abi.F16: torch.float16, abi.BF16: torch.bfloat16}
SCALE = 0.015625


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def prefill(ctx, k, v, q, kdt, vdt, start):
    """k, v: [start + T][8][64] fp32; q: [T][16][64]; returns out and the cache's rows."""
    cap = k.shape[0]
    arena = rt.KvArena(ctx, abi.SHAPE_GRANITE, 1, 1, cap, kdt, vdt)
    with rt.Graph(ctx) as g:
        rt.store_kv(g, arena, 0, 0, k[None].cuda(), v[None].cuda())
        out = rt.prefill_attention(g, arena, 0, start, q.cuda())
        kk, vv = arena.gather(g, 0, 0, 0, cap)
    return out.cpu().numpy(), kk.float().cpu().numpy(), vv.float().cpu().numpy()


def check(out, q, kk, vv, start, rows):
    worst = 0.0
    for t in rows:
        n = start + t + 1
        e = rel_err(out[t], attend64(q[t].numpy(), kk[:n], vv[:n], SCALE))
        assert e <= TOL_F32 / 2, (t, e)
        worst = max(worst, e)
    return worst


PLANS = [(abi.F32, abi.F16), (abi.F32, abi.F32), (abi.F32, abi.BF16), (abi.F16, abi.F32), (abi.BF16, abi.F32)]


@pytest.mark.parametrize("kdt,vdt", PLANS)
@pytest.mark.parametrize("start,T", [(0, 64), (0, 65), (63, 66), (1, 255), (700, 128), (300, 640)])
def test_edges_of_tiles_and_chunks(ctx, kdt, vdt, start, T):
    g = torch.Generator().manual_seed(start + T)
    k, v = (torch.randn((start + T, 8, 64), generator=g) for _ in range(2))
    q = 6 * torch.randn((T, 16, 64), generator=g)
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, start)
    e = check(out, q, kk, vv, start, sorted({0, 1, T // 2, max(0, T - 65), T - 1}))
    log(f"split prefill {kdt}/{vdt} {start}+{T}: vs float64 {e:.2e}")


@pytest.mark.parametrize("kdt,vdt", [(abi.F32, abi.F16), (abi.F32, abi.F32), (abi.BF16, abi.F32)])
@pytest.mark.parametrize("power", [-40, 30, 59, 64])
def test_operands_of_far_magnitudes(ctx, kdt, vdt, power):
    """One dim of every key times 2^power and of every query times 2^-power:
    the same scores, with pieces far apart; 64 is past the split's limit."""
    T = 200
    g = torch.Generator().manual_seed(power + 100)
    k, v = (torch.randn((T, 8, 64), generator=g) for _ in range(2))
    q = 6 * torch.randn((T, 16, 64), generator=g)
    k[:, :, 5] *= 2.0 ** power
    q[:, :, 5] *= 2.0 ** -power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    e = check(out, q, kk, vv, 0, [0, 63, 64, 150, 199])
    log(f"split prefill 2^{power} {kdt}/{vdt}: vs float64 {e:.2e}")


@pytest.mark.parametrize("vdt", [abi.F16, abi.F32, abi.BF16])
def test_infinities_stay_infinities(ctx, vdt):
    """An infinite value makes the rows that weigh it infinite in its dim, not
    NaN, and a key whose score is -inf drops out; the first tile's rows before
    either, and the other kv heads, are untouched."""
    T = 200
    g = torch.Generator().manual_seed(9)
    k, v = (torch.randn((T, 8, 64), generator=g) for _ in range(2))
    q = torch.randn((T, 16, 64), generator=g)
    q[:, :, 7] = 1.0 + q[:, :, 7].abs()
    v[70, 3, 11] = float("inf")
    k[90, 2, 7] = float("-inf")
    out, kk, vv = prefill(ctx, k, v, q, abi.F32, vdt, 0)
    assert np.all(np.isposinf(out[128:, 6:8, 11]))  # rows whose tiles hold no masked copy of it
    finite = np.delete(out[128:, 6:8], 11, axis=2)
    assert np.all(np.isfinite(finite)) and np.all(np.isfinite(out[:, :6])) and np.all(np.isfinite(out[:, 8:]))
    kk[90, 2] = 0.0  # attend64 without the dropped key
    for t in (128, 199):
        ref = np.zeros((16, 64))
        for h in range(16):
            keys = kk[:t + 1, h // 2].astype(np.float64)
            s = keys @ q[t, h].numpy().astype(np.float64) * SCALE
            if h // 2 == 2:
                s[90] = -np.inf
            w = np.exp(s - s.max())
            vals = vv[:t + 1, h // 2].astype(np.float64)
            vals = np.where(np.isfinite(vals), vals, 0.0)
            ref[h] = (w / w.sum()) @ vals
        got = np.where(np.isfinite(out[t]), out[t], 0.0)
        ref[6:8, 11] = 0.0
        assert rel_err(got, ref) <= TOL_F32 / 2
