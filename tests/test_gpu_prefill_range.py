"""The range of the fp32 and mixed-cache prefill (prefill_f32.hip): scores of any
size, infinities and NaN in later rows of the call, a large value under a small
weight, values next to either end of binary32, and the bits of each product.
Reference: float64 attention over the cache's own rows, within the fp32 bar's
5e-6 of the row's RMS unless a test derives its own."""
import numpy as np
import pytest
import torch

from qx_amd import abi
from qx_amd import runtime as rt
from tests.helpers import TOL_F32, attend64, log, rel_err

pytestmark = pytest.mark.gpu

SCALE = 0.015625
PLANS = [(abi.F32, abi.F16), (abi.F32, abi.F32), (abi.F32, abi.BF16), (abi.F16, abi.F32), (abi.BF16, abi.F32),
         (abi.F32, abi.I8_TIERED)]
WIDE_KEYS = [(k, v) for k, v in PLANS if k != abi.F16]  # keys past binary16's range


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def prefill(ctx, k, v, q, kdt, vdt, start):
    """k, v: [start + T][8][64] fp32; q: [T][16][64]; returns out and the cache's rows."""
    cap = k.shape[0]
    window = 64 if vdt == abi.I8_TIERED else 0
    arena = rt.KvArena(ctx, abi.SHAPE_GRANITE, 1, 1, cap, kdt, vdt, value_window=window)
    with rt.Graph(ctx) as g:
        rt.store_kv(g, arena, 0, 0, k[None].cuda(), v[None].cuda())
        out = rt.prefill_attention(g, arena, 0, start, q.cuda())
        kk, vv = arena.gather(g, 0, 0, 0, cap)
    return out.cpu().numpy(), kk.float().cpu().numpy(), vv.float().cpu().numpy()


def inputs(n, T, seed):
    g = torch.Generator().manual_seed(seed)
    k, v = (torch.randn((n, 8, 64), generator=g) for _ in range(2))
    return k, v, torch.randn((T, 16, 64), generator=g)


def check(out, q, kk, vv, start, rows, tol=TOL_F32 / 2):
    worst = 0.0
    for t in rows:
        n = start + t + 1
        e = rel_err(out[t], attend64(q[t].numpy(), kk[:n], vv[:n], SCALE))
        assert e <= tol, (t, e)
        worst = max(worst, e)
    return worst


# ---- large scores -----------------------------------------------------------------

@pytest.mark.parametrize("kdt,vdt", PLANS)
@pytest.mark.parametrize("size", [1e4, 3e4])
def test_large_scores(ctx, kdt, vdt, size):
    """Scores up to 2^29 in the exponent's units, too far apart for a second
    position to count: the largest of a row weighs exactly one, and the row is
    that position's values."""
    start, T = 70, 100
    k, v, q = inputs(start + T, T, int(size))
    k, q = (size * k).clamp(-65504, 65504), size * q
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, start)
    check(out, q, kk, vv, start, [0, 1, 57, 58, T - 1])


@pytest.mark.parametrize("kdt,vdt", WIDE_KEYS)
@pytest.mark.parametrize("power", [40, 59, 60, 64, 90])
def test_large_keys_under_ordinary_queries(ctx, kdt, vdt, power):
    """One dim decides every score, alike in no two positions (nor in bf16)."""
    T = 150
    k, v, q = inputs(T, T, power)
    k[:, :, 5] = torch.sign(k[:, :, 5]) * (1 + torch.arange(T)[:, None]) * 2.0 ** power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    check(out, q, kk, vv, 0, [0, 63, 64, 100, T - 1])


@pytest.mark.parametrize("kdt,vdt", PLANS)
@pytest.mark.parametrize("power", [59, 64, 90])
def test_large_queries_over_ordinary_keys(ctx, kdt, vdt, power):
    T = 150
    k, v, q = inputs(T, T, power + 1)
    q[::3, :, 5] *= 2.0 ** power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    check(out, q, kk, vv, 0, [0, 1, 63, 64, 99, T - 1])


@pytest.mark.parametrize("kdt,vdt", PLANS)
def test_a_query_past_the_limit_with_keys_as_small(ctx, kdt, vdt):
    """Queries of 2^64 over keys of 2^-64 (2^-14 in binary16, where the query's
    is 2^14): ordinary scores on the path of large magnitudes."""
    T, power = 150, 14 if kdt == abi.F16 else 64
    k, v, q = inputs(T, T, 64)
    k[:, :, 5] *= 2.0 ** -power
    q[:, :, 5] *= 2.0 ** power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    check(out, q, kk, vv, 0, [0, 63, 64, 100, T - 1])


# ---- infinities and NaN in later rows of the call ---------------------------------------

@pytest.mark.parametrize("kdt,vdt,bad", [(k, v, b) for k, v in PLANS if v != abi.I8_TIERED
                                         for b in (float("inf"), float("-inf"), float("nan"))] +
                         [(abi.F32, abi.F16, 1e5)])
@pytest.mark.parametrize("start,T,late", [(2400, 16, 15), (1600, 24, 7), (750, 48, 31), (0, 130, 70), (1400, 16, 12)])
def test_a_later_rows_value_stays_out_of_earlier_rows(ctx, kdt, vdt, bad, start, T, late):
    """A value that is no number, or that overflows the cache's binary16, in one
    row of the call: the rows before it do not see it, the rows from it on are
    not finite in its dim alone."""
    k, v, q = inputs(start + T, T, start + T)
    head, dim = 3, 11
    v[start + late, head, dim] = bad
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, start)
    finite = np.where(np.isfinite(vv), vv, 0.0)
    check(out, q, kk, finite, start, [0, late // 2, late - 1])
    assert not np.any(np.isfinite(out[late:, 2 * head:2 * head + 2, dim]))
    out[late:, 2 * head:2 * head + 2, dim] = 0.0
    for t in (late, T - 1):
        ref = attend64(q[t].numpy(), kk[:start + t + 1], finite[:start + t + 1], SCALE)
        ref[2 * head:2 * head + 2, dim] = 0.0
        assert rel_err(out[t], ref) <= TOL_F32 / 2, t


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_later_rows_value_in_the_tiered_window(ctx, bad):
    start, T, late = 3050, 16, 12
    k, v, q = inputs(start + T, T, 5)
    v[start + late, 3, 11] = bad
    out, kk, vv = prefill(ctx, k, v, q, abi.F32, abi.I8_TIERED, start)
    check(out, q, kk, np.where(np.isfinite(vv), vv, 0.0), start, [0, late - 1])


@pytest.mark.parametrize("vdt", [abi.F16, abi.F32, abi.BF16])
def test_a_later_rows_key_stays_out_of_earlier_rows(ctx, vdt):
    start, T, late = 2400, 16, 12
    k, v, q = inputs(start + T, T, 6)
    k[start + late, 3, 11] = float("nan")
    out, kk, vv = prefill(ctx, k, v, q, abi.F32, vdt, start)
    check(out, q, np.where(np.isfinite(kk), kk, 0.0), vv, start, [0, late - 1])


# ---- weights and values of all sizes ------------------------------------------------------

@pytest.mark.parametrize("kdt,vdt", PLANS)
@pytest.mark.parametrize("bits", [12, 16, 20, 24, 27, 30])
def test_a_large_value_under_a_small_weight(ctx, kdt, vdt, bits):
    """One position of weight 2^-bits whose value outweighs all the others': its
    weight counts with all of its bits.  (Tiered values hold it in the binary16
    window.)"""
    start, T = 60, 64
    n = start + T
    k, v, q = inputs(n, T, bits)
    k.zero_()
    q.fill_(1.0)
    at = start + 1  # in the window of the last 64 positions, seen by every row but the first
    k[at] = -round((bits + 0.3) * np.log(2.0) * 4) / 4  # 64 dims of it times 1/64, exact in any sum
    v *= 2.0 ** -18
    v[at] = 60000.0 * (1 + torch.arange(64) / 100.0) / 2
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, start)
    e = check(out, q, kk, vv, start, [1, 2, 3, 40, T - 1])
    log(f"large value under 2^-{bits} {kdt}/{vdt}: vs float64 {e:.2e}")


@pytest.mark.parametrize("kdt,vdt", [(k, v) for k, v in PLANS if v in (abi.F32, abi.BF16)])
@pytest.mark.parametrize("power", [-118, -112, -105, -60, 50, 59, 61, 100, 118])
def test_values_near_the_ends_of_binary32(ctx, kdt, vdt, power):
    """Values of one far magnitude, under weights within 2^-2 of each other."""
    T = 200
    k, v, q = inputs(T, T, power + 200)
    v *= 2.0 ** power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    for t in [0, 63, 64, 150, T - 1]:
        ref = attend64(q[t].numpy(), kk[:t + 1], vv[:t + 1], SCALE)
        e = rel_err(out[t] * 2.0 ** -power, ref * 2.0 ** -power)
        assert e <= TOL_F32 / 2, (t, e)


@pytest.mark.parametrize("kdt,vdt", [(k, v) for k, v in PLANS if v in (abi.F32, abi.BF16)])
def test_small_and_large_tiles_in_one_call(ctx, kdt, vdt):
    """Tiles of every range in turn, so that the sums pass from one way of
    forming the products to the other and back; each weighed so as to count."""
    T = 320
    k, v, q = inputs(T, T, 3)
    for tile, power in enumerate((0, 70, 3, -110, 66)):
        v[64 * tile:64 * tile + 64] *= 2.0 ** power
    out, kk, vv = prefill(ctx, k, v, q, kdt, vdt, 0)
    check(out, q, kk, vv, 0, [0, 63, 64, 130, 200, 300, T - 1])


# ---- the bits of a product -------------------------------------------------------------

@pytest.mark.parametrize("vdt", [abi.F16, abi.F32])
@pytest.mark.parametrize("bits", [0x3f80ff80, 0x3f807f80, 0x3f817fc0])
def test_product_bits(ctx, vdt, bits):
    """Two keys of nearly one score, one of the query's own 17 bits a dim and one
    of 8: the first needs every product of pieces.  Their values are 1 and -1,
    so the result errs by half of the scores' error.  In units of 2^-24 of the
    score: at most 1 is left out by the pieces and 1 goes to the rounding of
    each sum; a leading piece that is cut off leaves out up to 4."""
    x = np.array([bits], np.uint32).view(np.float32)[0].item()
    near = float(torch.tensor(x).to(torch.bfloat16))
    T, big = 64, 32.0
    k = torch.full((T, 8, 64), -big)  # the other positions weigh nothing
    v = torch.zeros((T, 8, 64))
    q = torch.full((T, 16, 64), x * big)
    k[0], k[1] = x * big, near * big
    v[0], v[1] = 1.0, -1.0
    out, kk, vv = prefill(ctx, k, v, q, abi.F32, vdt, 0)
    ref = attend64(q[1].numpy(), kk[:2], vv[:2], SCALE)
    unit = big * big * x * x * 64 * SCALE * 2.0 ** -24
    err = np.max(np.abs(out[1:] - ref)) * 2 / unit
    log(f"score error {err:.2f} units of 2^-24")
    assert err <= 3


# ---- workspace -------------------------------------------------------------------------

@pytest.mark.parametrize("kdt,vdt", PLANS)
@pytest.mark.parametrize("capacity", [300, 512, 1000])
def test_a_workspace_of_a_long_prompt_serves_shorter_ones(ctx, kdt, vdt, capacity):
    """A program asks once, for its longest prompt."""
    window = 64 if vdt == abi.I8_TIERED else 0
    arena = rt.KvArena(ctx, abi.SHAPE_GRANITE, 1, 1, capacity, kdt, vdt, value_window=window)
    sizes = [rt.prefill_workspace_bytes(arena, t) for t in range(1, capacity + 1)]
    assert sizes == sorted(sizes)
    workspace = torch.empty(sizes[-1], dtype=torch.uint8, device="cuda")
    q = torch.randn((127, 16, 64), device="cuda")
    with rt.Graph(ctx) as g:
        arena.fill_normal(g, seed=1, length=capacity)
        want = rt.prefill_attention(g, arena, 0, capacity - 127, q)
        out = rt.prefill_attention(g, arena, 0, capacity - 127, q, workspace=workspace)
    assert torch.equal(out, want)


# ---- tiered values at the edges of tiles and chunks -------------------------------------------

@pytest.mark.parametrize("window", [32, 128])
@pytest.mark.parametrize("start,T", [(0, 64), (0, 65), (63, 66), (1, 255), (700, 128), (300, 640)])
def test_tiered_values_at_edges(ctx, start, T, window):
    k, v, q = inputs(start + T, T, start + T + window)
    q *= 6
    cap = start + T
    arena = rt.KvArena(ctx, abi.SHAPE_GRANITE, 1, 1, cap, abi.F32, abi.I8_TIERED, value_window=window)
    with rt.Graph(ctx) as g:
        rt.store_kv(g, arena, 0, 0, k[None].cuda(), v[None].cuda())
        out = rt.prefill_attention(g, arena, 0, start, q.cuda())
        kk, vv = arena.gather(g, 0, 0, 0, cap)
    check(out.cpu().numpy(), q, kk.float().cpu().numpy(), vv.float().cpu().numpy(), start,
          sorted({0, 1, T // 2, max(0, T - 65), T - 1}))
