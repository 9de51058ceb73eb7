"""Few causal rows over equal 16-bit caches (a drafted block to verify, a short
chunk of a prompt), where several rows share a workgroup
(decode_mfma_rows_kernel): row counts around a workgroup's rows (two or four on
the Qwen shape, eight on Granite's), contexts around the rules' lines and the
split's granularity of 128, against float64 attention over the cache's rows at
the 16-bit bar; an infinite value in a later drafted row, which must not
reach the rows before it; and queries of another dtype, rounded to the cache's
or refused."""
import numpy as np
import pytest
import torch

from qx_amd import abi
from qx_amd import runtime as rt
from tests.helpers import TOL_16, attend64, log, rel_err

pytestmark = pytest.mark.gpu

TORCH = {abi.F32: torch.float32, abi.F16: torch.float16, abi.BF16: torch.bfloat16}
HEADS = {abi.SHAPE_GRANITE: (16, 8, 64, 0.015625), abi.SHAPE_QWEN3: (32, 4, 128, 128.0 ** -0.5)}


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def rows(ctx, shape, dt, start, T, seed, plant=None):
    hq, hk, d, scale = HEADS[shape]
    g = torch.Generator(device="cuda").manual_seed(seed)
    arena = rt.KvArena(ctx, shape, 1, 1, start + T, dt)
    k = torch.randn((1, start + T, hk, d), generator=g, device="cuda").to(TORCH[dt])
    v = torch.randn((1, start + T, hk, d), generator=g, device="cuda").to(TORCH[dt])
    if plant is not None:
        v[0, start + plant[0], plant[1], plant[2]] = float("inf")
    q = (2 * torch.randn((T, hq, d), generator=g, device="cuda")).to(TORCH[dt])
    with rt.Graph(ctx) as graph:
        rt.store_kv(graph, arena, 0, 0, k, v)
        out = rt.prefill_attention(graph, arena, 0, start, q, out_dtype=torch.float32)
    return [x.float().cpu().numpy() for x in (q, k[0], v[0], out)]


CASES = [(abi.SHAPE_QWEN3, s, T) for s, T in ((9999, 2), (6700, 3), (4091, 5), (2490, 8), (2220, 9), (1250, 17),
                                              (640, 32), (2528, 33), (2500, 63), (100, 63), (3000, 2),
                                              # two column blocks a workgroup: full and ragged last fours
                                              (33400, 3), (25100, 4), (40000, 5), (14280, 7), (7000, 15),
                                              (6100, 33), (29900, 32), (1530, 63), (7870, 63))]
CASES += [(abi.SHAPE_GRANITE, s, T) for s, T in ((4000, 3), (2191, 5), (1367, 8), (1216, 9), (1100, 16), (1130, 31),
                                                 (620, 33), (600, 63), (4033, 63), (64, 9), (700, 2))]


@pytest.mark.parametrize("dt", [abi.F16, abi.BF16])
@pytest.mark.parametrize("shape,start,T", CASES)
def test_rows_match_float64(ctx, shape, dt, start, T):
    q, k, v, out = rows(ctx, shape, dt, start, T, start + T)
    worst = 0.0
    for t in sorted({0, 1, T // 2, T - 2, T - 1}):
        n = start + t + 1
        worst = max(worst, rel_err(out[t], attend64(q[t], k[:n], v[:n], HEADS[shape][3])))
    log(f"causal rows {shape} {dt} {start}+{T}: {worst:.2e}")
    assert worst <= TOL_16


@pytest.mark.parametrize("shape,dt", [(abi.SHAPE_QWEN3, abi.BF16), (abi.SHAPE_QWEN3, abi.F16),
                                      (abi.SHAPE_GRANITE, abi.F16), (abi.SHAPE_GRANITE, abi.BF16)])
@pytest.mark.parametrize("start,T,late", [(6000, 5, 1), (6000, 5, 3), (6000, 5, 4),
                                          (14300, 7, 1), (14300, 7, 2), (14300, 7, 5)])
def test_an_infinite_draft_value_stays_out_of_earlier_rows(ctx, shape, dt, start, T, late):
    head, dim = 1, 9
    q, k, v, out = rows(ctx, shape, dt, start, T, late, plant=(late, head, dim))
    hq, hk, d, scale = HEADS[shape]
    group = hq // hk
    for t in range(T):
        n = start + t + 1
        vals = np.where(np.isfinite(v[:n]), v[:n], 0.0)
        ref = attend64(q[t], k[:n], vals, scale)
        got = out[t].copy()
        if t >= late:
            # inf, or NaN where bf16's second piece of the probability is negative
            assert not np.any(np.isfinite(got[head * group:(head + 1) * group, dim]))
            got[head * group:(head + 1) * group, dim] = ref[head * group:(head + 1) * group, dim]
        assert rel_err(got, ref) <= TOL_16, t


@pytest.mark.parametrize("shape,dt,start,T,taken", [
    (abi.SHAPE_QWEN3, abi.BF16, 12000, 16, True), (abi.SHAPE_QWEN3, abi.BF16, 13000, 16, False),
    (abi.SHAPE_QWEN3, abi.F16, 15000, 8, True), (abi.SHAPE_GRANITE, abi.F16, 2000, 34, True),
    (abi.SHAPE_GRANITE, abi.F16, 2100, 34, False), (abi.SHAPE_GRANITE, abi.BF16, 2600, 34, True),
    (abi.SHAPE_GRANITE, abi.BF16, 2700, 34, False)])
def test_a_query_of_another_dtype_is_taken_up_to_its_limit(ctx, shape, dt, start, T, taken):
    """The limit is the call's own: (T - 6) x context of 126000 on the Qwen
    shape, T x context of 70000 (f16) or 90000 (bf16) on Granite's."""
    hq, hk, d, _ = HEADS[shape]
    arena = rt.KvArena(ctx, shape, 1, 1, start + T, dt)
    arena.set_len(start + T)
    q = torch.zeros((T, hq, d), device="cuda")
    with rt.Graph(ctx) as graph:
        if taken:
            rt.prefill_attention(graph, arena, 0, start, q)
        else:
            with pytest.raises(abi.QxhError) as e:
                rt.prefill_attention(graph, arena, 0, start, q)
            assert e.value.code == abi.QXH_ERR_UNSUPPORTED


@pytest.mark.parametrize("qdt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,dt,start,T", [
    (abi.SHAPE_QWEN3, abi.BF16, 12000, 5), (abi.SHAPE_QWEN3, abi.F16, 12000, 13),  # one column block a workgroup
    (abi.SHAPE_QWEN3, abi.BF16, 15000, 7), (abi.SHAPE_QWEN3, abi.F16, 15000, 8),  # two
    (abi.SHAPE_QWEN3, abi.BF16, 10000, 12), (abi.SHAPE_QWEN3, abi.BF16, 3000, 2),
    (abi.SHAPE_GRANITE, abi.F16, 2000, 34), (abi.SHAPE_GRANITE, abi.BF16, 1300, 9)])
def test_a_query_of_another_dtype_is_rounded_to_the_caches(ctx, shape, dt, start, T, qdt):
    """Sequence 1 of three, in a cache with room past the call."""
    hq, hk, d, scale = HEADS[shape]
    g = torch.Generator(device="cuda").manual_seed(start + T)
    arena = rt.KvArena(ctx, shape, 1, 3, start + T + 77, dt)
    k, v = (torch.randn((3, start + T + 50, hk, d), generator=g, device="cuda").to(TORCH[dt]) for _ in range(2))
    q = (2 * torch.randn((T, hq, d), generator=g, device="cuda")).to(qdt)
    out = torch.full((T, hq, d), float("nan"), device="cuda")
    with rt.Graph(ctx) as graph:
        rt.store_kv(graph, arena, 0, 0, k, v)
        rt.prefill_attention(graph, arena, 0, start, q, out=out, sequence=1)
    qf = q.float().to(TORCH[dt]).float().cpu().numpy()
    kf, vf, out = k[1].float().cpu().numpy(), v[1].float().cpu().numpy(), out.cpu().numpy()
    for t in sorted({0, 1, T // 2, T - 2, T - 1}):
        n = start + t + 1
        assert rel_err(out[t], attend64(qf[t], kf[:n], vf[:n], scale)) <= TOL_16, t
    assert np.all(np.isfinite(out))
