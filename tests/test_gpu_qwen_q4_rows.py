"""The Qwen block's Q4 kernels read the hidden state and the norm weights 16
bytes at a time, from wherever the caller keeps them: element-aligned
addresses give the results of 16-byte-aligned ones bit for bit, and every
nibble and scale lands on its column (one-hot inputs read the weights back)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from qx_amd import abi
from qx_amd import runtime as rt
from tests.test_gpu_qwen_block import HID, dev, f16, to_device, weights, workspace_stages

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    return rt.Context(0)


def block(ctx, layer, hidden):
    arena = rt.KvArena(ctx, abi.SHAPE_QWEN3, 1, 1, 32, abi.F16)
    after = torch.empty(HID, dtype=torch.int16, device="cuda:0")
    moe = torch.empty_like(after)
    wsp = torch.zeros(rt.qwen_block_workspace_bytes(arena, 1), dtype=torch.uint8, device="cuda:0")
    with rt.Graph(ctx) as g:
        rt.qwen_attention_block(g, arena, 0, 0, layer, hidden, after, moe, wsp)
    return [x.cpu() for x in (after, moe)] + [x.cpu() for x in workspace_stages(wsp)]


@pytest.mark.parametrize("shift", [1, 2, 3, 5])
def test_element_aligned_inputs(ctx, shift):
    rng = np.random.default_rng(shift)
    mats, norms, layer = weights(rng)
    h = dev(rng.standard_normal(HID).astype(np.float16).view(np.int16))
    want = block(ctx, layer, h)
    moved = torch.zeros(HID + 8, dtype=torch.int16, device="cuda:0")
    moved[shift:shift + HID] = h
    n = torch.zeros(HID + 8, device="cuda:0")
    n[shift:shift + HID] = dev(norms[0])
    layer2 = rt.QwenQ4Layer(n[shift:shift + HID], *[to_device(m) for m in mats[:3]], dev(norms[1]), dev(norms[2]),
                            to_device(mats[3]), dev(norms[3]))
    for x, y in zip(want, block(ctx, layer2, moved[shift:shift + HID])):
        assert torch.equal(x, y)


@pytest.mark.parametrize("col", [0, 1, 4, 7, 31, 32, 1027, 2047])
def test_one_column_at_a_time(ctx, col):
    """A hidden state with one non-zero element: every q/k/v row is its own
    weight in that column times one activation, exact before the f16 rounding."""
    rng = np.random.default_rng(col)
    mats, norms, layer = weights(rng)
    h = np.zeros(HID, np.float16)
    h[col] = 2.0
    q, k, v = block(ctx, layer, dev(h.view(np.int16)))[2:5]
    act = O.qwen_rms_norm(h.astype(np.float32), norms[0]).astype(np.float16).astype(np.float32)
    for got, m in ((q, mats[0]), (k, mats[1]), (v, mats[2])):
        assert np.array_equal(f16(got), O.q4_mat_vec(m, act).astype(np.float16).astype(np.float32))
