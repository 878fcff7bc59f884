"""wz_moe_forward's chunks of a long prompt: a layer of many experts takes up to 65536 routed
pairs at once, a caller whose workspace holds 16384 pairs gets chunks of those.  The layer is
token-local, so the outputs and routing of chunks that run the prefill kernels are equal; a rest of
up to 16 tokens runs the decode kernels and is left out of that comparison."""

import ctypes
import dataclasses

import pytest
import torch

from tests.golden.cases import CASES, make_inputs
from tests.helpers import bf16_tensor
from wanferenz_amd import _native as N

pytestmark = pytest.mark.gpu


def _run(moe, x, ws):
    T, dev = x.size(0), moe.device
    y = torch.empty_like(x)
    w = torch.empty(T, moe.cfg.topk, device=dev, dtype=torch.float32)
    i = torch.empty(T, moe.cfg.topk, device=dev, dtype=torch.int64)
    N.call("wz_moe_workspace_init", ws.data_ptr(), ws.numel(), N.stream_handle(dev))
    N.call("wz_moe_forward", ctypes.byref(moe.desc), x.data_ptr(), None, T, y.data_ptr(), w.data_ptr(), i.data_ptr(),
           ws.data_ptr(), ws.numel(), N.stream_handle(dev))
    return y, w, i


# 65536 / 6 = 10922 tokens a chunk at 256 experts (64 count workgroups in the permutation), 5461 at
# 128; the small chunks of 2730 leave 2, 22, 20 and 17 tokens
@pytest.mark.parametrize("E,T", [(256, 10922), (256, 10942), (128, 5480), (128, 2731 + 16)])
def test_large_chunks_equal_small_ones(gpu, E, T):
    from tests.test_gpu_moe import upload_case

    case = dataclasses.replace(CASES["top6_t8"], name=f"chunks_e{E}_t{T}", dim=256, inter=128, n_experts=E, T=T)
    inp = make_inputs(case)
    moe = upload_case(case, inp, gpu)
    x = bf16_tensor(inp.x, gpu)
    small = 16384 // case.topk
    need = moe.workspace_bytes(T)
    assert need > moe.workspace_bytes(small)
    big = _run(moe, x, torch.empty(need, dtype=torch.uint8, device=gpu))
    few = _run(moe, x, torch.empty(moe.workspace_bytes(small), dtype=torch.uint8, device=gpu))
    n = T - T % small if T % small <= 16 else T
    for a, b in zip(big, few):
        assert torch.equal(a[:n], b[:n])
    # sampled rows against calls of their own, 32 tokens each
    for t in (0, small - 16, T - 32):
        assert torch.equal(big[0][t:t + 32], moe.forward(x[t:t + 32].contiguous()))


# the wide routed tiles against calls of 700 tokens, whose rows are in 64-row tiles: a partial last
# N-block of w2 (640 columns), five K-blocks (a ragged group of scales), experts of many tiles and of
# few rows, a skewed selection with empty experts (test_moe_routes.py: each case takes wide tiles)
WIDE = dict(dim=640, inter=384, topk=2)
WIDE_CASES = [(5, 5200, 0.0), (40, 3011, 0.0), (64, 1555, 0.05), (17, 4500, 1.0)]


@pytest.mark.parametrize("E,T,skew", WIDE_CASES)
def test_wide_tiles_equal_narrow_ones(gpu, E, T, skew):
    from tests.test_gpu_moe import upload_case

    case = dataclasses.replace(CASES["top6_t8"], name=f"wide_e{E}_t{T}", n_experts=E, T=T, **WIDE)
    inp = make_inputs(case)
    moe = upload_case(case, inp, gpu)
    if skew:
        moe.weights.gate_bias.copy_(torch.linspace(skew, -skew, E))
    x = bf16_tensor(inp.x, gpu)
    y, w, i = _run(moe, x, torch.empty(moe.workspace_bytes(T), dtype=torch.uint8, device=gpu))
    for at in range(0, T, 700):
        n = min(700, T - at)
        ws = torch.empty(moe.workspace_bytes(n), dtype=torch.uint8, device=gpu)
        for a, b in zip((y, w, i), _run(moe, x[at:at + n].contiguous(), ws)):
            assert torch.equal(a[at:at + n], b)


def test_captured_long_prompt(gpu):
    """The larger workspace of a captured long prompt belongs to the graph: replays, with eager
    calls of other lengths between them, give the eager bits."""
    from tests.test_gpu_moe import upload_case

    T = 2731 + 16
    case = dataclasses.replace(CASES["top6_t8"], name="captured_chunk", dim=256, inter=128, n_experts=128, T=T)
    inp = make_inputs(case)
    moe = upload_case(case, inp, gpu)
    x = bf16_tensor(inp.x, gpu)
    y = moe.forward(x)
    moe.reserve(T)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = moe.forward(x)
    for n in (32, 200, T):
        g.replay()
        assert torch.equal(out, y)
        assert torch.equal(moe.forward(x[:n].contiguous()), y[:n])
        out.zero_()
