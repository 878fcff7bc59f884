"""The scratch a HipMoE layer holds and what a long prompt adds to it, on the CPU (the library
sizes the workspace; the launches are replaced by a record of the calls)."""

import pytest
import torch

from tests.test_abi import _desc
from wanferenz_amd import _native as N
from wanferenz_amd import moe as M

D, I, E, K = 256, 128, 256, 6
SMALL = 16384 // K      # tokens of the chunk that every layer runs
LARGE = 65536 // K      # ... of the largest chunk of a layer of 256 experts


@pytest.fixture
def layer(monkeypatch):
    h = object.__new__(M.HipMoE)
    h.cfg = M.MoEConfig(dim=D, inter=I, n_experts=E, topk=K)
    h.desc, h.device, h.tid2eid = _desc(D, I, E, K), torch.device("cpu"), None
    h._ws, h._ws_tokens = None, 0
    h.calls = []
    monkeypatch.setattr(N, "call", lambda name, *a: h.calls.append((name, a)))
    monkeypatch.setattr(N, "stream_handle", lambda device=None: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    return h


def _forward(layer, T):
    """(pointer, bytes) of the workspace the forward of T tokens ran on, and whether it was cleared."""
    layer.calls.clear()
    layer.forward(torch.zeros(T, D, dtype=torch.bfloat16))
    name, args = layer.calls[-1]
    assert name == "wz_moe_forward"
    ws = (args[7], args[8])
    return ws, ("wz_moe_workspace_init", ws[0], ws[1]) in [(n, *a[:2]) for n, a in layer.calls]


@pytest.mark.parametrize("T", [SMALL + 1, LARGE, 3 * LARGE])
def test_a_long_prompt_leaves_a_small_workspace_behind(layer, T):
    held = layer.workspace_bytes(SMALL)
    (ptr, nbytes), cleared = _forward(layer, T)
    assert nbytes == layer.workspace_bytes(T) > held and cleared
    assert layer._ws.numel() == held
    assert _forward(layer, SMALL)[0] == (layer._ws.data_ptr(), held)
    # the same for an explicit reservation, after which nothing the layer holds moves
    ws = layer._ws
    layer.reserve(4 * LARGE)
    assert layer._ws is ws
    _forward(layer, T)
    assert layer._ws is ws


def test_a_long_prompt_runs_where_its_workspace_cannot_be_had(layer, monkeypatch):
    held, empty = layer.workspace_bytes(SMALL), torch.empty

    def small_device(n, *a, **kw):
        if kw.get("dtype") == torch.uint8 and n > held:
            raise torch.OutOfMemoryError("out of memory")
        return empty(n, *a, **kw)

    monkeypatch.setattr(torch, "empty", small_device)
    assert _forward(layer, LARGE)[0] == (layer._ws.data_ptr(), held)
    assert layer._ws.numel() == held


def test_short_calls_use_the_held_workspace(layer):
    layer.reserve(SMALL)
    ws = layer._ws
    for T in (1, 16, 17, 500, SMALL):
        assert _forward(layer, T) == ((ws.data_ptr(), ws.numel()), False)
