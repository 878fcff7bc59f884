"""GPU parity of sparse attention (wz_sparse_attn, kernels.sparse_attn) against the
oracle's restatement of torch_ops.py:114-146.

Bar: bf16 outputs within max|d|/max|ref| <= 1e-2 and cosine >= 0.9999 (the kernels
multiply a bf16 P by V, as the reference's GPU kernel does, reference.py:404-405;
the CPU reference keeps P in fp32); queries the reference turns into NaN (no valid
index in the first block of 64) are NaN here.  A workgroup holds one, two or four
tiles of 16 heads, and few queries are split over workgroups with a workspace.
"""

import numpy as np
import pytest
import torch

from oracle import moe as om
from oracle.numerics import bf16_bits
from tests.helpers import bf16_tensor, f32_of_bf16
from tests.test_oracle_attn import _inputs
from wanferenz_amd import _native as N
from wanferenz_amd import kernels

pytestmark = pytest.mark.gpu


def _dev(gpu, q, kv, sink, idx):
    return (bf16_tensor(bf16_bits(q), gpu).view(q.shape), bf16_tensor(bf16_bits(kv), gpu).view(kv.shape),
            torch.from_numpy(sink).to(gpu), torch.from_numpy(idx).to(gpu))


def _run(gpu, q, kv, sink, idx, scale):
    o = kernels.sparse_attn(*_dev(gpu, q, kv, sink, idx), scale)
    torch.cuda.synchronize()
    return f32_of_bf16(o).reshape(q.shape)


def _check(got, ref):
    rel, cos = om.max_rel_err(got, ref), om.cosine(got, ref)
    assert rel <= 1e-2 and cos >= 0.9999, (rel, cos)


@pytest.mark.parametrize("b,s,h,d,n,topk", [
    (1, 1, 64, 512, 2048, 640),    # V4 decode: 64 heads of 512, window 128 + 512 selected (split)
    (4, 1, 64, 512, 1024, 640),    # decode batch of 4 (split)
    (1, 4, 64, 512, 1024, 640),
    (1, 512, 64, 128, 700, 100),   # 512 queries: one workgroup per query, partial last block
    (2, 3, 128, 256, 300, 130),    # two 64-head groups
    (2, 3, 16, 128, 300, 100),     # 16-head kernel, partial last block
    (1, 2, 8, 256, 500, 64),       # 8 heads: padded to 16
    (1, 2, 32, 512, 400, 200),
])
def test_sparse_attn_matches_oracle(gpu, b, s, h, d, n, topk):
    q, kv, sink, idx = _inputs(b * 100 + h + topk + s, b, s, h, d, n, topk)
    idx[..., 0] = np.maximum(idx[..., 0], 0)  # every query sees at least one row in its first block
    scale = d ** -0.5
    _check(_run(gpu, q, kv, sink, idx, scale), om.sparse_attn(q, kv, sink, idx, scale))


def test_split_and_unsplit_agree(gpu):
    """The decode shape through the split path (workspace) and through one workgroup
    per query (no workspace): both meet the bar against the oracle."""
    b, s, h, d, n, topk = 2, 1, 64, 512, 900, 640
    q, kv, sink, idx = _inputs(11, b, s, h, d, n, topk)
    idx[..., 0] = np.maximum(idx[..., 0], 0)
    ref = om.sparse_attn(q, kv, sink, idx, d ** -0.5)
    assert kernels.sparse_attn_workspace_bytes(b, s, h, d, topk) > 0
    qt, kvt, st, it = _dev(gpu, q, kv, sink, idx)
    o = torch.empty_like(qt)
    N.call("wz_sparse_attn", N.ptr(qt), N.ptr(kvt), N.ptr(st), N.ptr(it), N.ptr(o), b, s, h, d, n, topk,
           d ** -0.5, None, 0, N.stream_handle(qt.device))
    torch.cuda.synchronize()
    _check(f32_of_bf16(o).reshape(q.shape), ref)
    _check(_run(gpu, q, kv, sink, idx, d ** -0.5), ref)


@pytest.mark.parametrize("h,s", [(16, 2), (64, 2), (64, 600)])
def test_unused_first_block_is_nan(gpu, h, s):
    q, kv, sink, idx = _inputs(7, 1, s, h, 128, 100, 130)
    idx[0, 0, :64] = -1        # query 0: nothing valid in its first block -> NaN (as the reference)
    idx[0, 1, 64:] = -1        # query 1: a fully unused later block contributes nothing
    idx[0, 1, 0] = 3
    idx[0, 2:, 0] = np.maximum(idx[0, 2:, 0], 0)
    got = _run(gpu, q, kv, sink, idx, 128 ** -0.5)
    ref = om.sparse_attn(q, kv, sink, idx, 128 ** -0.5)
    assert np.isnan(got[0, 0]).all() and np.isnan(ref[0, 0]).all()
    assert not np.isnan(got[0, 1:]).any()
    _check(got[0, 1:], ref[0, 1:])


@pytest.mark.parametrize("h", [16, 64])
def test_unused_slots_read_zeros(gpu, h):
    """Row 0 of the cache holds NaN and is never selected: unused (-1) slots must not
    bring it in (the reference zero-fills them)."""
    q, kv, sink, idx = _inputs(9, 1, 3, h, 256, 200, 192, invalid=0.5)
    kv[0, 0] = np.nan
    idx[idx == 0] = 1
    idx[..., 0] = 5
    got = _run(gpu, q, kv, sink, idx, 256 ** -0.5)
    assert not np.isnan(got).any()
    _check(got, om.sparse_attn(q, kv, sink, idx, 256 ** -0.5))


def test_bad_shapes_raise(gpu):
    q = torch.zeros(1, 1, 64, 96, dtype=torch.bfloat16, device=gpu)
    kv = torch.zeros(1, 10, 96, dtype=torch.bfloat16, device=gpu)
    with pytest.raises(N.WzError, match="head dim"):
        kernels.sparse_attn(q, kv, torch.zeros(64, device=gpu), torch.zeros(1, 1, 4, dtype=torch.int32, device=gpu),
                            1.0)


@pytest.mark.parametrize("h,d,s", [(64, 512, 1), (64, 128, 600), (16, 256, 3)])
def test_running_max_moves(gpu, h, d, s):
    """Rows grow block by block (row r scaled by 1 + 5 (r // 64)), so the running
    maximum moves by more than 8 at later blocks and the accumulated output is
    rescaled on the way; split (few queries) and unsplit (600 queries) paths."""
    topk = 320
    q, kv, sink, idx = _inputs(21 + h + d, 1, s, h, d, topk, topk, invalid=0.0)
    grow = (1.0 + 5.0 * (np.arange(topk) // 64)).astype(np.float32)
    kv = om.bf16_round((kv * grow[None, :, None]).astype(np.float32))
    idx[:] = np.arange(topk, dtype=np.int32)
    idx[..., 70] = -1  # an unused slot inside a later block as well
    scale = d ** -0.5
    ref = om.sparse_attn(q, kv, sink, idx, scale)
    _check(_run(gpu, q, kv, sink, idx, scale), ref)


@pytest.mark.parametrize("h", [16, 32, 48, 64, 80])
@pytest.mark.parametrize("s", [1, 260, 513])
def test_head_groups_and_empty_blocks(gpu, h, s):
    """Each number of head tiles a workgroup can hold (one, two, four with the last one
    missing, a second group of one), split over workgroups and not (from 512 head groups on),
    with blocks that have no valid index first-but-one, in the middle and last: they are
    skipped and add nothing."""
    d, topk = 512, 64 * 6 + 5
    q, kv, sink, idx = _inputs(31 + h + s, 1, s, h, d, 300, topk, invalid=0.3)
    idx[..., 0] = np.maximum(idx[..., 0], 0)
    idx[:, ::2, 64:128] = -1
    idx[:, 1::3, 192:320] = -1
    idx[:, ::4, 384:] = -1
    scale = d ** -0.5
    _check(_run(gpu, q, kv, sink, idx, scale), om.sparse_attn(q, kv, sink, idx, scale))


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("h", [32, 48, 80, 96, 144])
@pytest.mark.parametrize("s", [1, 257])
def test_head_groups_of_narrow_heads(gpu, d, h, s):
    """The same with heads of 128 (a wave per 16 heads past 32) and 256: last groups of one, two
    and three tiles, the running maximum moving by more than 8, and a NaN query head, whose
    products and rescales must not reach its neighbours."""
    topk = 64 * 4 + 5
    q, kv, sink, idx = _inputs(57 + h + s + d, 1, s, h, d, 300, topk, invalid=0.2)
    kv = om.bf16_round((kv * (1.0 + 5.0 * (np.arange(300) // 60))[None, :, None]).astype(np.float32))
    idx.sort(axis=-1)
    idx[..., 0] = np.maximum(idx[..., 0], 0)
    idx[:, ::2, 64:128] = -1
    idx[:, 1::3, 128:] = -1
    scale = d ** -0.5
    ref = om.sparse_attn(q, kv, sink, idx, scale)
    _check(_run(gpu, q, kv, sink, idx, scale), ref)
    q[:, :, 5] = np.nan
    got = _run(gpu, q, kv, sink, idx, scale)
    assert np.isnan(got[:, :, 5]).all()
    keep = np.arange(h) != 5
    _check(got[:, :, keep], ref[:, :, keep])
