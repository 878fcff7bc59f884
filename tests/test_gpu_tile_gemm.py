"""The tile GEMM (linear_gemm.hip) at its edges: remainders of every tile shape in M and N,
the shortest and odd K, each scale kind, unaligned and split outputs.  The cases reach every
compiled tile kernel, which test_tile_shapes.py checks without a GPU.

Every path of a weight form sums in one order, so a row of a wide call must have the bits of
the same row in a call of up to 16 rows, which the GEMV and skinny kernels serve (those are
held against the oracle in test_gpu_kernels.py): torch.equal, no tolerance."""

import pytest
import torch

from tests.helpers import bf16_tensor
from wanferenz_amd import _native as N
from wanferenz_amd import kernels, synth

pytestmark = pytest.mark.gpu


def _rows(M, K, dev):
    return bf16_tensor(synth.normal_bf16(synth.stream_key(M + K, synth.S_FP8_X), (M, K), 1.0), dev).view(M, K)


def _quant(x, act):
    return kernels.act_quant(x, 128, act, torch.float8_e8m0fnu if act else torch.float32)


def _narrow(gemm, q, qs):
    return torch.cat([gemm(q[i:i + 16].contiguous(), qs[i:i + 16].contiguous()) for i in range(0, q.size(0), 16)])


def _weight8(n, k, w_fp32, dev):
    from wanferenz_amd import stage

    return stage.synthetic_linear(n, k, n + k, dev, fp32_scales=w_fp32)


# (M, N, K): one row past a tile of each height; N of one and of nine 16-column tiles; a single
# K-block, K-block counts no stage divides, and grids that reach each larger tile shape.  Narrow
# calls with power-of-two scales stay on the skinny kernel (17 x 16 x 128)
ROW_SHAPES = [(17, 16, 128), (33, 144, 384), (65, 272, 640), (100, 4096, 512), (129, 8192, 1024),
              (257, 16400, 256), (700, 4096, 1152), (200, 4080, 8064)]
# MXFP4 rows are staged two K-blocks at a time: K of whole pairs, stages that end half full (an
# odd number of pairs: 256, 768, 1280) and, with K = 384, what the tile GEMM does not serve
FP4_SHAPES = [(33, 16, 256), (33, 144, 768), (65, 272, 1280), (31, 20496, 768), (100, 4096, 512),
              (333, 2048, 4096), (257, 8208, 256), (300, 5136, 768), (700, 4112, 1280), (1030, 8192, 768),
              (40, 144, 384)]
# packed weights: K = 1024 is one K-block a slice of the sum, 2048 and 4096 two, 8192 four, others all
PACKED_SHAPES = [(33, 144, 1024), (100, 4112, 1024), (300, 5136, 1024), (257, 16400, 1024), (520, 32784, 1024),
                 (300, 32656, 1024), (300, 2064, 4096), (300, 5136, 2048), (1030, 4112, 2048), (200, 272, 640), (200, 4080, 8192)]


@pytest.mark.parametrize("act", ["ue8m0", None])
@pytest.mark.parametrize("w_fp32", [False, True])
@pytest.mark.parametrize("M,Nn,K", ROW_SHAPES)
def test_fp8_rows_have_the_narrow_bits(gpu, M, Nn, K, w_fp32, act):
    w, ws = _weight8(Nn, K, w_fp32, gpu)
    q, qs = _quant(_rows(M, K, gpu), act)
    assert torch.equal(kernels.fp8_gemm(q, qs, w, ws), _narrow(lambda a, s: kernels.fp8_gemm(a, s, w, ws), q, qs))


@pytest.mark.parametrize("act", ["ue8m0", None])
@pytest.mark.parametrize("M,Nn,K", FP4_SHAPES)
def test_fp4_rows_have_the_narrow_bits(gpu, M, Nn, K, act):
    g = torch.Generator(device="cuda").manual_seed(M)
    w = torch.randint(0, 256, (Nn, K // 2), device=gpu, generator=g, dtype=torch.uint8).view(torch.float4_e2m1fn_x2)
    ws = torch.randint(118, 122, (Nn, K // 32), device=gpu, generator=g, dtype=torch.uint8).view(torch.float8_e8m0fnu)
    q, qs = _quant(_rows(M, K, gpu), act)
    assert torch.equal(kernels.fp4_gemm(q, qs, w, ws), _narrow(lambda a, s: kernels.fp4_gemm(a, s, w, ws), q, qs))


@pytest.mark.parametrize("act", ["ue8m0", None])
@pytest.mark.parametrize("w_fp32", [False, True])
@pytest.mark.parametrize("M,Nn,K", PACKED_SHAPES)
def test_packed_rows_have_the_narrow_bits(gpu, M, Nn, K, w_fp32, act):
    w, ws = _weight8(Nn, K, w_fp32, gpu)
    lin = kernels.PackedFp8Linear(w, ws, act)
    q, qs = _quant(_rows(M, K, gpu), act)
    y = lin.gemm(q, qs)
    # K outside the GEMV's set sums in one slice on every path: compared over the rows of one M-tile
    ref = _narrow(lin.gemm, q, qs)
    assert torch.equal(y, ref)


SPLITS = [(37, 128, 80), (300, 4096, 2064), (300, 32512, 144)]


@pytest.mark.parametrize("M,N0,N1", SPLITS)
def test_unaligned_and_split_outputs(gpu, M, N0, N1):
    """Outputs two bytes past a 16-byte boundary take the scalar stores; the split at N0 and
    the residual add give the unsplit, aligned bits."""
    K = 1024
    w, ws = _weight8(N0 + N1, K, False, gpu)
    lin = kernels.PackedFp8Linear(w, ws)
    q, qs = _quant(_rows(M, K, gpu), "ue8m0")
    ref = lin.gemm(q, qs)
    nsb = N0 // 128
    pair = kernels.PackedFp8Pair(w[:N0].contiguous(), ws[:nsb].contiguous(), w[N0:].contiguous(),
                                 ws[nsb:].contiguous())
    y0 = torch.empty(M * N0 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(M, N0)
    y1 = torch.empty(M * N1 + 1, dtype=torch.bfloat16, device=gpu)[1:].view(M, N1)
    pair.gemm(q, qs, out=(y0, y1))
    assert torch.equal(torch.cat([y0, y1], 1), ref)
    res = _rows(M, N0 + N1, gpu)
    need = int(N.lib().wz_fp8_gemm_packed_workspace_bytes(M, K, N.WZ_SCALE_UE8M0))
    wsp = torch.empty(max(need, 256), dtype=torch.uint8, device=gpu)
    for off in (0, 1):
        y = torch.empty(M * (N0 + N1) + off, dtype=torch.bfloat16, device=gpu)[off:]
        N.call("wz_fp8_gemm_packed_add", N.ptr(q), N.ptr(qs), N.ptr(lin.packed), N.ptr(ws), N.ptr(res), N.ptr(y), M,
               N0 + N1, K, N.WZ_SCALE_UE8M0, N.WZ_WSCALE_E8M0, N.ptr(wsp), wsp.numel(), N.stream_handle(gpu))
        assert torch.equal(y.view(M, -1), (ref.float() + res.float()).to(torch.bfloat16))
