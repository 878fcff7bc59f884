"""grouped_fp4_gemm at K = 2048 and 4096, where a workgroup keeps the row in LDS and reads a
quarter's weight scales at once, against fp4_gemm of each row (the same products in the same
order: equal bits), and at an unaligned row start, which the general body serves."""

import pytest
import torch

from tests.helpers import u8_tensor
from tests.test_gpu_kernels import _fp4_weight
from wanferenz_amd import kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("fmt,sd", [("ue8m0", torch.float8_e8m0fnu), ("ue8m0", torch.float32), (None, torch.float32)])
@pytest.mark.parametrize("G,N,shift", [(1, 128, 0), (5, 128, 0), (3, 384, 4)])
def test_grouped_rows_equal_fp4_gemm(gpu, K, fmt, sd, G, N, shift):
    g = torch.Generator(device=gpu).manual_seed(G * 100 + N + K)
    x = (torch.randn(G, K, device=gpu, generator=g) * torch.logspace(-3, 2, G, device=gpu)[:, None]).to(torch.bfloat16)
    q, s = kernels.act_quant(x, 128, fmt, sd)
    if shift:  # the codes at an address that is not a multiple of 16
        raw = torch.zeros(G * K + 16, dtype=torch.uint8, device=gpu)
        raw[shift:shift + G * K] = q.view(torch.uint8).flatten()
        q = raw[shift:shift + G * K].view(torch.float8_e4m3fn).view(G, K)
    w, ws = zip(*[_fp4_weight(N * 7 + K + e, N, K) for e in range(G)])
    wt = torch.stack([u8_tensor(a, gpu) for a in w]).view(torch.float4_e2m1fn_x2)
    wst = torch.stack([u8_tensor(a, gpu) for a in ws]).view(torch.float8_e8m0fnu)
    got = kernels.grouped_fp4_gemm(q, s, wt, wst, sd)
    rows = torch.cat([kernels.fp4_gemm(q[e:e + 1], s[e:e + 1], wt[e], wst[e], sd) for e in range(G)])
    assert torch.equal(got.view(torch.int16), rows.view(torch.int16))
