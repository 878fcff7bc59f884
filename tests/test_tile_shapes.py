"""Which tile GEMM kernels the host side selects (linear_gemm.hip), on a recording HIP runtime: every
compiled one is the choice of some call."""

import itertools
import re

import pytest

from tests.launch_recorder import record
from wanferenz_amd import _native as N

P = 1 << 20  # a 16-byte aligned stand-in for every operand: nothing is dereferenced
BIG = 1 << 40


def packed(M, n, k, w_fp32, a_kind=N.WZ_SCALE_UE8M0):
    return ("wz_fp8_gemm_packed", P, P, P, P, P, M, n, k, a_kind, N.WZ_WSCALE_F32 if w_fp32 else N.WZ_WSCALE_E8M0, P,
            BIG, None)


def fp8_rows(M, n, k, w_fp32, a_kind):
    return ("wz_fp8_gemm", P, P, P, P, P, M, n, k, a_kind, N.WZ_WSCALE_F32 if w_fp32 else N.WZ_WSCALE_E8M0, None)


def fp4_rows(M, n, k, a_kind):
    return ("wz_fp4_gemm", P, P, P, P, P, M, n, k, a_kind, None)


def tile_kernels(names):
    """(shape, weight form, power-of-two scales of a, of b, one-block slices) of each tile kernel named."""
    return {m.group(1) for n in names if (m := re.search(r"tile_gemm_kernel<(.*)>\(", n))}


def selected(tmp_path, calls):
    names, events = record(tmp_path, calls)
    got = tile_kernels(e["name"] for e in events if e["kind"] == "launch")
    assert got
    return tile_kernels(names), got


def test_every_tile_kernel_is_some_calls_choice(tmp_path):
    kinds = (N.WZ_SCALE_UE8M0, N.WZ_SCALE_F32)
    calls = []
    for M, n, k in itertools.product((17, 33, 65, 129, 300, 520, 2048), (16, 1024, 4096, 8192, 20480, 40960),
                                     (256, 1024, 4096, 8192)):
        for a in kinds:
            calls += [packed(M, n, k, w, a) for w in (False, True)] + [fp8_rows(M, n, k, w, a) for w in (False, True)]
            calls.append(fp4_rows(M, n, k, a))
    compiled, got = selected(tmp_path, calls)
    assert got == compiled, sorted(compiled - got)


F32, E8 = N.WZ_SCALE_F32, N.WZ_SCALE_UE8M0


# the choice counts on as many workgroups a CU as their LDS leaves room for.  Where float scales (or
# two K-blocks of MXFP4 a stage) leave room for one, the next larger tile took 0.57 to 0.67 of the time
@pytest.mark.parametrize("call,tile", [
    (packed(200, 4096, 8192, True, F32), "1, 2, 4, 2"), (packed(512, 2048, 12288, True, F32), "1, 2, 4, 2"),
    (fp8_rows(200, 4096, 8192, True, F32), "1, 2, 4, 2"), (fp8_rows(333, 2048, 12288, False, F32), "1, 2, 4, 2"),
    (fp4_rows(65, 4096, 8192, E8), "1, 2, 2, 2"), (fp4_rows(128, 4096, 8192, F32), "1, 2, 2, 2"),
    (fp4_rows(200, 2048, 12288, F32), "1, 2, 2, 2"),
    # two workgroups a CU fit: as before
    (packed(200, 4096, 8192, False, E8), "1, 2, 2, 2"), (fp8_rows(200, 4096, 4096, True, F32), "1, 2, 2, 2"),
    (fp4_rows(65, 4096, 2048, E8), "1, 1, 2, 2"),
])
def test_choice_counts_resident_workgroups(tmp_path, call, tile):
    _, got = selected(tmp_path, [call])
    assert [g[len("wz::TileCfg<"):].startswith(tile) for g in got] == [True], got


# (call, served by the skinny kernel): up to 32 rows of a K of up to 2048, and up to 28 of MXFP4 at any
# K, where both scales are powers of two and N / 16 workgroups fit the 256 CUs; 16 rows otherwise
@pytest.mark.parametrize("call,skinny", [
    (fp4_rows(16, 32768, 1024, F32), True), (fp4_rows(17, 2048, 4096, E8), True), (fp4_rows(28, 4096, 4096, E8), True),
    (fp4_rows(29, 4096, 4096, E8), False), (fp4_rows(17, 4112, 4096, E8), False),
    (fp4_rows(17, 2048, 4096, F32), False),
    (fp4_rows(28, 16, 12288, N.WZ_SCALE_UE8M0_F32), True), (fp4_rows(32, 4096, 2048, E8), True),
    (fp8_rows(16, 32768, 1024, True, F32), True), (fp8_rows(32, 4096, 2048, False, E8), True),
    (fp8_rows(33, 4096, 2048, False, E8), False), (fp8_rows(17, 4096, 2176, False, E8), False),
    (fp8_rows(17, 4096, 2048, True, E8), False), (fp8_rows(17, 4096, 2048, False, F32), False),
    (fp8_rows(17, 4112, 1024, False, E8), False),
])
def test_rows_of_the_skinny_kernel(tmp_path, call, skinny):
    _, events = record(tmp_path, [call])
    (name,) = [e["name"] for e in events if e["kind"] == "launch"]
    assert ("skinny_gemm_kernel" in name) == skinny, name


def test_bit_tests_reach_every_tile_kernel(tmp_path):
    """The cases that hold the tile GEMM to the narrow kernels' bits (test_gpu_tile_gemm.py)."""
    from tests.test_gpu_tile_gemm import FP4_SHAPES, PACKED_SHAPES, ROW_SHAPES, SPLITS

    calls = [fp4_rows(*s, a) for s in FP4_SHAPES for a in (E8, F32)]
    calls += [fp8_rows(*s, w, a) for s in ROW_SHAPES for a in (E8, F32) for w in (False, True)]
    calls += [packed(*s, w, a) for s in PACKED_SHAPES for a in (E8, F32) for w in (False, True)]
    compiled, got = selected(tmp_path, calls)
    assert got == compiled, sorted(compiled - got)
    # the one tile with two blocks of weight scales along N, with a split output as well
    (wide,) = [k for k in compiled if k.startswith("wz::TileCfg<8,")]
    assert wide in selected(tmp_path, [packed(M, a + b, 1024, False) for M, a, b in SPLITS])[1]
