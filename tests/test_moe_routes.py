"""Which routed tiles a prefill takes (prefill_tile_rows), on a recording HIP runtime."""

import ctypes

import pytest

from tests.launch_recorder import record
from tests.test_abi import _desc
from wanferenz_amd import _native as N

P = 1 << 20  # a stand-in for every operand: nothing is dereferenced
BIG = 1 << 40


def moe_desc(D=4096, I=2048, E=256, k=6, act=N.WZ_SCALE_UE8M0):
    d = _desc(D, I, E, k)
    d.act_scale_kind = act
    for name in ("w13p", "w13p_s", "w2p", "w2p_s", "sh13p", "sh2p", "sh_w1_s", "sh_w3_s", "sh_w2_s"):
        setattr(d, name, P)
    return ctypes.string_at(ctypes.byref(d), ctypes.sizeof(d))


# (layer, tokens, wide): from 1024 tokens, 32 rows an expert (48 where I < 2048) and 256 workgroups
# of w1/w3 on; float activation scales keep the 64-row tiles
@pytest.mark.parametrize("layer,T,wide", [
    (dict(), 1023, False), (dict(), 1365, False), (dict(), 1366, True), (dict(), 6000, True),
    (dict(E=4, k=2), 1023, False), (dict(E=4, k=2), 1024, True), (dict(act=N.WZ_SCALE_F32), 6000, False),
    (dict(D=5120, I=1536, E=160), 1279, False), (dict(D=5120, I=1536, E=160), 1280, True),
    (dict(D=2048, I=512, k=8), 1535, False), (dict(D=2048, I=512, k=8), 1536, True),
    (dict(D=4096, I=1024, E=96, k=1), 4096, False), (dict(D=4096, I=1024, E=96, k=1), 4608, True),
    (dict(D=1024, I=512, E=8, k=2), 3583, False), (dict(D=1024, I=512, E=8, k=2), 3584, True),
    (dict(D=512, I=256, E=16, k=2), 7167, False), (dict(D=512, I=256, E=16, k=2), 7168, True),
])
def test_wide_routed_tiles(tmp_path, layer, T, wide):
    _, events = record(tmp_path, [("wz_moe_forward", moe_desc(**layer), P, None, T, P, None, None, P, BIG, None)])
    names = [e["name"] for e in events if e["kind"] == "launch"]
    assert sum("prefill_wide_kernel" in n for n in names) == (2 if wide else 0), names
    assert sum("prefill_gemm_kernel" in n for n in names) == 2, names


def test_wide_cases_take_wide_tiles(tmp_path):
    """The cases that hold the wide tiles to the 64-row tiles' bits (test_gpu_moe_chunks.py) launch
    them, and their reference calls of 700 tokens do not."""
    from tests.test_gpu_moe_chunks import WIDE, WIDE_CASES

    for E, T, _ in WIDE_CASES:
        layer = moe_desc(WIDE["dim"], WIDE["inter"], E, WIDE["topk"])
        for n, wide in ((T, True), (700, False), (T % 700, False)):
            _, events = record(tmp_path, [("wz_moe_forward", layer, P, None, n, P, None, None, P, BIG, None)])
            assert any("prefill_wide_kernel" in e["name"] for e in events) == wide, (E, n)
