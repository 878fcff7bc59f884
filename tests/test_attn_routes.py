"""Which sparse attention kernels a call takes, on a recording HIP runtime."""

import pytest

from tests.launch_recorder import record

P = 1 << 20  # a 16-byte aligned stand-in for every operand: nothing is dereferenced
BIG = 1 << 40


def _launches(tmp_path, s, h, d):
    _, events = record(tmp_path, [("wz_sparse_attn", P, P, P, P, P, 1, s, h, d, 1000, 640, 0.1, P, BIG, None)])
    return [(e["name"].split("(")[0].split("wz::")[1], e["grid"], e["block"]) for e in events if e["kind"] == "launch"]


# ten blocks of 64 indices, one workgroup each: 3 queries are split and merged
@pytest.mark.parametrize("d", [128, 256, 512])
@pytest.mark.parametrize("h,tiles", [(16, 1), (32, 2), (48, 4), (64, 4), (80, 4), (96, 4), (112, 4), (192, 4)])
def test_split_queries(tmp_path, h, tiles, d):
    groups = 3 * ((h + 63) // 64)
    wave = tiles == 4 and d <= 256
    main = (f"sparse_attn_wave_kernel<{d}, true>", groups * 10, 256) if wave else \
        (f"sparse_attn_kernel<{d}, {tiles}, true>", groups * 10, 512)
    assert _launches(tmp_path, 3, h, d) == [main, (f"sparse_attn_combine_kernel<{d}>", groups * 16, 256)]


# from 512 groups on a workgroup takes all of a query's blocks; a last group of one or two tiles
# has a launch of its own
@pytest.mark.parametrize("d", [128, 256, 512])
@pytest.mark.parametrize("h,parts", [(16, [(1, 1)]), (32, [(2, 1)]), (48, [(4, 1)]), (64, [(4, 1)]),
                                     (80, [(4, 1), (1, 1)]), (96, [(4, 1), (2, 1)]), (112, [(4, 2)]),
                                     (144, [(4, 2), (1, 1)]), (192, [(4, 3)])])
def test_unsplit_queries(tmp_path, h, parts, d):
    want = [(f"sparse_attn_kernel<{d}, {tiles}, false>", 512 * groups, 512) for tiles, groups in parts]
    if d == 128 and h > 32:
        want = [(f"sparse_attn_wave_kernel<{d}, false>", 512 * ((h + 63) // 64), 256)]
    assert _launches(tmp_path, 512, h, d) == want
