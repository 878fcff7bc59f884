"""Which sparse attention kernel a call takes, on a recording HIP runtime."""

import pytest

from tests.launch_recorder import record

P = 1 << 20  # a 16-byte aligned stand-in for every operand: nothing is dereferenced
BIG = 1 << 40


# tiles of 16 heads in the largest group of 64 decide; heads of 128 in more than two tiles take a wave
# per tile.  From 512 groups on a query's blocks are not split and nothing is merged
@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("d", [128, 256, 512])
@pytest.mark.parametrize("h,tiles", [(16, 1), (32, 2), (48, 4), (64, 4), (80, 4), (192, 4)])
def test_kernel_of_a_shape(tmp_path, h, tiles, d, split):
    s = 3 if split else 512
    call = ("wz_sparse_attn", P, P, P, P, P, 1, s, h, d, 1000, 640, 0.1, P, BIG, None)
    _, events = record(tmp_path, [call])
    launches = [e for e in events if e["kind"] == "launch"]
    name = f"sparse_attn_wave_kernel<{d}, {str(split).lower()}>" if d == 128 and tiles == 4 else \
        f"sparse_attn_kernel<{d}, {tiles}, {str(split).lower()}>"
    assert name in launches[0]["name"]
    assert launches[0]["block"] == (256 if "wave" in name else 512)
    groups = s * ((h + 63) // 64)
    assert launches[0]["grid"] == groups * (10 if split else 1)
    assert [e["name"] for e in launches[1:]] == [e["name"] for e in launches if "combine" in e["name"]]
    assert len(launches) == (2 if split else 1)
