"""Dynamic LDS past 64 KB is granted to a kernel on the device that launches it
(hipFuncSetAttribute acts on the current device's function), before the launch, with several
devices and threads in one process.  On a recording HIP runtime: no GPU."""

import ctypes

from tests.launch_recorder import record
from tests.test_abi import _desc
from wanferenz_amd import _native as N

P = 1 << 20  # a 16-byte aligned stand-in for every operand: nothing is dereferenced
BIG = 1 << 40


def _moe_desc():
    d = _desc()
    for name in ("w13p", "w13p_s", "w2p", "w2p_s", "sh13p", "sh2p", "sh_w1_s", "sh_w3_s", "sh_w2_s"):
        setattr(d, name, P)
    return bytes(ctypes.string_at(ctypes.byref(d), ctypes.sizeof(d)))


# one call of each family whose dynamic LDS can pass 64 KB: tile GEMM on row-major FP8 and MXFP4
# and on packed weights, the one-tile GEMV of 16 rows, the fused norm GEMV, the wide MoE tiles
CALLS = [
    ("wz_fp8_gemm", P, P, P, P, P, 100, 4096, 4096, N.WZ_SCALE_F32, N.WZ_WSCALE_F32, None),
    ("wz_fp4_gemm", P, P, P, P, P, 333, 2048, 4096, N.WZ_SCALE_UE8M0, None),
    ("wz_fp8_gemm_packed", P, P, P, P, P, 300, 32656, 1024, N.WZ_SCALE_UE8M0, N.WZ_WSCALE_E8M0, P, BIG, None),
    ("wz_fp8_linear_packed", P, P, P, P, 16, 4096, 8192, N.WZ_SCALE_UE8M0_F32, N.WZ_WSCALE_E8M0, P, BIG, None),
    ("wz_moe_forward", _moe_desc(), P, None, 2048, P, None, None, P, BIG, None),
]


def _check(events, devices):
    granted = {}
    big = set()
    for e in events:
        key = (e["device"], e["name"])
        if e["kind"] == "grant":
            # the attribute is what the last call set: it never shrinks below an earlier launch's need
            assert e["bytes"] >= granted.get(key, 0), e
            granted[key] = e["bytes"]
        elif e["bytes"] > 64 * 1024:
            assert granted.get(key, 0) >= e["bytes"], f"no grant for {e}"
            big.add(key)
    for d in devices:
        assert len({n for dev, n in big if dev == d}) >= 5, sorted(big)


def test_each_device_is_granted(tmp_path):
    _, events = record(tmp_path, [("device", 0), *CALLS, ("device", 3), *CALLS, ("device", 0), *CALLS])
    _check(events, (0, 3))
    grants = [e for e in events if e["kind"] == "grant"]
    assert len(grants) == len({(e["device"], e["name"], e["bytes"]) for e in grants}), "granted once a device"


def test_threads_on_two_devices(tmp_path):
    # shapes of one kernel whose LDS grows and shrinks with K
    ks = [4096, 7168, 1024, 12288, 2048, 8192]
    calls = [("wz_fp8_gemm", P, P, P, P, P, 64, 4096, k, N.WZ_SCALE_UE8M0, N.WZ_WSCALE_E8M0, None) for k in ks * 20]
    lists = [[("device", t % 2)] + CALLS + calls[t:] for t in range(8)]
    _, events = record(tmp_path, [("threads", lists)])
    _check(events, (0, 1))
