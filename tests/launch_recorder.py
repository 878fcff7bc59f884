"""The library's host side without a GPU: which kernels a list of C calls launches, on a recording
stand-in for the HIP runtime (hip_recorder.c) in a process of its own.

``record(tmp, calls)`` runs ``calls`` in order and returns (names, events): the demangled names of
all kernels in the library, and per grant of dynamic LDS or launch a dict of kind ("grant" or
"launch"), device, name, bytes (of LDS), grid and block.  A call is ``("device", d)`` or
``(entry point, *arguments)``; pointers are integers that nothing dereferences, a descriptor is
its bytes, and ``("threads", [calls, calls, ...])`` runs lists of calls at once."""

import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def record(tmp, calls):
    so = os.path.join(str(tmp), "hip_recorder.so")
    if not os.path.exists(so):
        src = os.path.join(ROOT, "tests", "hip_recorder.c")
        subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-o", so, src], check=True)
    enc = json.dumps(calls, default=lambda b: {"bytes": bytes(b).hex()})
    r = subprocess.run([sys.executable, os.path.abspath(__file__), so], input=enc, capture_output=True, text=True,
                       cwd=ROOT, timeout=120)
    assert r.returncode == 0, r.stderr
    out = json.loads(r.stdout.splitlines()[-1])
    names = subprocess.run(["c++filt"], input="\n".join(out["names"]), capture_output=True, text=True,
                           check=True).stdout.splitlines()
    events = [dict(kind="launch" if k else "grant", device=d, name=names[i], bytes=b, grid=g, block=t)
              for k, d, i, b, g, t in out["events"]]
    return names, events


def _child(so):
    import ctypes
    import threading

    rec = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)  # before the library: its HIP calls bind here
    rec.rec_kernel_name.restype = ctypes.c_char_p
    sys.path.insert(0, ROOT)
    from wanferenz_amd import _native as N

    L = N.lib()

    def run(calls):
        for c in calls:
            if c[0] == "device":
                rec.rec_set_device(c[1])
            elif c[0] == "threads":
                ts = [threading.Thread(target=run, args=(part,)) for part in c[1]]
                [t.start() for t in ts]
                [t.join() for t in ts]
            else:
                args = [ctypes.create_string_buffer(bytes.fromhex(a["bytes"])) if isinstance(a, dict) else a
                        for a in c[1:]]
                N.check(getattr(L, c[0])(*args), c[0])

    run(json.loads(sys.stdin.read()))
    row = (ctypes.c_long * 6)()
    events = []
    for i in range(rec.rec_events()):
        rec.rec_event(i, row)
        events.append(list(row))
    names = [rec.rec_kernel_name(i).decode() for i in range(rec.rec_kernels())]
    print(json.dumps({"names": names, "events": events}))
    sys.stdout.flush()
    os._exit(0)  # the recorder's registrations need no teardown


if __name__ == "__main__":
    _child(sys.argv[1])
