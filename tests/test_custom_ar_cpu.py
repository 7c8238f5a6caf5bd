"""Regions of the one-shot all-reduce outlive their communicators (parallel/custom_ar.py): freed uncached memory gave
later tensors stale values on the GPU, so a closed communicator's regions are kept and handed to the next one."""
import ctypes
import subprocess
import sys

from githubrepostorag_amd.ops import _lib
from githubrepostorag_amd.parallel import custom_ar


def test_regions_are_kept_and_cleared_not_freed(monkeypatch):
    made, cleared, freed = [], [], []

    def alloc(nbytes, out):
        made.append(0x1000 * (len(made) + 1))
        ctypes.cast(out, ctypes.POINTER(ctypes.c_void_p))[0] = made[-1]
        return 0

    fake = {"grag_ar_region_bytes": lambda slot: 2 * slot + 256, "grag_ar_alloc": alloc,
            "grag_ar_clear": lambda p, n: cleared.append((p, n)) or 0, "grag_ar_free": lambda p: freed.append(p) or 0,
            "grag_ar_close_handle": lambda p: 0}
    monkeypatch.setattr(custom_ar, "_fn", fake.__getitem__)
    monkeypatch.setattr(custom_ar, "_KEPT", {})
    monkeypatch.setattr(custom_ar, "_KEY", {})
    monkeypatch.setattr(custom_ar.torch.cuda, "current_device", lambda: 0)

    def cycle(slot):
        comms = custom_ar.IpcAllReduce.simulated(2, "cpu", slot_bytes=slot)
        got = set(comms[0].regions)
        for c in comms:
            c.close()
            c.close()  # a second close gives nothing back twice
        return got

    first = cycle(1 << 20)
    assert cycle(1 << 20) == first and len(made) == 2
    assert {p for p, _ in cleared} == first and all(n == 2 * (1 << 20) + 256 for _, n in cleared)
    assert not cycle(4 << 20) & first and not freed  # another size: other regions

    exported = custom_ar.IpcAllReduce([made[0]], 0, "cpu", 1 << 20, [made[0]], [], exported=True)
    kept = {k: list(v) for k, v in custom_ar._KEPT.items()}
    exported.close()
    assert custom_ar._KEPT == kept and not freed  # a peer may still map it: kept, but not handed out again


STUBS = """
#include <stdio.h>
int hipMemset(void* p, int v, unsigned long n) { printf("memset %ld %d %lu\\n", (long)p, v, n); fflush(stdout); return 0; }
int hipDeviceSynchronize(void) { printf("wait\\n"); fflush(stdout); return 0; }
"""


def test_a_region_is_cleared_behind_what_is_in_flight(tmp_path):
    """grag_ar_clear waits for the device before it writes the zeros and after: the runtime's calls, by two stubs in their place."""
    src, so = tmp_path / "stubs.c", tmp_path / "stubs.so"
    src.write_text(STUBS)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    run = ("import ctypes; ctypes.CDLL({!r}, mode=ctypes.RTLD_GLOBAL); f = ctypes.CDLL({!r}).grag_ar_clear; "
           "f.argtypes = [ctypes.c_void_p, ctypes.c_long]; assert f(4096, 512) == 0").format(str(so), str(_lib.lib_path()))
    _lib.lib()  # (built)
    out = subprocess.run([sys.executable, "-c", run], check=True, capture_output=True, text=True, timeout=100).stdout
    assert out.split("\n") == ["wait", "memset 4096 0 512", "wait", ""]
