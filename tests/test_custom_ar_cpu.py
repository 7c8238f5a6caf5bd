"""Regions of the one-shot all-reduce outlive their communicators (parallel/custom_ar.py): freed uncached memory gave
later tensors stale values on the GPU, so a closed communicator's regions are kept and handed to the next one."""
import ctypes

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
