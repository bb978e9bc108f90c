"""The engine's host buffers for copies, without a device: a result belongs to the thread that asked
for it."""
import threading
import time

import torch

from omoknuni_quantum_amd.core import engine
from omoknuni_quantum_amd.core.engine import WaveEngine


class _SlowStream:
    """A stream whose waits take long enough for another thread to start its copies."""

    def synchronize(self):
        time.sleep(0.1)


def test_downloads_of_several_threads(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: _SlowStream())
    empty = torch.empty
    monkeypatch.setattr(engine.torch, "empty",
                        lambda *a, pin_memory=False, **k: empty(*a, **k))  # (no device to pin for)
    eng = WaveEngine.__new__(WaveEngine)
    eng.device = torch.device("cpu")
    eng._init_staging()
    got = {}

    def read(i):
        got[i] = eng._download(sampled=torch.full((6,), i, dtype=torch.int32))[0].tolist()

    threads = [threading.Thread(target=read, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got == {i: [i] * 6 for i in range(3)}
