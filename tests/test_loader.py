"""The provider's loader: checks of a built module, and threads that load together."""

from __future__ import annotations

import threading
import time
from types import SimpleNamespace

import tonari_amd._extensions as ext


def test_device_checks_of_several_threads_take_turns(monkeypatch):
    import torch

    inside, most = 0, 0

    def properties(index):
        nonlocal inside, most
        inside += 1
        most = max(most, inside)
        time.sleep(0.02)
        inside -= 1
        return SimpleNamespace(gcnArchName="gfx950:sramecc+")

    monkeypatch.setattr(torch.cuda, "get_device_properties", properties)
    monkeypatch.setattr(ext, "load_torch_hip",
                        lambda: SimpleNamespace(tnr_device_arch=lambda: b"gfx950"))
    threads = [threading.Thread(target=ext.check_device.__wrapped__, args=(0,)) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert most == 1
