"""The provider's loader: checks of a built module, and threads that load together."""

from __future__ import annotations

import sys
import threading
import time
from types import SimpleNamespace

import pytest
import torch

import tonari_amd._extensions as ext


def test_device_checks_of_several_threads_take_turns(monkeypatch):
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


def test_a_stale_native_module_is_refused():
    good = {"abi_version": ext.ABI_VERSION, "torch_version": ".".join(torch.__version__.split(".")[:2])}
    ext.check_native(SimpleNamespace(**good), torch.__version__)
    for abi in (ext.ABI_VERSION - 1, ext.ABI_VERSION + 1):
        with pytest.raises(ImportError, match=f"ABI version {abi}, expected .*rebuild it"):
            ext.check_native(SimpleNamespace(**dict(good, abi_version=abi)), torch.__version__)
    with pytest.raises(ImportError, match="ABI version None"):  # built before it said so
        ext.check_native(SimpleNamespace(), torch.__version__)
    for other in ("2.9.1+rocm7.0", "3.10.0", "2.1.0"):
        with pytest.raises(ImportError, match="built with torch .* but torch .*rebuild it"):
            ext.check_native(SimpleNamespace(**good), other)


def test_the_built_native_module_passes_its_check():
    module = ext.load_torch_native()
    assert module.abi_version == ext.ABI_VERSION
    assert torch.__version__.startswith(module.torch_version + ".")


def test_the_libraries_build_without_torch(monkeypatch, capsys):
    from tonari_amd import build

    built = []
    monkeypatch.setattr(build, "_run", lambda cmd, output, verbose, what: built.append(what))
    monkeypatch.setitem(sys.modules, "torch", None)  # as if it were not installed
    build.build()
    assert built == ["libtonari_hip.so", "libtonari_cpu.so"]
    assert "not built" in capsys.readouterr().err
    monkeypatch.undo()
    monkeypatch.setattr(build, "_run", lambda cmd, output, verbose, what: built.append(what))
    build.build()
    assert built[2:] == ["libtonari_hip.so", "libtonari_cpu.so", "_tonari_torch.so"]
