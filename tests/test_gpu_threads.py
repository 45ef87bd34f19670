"""GPU: concurrent Python callers on their own streams, and the loader's device check.

The library keeps no mutable state between calls (each call has its own
workspace; the frontend keeps its pinned status buffer and repeated-call
table per thread), and the frontend's native module runs without the GIL, so
calls from several threads overlap on the device.  After the reference's
``tests/backends/test_cpu_threads.py:160-215``: every thread's results must
equal the CPU oracle's.
"""

from __future__ import annotations

import threading
import time
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

from tests._util import assert_same_keys, keys_of, oracle_call
from tonari_amd import neighbor_list
from tonari_amd import workloads as W

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _cases():
    return {
        "batch": dict(W.c2(n_structures=40), algorithm="auto"),
        "box": W.c4(seed=31, n_atoms=12_000),
        "half": dict(W.c3(n_structures=64), sorted=True),
    }


def _call(cfg, t):
    return neighbor_list(
        "PS", t["positions"], t["cell"], t["pbc"], cfg["cutoff"], t["batch_ptr"],
        algorithm=cfg["algorithm"], half_list=cfg.get("half_list", False),
        include_self=cfg.get("include_self", False), sorted=cfg.get("sorted", False),
    )


def test_concurrent_calls_on_separate_streams():
    cases = _cases()
    expected = {name: keys_of(*oracle_call(cfg)) for name, cfg in cases.items()}
    tensors = {name: {k: torch.as_tensor(cfg[k]).to(DEV)
                      for k in ("positions", "cell", "pbc", "batch_ptr")}
               for name, cfg in cases.items()}
    torch.cuda.synchronize()

    def run(job):
        name, rep = job
        stream = torch.cuda.Stream(device=DEV)  # default priority
        # the inputs were written on the default stream, synchronised above
        with torch.cuda.stream(stream):
            results = []
            for _ in range(rep):
                P, S = _call(cases[name], tensors[name])
                results.append((P, S))
            stream.synchronize()
            return name, [keys_of(P, S) for P, S in results]

    jobs = [(name, 3) for name in cases] * 3
    print(f"[threads] {len(jobs)} jobs on 4 threads", flush=True)
    with ThreadPoolExecutor(max_workers=4) as pool:
        outcomes = list(pool.map(run, jobs))
    for name, keys in outcomes:
        for k in keys:
            assert_same_keys(k, expected[name])


def test_a_waiting_allocation_leaves_other_threads_running():
    # The call's allocations find the process's memory limit reached by a block that another
    # stream's pool holds, so the allocator frees that block, which waits for the device.
    cfg = W.c4(seed=5, n_atoms=60_000)
    t = {k: torch.as_tensor(cfg[k]).to(DEV) for k in ("positions", "cell", "pbc", "batch_ptr")}
    expected = _call(cfg, t)[0].shape[0]
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    start.record()
    torch.cuda._sleep(10_000_000)
    end.record()
    torch.cuda.synchronize()
    cycles = int(10_000_000 * 600.0 / start.elapsed_time(end))  # 0.6 s
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    limit = torch.cuda.memory_reserved(DEV) + (1 << 30)
    ticks, stop = [time.perf_counter()], threading.Event()

    def tick():
        while not stop.wait(0.002):
            ticks.append(time.perf_counter())

    try:
        torch.cuda.set_per_process_memory_fraction(limit / total, DEV)
        with torch.cuda.stream(torch.cuda.Stream(device=DEV)):
            del_me = torch.empty((1 << 30) - (4 << 20), dtype=torch.uint8, device=DEV)
        del del_me
        thread = threading.Thread(target=tick)
        thread.start()
        torch.cuda._sleep(cycles)
        P, _ = _call(cfg, t)
        stop.set()
        thread.join()
    finally:
        stop.set()
        torch.cuda.set_per_process_memory_fraction(1.0, DEV)
    gap = max(b - a for a, b in zip(ticks, ticks[1:]))
    print(f"[threads] {len(ticks)} ticks, longest gap {1000 * gap:.0f} ms", flush=True)
    assert P.shape[0] == expected
    assert ticks[-1] - ticks[0] > 0.3  # the call waited for the device
    assert gap < 0.2


def test_device_check_accepts_this_device_and_names_a_mismatch(monkeypatch):
    from tonari_amd import _extensions as ext

    ext.check_device(0)  # the box's device runs the library's target

    class Fake:
        def tnr_device_arch(self):
            return b"gfx942"

    monkeypatch.setattr(ext, "load_torch_hip", lambda: Fake())
    with pytest.raises(ImportError, match="holds gfx942 code only; device cuda:0 is gfx950"):
        ext.check_device.__wrapped__(0)
