"""What a repeated call reserves: outputs, bins and hit-mask words follow the counts of a shape."""

from __future__ import annotations

import gc
from types import SimpleNamespace

import pytest
import torch

import tonari_amd._torch_frontend as F
from tests._util import assert_same_keys, keys_of, oracle_call
from tonari_amd import neighbor_list
from tonari_amd import workloads as W


def test_settle_rule():
    assert F._settle(100, 100) == 100
    assert F._settle(100, 250) == 250  # never less than asked for
    old, steps = 1_000_000, 0
    while old > 8:
        new = F._settle(old, 8)
        assert 8 <= new < old
        old, steps = new, steps + 1
    assert steps < 800
    # the rows' margin covers the fall of a call, for counts up to half apart
    for big, small in ((15 * 10**8, 10**9), (5000, 4000), (10**6, 9 * 10**5)):
        assert F._settle_rows(F._capacity(big), F._capacity(small)) >= big
    assert F._settle_rows(F._capacity(10**9), F._capacity(10**6)) <= 1.5 * F._capacity(10**6)
    assert F._settle_bins(4096, 3000) == 4096 and F._settle_bins(3000, 4096) == 4096
    assert F._settle_bins(4096, 2000) == 2000 and F._settle_bins(64, 0) == 0


def test_run_rule():
    # a batch whose structures mostly fit the backward's direct table is not summed by runs
    assert F._run_atoms(1) == 2048
    assert 100 * 1000 <= F._run_atoms(100) < 100 * 2000


@pytest.fixture
def fates(monkeypatch):
    """What became of the rows each native search reserved, in order."""
    native, seen = F.load_torch_native(), []

    def search(*args):
        answer = native.search(*args)
        seen.append(answer[4])
        return answer

    monkeypatch.setattr(F, "load_torch_native", lambda: SimpleNamespace(search=search))
    F._speculation().clear()
    return seen


def _calls(boxes, calls, quantities="PS"):
    out = []
    for call in range(calls):
        c = boxes[call % len(boxes)]
        t = {k: torch.as_tensor(c[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
        out.append(neighbor_list(quantities, t["positions"], t["cell"], t["pbc"], c["cutoff"],
                                 t["batch_ptr"], algorithm="cell_list")[0])
    return out


@pytest.mark.gpu
def test_alternating_batches_emit_once(fates):
    # one shape, two densities: once both were seen, every call's writing pass fits
    boxes = [W.c4(seed=31 + k, n_atoms=6000, density=d) for k, d in enumerate((0.06, 0.09))]
    tensors = [{k: torch.as_tensor(c[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
               for c in boxes]
    expected = [keys_of(*oracle_call(c, algorithm="cell_list")) for c in boxes]
    F._speculation().clear()
    for call in range(8):
        c, t = boxes[call % 2], tensors[call % 2]
        reserved = [v[0] for v in F._speculation().values()]
        P, S = neighbor_list("PS", t["positions"], t["cell"], t["pbc"], c["cutoff"],
                             t["batch_ptr"], algorithm="cell_list")
        torch.cuda.synchronize()
        assert_same_keys(keys_of(P, S), expected[call % 2])
        # the list fits what was reserved before the call, and was written once
        assert call < 2 or reserved[0] >= P.shape[0], (call, reserved, P.shape)
        assert call < 2 or fates[-1] == F._FITTED, (call, fates)


@pytest.mark.gpu
def test_counts_far_apart_write_the_larger_list_again(fates):
    # beyond the 1.5 that a call reserves at most over its own count
    boxes = [W.c4(seed=31 + k, n_atoms=6000, density=d) for k, d in enumerate((0.055, 0.095))]
    _calls(boxes, 6)
    assert fates[2:] == [F._FITTED, F._MISSED, F._FITTED, F._MISSED], fates


@pytest.mark.gpu
def test_reserved_rows_beyond_the_memory_limit(fates):
    # the list fits the limit, the half more that the earlier call left reserved does not
    dense, sparse = (W.c4(seed=41, n_atoms=400_000, density=d) for d in (0.15, 0.1))
    q, row, slack = "PSDij", 56, 500 << 20  # the slack holds the workspace
    _calls([dense], 1, q)
    E = _calls([sparse], 1, q)[0].shape[0]
    (rows,) = [v[0] for v in F._speculation().values()]
    assert rows > 1.4 * E
    t = {k: torch.as_tensor(sparse[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties("cuda:0").total_memory
    held = torch.cuda.memory_reserved()  # with the free parts of segments in use
    limit = held + row * E + slack
    assert row * rows > row * E + slack + (held - torch.cuda.memory_allocated())
    try:
        torch.cuda.set_per_process_memory_fraction(limit / total)
        for call in range(2):
            out = neighbor_list(q, t["positions"], t["cell"], t["pbc"], sparse["cutoff"],
                                t["batch_ptr"], algorithm="cell_list")
            assert all(x.shape[0] == E for x in out)
            del out
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    # after the call without memory the rows are sized from the count alone
    assert fates[-2:] == [F._NO_MEMORY, F._FITTED], fates
