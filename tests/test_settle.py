"""What a repeated call reserves: outputs, bins and hit-mask words follow the counts of a shape."""

from __future__ import annotations

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


@pytest.mark.gpu
def test_alternating_batches_emit_once():
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
        # the list fits what was reserved before the call
        assert call < 2 or reserved[0] >= P.shape[0], (call, reserved, P.shape)
