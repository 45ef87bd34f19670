"""GPU: the backward over the sources' runs (sorted cell-list lists) against float64 autograd.

The frontend takes it from 2**20 pairs, 2,049 atoms and 1,537 per structure on; the small cases
lower both limits.  Sources without pairs, batches with empty structures,
wrapped atoms, all pair modes, tables of both kinds, and one list above the
limits.  Tolerances are those of tests/test_gpu_backward.py (1e-10 and 1e-4
of the largest gradient).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import tonari_amd._torch_frontend as F
from tests.test_gpu_backward import assert_close, fused_grads, small_box
from tonari_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture
def runs(monkeypatch):
    monkeypatch.setattr(F, "_RUN_PAIRS", 1)
    monkeypatch.setattr(F, "_RUN_ATOMS", 0)


def sparse_box(n):
    # most sources without pairs
    cfg = W.c4(seed=n, n_atoms=n, density=0.002)
    return dict(cfg, cutoff=3.0)


def slabs(sizes, seed):
    parts = [W.c5(seed=seed + k, n_structures=1, n_min=n, n_max=n) for k, n in enumerate(sizes) if n]
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    cells, pbc, it = [], [], iter(parts)
    for n in sizes:
        p = next(it) if n else parts[0]
        cells.append(p["cell"][0])
        pbc.append(p["pbc"][0])
    return {"positions": np.concatenate([p["positions"] for p in parts]), "cell": np.stack(cells),
            "pbc": np.stack(pbc), "batch_ptr": ptr, "cutoff": 5.0}


CASES = {
    "wrapped_box": lambda: small_box(seed=17, n=500),
    "sparse": lambda: sparse_box(900),
    "hashed": lambda: W.c4(seed=3, n_atoms=5000),
    "slabs": lambda: slabs([700, 0, 2300, 1, 65, 0], 5),
}


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("half_list,include_self", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("name", list(CASES))
def test_runs(runs, name, half_list, include_self, dtype):
    quantities = {(False, False): "dD", (True, False): "D", (False, True): "d"}[half_list, include_self]
    (gp, gc), (rp, rc) = fused_grads(CASES[name](), quantities, dtype, 7, algorithm="cell_list",
                                     sorted=True, half_list=half_list, include_self=include_self)
    assert_close(gp, rp, dtype)
    assert_close(gc, rc, dtype)


def test_other_lists_with_the_limits_lowered(runs):
    cfg = small_box(seed=19, n=300)
    for kw in ({"algorithm": "cell_list"}, {"algorithm": "brute_force", "sorted": True}):
        (gp, gc), (rp, rc) = fused_grads(cfg, "D", torch.float64, 7, **kw)
        assert_close(gp, rp, torch.float64)
        assert_close(gc, rc, torch.float64)


def test_list_above_the_limits():
    assert F._RUN_PAIRS <= 13_000 * 85 and F._RUN_ATOMS < 13_000
    (gp, gc), (rp, rc) = fused_grads(W.c4(seed=9, n_atoms=13_000), "d", torch.float64, 7,
                                     algorithm="cell_list", sorted=True)
    assert_close(gp, rp, torch.float64)
    assert_close(gc, rc, torch.float64)
