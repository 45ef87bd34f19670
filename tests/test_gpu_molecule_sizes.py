"""GPU: molecules at the edges of the molecule passes, against the oracle.

Atom counts around a chunk of 64 targets, a register pass of 8 chunks and the
largest molecule (2,048 atoms), one source per unit and many, lists longer
than the emitting pass's LDS list (a source with more than 1,792 targets),
and enough molecules that a wave's share of the units crosses structures.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests._util import assert_geometry_close, assert_same_keys, keys_of, oracle_call
from tonari_amd import neighbor_list

pytestmark = pytest.mark.gpu

SIZES = {
    "chunks": [1, 2, 63, 64, 65, 127, 128, 129, 0, 3],
    "passes": [511, 512, 513, 575, 577],
    "largest": [2047, 2048],
    "long_lists": [2048, 1800, 5],
    "shares": [40 + 7 * (k % 13) for k in range(1500)],
    "large_shares": [300 + 37 * (k % 11) for k in range(60)],
}


def molecules(name, dtype, seed):
    rng = np.random.default_rng(seed)
    sizes = SIZES[name]
    # "long_lists": every atom within the cutoff of every other
    radius = (lambda n: 1.0) if name == "long_lists" else (lambda n: (n / 0.1) ** (1 / 3))
    pos = [rng.uniform(0.0, radius(n), (n, 3)) for n in sizes]
    return {
        "positions": np.concatenate(pos).astype(dtype),
        "cell": np.zeros((len(sizes), 3, 3), dtype),
        "pbc": np.zeros((len(sizes), 3), bool),
        "batch_ptr": np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64),
        "cutoff": 4.0 if name != "large_shares" else 3.0,
    }


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("half_list,include_self", [(False, False), (True, True)])
@pytest.mark.parametrize("name", list(SIZES))
def test_sizes(name, half_list, include_self, dtype):
    cfg = dict(molecules(name, dtype, 3), half_list=half_list, include_self=include_self)
    expected = keys_of(*oracle_call(cfg, algorithm="brute_force"))
    t = {k: torch.as_tensor(cfg[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
    for _ in range(2):  # the full prologue, then the molecule one
        P, S, D = neighbor_list("PSD", t["positions"], t["cell"], t["pbc"], cfg["cutoff"],
                                t["batch_ptr"], half_list=half_list, include_self=include_self)
        torch.cuda.synchronize()
        assert_same_keys(keys_of(P, S), expected)
        assert_geometry_close(P, S, None, D, cfg)
        # by source, then target
        flat = P[:, 0] * len(cfg["positions"]) + P[:, 1]
        assert bool((flat[1:] > flat[:-1]).all())
