"""GPU: brute force in units far from 1, against the oracle.

Inputs scaled by a power of two are the same problem until squares leave the
type's normal range.  The bounds of an image walk are products of squares of
lengths (the search radius) and of inverse lengths (the dual vectors), which
leave it first: in float32 from about 2^59 on (an inverse length squared);
the pseudo-inverse of a float64 cell compares products of four lengths (2^256),
beyond which its duals are no bound.
Cells far below 1 are refused as linearly dependent.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests._util import assert_same_keys, keys_of, oracle_call
from tonari_amd import neighbor_list

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,exponent", [
    (np.float32, e) for e in (-40, 0, 40, 58, 59, 60)] + [
    (np.float64, e) for e in (-40, 0, 300, 500, 505)])
@pytest.mark.parametrize("n,edge", [(4, 9.0), (12, 14.0), (40, 20.0)])
def test_lists_in_scaled_units(n, edge, dtype, exponent):
    rng = np.random.Generator(np.random.PCG64(n))
    scale = 2.0**exponent
    cell = (np.eye(3) + rng.uniform(-0.1, 0.1, (3, 3))) * edge
    pos = rng.uniform(0.0, 1.0, (n, 3)) @ cell
    cfg = {"positions": (pos * scale).astype(dtype), "cell": (cell * scale).astype(dtype)[None],
           "pbc": np.ones((1, 3), bool), "batch_ptr": np.array([0, n]), "cutoff": 6.0 * scale}
    expected = keys_of(*oracle_call(cfg, algorithm="brute_force"))
    t = [torch.as_tensor(cfg[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")]
    P, S = neighbor_list("PS", t[0], t[1], t[2], cfg["cutoff"], t[3], algorithm="brute_force")
    assert_same_keys(keys_of(P, S), expected)
    # the same problem at scale 1, while the squares of its lengths are normal numbers
    if abs(exponent) <= (58 if dtype == np.float32 else 500):
        one = dict(cfg, positions=(pos.astype(dtype)), cell=cell.astype(dtype)[None], cutoff=6.0)
        assert_same_keys(expected, keys_of(*oracle_call(one, algorithm="brute_force")))
