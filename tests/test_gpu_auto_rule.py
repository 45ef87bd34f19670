"""GPU: algorithm='auto' at its lines, and the periodic brute-force walk on awkward cells, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests._util import assert_geometry_close, assert_same_keys, keys_of, oracle_call
from tonari_amd import neighbor_list
from tonari_amd import workloads as W
from tonari_amd._torch_frontend import _speculation

pytestmark = pytest.mark.gpu

BRUTE, CELL = 1, 2


def call(cfg, algorithm="auto", **kw):
    t = {k: torch.as_tensor(cfg[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
    _speculation().clear()
    for _ in range(2):
        P, S, D = neighbor_list("PSD", t["positions"], t["cell"], t["pbc"], cfg["cutoff"],
                                t["batch_ptr"], algorithm=algorithm, **kw)
        torch.cuda.synchronize()
        assert_same_keys(keys_of(P, S), keys_of(*oracle_call(dict(cfg, **kw), algorithm=algorithm)))
        assert_geometry_close(P, S, None, D, cfg)
    (entry,) = _speculation().values()
    return entry[1] & 3


def boxes(n, count, pbc=(True, True, True), dtype=np.float32, seed=0):
    rng = np.random.default_rng(seed)
    edge = (n / 0.05) ** (1 / 3)
    return {
        "positions": rng.uniform(0, edge, (n * count, 3)).astype(dtype),
        "cell": np.tile(np.eye(3) * edge, (count, 1, 1)).astype(dtype),
        "pbc": np.tile(np.array(pbc), (count, 1)),
        "batch_ptr": np.arange(0, n * count + 1, n, dtype=np.int64),
        "cutoff": float(0.9 * edge / 2),  # one image each way
    }


# atoms x 27 images around 1,500 and 2,700 (requests beyond 6,144 atoms) and
# 6,000 (up to it); slabs and wires by atoms x images up to 1,500, and as if
# fully periodic beyond
@pytest.mark.parametrize(
    "n,count,pbc,plan",
    [
        (55, 2, (1, 1, 1), BRUTE), (56, 2, (1, 1, 1), BRUTE),
        (222, 2, (1, 1, 1), BRUTE), (223, 2, (1, 1, 1), CELL),
        (100, 62, (1, 1, 1), BRUTE), (101, 61, (1, 1, 1), CELL),
        (222, 27, (1, 1, 1), BRUTE), (222, 28, (1, 1, 1), CELL),
        (166, 40, (1, 1, 0), BRUTE), (167, 40, (1, 1, 0), CELL), (222, 3, (1, 0, 1), BRUTE),
        (223, 3, (1, 0, 1), CELL), (500, 2, (0, 1, 0), BRUTE), (501, 2, (0, 1, 0), CELL),
    ],
)
def test_auto_lines(n, count, pbc, plan):
    cfg = boxes(n, count, tuple(bool(x) for x in pbc), seed=n)
    cfg["cutoff"] = min(cfg["cutoff"], 3.0)
    assert call(cfg) == plan


# beyond 16,384 atoms the line of 2,700 holds up to 2.5 + 110,000 / atoms iterations of
# the walk per atom (8 + ... with more than 27 images): 13.3 for 96 atoms at 0.9
# edges, 3.81 at 0.45, 2.54 for 64; 4.5 for 21 atoms at 1.1 edges (brute force took up
# to 1.7 times the cell list's time for 1,365 structures of 96 atoms)
@pytest.mark.parametrize("n,count,edges,plan", [
    (96, 170, 0.9, BRUTE), (96, 171, 0.9, CELL), (96, 860, 0.45, BRUTE), (96, 900, 0.45, CELL),
    (64, 1024, 0.45, BRUTE), (21, 900, 1.1, BRUTE), (101, 200, 0.3, CELL), (55, 400, 0.9, BRUTE),
])
def test_auto_line_of_large_requests(n, count, edges, plan):
    cfg = boxes(n, count, seed=n)
    t = {k: torch.as_tensor(cfg[k]).to("cuda:0") for k in ("positions", "cell", "pbc", "batch_ptr")}
    cutoff = float(edges * (n / 0.05) ** (1 / 3))
    call_ = lambda a: neighbor_list("PS", t["positions"], t["cell"], t["pbc"], cutoff,  # noqa: E731
                                    t["batch_ptr"], algorithm=a)
    other = call_("brute_force" if plan == CELL else "cell_list")
    _speculation().clear()
    for _ in range(2):
        P, S = call_("auto")
        assert P.shape == other[0].shape
        assert torch.equal(torch.bincount(P[:, 0]), torch.bincount(other[0][:, 0]))
        assert torch.equal(torch.bincount(P[:, 1]), torch.bincount(other[0][:, 1]))
        assert torch.equal(S.sum(0), other[1].sum(0))
    (entry,) = _speculation().values()
    assert entry[1] & 3 == plan


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("half_list,include_self", [(False, False), (True, True)])
def test_brute_walk_on_awkward_cells(dtype, half_list, include_self):
    # sheared cells (many rows per plane), needles and plates, open axes with
    # far coordinates, atoms outside the cell, one-atom structures, and more
    # pairs than one round of a unit
    rng = np.random.default_rng(7)
    shapes = [
        (W.triclinic_cell((4.0, 5.0, 6.0), (62.0, 118.0, 65.0)), (1, 1, 1), 9),
        (W.triclinic_cell((3.0, 3.2, 30.0), (80.0, 85.0, 61.0)), (1, 1, 1), 20),
        (W.triclinic_cell((25.0, 2.5, 20.0), (100.0, 75.0, 110.0)), (1, 1, 1), 70),
        (np.array([[6.0, 0, 0], [5.5, 6.0, 0], [-5.0, 5.5, 6.0]]), (1, 1, 1), 12),
        (W.triclinic_cell((7.0, 8.0, 9.0), (75.0, 100.0, 95.0)), (1, 0, 1), 40),
        (W.triclinic_cell((7.0, 8.0, 9.0), (75.0, 100.0, 95.0)), (0, 0, 1), 15),
        (np.eye(3) * 3.0, (1, 1, 1), 1),
        (np.eye(3) * 40.0, (1, 1, 1), 130),
    ]
    positions, cells, pbc, sizes = [], [], [], []
    for cell, periodic, n in shapes:
        frac = rng.uniform(-2.0, 2.0, (n, 3))
        frac[:, np.array(periodic) == 0] *= 3.0
        positions.append(frac @ cell if n < 100 else rng.uniform(0, 12.0, (n, 3)))
        cells.append(cell)
        pbc.append(np.array(periodic, bool))
        sizes.append(n)
    cfg = {
        "positions": np.concatenate(positions).astype(dtype),
        "cell": np.stack(cells).astype(dtype),
        "pbc": np.stack(pbc),
        "batch_ptr": np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64),
        "cutoff": 6.5,
    }
    assert call(cfg, "brute_force", half_list=half_list, include_self=include_self) == BRUTE
