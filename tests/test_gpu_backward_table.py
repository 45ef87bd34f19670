"""GPU: tnr_geometry_backward on synthetic lists at the edges of its table and ranges.

Lists with contiguous sources and random targets: structures at, below and
above the direct table's 2,048 atoms, a structure whose random targets
overflow the hashed table, batches with empty structures, structures more
than 64 boundaries apart, and pair counts around a round and a wave's range.
The oracle is the float64 sum of the same rows on the CPU.  Each entry may
err by the rounding of its sum: at most 128 roundings of partial sums lie on
any path (lane sums of 16 pairs, 6 steps across the lanes, 8 waves, the
workgroups that hold the atom), each within eps times the sum of absolute
values; the structures below keep every atom within 64 workgroups.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from tonari_amd._extensions import load_torch_hip

pytestmark = pytest.mark.gpu

DEV = "cuda:0"

CASES = {
    "one_pair": ([3], 1),
    "one_atom": ([1], 130),
    "round": ([700], 127),
    "two_rounds": ([700], 129),
    "direct_limit": ([2048], 20_000),
    "hashed": ([2049], 20_000),
    "overflow": ([40_000], 60_000),
    "batch": ([5, 0, 0, 40, 1, 300, 0, 2, 64, 65, 1800, 900, 0], 50_000),
    "wide_gaps": ([2] + [0] * 70 + [3] + [0] * 200 + [2] + [0] * 64 + [4], 500),
    "many": ([7] * 700, 30_000),
    "large_batch": ([3000, 10, 2500, 10], 40_000),
}


def synthetic(sizes, n_pairs, seed):
    rng = np.random.default_rng(seed)
    ptr = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    n = int(ptr[-1])
    src = np.sort(rng.integers(0, n, n_pairs))
    b = np.searchsorted(ptr, src, side="right") - 1
    lo, hi = ptr[b], ptr[b + 1]
    tgt = lo + np.floor(rng.random(n_pairs) * (hi - lo)).astype(np.int64)
    # within a structure the sources come in an order of their own
    for k in range(len(sizes)):
        at = np.flatnonzero(b == k)
        if len(at):
            perm = rng.permutation(np.arange(ptr[k], ptr[k + 1]))
            src[at] = perm[src[at] - ptr[k]]
    shifts = rng.integers(-3, 4, (n_pairs, 3)).astype(np.int32)
    return ptr, np.stack([src, tgt], 1), shifts, b


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("given", ["D", "d", "dD"])
@pytest.mark.parametrize("name", list(CASES))
def test_synthetic_lists(name, given, dtype):
    sizes, n_pairs = CASES[name]
    ptr, pairs, shifts, b = synthetic(sizes, n_pairs, 5)
    n, nb = int(ptr[-1]), len(sizes)
    g = torch.Generator().manual_seed(9)
    rand = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64).to(dtype)  # noqa: E731
    vec, gD, gd = rand(n_pairs, 3), rand(n_pairs, 3), rand(n_pairs)
    vec[:: max(2, n_pairs // 7)] = 0  # d = 0: no gradient of d
    dist = torch.linalg.vector_norm(vec.double(), dim=1).to(dtype)
    total = torch.zeros(n_pairs, 3, dtype=torch.float64)
    # sum of absolute terms: gD and k vec round (and may cancel) before they are summed
    terms = torch.zeros(n_pairs, 3, dtype=torch.float64)
    if "D" in given:
        total += gD.double()
        terms += gD.double().abs()
    if "d" in given:
        k = torch.where(dist > 0, gd / dist, torch.zeros_like(gd)).double()
        total += k[:, None] * vec.double()
        terms += (k[:, None] * vec.double()).abs()
    P, S, B = torch.as_tensor(pairs), torch.as_tensor(shifts).double(), torch.as_tensor(b)

    def sums(x, y):
        # positions and cell of rows x (targets) and y (sources), and outer products
        pos = torch.zeros(n, 3, dtype=torch.float64)
        pos.index_add_(0, P[:, 1], x)
        pos.index_add_(0, P[:, 0], y)
        return pos

    exp_pos, abs_pos = sums(total, -total), sums(terms, terms)
    cell = lambda s, x: torch.zeros(nb, 3, 3, dtype=torch.float64).index_add_(  # noqa: E731
        0, B, s[:, :, None] * x[:, None, :])
    exp_cell, abs_cell = cell(S, total), cell(S.abs(), terms)

    dev = [torch.as_tensor(x).to(DEV) for x in (ptr, pairs, shifts)]
    dvec, ddist, dgD, dgd = (x.to(DEV) for x in (vec, dist, gD, gd))
    gp = torch.zeros(n, 3, dtype=dtype, device=DEV)
    gc = torch.zeros(nb, 3, 3, dtype=dtype, device=DEV)
    err = ctypes.create_string_buffer(512)
    code = load_torch_hip().tnr_geometry_backward(
        0 if dtype == torch.float32 else 1, n_pairs, n, nb, dev[0].data_ptr(), dev[1].data_ptr(),
        dev[2].data_ptr(), dvec.data_ptr(), ddist.data_ptr(),
        dgD.data_ptr() if "D" in given else None, dgd.data_ptr() if "d" in given else None,
        gp.data_ptr(), gc.data_ptr(), torch.cuda.current_stream().cuda_stream, err, len(err))
    assert code == 0, err.value
    eps = torch.finfo(dtype).eps
    # a pair's own gradient: the division, the product and the sum round in the working precision
    for got, exp, scale in ((gp, exp_pos, abs_pos), (gc, exp_cell, abs_cell)):
        off = (got.double().cpu() - exp).abs()
        assert bool((off <= (128 + 4) * eps * scale).all()), float((off / (eps * scale + 1e-300)).max())
