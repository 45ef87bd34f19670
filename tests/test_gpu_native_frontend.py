"""GPU: the native frontend module: autograd around its node, streams, and calls without batch_ptr."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_backward import assert_close, reference_grads, small_box
from tests._util import assert_same_keys, keys_of
from tonari_amd import neighbor_list

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def inputs(seed=5, n=200, dtype=torch.float64):
    cfg = small_box(seed=seed, n=n)
    pos = torch.as_tensor(cfg["positions"]).to(DEV, dtype).requires_grad_()
    cell = torch.as_tensor(cfg["cell"]).to(DEV, dtype).requires_grad_()
    return cfg, pos, cell, torch.as_tensor(cfg["pbc"]).to(DEV), torch.as_tensor(cfg["batch_ptr"]).to(DEV)


@pytest.mark.parametrize("quantities", ["PSD", "PSd", "PSdD"])
def test_saved_tensor_hooks_and_retained_graphs(quantities):
    cfg, pos, cell, pbc, ptr = inputs()
    with torch.autograd.graph.save_on_cpu():
        out = dict(zip(quantities, neighbor_list(quantities, pos, cell, pbc, cfg["cutoff"], ptr)))
    wD = torch.ones_like(out["D"]) * 0.5 if "D" in out else None
    wd = torch.linspace(-1, 1, len(out["P"]), dtype=pos.dtype, device=DEV) if "d" in out else None
    loss = sum((w * out[q]).sum() for q, w in (("D", wD), ("d", wd)) if w is not None)
    exp = reference_grads(pos, cell, ptr, out["P"], out["S"], wD, wd)
    for _ in range(2):
        got = torch.autograd.grad(loss, (pos, cell), retain_graph=True)
        for g, e in zip(got, exp):
            assert_close(g, e, torch.float64)


def test_only_one_output_has_a_gradient():
    cfg, pos, cell, pbc, ptr = inputs(seed=8)
    P, S, d, D = neighbor_list("PSdD", pos, cell, pbc, cfg["cutoff"], ptr)
    for wD, wd in ((torch.ones_like(D), None), (None, torch.ones_like(d))):
        loss = (wD * D).sum() if wD is not None else (wd * d).sum()
        exp = reference_grads(pos, cell, ptr, P, S, wD, wd)
        for create in (False, True):
            got = torch.autograd.grad(loss, (pos, cell), retain_graph=True, create_graph=create)
            for g, e in zip(got, exp):
                assert_close(g, e, torch.float64)
    with torch.no_grad():
        assert not neighbor_list("D", pos, cell, pbc, cfg["cutoff"], ptr)[0].requires_grad
    assert not neighbor_list("PS", pos, cell, pbc, cfg["cutoff"], ptr)[0].requires_grad


def test_without_batch_ptr_on_a_side_stream():
    cfg, pos, cell, pbc, ptr = inputs(seed=9, n=120)
    expected = keys_of(*neighbor_list("PS", pos, cell, pbc, cfg["cutoff"], ptr))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(3):
            P, S, D = neighbor_list("PSD", pos, cell[0], pbc[0], cfg["cutoff"])
            gp, gc = torch.autograd.grad(D.sum(), (pos, cell))
            stream.synchronize()
            assert_same_keys(keys_of(P, S), expected)
            rp, rc = reference_grads(pos, cell, ptr, P, S, torch.ones_like(D), None)
            assert_close(gp, rp, torch.float64)
            assert_close(gc, rc, torch.float64)


@pytest.mark.parametrize("n", [0, 1])
def test_smallest_structures_without_batch_ptr(n):
    pos = torch.zeros((n, 3), device=DEV, requires_grad=True)
    cell, pbc = torch.eye(3, device=DEV) * 3, torch.ones(3, dtype=torch.bool, device=DEV)
    for _ in range(2):
        P, S, D = neighbor_list("PSD", pos, cell, pbc, 3.5)
        assert P.shape == (6 * n, 2) and S.shape == (6 * n, 3) and D.shape == (6 * n, 3)
        (g,) = torch.autograd.grad(D.sum(), pos)
        assert g.shape == (n, 3) and float(g.abs().sum()) == 0.0


def test_errors_keep_their_types():
    cfg, pos, cell, pbc, ptr = inputs(seed=10, n=50)
    bad = pos.detach().clone()
    bad[3, 1] = float("nan")
    for _ in range(2):
        with pytest.raises(RuntimeError, match="positions must contain only finite values"):
            neighbor_list("PS", bad, cell, pbc, cfg["cutoff"], ptr)
        with pytest.raises(ValueError, match="batch_ptr must end at N_total"):
            neighbor_list("PS", pos, cell, pbc, cfg["cutoff"], ptr - torch.tensor([0, 1], device=DEV))
    assert np.isfinite(float(neighbor_list("d", pos, cell, pbc, cfg["cutoff"], ptr)[0].detach().sum()))


def test_gradients_are_independent_tensors():
    cfg, pos, cell, pbc, ptr = inputs(seed=11)
    (D,) = neighbor_list("D", pos, cell, pbc, cfg["cutoff"], ptr)
    (D * D).sum().backward()
    gp, gc = pos.grad, cell.grad
    assert gp.shape == pos.shape and gc.shape == cell.shape
    assert gp.is_contiguous() and gc.is_contiguous()
    before = gc.clone()
    w = torch.ones((), dtype=gc.dtype, device=DEV, requires_grad=True)
    y = (gc * w).sum()  # saves gc
    gp.mul_(2.0)
    y.backward()
    assert torch.equal(gc, before) and float((w.grad - before.sum()).abs()) == 0.0


def test_gradients_own_their_storage():
    cfg, pos, cell, pbc, ptr = inputs(seed=12, n=301, dtype=torch.float32)
    (D,) = neighbor_list("D", pos, cell, pbc, cfg["cutoff"], ptr)
    (D * D).sum().backward()
    for g in (pos.grad, cell.grad):
        assert g.untyped_storage().nbytes() == g.numel() * g.element_size()
        assert g.data_ptr() % 256 == 0  # as a fresh allocation
    kept = cell.grad.clone()
    pos.grad.untyped_storage().resize_(0)
    assert torch.equal(cell.grad, kept)
