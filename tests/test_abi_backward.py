"""The C ABI of the backward without a GPU: layout, and requests refused before a launch."""

from __future__ import annotations

import ctypes

import pytest

from tonari_amd import _extensions as ext
from tests.test_abi import _request, lib  # noqa: F401

PTR = 1 << 20  # never dereferenced: every call here returns before a launch


def _backward(**kw):
    base = dict(dtype=0, n_pairs=5, n_atoms=4, n_structures=1, batch_ptr=PTR, pairs=PTR, shifts=PTR,
                vectors=PTR, distances=PTR, grad_vectors=PTR, grad_distances=PTR,
                grad_positions=PTR, grad_cell=PTR, source_runs=None)
    base.update(kw)
    return ext.Backward(**base)


def test_struct_layout_matches_header():
    assert ctypes.sizeof(ext.Backward) == 112
    assert ext.Backward.n_pairs.offset == 8 and ext.Backward.batch_ptr.offset == 32
    assert ext.Backward.grad_positions.offset == 88 and ext.Backward.source_runs.offset == 104


def _call(f, req):
    err = ctypes.create_string_buffer(256)
    code = f(req if req is None else ctypes.byref(req), None, err, len(err))
    return code, err.value.decode()


@pytest.mark.parametrize("name", ["tnr_backward_list", "tnr_zero_gradients"])
def test_refused_requests(lib, name):  # noqa: F811
    f = getattr(lib, name)
    bad = [(None, "request is null"), (_backward(dtype=2), "dtype must be float32 or float64"),
           (_backward(n_atoms=-1), "invalid sizes"), (_backward(n_structures=0), "invalid sizes"),
           (_backward(grad_positions=None), "required pointers are null"),
           (_backward(grad_cell=None), "required pointers are null")]
    if name == "tnr_backward_list":
        bad += [(_backward(n_pairs=-1), "invalid sizes"),
                (_backward(pairs=None), "required pointers are null"),
                (_backward(distances=None), "the gradient of d needs the distances and vectors"),
                (_backward(vectors=None), "the gradient of d needs the distances and vectors")]
    for req, message in bad:
        assert _call(f, req) == (ext.TNR_INPUT_ERROR, message)


def test_nothing_to_add(lib):  # noqa: F811
    # no pairs, or no upstream gradient: accepted without a launch
    assert _call(lib.tnr_backward_list, _backward(n_pairs=0, pairs=None))[0] == ext.TNR_OK
    assert _call(lib.tnr_backward_list,
                 _backward(grad_vectors=None, grad_distances=None))[0] == ext.TNR_OK


def test_source_runs_refused(lib):  # noqa: F811
    err = ctypes.create_string_buffer(256)
    req = _request()
    need = lib.tnr_workspace_size(ctypes.byref(req))
    for workspace, size, runs in ((PTR, need - 1, PTR), (None, need, PTR), (PTR, need, None)):
        assert lib.tnr_source_runs(ctypes.byref(req), workspace, size, runs, None, err,
                                   len(err)) == ext.TNR_INPUT_ERROR
    empty = _request(n_atoms=0)
    assert lib.tnr_source_runs(ctypes.byref(empty), PTR, lib.tnr_workspace_size(ctypes.byref(empty)),
                               None, None, err, len(err)) == ext.TNR_OK
