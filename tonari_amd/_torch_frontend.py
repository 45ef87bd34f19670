"""PyTorch frontend of ``neighbor_list``.

Restates the reference frontend (``src/tonari/_torch_frontend.py``): the same
single-structure normalisation (``:25-48``), validation and messages
(``:51-75``), detached contiguous arguments (``:128-137``) and quantity order
(``:78-105``).  The native call goes to the HIP C ABI instead of the pybind11
CUDA provider (``:138-145``); i/j/P/S/d/D are written by the emit kernel
instead of being assembled with Torch gathers.

When ``d`` or ``D`` is requested and ``positions`` or ``cell`` requires
gradients, the kernel's d/D carry autograd to both through a fused backward
kernel, the gradient of the reference's Torch expression.  The calls into the
C ABI, the allocations and the autograd node are native
(``csrc/torch/frontend.cpp``); what a shape's next call reserves is kept here.

CPU tensors go to this build's host provider (``_cpu_provider``), and i/j/d/D
are assembled from its P and S as the reference does (``:78-105``).
"""

from __future__ import annotations

import threading
from math import isfinite

import torch
from torch import Tensor

from . import _cpu_provider
from ._extensions import (
    ALGORITHMS,
    HOST_RESULT_SLOTS,
    TNR_INPUT_ERROR,
    TNR_OK,
    check_device,
    load_torch_native,
)


def _require_torch_tensors(*, cell: object, pbc: object, batch_ptr: object | None) -> None:
    for name, tensor in (("cell", cell), ("pbc", pbc), ("batch_ptr", batch_ptr)):
        if tensor is not None and not isinstance(tensor, Tensor):
            raise TypeError(
                "positions, cell, pbc, and batch_ptr must all be PyTorch tensors; "
                f"{name} has type {type(tensor).__name__}"
            )


def normalize_torch_inputs(
    positions: Tensor, cell: Tensor, pbc: Tensor, batch_ptr: Tensor | None
) -> tuple[Tensor, Tensor, Tensor, Tensor]:
    if positions.ndim != 2 or positions.shape[1] != 3:
        raise ValueError("positions must have shape (N_total, 3)")
    if batch_ptr is None:
        if cell.ndim != 2 or cell.shape != (3, 3):
            raise ValueError("single-structure cell must have shape (3, 3)")
        if pbc.ndim != 1 or pbc.shape != (3,):
            raise ValueError("single-structure pbc must have shape (3,)")
        n = positions.shape[0]
        if positions.is_cuda and n > 0:
            # written by a kernel: a copy from the host would wait for the stream
            batch_ptr = torch.arange(0, n + 1, n, dtype=torch.int64, device=positions.device)
        else:
            batch_ptr = torch.tensor([0, n], dtype=torch.int64, device=positions.device)
        cell = cell.unsqueeze(0)
        pbc = pbc.unsqueeze(0)
    else:
        if cell.ndim != 3:
            raise ValueError("batched cell must have shape (B, 3, 3)")
        if pbc.ndim != 2:
            raise ValueError("batched pbc must have shape (B, 3)")
    return positions, cell, pbc, batch_ptr


def validate_torch_inputs(
    positions: Tensor, cell: Tensor, pbc: Tensor, cutoff: float, batch_ptr: Tensor
) -> None:
    if positions.device.type not in ("cpu", "cuda"):
        raise ValueError("positions must be a CPU or CUDA tensor")
    if positions.dtype not in (torch.float32, torch.float64):
        raise ValueError("positions must have dtype float32 or float64")
    if batch_ptr.ndim != 1 or batch_ptr.numel() == 0 or batch_ptr.dtype != torch.int64:
        raise ValueError("batch_ptr must be int64 with shape (B + 1,)")
    if cell.shape != (batch_ptr.numel() - 1, 3, 3):
        raise ValueError("cell must have shape (B, 3, 3)")
    if cell.dtype != positions.dtype:
        raise ValueError("cell and positions must have the same dtype")
    if pbc.shape != (batch_ptr.numel() - 1, 3) or pbc.dtype != torch.bool:
        raise ValueError("pbc must be bool with shape (B, 3)")
    if any(tensor.device != positions.device for tensor in (cell, pbc, batch_ptr)):
        raise ValueError("positions, cell, pbc, and batch_ptr must be on the same device")
    if not isfinite(cutoff) or cutoff <= 0:
        raise ValueError("cutoff must be finite and positive")


def _torch_geometry(positions: Tensor, cell: Tensor, batch_ptr: Tensor, pairs: Tensor,
                    shifts: Tensor) -> Tensor:
    """The reference's Torch expression for D (``_torch_frontend.py:92-101``)."""
    source = pairs[:, 0].contiguous()
    target = pairs[:, 1].contiguous()
    pair_batch = torch.bucketize(source, batch_ptr[1:], right=True)
    return positions[target] - positions[source] + torch.einsum(
        "ei,eij->ej", shifts.to(positions.dtype), cell[pair_batch]
    )


_HOST = threading.local()


def _host_result(device: torch.device):
    """Pinned status words of this thread for `device`, an event, and their addresses.

    The count writes its status words into the buffer on the stream; the
    event, recorded right after, tells when they have arrived.  One buffer
    per thread and device is reused across calls (a fresh pinned allocation
    per call costs more than the search of a small structure).
    """
    cache = getattr(_HOST, "buffers", None)
    if cache is None:
        cache = _HOST.buffers = {}
    entry = cache.get(device)
    if entry is None:
        host = torch.empty(HOST_RESULT_SLOTS, dtype=torch.int64, pin_memory=True)
        event = torch.cuda.Event()
        event.record(torch.cuda.current_stream(device))  # the handle exists from the first record
        entry = cache[device] = (host, event, host.data_ptr(), event.cuda_event)
    return entry


def _speculation() -> dict:
    """This thread's last (output capacity, plan, bins, hit-mask words) per request shape."""
    table = getattr(_HOST, "speculation", None)
    if table is None:
        table = _HOST.speculation = {}
    return table


# Output capacity of the next call of a shape: the last pair count plus
# 1/32 and a constant, which covers the drift of a molecular-dynamics step.
def _capacity(n_pairs: int) -> int:
    return n_pairs + (n_pairs >> 5) + 4096


# Hit-mask words per atom of the next call's workspace: the longest row the
# last count wanted (host_result[5]) plus one for the drift of the densest
# bin; a bin that outgrows it takes the slow path, with the same results.
def _mask_words(need: int) -> int:
    return min(need + 1, 64) if need > 0 else 1


_FITTED, _MISSED, _NO_MEMORY = 1, 2, 3  # what became of the rows a call reserved


# What the next call of a shape reserves, given what the last one reserved
# (old) and what its count asks for (new): never less than asked for, and
# falling by a 64th of the difference per call, so that batches of one shape
# whose counts differ by more than the margin keep fitting when they take
# turns (the margin of 1/32 covers the fall of a call; rows: for counts up to
# 1.5 times apart, see below).  Two alternating float64 slab batches took the writing pass
# again on every second call, and the slow path of stencils beyond their
# hit-mask rows.
def _settle(old: int, new: int) -> int:
    return max(new, old - ((old - new + 63) >> 6))


# Output rows: at most half more than the call asks for, so that results kept
# alive stay near their size when a shape's counts fall for good.  Counts
# further apart that take turns write the larger list twice.
def _settle_rows(old: int, new: int) -> int:
    return min(_settle(old, new), new + (new >> 1))


# The cell-list bins a launch covers have no margin: the larger count is kept
# (surplus workgroups leave at once) until it is more than twice what a call
# asks for.
def _settle_bins(old: int, new: int) -> int:
    return max(old, new) if old <= 2 * new else new


_ROWS = {
    "P": ((2,), torch.int64),
    "S": ((3,), torch.int32),
    "i": ((), torch.int64),
    "j": ((), torch.int64),
}


# Internal quantity of the native search: the edge-first index (2, E) of the
# graph adapter.
EDGE_INDEX = "E"


def _allocate(want: set, rows: int, dtype: torch.dtype, device: torch.device) -> dict:
    out = {}
    for q in ("P", "S", "i", "j", "d", "D"):
        if q not in want:
            continue
        if q in _ROWS:
            tail, qdtype = _ROWS[q]
        else:
            tail, qdtype = ((3,) if q == "D" else ()), dtype
        out[q] = torch.empty((rows, *tail), dtype=qdtype, device=device)
    return out


def _rows(out: dict, count: int) -> dict:
    """The first `count` rows of each output."""
    return {q: t[:count] for q, t in out.items()}


# A list in index order whose structures come from a cell list is summed by
# its sources' runs in binned order from this many pairs on: the kernels gain
# from 0.3 M pairs (float32 d, one box: 23 + 4 against 32 us; 28 + 4 against 76
# at 1.1 M, 203 + 4 against 561 at 9 M), but the call pays the runs' allocation
# and launch (155 against 162 us at 0.5 M, 168 against 187 at 1.1 M).
# Structures of up to 2,048 atoms have a table without hashing, and pairs in
# index order serve those better (100 structures of 1,000 atoms, 9 M pairs: 531
# us, 561 by runs; 50 of 2,000: 449 and 438).
_RUN_PAIRS = 1 << 20
_RUN_ATOMS = 2048


def _run_atoms(n_structures: int) -> int:
    """Atoms beyond which a request may be summed by runs: 1,536 per structure, 2,048 in all."""
    return max(_RUN_ATOMS, _RUN_ATOMS * 3 // 4 * n_structures)


def _raise(code: int, message: str) -> None:
    if code == TNR_INPUT_ERROR:
        raise ValueError(message)
    raise RuntimeError(message)


def neighbor_list_hip(
    quantities: str,
    positions: Tensor,
    batch_ptr: Tensor,
    cell: Tensor,
    pbc: Tensor,
    cutoff: float,
    *,
    half_list: bool,
    include_self: bool,
    algorithm: str,
    sorted: bool,
    grad_positions: Tensor | None = None,
    grad_cell: Tensor | None = None,
) -> tuple[Tensor, ...]:
    """Run count + emit on the tensors' HIP device; returns one tensor per quantity.

    The first call of a request shape (device, dtype, sizes, pair policy,
    algorithm, quantities) counts, waits for the pair count E and writes
    outputs of exactly E rows, as the reference does.  A repeated call of
    the same shape launches the writing pass right behind the count, into
    outputs sized from the previous calls' counts plus a margin, and waits
    only for the count: when E fits (and the plan and bins match the
    launch) the results are the first E rows of those outputs; otherwise,
    or where memory does not hold those outputs, the writing pass runs with
    exact sizes.  Either way the returned values are the same; a repeated
    call's tensors may be views of allocations of up to half more rows.
    """
    device = positions.device
    try:
        native = load_torch_native()
        check_device(device.index if device.index is not None else torch.cuda.current_device())
    except ImportError as error:
        raise RuntimeError(f"the CUDA provider is unavailable: {error}") from error
    if positions.shape[0] >= 2**31:
        raise ValueError("the current implementation supports fewer than 2^31 atoms")
    if grad_positions is None:
        grad_positions = positions
    if grad_cell is None:
        grad_cell = cell
    need_grad = (
        ("d" in quantities or "D" in quantities)
        and (grad_positions.requires_grad or grad_cell.requires_grad)
        and torch.is_grad_enabled()
    )
    # the cutoff is part of the shape: a call at another cutoff takes the
    # plain count -> emit path instead of a speculative emit sized for the
    # old one (the cell is not: it drifts a little on every step of NPT
    # dynamics, and a miss only re-runs the emit)
    key = (device, positions.dtype, positions.shape[0], batch_ptr.numel() - 1, half_list,
           include_self, algorithm, cutoff, frozenset(quantities), need_grad)
    table = _speculation()
    guess = table.get(key)
    _, _, host, event = _host_result(device)
    code, message, tensors, (count, plan, bins, mask_need), reserved = native.search(
        quantities, grad_positions, grad_cell, pbc, batch_ptr, cutoff, ALGORITHMS[algorithm],
        sorted, half_list, include_self, need_grad, guess, host, event, _RUN_PAIRS,
        _run_atoms(batch_ptr.numel() - 1),
    )
    if code != TNR_OK:
        _raise(code, message)
    entry = (_capacity(count), plan, bins, _mask_words(mask_need))
    if guess is not None and reserved != _NO_MEMORY:
        entry = (_settle_rows(guess[0], entry[0]), plan, _settle_bins(guess[2], bins),
                 _settle(guess[3], entry[3]))
    table[key] = entry
    return tuple(tensors)


def _select_torch_quantities(quantities: str, positions: Tensor, cell: Tensor,
                             batch_ptr: Tensor, pairs: Tensor, shifts: Tensor) -> tuple[Tensor, ...]:
    """i/j/P/S/d/D from the CPU provider's P and S, as the reference assembles them
    (``_torch_frontend.py:78-105``): D and d by the Torch expression, so they
    carry autograd to positions and cell."""
    values: dict[str, Tensor] = {"P": pairs, "S": shifts}
    if "i" in quantities:
        values["i"] = pairs[:, 0].contiguous()
    if "j" in quantities:
        values["j"] = pairs[:, 1].contiguous()
    if "D" in quantities or "d" in quantities:
        values["D"] = _torch_geometry(positions, cell, batch_ptr, pairs, shifts)
        if "d" in quantities:
            values["d"] = torch.linalg.vector_norm(values["D"], dim=1)
    return tuple(values[q] for q in quantities)


def _neighbor_list_cpu(quantities: str, positions: Tensor, cell: Tensor, pbc: Tensor,
                       cutoff: float, batch_ptr: Tensor, *, algorithm: str,
                       cpu_threads: int | None, half_list: bool,
                       include_self: bool) -> tuple[Tensor, ...]:
    """CPU tensors: the host provider (``_cpu_provider``) on ``cpu_threads``
    threads (1 by default), replacing the reference's ``_torch_cpu`` module
    (``_torch_frontend.py:147-156``).  Sources come in index order."""
    pos = positions.detach().contiguous()
    cel = cell.detach().contiguous()
    bp = batch_ptr.contiguous()
    flags = pbc.contiguous()  # bool: one byte per entry, 0 or 1

    def allocate(n_pairs: int):
        pairs = torch.empty((n_pairs, 2), dtype=torch.int64)
        shifts = torch.empty((n_pairs, 3), dtype=torch.int32)
        return pairs, shifts, pairs.data_ptr(), shifts.data_ptr()

    try:
        pairs, shifts = _cpu_provider.search(
            pos.dtype == torch.float64, pos.data_ptr() if pos.numel() else None, pos.shape[0],
            bp.data_ptr(), bp.numel() - 1, cel.data_ptr() if cel.numel() else None,
            flags.data_ptr() if flags.numel() else None, cutoff, half_list, include_self,
            algorithm, 1 if cpu_threads is None else cpu_threads, allocate,
        )
    except ImportError as error:
        raise RuntimeError(f"the Torch CPU provider is unavailable: {error}") from error
    return _select_torch_quantities(quantities, positions, cell, batch_ptr, pairs, shifts)


def neighbor_list_torch(
    quantities: str,
    positions: Tensor,
    cell: Tensor,
    pbc: Tensor,
    cutoff: float,
    batch_ptr: Tensor | None,
    *,
    algorithm: str,
    cpu_threads: int | None,
    sorted: bool,
    half_list: bool,
    include_self: bool,
) -> tuple[Tensor, ...]:
    _require_torch_tensors(cell=cell, pbc=pbc, batch_ptr=batch_ptr)
    positions, cell, pbc, batch_ptr = normalize_torch_inputs(positions, cell, pbc, batch_ptr)
    cutoff = float(cutoff)
    validate_torch_inputs(positions, cell, pbc, cutoff, batch_ptr)
    if not positions.is_cuda:
        return _neighbor_list_cpu(
            quantities, positions, cell, pbc, cutoff, batch_ptr, algorithm=algorithm,
            cpu_threads=cpu_threads, half_list=half_list, include_self=include_self,
        )
    if cpu_threads is not None:
        raise ValueError("cpu_threads only applies to CPU inputs")
    return neighbor_list_hip(
        quantities,
        positions,
        batch_ptr,
        cell,
        pbc,
        cutoff,
        half_list=half_list,
        include_self=include_self,
        algorithm=algorithm,
        sorted=sorted,
    )
