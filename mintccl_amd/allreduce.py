"""Ring allreduce: the collective the reference lists as planned
(``8_allreduce.py``, ``README.md:23,49``), built from the pieces of
``7_reducescatter.py`` and ``6_allgather.py``: the buffer is cut into
``world`` chunks of whole 16-byte vectors (the last ones may be short or
empty); chunk c is summed round the ring starting from rank c's own value
(the reduce-scatter order of ``7_reducescatter.py:54-73``) and the finished sum
is handed round until every rank has stored it.  In place; after the call all
ranks hold the same bits.

Two ways to run it, same result bit for bit:

* fused (``fused=True`` or ``MINTCCL_ALLREDUCE=fused``; the default where the
  rings run inside compute units, else below 32 MiB per rank): one launch, one pass round the ring of 2 * world - 1
  positions - what the reference plans.  Its two phases share the staging
  slots and the wavefronts.
* split (``fused=False`` or ``MINTCCL_ALLREDUCE=split``; the default of the
  rings through staging from 32 MiB per rank): a reduce-scatter launch followed by an allgather launch on
  the same chunks; each launch can use the whole wavefront budget, and the
  allgather's origins get compute units of their own.
"""
from __future__ import annotations

import torch

from . import _lib
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_ALLREDUCE


# Through staging, two launches are faster than one pass from this size per rank
# on (measured on MI355X, 8 ranks, f16: 104 / 110 us at 16 MiB, 199 / 192 at 32 MiB, 1510 /
# 1384 at 256 MiB; below, the second launch costs more than it gains: 12 / 18 us
# at 64 KiB).  Inside compute units the two phases share nothing: one pass is
# 161 us at 64 MiB of bf16 where two launches through staging take 368.
SPLIT_FROM_BYTES = 32 << 20


def chunk_bytes(count: int, world: int) -> int:
    """Bytes of one chunk: ceil(count / world) rounded up to whole 16-byte vectors."""
    return (-(-count // world) + 15) // 16 * 16


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, dtype, _, variant, ptrs, _, _ = posted
    fused = count < SPLIT_FROM_BYTES or comm._runs_inside() if variant < 0 else bool(variant)
    ring = ring_of(comm)
    if fused:
        comm.enqueue(_lib.OP_ALLREDUCE, dtype, count, ptrs, ptrs, ring)
        return
    row = chunk_bytes(count, comm.world_size)
    comm.enqueue(_lib.OP_REDUCESCATTER, dtype, row, ptrs, ptrs, ring, row_stride=row,
                 total_bytes=count)
    comm.enqueue(_lib.OP_ALLGATHER, _lib.BYTES, row, ptrs, ptrs, ring, row_stride=row,
                 total_bytes=count)


@front(_KIND, _go_on)
def allreduce(buff: torch.Tensor, comm: VirtualComm | None = None,
              fused: bool | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, 0, fused)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("allreduce"))
