"""Alltoall (the reference plans it as ``9_alltoall.py``, ``README.md:24,50``):
``buff`` and ``out`` are ``(world, n)``; after the call row ``s`` of rank
``d``'s ``out`` holds row ``d`` of rank ``s``'s ``buff`` - the transpose of the
ranks' buffers, MPI_Alltoall.  Every row travels straight to its destination
through the destination's staging slots as LL128 lines (or with the Simple
protocol): ``world x world`` pipelines of two positions in one fused launch.
``out`` must not overlap any rank's ``buff``: every row is read while others
are being written."""
from __future__ import annotations

import torch

from . import _lib
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_ALLTOALL


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, _, _, _, ins, outs, _ = posted
    row = count // comm.world_size
    comm.enqueue(_lib.OP_ALLTOALL, _lib.BYTES, row, ins, outs, ring_of(comm), row_stride=row)


@front(_KIND, _go_on)
def alltoall(buff: torch.Tensor, out: torch.Tensor, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, 0, None, out)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("alltoall"))
