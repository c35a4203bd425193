"""Ring allgather (``6_allgather.py``): ``buff`` is ``(world, n)``; rank r
contributes row r and ends up with every rank's row, in place.

The reference has two kernels that leave the same bytes.  *Spatial*
(``6_allgather.py:79-138``): every source rank's row has its own blocks and
its own share of the staging - the default here, it is the faster one.
*Temporal* (``:25-77``, the one the reference's host function launches): the
whole grid moves rank 0's row round the ring, then rank 1's, and so on,
through staging for one row - ``schedule="temporal"`` or
``MINTCCL_ALLGATHER=temporal`` (LL128 only).  ``MINTCCL_TOPOLOGY=hypercube``
doubles recursively over a hypercube instead (``mintccl_amd.hypercube``)."""
from __future__ import annotations

import torch

from . import _lib, hypercube
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_ALLGATHER


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, _, _, temporal, ptrs, _, _ = posted
    row = count // comm.world_size
    if temporal:
        comm.launch(comm.make_op(_lib.OP_ALLGATHER_TEMPORAL, _lib.BYTES, row, ptrs, ptrs,
                                 ring_of(comm), row_stride=row, protocol=_lib.PROTO_LL128))
    else:
        comm.enqueue(_lib.OP_ALLGATHER, _lib.BYTES, row, ptrs, ptrs, ring_of(comm), row_stride=row)


@front(_KIND, _go_on)
def allgather(buff: torch.Tensor, comm: VirtualComm | None = None,
              schedule: str | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, 0, schedule)
    if posted is False:
        return hypercube.allgather(buff, comm)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("allgather"))
