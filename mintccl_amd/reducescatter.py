"""Ring reduce-scatter (``7_reducescatter.py``): ``buff`` is ``(world, n)``;
after the call row r of rank r holds the sum over ranks of their row r,
accumulated in ring order starting from rank r's own value.
``MINTCCL_TOPOLOGY=hypercube`` halves recursively instead
(``mintccl_amd.hypercube``)."""
from __future__ import annotations

import torch

from . import _lib, hypercube
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_REDUCESCATTER


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, dtype, _, _, ptrs, _, _ = posted
    row = count // comm.world_size
    comm.enqueue(_lib.OP_REDUCESCATTER, dtype, row, ptrs, ptrs, ring_of(comm), row_stride=row)


@front(_KIND, _go_on)
def reducescatter(buff: torch.Tensor, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff)
    if posted is False:
        return hypercube.reducescatter(buff, comm)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("reducescatter"))
