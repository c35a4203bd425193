"""Ring reduce-scatter (``7_reducescatter.py``): ``buff`` is ``(world, n)``;
after the call row r of rank r holds the sum over ranks of their row r,
accumulated in ring order starting from rank r's own value.
``MINTCCL_TOPOLOGY=hypercube`` halves recursively instead
(``mintccl_amd.hypercube``)."""
from __future__ import annotations

import torch

from . import _lib, hypercube
from ._ops import ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_REDUCESCATTER


def reducescatter(buff: torch.Tensor, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff)
    if posted is None:               # not all ranks are here yet, or launched
        return
    if posted is False:
        return hypercube.reducescatter(buff, comm)
    count, dtype, _, _, ptrs, _, _ = posted
    row = count // comm.world_size
    comm.enqueue(_lib.OP_REDUCESCATTER, dtype, row, ptrs, ptrs, ring_of(comm), row_stride=row)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("reducescatter"))
