"""Ring reduce (``5_reduce.py``): elementwise sum in ring order, in place at
the root; the other ranks' buffers are left as they were.
``MINTCCL_TOPOLOGY=tree`` adds up a binary tree instead (``mintccl_amd.tree``)."""
from __future__ import annotations

import torch

from . import _lib, tree
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_REDUCE


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, dtype, root, _, ptrs, _, _ = posted
    # inputbuff on every rank, outputbuff only at the root (5_reduce.py:117-118)
    comm.enqueue(_lib.OP_REDUCE, dtype, count, ptrs, {root: ptrs[root]}, ring_of(comm), root=root)


@front(_KIND, _go_on)
def reduce(buff: torch.Tensor, root: int, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, root)
    if posted is False:
        return tree.reduce(buff, root, comm)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("reduce"))
