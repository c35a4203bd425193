"""Ring reduce (``5_reduce.py``): elementwise sum in ring order, in place at
the root; the other ranks' buffers are left as they were.
``MINTCCL_TOPOLOGY=tree`` adds up a binary tree instead (``mintccl_amd.tree``)."""
from __future__ import annotations

import torch

from . import _lib, tree
from ._ops import ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_REDUCE


def reduce(buff: torch.Tensor, root: int, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, root)
    if posted is None:               # not all ranks are here yet, or launched
        return
    if posted is False:
        return tree.reduce(buff, root, comm)
    count, dtype, root, _, ptrs, _, _ = posted
    # inputbuff on every rank, outputbuff only at the root (5_reduce.py:117-118)
    comm.enqueue(_lib.OP_REDUCE, dtype, count, ptrs, {root: ptrs[root]}, ring_of(comm), root=root)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("reduce"))
