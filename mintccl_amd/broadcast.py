"""Ring broadcast (``4_broadcast.py``): after the call every rank's ``buff``
holds the root's bytes.  ``MINTCCL_TOPOLOGY=tree`` sends them down a binary tree
instead (``mintccl_amd.tree``)."""
from __future__ import annotations

import torch

from . import _lib, tree
from ._ops import front, ring_of
from .common import VirtualComm, get_comm

_KIND = _lib.KIND_BROADCAST


def _go_on(comm: VirtualComm, posted: tuple) -> None:
    """All ranks are here, and it is not the board's to launch."""
    count, _, root, _, ptrs, _, _ = posted
    # root has the input, everyone else an output (4_broadcast.py:97-98)
    comm.enqueue(_lib.OP_BROADCAST, _lib.BYTES, count, {root: ptrs[root]},
                 {r: p for r, p in ptrs.items() if r != root}, ring_of(comm), root=root)


@front(_KIND, _go_on)
def broadcast(buff: torch.Tensor, root: int, comm: VirtualComm | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    posted = comm._post(_KIND, buff, root)
    if posted is False:
        return tree.broadcast(buff, root, comm)
    if posted is not None:           # (None: not all ranks are here yet, or launched)
        _go_on(comm, posted)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("broadcast"))
