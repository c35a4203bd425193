"""Multi-hop LL128 send / recv through fixed circular staging
(``3_sendrecv_buffer.py``).

``send`` and ``recv`` only record their arguments (``:78-92``); ``sync``,
called by every rank (``:98``), matches them, picks the route and enqueues one
launch in which every rank on the route runs its hop.
"""
from __future__ import annotations

import torch

from . import _lib
from ._ops import front
from .common import VirtualComm, get_comm
from .protocol import packed_bytes


@front(_lib.SEND)
def send(buff: torch.Tensor, peer: int, comm: VirtualComm | None = None) -> None:
    (comm if comm is not None else get_comm())._board.send(buff, peer)


@front(_lib.RECV)
def recv(buff: torch.Tensor, peer: int, comm: VirtualComm | None = None) -> None:
    (comm if comm is not None else get_comm())._board.recv(buff, peer)


def _launch(comm: VirtualComm, matched: tuple, full_size_staging: bool = False) -> None:
    src, dst, sptr, dptr, count, route, _ = matched
    args = (_lib.OP_SENDRECV, _lib.BYTES, count, {src: sptr}, {dst: dptr}, route)
    if not full_size_staging:
        comm.enqueue(*args, route_len=len(route))
        return
    # every line of the message gets a slot of its own, so no hop ever waits for
    # a credit (2_sendrecv_indirect.py:147-149); zeroed like the reference's, and
    # kept alive until the next transfer replaces it, since the launch is
    # asynchronous
    d = comm.make_op(*args, route_len=len(route))
    slot = d.slot_bytes
    d.nslots = max(1, -(-packed_bytes(count) // slot))
    per_rank = d.nslots * slot + max(4096, slot // 4) + _lib.TICKET_BYTES
    hops = torch.zeros(comm.world_size * per_rank, dtype=torch.uint8, device=comm.device)
    comm._indirect_staging = hops
    for k in range(comm.world_size):
        d.staging[k] = hops.data_ptr() + k * per_rank
    d.staging_bytes = per_rank
    d.credit_offset = 0                      # right after this staging's own slots
    comm.launch(d)


@front(_lib.SYNC, _launch)
def sync(comm: VirtualComm | None = None, route: list[int] | None = None) -> None:
    """Every rank calls this; the first call that finds a matched send / recv
    pair launches, the others find nothing left to do."""
    comm = comm if comm is not None else get_comm()
    matched = comm._board.sync(route, False)
    if matched is not None:                  # (not launched by the board)
        _launch(comm, matched)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("sendrecv_buffer"))
