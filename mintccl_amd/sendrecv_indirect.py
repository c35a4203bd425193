"""Multi-hop LL128 send / recv with full-size staging
(``2_sendrecv_indirect.py``): every line of the message has a staging slot of
its own (``:147-149``), so no hop ever waits for a credit."""
from __future__ import annotations

from . import sendrecv_buffer as _buffered
from .common import VirtualComm, get_comm

send = _buffered.send
recv = _buffered.recv


def sync(comm: VirtualComm | None = None, route: list[int] | None = None) -> None:
    comm = comm if comm is not None else get_comm()
    matched = comm._board.sync(route, True)
    if matched is not None:
        _buffered._launch(comm, matched, full_size_staging=True)


if __name__ == "__main__":      # the reference runs its self-test from here
    import sys

    from .selftest import main
    sys.exit(main("sendrecv_indirect"))
