"""Rings inside compute units (what the operators run when nothing about the
wire is named): rows around every edge of the walk - less than a lane's 16
bytes, around one 1 KiB block, around the rounds of four steps, one channel
more or less than a grid holds, around the size from which the copying
collectives move 4 KiB per step - bit for bit against the oracle."""
import numpy as np
import pytest
import torch

from oracle import ring
from tests.helpers import as_bytes, rank_rows

pytestmark = pytest.mark.gpu

# bytes of a row (even: whole f16 values)
ROWS = [2, 14, 16, 18, 1022, 1024, 1026, 3 * 1024, 4 * 1024 + 2, 64 * 1024 - 2, 65 * 1024 + 16,
        5 * 64 * 1024 + 1040, 7 * 64 * 1024 - 6]


def make_comm(world, **kw):
    from mintccl_amd.common import VirtualComm
    comm = VirtualComm(world_size=world, spin_budget=400000, **kw)
    assert comm.inside_cu
    return comm


@pytest.mark.parametrize("world,dt", [(8, "f16"), (8, "bf16"), (8, "f32"), (3, "f16"), (2, "bf16")])
def test_reducing_rows(dev, world, dt):
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.reduce import reduce
    from mintccl_amd.reducescatter import reducescatter
    size = 4 if dt == "f32" else 2
    comm = make_comm(world)
    for i, nbytes in enumerate(ROWS):
        n = max(1, nbytes // size)
        host = rank_rows(world, n, dt, seed0=50 * i)
        raw = [as_bytes(h) for h in host]
        for what, run, want in (
                ("reducescatter", lambda b: comm.run(lambda r: reducescatter(b[r], comm)),
                 ring.reducescatter(raw, dt)),
                ("reduce", lambda b: comm.run(lambda r: reduce(b[r], world - 1, comm)),
                 ring.reduce(raw, world - 1, dt)),
                ("allreduce", lambda b: comm.run(lambda r: allreduce(b[r].view(-1), comm)),
                 ring.allreduce(raw, dt)),
                ("allreduce split", lambda b: comm.run(lambda r: allreduce(b[r].view(-1), comm, fused=False)),
                 ring.allreduce(raw, dt))):
            bufs = [h.to(dev) for h in host]
            run(bufs)
            comm.check()
            for r in range(world):
                assert ring.same_values(as_bytes(bufs[r]), want[r], dt), (what, n, r)


@pytest.mark.parametrize("world", [2, 3, 8])
@pytest.mark.parametrize("nbytes", ROWS + [4 << 20, (4 << 20) - 1, (4 << 20) + 4097, (9 << 20) + 5 * 1024 + 3])
def test_copying_rows(dev, world, nbytes):
    from mintccl_amd import sendrecv_buffer
    from mintccl_amd.allgather import allgather
    from mintccl_amd.alltoall import alltoall
    from mintccl_amd.broadcast import broadcast
    comm = make_comm(world)
    g = torch.Generator().manual_seed(nbytes)
    host = [torch.randint(0, 256, (world, nbytes), dtype=torch.uint8, generator=g) for _ in range(world)]
    bufs = [h.to(dev) for h in host]
    outs = [torch.zeros_like(b) for b in bufs]
    comm.run(lambda r: alltoall(bufs[r], outs[r], comm))
    route = [0] + list(range(2, world)) + [1]                 # over every other rank
    dst = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
    with comm.rank(0):
        sendrecv_buffer.send(bufs[0][0], 1, comm)
    with comm.rank(1):
        sendrecv_buffer.recv(dst, 0, comm)
    comm.run(lambda r: sendrecv_buffer.sync(comm, route=route))
    comm.run(lambda r: allgather(bufs[r], comm))
    flat = [h[r].to(dev) for r, h in enumerate(host)]
    comm.run(lambda r: broadcast(flat[r], world - 1, comm))
    comm.check()
    assert torch.equal(dst.cpu(), host[0][0])
    gathered = torch.stack([host[r][r] for r in range(world)])
    for r in range(world):
        assert torch.equal(outs[r].cpu(), torch.stack([host[q][r] for q in range(world)])), r
        assert torch.equal(bufs[r].cpu(), gathered), r
        assert torch.equal(flat[r].cpu(), host[world - 1][world - 1]), r


@pytest.mark.parametrize("shift", [1, 3, 8])
def test_rows_at_any_byte_touch_nothing_else(dev, shift):
    from mintccl_amd import _lib
    from mintccl_amd.broadcast import broadcast
    world, n = 8, 3001
    comm = make_comm(world)
    host = rank_rows(world, n, "f16", seed0=900)
    backing = [torch.full((world * n * 2 + 32,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(world)]
    want = ring.reducescatter([as_bytes(h) for h in host], "f16")
    for r in range(world):
        backing[r][shift: shift + world * n * 2] = torch.from_numpy(as_bytes(host[r])).to(dev)
    # (torch has no f16 view at an odd byte: through the descriptor)
    ptrs = {r: backing[r].data_ptr() + shift for r in range(world)}
    comm.enqueue(_lib.OP_REDUCESCATTER, _lib.F16, 2 * n, ptrs, ptrs, list(range(world)) + [0], row_stride=2 * n)
    comm.check()
    for r in range(world):
        assert np.array_equal(as_bytes(backing[r])[shift: shift + world * n * 2], want[r]), r
        assert torch.all(backing[r][:shift] == 0x5A) and torch.all(backing[r][shift + world * n * 2:] == 0x5A)
    views = [b[shift: shift + world * n * 2] for b in backing]
    root = views[2].clone()
    comm.run(lambda r: broadcast(views[r], 2, comm))
    comm.check()
    for r in range(world):
        assert torch.equal(views[r], root)
        assert torch.all(backing[r][:shift] == 0x5A) and torch.all(backing[r][shift + world * n * 2:] == 0x5A)


def test_a_wait_that_runs_out_is_reported_and_the_grid_drains(dev):
    """A spin limit of one poll: the positions behind the origin find nothing in
    their first slot - the row is still on its way from HBM - and say so."""
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.common import RingTimeout
    world, n = 8, 1 << 22
    comm = make_comm(world)
    comm.spin_budget = 1
    host = torch.randint(0, 256, (n,), dtype=torch.uint8, generator=torch.Generator().manual_seed(1))
    bufs = [host.to(dev) if r == 0 else torch.zeros(n, dtype=torch.uint8, device=dev) for r in range(world)]
    comm.run(lambda r: broadcast(bufs[r], 0, comm))
    with pytest.raises(RingTimeout):
        comm.check()
    comm.spin_budget = 400000
    comm.run(lambda r: broadcast(bufs[r], 0, comm))
    comm.check()
    assert all(torch.equal(b.cpu(), host) for b in bufs)


def test_naming_anything_about_the_wire_goes_through_staging(dev, monkeypatch):
    from mintccl_amd import _lib
    from mintccl_amd.common import VirtualComm
    for kw in (dict(placement=_lib.PLACE_LOCAL), dict(cache_policy=0), dict(threads_per_block=256),
               dict(row_fetch=_lib.FETCH_LDS), dict(origin_cus=9), dict(nslots=2), dict(buff_size_=1 << 22),
               dict(waves_per_rank=64)):
        assert not VirtualComm(8, **kw).inside_cu, kw
    monkeypatch.setenv("MINTCCL_NSLOTS", "4")
    assert not VirtualComm(8).inside_cu
