"""The native host side of the operators: what it refuses, that it follows the
communicator's attributes and the environment, and whose rank a thread speaks for."""
import threading

import numpy as np
import pytest
import torch

from oracle import ring
from tests.helpers import as_bytes, rank_rows

pytestmark = pytest.mark.gpu


def make_comm(world, **kw):
    from mintccl_amd.common import VirtualComm
    return VirtualComm(world_size=world, spin_budget=400000, **kw)


def test_refusals_leave_the_communicator_usable(dev):
    from mintccl_amd.allgather import allgather
    from mintccl_amd.alltoall import alltoall
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.reduce import reduce
    comm = make_comm(2)
    a, b = torch.zeros(8, device=dev), torch.zeros(8, device=dev, dtype=torch.float16)

    def pair(first, second, match):
        with comm.rank(0):
            first()
        with comm.rank(1), pytest.raises(ValueError, match=match):
            second()

    pair(lambda: broadcast(a, 0, comm), lambda: broadcast(a, 1, comm), "ranks disagree on the root")
    pair(lambda: broadcast(a, 0, comm), lambda: broadcast(b, 0, comm), "byte count: .'16', '32'.")
    pair(lambda: reduce(b, 0, comm), lambda: reduce(b.bfloat16(), 0, comm), "the dtype")
    pair(lambda: allgather(a, comm), lambda: allgather(a, comm, schedule="temporal"),
         "the schedule: .'spatial', 'temporal'.")
    pair(lambda: alltoall(a, torch.zeros_like(a), comm), lambda: alltoall(b.float(), a, comm), "overlaps")
    with comm.rank(0):
        with pytest.raises(ValueError, match="schedule is"):
            allgather(a, comm, schedule="both")
        with pytest.raises(ValueError, match="differ in size"):
            alltoall(a, b, comm)
        reduce(a, 0, comm)
        with pytest.raises(RuntimeError, match="called reduce twice"):
            reduce(a, 0, comm)
    with comm.rank(1):
        reduce(a, 0, comm)
    with pytest.raises(ValueError):
        comm.rank(2)
    comm.check()


def test_launches_follow_attributes_and_environment(dev, monkeypatch):
    """A ring set after the first launch is the ring of the next one (f16 sums
    depend on the order), and MINTCCL_TOPOLOGY / _ALLREDUCE / _ALLGATHER are read
    when an operator runs."""
    from mintccl_amd._ops import ring_of
    from mintccl_amd.allgather import allgather
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.reducescatter import reducescatter
    world, n = 4, 5000
    comm = make_comm(world)
    host = rank_rows(world, n, "f16", seed0=70)
    raw = [as_bytes(h) for h in host]

    def summed():
        bufs = [h.to(dev) for h in host]
        comm.run(lambda r: reducescatter(bufs[r], comm))
        comm.check()
        return [as_bytes(x) for x in bufs]

    plain = summed()
    assert all(np.array_equal(x, y) for x, y in zip(plain, ring.reducescatter(raw, "f16")))
    # only the links of the ring 0 -> 2 -> 1 -> 3 -> 0
    links = [(0, 2), (2, 1), (1, 3), (3, 0)]
    comm.topology = {u: [(v, 1.0) for a, b in links for v in ((b,) if a == u else (a,) if b == u else ())]
                     for u in range(world)}
    turned = summed()
    order = ring_of(comm)
    assert order in ([0, 2, 1, 3, 0], [0, 3, 1, 2, 0])
    assert all(np.array_equal(x, y) for x, y in zip(turned, ring.reducescatter(raw, "f16", order)))
    assert any(not np.array_equal(x, y) for x, y in zip(plain, turned))
    comm.topology = None
    monkeypatch.setenv("MINTCCL_TOPOLOGY", "hypercube")
    cube = summed()
    assert all(np.array_equal(x, y) for x, y in zip(cube, ring.hypercube_reducescatter(raw, "f16")))
    monkeypatch.delenv("MINTCCL_TOPOLOGY")
    for var, value, op, want in (("MINTCCL_ALLREDUCE", "split", allreduce, ring.allreduce(raw, "f16")),
                                 ("MINTCCL_ALLGATHER", "temporal", allgather, ring.allgather(raw))):
        monkeypatch.setenv(var, value)
        bufs = [h.to(dev) for h in host]
        comm.run(lambda r: op(bufs[r], comm))
        comm.check()
        assert all(np.array_equal(as_bytes(b), w) for b, w in zip(bufs, want)), var
        monkeypatch.delenv(var)


def test_a_rank_belongs_to_its_thread_and_communicator(dev):
    from mintccl_amd.broadcast import broadcast
    comm, other = make_comm(3), make_comm(2)
    bufs = [torch.full((1000,), float(r), device=dev) for r in range(3)]
    seen = []

    def rank(r):
        with comm.rank(r), other.rank(0):
            with comm.rank((r + 1) % 3):
                assert comm.Get_rank() == (r + 1) % 3
            assert comm.Get_rank() == r and other.Get_rank() == 0
            broadcast(bufs[r], 1, comm)
        try:
            comm.Get_rank()
        except RuntimeError:
            seen.append(r)

    threads = [threading.Thread(target=rank, args=(r,)) for r in range(3)]
    for t in threads:
        t.start()
        t.join()
    comm.check()
    assert seen == [0, 1, 2]
    assert all(torch.all(b == 1.0) for b in bufs)


def test_codec_refuses_what_it_cannot_take(dev):
    from mintccl_amd import _lib, protocol
    raw = torch.zeros(960, dtype=torch.uint8, device=dev)
    msg = protocol.pack(raw)
    for bad in (lambda: protocol.pack(raw.cpu()), lambda: protocol.pack(raw.view(2, 480).t()),
                lambda: protocol.pack(raw, out=raw), lambda: protocol.unpack(msg[:512], raw),
                lambda: protocol.unpack(msg.cpu(), raw)):
        with pytest.raises(ValueError):
            bad()
    with pytest.raises(_lib.MintError):
        protocol.pack(raw, layout=7)
    with pytest.raises(_lib.MintError) as e:
        protocol.pack(torch.zeros(976, dtype=torch.uint8, device=dev)[1:961])
    assert e.value.code == _lib.ERR_ALIGN


def test_codec_takes_its_arguments_in_every_form(dev):
    """Positional, by name, defaults, a name made at run time; what does not fit is
    the function's own TypeError."""
    import inspect
    import pickle

    from mintccl_amd import _lib, protocol
    raw = torch.arange(2001, dtype=torch.int32, device=dev)
    bad = torch.zeros(1, dtype=torch.int64, device=dev)
    wave, pair = _lib.LAYOUT_WAVE64, _lib.LAYOUT_PAIR
    want = {(base, layout, stride): protocol.pack.__wrapped__(raw, base, layout, stride)
            for base, layout, stride in ((1, wave, 1), (9, pair, 1), (9, wave, 3), (2**64 - 1, wave, 1))}
    into = torch.zeros_like(want[1, wave, 1])
    assert protocol.pack(raw, out=into) is into
    made = "".join(["flag", "_", "base"])              # (another object than the name in the code)
    assert made is not inspect.signature(protocol.pack.__wrapped__).parameters["flag_base"].name
    for msg, kept in ((into, (1, wave, 1)), (protocol.pack(raw), (1, wave, 1)), (protocol.pack(raw=raw), (1, wave, 1)),
                      (protocol.pack(raw, 9, pair), (9, pair, 1)), (protocol.pack(raw, layout=pair, flag_base=9), (9, pair, 1)),
                      (protocol.pack(raw, 9, flag_stride=3), (9, wave, 3)), (protocol.pack(raw, **{made: -1}), (2**64 - 1, wave, 1))):
        base, layout, stride = kept
        assert torch.equal(msg, want[kept])
        for form in (lambda o: protocol.unpack(msg, o, base, layout, stride, bad),
                     lambda o: protocol.unpack(out=o, msg=msg, flag_stride=stride, bad_flags=bad, flag_base=base, layout=layout)):
            back = torch.zeros_like(raw)
            assert form(back) is back and torch.equal(back, raw)
    assert int(bad) == 0
    for call in (lambda: protocol.pack(), lambda: protocol.pack(raw, raws=1), lambda: protocol.pack(raw, raw=raw),
                 lambda: protocol.pack(raw, 1, wave, 1, None, 5), lambda: protocol.unpack(into),
                 lambda: protocol.pack(raw, "1"), lambda: protocol.unpack(into, raw, bad_flags=3)):
        with pytest.raises(TypeError):
            call()
    assert list(inspect.signature(protocol.unpack).parameters) == ["msg", "out", "flag_base", "layout", "flag_stride", "bad_flags"]
    assert pickle.loads(pickle.dumps(protocol.pack)) is protocol.pack


def test_operators_take_their_arguments_in_every_form(dev, monkeypatch):
    """Positional, by name, the default communicator; what does not fit is the
    operator's own TypeError; MINTCCL_TOPOLOGY still reaches the other modules."""
    from mintccl_amd import sendrecv_buffer
    from mintccl_amd.allgather import allgather
    from mintccl_amd.alltoall import alltoall
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.common import get_comm, set_comm
    world, n = 4, 999
    comm, before = make_comm(world), get_comm()
    src = [torch.full((world, n), r + 1, dtype=torch.int32, device=dev) for r in range(world)]
    out = [torch.zeros_like(s) for s in src]
    rows = torch.arange(1, world + 1, dtype=torch.int32, device=dev)[:, None].expand(world, n)

    def fresh():
        return [s.clone() for s in src]
    set_comm(comm)
    try:
        for call in (lambda b: allgather(b), lambda b: allgather(b, comm), lambda b: allgather(buff=b, comm=comm),
                     lambda b: allgather(b, comm=comm, schedule="spatial"), lambda b: allgather(b, None, "temporal"),
                     lambda b: allgather(b, **{"co" + "mm": comm})):
            bufs = fresh()
            comm.run(lambda r: call(bufs[r]))
            comm.check()
            assert all(torch.equal(b, rows) for b in bufs)
        for topology in ("", "tree"):
            monkeypatch.setenv("MINTCCL_TOPOLOGY", topology)
            bufs = fresh()
            comm.run(lambda r: broadcast(bufs[r], comm=comm, root=2))
            comm.check()
            assert all(torch.equal(b, src[2]) for b in bufs)
        comm.run(lambda r: alltoall(src[r], comm=comm, out=out[r]))
        with comm.rank(1):
            sendrecv_buffer.send(peer=3, buff=src[1])
        with comm.rank(3):
            sendrecv_buffer.recv(bufs[3], 1, comm=comm)
        comm.run(lambda r: sendrecv_buffer.sync(route=[1, 0, 3], comm=comm))
        assert comm.last_route == [1, 0, 3]
        comm.check()
        assert all(torch.equal(o, rows) for o in out) and torch.equal(bufs[3], src[1])
        for bad in (lambda: allgather(), lambda: allgather(src[0], comm, None, None),
                    lambda: allgather(src[0], comm, comm=comm), lambda: broadcast(src[0], comm=comm)):
            with pytest.raises(TypeError, match="allgather|broadcast"):
                bad()
    finally:
        set_comm(before)


def test_methods_of_ones_own_are_called(dev, monkeypatch):
    """A subclass's launch, make_op, Get_rank and rank are what an operator goes
    through, on the object and on the class as well, also when they are set
    after a launch."""
    from mintccl_amd import _lib, common
    from mintccl_amd.allgather import allgather
    from mintccl_amd.broadcast import broadcast
    world, n = 3, 1000
    src = [torch.full((world, n), float(r), device=dev) for r in range(world)]
    rows = torch.arange(world, device=dev, dtype=torch.float32)[:, None].expand(world, n)
    calls = []

    class Own(common.VirtualComm):
        def launch(self, d):
            calls.append(("launch", d.op, d.placement))
            super().launch(d)

    class Described(common.VirtualComm):
        def make_op(self, *args, **kw):
            calls.append("make_op")
            return super().make_op(*args, **kw)

    class Elsewhere(common.VirtualComm):
        speaker = None

        def Get_rank(self):
            return self.speaker

        def rank(self, r):
            calls.append(r)
            return super().rank(r)

    def gather(comm, run=None):
        calls.clear()
        bufs = [s.clone() for s in src]
        (run or comm.run)(lambda r: allgather(bufs[r], comm))
        comm.check()
        assert all(torch.equal(b, rows) for b in bufs)
    gather(Own(world, dev))
    assert calls == [("launch", _lib.OP_ALLGATHER, _lib.PLACE_CU)]
    comm = Described(world, dev)
    gather(comm)
    assert calls == ["make_op"] and comm.epoch == 1
    comm = Elsewhere(world, dev)

    def in_turn(fn):
        for comm.speaker in range(world):
            fn(comm.speaker)
    gather(comm, in_turn)
    comm.speaker = world
    with pytest.raises(ValueError, match="rank 3"):
        broadcast(src[0], 0, comm)
    comm.speaker = 0
    comm.run(calls.append)
    assert calls == [0, 0, 1, 1, 2, 2]
    # after launches of an ordinary communicator: on the object, on its class
    comm = make_comm(world)
    gather(comm)
    assert not calls
    comm.launch = lambda d: (calls.append("own"), common.VirtualComm.launch(comm, d))
    gather(comm)
    assert calls == ["own"]
    del comm.launch
    gather(comm)
    assert not calls
    plain = common.VirtualComm.launch
    with monkeypatch.context() as m:
        m.setattr(common.VirtualComm, "launch", lambda self, d: (calls.append("class"), plain(self, d)))
        gather(comm)
        assert calls == ["class"]
    gather(comm)
    assert not calls


def test_an_attribute_of_the_wire_set_after_a_launch_is_in_the_next_one(dev):
    from mintccl_amd.allgather import allgather
    world, n = 8, 5000
    comm = make_comm(world)
    for launch in range(3):
        bufs = [torch.zeros(world, n, device=dev) for _ in range(world)]
        for r, b in enumerate(bufs):
            b[r] = r + 1
        comm.run(lambda r: allgather(bufs[r], comm))
        comm.check()
        assert comm.epoch == launch and all(torch.equal(b, bufs[0]) and b[-1, -1] == world for b in bufs)
        comm.threads_per_block = 128


def test_a_topology_changed_in_place_changes_the_next_route(dev):
    from mintccl_amd import sendrecv_buffer
    comm = make_comm(4)
    comm.topology = {0: [(1, 2.0)], 1: [(0, 2.0), (3, 2.0)], 2: [], 3: [(1, 2.0)]}
    src, dst = torch.arange(1000, device=dev), torch.zeros(1000, dtype=torch.int64, device=dev)

    def route():
        dst.zero_()
        with comm.rank(0):
            sendrecv_buffer.send(src, 3, comm)
        with comm.rank(3):
            sendrecv_buffer.recv(dst, 0, comm)
        comm.run(lambda r: sendrecv_buffer.sync(comm))
        comm.check()
        assert torch.equal(src, dst)
        return comm.last_route
    assert route() == [0, 1, 3]
    comm.topology[0].append((2, 5.0))
    comm.topology[2].append((3, 5.0))
    assert route() == [0, 2, 3]
    comm.topology[0].append((3, 1.0))
    assert route() == [0, 3]
    del comm.topology[0][-1]
    assert route() == [0, 2, 3]
    del comm.topology
    assert route() == [0, 3]


def test_the_allocation_of_a_message_is_seen(dev):
    """By dispatch modes, function modes and the profiler, as any allocation."""
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from mintccl_amd import protocol
    raw = torch.arange(2000, dtype=torch.int32, device=dev)
    seen = []

    class Dispatched(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    class Functions(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))
    want = protocol.pack(raw)
    with Dispatched():
        msg = protocol.pack(raw)
    assert any("aten.empty" in str(f) for f in seen) and torch.equal(msg, want)
    seen.clear()
    with Functions():
        msg = protocol.pack(raw)
    assert torch.empty in seen and torch.equal(msg, want)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        protocol.pack(raw)
    assert any(e.key == "aten::empty" for e in prof.key_averages())


def test_a_launch_without_an_epoch_advances_none(dev):
    """With the epoch in device memory: a ring inside compute units leaves it (and
    the staging that is cleared when it starts over) alone, one through staging
    advances it."""
    from mintccl_amd.allgather import allgather
    world = 4
    comm = make_comm(world, device_epoch=True)
    comm.epoch_word[0] = 4094
    comm.staging.fill_(7)
    bufs = [torch.zeros(world, 1000, device=dev) for _ in range(world)]
    for r, b in enumerate(bufs):
        b[r] = r + 1
    rows = torch.arange(1, world + 1, dtype=torch.float32, device=dev)[:, None].expand(world, 1000)
    for _ in range(3):
        comm.run(lambda r: allgather(bufs[r], comm))
    comm.check()
    assert all(torch.equal(b, rows) for b in bufs)
    assert int(comm.epoch_word[0]) == 4094 and torch.all(comm.staging == 7)
    comm.staging.zero_()
    comm.run(lambda r: allgather(bufs[r], comm, schedule="temporal"))
    comm.check()
    assert int(comm.epoch_word[0]) == 4095 and all(torch.equal(b, rows) for b in bufs)
