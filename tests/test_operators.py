"""The operators and the communicator as Python objects (no GPU needed): what a
function and a context manager can do."""
import copy
import importlib
import inspect
import pickle
import weakref

import pytest

from mintccl_amd import _lib, common

OPERATORS = [("broadcast", "broadcast"), ("reduce", "reduce"), ("allgather", "allgather"),
             ("reducescatter", "reducescatter"), ("allreduce", "allreduce"), ("alltoall", "alltoall"),
             ("sendrecv_buffer", "send"), ("sendrecv_buffer", "recv"), ("sendrecv_buffer", "sync")]


@pytest.fixture
def make_comm(monkeypatch):
    """A communicator whose memory lies on the host: nothing can be launched."""
    monkeypatch.setattr(common, "_xcd_count", lambda device: 8)
    for knob in ("NUM_BLOCKS", "NUM_WARPS", "BUFFSIZE", "NSLOTS", "PLACEMENT", "THREADS", "CACHE",
                 "ROW_FETCH", "ORIGIN_CUS", "PROTOCOL"):
        monkeypatch.delenv("MINTCCL_" + knob, raising=False)
    return lambda world=4, cls=common.VirtualComm, **kw: cls(world, device="cpu", **kw)


@pytest.mark.parametrize("module,name", OPERATORS)
def test_an_operator_can_be_handed_on_like_a_function(module, name):
    """Pickled by its name (a spawned process gets the operator), copied as
    itself, referred to weakly, bound where a class holds it."""
    op = getattr(importlib.import_module("mintccl_amd." + module), name)
    assert pickle.loads(pickle.dumps(op)) is op
    assert copy.copy(op) is op and copy.deepcopy({"op": [op]})["op"][0] is op
    assert weakref.ref(op)() is op
    assert op.__name__ == name and "comm" in inspect.signature(op).parameters

    class Holder:
        held = op
    holder = Holder()
    assert Holder.held is op
    assert holder.held.__self__ is holder and holder.held.__func__ is op


def test_a_rank_as_a_decorator(make_comm):
    comm = make_comm()

    @comm.rank(2)
    def who(x, *, y):
        """docs"""
        return comm.Get_rank(), x, y
    assert who.__name__ == "who" and who.__doc__ == "docs"
    for _ in range(2):
        assert who(1, y=3) == (2, 1, 3)
        with comm.rank(1):
            assert who(4, y=5) == (2, 4, 5) and comm.Get_rank() == 1

    @comm.rank(3)
    def nested(depth):
        return nested(depth - 1) if depth else comm.Get_rank()
    assert nested(2) == 3
    with pytest.raises(RuntimeError, match="no current rank"):
        comm.Get_rank()


def test_a_rank_context_is_not_entered_twice_at_a_time(make_comm):
    """The second way in would forget whose rank the thread had before the first."""
    comm = make_comm()
    context = comm.rank(1)
    with context:
        with pytest.raises(RuntimeError, match="entered"):
            with context:
                pass
        assert comm.Get_rank() == 1
    with pytest.raises(RuntimeError, match="no current rank"):
        comm.Get_rank()


def test_a_make_op_of_ones_own_is_the_one_that_is_used(make_comm):
    """In a subclass or on the object: it describes launches through staging."""
    class Own(common.VirtualComm):
        def make_op(self, *args, **kw):
            d = super().make_op(*args, **kw)
            d.nslots = 2
            return d
    comm, plain = make_comm(cls=Own), make_comm()
    plain.make_op = lambda *args, **kw: "mine"
    seen = []
    for c in (comm, plain):
        c.launch = seen.append
        ptrs = {r: 4096 * (r + 1) for r in range(4)}
        c.enqueue(_lib.OP_BROADCAST, _lib.BYTES, 64, {0: ptrs[0]}, ptrs, [0, 1, 2, 3, 0])
    assert seen[0].nslots == 2 and seen[0].placement != _lib.PLACE_CU and seen[1] == "mine"


@pytest.mark.parametrize("name,value", [("placement", _lib.PLACE_SPREAD), ("cache_policy", 0),
                                        ("row_fetch", _lib.FETCH_LDS), ("origin_cus", 9),
                                        ("threads_per_block", 512), ("waves_per_rank", 64), ("nslots", 2),
                                        ("slot_bytes", 1 << 16), ("auto_geometry", False)])
def test_naming_the_wire_after_construction_goes_through_staging(make_comm, name, value):
    """As naming it in the constructor does, and what is named is in the next
    launch's descriptor."""
    comm = make_comm(8)
    launched = []
    comm.launch = launched.append
    ptrs = {r: 4096 * (r + 1) for r in range(8)}
    ring = list(range(8)) + [0]

    def launch():
        comm.enqueue(_lib.OP_ALLGATHER, _lib.BYTES, 1 << 20, ptrs, ptrs, ring, row_stride=1 << 20)
        return launched[-1]
    assert comm.inside_cu and launch().placement == _lib.PLACE_CU
    if name == "placement":
        comm.cache_policy = 0           # (agent scope: what the spread placement takes)
    setattr(comm, name, value)
    d = launch()
    assert not comm.inside_cu and d.placement != _lib.PLACE_CU and d.nslots
    if name in ("placement", "cache_policy", "row_fetch", "origin_cus", "threads_per_block", "nslots"):
        assert getattr(d, name) == value


def test_the_protocol_says_how_a_hop_through_staging_is_made(make_comm, monkeypatch):
    """It alone does not ask for staging (inside a compute unit there is no hop to
    make safe); with anything else of the wire named it is the launch's."""
    assert make_comm(protocol=_lib.PROTO_SIMPLE).inside_cu
    monkeypatch.setenv("MINTCCL_PROTOCOL", "simple")
    assert make_comm().inside_cu
    comm = make_comm(8, placement=_lib.PLACE_LOCAL)
    assert not comm.inside_cu
    ptrs = {r: 4096 * (r + 1) for r in range(8)}
    d = comm.make_op(_lib.OP_ALLGATHER, _lib.BYTES, 4096, ptrs, ptrs, list(range(8)) + [0], row_stride=4096)
    assert d.protocol == _lib.PROTO_SIMPLE and d.staging[0]
