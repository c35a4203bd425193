"""The operators as Python objects (no GPU needed): what a function can do."""
import copy
import importlib
import inspect
import pickle
import weakref

import pytest

OPERATORS = [("broadcast", "broadcast"), ("reduce", "reduce"), ("allgather", "allgather"),
             ("reducescatter", "reducescatter"), ("allreduce", "allreduce"), ("alltoall", "alltoall"),
             ("sendrecv_buffer", "send"), ("sendrecv_buffer", "recv"), ("sendrecv_buffer", "sync")]


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
