"""The work that programs have this package do, as cases that can be timed: the
collectives through their operators on eight (and fewer) virtual ranks, a
point-to-point transfer, and the stand-alone LL128 codec, from the smallest
message of the benchmark configurations to the largest.

A case is a dict of plain values:

    name   listed cases only
    op     sendrecv | broadcast | reduce | allgather | reducescatter |
           allreduce | alltoall | codec
    world  virtual ranks of the communicator (codec: 1)
    count  elements: of one rank's buffer (sendrecv, broadcast, reduce,
           allreduce), of one row of it (allgather, reducescatter, alltoall:
           a buffer has `world` rows), of the raw side (codec)
    dtype  f16 | bf16 | f32
    proto  ll128 (what a communicator speaks unless told otherwise) | simple
    root   broadcast and reduce: the root; sendrecv: the sender (the receiver
           is the rank before it)
"""
import math

import torch

from mintccl_amd import _lib, protocol, sendrecv_buffer
from mintccl_amd.allgather import allgather
from mintccl_amd.allreduce import allreduce
from mintccl_amd.alltoall import alltoall
from mintccl_amd.broadcast import broadcast
from mintccl_amd.common import VirtualComm
from mintccl_amd.reduce import reduce
from mintccl_amd.reducescatter import reducescatter

DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}
REDUCING = ("reduce", "reducescatter", "allreduce")
ROWWISE = ("allgather", "reducescatter", "alltoall")

#: Bytes of one rank's buffer (rowwise: of one row of it; codec: of the raw side), least and most.
RANGE = {
    "sendrecv": (1 << 10, 256 << 20),
    "broadcast": (1 << 10, 64 << 20),
    "reduce": (1 << 10, 128 << 20),
    "allgather": (512, 128 << 20),
    "reducescatter": (512, 32 << 20),
    "allreduce": (1 << 10, 64 << 20),
    "alltoall": (512, 16 << 20),
    "codec": (64 << 10, 64 << 20),
}


def _case(op, world, count, dtype, proto="ll128", root=0):
    return {"op": op, "world": world, "count": count, "dtype": dtype, "proto": proto, "root": root}


def listed():
    cases = {
        # the smallest message of the allgather sweep: a step counter, a loss value, a handful of flags
        "allgather_512B": _case("allgather", 8, 256, "f16"),
        # a bias or a layer norm's gradients
        "allreduce_64KiB": _case("allreduce", 8, 32 << 10, "bf16"),
        # the codec configuration: 1 MiB to LL128 lines and back
        "codec_1MiB": _case("codec", 1, 512 << 10, "f16"),
        # gradients of a small tensor cut over six ranks, no size a power of two
        "reducescatter_700KB_6": _case("reducescatter", 6, 174763, "f32"),
        # tokens handed to experts on five ranks, rows of an odd length
        "alltoall_3MB_5": _case("alltoall", 5, 1500007, "bf16"),
        # weights handed to every rank (configuration: broadcast of 64 MiB)
        "broadcast_64MiB": _case("broadcast", 8, 32 << 20, "f16"),
        # a gradient bucket of a training step
        "allreduce_64MiB": _case("allreduce", 8, 32 << 20, "bf16"),
        # the point-to-point configuration: 256 MiB between two ranks
        "sendrecv_256MiB": _case("sendrecv", 2, 128 << 20, "f16"),
        # the reduction configuration, 32 Mi elements per rank, in its widest type
        "reduce_32Mi_f32": _case("reduce", 8, 32 << 20, "f32"),
        # the same configuration as a reduce-scatter, over the other protocol
        "reducescatter_32Mi_simple": _case("reducescatter", 8, 4 << 20, "bf16", "simple"),
        # the headline: 256 MiB per rank
        "reducescatter_256MiB": _case("reducescatter", 8, 16 << 20, "f16"),
        # the largest message of the allgather sweep: sharded weights gathered
        "allgather_128MiB": _case("allgather", 8, 64 << 20, "f16"),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def draw(rng):
    op = rng.choice(sorted(RANGE))
    lo, hi = RANGE[op]
    nbytes = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    world = rng.choice([2, 3, 4, 5, 6, 7, 8, 8, 8, 8])
    dtype = rng.choice(["f16", "bf16", "f32"])
    count = max(1, int(nbytes) // SIZE[dtype])
    if rng.random() < 0.5:                     # half of them in whole 16-byte vectors, the others as they fall
        count = max(8, count // 8 * 8)
    if op == "codec":
        return _case(op, 1, count, dtype)
    return _case(op, world, count, dtype, rng.choice(["ll128", "ll128", "ll128", "simple"]),
                 rng.randrange(world) if op in ("sendrecv", "broadcast", "reduce") else 0)


def prepare(case, seed):
    dev = torch.device("cuda:0")
    op, world, n, dt = case["op"], case["world"], case["count"], DTYPE[case["dtype"]]

    def values(rank, *shape):
        # activations and gradients: normal values
        g = torch.Generator(device=dev).manual_seed(seed * 16 + rank)
        return torch.randn(*shape, generator=g, device=dev, dtype=dt)

    state = {"case": case}
    if op == "codec":
        state["raw"] = values(0, n)
        state["out"] = torch.zeros_like(state["raw"])
        return state
    state["comm"] = VirtualComm(world, dev, protocol=_lib.PROTO_SIMPLE if case["proto"] == "simple" else None)
    if op in ("reduce", "allreduce"):
        state["bufs"] = [values(r, n) for r in range(world)]
    elif op == "reducescatter":
        state["bufs"] = [values(r, world, n) for r in range(world)]
    elif op == "alltoall":
        state["bufs"] = [values(r, world, n) for r in range(world)]
        state["outs"] = [torch.zeros_like(b) for b in state["bufs"]]
    elif op == "allgather":
        # every rank brings its own row
        state["bufs"] = [torch.zeros(world, n, device=dev, dtype=dt) for _ in range(world)]
        for r, b in enumerate(state["bufs"]):
            b[r] = values(r, n)
    elif op == "broadcast":
        state["bufs"] = [values(r, n) if r == case["root"] else torch.zeros(n, device=dev, dtype=dt)
                         for r in range(world)]
    else:
        state["bufs"] = [values(0, n), torch.zeros(n, device=dev, dtype=dt)]
    return state


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "codec":
        msg = protocol.pack(state["raw"])
        return [msg, protocol.unpack(msg, state["out"])]
    comm, bufs, root = state["comm"], state["bufs"], case["root"]
    if op == "sendrecv":
        src, dst = root, (root - 1) % case["world"]
        with comm.rank(src):
            sendrecv_buffer.send(bufs[0], dst, comm)
        with comm.rank(dst):
            sendrecv_buffer.recv(bufs[1], src, comm)
        comm.run(lambda r: sendrecv_buffer.sync(comm))
        return bufs[1]
    if op == "broadcast":
        comm.run(lambda r: broadcast(bufs[r], root, comm))
    elif op == "reduce":
        comm.run(lambda r: reduce(bufs[r], root, comm))
    elif op == "allgather":
        comm.run(lambda r: allgather(bufs[r], comm))
    elif op == "reducescatter":
        comm.run(lambda r: reducescatter(bufs[r], comm))
    elif op == "allreduce":
        comm.run(lambda r: allreduce(bufs[r], comm))
    else:
        outs = state["outs"]
        comm.run(lambda r: alltoall(bufs[r], outs[r], comm))
        return outs
    return bufs


def work(case):
    """Every rank's input read once, every output written once, an addition for every value that is combined."""
    op, world, n = case["op"], case["world"], case["count"]
    size = n * SIZE[case["dtype"]]
    if op == "codec":
        # read raw, write lines, read lines, write raw
        return {"bytes": 2 * size + 2 * protocol.packed_bytes(size), "flops": 0}
    moved = {"sendrecv": 2, "broadcast": world, "reduce": world + 1, "allgather": world * world,
             "reducescatter": world * world + world, "allreduce": 2 * world, "alltoall": 2 * world * world}[op]
    added = {"reduce": world - 1, "allreduce": world - 1, "reducescatter": world * (world - 1)}.get(op, 0)
    return {"bytes": moved * size, "flops": added * n}


def tolerance(case):
    # bytes that are moved stay the same; sums are formed in the ring's order,
    # one rounding per addition, which fixes every bit of them
    return "exact"
