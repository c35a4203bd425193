"""Rings inside compute units (what the operators run when nothing about the
staging is named): rows around every edge of the walk - less than a lane's 16
bytes, around a wavefront's 1 KiB and a tile's 2, at any byte, in both forms of
the kernels - bit for bit against the oracle or, for the large rows, against the
same additions in torch."""
import numpy as np
import pytest
import torch

from oracle import ring
from tests.helpers import as_bytes, rank_rows

pytestmark = pytest.mark.gpu

# bytes of a row (even: whole f16 values)
ROWS = [2, 14, 16, 18, 1022, 1024, 1026, 2046, 2050, 3 * 1024, 4 * 1024 - 2, 4 * 1024 + 2, 64 * 1024 - 2, 65 * 1024 + 16,
        5 * 64 * 1024 + 1040, 7 * 64 * 1024 - 6]


def make_comm(world, **kw):
    from mintccl_amd.common import VirtualComm
    comm = VirtualComm(world_size=world, spin_budget=400000, **kw)
    assert comm.inside_cu
    return comm


def staged_comm(world):
    """The same collectives through staging: another path to the same bits."""
    from mintccl_amd import _lib
    from mintccl_amd.common import VirtualComm
    comm = VirtualComm(world_size=world, spin_budget=400000, placement=_lib.PLACE_LOCAL)
    assert not comm.inside_cu
    return comm


@pytest.mark.parametrize("world,dt", [(8, "f16"), (8, "bf16"), (8, "f32"), (7, "bf16"), (6, "f32"), (5, "f16"),
                                      (4, "bf16"), (3, "f16"), (2, "bf16")])
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
@pytest.mark.parametrize("nbytes", ROWS + [(4 << 20) + 4097, (8 << 20) - 1, (9 << 20) + 5 * 1024 + 3])
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


@pytest.mark.parametrize("world,dt", [(8, "f16"), (7, "bf16"), (6, "f32")])
def test_sums_far_beyond_the_cache(dev, world, dt):
    """More than 640 MiB touched, rows that end in the middle of a vector."""
    from mintccl_amd.reduce import reduce
    from mintccl_amd.reducescatter import reducescatter
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dt]
    comm = make_comm(world)
    n = (648 << 20) // (world * world * dtype.itemsize) + 5
    g = torch.Generator(device=dev).manual_seed(world)
    made = [torch.randn((world, n), generator=g, device=dev, dtype=torch.float32).to(dtype) for _ in range(world)]
    for op, root in ((reducescatter, None), (reduce, 2)):
        bufs = [m.clone() for m in made]
        comm.run(lambda r: op(bufs[r], comm) if root is None else op(bufs[r], root, comm))
        comm.check()
        for r in range(world):
            want = made[r].clone()
            for row in [r] if root is None else range(world) if r == root else []:
                x = made[r][row]
                for h in range(1, world):
                    x = made[(r + h) % world][row] + x
                want[row] = x
            assert torch.equal(bufs[r].view(torch.uint8), want.view(torch.uint8)), (op.__name__, r)


def added(rows, first):
    """rows[first] + ... around the ring, one rounding per addition."""
    x = rows[first]
    for h in range(1, len(rows)):
        x = rows[(first + h) % len(rows)] + x
    return x


@pytest.mark.parametrize("world", [2, 3, 8])
def test_every_bf16_pattern_in_a_sum(dev, world):
    """Each of the 65536 patterns on the first, the second and the last rank that is added, the
    others with zeros, subnormals, the largest values, infinities and NaNs of every kind: bit for bit, a
    NaN as the canonical one, wherever on the ring it came in."""
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.reduce import reduce
    comm = make_comm(world)
    special = np.array([0x0000, 0x8000, 0x0001, 0x807F, 0x3F80, 0xBF80, 0x7F7F, 0xFF7F, 0x7F80, 0xFF80, 0x7F81, 0xFF81,
                        0x7FBF, 0x7FC0, 0xFFC0, 0x7FFF, 0xFFFF], dtype=np.uint16)
    for at in sorted({0, 1, world - 1}):
        pick = np.random.default_rng(world + at)
        host = [pick.choice(special, 65536) if pick.random() < 0.7 or r == (at + 1) % world
                else (pick.standard_normal(65536).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16) for r in range(world)]
        host[at] = np.arange(65536, dtype=np.uint16)
        for op, want in ((lambda b: reduce(b, 0, comm), ring.reduce(host, 0, "bf16")[:1]),
                         (lambda b: allreduce(b, comm), ring.allreduce(host, "bf16"))):
            bufs = [torch.from_numpy(h.view(np.int16).copy()).to(dev).view(torch.bfloat16) for h in host]
            comm.run(lambda r: op(bufs[r]))
            comm.check()
            for r, w in enumerate(want):
                assert np.array_equal(as_bytes(bufs[r]), w.view(np.uint8)), (at, r)


@pytest.fixture(scope="module")
def wide(dev):
    """One allocation of somewhat more than 4 GiB, in which buffers lie wherever a test wants them."""
    return torch.empty((4 << 30) + (64 << 20), dtype=torch.uint8, device=dev)


# span: bytes from the lowest buffer to the end of the last row.  Up to 2^32 - 1 a launch
# in place names its buffers by their distances, beyond by their addresses.
@pytest.mark.parametrize("shift", [0, 6])
@pytest.mark.parametrize("world", range(2, 9))
def test_buffers_near_and_far(dev, wide, world, shift):
    """The same collective on buffers that lie together, as far apart as 32 bits reach, and one
    byte further: the same bytes, those between the buffers included.  The ring is not in the order of the ranks, rows are
    cut, or have gaps between them, and every rank is the lowest once."""
    from mintccl_amd import _lib
    comm = make_comm(world)
    order = list(range(1, world, 2)) + list(range(0, world, 2))
    cycle = order + order[:1]
    row = 4096 + 66                                             # of f16, three tiles, a ragged end
    room = 64 << 10
    ops = [("reduce", _lib.OP_REDUCE, dict(root=world - 1)), ("broadcast", _lib.OP_BROADCAST, dict(root=world // 2)),
           ("allreduce", _lib.OP_ALLREDUCE, {}), ("allgather", _lib.OP_ALLGATHER, dict(row_stride=row)),
           ("reducescatter", _lib.OP_REDUCESCATTER, dict(row_stride=row)),
           ("reducescatter, gaps", _lib.OP_REDUCESCATTER, dict(row_stride=row + 190)),
           ("allgather, cut", _lib.OP_ALLGATHER, dict(row_stride=row, total_bytes=(world - 1) * row - 34)),
           ("reducescatter, cut", _lib.OP_REDUCESCATTER, dict(row_stride=row, total_bytes=(world - 1) * row - 34)),
           ("reducescatter, gaps and cut", _lib.OP_REDUCESCATTER, dict(row_stride=row + 190, total_bytes=world * row - 38))]
    g = torch.Generator(device=dev).manual_seed(world)
    made = torch.randn((world, room // 2), generator=g, device=dev).to(torch.float16).view(torch.uint8)
    for i, (name, op, kw) in enumerate(ops):
        rows = world if "row_stride" in kw else 1
        need = (rows - 1) * kw.get("row_stride", 0) + row
        at = [(r + i) % world * room + shift for r in range(world)]           # from the lowest
        lowest, highest = at.index(min(at)), at.index(max(at))
        results = []
        for span in (None, (1 << 32) - 2, 1 << 32):
            place = list(at)
            if span is not None:
                place[highest] = at[lowest] + span - need
            bufs = [wide[x: x + room - shift] for x in place]
            for b, m in zip(bufs, made):
                b.copy_(m[:room - shift])
            ptrs = {r: b.data_ptr() for r, b in enumerate(bufs)}
            dtype = _lib.BYTES if op in (_lib.OP_BROADCAST, _lib.OP_ALLGATHER) else _lib.F16
            comm.enqueue(op, dtype, row, ptrs, ptrs, cycle, **kw)
            comm.check()
            results.append([b.clone() for b in bufs])
        for got in results[1:]:
            assert all(torch.equal(x, y) for x, y in zip(got, results[0])), name
        if op == _lib.OP_REDUCESCATTER and "cut" not in name:                # against the additions themselves
            for r in range(world):
                part = slice(r * kw["row_stride"], r * kw["row_stride"] + row)
                want = added([made[q][part].view(torch.float16) for q in order], order.index(r))
                assert torch.equal(results[0][r][part], want.view(torch.uint8)), (name, r)


# row: one tile and less, ragged, an eighth of the row to each XCD, in the large form
@pytest.mark.parametrize("row", [2, 2048, 3 * 2048 + 50, (1 << 20) + 16, (1 << 20) + 18, (7 << 20) + 6])
@pytest.mark.parametrize("world", [2, 3, 4, 5])
def test_alltoall_by_distances_and_by_addresses(dev, wide, world, row):
    """An alltoall of up to four ranks names its buffers by their distances in units of 256 bytes, others by
    tables of distances or of addresses: whole units apart (in three orders, as far apart as the
    allocation lets them), 16 and 6 bytes off a unit, and with gaps between the rows, the same bytes and nothing beside them."""
    from mintccl_amd import _lib
    comm = make_comm(world)
    g = torch.Generator(device=dev).manual_seed(world + row)
    cycle = list(range(world)) + [0]
    for turn, far, shift, gap in [(0, False, 0, 0), (1, True, 0, 0), (world, False, 0, 0), (0, True, 16, 0), (1, False, 6, 0),
                                  (0, False, 0, 190)]:
        step = -(-(world * (row + gap) + 64) // 256) * 256
        # inputs and outputs by turns around each other; the last of them far away
        at = [(i + turn) % (2 * world) * step + shift * (i % 2) for i in range(2 * world)]
        if far:
            at[at.index(max(at))] += (wide.numel() - 2 * world * step) // 256 * 256 - 256
        views = [wide[x: x + world * (row + gap) + 32] for x in at]
        for v in views:
            v.fill_(0x5A)
        made = torch.randint(0, 256, (world, world, row), dtype=torch.uint8, generator=g, device=dev)
        rows = [v[: world * (row + gap)].view(world, row + gap) for v in views]
        for r in range(world):
            rows[r][:, :row] = made[r]
        ins = {r: views[r].data_ptr() for r in range(world)}
        outs = {r: views[world + r].data_ptr() for r in range(world)}
        comm.enqueue(_lib.OP_ALLTOALL, _lib.BYTES, row, ins, outs, cycle, row_stride=row + gap)
        comm.check()
        for r in range(world):
            assert torch.equal(rows[world + r][:, :row], made[:, r]), (turn, far, shift, gap, r)
            assert torch.equal(rows[r][:, :row], made[r])
        for v, x in zip(views, rows):
            assert torch.all(v[world * (row + gap):] == 0x5A) and torch.all(x[:, row:] == 0x5A)


# MiB touched: in the small form, between, large, far beyond the cache
@pytest.mark.parametrize("mib", [30, 150, 300, 660])
@pytest.mark.parametrize("world,dt", [(2, "f32"), (4, "bf16"), (5, "f32"), (6, "f16"), (7, "bf16"), (8, "f16")])
def test_every_form_near_and_far(dev, wide, world, dt, mib):
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.reduce import reduce
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dt]
    comm = make_comm(world)
    n = (mib << 20) // (world * dtype.itemsize) + 5
    g = torch.Generator(device=dev).manual_seed(world + mib)
    made = [torch.randn(n, generator=g, device=dev).to(dtype) for _ in range(world)]
    nbytes = n * dtype.itemsize
    step = -(-nbytes // 4096) * 4096 + 16
    total = wide.numel() - 64
    summed = added(made, 1)
    for far in (False, True):
        places = [r * step for r in range(world - 1)] + [(total - nbytes) // 16 * 16 if far else (world - 1) * step]
        bufs = [wide[x: x + nbytes].view(dtype) for x in places]
        for op, want in ((lambda r: reduce(bufs[r], 1, comm), lambda r: summed if r == 1 else made[r]),
                         (lambda r: broadcast(bufs[r], 1, comm), lambda r: made[1]),
                         (lambda r: allreduce(bufs[r], comm), None)):
            for b, m in zip(bufs, made):
                b.copy_(m)
            comm.run(op)
            comm.check()
            for r in range(world):
                if want:
                    assert torch.equal(bufs[r].view(torch.uint8), want(r).view(torch.uint8)), (far, r)
                elif far or r:
                    assert torch.equal(bufs[r].view(torch.uint8), same.view(torch.uint8)), (far, r)
                else:
                    same = bufs[0].clone()
    per = (-(-nbytes // world) + 15) // 16 * 16 // dtype.itemsize
    assert torch.equal(same[:per].view(torch.uint8), added([m[:per] for m in made], 0).view(torch.uint8))


# MiB touched: in the small form, between, large, streamed far beyond the cache
@pytest.mark.parametrize("world,mib", [(2, 30), (2, 150), (2, 300), (3, 150), (3, 300), (3, 400), (5, 150), (5, 300), (6, 660), (7, 300),
                                       (8, 30), (8, 300), (8, 660)])
def test_bf16_specials_in_every_form(dev, world, mib):
    """NaNs of several payloads, infinities of both signs, the largest values and subnormals scattered over rows of normal ones:
    the sums bit for bit, a NaN as the canonical one."""
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.reduce import reduce
    from mintccl_amd.reducescatter import reducescatter
    comm = make_comm(world)
    special = torch.tensor([0x7F80, 0xFF80, 0x7F81, 0xFFA3, 0x7FC0, 0xFFC1, 0x7FFF, 0xFFFF, 0x7F7F, 0xFF7F, 0x0001, 0x8000],
                           dtype=torch.int32, device=dev).to(torch.int16)
    n = ((mib << 20) // (2 * world * world) // 8 * 8) * world + world             # rows of whole elements, ragged
    g = torch.Generator(device=dev).manual_seed(world * mib)
    made = []
    for _ in range(world):
        m = torch.randn(n, generator=g, device=dev).to(torch.bfloat16).view(torch.int16)
        at = torch.randint(0, n, (n // 8,), generator=g, device=dev)
        m[at] = special[torch.randint(0, len(special), (n // 8,), generator=g, device=dev)]
        made.append(m)

    def want(first, part=slice(None)):
        x = added([m[part].view(torch.bfloat16) for m in made], first)
        return torch.where(torch.isnan(x), torch.tensor(0x7FC0, dtype=torch.int16, device=dev), x.view(torch.int16))

    def run(call):
        bufs = [m.clone() for m in made]
        comm.run(lambda r: call(bufs[r].view(torch.bfloat16)))
        comm.check()
        return bufs

    got = run(lambda b: reduce(b, 1, comm))
    assert torch.equal(got[1], want(1)) and torch.equal(got[0], made[0])
    got = run(lambda b: reducescatter(b.view(world, -1), comm))
    row = n // world
    for r in range(world):
        part = slice(r * row, r * row + row)
        assert torch.equal(got[r][part], want(r, part)), r
    got = run(lambda b: allreduce(b, comm))
    row = (-(-2 * n // world) + 15) // 16 * 8                                      # (cut in whole vectors)
    for p in range(world):
        part = slice(p * row, min(n, p * row + row))
        result = want(p, part)
        assert all(torch.equal(b[part], result) for b in got), p


# What a launch by distances reaches: rows up to 2^30 bytes, the last one's end up to 2^32 - 1 from the lowest
# address; here both sides of each.
@pytest.mark.parametrize("end", [(1 << 32) - 2, 1 << 32])
@pytest.mark.parametrize("row", [(1 << 30) - 6, 1 << 30, (1 << 30) + 2])
@pytest.mark.parametrize("world", [2, 3])
def test_the_longest_rows_by_distances(dev, wide, world, row, end):
    """A broadcast and a reduce of rows that begin at any byte and lie as far apart as they may: whole
    rows, and the bytes around them."""
    from mintccl_amd import _lib
    comm = make_comm(world)
    cycle = list(range(world)) + [0]
    guard = 64
    # (the ranks' order is not that of the addresses)
    at = [guard + 6 + x for x in ([end - row, 0] if world == 2 else [end - row, 0, (end - row) // 2 // 16 * 16 + 10])]
    g = torch.Generator(device=dev).manual_seed(row % 1000 + world)
    made = [torch.randint(0, 2048, (row // 2,), generator=g, device=dev, dtype=torch.int32).to(torch.float16).view(torch.uint8)
            for _ in range(world)]

    def fresh():
        for x, m in zip(at, made):
            wide[x - guard: x + row + guard].fill_(0x5A)
            wide[x: x + row].copy_(m)

    def same(wanted, what):
        comm.check()
        for r, (x, w) in enumerate(zip(at, wanted)):
            assert torch.equal(wide[x: x + row], w), (what, r)
            assert torch.all(wide[x - guard: x] == 0x5A) and torch.all(wide[x + row: x + row + guard] == 0x5A), (what, r)

    pointers = {r: wide.data_ptr() + x for r, x in enumerate(at)}
    fresh()
    comm.enqueue(_lib.OP_BROADCAST, _lib.BYTES, row, pointers, pointers, cycle, root=1)
    same([made[1]] * world, "broadcast")
    fresh()
    comm.enqueue(_lib.OP_REDUCE, _lib.F16, row, pointers, {0: pointers[0]}, cycle, root=0)
    summed = added([m.view(torch.float16) for m in made], 0).view(torch.uint8)
    same([summed] + made[1:], "reduce")


# MiB touched (bytes loaded and stored, sums: loaded), elements more than that in every row
@pytest.mark.parametrize("mib,more", [(1, 5), (8, 1), (11, 3), (19, 3), (21, 0), (21, 3), (25, 9), (31, 2), (33, 3), (41, 7),
                                      (47, 1021), (72, 6), (74, 1), (85, 3), (89, 5), (105, 2051), (158, 9), (170, 9), (178, 3),
                                      (194, 7), (198, 1), (206, 1), (210, 3), (262, 1), (270, 1)])
@pytest.mark.parametrize("world,dt", [(2, "f32"), (3, "f16"), (4, "f16"), (5, "bf16"), (6, "f32"), (7, "f16"), (8, "bf16")])
def test_every_form(dev, world, dt, mib, more):
    """Sizes on both sides of what a launch's form is chosen by, rows that end in
    the middle of a vector, a tile and an XCD's part of the tiles."""
    from mintccl_amd.allgather import allgather
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.alltoall import alltoall
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.reduce import reduce
    from mintccl_amd.reducescatter import reducescatter
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dt]
    comm = make_comm(world)
    g = torch.Generator(device=dev).manual_seed(100 * world + mib)

    def make(rows, touched):
        n = int(touched * 2**20) // (rows * world * dtype.itemsize) + more
        return [torch.randn((rows, n), generator=g, device=dev, dtype=torch.float32).to(dtype) for _ in range(world)]

    def same(got, want, what):
        comm.check()
        for r, (x, y) in enumerate(zip(got, want)):
            assert torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8)), (what, r)

    made = make(world, mib)
    bufs = [m.clone() for m in made]
    comm.run(lambda r: reducescatter(bufs[r], comm))
    same([b[r] for r, b in enumerate(bufs)], [added([m[r] for m in made], r) for r in range(world)], "reducescatter")
    for r, (b, m) in enumerate(zip(bufs, made)):
        keep = [q for q in range(world) if q != r]
        assert torch.equal(b[keep].view(torch.uint8), m[keep].view(torch.uint8)), ("reducescatter, others' rows", r)
    bufs = [m.clone() for m in made]
    comm.run(lambda r: allgather(bufs[r], comm))
    same(bufs, [torch.stack([made[q][q] for q in range(world)])] * world, "allgather")
    bufs = [m.clone() for m in made]
    comm.run(lambda r: allreduce(bufs[r], comm))
    # (rows of the reduction: the buffer cut into as many as there are ranks, in bytes)
    flat = [m.view(-1) for m in made]
    lone = [f.clone() for f in flat]
    apart = staged_comm(world)
    apart.run(lambda r: allreduce(lone[r], apart))
    same([b.view(-1) for b in bufs], lone, "allreduce")
    made = make(1, mib)
    bufs = [m.clone() for m in made]
    comm.run(lambda r: reduce(bufs[r], 1, comm))
    same(bufs, [added(made, 1) if r == 1 else made[r] for r in range(world)], "reduce")
    comm.run(lambda r: broadcast(bufs[r], world - 1, comm))
    same(bufs, [bufs[world - 1]] * world, "broadcast")
    made = make(world, mib / 2)                       # (as much again is stored)
    outs = [torch.zeros_like(m) for m in made]
    comm.run(lambda r: alltoall(made[r], outs[r], comm))
    same(outs, [torch.stack([made[q][r] for q in range(world)]) for r in range(world)], "alltoall")


@pytest.mark.parametrize("world,mib", [(2, 402), (5, 398), (5, 402), (8, 402)])
def test_a_row_to_one_place_far_beyond_the_cache(dev, world, mib):
    """Both sides of where the wavefronts of an alltoall wait before they store, and a transfer
    between two ranks, which wait throughout: rows that end in the middle of a vector."""
    from mintccl_amd import sendrecv_buffer
    from mintccl_amd.alltoall import alltoall
    comm = make_comm(world)
    n = (mib << 20) // (2 * world * world) + 1029
    g = torch.Generator(device=dev).manual_seed(world + mib)
    bufs = [torch.randint(0, 256, (world, n), dtype=torch.uint8, generator=g, device=dev) for _ in range(world)]
    taken = [torch.full((world * n + 64,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(world)]
    outs = [t[32: 32 + world * n].view(world, n) for t in taken]
    comm.run(lambda r: alltoall(bufs[r], outs[r], comm))
    comm.check()
    for r in range(world):
        assert torch.equal(outs[r], torch.stack([b[r] for b in bufs])), r
        assert torch.all(taken[r][:32] == 0x5A) and torch.all(taken[r][32 + world * n:] == 0x5A), r
    sent = torch.cat([b.view(-1) for b in bufs])[: (mib << 19) + 1029]
    backing = torch.full((sent.numel() + 64,), 0x5A, dtype=torch.uint8, device=dev)
    with comm.rank(0):
        sendrecv_buffer.send(sent, 1, comm)
    with comm.rank(1):
        sendrecv_buffer.recv(backing[32: 32 + sent.numel()], 0, comm)
    comm.run(lambda r: sendrecv_buffer.sync(comm))
    comm.check()
    assert torch.equal(backing[32: 32 + sent.numel()], sent)
    assert torch.all(backing[:32] == 0x5A) and torch.all(backing[32 + sent.numel():] == 0x5A)


@pytest.mark.parametrize("world,mib", [(6, 1284), (7, 704), (8, 2564)])
def test_copies_far_beyond_the_cache(dev, world, mib):
    """Just beyond where a wavefront moves 4 KiB, rows that end in the middle of such a
    tile and of a vector; what lies around the rows stays as it was."""
    from mintccl_amd.allgather import allgather
    from mintccl_amd.broadcast import broadcast
    comm = make_comm(world)
    nbytes = (mib << 20) // (world * world) + 2 * 1024 + 3

    def blocks(row):                       # (a row's first tile may begin up to 1023 bytes before it; one block for the ends)
        return -(-(row + 1023) // 4096) + 1

    g = torch.Generator(device=dev).manual_seed(world)
    rows = [torch.randint(0, 256, (nbytes,), dtype=torch.uint8, generator=g, device=dev) for _ in range(world)]
    backing = [torch.full((world * nbytes + 64,), 0x5A, dtype=torch.uint8, device=dev) for _ in range(world)]
    bufs = [b[32: 32 + world * nbytes].view(world, nbytes) for b in backing]
    for r, b in enumerate(bufs):
        b[r] = rows[r]
    comm.run(lambda r: allgather(bufs[r], comm))
    comm.check()
    assert comm.last_grid == world * blocks(nbytes)
    want = torch.stack(rows)
    for r in range(world):
        assert torch.equal(bufs[r], want), r
        assert torch.all(backing[r][:32] == 0x5A) and torch.all(backing[r][32 + world * nbytes:] == 0x5A), r
    flat = [b[7: 7 + world * nbytes] for b in backing]
    flat[1].copy_(torch.randint(0, 256, (world * nbytes,), dtype=torch.uint8, generator=g, device=dev))
    comm.run(lambda r: broadcast(flat[r], 1, comm))
    comm.check()
    assert comm.last_grid == blocks(world * nbytes)
    for r in range(world):
        assert torch.equal(flat[r], flat[1]), r


@pytest.mark.parametrize("shift", [1, 3, 8, 16, 30])
def test_rows_at_any_byte_touch_nothing_else(dev, shift):
    from mintccl_amd import _lib
    from mintccl_amd.alltoall import alltoall
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
    # (addresses that are no multiples of 256 bytes from each other)
    taken = [torch.full((world * n * 2 + 32 + 2 * r,), 0x5A, dtype=torch.uint8, device=dev)[2 * r:] for r in range(world)]
    outs = [t[shift: shift + world * n * 2] for t in taken]
    comm.run(lambda r: alltoall(views[r], outs[r], comm))
    comm.check()
    for r in range(world):
        row = slice(r * n * 2, (r + 1) * n * 2)
        assert torch.equal(outs[r], torch.cat([v[row] for v in views])), r
        assert torch.all(taken[r][:shift] == 0x5A) and torch.all(taken[r][shift + world * n * 2:] == 0x5A)
    root = views[2].clone()
    comm.run(lambda r: broadcast(views[r], 2, comm))
    comm.check()
    for r in range(world):
        assert torch.equal(views[r], root)
        assert torch.all(backing[r][:shift] == 0x5A) and torch.all(backing[r][shift + world * n * 2:] == 0x5A)


@pytest.mark.parametrize("world,dt", [(8, "bf16"), (7, "f16"), (5, "f32"), (3, "f16"), (2, "f32")])
def test_rows_beyond_the_cache(dev, world, dt):
    """Just beyond 100 MiB touched (the large form; sums of two to six ranks to one place the
    form between, small copies of two ranks), buffers that start 6 or 12 bytes
    behind a 16-byte boundary and rows that end in the middle of a vector."""
    from mintccl_amd.allgather import allgather
    from mintccl_amd.allreduce import allreduce
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.reduce import reduce
    from mintccl_amd.reducescatter import reducescatter
    dtype = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}[dt]
    comm = make_comm(world)
    n = (100 << 20) // (world * world * dtype.itemsize) + 13
    g = torch.Generator(device=dev).manual_seed(world)
    made = [torch.randn(world * n + 3, generator=g, device=dev, dtype=dtype)[3:] for _ in range(world)]
    total = made[0].numel()
    per = (-(-total * dtype.itemsize // world) + 15) // 16 * 16 // dtype.itemsize     # a chunk of the allreduce

    def summed(start, lo, hi):
        x = made[start][lo:hi]
        for h in range(1, world):
            x = made[(start + h) % world][lo:hi] + x
        return x

    def run(op):
        bufs = [torch.empty(total + 3, device=dev, dtype=dtype)[3:].copy_(m) for m in made]
        comm.run(lambda r: op(bufs[r]))
        comm.check()
        return bufs

    def same(a, b):
        return torch.equal(a.view(torch.uint8), b.view(torch.uint8))

    scattered = run(lambda b: reducescatter(b.view(world, n), comm))
    reduced = run(lambda b: reduce(b, world - 1, comm))
    everywhere = run(lambda b: allreduce(b, comm))
    gathered = run(lambda b: allgather(b.view(world, n), comm))
    cast = run(lambda b: broadcast(b, world - 1, comm))
    want = torch.cat([summed(c, c * per, min(total, (c + 1) * per)) for c in range(world)])
    rows = torch.cat([made[r][r * n: (r + 1) * n] for r in range(world)])
    for r in range(world):
        own = made[r].clone()
        own[r * n: (r + 1) * n] = summed(r, r * n, (r + 1) * n)
        assert same(scattered[r], own), r
        assert same(reduced[r], summed(r, 0, total) if r == world - 1 else made[r]), r
        assert same(everywhere[r], want) and same(gathered[r], rows) and same(cast[r], made[world - 1]), r


def test_nothing_waits(dev):
    """A spin limit of one poll, and the abort flag of an earlier launch: the
    launch has nobody to wait for, runs all the same and is counted."""
    from mintccl_amd.broadcast import broadcast
    from mintccl_amd.common import RingTimeout
    world, n = 8, 1 << 22
    comm = make_comm(world)
    comm.spin_budget = 1
    host = torch.randint(0, 256, (n,), dtype=torch.uint8, generator=torch.Generator().manual_seed(1))
    for flag in (0, 1):
        bufs = [host.to(dev) if r == 0 else torch.zeros(n, dtype=torch.uint8, device=dev) for r in range(world)]
        comm.status[0] = comm.status[3] = flag
        comm.run(lambda r: broadcast(bufs[r], 0, comm))
        if flag:
            with pytest.raises(RingTimeout, match="1 later launch"):
                comm.check()
        else:
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
