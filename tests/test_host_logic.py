"""Host-side logic that needs no GPU: knobs and wave-count selection."""
import os
import subprocess
import sys

import pytest

from mintccl_amd import _lib, common, protocol

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_reference_constants():
    assert common.NULL == 0 and common.VECTORIZED_BYTES == 16 and common.WARP_SIZE == 64
    assert protocol.BYTES_LL128_MSG == 128 and protocol.BYTES_LL128_RAW == 120
    assert protocol.WORKGROUP_SIZE == 8 and protocol.PAYLOAD_FLAG_THREAD == 8
    assert protocol.BYTES_BLOCK_MSG == 1024 and protocol.BYTES_BLOCK_RAW == 960


def test_env_knobs_are_read_at_call_time(monkeypatch):
    assert common.num_blocks() == 16 and common.num_warps() == 16
    assert common.buff_size() == 4194304 and common.test_count() == 67108864
    monkeypatch.setenv("MINTCCL_NUM_BLOCKS", "32")
    monkeypatch.setenv("MINTCCL_BUFFSIZE", "8388608")
    monkeypatch.setenv("MINTCCL_TEST_MODE", "0")      # any non-empty string (common.py:113)
    assert common.num_blocks() == 32 and common.buff_size() == 8388608
    assert common.test_mode() is True
    monkeypatch.setenv("MINTCCL_PROTOCOL", "simple")
    assert common.protocol_env() == 1


@pytest.mark.parametrize("n,cap,want", [(64, 16, 16), (64, 100, 64), (60, 16, 15), (7, 4, 1),
                                        (512, 128, 128), (1, 5, 1)])
def test_largest_divisor(n, cap, want):
    assert common._largest_divisor_at_most(n, cap) == want


@pytest.mark.parametrize("world", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("row_blocks", [None, 1, 37, 5000])
@pytest.mark.parametrize("op", [_lib.OP_SENDRECV, _lib.OP_BROADCAST, _lib.OP_REDUCE, _lib.OP_ALLGATHER,
                                _lib.OP_REDUCESCATTER, _lib.OP_ALLREDUCE, _lib.OP_ALLTOALL,
                                _lib.OP_TREE_BROADCAST, _lib.OP_TREE_REDUCE,
                                _lib.OP_ALLGATHER_TEMPORAL])
def test_tuned_geometry_is_always_launchable(op, world, row_blocks):
    """Whatever the collective and the world size, the tuned geometry passes the
    library's own plan check, deals whole channels to the 8 XCDs, fits its
    staging budget and stays inside the wavefront budget."""
    from tests.test_abi import make_op
    reducing = op in (_lib.OP_REDUCE, _lib.OP_REDUCESCATTER, _lib.OP_ALLREDUCE, _lib.OP_TREE_REDUCE)
    pairs = op in (_lib.OP_REDUCE, _lib.OP_REDUCESCATTER, _lib.OP_ALLREDUCE, _lib.OP_SENDRECV,
                   _lib.OP_ALLTOALL)
    threads = common.TUNED_THREADS_REDUCING if pairs else 256
    slot, nslots, waves = common.tuned_geometry(op, world, 2, threads, common.TUNED_NSLOTS,
                                                row_blocks=row_blocks)
    assert slot % 1024 == 0 and slot <= common.TUNED_SLOT_BUDGET and nslots >= 1
    # (staging is allocated for TUNED_NSLOTS slots of TUNED_SLOT_BUDGET)
    assert nslots * slot <= common.TUNED_NSLOTS * common.TUNED_SLOT_BUDGET
    multi = op == _lib.OP_ALLTOALL
    d = make_op(op=op, world=world, slot_bytes=slot, nslots=nslots, waves_per_channel_group=waves,
                placement=_lib.PLACE_LOCAL, cache_policy=2, route_len=2, threads_per_block=threads,
                dtype=_lib.F16 if reducing else _lib.BYTES)
    pipes = world if op in (_lib.OP_ALLGATHER, _lib.OP_REDUCESCATTER, _lib.OP_ALLREDUCE) else 1
    if op == _lib.OP_ALLTOALL:
        pipes = world * world
    d.origin_cus = common.tuned_origin_cus(op, 2 if op in (_lib.OP_SENDRECV, _lib.OP_ALLTOALL) else world,
                                           pipes * -(-waves // (threads // 64)), threads // 64)
    if op == _lib.OP_ALLTOALL:
        for r in range(8):
            d.output[r] = 0x40000000 + r * 0x1000000
    for i in range(9):
        d.ring[i] = i % world if i < world else 0
    d.ring[world] = 0
    if op == _lib.OP_SENDRECV:
        d.ring[0], d.ring[1] = 0, 1
    if op == _lib.OP_ALLREDUCE:
        d.row_stride = 0
    blocks = _lib.lib().mint_ring_grid_blocks(d)
    assert blocks > 0, blocks
    assert blocks % 8 == 0
    # (CUs set apart for origins fill the grid up to whole rounds over the 256
    # CUs, at most 24 wavefronts each)
    budget = common.TUNED_TOTAL_WAVES_ALLTOALL_SIMPLE if multi else common.TUNED_TOTAL_WAVES
    assert blocks * (threads // 64) <= (24 * 256 if d.origin_cus else budget)
    d.origin_cus = 0
    assert 0 < _lib.lib().mint_ring_grid_blocks(d) <= blocks
    assert _lib.lib().mint_ring_grid_blocks(d) * (threads // 64) <= budget


CU_OPS = [_lib.OP_SENDRECV, _lib.OP_BROADCAST, _lib.OP_REDUCE, _lib.OP_ALLGATHER, _lib.OP_REDUCESCATTER,
          _lib.OP_ALLREDUCE, _lib.OP_ALLTOALL]
CU_SUMS = (_lib.OP_REDUCE, _lib.OP_REDUCESCATTER, _lib.OP_ALLREDUCE)


def inside_compute_units(op, world, row):
    """Descriptor of a collective inside compute units, rows of `row` bytes."""
    from tests.test_abi import make_op
    alltoall, one = op == _lib.OP_ALLTOALL, op in (_lib.OP_SENDRECV, _lib.OP_BROADCAST, _lib.OP_REDUCE)
    d = make_op(op=op, world=world, placement=_lib.PLACE_CU, dtype=_lib.F16 if op in CU_SUMS else _lib.BYTES,
                count_bytes=row * (world if op == _lib.OP_ALLREDUCE else 1),
                row_stride=0 if one or op == _lib.OP_ALLREDUCE else row, route_len=2 if op == _lib.OP_SENDRECV else 0)
    for i in range(9):
        d.ring[i] = i % world if i <= world else 0
    for r in range(8):
        d.input[r] = d.output[r] = 0x100000000000 + r * 0x4000000000 if r < world else 0
        if alltoall and r < world:
            d.output[r] += 0x200000000000
    return d


def cu_grid(op, world, mib):
    """Thread blocks per row, and the bytes of a row, of a collective inside compute
    units whose ranks touch `mib` MiB in all; rows in whole 4 KiB."""
    pipes = world * world if op == _lib.OP_ALLTOALL else 1 if op in CU_OPS[:3] else world
    touching = 2 if op in (_lib.OP_ALLTOALL, _lib.OP_SENDRECV) else world
    row = int(mib * 2**20) // (pipes * touching) // 4096 * 4096
    blocks = _lib.lib().mint_ring_grid_blocks(inside_compute_units(op, world, row))
    assert blocks > 0 and blocks % pipes == 0
    return blocks // pipes, row


@pytest.mark.parametrize("op,world", [(_lib.OP_SENDRECV, 2), (_lib.OP_SENDRECV, 8), (_lib.OP_BROADCAST, 2),
                                      (_lib.OP_ALLGATHER, 2)] + [(_lib.OP_ALLTOALL, w) for w in range(2, 9)])
def test_a_row_copied_once_moves_in_small_tiles_up_to_192_mib(op, world):
    """Where the same buffers are used again the large form costs 2 - 12 % there."""
    for mib, tile in ((150, 2048), (167, 2048), (172, 2048), (190, 2048), (193, 1024), (300, 1024)):
        blocks, row = cu_grid(op, world, mib)
        assert 0 <= blocks - -(-row // tile) < 8, (mib, blocks, row)


@pytest.mark.parametrize("op", [_lib.OP_REDUCE, _lib.OP_REDUCESCATTER])
@pytest.mark.parametrize("world", [2, 3, 4, 5, 6, 7, 8])
def test_small_sums_do_not_stream_their_rows(op, world):
    """A form that streams its rows moves them in tiles of one wavefront.  Rows of a few MiB
    would leave the caches that the next kernel finds them in."""
    for mib in (1, 8, 12, 16, 19, 22, 28, 31, 33, 39, 41, 60, 75):
        blocks, row = cu_grid(op, world, mib)
        assert 0 <= blocks - -(-row // 2048) < 8, (mib, blocks, row)


@pytest.mark.parametrize("op", [_lib.OP_BROADCAST, _lib.OP_ALLGATHER])
@pytest.mark.parametrize("world", [3, 4, 5, 6, 7, 8])
def test_rows_copied_to_several_places_stay_in_the_cache_up_to_88_mib(op, world):
    """The large form (tiles of 1 KiB, of eight ranks 2 KiB at whole KiB) stores past the
    last-level cache; a kernel that reads the results next misses them there."""
    for mib in (70, 72.5, 73.5, 75.5, 76.5, 80, 87.5, 88.5, 100):
        blocks, row = cu_grid(op, world, mib)
        tile = 2048 if mib < 88 or world == 8 else 1024
        assert 0 <= blocks - -(-row // tile) < 8, (mib, blocks, row)


@pytest.mark.parametrize("op,world,least,most", [
    (_lib.OP_REDUCE, 2, 12, 100), (_lib.OP_REDUCE, 6, 20, 100), (_lib.OP_REDUCE, 7, 20, 100), (_lib.OP_REDUCE, 8, 20, 100), (_lib.OP_BROADCAST, 3, 20, 73), (_lib.OP_BROADCAST, 8, 20, 73),
    (_lib.OP_ALLGATHER, 4, 20, 73), (_lib.OP_ALLGATHER, 8, 99, 0), (_lib.OP_SENDRECV, 2, 20, 192)])
def test_where_an_xcd_takes_an_eighth_of_every_row(op, world, least, most):
    """Then a row has a multiple of eight thread blocks, else one per tile.  Not where a reduce
    of seven or eight ranks just outgrows the L2s: the same buffers again up to 1.7 of the time."""
    for mib in (11, 13, 17, 19, 21, 30, 31.5, 33, 45, 55.5, 57, 59, 71, 72.9, 73.1, 80, 87):
        row = int(mib * 2**20) // (2 if op == _lib.OP_SENDRECV else world) // (world if op == _lib.OP_ALLGATHER else 1)
        row = row // 16384 * 16384 + 2048 * 3                     # tiles: 3 more than a multiple of 8
        blocks = _lib.lib().mint_ring_grid_blocks(inside_compute_units(op, world, row))
        tiles = row // 2048 * (world if op == _lib.OP_ALLGATHER else 1)
        if op == _lib.OP_ALLGATHER:
            blocks, tiles = blocks // world, tiles // world
        outgrows = op == _lib.OP_REDUCE and world >= 7 and 32 < mib < 56
        assert blocks == (tiles + 5 if least <= mib <= most and not outgrows else tiles), (mib, blocks, tiles)


def cu_tile(op, world, touched):
    """Bytes of a tile inside compute units, and of what it begins at whole ones."""
    mib = touched / 2**20
    if op in CU_SUMS:
        if mib <= 100:
            return 2048, 128
        if op != _lib.OP_ALLREDUCE and mib <= {2: 196, 3: 264, 4: 208, 5: 176, 6: 160}.get(world, 0):
            return (2048 if world <= 4 else 1024), 128
        return 1024, 1024
    if op in (_lib.OP_SENDRECV, _lib.OP_ALLTOALL) or world == 2:
        return (2048, 128) if mib <= 192 else (1024, 1024)
    if mib <= 88:
        return 2048, 128
    if mib > {6: 1280, 7: 700, 8: 2560}.get(world, 1 << 30):
        return 4096, 1024
    return (2048 if world == 8 else 1024), 1024


@pytest.mark.parametrize("world", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("op", CU_OPS)
def test_every_tile_of_a_row_has_its_block_inside_compute_units(op, world):
    """The grid has a thread block for every tile of a row and one for its ragged ends, and
    no others but what makes a row's a multiple of eight where the XCDs take an eighth of it
    each; on both sides of every line between the forms."""
    alltoall, one = op == _lib.OP_ALLTOALL, op in CU_OPS[:3]
    copies = op in (_lib.OP_BROADCAST, _lib.OP_ALLGATHER) and world > 2
    pipes, rows = (world * world, world) if alltoall else (1, 1) if one else (world, world)
    touching = 2 if alltoall or op == _lib.OP_SENDRECV else world
    for mib in (1, 8, 11, 13, 19, 21, 23, 33, 41, 50, 72, 74, 87, 89, 99, 101, 150, 159, 161, 175, 177, 191, 193, 195, 197, 207, 209, 263, 265,
                639, 641, 699, 701, 1279, 1281, 2559, 2561):
        for more in (0, 2, 30, 1022, 2046, 4094, 4096):
            row = (mib << 20) // (pipes * touching) // 4096 * 4096 + more
            d = inside_compute_units(op, world, row)
            blocks = _lib.lib().mint_ring_grid_blocks(d)
            assert blocks > 0 and blocks % pipes == 0, (mib, more, blocks)
            held = -(-row // 16) * 16 if op == _lib.OP_ALLREDUCE else row       # (cut in whole vectors)
            touched = pipes * held * touching
            tile, align = cu_tile(op, world, touched)
            slack = align - 1 if not one and held % align else 0
            # (the last row of an allreduce is what the others leave of the buffer)
            last = d.count_bytes - (world - 1) * held if op == _lib.OP_ALLREDUCE else row
            want = -(-(held + slack) // tile) + (last % 16 != 0 or held % 16 != 0)
            least = 12 if op == _lib.OP_REDUCE and world == 2 else 20
            outgrows = op == _lib.OP_REDUCE and world >= 7 and 32 << 20 < touched <= 56 << 20
            if rows % 8 and align == 128 and touched >= least << 20 and not (copies and touched > 73 << 20) and not outgrows:
                want = -(-want // 8) * 8
            assert blocks // pipes == want, (mib, more, blocks // pipes, want)


def test_headline_geometry():
    assert common.tuned_geometry(_lib.OP_REDUCESCATTER, 8, 0, 128, 3) == (448 * 1024, 3, 56)
    assert common.tuned_geometry(_lib.OP_ALLREDUCE, 8, 0, 128, 3) == (512 * 1024, 3, 32)
    assert common.tuned_geometry(_lib.OP_ALLGATHER, 8, 0, 256, 3) == (512 * 1024, 3, 64)
    assert common.tuned_geometry(_lib.OP_BROADCAST, 8, 0, 256, 3) == (512 * 1024, 3, 512)
    assert common.tuned_geometry(_lib.OP_SENDRECV, 8, 2, 128, 3) == (1536 * 1024, 4, 1536)
    assert common.tuned_geometry(_lib.OP_SENDRECV, 8, 3, 128, 3) == (1536 * 1024, 3, 1536)
    assert common.tuned_geometry(_lib.OP_SENDRECV, 8, 2, 128, 3, ll128=False) == (2304 * 1024, 3, 2304)
    assert common.tuned_origin_cus(_lib.OP_SENDRECV, 2, 768, 2) == 20
    assert common.tuned_origin_cus(_lib.OP_ALLGATHER, 8, 8 * 16, 4) == 9
    assert common.tuned_origin_cus(_lib.OP_BROADCAST, 8, 128, 4) == 9
    assert common.tuned_origin_cus(_lib.OP_REDUCESCATTER, 8, 128, 4) == 0
    assert common.tuned_geometry(_lib.OP_ALLTOALL, 8, 0, 128, 3) == (8 * 20 * 1024, 6, 20)
    assert common.tuned_geometry(_lib.OP_ALLTOALL, 8, 0, 128, 3, ll128=False) == (8 * 44 * 1024, 2, 44)
    assert common.tuned_origin_cus(_lib.OP_ALLTOALL, 2, 64 * 10, 2) == 20
    # a small message takes a small grid: the wave-channels are capped at the
    # blocks of one row, in whole thread blocks that the 8 XCDs divide
    assert common.tuned_geometry(_lib.OP_ALLGATHER, 8, 0, 256, 3, row_blocks=1) == (32 * 1024, 3, 4)
    assert common.tuned_geometry(_lib.OP_ALLGATHER, 8, 0, 256, 3, row_blocks=61) == (512 * 1024, 3, 64)
    assert common.tuned_geometry(_lib.OP_ALLGATHER, 8, 0, 256, 3, row_blocks=53) == (448 * 1024, 3, 56)
    assert common.tuned_geometry(_lib.OP_ALLGATHER, 8, 0, 256, 3, row_blocks=10 ** 6) == (512 * 1024, 3, 64)
    assert common.tuned_geometry(_lib.OP_BROADCAST, 8, 0, 256, 3, row_blocks=5) == (32 * 1024, 3, 32)
    assert common.tuned_geometry(_lib.OP_TREE_REDUCE, 8, 0, 256, 3, row_blocks=5) == (2 * 32 * 1024, 3, 32)
    assert common.tuned_geometry(_lib.OP_TREE_REDUCE, 8, 0, 256, 3) == (2 * 512 * 1024, 3, 512)


def test_codec_front_before_the_library_is_bound():
    """A call goes to the function as it came, one that does not fit included."""
    code = """if True:
        from mintccl_amd import _host
        def pack(raw, flag_base=1, layout=2, flag_stride=3, out=None):
            return raw, flag_base, layout, flag_stride, out
        front = _host.Front(pack, _host.PACK, None)
        assert front(5) == (5, 1, 2, 3, None) and front(out=4, raw=5) == (5, 1, 2, 3, 4)
        assert front(5, 6, 7, 8, 9) == (5, 6, 7, 8, 9)
        for args, names in (((), {}), ((1, 2, 3, 4, 5, 6), {}), ((5,), {"raw": 5}), ((5,), {"raws": 5})):
            try:
                front(*args, **names)
            except TypeError as e:
                assert "pack()" in str(e)
            else:
                raise AssertionError(args)
        print("DONE")
    """
    assert "DONE" in subprocess.check_output([sys.executable, "-c", code], cwd=ROOT).decode()
