"""The rules that say how many wavefronts of a launch inside compute units a compute unit
holds (csrc/cu_rules.hpp), compiled by the host's compiler alone."""
import os
import subprocess

import pytest

from mintccl_amd import _lib

CSRC = os.path.join(os.path.dirname(_lib.__file__), "csrc")
OPS = {"broadcast": _lib.OP_BROADCAST, "allgather": _lib.OP_ALLGATHER, "reduce": _lib.OP_REDUCE,
       "reducescatter": _lib.OP_REDUCESCATTER, "allreduce": _lib.OP_ALLREDUCE}
TYPES = {"f16": _lib.F16, "bf16": _lib.BF16, "f32": _lib.F32, "bytes": _lib.BYTES}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """rule(expression) -> its value as a whole number."""
    where = tmp_path_factory.mktemp("rules")
    known = {}

    def evaluate(*expressions):
        new = [e for e in expressions if e not in known]
        if new:
            source, program = str(where / "rules.cpp"), str(where / "rules")
            with open(source, "w") as f:
                f.write('#include "cu_rules.hpp"\n#include <cstdio>\nusing namespace mint;\nint main() {\n')
                f.writelines(f'    printf("%lld\\n", (long long)({e}));\n' for e in new)
                f.write("}\n")
            subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, source, "-o", program], check=True)
            known.update(zip(new, map(int, subprocess.check_output([program]).split())))
        return [known[e] for e in expressions]
    return evaluate


def waves(op, dtype, ranks, mib, vast=False):
    """The large form's count for `mib` MiB touched."""
    return f"cu_waves({OPS[op]}, {TYPES[dtype]}, {ranks}, {str(vast).lower()}, {(mib << 20) // ranks}ull)"


def test_a_block_at_least(rule):
    """However few wavefronts a rule names, a compute unit holds a block of them, and no less LDS
    than that leaves is asked for."""
    lds, unit = rule("kCuLds", "kCuLdsUnit")
    cases = [(w, t) for t in (64, 128, 256) for w in range(1, 33)]
    for (w, t), share in zip(cases, rule(*(f"cu_lds_share({w}, {t})" for w, t in cases))):
        blocks = max(1, w * 64 // t)
        if w == 32:
            assert share == 0
        else:
            assert share % unit == 0 and share * blocks <= lds < (share + unit) * blocks, (w, t, share)


def test_every_rule_names_whole_blocks(rule):
    """No form has more than two wavefronts to a block."""
    sizes = (1, 20, 24, 25, 28, 30, 32, 40, 90, 101, 129, 131, 150, 164, 166, 210, 300, 330, 470, 490, 700, 3000)
    asked = [e for r in range(2, 9) for m in sizes for e in (
        [waves(op, dt, r, m) for op in ("reduce", "reducescatter", "allreduce") for dt in ("f16", "bf16", "f32")] +
        [waves(op, "bytes", r, m, vast) for op in ("broadcast", "allgather") for vast in (False, True)] +
        [f"cu_mid_waves({r}, {m << 20}ull)"] + [f"cu_small_waves({op}, {r}, {m << 20}ull)" for op in OPS.values()])]
    for e, value in zip(asked, rule(*asked)):
        assert 2 <= value <= 32, e


@pytest.mark.parametrize("op", ["broadcast", "allgather"])
def test_copies_of_rows_that_no_translation_is_at_hand_for(rule, op):
    """On buffers that 1.3 GB and more lie between two uses of, every access waits for its address to be
    translated too, and fewer wavefronts than these leave HBM idle: five to eight ranks with 8, 8, 5 and 6
    of them up to 72 MiB copied took 1.02 - 1.2 of the time."""
    for ranks, least in ((3, 18), (4, 16), (5, 14), (6, 12), (7, 8), (8, 8)):
        sizes = (89, 120, 200, 72 * ranks - 1, 72 * ranks, 72 * ranks + ranks, 640)
        for mib, value in zip(sizes, rule(*(waves(op, "bytes", ranks, m) for m in sizes))):
            assert value == (10 if ranks >= 7 and mib > 72 * ranks else least), (ranks, mib, value)


def test_no_wait_where_none_was_worth_it(rule):
    """An allreduce of bf16 and fewer than eight ranks: its additions are the wait (seven ranks with
    512 clocks more: 1.002 of the time, the same buffers again up to 1.010)."""
    sizes = (101, 113, 130, 149, 151, 700)
    asked = [f"cu_pauses({_lib.OP_ALLREDUCE}, {_lib.BF16}, {r}, {m << 20}ull)" for r in range(2, 8) for m in sizes]
    assert rule(*asked) == [0] * len(asked)
