"""Slots of the dense core's item list (trust_amd/csrc/core_items.h), on the CPU.

A row with at least t targets takes a slot from the back of the list; one with
more than 2048 also takes a slot per 2048 targets from the front.  The list has
to hold both ends at any t and any row lengths."""
import ctypes
import os
import random
import subprocess

import pytest

from conftest import ROOT

PART = 2048


@pytest.fixture(scope="module")
def slots(tmp_path_factory):
    d = tmp_path_factory.mktemp("core_items")
    src, so = d / "slots.cpp", d / "slots.so"
    src.write_text('#include "core_items.h"\n'
                   'extern "C" long long slots(long long rows, long long E) { return trust::core_item_slots(rows, E); }\n'
                   'extern "C" int part(void) { return trust::kCorePart; }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "trust_amd", "csrc"),
                    str(src), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    assert lib.part() == PART
    lib.slots.restype = ctypes.c_longlong
    return lambda rows, E: lib.slots(ctypes.c_longlong(rows), ctypes.c_longlong(E))


def used(degrees):
    """Slots taken by candidate rows of which every entry is a target."""
    return len(degrees) + sum(-(-d // PART) for d in degrees if d > PART)


def one_slot_list(t, E):
    """A size that counts a row at one end only."""
    return E // t + E // PART + 2


@pytest.mark.parametrize("t", [2, 384, 1024, 1025, 2048, 4096])
def test_both_ends_fit(slots, t):
    for n in (1, 2, 7, 6000):
        for d in range(t, max(t, 3 * PART) + 2):
            assert used([d]) * n <= slots(n, n * d), (t, n, d)
    rng = random.Random(t)
    for _ in range(200):
        rows = [rng.choice([t, max(t, PART), max(t, PART + 1), t + rng.randrange(3 * PART)]) for _ in range(50)]
        assert used(rows) <= slots(len(rows), sum(rows)), (t, rows)
        # entries of rows below t only add room
        assert used(rows) <= slots(len(rows), sum(rows) + rng.randrange(10 ** 6))


def test_one_slot_a_row_is_too_few():
    # 6000 rows over 2200 targets and 2100 candidate rows without any
    rows, E = [2200] * 6000, 6000 * 2200 + 2100 * 2100
    assert used(rows) + 2100 > one_slot_list(2048, E)
