"""The indices that a tile of a K-major operand loads and stores in the split
Linear products (novann_amd/csrc/novaq_split_index.h), for every operand size up
to three tiles: runs stay inside the operand, and each index of a tile is stored
by exactly one lane, none before the tile or past the operand -- also where
fewer indices than a run are left of it.  CPU only (the header is built with
g++); the kernel runs the same functions."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("T", [2, 4])
def test_each_index_is_stored_once_and_none_outside(T, tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "split_index_dump")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "native", "split_index_dump.cpp")], check=True)
    out = subprocess.run([exe, str(T), str(3 * 16 * T + 1)], check=True, capture_output=True,
                         text=True).stdout
    tiles = moved = 0
    for line in out.splitlines():
        fields = line.split()
        count, i0 = int(fields[0]), int(fields[1])
        held = [tuple(map(int, e.split(","))) for e in fields[2:]]
        assert len(held) == 16 * T
        # what is loaded lies in the operand
        assert all(0 <= i0 + i < count for i, _ in held), (count, i0)
        # runs are T consecutive indices
        for r in range(16):
            assert [i - held[T * r][0] for i, _ in held[T * r:T * r + T]] == list(range(T))
        # what is stored: the tile's indices, each once
        stored = sorted(i for i, own in held if own)
        assert stored == list(range(min(16 * T, count - i0))), (count, i0)
        tiles += 1
        moved += any(i < 0 for i, _ in held)
    assert tiles > 0 and moved > 0  # runs that start before their tile occur
