"""What a block of the deposition's tile kernel takes (lcode3d_amd/csrc/tile_order.hpp),
on the CPU: the words of the host's table come back as they went in at the limits
of their fields, and without a table (lcode_deposit_noalloc, whose grids are not
limited) a block's index is its tile, also beyond 65536 tiles (24-cell tiles from
6145^2 on)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(__file__), os.pardir, "lcode3d_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include "tile_order.hpp"
using namespace lcode;
static void show(DepBlock b) { std::printf("%d %d %d\n", b.tile, b.slot, b.part); }
int main() {
    for (int lin : {0, 65535, 65536, 66048, 1 << 20}) show(dep_block(false, 0, lin));
    for (int tile : {0, 7, 65535})
        for (int slot : {-1, 0, 32766})
            for (int part : {0, 1}) show(dep_block(true, dep_entry(tile, slot, part), 12345));
    std::printf("%d %d %d %d\n", dep_entries_fit(65536, 32767), dep_entries_fit(65537, 0),
                dep_entries_fit(1, 32768), dep_entries_fit(7396, 7396));
    return 0;
}
"""


def test_block_words(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "h.cpp", tmp_path / "h"
    src.write_text(HARNESS)
    subprocess.run([gxx, "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    got = [tuple(map(int, line.split())) for line in
           subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()]
    want = [(lin, -1, 0) for lin in (0, 65535, 65536, 66048, 1 << 20)]
    want += [(t, s, p) for t in (0, 7, 65535) for s in (-1, 0, 32766) for p in (0, 1)]
    assert got[:-1] == want
    assert got[-1] == (1, 0, 0, 1)


def test_kernel_takes_its_block_from_there():
    """The kernel decodes no word of its own, and the launch checks the fit."""
    with open(os.path.join(CSRC, "particles.hip")) as f:
        text = f.read()
    kernel = text[text.index("deposit_tile_kernel(DepositArgs a)"):]
    assert "dep_block(a.tile_order," in kernel
    assert ">> 16" not in kernel and "0xFFFF" not in kernel
    launch = text[text.index("int launch_deposit(const DepositArgs"):]
    assert "dep_entries_fit(" in launch
