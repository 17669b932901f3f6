"""How the sweeps are dealt out over waves (csrc/hp_tiling.h), checked on the
host: every cell is walked by exactly one lane, narrow boxes fill their waves,
the launch fits the 2^32 threads of a grid for every box that can be created,
and choosing a segment length takes a bounded number of steps."""
import ctypes
import os
import subprocess

import pytest

from hydropad_amd import build

SRC = r"""
#include <vector>
#include "hp_tiling.h"
extern "C" {
long items(long npen, long nseg) { return hp::stream_items(npen, nseg); }
void item(unsigned wave, unsigned lane, unsigned npen, unsigned nseg, int* out)
{
    const hp::StreamItem i = hp::stream_item(wave, lane, npen, nseg);
    out[0] = i.active; out[1] = (int)i.pen; out[2] = (int)i.seg;
}
int seglen(int nax, long npen, int simds, int* tried)
{
    int n = 0;
    const int len = hp::stream_seglen(nax, simds, 3, [&](int nseg) { ++n; return hp::stream_items(npen, nseg); });
    *tried = n;
    return len;
}
void forms(const int* boxes, int n, int form, int blocks, int ncu, int* out)
{
    std::vector<hp::BatchShape> v;
    for (int i = 0; i < n; ++i, boxes += 5) v.push_back({boxes[0], boxes[1], boxes[2], boxes[3] != 0, boxes[4] != 0});
    const hp::FormTiling t = hp::form_tiling(v.data(), n, form, blocks, ncu);
    out[0] = t.chunks; out[1] = t.len;
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("tiling")
    (d / "rules.cpp").write_text(SRC)
    so = str(d / "rules.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", build.CSRC, str(d / "rules.cpp"), "-o", so],
                   check=True)
    L = ctypes.CDLL(so)
    L.items.restype = ctypes.c_long
    L.items.argtypes = [ctypes.c_long, ctypes.c_long]
    L.item.argtypes = [ctypes.c_uint] * 4 + [ctypes.POINTER(ctypes.c_int)]
    L.seglen.argtypes = [ctypes.c_int, ctypes.c_long, ctypes.c_int, ctypes.POINTER(ctypes.c_int)]
    return L


@pytest.mark.parametrize("npen", [9, 12, 16, 21, 31, 32, 33, 63, 64, 65, 100, 255, 256, 257, 1000])
@pytest.mark.parametrize("nseg", [1, 2, 6, 7, 8, 33])
def test_every_segment_of_every_pencil_once(rules, npen, nseg):
    out = (ctypes.c_int * 3)()
    seen = []
    waves = rules.items(npen, nseg)
    for wave in range(waves + 4):                   # the last block's waves past the end are idle
        for lane in range(64):
            rules.item(wave, lane, npen, nseg, out)
            assert 0 <= out[1] < npen and 0 <= out[2] < nseg
            if out[0]:
                assert wave < waves
                seen.append((out[1], out[2]))
    assert sorted(seen) == [(p, s) for p in range(npen) for s in range(nseg)]


def test_narrow_boxes_fill_their_waves(rules):
    """Over many segments at least half of the lanes have a pencil."""
    nseg = 10000
    for npen in range(9, 200):
        assert rules.items(npen, nseg) * 64 <= 2 * npen * nseg, npen


def largest(nx, ny):
    """Interior length of the longest (nx, ny, nz) box of fewer than 2^31 cells."""
    return ((1 << 31) - 1) // (nx * ny) - 6


def test_threads_fit_a_grid(rules):
    """One-cell segments, the shortest that can be asked for."""
    for n1 in (3, 4, 5, 7, 8, 9, 13, 16, 33, 64, 65, 100, 500):
        for n2 in (3, 4, 5, 8, 11, 22):
            nax = largest(n1 + 6, n2 + 6)
            assert rules.items(n1 * n2, nax) * 64 + 256 < 1 << 32, (n1, n2)


@pytest.mark.parametrize("nax", [3, 24, 25, 64, 100, 512, 100000, largest(9, 9)])
def test_segment_length_takes_few_steps(rules, nax):
    tried = ctypes.c_int()
    for npen in (9, 64, 4096, 1 << 18):
        n = rules.seglen(nax, npen, 1024, ctypes.byref(tried))
        assert 1 <= n <= min(nax, 24), npen
        assert tried.value <= 24, npen


def test_each_form_of_a_batch_is_dealt_out_by_itself(rules):
    """A launch of a batch holds the boxes of one form (precision and gamma =
    5/3 or not), so the others do not lengthen its segments."""
    def tiling(boxes, g53, mixed, blocks=1024):
        flat = (ctypes.c_int * (5 * len(boxes)))(*[v for b in boxes for v in b])
        out = (ctypes.c_int * 2)()
        rules.forms(flat, len(boxes), 2 * mixed + g53, blocks, 256, out)
        return tuple(out)

    all_boxes = [(n, n, n, g53, mixed) for n in (32, 48, 64) for g53 in (0, 1) for mixed in (0, 1)]
    for g53 in (0, 1):
        for mixed in (0, 1):
            alone = [b for b in all_boxes if b[3:] == (g53, mixed)]
            assert tiling(all_boxes, g53, mixed) == tiling(alone, g53, mixed)
    for n in (64, 96, 128, 160):
        tried = ctypes.c_int()
        assert tiling([(n, n, n, 1, 0)], 1, 0)[1] == rules.seglen(n, n * n, 1024, ctypes.byref(tried))
