"""The host code's rules on sizes (dwf_rules.h, plain C++), compiled here and
called through ctypes."""

import ctypes
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "dwf_rules.h"
extern "C" void split_blocks(int64_t nblk, int block, uint32_t* xy)
{
  const qdwf::Grid2 g = qdwf::split_blocks(nblk, block);
  xy[0] = g.x;
  xy[1] = g.y;
}
extern "C" int three_phase_sites(int ls, int64_t vh) { return qdwf::three_phase_sites(ls, vh); }
extern "C" int ring_pays(size_t bytes, int without) { return qdwf::ring_pays(bytes, without); }
extern "C" int z_tile(int xh, int by, int nz) { return qdwf::z_tile(xh, by, nz); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SOURCE)
    lib = str(d / "librules.so")
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "qlattice_amd", "csrc"),
                    str(d / "rules.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib)


@pytest.mark.parametrize("nelem", [1, 256, 257, 2**32 - 256, 2**32 - 255, 2**32, 2**32 + 4, 3 * 2**32, 2**35 + 12])
def test_a_launch_stays_below_the_grid_limit(rules, nelem):
    """128^3 x 64 Ls 8 has 2^32 QED elements: one thread each is one more than
    a grid dimension takes."""
    nblk = (nelem + 255) // 256
    xy = (ctypes.c_uint32 * 2)()
    rules.split_blocks(ctypes.c_int64(nblk), 256, xy)
    x, y = xy
    assert x * 256 < 2**32 and y < 65536
    assert nblk <= x * y < nblk + y
    if nelem <= 2**32 - 256:
        assert y == 1


def test_z_tiles_keep_whole_lines(rules):
    """A tile divides Z, and where the t neighbours are whole 128-byte lines (8
    sites) away without tiles they still are: 20^3 and 28^3 took tiles of 10
    and 7 planes, 500 and 686 sites."""
    for nz in range(2, 98, 2):
        for by in (1, 2, 4, 5, 6, 7, 9, 11):
            for xh in range(1, 25):
                b = rules.z_tile(xh, by, nz)
                assert nz % b == 0
                if xh * by * nz % 8 == 0:
                    assert xh * by * b % 8 == 0
                assert max(b * b / 97, 97 / (b * b)) <= max(nz * nz / 97, 97 / (nz * nz))
    assert [rules.z_tile(8, 4, 16), rules.z_tile(12, 6, 24), rules.z_tile(16, 4, 32)] == [8, 12, 8]
    assert [rules.z_tile(10, 5, 20), rules.z_tile(14, 7, 28)] == [20, 4]


@pytest.mark.parametrize("ls", [6, 8, 10, 12, 14, 16, 20, 24])
def test_sites_per_block_have_a_kernel(rules, ls):
    """Whole waves and the sites the kernels are built for at this Ls; 32 at Ls
    8 on every lattice (blocks of 16 lost up to 10% below 16^3x32)."""
    for vh in (8, 256, 4096, 8192, 8200, 13824, 65535, 65536, 442368):
        sb = rules.three_phase_sites(ls, ctypes.c_int64(vh))
        assert sb in ((8, 16) if ls == 24 else (16, 32) if ls <= 16 else (16,))
        assert sb * ls % 64 == 0
        if ls == 8:
            assert sb == 32
        if ls == 24:
            assert sb == (8 if vh > 8192 else 16)


def test_the_ring_waits_for_a_second_call(rules):
    """A new inverter's first call on a small host array, one transfer in and
    one out, makes no ring (its pinned memory takes longer than their copies);
    the next one does, and a large array at once."""
    mb = 1 << 20

    def pays(bytes_, without):
        return bool(rules.ring_pays(ctypes.c_size_t(bytes_), without))

    for size in (4, 12, 18, 25, 32):
        assert not pays(size * mb, 0) and not pays(size * mb, 1) and pays(size * mb, 2)
    assert pays(45 * mb, 0) and pays(96 * mb, 0)
