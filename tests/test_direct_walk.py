"""CPU tests of how the direct contraction kernels walk through their K steps (tal_sh_amd/csrc/direct_index.hpp)."""
import ctypes
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("walk") / "libdirect_walk.so")
    csrc = os.path.join(REPO, "tal_sh_amd", "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + csrc, "-I" + os.path.join(REPO, "include"),
                    os.path.join(csrc, "direct_args.cpp"), os.path.join(csrc, "plan.cpp"),
                    os.path.join(REPO, "tests", "cxx", "direct_walk_shim.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    return build(tmp_path_factory)


@pytest.mark.parametrize("ahead", (0, 1))
@pytest.mark.parametrize("kb", (8, 16, 32))
def test_table_halves_are_not_read_while_they_are_filled(walk, ahead, kb):
    """Waves of a workgroup are ordered by barriers only: what one writes between two of them, no other may read there."""
    for pf in (1, 2, 3):
        for n in (1, kb, 255, 256, 257, 511, 512, 513, 640, 768, 769, 840, 1024, 1025, 1279, 1280, 1281, 5000):
            assert walk.table_walk(n, kb, 256, pf, ahead) == 0, (n, kb, pf, ahead)


# Contractions in 128 x 128 tiles whose contracted indices lie in runs shorter than a K step (offsets by table, which
# these tiles read in the call that uses them) and reach past two halves of the table.
SHORT_RUNS = [("D(a,b)+=L(i,a,j)*R(i,j,b)", dict(a=65536, b=128, i=8, j=160)),
              ("D(a,b)+=L(i,a,j)*R(i,j,b)", dict(a=65500, b=121, i=9, j=113)),
              ("D(b,a,c)+=L(i,a,j)*R(b,j,c,i)", dict(a=127, b=201, c=301, i=11, j=97))]


def labels_of(pattern):
    return [x[x.index("(") + 1:x.index(")")].split(",") for x in pattern.replace("+=", "*").split("*")]


def variant(walk, pattern, ext, dk):
    """(mode, tile, K range) of a contraction on 256 compute units."""
    dims = [(ctypes.c_int * len(lab))(*[ext[x] for x in lab]) for lab in labels_of(pattern)]
    out = (ctypes.c_int * 3)()
    assert walk.direct_variant(pattern.encode(), *dims, dk, 256, out) == 0, (pattern, ext)
    return tuple(out)


@pytest.mark.parametrize("dk", (4, 8))
@pytest.mark.parametrize("case", SHORT_RUNS)
def test_short_runs_take_tables_in_large_tiles(walk, dk, case):
    mode, tile, krange = variant(walk, *case, dk)
    assert (mode, tile) == (2, 0) and krange > 512
