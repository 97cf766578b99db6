"""CPU tests of how the direct contraction kernels walk through their K steps (tal_sh_amd/csrc/direct_index.hpp)."""
import ctypes
import os
import random
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def build(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("walk") / "libdirect_walk.so")
    csrc = os.path.join(REPO, "tal_sh_amd", "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + csrc, "-I" + os.path.join(REPO, "include"),
                    os.path.join(csrc, "direct_args.cpp"), os.path.join(csrc, "plan.cpp"), os.path.join(csrc, "route.cpp"),
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


def lane_offsets(walk, pattern, ext, dk):
    dims = [(ctypes.c_int * len(lab))(*[ext[x] for x in lab]) for lab in labels_of(pattern)]
    modes = ctypes.c_int()
    return walk.lane_offsets(pattern.encode(), *dims, dk, ctypes.byref(modes)), modes.value


# R below 2 GiB, its next run of k far lower in memory than the end of the one before
BACKWARDS = [("D(a,b,c)+=L(i,a,j)*R(b,j,i,c)", dict(a=128, b=1500, c=2, i=20, j=3300)),
             ("D(a,b,c)+=L(i,a,j)*R(b,j,i,c)", dict(a=64, b=1600, c=4, i=18, j=2000)),
             ("D(a,b)+=L(i,a,j,k)*R(k,j,b,i)", dict(a=64, b=37, i=18, j=500, k=700)),
             ("D(a,b,c)+=L(i,a,j)*R(b,i,c,j)", dict(a=40, b=300, c=1200, i=33, j=21))]


@pytest.mark.parametrize("case", BACKWARDS)
def test_large_operands_stay_in_range_backwards(walk, case):
    """Every lane's 32-bit offset stays in its resource's range where the element is inside the operand."""
    assert lane_offsets(walk, *case, 8)[0] in (0, -1)


@pytest.mark.parametrize("dk", (4, 8, 14, 18))
def test_operands_up_to_2gib_stay_in_range(walk, dk):
    rng = random.Random(dk)
    seen = 0
    size = {4: 4, 8: 8, 14: 8, 18: 16}[dk]
    for _ in range(60):
        nl, nr, nk = rng.randint(1, 2), rng.randint(1, 2), rng.randint(1, 3)
        x = [chr(ord("a") + i) for i in range(nl + nr + nk)]
        lu, ru, cc = x[:nl], x[nl:nl + nr], x[nl + nr:]
        ext = {q: rng.choice((3, 9, 18, 33, 40)) for q in cc}
        ext.update({q: rng.choice((5, 16, 129)) for q in lu})
        ext.update({q: 2 for q in ru})
        # one index of R grows until R is just below 2 GiB, or a third of that
        grow, goal = rng.choice(ru + cc), rng.choice((1.0, 1.0, 0.34)) * (0x7FFFFF00 / size)
        rest = 1
        for q in ru + cc:
            rest *= ext[q] if q != grow else 1
        ext[grow] = max(1, int(goal / rest))
        k = 1
        for q in cc:
            k *= ext[q]
        left = 1
        for q in lu + cc:
            left *= ext[q]
        if k > 60000 or left * size > 0x7FFFFF00:
            continue
        l, r, d = lu + cc, ru + cc, lu + ru
        for q in (l, r, d):
            rng.shuffle(q)
        pattern = "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))
        rc, modes = lane_offsets(walk, pattern, ext, dk)
        assert rc in (0, -1), (rc, pattern, ext)
        seen |= modes
    assert seen & 7 == 7


def high_rank(rng):
    """A contraction of many indices of extent 2: the labels of D, L and R."""
    nl, nr, nk = rng.choice(((9, 9, 6), (10, 9, 6), (10, 10, 6), (8, 9, 3)))
    x = ["x%d" % i for i in range(nl + nr + nk)]
    l, r, d = x[:nl] + x[nl + nr:], x[nl:], x[:nl + nr]
    for q in (l, r, d):
        rng.shuffle(q)
    return d, l, r


def test_high_ranks_are_addressable(walk):
    """Contractions of many short indices: where D's rows or columns are too many numbers to be written in place, D'
    takes their place and the product is a plain one."""
    rng = random.Random(5)
    seen = set()
    for _ in range(60):
        d, l, r = high_rank(rng)
        pattern = "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))
        dims = [(ctypes.c_int * len(lab))(*[2] * len(lab)) for lab in (d, l, r)]
        in_place = ctypes.c_int()
        for dk in (4, 8, 14, 18):
            assert walk.mat_addressable(pattern.encode(), *dims, dk, ctypes.byref(in_place)) == 1, pattern
        seen.add(in_place.value)
    assert seen == {0, 1}


# Operands whose rows or contracted indices lie 64 MiB or more apart: tall ones along their rows, long ones along k.
MODE_FAR, ROUTE_COPIES = 3, 1
FAR = {8: [("D(a,q)+=L(a,p)*R(p,q)", dict(a=8400000, p=37, q=24)),      # 16-byte loads, a partial K step
           ("D(a,q)+=L(a,p)*R(q,p)", dict(a=8400001, p=16, q=47)),      # element loads, a partial tile
           ("D(q,a)+=L(p,q)*R(a,p)", dict(a=8400003, p=5, q=70)),       # K below a step
           ("D(a,q)+=L(a,p)*R(p,q)", dict(a=8388610, p=33, q=130)),
           ("D(a,b,c,q)+=L(a,b,c,p)*R(p,q)", dict(a=210, b=200, c=201, p=40, q=9)),
           ("D(a,b)+=L(k,a)*R(k,b)", dict(a=130, b=30, k=2200001)),     # both along k, element loads
           ("D(a,b)+=L(k,a)*R(k,b)", dict(a=130, b=140, k=2200002)),
           ("D(a,b)+=L(k,a)*R(b,k)", dict(a=129, b=31, k=2200000)),
           ("D(b,a)+=L(a,k)*R(k,b)", dict(a=30, b=135, k=2150002)),
           ("D(a,b,h)+=L(a,k,h)*R(k,b,h)", dict(a=8400001, b=5, k=7, h=3))],  # batch entries
       4: [("D(a,q)+=L(a,p)*R(p,q)", dict(a=16800000, p=35, q=24)),
           ("D(a,q)+=L(a,p)*R(q,p)", dict(a=16800001, p=64, q=33)),
           ("D(a,b)+=L(k,a)*R(k,b)", dict(a=130, b=33, k=4400001)),
           ("D(a,b)+=L(k,a)*R(b,k)", dict(a=130, b=33, k=4400000))],
       18: [("D(a,q)+=L(a,p)*R(p,q)", dict(a=4200001, p=35, q=24)),
            ("D(a,b)+=L(k,a)*R(k,b)", dict(a=130, b=33, k=1100001))],
       14: [("D(a,q)+=L(a,p)*R(p,q)", dict(a=8400001, p=35, q=24)),
            ("D(a,b)+=L(k,a)*R(b,k)", dict(a=130, b=33, k=2200001))]}


# Operands of 2 GiB and more whose tiles are reached by 32-bit offsets from a 64-bit base.
LARGE = [("D(a,b)+=L(a,k)*R(k,b)", dict(a=100003, b=37, k=2700)), ("D(a,b)+=L(a,k)*R(k,b)", dict(a=100002, b=38, k=2702)),
         ("D(b,a)+=L(k,a)*R(b,k)", dict(a=2701, b=65, k=100003)), ("D(a,b)+=L(a,k)*R(k,b)", dict(a=4000, b=70, k=70001))]


def test_large_operands_take_a_moving_base(walk):
    for pattern, ext in LARGE:
        dims = [(ctypes.c_int * len(lab))(*[ext[x] for x in lab]) for lab in labels_of(pattern)]
        out = (ctypes.c_int * 3)()
        assert walk.route_of(pattern.encode(), *dims, 8, 256, out) in (0, ROUTE_COPIES) and out[0] == 1, (pattern, ext)


@pytest.mark.parametrize("dk", (4, 8, 14, 18))
def test_far_operands_take_the_direct_kernels(walk, dk):
    for pattern, ext in FAR[dk]:
        dims = [(ctypes.c_int * len(lab))(*[ext[x] for x in lab]) for lab in labels_of(pattern)]
        out = (ctypes.c_int * 3)()
        assert walk.route_of(pattern.encode(), *dims, dk, 256, out) == ROUTE_COPIES, (pattern, ext)
        assert out[0] == MODE_FAR, (pattern, ext)


@pytest.mark.parametrize("dk", (4, 8, 14, 18))
def test_launches_hold_fewer_threads_than_a_grid_can(walk, dk):
    """Products of up to 2^31 rows: every unit is launched once, in grids of fewer than 2^32 threads."""
    LL = ctypes.c_longlong
    walk.launch_units.restype, walk.launch_units.argtypes = LL, [LL, LL, ctypes.c_uint]
    walk.choose_units.argtypes = [ctypes.c_int, LL, LL, LL, ctypes.c_int, ctypes.POINTER(LL)]
    for M in (1, 1000, 536870913, 1073741825, 1100000000, 2147483520):
        for N in (1, 24, 100):
            for swap in (0, 1):
                units = LL()
                assert walk.choose_units(dk, N if swap else M, M if swap else N, 2, 256, ctypes.byref(units)) == 1
                assert 0 < units.value < 2 ** 31
                for threads in (256, 512):
                    at = 0
                    while at < units.value:
                        n = walk.launch_units(units.value, at, threads)
                        assert n > 0 and n * threads < 2 ** 32
                        at += n
                    assert at == units.value and walk.launch_units(units.value, at, threads) == 0


def test_k_past_one_launch(walk):
    for d, l, r, ext in (([], ["a", "b"], ["a", "b"], dict(a=65536, b=33000)),
                         (["m", "n"], ["a", "m", "b"], ["b", "n", "a"], dict(a=65536, b=33000, m=2, n=3))):
        pattern = "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))
        dims = [(ctypes.c_int * max(1, len(lab)))(*[ext[x] for x in lab]) for lab in (d, l, r)]
        in_place = ctypes.c_int()
        for dk in (4, 8, 14, 18):
            assert walk.mat_addressable(pattern.encode(), *dims, dk, ctypes.byref(in_place)) == 1


# Products by tile shape (its number in direct_tiles; complex kinds have one shape for 0 and 1): a, b and k with partial
# tiles and partial K steps, 16-byte and element loads, and with k of two dimensions (a, b, i, j).
LAYOUTS = ["D(a,b)+=L(a,k)*R(k,b)", "D(a,b)+=L(k,a)*R(k,b)", "D(b,a)+=L(a,k)*R(b,k)", "D(a,b)+=L(k,a)*R(b,k)"]
RUN_LAYOUTS = ["D(a,b)+=L(i,a,j)*R(i,j,b)", "D(a,b)+=L(i,a,j)*R(b,i,j)", "D(b,a)+=L(a,i,j)*R(j,b,i)"]
SMALL = [(129, 65, 259), (15, 1, 1), (33, 31, 7)]
TILES = {
    8: {0: [(16390, 2052, 70), (16389, 2051, 259)], 1: [(4100, 2052, 70), (4097, 2051, 133)],
        2: [(8200, 66, 70), (8201, 65, 133)], 3: [(130, 66, 70)] + SMALL},
    4: {0: [(4100, 8196, 260), (8197, 8199, 67)], 1: [(8200, 2052, 132), (8200, 2052, 130)],
        2: [(2052, 2052, 68), (8200, 66, 70)], 3: [(132, 68, 68)] + SMALL},
    18: {0: [(2500, 1598, 259)], 2: [(8200, 66, 70)], 3: SMALL},
    14: {0: [(4100, 2052, 70), (4097, 2051, 133)], 2: [(8200, 66, 70), (8201, 65, 133)], 3: [(130, 66, 70)] + SMALL}}
TILE_RUNS = {
    8: {0: [(16390, 2052, 33, 4), (16390, 2052, 36, 6)], 1: [(4097, 2052, 17, 3), (8200, 1030, 16, 5), (4097, 2052, 3, 11)],
        2: [(8200, 66, 17, 3), (8200, 66, 20, 7), (8200, 66, 5, 51)],
        3: [(131, 31, 17, 3), (130, 34, 20, 7), (129, 33, 5, 51)]},
    4: {0: [(16390, 1030, 33, 4)], 1: [(8200, 2052, 17, 3)], 2: [(8200, 66, 33, 4), (8200, 68, 36, 5), (8200, 66, 17, 5)],
        3: [(131, 31, 33, 4), (132, 36, 36, 7), (129, 33, 5, 51)]},
    18: {0: [(65537, 33, 5, 51)], 2: [(8200, 66, 17, 3), (8200, 66, 3, 51)], 3: [(131, 31, 17, 3), (129, 33, 3, 51)]},
    14: {0: [(4097, 2052, 33, 4), (4097, 2052, 36, 7), (33000, 33, 5, 51)],
         2: [(8200, 66, 17, 3), (8200, 66, 20, 7), (8200, 66, 5, 51)],
         3: [(131, 31, 17, 3), (130, 34, 20, 7), (129, 33, 5, 51)]}}


@pytest.mark.parametrize("dk", (4, 8, 14, 18))
def test_tiles_are_chosen(walk, dk):
    """The shapes above take the tiles they are listed under, with both load widths, and walk or look up their runs."""
    wide = {4: 4, 8: 2, 14: 2, 18: 1}[dk]
    out = (ctypes.c_int * 3)()

    def route(pattern, ext):
        dims = [(ctypes.c_int * len(lab))(*[ext[x] for x in lab]) for lab in labels_of(pattern)]
        return walk.route_of(pattern.encode(), *dims, dk, 256, out)

    assert set(TILES[dk]) == set(TILE_RUNS[dk]) == ({0, 1, 2, 3} if dk in (4, 8) else {0, 2, 3})
    for tile, sizes in TILES[dk].items():
        widths = set()
        for size in sizes:
            for pattern in LAYOUTS:
                assert route(pattern, dict(zip("abk", size))) == ROUTE_COPIES, (pattern, size)
                # as D(b,a), two shapes of equal cost may change places
                assert out[0] == 0 and (out[2] == tile or pattern == LAYOUTS[2]), (pattern, size)
                widths.add(out[1])
        assert widths == {1, wide}, (tile, widths)
    modes = set()
    for tile, sizes in TILE_RUNS[dk].items():
        for size in sizes:
            for pattern in RUN_LAYOUTS[:2]:
                assert route(pattern, dict(zip("abij", size))) == 0, (pattern, size)
                assert out[2] == tile and out[0] in (1, 2), (pattern, size)
                modes.add((tile, out[0]))
    assert {m for _, m in modes} == {1, 2}
