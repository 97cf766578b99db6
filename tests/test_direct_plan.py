"""CPU tests of the direct contraction kernels' planning (tal_sh_amd/csrc/plan.cpp, direct_args.cpp).

Every form that the planner accepts is evaluated on the CPU with the addresses the kernel forms (the same inline
functions, k walked in the kernel's steps) and compared with the pattern's loop nest: ranks 1-5, labels in any order,
hyper indices, unit, odd and even extents, both ways round, straight from the tensors and on transposed copies."""
import ctypes
import os
import random
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KINDS = (4, 8, 14, 18)


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("direct") / "libdirect_shim.so")
    csrc = os.path.join(REPO, "tal_sh_amd", "csrc")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I" + csrc, "-I" + os.path.join(REPO, "include"),
                    os.path.join(csrc, "direct_args.cpp"), os.path.join(csrc, "plan.cpp"),
                    os.path.join(REPO, "tests", "cxx", "direct_shim.cpp"), "-o", out], check=True)
    lib = ctypes.CDLL(out)
    I, LL = ctypes.c_int, ctypes.c_longlong
    IP = ctypes.POINTER(I)
    lib.direct_check.argtypes = [ctypes.c_char_p, IP, IP, IP, I, I, I, I, IP]
    lib.direct_choice.argtypes = [I, LL, LL, LL, LL, I, ctypes.POINTER(LL)]
    return lib


def _ints(v):
    return (ctypes.c_int * max(1, len(v)))(*v)


def random_contraction(rng):
    """Pattern with shuffled labels, up to two hyper indices; extents 1-9 or multiples of 4, few elements in all."""
    while True:
        nl, nr, nk, nh = rng.randint(0, 3), rng.randint(0, 3), rng.randint(0, 3), rng.choice((0, 0, 0, 1, 2))
        if nl + nk + nh == 0 or nr + nk + nh == 0:
            continue
        labels = [chr(ord("a") + i) for i in range(nl + nr + nk + nh)]
        lu, ru, cc, hh = (labels[:nl], labels[nl:nl + nr], labels[nl + nr:nl + nr + nk], labels[nl + nr + nk:])
        ext = {x: rng.choice((1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 18, 20)) for x in labels}
        total = 1
        for x in labels:
            total *= ext[x]
        if total > 60000:
            continue
        d, l, r = lu + ru + hh, lu + cc + hh, ru + cc + hh
        for x in (d, l, r):
            rng.shuffle(x)
        return ("D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r)), [ext[x] for x in d],
                [ext[x] for x in l], [ext[x] for x in r])


@pytest.mark.parametrize("seed", range(4))
def test_forms_address_the_contraction(shim, seed):
    rng = random.Random(seed)
    seen = {}
    for _ in range(150):
        pat, dd, ld, rd = random_contraction(rng)
        for dk in KINDS:
            for form in (0, 1):
                for kstep in (8, 16, 32):
                    swap = rng.randint(0, 1)
                    info = (ctypes.c_int * 4)()
                    rc = shim.direct_check(pat.encode(), _ints(dd), _ints(ld), _ints(rd), dk, form, kstep, swap, info)
                    assert rc in (0, -1), (rc, pat, dd, ld, rd, dk, form, kstep, swap, list(info))
                    if rc == 0:
                        key = (form, info[0], info[1] > 1)
                        seen[key] = seen.get(key, 0) + 1
    # every way of addressing k, with element and wide loads, was met
    for form, modes in ((0, (0, 1, 2)), (1, (0,))):
        for mode in modes:
            assert seen.get((form, mode, False), 0) > 0, (form, mode, seen)
    assert seen.get((0, 0, True), 0) > 0 and seen.get((1, 0, True), 0) > 0, seen


@pytest.mark.parametrize("dk", KINDS)
def test_choice_covers_the_product(shim, dk):
    """Tiles cover M x N once, K ranges cover K once, partial sums stay within their bound."""
    rng = random.Random(dk)
    out = (ctypes.c_longlong * 9)()
    sizes = [1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 1000, 2809, 9216, 97344]
    for _ in range(400):
        M, N, K = (rng.choice(sizes) for _ in range(3))
        batch = rng.choice((1, 1, 1, 3, 300))
        rc = shim.direct_choice(dk, M, N, K, batch, rng.choice((1, 64, 256, 304)), out)
        assert rc == 0, (rc, M, N, K, batch, list(out))
        assert out[8] <= 64 << 20
