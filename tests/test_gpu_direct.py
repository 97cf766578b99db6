"""The direct contraction kernels (tal_sh_amd/csrc/direct_kernel.hpp) where they can go wrong: tile edges in m and n,
K below, at and past whole K steps, every operand layout, k linear, in runs and in short pieces, D stored along m, along
n and scattered, tiles split along K, batch entries, conjugation, operands that allow no wide load.

Every element is within the forward error bound of a K-term dot product in the kind's precision:
|got - want| <= c * ((K + 4) * |alpha| * sum |l||r| + |d|) * eps, c = 1 real, 4 complex (four real products and the
scale by alpha), against the same contraction in extended precision."""
import random

import numpy as np
import pytest

from tal_common import C4, C8, R4, R8, tensor

pytestmark = pytest.mark.gpu
EDGES = (1, 7, 16, 31, 33, 64, 65, 129)
DEPTHS = (1, 5, 8, 15, 16, 17, 31, 32, 33, 100)


def check(ts, dk, pattern, ext, seed, acc):
    d, l, r = [p[p.index("(") + 1:p.index(")")].split(",") for p in pattern.replace("+=", "*").split("*")]
    dims = [[ext[x] for x in t] for t in (d, l, r)]
    D, L, R = (tensor(dk, n, seed + i) for i, n in enumerate(dims))
    alpha = complex(0.5, -0.25) if dk in (C4, C8) else 0.5
    ten = []
    for n, a in zip(dims, (D, L, R)):
        t = ts.Tensor(dk, n, 0, data=a)
        t.place(ts.gpu_flat(0))
        ten.append(t)
    ts.check(ts.contract(pattern, ten[0], ten[1], ten[2], alpha=alpha, accumulative=acc), pattern)
    got = ten[0].host_array()
    for t in ten:
        t.destruct()
    wide = np.clongdouble if dk in (C4, C8) else np.longdouble
    lo, ro, do = (a.reshape(n[::-1]).astype(wide) for a, n in zip((L, R, D), (dims[1], dims[2], dims[0])))
    if "L+(" in pattern:
        lo = lo.conj()
    sub = "%s,%s->%s" % ("".join(l)[::-1], "".join(r)[::-1], "".join(d)[::-1])
    want = alpha * np.einsum(sub, lo, ro) + (do if acc else 0)
    size = abs(alpha) * np.einsum(sub, abs(lo), abs(ro))
    k = int(np.prod([ext[x] for x in set(l) & set(r) - set(d)] or [1]))
    eps = np.finfo(np.float64 if dk in (R8, C8) else np.float32).eps
    bound = (4 if dk in (C4, C8) else 1) * ((k + 4) * size + abs(do)) * eps
    assert np.all(abs(got - want.reshape(-1)) <= bound.reshape(-1)), (dk, pattern, ext, acc)


@pytest.mark.parametrize("dk", [R8, R4, C8, C4])
def test_direct_edges(talsh_gpu, dk):
    rng = random.Random(dk)
    forms = ["D(a,b)+=L(a,k)*R(k,b)", "D(a,b)+=L(k,a)*R(k,b)", "D(a,b)+=L(a,k)*R(b,k)", "D(a,b)+=L(k,a)*R(b,k)",
             "D(b,a)+=L(a,k)*R(k,b)", "D(a,b)+=L+(k,a)*R(b,k)"]
    for i in range(48):
        ext = {"a": rng.choice(EDGES), "b": rng.choice(EDGES), "k": rng.choice(DEPTHS)}
        check(talsh_gpu, dk, forms[i % len(forms)], ext, 3 * i, i // len(forms) % 2)


@pytest.mark.parametrize("dk", [R8, R4, C8, C4])
def test_direct_layouts(talsh_gpu, dk):
    cases = [("D(a,b,c,d)+=L(c,i,b,j)*R(d,j,a,i)", dict(a=9, b=7, c=11, d=8, i=6, j=10)),   # short runs of k
             ("D(a,b,c,d)+=L(c,i,b,j)*R(d,j,a,i)", dict(a=12, b=8, c=20, d=16, i=36, j=3)),  # runs of k past a step
             ("D(a,b,c,d)+=L(c,i,b,j)*R(d,j,a,i)", dict(a=5, b=6, c=7, d=9, i=33, j=34)),
             ("D(a,b)+=L(i,a,j)*R(i,j,b)", dict(a=40, b=33, i=37, j=5)),                     # one run in R, two in L
             ("D(a,b)+=L(i,a,j,e)*R(i,e,b,j)", dict(a=17, b=18, i=34, j=3, e=4)),            # three dims of k
             ("D(a,b,c)+=L(b,d,a)*R(d,c)", dict(a=21, b=40, c=24, d=50)),                    # D scattered
             ("D(a,b,h)+=L(a,k,h)*R(k,b,h)", dict(a=33, b=20, k=19, h=5)),                   # batch entries
             ("D(a,h,b)+=L(a,k,h)*R(k,h,b)", dict(a=16, b=9, k=40, h=3)),
             ("D(a,b)+=L(a,k)*R(k,b)", dict(a=130, b=70, k=2000)),                           # split along k
             ("D(a,b)+=L(k,a)*R(b,k)", dict(a=65, b=33, k=1999)),
             ("D(a,b)+=L(a)*R(b)", dict(a=65, b=130)),                                       # no k
             ("D(a,b,c,d,e,f)+=L(d,e,g,a)*R(g,f,b,c)", dict(a=4, b=5, c=6, d=7, e=3, f=4, g=9))]
    for i, (pattern, ext) in enumerate(cases):
        for acc in (0, 1):
            check(talsh_gpu, dk, pattern, ext, 100 + i, acc)
