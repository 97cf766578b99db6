"""Contractions whose contracted indices lie in short runs (offsets by table in the direct kernel): K around the sizes
of the table's halves and of a K step, cut into K ranges, with D accumulated or not and stored along either operand's
indices, against 64 bits."""
import numpy as np
import pytest

from tal_common import C4, C8, R4, R8, tensor

pytestmark = pytest.mark.gpu

K = [(1, 1), (3, 5), (3, 11), (5, 51), (4, 64), (3, 171), (7, 110), (2, 650), (37, 9), (33, 33)]
PATTERNS = ["D(a,b,c,d)+=L(c,i,b,j)*R(d,j,a,i)", "D(c,b,d,a)+=L(i,c,j,b)*R(j,d,i,a)"]


def upload(ts, dk, dims, data):
    t = ts.Tensor(dk, dims, ts.gpu_flat(0))
    h = ts.Tensor(dk, dims, 0, data=data)
    lab = ",".join("i%d" % k for k in range(len(dims)))
    ts.check(ts.copy("D(%s)=L(%s)" % (lab, lab), t, h), "upload")
    h.destruct()
    return t


@pytest.mark.parametrize("dk", (R4, R8, C4, C8))
@pytest.mark.parametrize("pattern", PATTERNS)
@pytest.mark.parametrize("k", K)
def test_table_offsets(talsh_gpu, dk, pattern, k):
    ts = talsh_gpu
    print("[case] tables", dk, pattern, k, flush=True)
    ext = {"a": 5, "b": 7, "c": 9, "d": 6, "i": k[0], "j": k[1]}
    labels = [x[x.index("(") + 1:x.index(")")].split(",") for x in pattern.replace("+=", "*").split("*")]
    dims = [[ext[x] for x in lab] for lab in labels]
    data = [tensor(dk, d, 7 * n + k[0]) for n, d in enumerate(dims)]
    wide = np.complex128 if dk in (C4, C8) else np.float64
    body = [x.astype(wide).reshape(d, order="F") for x, d in zip(data, dims)]
    spec = "%s,%s->%s" % tuple("".join(labels[n]) for n in (1, 2, 0))
    prod = np.einsum(spec, body[1], body[2])
    mag = np.einsum(spec, abs(body[1]), abs(body[2]))
    n = k[0] * k[1]
    # sums of n products (complex: 4 real ones each), alpha and the sum with D: one rounding each
    eps = 2.0 ** (-23 if dk in (R4, C4) else -52)
    tol = (n + 6) * (2 if dk in (C4, C8) else 1) * eps * (0.5 * mag + abs(body[0]))
    l, r = upload(ts, dk, dims[1], data[1]), upload(ts, dk, dims[2], data[2])
    for acc in (ts.YEP, ts.NOPE):
        d = upload(ts, dk, dims[0], data[0])
        ts.check(ts.contract(pattern, d, l, r, alpha=0.5, accumulative=acc), "contract")
        got = d.host_array().astype(wide).reshape(dims[0], order="F")
        want = 0.5 * prod + (body[0] if acc == ts.YEP else 0)
        assert (abs(got - want) <= tol).all(), acc
