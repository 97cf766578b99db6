"""Work queues of the batch kernel where they run dry: from one item to more items than the resident workgroups
start with.  The queues' counters are cleared by the launch itself, so executions follow one another with eager work in
between, each checked against the product in 64 bits."""
import numpy as np
import pytest

from tal_common import R4, R8, tensor

pytestmark = pytest.mark.gpu


def upload(ts, dk, dims, data):
    t = ts.Tensor(dk, dims, ts.gpu_flat(0))
    h = ts.Tensor(dk, dims, 0, data=data)
    lab = ",".join("i%d" % k for k in range(len(dims)))
    ts.check(ts.copy("D(%s)=L(%s)" % (lab, lab), t, h), "upload")
    h.destruct()
    return t


# (contractions, extent of a and b): items = contractions x ceil(extent / 64)^2
@pytest.mark.parametrize("dk", (R8, R4))
@pytest.mark.parametrize("ntask,ext", [(1, 5), (7, 33), (9, 64), (40, 65), (23, 600)])
def test_every_item_runs_once(talsh_gpu, dk, ntask, ext):
    ts = talsh_gpu
    k = 19
    # D's fastest index comes from L in every other contraction
    pats = ("D(a,b)+=L(a,k)*R(k,b)", "D(b,a)+=L(k,a)*R(b,k)")
    b, tasks = ts.Batch(), []
    for t in range(ntask):
        p = t % 2
        ld, rd = ([ext, k], [k, ext]) if p == 0 else ([k, ext], [ext, k])
        L, R = tensor(dk, ld, 2 * t + 1), tensor(dk, rd, 2 * t + 2)
        lm = L.astype(np.float64).reshape(ld, order="F")
        rm = R.astype(np.float64).reshape(rd, order="F")
        want = (lm @ rm) if p == 0 else (rm @ lm)
        mag = (abs(lm) @ abs(rm)) if p == 0 else (abs(rm) @ abs(lm))
        lt, rt = upload(ts, dk, ld, L), upload(ts, dk, rd, R)
        dt = ts.Tensor(dk, [ext, ext], ts.gpu_flat(0))
        assert b.add(pats[p], dt, lt, rt, alpha=1.0, accumulative=ts.YEP) == 0
        tasks.append((dt, lt, rt, want.reshape(-1, order="F"), mag.reshape(-1, order="F")))
    # k products summed in order, `reps` sums: |error| <= (k + reps) eps sum |l r| per element
    eps = 2.0 ** -52 if dk == R8 else 2.0 ** -23
    reps = 4
    for rep in range(1, reps + 1):
        print("[case] queues", dk, ntask, ext, rep, flush=True)
        assert b.execute() == 0
        for dt, _, _, want, mag in tasks:
            got = dt.host_array().astype(np.float64)
            assert (abs(got - rep * want) <= (k + reps) * eps * rep * mag).all(), rep
            dt.place(ts.gpu_flat(0))
    b.destroy()
