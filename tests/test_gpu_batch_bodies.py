"""A batch whose operands' bodies change between executions: every execution works on what its tensors hold then. All
values are small whole numbers, so results are exact."""
import ctypes

import pytest
import torch

from tal_common import R4, R8

pytestmark = pytest.mark.gpu


def body(dtype, n, seed):
    return torch.randint(-4, 5, (n,), generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def rebuild(ts, t, dims, b):
    """The tensor's struct, destructed and constructed again over another caller-owned body."""
    ts.check(t.lib.talshTensorDestruct(t.ptr), "talshTensorDestruct")
    ts.check(t.lib.talshTensorClean(t.ptr), "talshTensorClean")
    ts.check(t.lib.talshTensorConstruct(t.ptr, t.dk, len(dims), (ctypes.c_int * len(dims))(*dims), ts.gpu_flat(0),
                                        b.data_ptr(), -1, None, 0.0, 0.0), "talshTensorConstruct")


@pytest.mark.parametrize("dk", (R8, R4))
@pytest.mark.parametrize("which", (0, 1, 2))
def test_rebuilt_operand(talsh_gpu, dk, which):
    ts = talsh_gpu
    print("[case] rebuilt operand", dk, which, flush=True)
    dtype = torch.float64 if dk == R8 else torch.float32
    dims = [[40, 24], [40, 31], [31, 24]]
    old = [body(dtype, d[0] * d[1], i) for i, d in enumerate(dims)]
    new = body(dtype, dims[which][0] * dims[which][1], 9)
    torch.cuda.synchronize()
    ten = [ts.Tensor(dk, d, ts.gpu_flat(0), ext=b.data_ptr()) for d, b in zip(dims, old)]
    b = ts.Batch()
    assert b.add("D(a,b)+=L(a,k)*R(k,b)", *ten, alpha=1.0, accumulative=ts.NOPE) == 0

    def product(bodies):  # bodies are column-major
        m = [x.double().view(d[::-1]) for x, d in zip(bodies, dims)]
        return (m[2] @ m[1]).reshape(-1)

    for _ in range(2):  # twice: the second one replays
        task = ts.Task()
        assert b.execute(task) == 0
        task.wait()
        task.destruct()
    assert torch.equal(old[0].double(), product(old))
    now = list(old)
    now[which] = new
    rebuild(ts, ten[which], dims[which], new)
    kept = old[0].clone()
    for rep in range(3):
        now[0].zero_()
        torch.cuda.synchronize()
        assert b.execute() == 0
        assert torch.equal(now[0].double(), product(now)), rep
    if which == 0:
        assert torch.equal(old[0], kept)  # the body that the tensor left
    b.destroy()
    for t in ten:
        t.destruct()


@pytest.mark.parametrize("dk", (R8, R4))
def test_added_while_it_runs(talsh_gpu, dk):
    """A contraction added behind an asynchronous execution: the plan is made anew, and both executions are whole."""
    ts = talsh_gpu
    print("[case] added while it runs", dk, flush=True)
    dtype = torch.float64 if dk == R8 else torch.float32
    n = 512
    bodies = [body(dtype, n * n, i) for i in range(4)]
    out = [torch.zeros(n * n, dtype=dtype, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    mk = lambda x: ts.Tensor(dk, [n, n], ts.gpu_flat(0), ext=x.data_ptr())  # noqa: E731
    ten, d = [mk(x) for x in bodies], [mk(x) for x in out]
    want = [(bodies[2 * i + 1].double().view(n, n) @ bodies[2 * i].double().view(n, n)).reshape(-1) for i in range(2)]
    for rep in range(3):
        b = ts.Batch()
        assert b.add("D(a,b)+=L(a,k)*R(k,b)", d[0], ten[0], ten[1], alpha=1.0, accumulative=ts.NOPE) == 0
        first, second = ts.Task(), ts.Task()
        assert b.execute(first) == 0
        assert b.add("D(a,b)+=L(a,k)*R(k,b)", d[1], ten[2], ten[3], alpha=1.0, accumulative=ts.NOPE) == 0
        assert b.execute(second) == 0
        for t in (first, second):
            t.wait()
            t.destruct()
        for o, w in zip(out, want):
            assert torch.equal(o.double(), w), rep
            o.zero_()
        torch.cuda.synchronize()
        b.destroy()
    for t in ten + d:
        t.destruct()
