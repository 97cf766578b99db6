"""Tensors of many indices of extent 2: permutations take a block per 8 elements, more than one grid holds from 2^27
elements on. Values are whole numbers that FP32 holds."""
import pytest
import torch

from tal_common import R4

pytestmark = pytest.mark.gpu


def permuted_index(order):
    """For every element e of a tensor whose index i is the source's index order[i]: its place in the source."""
    e = torch.arange(1 << len(order), device="cuda", dtype=torch.int64)
    out = torch.zeros_like(e)
    for i, o in enumerate(order):
        out |= ((e >> i) & 1) << o
    return out


def body(rank):
    return (torch.arange(1 << rank, device="cuda", dtype=torch.int64) * 40503 % 4093 - 2046).to(torch.float32)


@pytest.mark.parametrize("rank,add", [(26, False), (27, False), (28, True)])
def test_reversal(talsh_gpu, rank, add):
    ts = talsh_gpu
    print("[case] reversal", rank, add, flush=True)
    src = body(rank)
    dst = torch.ones_like(src)
    torch.cuda.synchronize()
    lab = ["x%d" % i for i in range(rank)]
    d, s = (ts.Tensor(R4, [2] * rank, ts.gpu_flat(0), ext=x.data_ptr()) for x in (dst, src))
    labels = ",".join(lab), ",".join(lab[::-1])
    if add:
        ts.check(ts.add("D(%s)+=L(%s)" % labels, d, s, alpha=2.0), "add")
    else:
        ts.check(ts.copy("D(%s)=L(%s)" % labels, d, s), "copy")
    want = src[permuted_index(list(range(rank))[::-1])]
    assert torch.equal(dst, 2.0 * want + 1.0 if add else want)
    d.destruct()
    s.destruct()
    torch.cuda.empty_cache()


def test_contraction(talsh_gpu):
    """L of rank 28 is copied in another order before the product."""
    ts = talsh_gpu
    print("[case] contraction of rank 28", flush=True)
    free = ["x%d" % i for i in range(27)]
    left = free[::-2] + ["k"] + free[1::2]
    L = body(28)
    R = torch.tensor([3.0, -1.0, 2.0, 5.0], device="cuda")  # R(k,n), k first
    D = torch.zeros(1 << 28, device="cuda")
    torch.cuda.synchronize()
    ten = [ts.Tensor(R4, [2] * n, ts.gpu_flat(0), ext=x.data_ptr()) for n, x in ((28, D), (28, L), (2, R))]
    d = free[9:] + ["n"] + free[:9]
    ts.check(ts.contract("D(%s)+=L(%s)*R(k,n)" % (",".join(d), ",".join(left)), *ten, alpha=1.0,
                         accumulative=ts.YEP), "contract")
    e = torch.arange(1 << 28, device="cuda", dtype=torch.int64)
    at = torch.zeros_like(e)
    for i, x in enumerate(d):
        if x != "n":
            at |= ((e >> i) & 1) << left.index(x)
    n = (e >> d.index("n")) & 1
    want = L[at] * R[2 * n] + L[at | 1 << left.index("k")] * R[2 * n + 1]
    assert torch.equal(D, want)
    for t in ten:
        t.destruct()
    torch.cuda.empty_cache()
