"""Partial sums of products that are cut along K do not come from the buffer pool: with the pool all but full, a
contraction is accepted as before and gives the same bits."""
import pytest
import torch

from tal_common import C4, C8, R4, R8

pytestmark = pytest.mark.gpu
DTYPE = {R4: torch.float32, R8: torch.float64, C4: torch.complex64, C8: torch.complex128}


def fill_pool(ts, leave):
    """Tensors in the pool until `leave` bytes (a multiple of 1 MiB) are free in one range."""
    free = ts.load().talshDeviceBufferFreeSize(0, ts.DEV_NVIDIA_GPU)
    rows = (free - leave) >> 20
    return ts.Tensor(R8, [1 << 17, rows], ts.gpu_flat(0)) if rows > 0 else None


@pytest.mark.parametrize("dk,m,n,k,split", [(R8, 189, 278, 40001, None), (R4, 300, 400, 60000, None),
                                            (C4, 65, 70, 9000, None), (C8, 40, 50, 7777, None),
                                            (R4, 300, 260, 8192, "SPLIT_FP16X3"), (R4, 300, 260, 8192, "SPLIT_BF16X6")])
def test_full_pool(talsh_gpu, dk, m, n, k, split):
    ts = talsh_gpu
    print("[case] full pool", dk, m, n, k, split, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    L, R = (torch.rand(x * k, generator=gen, device="cuda", dtype=torch.float64).to(DTYPE[dk]) for x in (m, n))
    D = torch.zeros(m * n, dtype=DTYPE[dk], device="cuda")
    torch.cuda.synchronize()
    ten = [ts.Tensor(dk, d, ts.gpu_flat(0), ext=b.data_ptr()) for d, b in (([m, n], D), ([k, m], L), ([k, n], R))]
    # room for the planes of the fast-math operands alone: 2 bytes a value and plane, padded to 256 x 128 x 32
    planes = 3 if split == "SPLIT_BF16X6" else 2
    room = 0 if not split else planes * 2 * (512 + 384) * 8192 + (1 << 20)
    if split:
        ts.check(ts.fast_math(True, getattr(ts, split)), "fast math")
    try:
        got = []
        for full in (False, True):
            filler = fill_pool(ts, -(-room >> 20) << 20) if full else None
            ts.check(ts.contract("D(a,b)=L(k,a)*R(k,b)", *ten, alpha=1.0, accumulative=ts.NOPE), "contract")
            got.append(D.clone())
            if filler:
                filler.destruct()
        assert torch.equal(got[0], got[1])
    finally:
        if split:
            ts.fast_math(False)
        for t in ten:
            t.destruct()
