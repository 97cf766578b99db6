"""Fast-math products of R4 tensors (bf16x6, fp16x3) at the edges of the pre-split path: fewer K steps than LDS stages,
partial steps, rows longer than a block keeps in registers, unaligned rows, partial tiles, a partial round of tiles cut
into K ranges, operands contiguous along k or along their rows, D in place or accumulated."""
import numpy as np
import pytest
import torch

from tal_common import R4

pytestmark = pytest.mark.gpu

# a, b, c of D(a,b)+=L(..)*R(..)
SIZES = [(1, 1, 1), (5, 3, 33), (257, 129, 31), (130, 70, 65), (255, 128, 97), (300, 260, 128), (96, 80, 8229),
         (70, 40, 16411), (2100, 2053, 515), (1537, 1281, 1030),
         (3000, 33, 48), (700, 600, 250), (300, 200, 2049)]
PATTERNS = ["D(a,b)+=L(c,a)*R(c,b)", "D(a,b)+=L(a,c)*R(b,c)", "D(b,a)+=L(a,c)*R(c,b)"]


@pytest.mark.parametrize("method", ("SPLIT_BF16X6", "SPLIT_FP16X3"))
@pytest.mark.parametrize("pattern", PATTERNS)
@pytest.mark.parametrize("size", SIZES)
def test_split_edges(talsh_gpu, method, pattern, size):
    ts = talsh_gpu
    print("[case]", method, pattern, size, flush=True)
    ext = dict(zip("abc", size))
    labels = [p[p.index("(") + 1:p.index(")")].split(",") for p in pattern.replace("+=", "*").split("*")]
    gen = torch.Generator().manual_seed(sum(size))
    # bodies start at an odd element for odd seeds, so that rows are not 16-byte aligned
    shift = size[2] % 2
    host = []
    for lab in labels:
        n = int(np.prod([ext[x] for x in lab]))
        host.append((torch.rand(n, generator=gen, dtype=torch.float32) * 2 - 1))
    dev = []
    for h in host:
        buf = torch.zeros(h.numel() + 4, dtype=torch.float32, device="cuda")
        buf[shift:shift + h.numel()] = h.cuda()
        dev.append(buf[shift:shift + h.numel()])
    torch.cuda.synchronize()
    tens = [ts.Tensor(R4, [ext[x] for x in lab], ts.gpu_flat(0), ext=d.data_ptr()) for lab, d in zip(labels, dev)]
    ts.check(ts.fast_math(True, getattr(ts, method)), "fast math")
    try:
        ts.check(ts.contract(pattern, tens[0], tens[1], tens[2], alpha=0.5, accumulative=ts.YEP), "contract")
    finally:
        ts.fast_math(False)
    got = dev[0].cpu().double()

    def mat(i, rows):  # operand i as (rows, c)
        x = host[i].double().view([ext[q] for q in labels[i]][::-1])
        return x.T if labels[i][0] == rows else x

    A, B = mat(1, "a"), mat(2, "b")
    want = 0.5 * A @ B.T
    mag = 0.5 * A.abs() @ B.abs().T
    k = size[2]
    # sums: at most one rounding per product plus a few; operands: 3 x 2^-22 of the row's (column's) largest each
    tol = (k + 24) * 2.0 ** -23 * mag
    if method == "SPLIT_FP16X3":
        tol = tol + 0.5 * 3 * 2.0 ** -22 * k * A.abs().max(1).values[:, None] * B.abs().max(1).values[None, :]
    order = (lambda m: m.T.reshape(-1)) if labels[0][0] == "a" else (lambda m: m.reshape(-1))
    old = host[0].double()
    tol = order(tol) + 2.0 ** -23 * (old.abs() + order(mag))
    assert ((got - old - order(want)).abs() <= tol).all()
