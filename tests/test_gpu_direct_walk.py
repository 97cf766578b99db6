"""Direct contractions where their walk through the operands is long: in 128 x 128 tiles with offsets by table, over K
ranges of several table halves; with runs of k that lie far back from each other; with rows too far apart for 32-bit
offsets; with many indices. The bodies hold small whole numbers, so every sum is exact and in any order."""
import math
import random

import numpy as np
import pytest
import torch

from tal_common import C4, C8, R4, R8
from test_direct_walk import BACKWARDS, FAR, LARGE, SHORT_RUNS, high_rank, labels_of

pytestmark = pytest.mark.gpu


DTYPE = {R4: torch.float32, R8: torch.float64, C4: torch.complex64, C8: torch.complex128}


def matrix(body, labels, ext, rows, cols):
    """A body (its shape is the labels reversed) as a matrix in 64 bits."""
    order = [len(labels) - 1 - labels.index(x) for x in rows + cols]
    return body.view([ext[x] for x in labels][::-1]).permute(order).reshape(
        math.prod([ext[x] for x in rows]), -1).to(torch.complex128 if body.is_complex() else torch.float64).contiguous()


def check_batch(ts, dk, pattern, ext, body, h):
    """A hyper index that runs slowest in every tensor: one product per entry."""
    labels = labels_of(pattern)
    assert all(lab[-1] == h for lab in labels)
    part = [[b.view(ext[h], -1)[q] for b in body] for q in range(ext[h])]
    d, l, r = (lab[:-1] for lab in labels)
    k = [x for x in l if x in r]
    m, n = [x for x in d if x in l], [x for x in d if x in r]
    want = [matrix(p[0], d, ext, m, n) + matrix(p[1], l, ext, m, k) @ matrix(p[2], r, ext, k, n) for p in part]
    torch.cuda.synchronize()
    ten = [ts.Tensor(dk, [ext[x] for x in lab], ts.gpu_flat(0), ext=b.data_ptr()) for lab, b in zip(labels, body)]
    ts.check(ts.contract(pattern, *ten, alpha=1.0, accumulative=ts.YEP), "contract")
    for p, w in zip(part, want):
        assert torch.equal(matrix(p[0], d, ext, m, n), w)
    for t in ten:
        t.destruct()


def check(ts, dk, pattern, ext, largest=8):
    """largest: magnitude of the bodies' whole numbers; no sum may leave the kind's exact range."""
    print("[case] walk", dk, pattern, ext, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    labels = labels_of(pattern)

    def draw(n):
        x = torch.empty(n, dtype=torch.float32, device="cuda")
        return x.random_(-largest, largest + 1, generator=gen)

    body = []
    for lab in labels:
        n = math.prod(ext[x] for x in lab)
        body.append((torch.complex(draw(n), draw(n)) if dk in (C4, C8) else draw(n)).to(DTYPE[dk]))
    d, l, r = labels
    k = [x for x in l if x in r and x not in d]
    h = [x for x in d if x in l and x in r]
    if h:
        check_batch(ts, dk, pattern, ext, body, h[0])
        return
    m, n = [x for x in d if x in l], [x for x in d if x in r]
    total = math.prod(ext[x] for x in k) * largest ** 2 * (2 if dk in (C4, C8) else 1) + largest
    assert total < (2 ** 24 if dk in (R4, C4) else 2 ** 53)
    left = matrix(body[1], l, ext, m, k)
    want = matrix(body[0], d, ext, m, n) + (left.conj().resolve_conj() if "L+(" in pattern else left) @ matrix(
        body[2], r, ext, k, n)
    torch.cuda.synchronize()
    ten = [ts.Tensor(dk, [ext[x] for x in lab], ts.gpu_flat(0), ext=b.data_ptr()) for lab, b in zip(labels, body)]
    ts.check(ts.contract(pattern, ten[0], ten[1], ten[2], alpha=1.0, accumulative=ts.YEP), "contract")
    assert torch.equal(matrix(body[0], d, ext, m, n), want)
    for t in ten:
        t.destruct()


@pytest.mark.parametrize("dk", (R4, R8))
@pytest.mark.parametrize("case", SHORT_RUNS)
def test_short_runs_in_large_tiles(talsh_gpu, dk, case):
    check(talsh_gpu, dk, *case)


@pytest.mark.parametrize("case", BACKWARDS)
def test_runs_far_back(talsh_gpu, case):
    check(talsh_gpu, R8, *case)


@pytest.mark.parametrize("seed", range(6))
def test_high_ranks(talsh_gpu, seed):
    """Indices of extent 2, up to 20 of them in D: written in place or through D'."""
    ts = talsh_gpu
    d, l, r = high_rank(random.Random(seed))
    print("[case] high rank", d, l, r, flush=True)
    rng = np.random.default_rng(seed)
    body = [rng.integers(-8, 9, 2 ** len(x)).astype(np.float64) for x in (d, l, r)]
    k = [x for x in l if x not in d]
    m, n = [x for x in d if x in l], [x for x in d if x in r]

    def mat(i, labels, rows, cols):
        order = [len(labels) - 1 - labels.index(x) for x in rows + cols]
        return body[i].reshape([2] * len(labels)).transpose(order).reshape(2 ** len(rows), 2 ** len(cols))

    want = mat(0, d, m, n) + mat(1, l, m, k) @ mat(2, r, k, n)
    dev = [torch.from_numpy(b).cuda() for b in body]
    torch.cuda.synchronize()
    ten = [ts.Tensor(R8, [2] * len(x), ts.gpu_flat(0), ext=b.data_ptr()) for x, b in zip((d, l, r), dev)]
    pattern = "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))
    ts.check(ts.contract(pattern, ten[0], ten[1], ten[2], alpha=1.0, accumulative=ts.YEP), "contract")
    body[0] = dev[0].cpu().numpy()
    assert np.array_equal(mat(0, d, m, n), want)
    for t in ten:
        t.destruct()


@pytest.mark.parametrize("case", LARGE)
def test_large_operands(talsh_gpu, case):
    """2 GiB and more, within reach of a base that moves along k."""
    check(talsh_gpu, R8, *case)
    torch.cuda.empty_cache()


@pytest.mark.parametrize("dk,case", [(dk, i) for dk in FAR for i in range(len(FAR[dk]))])
def test_far_operands(talsh_gpu, dk, case):
    """Rows or contracted indices 64 MiB and more apart."""
    pattern, ext = FAR[dk][case]
    check(talsh_gpu, dk, pattern, ext, largest=1 if dk in (R4, C4) else 8)
    torch.cuda.empty_cache()


def test_more_rows_than_one_grid_holds(talsh_gpu):
    ts = talsh_gpu
    M = 1100000000
    print("[case] rows", M, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    L = torch.empty(2 * M, device="cuda").random_(-8, 9, generator=gen)
    R = torch.tensor([3.0, -2.0], device="cuda")
    D = torch.full((M,), 5.0, device="cuda")
    torch.cuda.synchronize()
    ten = [ts.Tensor(R4, d, ts.gpu_flat(0), ext=b.data_ptr()) for d, b in (([M], D), ([M, 2], L), ([2], R))]
    ts.check(ts.contract("D(a)+=L(a,k)*R(k)", *ten, alpha=1.0, accumulative=ts.YEP), "contract")
    for at in range(0, M, 1 << 28):  # a piece at a time
        b = slice(at, min(M, at + (1 << 28)))
        assert torch.equal(D[b], 5.0 + 3.0 * L[:M][b] - 2.0 * L[M:][b]), at
    for t in ten:
        t.destruct()
    torch.cuda.empty_cache()


def test_more_contracted_indices_than_one_launch_takes(talsh_gpu):
    """Longer than 2^31: ranges of 2^30 are summed one after the other. Sums of K products of -1, 0 and 1 stay far below
    2^24 (standard deviation 2/3 sqrt(K) = 31,000), so the result is exact."""
    ts = talsh_gpu
    dims = [65536, 33000]
    print("[case] contracted indices", dims, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    L, R = (torch.empty(dims[0] * dims[1], device="cuda").random_(-1, 2, generator=gen) for _ in range(2))
    D = torch.full((1,), 5.0, device="cuda")
    want = 5.0 - 2.0 * sum((L[at:at + (1 << 28)] * R[at:at + (1 << 28)]).sum(dtype=torch.float64).item()
                           for at in range(0, L.numel(), 1 << 28))
    torch.cuda.synchronize()
    ten = [ts.Tensor(R4, d, ts.gpu_flat(0), ext=b.data_ptr()) for d, b in (([], D), (dims, L), (dims, R))]
    ts.check(ts.contract("D()+=L(a,b)*R(a,b)", *ten, alpha=-2.0, accumulative=ts.YEP), "contract")
    assert D.item() == want
    for t in ten:
        t.destruct()
    torch.cuda.empty_cache()


def test_more_short_rows_than_one_grid_splits(talsh_gpu):
    """Fast math (bf16x6, exact for small whole numbers): 140 million rows of 8 contracted indices."""
    ts = talsh_gpu
    M, K = 140000000, 8
    print("[case] short rows", M, K, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    L = torch.empty(M * K, device="cuda").random_(-8, 9, generator=gen)
    R = torch.empty(K, device="cuda").random_(-8, 9, generator=gen)
    D = torch.full((M,), 5.0, device="cuda")
    torch.cuda.synchronize()
    ten = [ts.Tensor(R4, d, ts.gpu_flat(0), ext=b.data_ptr()) for d, b in (([M, 1], D), ([K, M], L), ([K, 1], R))]
    ts.check(ts.fast_math(True, ts.SPLIT_BF16X6), "fast math")
    try:
        ts.check(ts.contract("D(a,b)+=L(k,a)*R(k,b)", *ten, alpha=1.0, accumulative=ts.YEP), "contract")
    finally:
        ts.fast_math(False)
    for at in range(0, M, 1 << 24):
        b = slice(at, min(M, at + (1 << 24)))
        assert torch.equal(D[b], 5.0 + (L.view(M, K)[b] * R).sum(1)), at
    for t in ten:
        t.destruct()
    torch.cuda.empty_cache()
