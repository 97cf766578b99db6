"""Direct contractions in 128 x 128 tiles with offsets by table, over K ranges of several table halves, and of operands
whose runs of k lie far back from each other. The bodies hold small whole numbers, so every sum is exact in both
precisions and in any order."""
import math
import random

import numpy as np
import pytest
import torch

from tal_common import R4, R8
from test_direct_walk import BACKWARDS, SHORT_RUNS, high_rank, labels_of

pytestmark = pytest.mark.gpu


def matrix(body, labels, ext, rows, cols):
    """A body (its shape is the labels reversed) as a matrix in 64 bits."""
    order = [len(labels) - 1 - labels.index(x) for x in rows + cols]
    return body.view([ext[x] for x in labels][::-1]).permute(order).reshape(
        math.prod([ext[x] for x in rows]), -1).to(torch.float64).contiguous()


def check(ts, dk, pattern, ext):
    print("[case] walk", dk, pattern, ext, flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    labels = labels_of(pattern)
    dtype = torch.float32 if dk == R4 else torch.float64
    # |sum| <= 64 K + 8: below 2^24 for every R4 case
    body = [torch.randint(-8, 9, (math.prod(ext[x] for x in lab),), generator=gen, device="cuda").to(dtype)
            for lab in labels]
    d, l, r = labels
    k = [x for x in l if x in r and x not in d]
    m, n = [x for x in d if x in l], [x for x in d if x in r]
    want = matrix(body[0], d, ext, m, n) + matrix(body[1], l, ext, m, k) @ matrix(body[2], r, ext, k, n)
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
