"""Performance cases of the tensor-contraction path: what a TAL-SH program has the GPU do.

Each case is one pass through the library's public calls (talshTensorContract, talshTensorCopy, talshTensorAdd,
talshAmdBatchExecute, ...) on operands that are resident on the GPU, as in an iterative many-body solver:

  contract  one blocking talshTensorContract; `split` names the fast-math method of an R4 contraction, or is empty
  copy      one blocking talshTensorCopy (a permutation)
  update    a residual update, one blocking call after another: initialise, two permuted adds, scale, cut a block
            out, add it back elsewhere, squared norm
  batch     many small contractions collected once and executed in one call

Tensor bodies are torch tensors whose shape is the TAL-SH shape reversed (TAL-SH runs its first index fastest).
"""
import math
import random

import torch

import tal_sh_amd as ts

KINDS = {"R4": ts.R4, "R8": ts.R8, "C4": ts.C4, "C8": ts.C8}
DTYPES = {"R4": torch.float32, "R8": torch.float64, "C4": torch.complex64, "C8": torch.complex128}
BYTES = {"R4": 4, "R8": 8, "C4": 8, "C8": 16}
SPLITS = {"bf16x6": ts.SPLIT_BF16X6, "fp16x3": ts.SPLIT_FP16X3}

# Contraction patterns in use: the 32^4 and 96^4 headline contractions, the particle ladder, a matrix product, index
# transformations by a small matrix, a product over two indices of rank-3 tensors, rank-6 outer-like products, a
# hyper-contraction (h in all three tensors).
PATTERNS = (
    "D(a,b,c,d)+=L(c,i,b,j)*R(d,j,a,i)",
    "D(a,b,c,d)+=L(a,i,c,j)*R(j,b,i,d)",
    "D(a,b,i,j)+=L(a,b,c,d)*R(c,d,i,j)",
    "D(a,b)+=L(a,c)*R(c,b)",
    "D(a,b,c)+=L(b,d,a)*R(d,c)",
    "D(a,b,c,d)+=L(e,b)*R(a,e,c,d)",
    "D(a,b)+=L(c,a,d)*R(d,c,b)",
    "D(a,b,c,d,e,f)+=L(d,e,g,a)*R(g,f,b,c)",
    "D(a,b,h)+=L(a,k,h)*R(k,b,h)",
)
PERMUTATIONS = ("f,e,d,c,b,a", "c,f,b,e,a,d", "c,a,f,b,e,d", "d,c,b,a", "b,a,d,c", "c,d,a,b", "a,c,b", "c,b,a", "b,a")


def listed():
    def contract(name, pattern, ext, kind, alpha=1.0, acc=True, split=""):
        return {"name": name, "op": "contract", "pattern": pattern, "ext": ext, "kind": kind, "alpha": alpha,
                "acc": acc, "split": split}

    return [
        # a block of a blocked tensor: a few microseconds of work, so launches and the host path count
        contract("contract_small_r8", PATTERNS[0], "a=9,b=7,c=11,d=8,i=6,j=10", "R8", 0.5),
        # the 2 GFLOP contraction of the library's own benchmark
        contract("contract_32_r8", PATTERNS[0], "a=32,b=32,c=32,d=32,i=32,j=32", "R8"),
        # the headline contraction, full size
        contract("contract_96_r8", PATTERNS[1], "a=96,b=96,c=96,d=96,i=96,j=96", "R8"),
        # particle ladder of a coupled-cluster step: 53 virtual and 19 occupied orbitals, every extent odd
        contract("ladder_odd_r8", PATTERNS[2], "a=53,b=53,c=53,d=53,i=19,j=19", "R8", 0.5),
        # one index of a rank-3 tensor transformed to a basis of 24 (a shape of the reference's benchmark list)
        contract("transform_24_r8", PATTERNS[4], "a=312,b=312,c=24,d=312", "R8", 1.0, False),
        # single precision, ragged extents
        contract("contract_ragged_r4", PATTERNS[1], "a=66,b=57,c=61,d=70,i=63,j=58", "R4"),
        # the headline contraction in single precision by both fast-math methods, the second at a smaller size
        contract("contract_96_bf16x6", PATTERNS[1], "a=96,b=96,c=96,d=96,i=96,j=96", "R4", 1.0, True, "bf16x6"),
        contract("contract_72_fp16x3", PATTERNS[1], "a=72,b=72,c=72,d=72,i=72,j=72", "R4", 1.0, True, "fp16x3"),
        # complex amplitudes with a conjugated operand
        contract("contract_conj_c8", "D(a,b,c,d)+=L+(c,i,b,j)*R(d,j,a,i)", "a=44,b=40,c=45,d=42,i=40,j=43", "C8", 0.5),
        # full index reversal of a 134 MB tensor
        {"name": "reverse_16p6_r8", "op": "copy", "perm": PERMUTATIONS[0], "ext": "a=16,b=16,c=16,d=16,e=16,f=16",
         "kind": "R8"},
        # residual update, odd extents
        {"name": "update_odd_r4", "op": "update", "nv": 83, "no": 41, "kind": "R4"},
        # 4,096 contractions of ranks 2-4 with extents 2-24, planned once and executed every iteration
        {"name": "batch_4096_r8", "op": "batch", "tasks": 4096, "gen": 4104, "kind": "R8"},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _random_pattern(rng):
    """Labels of every operand in any order, as a general code produces them."""
    while True:
        rl, rr = rng.randint(2, 5), rng.randint(2, 5)
        nc = rng.randint(1, min(3, rl, rr))
        nl, nr = rl - nc, rr - nc
        if 2 <= nl + nr <= 6:
            break
    labels = [chr(ord("a") + i) for i in range(nl + nr + nc)]
    d, l, r = labels[:nl + nr], labels[:nl] + labels[nl + nr:], labels[nl:]
    for x in (d, l, r):
        rng.shuffle(x)
    return "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))


def _extents(rng, labels, product):
    """Extents around the `product`'s root, a fifth of the sets multiples of eight."""
    n = product ** (1.0 / len(labels))
    mult = rng.choice((1, 1, 1, 1, 8))
    return {x: max(2, mult * int(round(n * math.exp(rng.uniform(-0.6, 0.6)) / mult))) for x in labels}


def _ext_text(ext):
    return ",".join("%s=%d" % (x, ext[x]) for x in sorted(ext))


def draw(rng):
    op = rng.choice(("contract", "contract", "contract", "contract", "contract", "copy", "update", "batch"))
    if op == "copy":
        perm = rng.choice(PERMUTATIONS)
        kind = rng.choice(("R4", "R8", "C4", "C8"))
        vol = _log_uniform(rng, 1e4, 1e9 / BYTES[kind])
        ext = _extents(rng, sorted(perm.split(",")), vol)
        if math.prod(ext.values()) * BYTES[kind] > 2e9:
            return draw(rng)
        return {"op": "copy", "perm": perm, "ext": _ext_text(ext), "kind": kind}
    if op == "update":
        kind = rng.choice(("R4", "R8", "C4", "C8"))
        nv = int(_log_uniform(rng, 12, 140))
        return {"op": "update", "nv": nv, "no": max(4, int(nv * rng.uniform(0.25, 0.6))), "kind": kind}
    if op == "batch":
        return {"op": "batch", "tasks": int(_log_uniform(rng, 64, 2048)), "gen": rng.randrange(1 << 20),
                "kind": rng.choice(("R4", "R8"))}
    kind = rng.choice(("R8", "R8", "R8", "R4", "R4", "C8", "C4"))
    split = rng.choice(("", "bf16x6", "fp16x3")) if kind == "R4" else ""
    pattern = rng.choice(PATTERNS) if rng.random() < 0.5 else _random_pattern(rng)
    if kind[0] == "C" and rng.random() < 0.5:
        pattern = pattern.replace("=L(", "=L+(")
    labels = sorted(set(x for part in _labels(pattern) for x in part))
    top = 4e10 if kind[0] == "C" else 2e11
    while True:
        ext = _extents(rng, labels, _log_uniform(rng, 1e5, top))
        case = {"op": "contract", "pattern": pattern, "ext": _ext_text(ext), "kind": kind, "alpha": 0.5,
                "acc": rng.random() < 0.7, "split": split}
        if math.prod(ext.values()) <= 2 * top and work(case)["bytes"] <= 2e9:
            return case


def _labels(pattern):
    """Index labels of D, L and R."""
    return [part[part.index("(") + 1:part.index(")")].split(",")
            for part in pattern.replace("+=", "=").replace("*", "=").split("=")]


def _ext(case):
    return {x.split("=")[0]: int(x.split("=")[1]) for x in case["ext"].split(",")}


def _batch_tasks(case):
    """Contractions of a batch: D, L and R of rank 2-4, 1-2 contracted indices, extents 2-24, labels shuffled."""
    rng = random.Random(case["gen"])
    out = []
    while len(out) < case["tasks"]:
        rl, rr = rng.randint(2, 4), rng.randint(2, 4)
        nc = rng.randint(1, min(2, rl, rr))
        nl, nr = rl - nc, rr - nc
        if not 2 <= nl + nr <= 4:
            continue
        labels = [chr(ord("a") + i) for i in range(nl + nr + nc)]
        ext = {x: rng.randint(2, 24) for x in labels}
        d, l, r = labels[:nl + nr], labels[:nl] + labels[nl + nr:], labels[nl:]
        for x in (d, l, r):
            rng.shuffle(x)
        out.append((d, l, r, ext))
    return out


def _update_shapes(case):
    """Residual and amplitude extents, the block's extents and the offsets it is cut from and added to."""
    v, o = case["nv"], case["no"]
    block = [v // 2, v // 2 + 1, o // 2, o // 2 + 1]
    return [v, v, o, o], [o, o, v, v], block, [1, 0, o // 4, 1], [v // 4, 1, 0, o // 3]


def work(case):
    e = BYTES[case["kind"]]
    cplx = case["kind"][0] == "C"
    if case["op"] == "contract":
        ext = _ext(case)
        vd, vl, vr = (math.prod(ext[x] for x in part) for part in _labels(case["pattern"]))
        return {"bytes": e * (vd * (2 if case["acc"] else 1) + vl + vr),
                "flops": (8 if cplx else 2) * math.prod(ext.values())}
    if case["op"] == "copy":
        return {"bytes": 2 * e * math.prod(_ext(case).values()), "flops": 0}
    if case["op"] == "update":
        full, _, block, _, _ = _update_shapes(case)
        vol, small = math.prod(full), math.prod(block)
        # both inputs read, the residual written, the block written
        return {"bytes": e * (3 * vol + small), "flops": (22 if cplx else 7) * vol}
    nbytes = flops = 0
    for d, l, r, ext in _batch_tasks(case):
        nbytes += e * sum(math.prod(ext[x] for x in part) for part in (d, l, r))
        flops += 2 * math.prod(ext.values())
    return {"bytes": nbytes, "flops": flops}


class _Batch(ts.Batch):
    def __del__(self):
        self.destroy()


def _start():
    """The runtime, once per process; its buffer pool holds the temporaries of the calls."""
    if not _start.done:
        ts.check(ts.init(host_buf_size=1 << 26, dev_buffer_size=16 << 30), "talshInit")
        _start.done = True


_start.done = False


def _bodies(kind, seed, dims_list):
    """Bodies with elements uniform in [-1, 1], from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[kind]
    out = []
    for dims in dims_list:
        n = math.prod(dims)
        if dtype.is_complex:
            real = torch.float32 if dtype == torch.complex64 else torch.float64
            x = torch.view_as_complex(torch.rand(n, 2, generator=gen, device="cuda", dtype=real).mul_(2).sub_(1))
        else:
            x = torch.rand(n, generator=gen, device="cuda", dtype=dtype).mul_(2).sub_(1)
        out.append(x.view(list(dims)[::-1]))
    return out


def _tensor(kind, dims, body):
    return ts.Tensor(KINDS[kind], dims, ts.gpu_flat(0), ext=body.data_ptr())


def _inputs(case, seed):
    """The bodies a case starts from."""
    kind = case["kind"]
    if case["op"] == "contract":
        ext = _ext(case)
        return _bodies(kind, seed, [[ext[x] for x in part] for part in _labels(case["pattern"])])
    if case["op"] == "copy":
        ext = _ext(case)
        return _bodies(kind, seed, [[ext[x] for x in sorted(ext)]])
    if case["op"] == "update":
        full, rev, _, _, _ = _update_shapes(case)
        return _bodies(kind, seed, [rev, full])
    tasks = _batch_tasks(case)
    sizes = [[math.prod(t[3][x] for x in part) for part in t[1:3]] for t in tasks]
    # 256-byte aligned bodies, as the library's own pool gives them
    step = 256 // BYTES[kind]
    total = sum(-(-n // step) * step for pair in sizes for n in pair)
    return _bodies(kind, seed, [[total]])


def prepare(case, seed):
    _start()
    kind = case["kind"]
    split = case.get("split", "")
    ts.check(ts.fast_math(bool(split), SPLITS.get(split, ts.SPLIT_BF16X6)), "fast math")
    bodies = _inputs(case, seed)
    state = {"case": case, "bodies": bodies}
    if case["op"] == "contract":
        ext = _ext(case)
        dims = [[ext[x] for x in part] for part in _labels(case["pattern"])]
        state["tensors"] = [_tensor(kind, n, b) for n, b in zip(dims, bodies)]
    elif case["op"] == "copy":
        ext = _ext(case)
        order = case["perm"].split(",")
        src = [ext[x] for x in order]
        out = torch.empty([ext[x] for x in sorted(ext)][::-1], dtype=DTYPES[kind], device="cuda")
        state["bodies"] = bodies = [out, bodies[0].view(src[::-1])]
        state["tensors"] = [_tensor(kind, [ext[x] for x in sorted(ext)], out), _tensor(kind, src, bodies[1])]
        state["pattern"] = "D(%s)=L(%s)" % (",".join(sorted(ext)), ",".join(order))
    elif case["op"] == "update":
        full, rev, block, _, _ = _update_shapes(case)
        made = [torch.empty(list(n)[::-1], dtype=DTYPES[kind], device="cuda") for n in (full, block, [])]
        state["bodies"] = bodies = bodies + made
        state["tensors"] = [_tensor(kind, n, b) for n, b in zip((rev, full, full, block, []), bodies)]
    else:
        tasks = _batch_tasks(case)
        step = 256 // BYTES[kind]
        pad = lambda n: -(-n // step) * step  # noqa: E731
        src = bodies[0]
        dst = torch.zeros(sum(pad(math.prod(t[3][x] for x in t[0])) for t in tasks), dtype=DTYPES[kind],
                          device="cuda")
        state["bodies"] = [src, dst]
        state["tensors"] = []
        state["batch"] = _Batch()
        at, to = 0, 0
        for d, l, r, ext in tasks:
            dims = [[ext[x] for x in part] for part in (d, l, r)]
            n = [math.prod(x) for x in dims]
            dt = _tensor(kind, dims[0], dst[to:])
            lt = _tensor(kind, dims[1], src[at:])
            rt = _tensor(kind, dims[2], src[at + pad(n[1]):])
            to += pad(n[0])
            at += pad(n[1]) + pad(n[2])
            state["tensors"] += [dt, lt, rt]
            pattern = "D(%s)+=L(%s)*R(%s)" % (",".join(d), ",".join(l), ",".join(r))
            ts.check(state["batch"].add(pattern, dt, lt, rt, alpha=1.0, accumulative=ts.NOPE), "talshAmdBatchAdd")
    torch.cuda.synchronize()  # the bodies are written before the library's streams read them
    return state


def run(state):
    case, t = state["case"], state["tensors"]
    if case["op"] == "contract":
        ts.check(ts.contract(case["pattern"], t[0], t[1], t[2], alpha=case["alpha"],
                             accumulative=ts.YEP if case["acc"] else ts.NOPE), "talshTensorContract")
        return state["bodies"][0]
    if case["op"] == "copy":
        ts.check(ts.copy(state["pattern"], t[0], t[1]), "talshTensorCopy")
        return state["bodies"][0]
    if case["op"] == "update":
        _, _, _, cut, put = _update_shapes(case)
        integrals, amplitudes, residual, block, norm = t
        ts.check(ts.init_value(residual, 0.25), "talshTensorInit")
        ts.check(ts.add("D(a,b,i,j)+=L(i,j,a,b)", residual, integrals, alpha=1.0), "talshTensorAdd")
        ts.check(ts.add("D(a,b,i,j)+=L(b,a,j,i)", residual, amplitudes, alpha=-0.5), "talshTensorAdd")
        ts.check(ts.scale(residual, 0.75), "talshTensorScale")
        ts.check(ts.slice(block, residual, cut), "talshTensorSlice")
        ts.check(ts.insert(residual, block, put, accumulative=ts.YEP), "talshTensorInsert")
        ts.check(ts.norm2(norm, residual), "talshTensorNorm2")
        return state["bodies"][2:]
    ts.check(state["batch"].execute(), "talshAmdBatchExecute")
    return state["bodies"][1]


def _einsum(labels, left, right):
    """D of one contraction in 64 bits, as a body (reversed shape)."""
    d, l, r = ("".join(part)[::-1] for part in labels)
    return torch.einsum("%s,%s->%s" % (l, r, d), left, right)


def exact(case, seed):
    bodies = [b.to(torch.complex128 if b.is_complex() else torch.float64) for b in _inputs(case, seed)]
    if case["op"] == "contract":
        left = bodies[1].conj().resolve_conj() if "L+(" in case["pattern"] else bodies[1]
        out = case["alpha"] * _einsum(_labels(case["pattern"]), left, bodies[2])
        return out + bodies[0] if case["acc"] else out
    if case["op"] == "copy":
        ext = _ext(case)
        order = case["perm"].split(",")
        src = bodies[0].view([ext[x] for x in order][::-1])
        return torch.einsum("%s->%s" % ("".join(order)[::-1], "".join(sorted(ext))[::-1]), src).contiguous()
    if case["op"] == "update":
        _, _, block, cut, put = _update_shapes(case)
        box = lambda off: tuple(slice(o, o + n) for o, n in zip(off, block))[::-1]  # noqa: E731
        integrals, amplitudes = bodies
        residual = 0.25 + torch.einsum("baji->jiba", integrals) - 0.5 * torch.einsum("ijab->jiba", amplitudes)
        residual = residual * 0.75
        part = residual[box(cut)].clone()
        residual[box(put)] += part
        return [residual, part, (residual.abs() ** 2).sum().to(residual.dtype)]
    tasks = _batch_tasks(case)
    step = 256 // BYTES[case["kind"]]
    pad = lambda n: -(-n // step) * step  # noqa: E731
    src = bodies[0]
    dst = torch.zeros(sum(pad(math.prod(t[3][x] for x in t[0])) for t in tasks), dtype=src.dtype, device="cuda")
    at, to = 0, 0
    for d, l, r, ext in tasks:
        dims = [[ext[x] for x in part][::-1] for part in (d, l, r)]
        n = [math.prod(x) for x in dims]
        right = src[at + pad(n[1]):at + pad(n[1]) + n[2]].view(dims[2])
        dst[to:to + n[0]] = _einsum((d, l, r), src[at:at + n[1]].view(dims[1]), right).reshape(-1)
        to += pad(n[0])
        at += pad(n[1]) + pad(n[2])
    return dst
