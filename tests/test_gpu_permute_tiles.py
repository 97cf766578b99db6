"""Transposing copies and adds (tal_sh_amd/csrc/permute.hip) at the edges of their tiles: the written dimension around
32, 64 and 128 elements and their multiples, where element accesses change tile, the read one around 24 and 32, odd
extents (element accesses) and even ones, with a third dimension and an outer one.  Copies and real adds are the same
bits as numpy's; complex adds too, alpha's imaginary part being zero and its real part a power of two."""
import numpy as np
import pytest

from tal_common import C4, C8, R4, R8, tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dk", [R8, R4, C8, C4])
def test_permute_tile_edges(talsh_gpu, dk):
    ts = talsh_gpu
    for a in (23, 24, 33, 67):
        for b in (31, 32, 33, 63, 64, 65, 83, 128, 129, 193, 257):
            for pattern, src in (("D(b,a)%s=L(a,b)", [a, b]),
                                 ("D(b,c,a)%s=L(a,b,c)", [a, b, 5]),
                                 ("D(b,d,c,a)%s=L(a,d,c,b)", [a, 2, 3, b])):
                names = pattern[pattern.index("L(") + 2:-1].split(",")
                out = pattern[2:pattern.index(")")].split(",")
                dst = [src[names.index(x)] for x in out]
                L, D = tensor(dk, src, a), tensor(dk, dst, b)
                moved = L.reshape(src[::-1]).transpose([names[::-1].index(x) for x in out[::-1]]).reshape(-1)
                lt, dt = ts.Tensor(dk, src, 0, data=L), ts.Tensor(dk, dst, 0, data=D)
                for t in (lt, dt):
                    t.place(ts.gpu_flat(0))
                ts.check(ts.add(pattern % "+", dt, lt, alpha=0.5), pattern)
                assert dt.host_array().tobytes() == (D + moved * L.dtype.type(0.5)).tobytes(), (dk, pattern, src)
                ts.check(ts.copy(pattern % "", dt, lt), pattern)
                assert dt.host_array().tobytes() == moved.tobytes(), (dk, pattern, src)
                lt.destruct()
                dt.destruct()
