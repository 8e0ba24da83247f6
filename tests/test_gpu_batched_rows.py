"""Members of a batched plan do not touch each other in the plain transforms.

The x rows go two to a complex transform.  With an odd number of rows a
member's last row and the next member's first must not share one: each member
then equals its own plain plan bit for bit, and a member that has overflowed
leaves the others finite."""

import numpy as np
import pytest

from helpers import random_x
from test_gpu_kernels import case, hip

pytestmark = pytest.mark.gpu


# mixed-radix rows with one, two and eight row pairs to a workgroup, a row
# count that leaves most of a workgroup empty, the general row kernel (576),
# an even row count, and the size-specialised rows
@pytest.mark.parametrize("f32", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("batch,shape", [(3, (5, 20)), (33, (75, 90)), (301, (45, 30)), (700, (3, 40)), (64, (15, 360)),
                                         (2, (9, 576)), (8, (48, 48)), (5, (75, 64)), (90, (9, 128)), (3, (27, 256)),
                                         (40, (45, 512)), (1, (9, 64))], ids=str)
def test_members_are_independent(batch, shape, f32):
    hp = hip()
    case("batched rows", batch, shape, f32)
    L = (2 * np.pi, 3.0)
    prec = hp.F32 if f32 else hp.F64
    many, one = hp.Plan(shape, L, prec, batch=batch), hp.Plan(shape, L, prec)
    x = np.stack([random_x(shape, 100 + i) for i in range(batch)])
    bad = batch // 2
    if batch > 1:
        x[bad] = 1e30 if f32 else 1e300
        x[bad, -1, -1] = np.inf
    xd, kd, yd = many.alloc_x(), many.alloc_k(), many.alloc_x()
    many.upload_x(xd, x)
    many.fwd(xd, kd)
    many.bwd(kd, yd)
    k, y = many.download_k(kd), many.download_x(yd)
    x1, k1, y1 = one.alloc_x(), one.alloc_k(), one.alloc_x()
    for i in sorted({0, 1, bad - 1, bad + 1, batch - 1} & set(range(batch)) - ({bad} if batch > 1 else set())):
        one.upload_x(x1, x[i])
        one.fwd(x1, k1)
        one.bwd(k1, y1)
        assert np.array_equal(k[i], one.download_k(k1)), i
        assert np.array_equal(y[i], one.download_x(y1)), i
