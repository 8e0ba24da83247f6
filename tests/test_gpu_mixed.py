"""Mixed-radix passes (extents other than 64, 128, 256, 512) against the oracle.

The shapes cover every last radix of the x rows (4, 5, 6), plans of one, two
and three radices, rows without a mixed plan (the general row kernel), odd
row counts (the last row pair is half empty), partial column tiles, single
radix columns and the first-radix-12 reordering (16 x 12, 15 x 5).
"""

import numpy as np
import pytest

from helpers import kfields, random_x, rel_l2
from oracle import numpy_path as npth
from test_gpu_kernels import FIELDS, case, download_fields, hip, params_struct, upload_fields

pytestmark = pytest.mark.gpu

SHAPES = [(4, 2), (5, 4), (3, 6), (9, 10), (16, 36), (15, 48), (75, 90), (125, 50), (192, 54),
          (9, 576), (625, 20), (2, 200), (75, 96, 120), (27, 36, 40), (15, 9, 50), (10, 12, 54), (4, 45, 30)]


# Rounding: a transform of N points in P passes loses about eps sqrt(P) per
# pass with table twiddles, below 1e-15 (FP64) and 6e-7 (FP32) here; the
# bounds of the other transform tests (1e-14, 2e-6) stand.
@pytest.mark.parametrize("f32", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_transforms(shape, f32):
    hp = hip()
    L = (2 * np.pi,) * len(shape)
    case("mixed transforms", shape, f32)
    plan = hp.Plan(shape, L, hp.F32 if f32 else hp.F64)
    tol = 2e-6 if f32 else 1e-14
    xs, ks = [plan.alloc_x() for _ in range(3)], [plan.alloc_k() for _ in range(3)]
    refs = []
    for i in range(3):
        x = random_x(shape, 7 + i)
        c = npth.Component(shape, L)
        c['xspace'] = x
        refs.append(c['kspace'].copy())
        plan.upload_x(xs[i], x)
    plan.fwd_many(xs, ks)
    for i in range(3):
        got = plan.download_k(ks[i])
        d = npth.Component(shape, L)
        d['kspace'] = refs[i]
        d.dealias()
        ref = d['kspace'].copy()
        assert rel_l2(got, ref) < tol, i
        plan.upload_k(ks[i], ref)
        refs[i] = d['xspace'].copy()
    plan.bwd_many(ks, xs)
    for i in range(3):
        assert rel_l2(plan.download_x(xs[i]), refs[i]) < tol, i


@pytest.mark.parametrize("kind", ["hydro", "boussinesq", "mhd"])
@pytest.mark.parametrize("shape", [(75, 48), (45, 50), (25, 54), (90, 360), (9, 576), (15, 12, 40), (9, 10, 50),
                                   (12, 15, 54), (5, 27, 96)], ids=str)
def test_rhs(kind, shape):
    hp = hip()
    nd = len(shape)
    L = (2 * np.pi,) * nd
    p = {'nu': 1e-3}
    if kind == 'boussinesq':
        p.update(kappa=1e-3, boussinesq_direction='y')
    elif kind == 'mhd':
        p.update(eta=1e-3, rho0=1.5)
    case("mixed rhs", kind, shape)
    kf = kfields(kind, shape, 31, L)
    ref = npth.rhs(kind, shape, kf, L, **dict(p))
    plan = hp.Plan(shape, L)
    st = upload_fields(plan, kind, kf)
    dv = [plan.alloc_k() for _ in st]
    plan.rhs(params_struct(hp, kind, nd, p), st, dv)
    got = download_fields(plan, kind, nd, dv)
    for name in FIELDS[kind]:
        for c in range(len(ref[name])):
            assert rel_l2(got[name][c], ref[name][c]) < 1e-12, (name, c)
