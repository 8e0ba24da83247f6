"""Mixed-radix passes where their launches have remainders: several rows (or
row pairs) to a workgroup and a last workgroup that is not full, in the
transforms, the right-hand sides (also with a forcing in x space) and whole
steps, FP64 and FP32, boxes other than 2 pi; short columns; and columns whose
slab spans more than 4 GB (64-bit offsets)."""

import numpy as np
import pytest

from helpers import kfields, random_x, rel_l2
from oracle import numpy_path as npth
from test_gpu_kernels import FIELDS, case, download_fields, hip, params_struct, upload_fields

pytestmark = pytest.mark.gpu

BOX = {2: (3.0, 2 * np.pi), 3: (1.5, 2 * np.pi, 4.0)}


def parameters(kind):
    p = {'nu': 1e-3}
    if kind == 'boussinesq':
        p.update(kappa=1e-3, boussinesq_direction='y')
    elif kind == 'mhd':
        p.update(eta=1e-3, rho0=1.5)
    return p


# 1215 and 1125 rows, two to a workgroup, last radix 4, 5 and 6; two passes of
# a short column.  FP32: the transforms' bound of 2e-6 grows by the largest
# wavenumber, which a derivative multiplies their rounding by.
@pytest.mark.parametrize("f32", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("kind", ["hydro", "boussinesq", "mhd"])
@pytest.mark.parametrize("shape", [(27, 45, 40), (25, 45, 50), (27, 45, 54), (1125, 20), (8, 12, 10)], ids=str)
def test_rhs_remainders(kind, shape, f32):
    hp = hip()
    nd, L = len(shape), BOX[len(shape)]
    case("mixed rhs", kind, shape, f32)
    p = parameters(kind)
    tol = 2e-6 * max(2 * np.pi / l * n / 3 for n, l in zip(shape, L)) if f32 else 1e-12
    kf = kfields(kind, shape, 31, L)
    ref = npth.rhs(kind, shape, kf, L, **dict(p))
    plan = hp.Plan(shape, L, hp.F32 if f32 else hp.F64)
    st = upload_fields(plan, kind, kf)
    dv = [plan.alloc_k() for _ in st]
    plan.rhs(params_struct(hp, kind, nd, p), st, dv)
    got = download_fields(plan, kind, nd, dv)
    for name in FIELDS[kind]:
        for c in range(len(ref[name])):
            assert rel_l2(got[name][c], ref[name][c]) < tol, (name, c)


# 35 members of 45 x 30: 1575 rows
@pytest.mark.parametrize("kind", ["hydro", "boussinesq", "mhd"])
def test_rhs_members(kind):
    hp = hip()
    shape, nb, L = (45, 30), 35, BOX[2]
    case("mixed rhs, members", kind)
    p = parameters(kind)
    prm = params_struct(hp, kind, 2, p)
    many, one = hp.Plan(shape, L, batch=nb), hp.Plan(shape, L)
    kfs = [kfields(kind, shape, 100 + 7 * m, L) for m in range(nb)]
    st = []
    for name in FIELDS[kind]:
        for c in range(len(kfs[0][name])):
            b = many.alloc_k()
            many.upload_k(b, np.stack([kf[name][c] for kf in kfs]))
            st.append(b)
    dv = [many.alloc_k() for _ in st]
    many.rhs(prm, st, dv)
    got = [many.download_k(b) for b in dv]
    for m in (0, 1, 17, nb - 1):
        s1 = upload_fields(one, kind, kfs[m])
        d1 = [one.alloc_k() for _ in s1]
        one.rhs(prm, s1, d1)
        for g, b in zip(got, d1):
            assert np.array_equal(g[m], one.download_k(b)), m
    ref = npth.rhs(kind, shape, kfs[nb - 1], L, **dict(p))
    flat = [a for name in FIELDS[kind] for a in ref[name]]
    for g, r in zip(got, flat):
        assert rel_l2(g[nb - 1], r) < 1e-12


# 1013 row pairs, four to a workgroup with three fields and one with one; 1013
# is prime, so no count of pairs divides it
@pytest.mark.parametrize("f32", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("nf", [1, 3, 16])
def test_transform_remainders(nf, f32):
    hp = hip()
    shape, L = (45, 45, 30), BOX[3]
    case("mixed transforms", nf, f32)
    plan = hp.Plan(shape, L, hp.F32 if f32 else hp.F64)
    tol = 2e-6 if f32 else 1e-14
    xs, ks = [plan.alloc_x() for _ in range(nf)], [plan.alloc_k() for _ in range(nf)]
    refs = []
    for i in range(nf):
        c = npth.Component(shape, L)
        x = random_x(shape, 70 + i)
        c['xspace'] = x
        refs.append(c['kspace'].copy())
        plan.upload_x(xs[i], x)
    plan.fwd_many(xs, ks)
    for i in range(nf):
        d = npth.Component(shape, L)
        d['kspace'] = refs[i]
        d.dealias()
        ref = d['kspace'].copy()
        assert rel_l2(plan.download_k(ks[i]), ref) < tol, i
        plan.upload_k(ks[i], ref)
        refs[i] = d['xspace'].copy()
    plan.bwd_many(ks, xs)
    for i in range(nf):
        assert rel_l2(plan.download_x(xs[i]), refs[i]) < tol, i


# steps, and a forcing in x space that joins the products on the mixed rows:
# equal to its transform given in k space, to rounding
@pytest.mark.parametrize("f32", [False, True], ids=["f64", "f32"])
@pytest.mark.parametrize("kind,shape,integ", [('hydro', (27, 45, 40), 'RK2mid'), ('mhd', (75, 90), 'RK2trap'),
                                              ('boussinesq', (25, 45, 50), 'RK2mid')], ids=str)
def test_steps(kind, shape, integ, f32):
    hp = hip()
    nd, L = len(shape), BOX[len(shape)]
    case("mixed steps", kind, shape, integ, f32)
    p = parameters(kind)
    kf = kfields(kind, shape, 55, L)
    ref = npth.run(kind, shape, kf, 2e-3, 3, integ, L, **dict(p))
    plan = hp.Plan(shape, L, hp.F32 if f32 else hp.F64)
    prm = params_struct(hp, kind, nd, p)
    code = hp.RK2MID if integ == 'RK2mid' else hp.RK2TRAP
    tol = 2e-5 if f32 else 1e-12
    bufs = [[plan.alloc_k() for name in FIELDS[kind] for _ in kf[name]] for _ in range(2)]
    st = upload_fields(plan, kind, kf)
    plan.step(code, prm, st, bufs[0], bufs[1], None, 3, 2e-3)
    got = download_fields(plan, kind, nd, st)
    for name in FIELDS[kind]:
        for c in range(len(ref[name])):
            assert rel_l2(got[name][c], ref[name][c]) < tol, (name, c)
    xf, kfc = [plan.alloc_x() for _ in range(nd)], [plan.alloc_k() for _ in range(nd)]
    for c in range(nd):
        plan.upload_x(xf[c], random_x(shape, 80 + c))
    plan.fwd_many(xf, kfc)
    none = [None] * (len(st) - nd)
    sa, sb = upload_fields(plan, kind, kf), upload_fields(plan, kind, kf)
    plan.step(code, prm, sa, bufs[0], bufs[1], None, 3, 2e-3, xforcing=xf + none)
    plan.step(code, prm, sb, bufs[0], bufs[1], None, 3, 2e-3, forcing=kfc + none)
    for a, b in zip(sa, sb):
        assert rel_l2(plan.download_k(a), plan.download_k(b)) < tol


def test_columns_over_4_gb():
    """Three plane waves through (2025, 2025, 300): the y columns of one z
    plane's workspace are 4.5 GB apart from first to last row.  Their sum and
    their coefficients are known, so no reference transform is needed."""
    torch = pytest.importorskip("torch")
    hp = hip()
    n = (2025, 2025, 300)
    case("columns over 4 GB", n)
    plan = hp.Plan(n, (2 * np.pi,) * 3)
    ky, kz, kxp = plan.kc_shape
    assert ky * n[0] * kxp * 16 > 2 ** 32
    waves = [((3, -5, 7), 0.75), ((-640, 650, 99), -1.25), ((600, 1, 0), 0.5)]   # (kz, ky, kx), amplitude
    ax = [torch.arange(m, dtype=torch.float64, device="cuda") for m in n]
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    for k, a in waves:
        # cos of the sum of three phases, from cosines and sines per axis, a
        # plane at a time
        ph = [2 * np.pi / m * ((q * t) % m) for m, q, t in zip(n, k, ax)]
        cz, sz, cy, sy = ph[0].cos(), ph[0].sin(), ph[1].cos(), ph[1].sin()
        c, s = ph[2].cos(), ph[2].sin()
        for i0 in range(0, n[0], 225):
            i = slice(i0, i0 + 225)
            czy = cz[i, None] * cy - sz[i, None] * sy
            szy = sz[i, None] * cy + cz[i, None] * sy
            x[i] += a * (czy[:, :, None] * c - szy[:, :, None] * s)
    kc = torch.full((ky, kz, kxp, 2), float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    plan.fwd(x.data_ptr(), kc.data_ptr())
    plan.sync()
    for k, a in waves:
        # a cosine is half a wave at k and half at -k, of which kx > 0 (both
        # for kx = 0) are stored
        for sgn in ([1, -1] if k[2] == 0 else [1]):
            at = (sgn * k[1] % ky, sgn * k[0] % kz, k[2], 0)
            assert abs(float(kc[at]) - a / 2) < 1e-13
            kc[at] -= a / 2
    assert float(kc.abs().amax()) < 1e-13
    for k, a in waves:
        for sgn in ([1, -1] if k[2] == 0 else [1]):
            kc[sgn * k[1] % ky, sgn * k[0] % kz, k[2], 0] += a / 2
    y = torch.full(n, float("nan"), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    plan.bwd(kc.data_ptr(), y.data_ptr())
    plan.sync()
    assert float(y.sub_(x).abs_().amax()) < 1e-12
