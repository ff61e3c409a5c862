"""Kernels at the sizes where they can go wrong: tile edges, remainders, the smallest problems.

Each is compared with the CPU oracle (or numpy) in FP64.
"""
import numpy as np
import pytest

from oracle import fem
from opencmp_amd import _lib as L
from opencmp_amd.mesh import unit_cube, unit_square

pytestmark = pytest.mark.gpu


def core():
    from opencmp_amd import core as C
    return C


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


# ------------------------------------------------------------------------------------------ load vectors

POLY = {2: [0.3, -1.0, 2.0, 0.7, -0.4, 1.1], 3: [0.3, -1.0, 2.0, 0.5, 0.7, -0.4, 1.1, 0.2, -0.6, 0.9]}


def poly(dim):
    c = POLY[dim]
    if dim == 2:
        return lambda x, y: c[0] + c[1] * x + c[2] * y + c[3] * x * x + c[4] * x * y + c[5] * y * y
    return lambda x, y, z: (c[0] + c[1] * x + c[2] * y + c[3] * z + c[4] * x * x + c[5] * y * y + c[6] * z * z +
                            c[7] * x * y + c[8] * x * z + c[9] * y * z)


# 2, 18 and 98 triangles, 6, 48 and 162 tetrahedra: one element tile of 16 and less, several with a rest
@pytest.mark.parametrize('dim,n', [(2, 1), (2, 3), (2, 7), (3, 1), (3, 2), (3, 3)])
@pytest.mark.parametrize('order', [1, 2, 3])
def test_load_vector_tiles(gpu_ctx, dim, n, order):
    """Volume loads of every order on tile edges, written and then accumulated, against the oracle's
    quadrature (both rules exact for the data, so the difference is rounding: sums of at most 64 points and
    24 elements, 1e-14 relative)."""
    C = core()
    hm = unit_square(n) if dim == 2 else unit_cube(n)
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.H1(order)])
    f = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, POLY[dim]))])
    f.Assemble()
    cs = fem.Compound([fem.Space(fem.Topology(hm), 'H1', order)])
    ref = fem.assemble_source(cs, 0, poly(dim))
    assert rel(f.vec.cpu().numpy(), ref) < 1e-14
    # nine terms: a second launch adds to the first's vector
    f9 = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, POLY[dim]), coef=k + 1.0) for k in range(9)])
    f9.Assemble()
    assert rel(f9.vec.cpu().numpy(), 45.0 * ref) < 1e-14
    f.Assemble()
    assert rel(f.vec.cpu().numpy(), ref) < 1e-14


def test_load_vector_blocks_and_facets(gpu_ctx):
    """A compound space with terms on some blocks only, a boundary source on one marker, and no terms at
    all: untouched blocks are zero."""
    C = core()
    hm = unit_square(5)
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.VectorH1(2), C.H1(1)])
    t = fem.Topology(hm)
    cs = fem.Compound([fem.Space(t, 'H1', 2, ncomp=2), fem.Space(t, 'H1', 1)])
    right = hm.marker_mask('right')
    f = C.LinearForm(fes, [C.Source(1, (L.FN_POLY2, POLY[2])), C.BndSource(0, right, fn=(L.FN_CONST, (2.0,)))])
    f.Assemble()
    ref = fem.assemble_source(cs, 0, [lambda x, y: 0 * x, poly(2)]) + \
        fem.assemble_bnd_source(cs, 0, 2.0, right)
    assert rel(f.vec.cpu().numpy(), ref) < 1e-14
    only = C.LinearForm(fes, [C.BndSource(0, right, fn=(L.FN_CONST, (2.0,)))])
    only.Assemble()
    assert rel(only.vec.cpu().numpy(), fem.assemble_bnd_source(cs, 0, 2.0, right)) < 1e-14
    none = C.LinearForm(fes, [])
    none.vec.fill_(1.0)
    none.Assemble()
    assert float(none.vec.abs().max()) == 0.0


# ------------------------------------------------------------------------------------------ SpMV row blocks


def fan(n):
    """n triangles around one vertex: its P3 row has 6 n + 1 nonzeros per component (at most 256 triangles,
    the space's colours)."""
    from opencmp_amd.mesh import Mesh
    t = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(t), np.sin(t)], 1)
    k = np.arange(n)
    el = np.stack([np.zeros(n, int), 1 + k, 1 + (k + 1) % n], 1).astype(np.int32)
    return Mesh(np.concatenate([[[0.0, 0.0]], ring]), el, el[:, 1:].copy(), np.zeros(n, np.int32), ['rim'])


def shuffled(m, seed):
    """The mesh with its vertices renumbered at random: neighbouring rows share few columns."""
    from opencmp_amd.mesh import Mesh
    p = np.random.default_rng(seed).permutation(m.nv)
    c = np.empty_like(m.coords)
    c[p] = m.coords
    return Mesh(c, p[m.elems].astype(np.int32), p[m.bnd_facets].astype(np.int32), m.bnd_markers, m.bnd_names)


@pytest.mark.parametrize('name,make,order', [
    ('one block', lambda: unit_square(1), 1),
    ('several small blocks', lambda: unit_square(23), 3),
    ('large blocks', lambda: unit_cube(15), 3),
    ('large blocks of long rows', lambda: unit_cube(14), 3),
    ('rows of 4,503 nonzeros', lambda: fan(250), (3, 3)),
    ('rows of 2,042 nonzeros, longer than a block', lambda: fan(170), (3, 2)),
    ('rows of 2,030 nonzeros, each a block', lambda: fan(169), (3, 2)),
    ('blocks with too many distinct columns', lambda: shuffled(unit_square(310), 1), 2),
])
def test_spmv_row_blocks(gpu_ctx, name, make, order):
    """y = A x against scipy on the same values: rows of at most 4,503 terms, 1e-14 relative."""
    import torch
    C = core()
    order, ncomp = order if isinstance(order, tuple) else (order, 1)
    fes = C.FESpace(C.Mesh(make(), gpu_ctx), [C.H1(order)] * ncomp)
    a = C.BilinearForm(fes, [C.Vol(k, i, i, coef=c) for i in range(ncomp) for k, c in (('gradgrad', 1.0), ('mass', 3.0))])
    a.Assemble()
    x = np.random.default_rng(2).standard_normal(fes.ndof)
    y = gpu_ctx.zeros(fes.ndof)
    a.mult(torch.tensor(x, device='cuda'), y)
    ref = a.to_scipy() @ x
    assert rel(y.cpu().numpy(), ref) < 1e-14
    if fes.ndof > 1000:
        # FP32 blocks inside FP64 refinement
        f = C.LinearForm(fes, [C.Source(0, (L.FN_CONST, (1.0,)))])
        f.Assemble()
        pre = C.Preconditioner(a, 'local', precision='mixed')
        pre.Update()
        u = C.GridFunction(fes)
        r = C.solve(a, f.vec, u.vec, pre, 'CG', tol=1e-10, precision='mixed')
        assert r.converged and r.rel_residual <= 1e-10


def test_spmv_infinite_x(gpu_ctx):
    """An infinite entry of x reaches the rows that have its column, and no other: every column in turn
    (rows in blocks, so the first and last thread of a block see its neighbours' nonzeros)."""
    import torch
    C = core()
    fes = C.FESpace(C.Mesh(unit_square(13), gpu_ctx), [C.H1(3)])
    a = C.BilinearForm(fes, [C.Vol('gradgrad', 0, 0), C.Vol('mass', 0, 0)])
    a.Assemble()
    rp, col = a.pattern()
    has = np.zeros((fes.ndof, fes.ndof), bool)
    has[np.repeat(np.arange(fes.ndof), np.diff(rp)), col] = True
    finite = torch.empty((fes.ndof, fes.ndof), dtype=torch.bool, device='cuda')
    x = torch.ones(fes.ndof, dtype=torch.float64, device='cuda')
    y = gpu_ctx.zeros(fes.ndof)
    for j in range(fes.ndof):
        x[j] = float('inf')
        a.mult(x, y)
        finite[:, j] = torch.isfinite(y)
        x[j] = 1.0
    assert np.array_equal(finite.cpu().numpy(), ~has)


@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
def test_spmv_rows_without_nonzeros(gpu_ctx, precision):
    """FGMRES multiplies by the operator without untouched block pairs: with terms on one of two
    components, half of its rows are empty. The solution equals that of the one component alone."""
    C = core()
    hm = unit_square(9)
    sol = []
    for comps in ([C.H1(2, 'left'), C.H1(2, 'left')], [C.H1(2, 'left')]):
        fes = C.FESpace(C.Mesh(hm, gpu_ctx), comps)
        a = C.BilinearForm(fes, [C.Vol('gradgrad', 0, 0), C.Vol('mass', 0, 0)])
        f = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, POLY[2]))])
        a.Assemble()
        f.Assemble()
        pre = C.Preconditioner(a, 'local', precision=precision)
        pre.Update()
        u = C.GridFunction(fes)
        r = C.solve(a, f.vec, u.vec, pre, 'FGMRes', tol=1e-12, precision=precision, restart=60, inner_tol=1e-4)
        assert r.converged
        sol.append(u.vec.cpu().numpy())
    n = len(sol[1])
    assert rel(sol[0][:n], sol[1]) < 1e-10 and not sol[0][n:].any()


# rows without nonzeros before, behind and between the others, whole blocks of them, blocks of 4096 nonzeros
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('make,order,live', [
    (lambda: unit_square(1), 1, (0, 1)), (lambda: unit_square(12), 1, (1, 0, 0)), (lambda: unit_square(40), 2, (0, 1, 0)),
    (lambda: unit_square(30), 3, (0, 0, 1)), (lambda: unit_cube(15), 3, (1, 0)),
])
def test_spmv_some_rows_without_nonzeros(gpu_ctx, make, order, live, precision):
    """As above with the live component first, last or in the middle: the solution solves the system, by
    scipy's product with the same matrix. The solver's residual is at most 1e-12 |f|; the two products
    differ by the rounding of rows of at most 100 terms, below 100 * 1.1e-16 | |A| |u| |."""
    C = core()
    hm = make()
    k = live.index(1)
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.H1(order if c else 1) for c in live])
    a = C.BilinearForm(fes, [C.Vol('gradgrad', k, k, coef=1e-4), C.Vol('mass', k, k)])
    f = C.LinearForm(fes, [C.Source(k, (L.FN_POLY2, POLY[hm.dim]))])
    a.Assemble()
    f.Assemble()
    pre = C.Preconditioner(a, 'local', precision=precision)
    pre.Update()
    u = C.GridFunction(fes)
    r = C.solve(a, f.vec, u.vec, pre, 'FGMRes', tol=1e-12, precision=precision, restart=60, inner_tol=1e-4)
    assert r.converged
    off = fes.block_offsets()
    v, b, A = u.vec.cpu().numpy(), f.vec.cpu().numpy(), a.to_scipy()
    assert not v[:off[k]].any() and not v[off[k + 1]:].any()
    assert np.linalg.norm(b - A @ v) <= 1e-12 * np.linalg.norm(b) + 1.1e-14 * np.linalg.norm(abs(A) @ abs(v))


# ------------------------------------------------------------------------------------------ row gather


@pytest.mark.parametrize('make,order', [
    (lambda: unit_square(1), 1), (lambda: unit_square(6), 2), (lambda: unit_cube(2), 1), (lambda: unit_cube(3), 3),
    (lambda: fan(16), 3),     # exactly one unit of 16 entries for the centre's row
    (lambda: fan(17), 2),     # and one entry more
    (lambda: fan(200), 3),    # a block grown to one row's 200 entries
    (lambda: fan(250), 3),    # and to 250: 33 KB of LDS
])
def test_gather_units(gpu_ctx, make, order):
    """Matrix values against the oracle's quadrature, written, accumulated in a second launch (33 terms)
    and with coefficients that make terms share a table or not (relative Frobenius 1e-13)."""
    C = core()
    hm = make()
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.H1(order), C.H1(1)])
    t = fem.Topology(hm)
    cs = fem.Compound([fem.Space(t, 'H1', order), fem.Space(t, 'H1', 1)])

    def ref(g, m, c):
        A = fem.Assembler(cs)
        fem.assemble_volume(A, [dict(kind='grad_grad', trial=0, test=0, coef=g),
                                dict(kind='mass', trial=0, test=0, coef=m),
                                dict(kind='mass', trial=1, test=0, coef=c)])
        return A.matrix().data

    def gpu(terms):
        a = C.BilinearForm(fes, terms)
        assert 'assemble_h1_gather' in _timed(gpu_ctx, a.Assemble)
        return a.values()

    G, M, X = (lambda c: C.Vol('gradgrad', 0, 0, coef=c)), (lambda c: C.Vol('mass', 0, 0, coef=c)), \
        (lambda c: C.Vol('mass', 1, 0, coef=c))
    assert rel(gpu([G(2.0), M(3.0), X(0.5)]), ref(2.0, 3.0, 0.5)) < 1e-13
    assert rel(gpu([G(2.0), G(2.0), M(0.5), X(0.5)]), ref(4.0, 0.5, 0.5)) < 1e-13
    assert rel(gpu([G(2.0), G(1.0), M(0.5), X(0.25)]), ref(3.0, 0.5, 0.25)) < 1e-13
    assert rel(gpu([G(1.0)] * 31 + [M(1.0), X(1.0)]), ref(31.0, 1.0, 1.0)) < 1e-13


def _timed(ctx, f):
    """The classes of the kernels that f launches."""
    ctx.timing_report()
    ctx.timing(True)
    f()
    ctx.timing(False)
    return ctx.timing_report()


def test_element_scatter_of_long_rows(gpu_ctx):
    """A row whose 250 entries of 20 values are more than LDS takes: the elements are scattered colour by
    colour, also in a call of 33 terms that adds to the first 32 (against the oracle as above)."""
    C = core()
    hm = fan(250)
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.H1(3), C.H1(3)])
    t = fem.Topology(hm)
    cs = fem.Compound([fem.Space(t, 'H1', 3), fem.Space(t, 'H1', 3)])
    for n in (1, 31):
        a = C.BilinearForm(fes, [C.Vol('gradgrad', 0, 0, coef=2.0)] * n + [C.Vol('mass', 1, 1, coef=3.0),
                                                                           C.Vol('mass', 1, 0, coef=0.5)])
        assert 'assemble_h1_gather' not in _timed(gpu_ctx, a.Assemble)
        A = fem.Assembler(cs)
        fem.assemble_volume(A, [dict(kind='grad_grad', trial=0, test=0, coef=2.0 * n),
                                dict(kind='mass', trial=1, test=1, coef=3.0),
                                dict(kind='mass', trial=1, test=0, coef=0.5)])
        assert rel(a.values(), A.matrix().data) < 1e-13


def _field_case(C, ctx, gm, hm, t, order, seed, ncomp=1):
    """A grid function of random values on a space of its own, and the oracle's evaluation of it."""
    import torch
    fes = C.FESpace(gm, [C.H1(order, ncomp=ncomp)])
    v = np.random.default_rng(seed).standard_normal(fes.ndof)
    gf = C.GridFunction(fes, torch.tensor(v, device=ctx.torch_device))
    return gf, fem.GridFunctionEval(fem.Space(t, 'H1', order, ncomp=ncomp), v)


def _assert_volume(C, fes, cs, terms, ref):
    a = C.BilinearForm(fes, terms)
    a.Assemble()
    A = fem.Assembler(cs)
    fem.assemble_volume(A, ref, qdeg=8)     # exact: P2 test and trial, a P3 weight
    r = A.matrix().data
    assert rel(a.values(), r) < 1e-13


def test_tables_of_the_weighting_field(gpu_ctx):
    """Forms of one space with the same list of fields, whose last term is weighted by the P1 field in
    one and by the P2 or P3 field in the others: each has tables of its own."""
    C = core()
    hm = unit_square(4)
    gm, t = C.Mesh(hm, gpu_ctx), fem.Topology(hm)
    fes, cs = C.FESpace(gm, [C.H1(2)]), fem.Compound([fem.Space(t, 'H1', 2)])
    f = [_field_case(C, gpu_ctx, gm, hm, t, p, p) for p in (1, 2, 3)]
    for k in (0, 1, 2, 0):
        terms = [C.Vol('mass', 0, 0, weight_gf=(gf, 0, L.WEIGHT_FIELD)) for gf, _ in f] + \
                [C.Vol('gradgrad', 0, 0, coef=2.0, weight_gf=(f[k][0], 0, L.WEIGHT_FIELD))]
        ref = [dict(kind='mass', trial=0, test=0, coef=('field', e, 1, 1.0)) for _, e in f] + \
              [dict(kind='grad_grad', trial=0, test=0, coef=('field', f[k][1], 1, 2.0))]
        _assert_volume(C, fes, cs, terms, ref)


@pytest.mark.parametrize('path', ['row gather', 'element scatter', 'load vector'])
def test_tables_of_a_later_field_space(gpu_ctx, path):
    """Spaces of fields that come and go, each of another order than the one before it and mostly at its
    address: no table of an earlier one is taken."""
    import gc
    C = core()
    hm = unit_square(4)
    gm, t = C.Mesh(hm, gpu_ctx), fem.Topology(hm)
    fes, cs = C.FESpace(gm, [C.H1(2)]), fem.Compound([fem.Space(t, 'H1', 2)])
    for order in (1, 3, 2, 1):
        gf, e = _field_case(C, gpu_ctx, gm, hm, t, order, order)
        if path == 'row gather':
            _assert_volume(C, fes, cs, [C.Vol('gradgrad', 0, 0, coef=2.0, weight_gf=(gf, 0, L.WEIGHT_FIELD))],
                           [dict(kind='grad_grad', trial=0, test=0, coef=('field', e, 1, 2.0))])
        elif path == 'element scatter':
            # a wind and a weight in one term; the quadrature follows the weight's order
            w, ew = _field_case(C, gpu_ctx, gm, hm, t, 1, 7, ncomp=2)
            _assert_volume(C, fes, cs, [C.Vol('conv', 0, 0, wind_gf=(w, w.space.comp_blocks[0]),
                                              weight_gf=(gf, 0, L.WEIGHT_FIELD))],
                           [dict(kind='conv', trial=0, test=0, coef=('field', e, 1, 1.0), wind=ew)])
            del w
        else:
            b = C.LinearForm(fes, [C.Source(0, field_gf=(gf, 0), weight_gf=(gf, 0, L.WEIGHT_FIELD))])
            b.Assemble()
            lam, w = fem.simplex_rule(2, 8)
            phi, _ = fem.ref_basis('H1', 2, 2, lam)
            c = e.at(lam)[0][..., 0] ** 2 * (w[None, :] * t.absdet[:, None])
            ref = np.zeros(cs.ndof)
            np.add.at(ref, cs.spaces[0].edofs1, np.einsum('eq,qi->ei', c, phi))
            assert rel(b.vec.cpu().numpy(), ref) < 1e-13
            del b
        del gf
        gc.collect()


# ------------------------------------------------------------------------------------------ U-net


@pytest.mark.parametrize('N', [4, 12, 16])
def test_unet_tiles(gpu_ctx, N):
    """Forward and parameter gradients where the 16-voxel tiles end inside a row: coarsest grids of 8, 64
    and 125 voxels. The activations and the gradients of each layer are compared with the oracle's product
    of the GPU's own stored inputs, so bf16 rounding does not travel: FP32 sums of at most 864 products
    (1e-5 relative; an activation may differ by its own bf16 rounding, 2^-8, 4 % of them at most)."""
    import torch
    from opencmp_amd.learned import UNetPrecond
    from oracle import unet as ou
    from oracle.mlp import bf16_round
    rng = np.random.default_rng(N)
    p = (ou.init_params(N) + 0.05 * rng.standard_normal(ou.NPARAM)).astype(np.float32)
    U = UNetPrecond(N, gpu_ctx, params=p)
    n = [N + 1, N // 2 + 1, N // 4 + 1]
    x = rng.standard_normal((4,) + (n[0],) * 3).astype(np.float32)
    gy = rng.standard_normal((4,) + (n[0],) * 3).astype(np.float32)
    g = U.grad(torch.tensor(x.reshape(4, -1), device='cuda'), torch.tensor(gy.reshape(4, -1), device='cuda'))
    shapes = [(4, 0), (8, 0), (16, 1), (16, 1), (32, 2), (32, 2), (16, 1), (8, 0), (4, 0)]
    a = [U.activation(l - 1).cpu().numpy().reshape((c,) + (n[lv],) * 3).astype(np.float64)
         for l, (c, lv) in enumerate(shapes)]
    q = {k: bf16_round(v).astype(np.float64) for k, v in ou.unpack(p).items()}
    skip = {5: a[3], 6: a[1]}
    for l, (name, kind, ci, co, s) in enumerate(ou.LAYERS):
        W, b = q[name + '.W'], q[name + '.b']
        z = ou.conv(a[l], W, b, s) if kind == 'c' else ou.tconv(a[l], W, b, a[l + 1].shape[1])
        z = z + skip.get(l, 0.0)
        if l < 7:
            z = np.maximum(z, 0.0)
            d = np.abs(a[l + 1] - z)
            assert (d <= 2.0 ** -8 * np.abs(z) + 1e-5 * np.abs(z).max()).all(), name
            r = bf16_round(z.astype(np.float32))
            assert (a[l + 1] != r).mean() <= 0.04, name
        else:
            assert rel(a[8], z) < 1e-5
    acts = {'x': a[0], **{f'a{l}': a[l + 1] for l in range(7)}}
    _, gt = ou.backward(p, x, gy, bf16=True, acts=acts)
    o = 0
    g = g.cpu().numpy()
    for name, kind, ci, co, s in ou.LAYERS:
        for size in (ci * co * 27, co):
            assert rel(g[o:o + size], gt[o:o + size]) < 1e-5, name
            o += size


def test_unet_gradient_of_a_large_grid(gpu_ctx):
    """Sums over 129^3 voxels, known exactly: all weights zero, the last hidden layer's bias 1, so that the
    last layer's weight gradient is the output gradient summed over the voxels that a tap reaches, and its
    bias gradient over all. Constant output gradients let every rounding of a long FP32 sum fall on the
    same side. FP32 sums of 128 products and of 17 such sums, four wavefronts, FP64 beyond and one rounding:
    at most (128 + 17 + 2 + 1) 2^-24 relative."""
    import torch
    from opencmp_amd.learned import UNetPrecond
    from oracle import unet as ou
    N = 128
    n = N + 1
    p = {k: np.zeros_like(v) for k, v in ou.unpack(np.zeros(ou.NPARAM, np.float32)).items()}
    flat, o, at = np.zeros(ou.NPARAM, np.float32), 0, {}
    for name, kind, ci, co, s in ou.LAYERS:
        at[name] = (o, o + ci * co * 27, o + ci * co * 27 + co)
        o = at[name][2]
    assert o == ou.NPARAM and set(p) == {f'{k}.{w}' for k in at for w in 'Wb'}
    hidden, last = ou.LAYERS[6][0], ou.LAYERS[7][0]
    flat[at[hidden][1]:at[hidden][2]] = 1.0
    c = np.array([1.167053, 1.8018806, 1.0147063, 1.6719949], np.float32)
    U = UNetPrecond(N, gpu_ctx, params=flat)
    x = torch.zeros((4, n ** 3), device='cuda')
    gy = torch.from_numpy(c).cuda().reshape(4, 1).expand(4, n ** 3).contiguous()
    g = U.grad(x, gy).cpu().numpy().astype(np.float64)
    d = np.array([n - 1, n, n - 1], np.float64)     # voxels that a tap of -1, 0, 1 reaches along an axis
    taps = np.einsum('i,j,k->ijk', d, d, d).ravel()
    ci, co = ou.LAYERS[7][2], ou.LAYERS[7][3]
    W = g[at[last][0]:at[last][1]].reshape(co, ci, 27)
    ref = c.astype(np.float64)[:, None, None] * taps
    assert np.abs(W / ref - 1.0).max() <= 148 * 2.0 ** -24
    b = g[at[last][1]:at[last][2]]
    assert np.abs(b / (c.astype(np.float64) * n ** 3) - 1.0).max() <= 148 * 2.0 ** -24


# ------------------------------------------------------------------------------------------ MLP tiles


# 64 rows a wave from 131,072 rows: the first of them with and without a rest, and one past a whole block
@pytest.mark.parametrize('n', [127, 129, 130944, 130945, 131072, 131073 + 63, 262145])
def test_mlp_rows(gpu_ctx, n):
    """Forward and guess against the oracle; 2e-3 bounds the bf16 roundings that an FP32 sum puts one unit
    apart (as in the tests of the network)."""
    import torch
    from oracle import mlp as om
    from opencmp_amd.learned import MLPGuess
    p = om.init_params(3).astype(np.float32)
    net = MLPGuess(gpu_ctx, params=p, max_batch=128)
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 4)).astype(np.float32)
    y = net.forward(torch.from_numpy(X).cuda()).cpu().numpy().astype(np.float64)
    yo = om.forward(p, X, bf16=True)
    assert rel(y, yo) <= 2e-3
    tail = slice(n - min(n, 70), n)     # the last rows on their own: a wrong rest hides in the norm
    assert rel(y[tail], yo[tail]) <= 1e-2
    u = [rng.standard_normal(n) for _ in range(4)]
    off, sc, U = [0, n // 3, n], [0.5, 2.0], [1.0, 1.5]
    net.set_scales(off, sc, U)
    g = net.guess([torch.from_numpy(v).cuda() for v in u]).cpu().numpy()
    go = om.guess(p, u, off, sc, U, bf16=True)
    assert rel(g - u[0], go - u[0]) <= 2e-3


@pytest.mark.parametrize('B', [1, 63, 65, 257, 16385])
def test_mlp_gradient_rows(gpu_ctx, B):
    """Chunks of 64 rows, blocks of 256, of 64 rows or more for the small sums; 2e-2 as above for gradients."""
    import torch
    from oracle import mlp as om
    from opencmp_amd.learned import MLPGuess
    p = om.init_params(5).astype(np.float32)
    net = MLPGuess(gpu_ctx, params=p, max_batch=B)
    rng = np.random.default_rng(B)
    X = rng.standard_normal((B, 4)).astype(np.float32)
    T = rng.standard_normal(B).astype(np.float32)
    g, loss = net.grad(torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda())
    lo, go = om.loss_and_grad(p, X, T, bf16=True)
    g = g.cpu().numpy()
    assert rel(g, go) <= 2e-2 and abs(loss - lo) <= 1e-3 * lo


# ------------------------------------------------------------------------------------------ solvers' forms


def _apply(a, x):
    import torch
    y = torch.empty_like(x)
    a.mult(x, y)
    return y


def _poisson(C, ctx, n, kappa):
    fes = C.FESpace(C.Mesh(unit_square(n), ctx), [C.H1(2, 'left|top')])
    a = C.BilinearForm(fes, [C.Vol('gradgrad', 0, 0, coef=kappa)])
    f = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, POLY[2]))])
    return fes, a, f


# scalars summed by every block (up to 512 row blocks), by one block in its own launch beyond 2048
@pytest.mark.parametrize('precision', ['fp64', 'mixed'])
@pytest.mark.parametrize('n', [2, 40, 240, 520])
def test_cg_forms(gpu_ctx, n, precision):
    """The solution solves the system: residual of the returned vector, by the operator's own product."""
    import torch
    C = core()
    fes, a, f = _poisson(C, gpu_ctx, n, 1.3)
    a.Assemble()
    f.Assemble()
    pre = C.Preconditioner(a, 'local', precision=precision)
    pre.Update()
    u = C.GridFunction(fes)
    tol = 1e-9
    st = C.solve(a, f.vec, u.vec, pre, 'CG', tol=tol, precision=precision,
                 inner_tol=1e-4 if precision == 'mixed' else 0.0)
    assert st.converged
    free = torch.from_numpy(fes.FreeDofs()).to(u.vec.device)
    y = _apply(a, u.vec)
    r = torch.where(free, f.vec - y, torch.zeros_like(y))
    b = torch.where(free, f.vec, torch.zeros_like(y))
    # the stopping rule bounds the recurred residual; the true one is off by its rounding, some units of
    # 1.1e-16 |A| |x| with |A| <= 40 (rows of the P2 stiffness matrix, kappa = 1.3)
    assert float(r.norm()) <= 1.01 * tol * float(b.norm()) + 1e-15 * 40 * float(u.vec.norm())


# the s-step factor made by every block (up to 864 Gram partials an entry: 192^2 FP64) and in its own launch
@pytest.mark.parametrize('n,precision', [(2, 'fp64'), (17, 'fp64'), (17, 'mixed'), (192, 'fp64'), (193, 'fp64'),
                                         (216, 'fp64'), (300, 'mixed')])
def test_s_step_blocks(gpu_ctx, n, precision):
    import torch
    C = core()
    hm = unit_square(n)
    fes = C.FESpace(C.Mesh(hm, gpu_ctx), [C.L2(2)], dgjumps=True)
    a = C.BilinearForm(fes, [C.Vol('mass', 0, 0, coef=400.0), C.Vol('gradgrad', 0, 0, coef=1e-3),
                             C.DGFacet(0, eps=1e-3, alpha=40.0, dirichlet=hm.marker_mask(hm.bnd_names))])
    f = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, POLY[2]))])
    a.Assemble()
    f.Assemble()
    pre = C.Preconditioner(a, 'local', precision=precision)
    pre.Update()
    u = C.GridFunction(fes)
    st = C.solve(a, f.vec, u.vec, pre, 'GMRes', tol=1e-9, restart=50, precision=precision,
                 inner_tol=1e-4 if precision == 'mixed' else 0.0, s_step=5)
    assert st.converged and not st.fallback
    r = f.vec - _apply(a, u.vec)
    assert float(r.norm()) <= 1.01e-9 * float(f.vec.norm())


def test_inner_iteration_cap_costs_few_outer_iterations(gpu_ctx):
    """The Schur PCG's launches of a step are capped by the counts of the steps before. In one cycle of the
    two Stokes steps here FGMRES takes 109 and 102 iterations without a cap (one batch for the whole cycle,
    so no count is known in it); caps with three tenths plus ten of room take 111 and 107, with a tenth plus
    four 118 and 115. Half of the way between the sums, 6 % more than without a cap, is allowed."""
    C = core()
    from opencmp_amd.models import Stokes, const
    inflow = [(L.FN_POLY2, [0, 0, 4.0, 0, 0, -4.0]), const(0.0)]
    wall = [const(0.0), const(0.0)]
    its = {1: 0, 150: 0}
    for n, dt in ((16, 1e-2), (32, 1e-3)):
        m = Stokes(unit_square(n), kv=1.0, interp_ord=2, dirichlet={'u': {'left': inflow, 'top': wall, 'bottom': wall}},
                   linear_solver='GMRes', preconditioner='schur', linear_tolerance=1e-10, restart=150,
                   schur_iters=200, schur_tol=0.1, ctx=gpu_ctx)
        a = C.BilinearForm(m.fes, m.time_derivative_terms() + m.construct_bilinear_time_coefficient(dt) +
                           m.construct_bilinear_time_ODE(dt))
        f = C.LinearForm(m.fes, m.construct_linear(dt))
        a.Assemble()
        f.Assemble()
        for check in its:
            pre = m.construct_preconditioners(a)
            pre.Update()
            x = C.GridFunction(m.fes)
            m.apply_dirichlet_bcs_to(x)
            r = C.solve(a, f.vec, x.vec, pre, 'FGMRes', tol=1e-8, restart=150, maxit=150, check_every=check)
            assert r.converged and r.outer == 1
            its[check] += r.iters
    assert its[1] <= 1.06 * its[150]


def test_kept_plans_follow_the_form(gpu_ctx):
    """A form assembled again takes the coefficients, sources and field values of the moment, also after
    another form of the same space was assembled in between."""
    import torch
    C = core()
    fes, a, f = _poisson(C, gpu_ctx, 9, 1.0)
    a2 = C.BilinearForm(fes, [C.Vol('gradgrad', 0, 0, coef=2.5), C.Vol('mass', 0, 0, coef=1.0)])
    f2 = C.LinearForm(fes, [C.Source(0, (L.FN_POLY2, [2.0 * c for c in POLY[2]]))])
    x = torch.linspace(-1, 1, fes.ndof, dtype=torch.float64, device='cuda')
    a.Assemble()
    y1 = _apply(a, x).clone()
    a2.Assemble()
    a.Assemble()
    assert torch.equal(_apply(a, x), y1)
    f.Assemble()
    b1 = f.vec.clone()
    f2.Assemble()
    f.Assemble()
    assert torch.equal(f.vec, b1)
    # twice the source is twice the vector, to the rounding of its sums
    assert float((f2.vec - 2 * b1).abs().max()) <= 1e-15 * float(b1.abs().max()) * 8


def test_kept_plans_follow_what_changes(gpu_ctx):
    """The same form assembled again after a coefficient, the contents of a per-element coefficient, the
    values of a wind or a weight or the weighting field itself changed: bit for bit what a new form of the
    same terms gives, and not what it gave before."""
    import torch
    C = core()
    hm = unit_square(6)
    gm = C.Mesh(hm, gpu_ctx)
    fes = C.FESpace(gm, [C.H1(2)])
    wind, w1, w2 = (C.GridFunction(C.FESpace(gm, [C.H1(p, ncomp=c)])) for p, c in ((2, 2), (1, 1), (2, 1)))
    rng = np.random.default_rng(5)

    def fill(v):
        v.copy_(torch.from_numpy(rng.random(v.numel())).to(v.device))

    kappa = torch.empty(hm.nel, dtype=torch.float64, device='cuda')
    for v in (kappa, wind.vec, w1.vec, w2.vec):
        fill(v)
    terms = [C.Vol('gradgrad', 0, 0, elem_coef=kappa),
             C.Vol('conv', 0, 0, wind_gf=(wind, wind.space.comp_blocks[0])),
             C.Vol('mass', 0, 0, coef=2.0, weight_gf=(w1, 0, L.WEIGHT_FIELD)),
             C.Vol('mass', 0, 0, coef=0.5, weight_gf=(w2, 0, L.WEIGHT_ONE_MINUS_FIELD))]
    # alone, and as the last of 33 terms, which are added in a second launch
    for terms in (terms, [C.Vol('gradgrad', 0, 0, elem_coef=kappa)] * 32 + terms[2:]):
        a = C.BilinearForm(fes, terms)
        a.Assemble()
        last = a.values()

        def again():
            nonlocal last
            a.Assemble()
            fresh = C.BilinearForm(fes, list(terms))
            fresh.Assemble()
            assert np.array_equal(a.values(), fresh.values()) and not np.array_equal(a.values(), last)
            last = a.values()

        terms[-1].coef += 1.25
        again()
        for v in (kappa, w1.vec, w2.vec):
            fill(v)
            again()
        if len(terms) == 4:
            fill(wind.vec)
            again()
        terms[-1].weight_gf = (w1, 0, L.WEIGHT_ONE_MINUS_FIELD)
        again()
        terms[-1].weight_gf = (w2, 0, L.WEIGHT_FIELD)
        again()


def test_kept_load_plans_follow_what_changes(gpu_ctx):
    """As above for load vectors, and with more of them in turn (12) than a space keeps plans (8)."""
    import torch
    C = core()
    hm = unit_square(6)
    gm = C.Mesh(hm, gpu_ctx)
    fes = C.FESpace(gm, [C.H1(2)])
    g, w = (C.GridFunction(C.FESpace(gm, [C.H1(p)])) for p in (2, 1))
    rng = np.random.default_rng(6)

    def fill(v):
        v.copy_(torch.from_numpy(rng.random(v.numel())).to(v.device))

    fill(g.vec)
    fill(w.vec)
    forms = [C.LinearForm(fes, [C.Source(0, field_gf=(g, 0), coef=1.0 + k, weight_gf=(w, 0, L.WEIGHT_FIELD)),
                                C.Source(0, (L.FN_CONST, (0.1 * k,)))]) for k in range(12)]

    def vectors(fs):
        for f in fs:
            f.Assemble()
        return [f.vec.clone() for f in fs]

    last = vectors(forms)
    for change in ('field', 'weight', 'coefficient', 'source'):
        if change == 'field':
            fill(g.vec)
        elif change == 'weight':
            fill(w.vec)
        for f in forms:
            if change == 'coefficient':
                f.terms[0].coef += 0.25
            elif change == 'source':
                f.terms[1].fn = (L.FN_CONST, (f.terms[1].fn[1][0] + 1.0,))
        now = vectors(forms)
        fresh = vectors([C.LinearForm(fes, list(f.terms)) for f in reversed(forms)])[::-1]
        for a, b, c in zip(now, fresh, last):
            assert torch.equal(a, b) and not torch.equal(a, c)
        last = now
