"""The box apply (element factors, needs an MI355X) at the edges of its
decomposition.

Its workgroups march columns of 16, 32 or 64 element slots along z, duplicate
the elements of tile and chunk faces and choose slots, tile and chunk from the
mesh and the number of right-hand sides.  Against the quadrature-point factors
of the same operator (the tile kernels, which the tests of tile variants pin to
the oracle in factor mode 0): meshes of one
element per direction, edges just below, at and above tile and chunk sizes, the
block pairs of order 1 split by an odd edge, partial PEC, and sizes that take
each number of slots.  Both sides carry rounding errors of a few units of
2^-53 (1e-15 .. 3e-15 relative to 64-bit references), so 2e-14 bounds their
difference with a margin; FP32 vectors differ by their own rounding, 2^-24 per
entry of x and y, and the tile kernel's FP32 sums (1e-7 measured).  A result
must not depend on the decomposition: several right-hand sides in one launch
(another tile and chunk) are bitwise those of single launches.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import hephaestus_amd as H
    H.load()
    return torch, H


SIZES = [(1, 1, 1), (2, 1, 1), (1, 5, 2), (1, 1, 40), (3, 4, 5), (4, 4, 4), (5, 7, 9), (7, 8, 2), (8, 9, 17), (64, 2, 3),
         (65, 1, 2), (9, 63, 5), (16, 15, 33), (48, 48, 11)]


@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("n", SIZES)
def test_box_apply_edges(env, p, n):
    torch, H = env
    pec = (0x3F, 0x19, 0x00, 0x26)[sum(n) % 4]
    print(f"case box edges p={p} n={n} pec={pec:#x}", flush=True)
    g = torch.Generator().manual_seed(sum(n) + p)
    E = n[0] * n[1] * n[2]
    nu = (0.5 + torch.rand(E, generator=g, dtype=torch.float64)).numpy()
    sig = (10.0 ** (2.0 * torch.rand(E, generator=g, dtype=torch.float64))).numpy()
    op = H.Operator(n, p, nu, sig, pec_faces=pec, length=(1.0, 0.7, 1.3)).setup(0.37)
    X = (2.0 * torch.rand((5, op.ndofs), generator=g, dtype=torch.float64) - 1.0).cuda()
    Y = op.apply(X)
    y32 = op.apply_f32(X.float())
    k = op.apply_curl(X[0].contiguous())
    for r in range(5):
        assert torch.equal(op.apply(X[r].contiguous()), Y[r]), r
        assert torch.equal(op.apply_f32(X[r].float().contiguous()), y32[r]), r
    op.set_factor_mode(0)
    Yq, kq = op.apply(X), op.apply_curl(X[0].contiguous())
    assert float((Y - Yq).norm()) <= 2e-14 * float(Yq.norm())
    assert float((k - kq).norm()) <= 2e-14 * float(kq.norm())
    assert float((y32.double() - Yq).norm()) <= 4e-7 * float(Yq.norm())
    op.close()


@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("n,pec", [((1, 1, 1), 0x3F), ((1, 1, 1), 0x00), ((2, 1, 3), 0x15), ((5, 4, 6), 0x2A), ((7, 33, 2), 0x3F)])
def test_box_diagonals(env, p, n, pec):
    """The closed-form Jacobi and node diagonals of a box mesh (the latter
    through the gradient-corrected preconditioner) and its term ratio equal
    those of the same mesh given by its vertices, which are summed over the
    quadrature-point factors.  Every entry is a sum of positive terms, so both
    are within some 50 roundings of the exact value: 1e-13."""
    torch, H = env
    import numpy as np
    print(f"case box diagonals p={p} n={n} pec={pec:#x}", flush=True)
    rng = np.random.default_rng(11 * p + sum(n))
    E = n[0] * n[1] * n[2]
    nu, sig = rng.uniform(0.5, 2.0, E), 10.0 ** rng.uniform(-3, 3, E)
    L = (1.0, 0.6, 1.5)
    Z, Y, X = np.meshgrid(*[L[a] * np.arange(n[a] + 1) / n[a] for a in (2, 1, 0)], indexing="ij")
    vert = np.stack([X, Y, Z], -1).reshape(-1, 3)
    box = H.Operator(n, p, nu, sig, pec_faces=pec, length=L).setup(0.25)
    ref = H.Operator(n, p, nu, sig, pec_faces=pec, vert=vert).setup(0.25)
    d, dr = box.diagonal(), ref.diagonal()
    assert float(((d - dr) / dr).abs().max()) <= 1e-13
    r = torch.from_numpy(rng.uniform(-1, 1, box.ndofs)).cuda()
    for mode in (H.SOLVE_FP64, H.SOLVE_FP64 | H.SOLVE_AUX):
        z, zr = box.precond_apply(r, mode), ref.precond_apply(r, mode)
        assert float((z - zr).norm()) <= 1e-12 * float(zr.norm()), mode
    assert abs(box.term_ratio / ref.term_ratio - 1.0) <= 1e-13
    box.close()
    ref.close()


@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 3), (1, 1, 40), (4, 4, 4), (5, 7, 9), (8, 9, 17), (65, 1, 2), (9, 23, 5), (33, 26, 11)])
def test_hex_apply_edges(env, p, n):
    """The trilinear form of the box apply, which takes the point factors from
    the vertices, against the stored factors: distorted elements (vertices moved
    by up to 0.15 of an edge), also with the x axis reversed (negative
    determinants).  The point factors are sums of products of Jacobian entries
    with at most a few digits of cancellation on both sides: 4e-14."""
    torch, H = env
    import numpy as np
    pec = (0x3F, 0x19, 0x00, 0x26)[sum(n) % 4]
    print(f"case hex edges p={p} n={n} pec={pec:#x}", flush=True)
    rng = np.random.default_rng(sum(n) + p)
    E = n[0] * n[1] * n[2]
    nu, sig = rng.uniform(0.5, 1.5, E), 10.0 ** rng.uniform(0, 2, E)
    L = (1.0 if n[1] % 2 else -1.0, 0.7, 1.3)
    Z, Y, X = np.meshgrid(*[L[a] * np.arange(n[a] + 1) / n[a] for a in (2, 1, 0)], indexing="ij")
    h = np.array([abs(L[a]) / n[a] for a in range(3)])
    vert = np.stack([X, Y, Z], -1).reshape(-1, 3) + 0.15 * h * rng.uniform(-1, 1, (X.size, 3))
    op = H.Operator(n, p, nu, sig, pec_faces=pec, vert=vert).setup(0.37)
    X = torch.from_numpy(rng.uniform(-1, 1, (5, op.ndofs))).cuda()
    Y = op.apply(X)
    y32 = op.apply_f32(X.float())
    k = op.apply_curl(X[0].contiguous())
    for r in range(5):
        assert torch.equal(op.apply(X[r].contiguous()), Y[r]), r
        assert torch.equal(op.apply_f32(X[r].float().contiguous()), y32[r]), r
    op.set_factor_mode(0)
    Yq, kq = op.apply(X), op.apply_curl(X[0].contiguous())
    assert float((Y - Yq).norm()) <= 4e-14 * float(Yq.norm())
    assert float((k - kq).norm()) <= 4e-14 * float(kq.norm())
    assert float((y32.double() - Yq).norm()) <= 4e-7 * float(Yq.norm())
    op.close()


@pytest.mark.parametrize("p", [1, 2, 3])
def test_hex_table(env, p):
    """Trilinear instances of one order in one launch of a batch, with several
    right-hand sides: every column reaches the asked residual of the operator on
    stored factors (the factor 1.05 covers the difference of the recurred from
    the true residual and of the two products)."""
    torch, H = env
    import numpy as np
    print(f"case hex table p={p}", flush=True)
    rng = np.random.default_rng(p)
    bt, ops, bs, xs = H.Batch(), [], [], []
    for n in ((3, 5, 4), (9, 2, 6)):
        Z, Y, X = np.meshgrid(*[np.arange(n[a] + 1) / n[a] for a in (2, 1, 0)], indexing="ij")
        vert = np.stack([X, Y, Z], -1).reshape(-1, 3) + 0.1 * rng.uniform(-1, 1, (X.size, 3)) / max(n)
        E = n[0] * n[1] * n[2]
        op = H.Operator(n, p, rng.uniform(0.5, 2.0, E), rng.uniform(0.5, 2.0, E), vert=vert).setup(1.0)
        ops.append(op)
        bs.append(torch.stack([op.rhs_coil(7 * r + p) for r in range(3)]))
        xs.append(torch.zeros_like(bs[-1]))
        bt.add(op, bs[-1], xs[-1], rtol=1e-10, maxit=5000)
    _, st = bt.solve(mode=H.SOLVE_FP64)
    assert all(s["converged"] for s in st), st
    for op, b, x in zip(ops, bs, xs):
        op.set_factor_mode(0)
        r = b - op.apply(x)
        assert bool((r.norm(dim=1) <= 1.05e-10 * b.norm(dim=1)).all())
    bt.close()
    for op in ops:
        op.close()


@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("n,pec", [((1, 1, 1), 0x3F), ((1, 1, 1), 0x00), ((2, 1, 3), 0x15), ((5, 4, 6), 0x2A), ((17, 9, 5), 0x3F),
                                   ((8, 3, 41), 0x19)])
def test_box_av_edges(env, p, n, pec):
    """The mass-only and the adding form of the box apply, through the A-V block
    operator, against the stored factors of the same operator (general product
    and a sum afterwards).  Random inputs, no cancellation beyond that of a
    difference of neighbours: 4e-14 as for a product."""
    torch, H = env
    import numpy as np
    print(f"case box av p={p} n={n} pec={pec:#x}", flush=True)
    rng = np.random.default_rng(3 * p + sum(n))
    E = n[0] * n[1] * n[2]
    op = H.Operator(n, p, rng.uniform(0.5, 2.0, E), 10.0 ** rng.uniform(-2, 2, E), pec_faces=pec, length=(1.0, 0.8, 1.4)).setup(0.3)
    a = torch.from_numpy(rng.uniform(-1, 1, op.ndofs)).cuda()
    v = torch.from_numpy(rng.uniform(-1, 1, op.nnodes)).cuda()
    ya, yv = op.av_apply(a, v)
    op.set_factor_mode(0)
    ra, rv = op.av_apply(a, v)
    assert float((ya - ra).norm()) <= 4e-14 * float(ra.norm())
    assert float((yv - rv).norm()) <= 4e-14 * float(rv.norm())
    op.close()


def _polar(n, axis):
    """Vertices of a sector around the z axis: the radius runs along `axis`, the
    angle along the other, so that the first elements have a collapsed edge (the
    determinant is zero on the z axis and positive at every quadrature point)."""
    import numpy as np
    k, j, i = np.meshgrid(*[np.arange(n[a] + 1) / n[a] for a in (2, 1, 0)], indexing="ij")
    r, t = (i, 1.2 * j) if axis == "x" else (j, 1.2 * (1.0 - i))
    return np.stack([r * np.cos(t), r * np.sin(t), k], -1).reshape(-1, 3)


@pytest.mark.parametrize("axis", ["x", "y"])
@pytest.mark.parametrize("p", [1, 2, 3])
@pytest.mark.parametrize("n,pec", [((3, 4, 2), 0x3F), ((5, 3, 4), 0x00), ((2, 7, 3), 0x15)])
def test_hex_collapsed_edge(env, p, n, pec, axis):
    """Elements with a collapsed edge (wedges on the axis of a polar mesh): the
    trilinear form takes factors at quadrature points only, where they are
    finite.  The point nearest to the collapsed edge lies at 0.069 of the element
    or more, which amplifies the roundings of the factors by at most 15: 4e-14
    against the stored factors, as for the other distorted meshes."""
    torch, H = env
    import numpy as np
    print(f"case hex collapsed p={p} n={n} pec={pec:#x} {axis}", flush=True)
    rng = np.random.default_rng(sum(n) + 7 * p)
    E = n[0] * n[1] * n[2]
    op = H.Operator(n, p, rng.uniform(0.5, 1.5, E), 10.0 ** rng.uniform(0, 2, E), pec_faces=pec, vert=_polar(n, axis)).setup(0.37)
    x = torch.from_numpy(rng.uniform(-1, 1, (2, op.ndofs))).cuda()
    v = torch.from_numpy(rng.uniform(-1, 1, op.nnodes)).cuda()

    def products():
        return [op.apply(x), op.apply_curl(x[0].contiguous()), *op.av_apply(x[0].contiguous(), v)]

    ys = products()
    op.set_factor_mode(0)
    for i, (y, r) in enumerate(zip(ys, products())):
        assert bool(torch.isfinite(y).all()), i
        assert float((y - r).norm()) <= 4e-14 * float(r.norm()), i
    op.close()


@pytest.mark.parametrize("mesh", ["box", "hex"])
@pytest.mark.parametrize("p", [1, 2, 3])
def test_non_finite_entries_stay_in_their_elements(env, p, mesh):
    """An entry of x that is not finite, or that overflows in the product, makes
    outputs of the elements that hold it non-finite and no others: elsewhere the
    bits are those of the product with a zero in its place."""
    torch, H = env
    import numpy as np
    from brute import elem_gids
    n = (5, 4, 6)
    print(f"case non-finite p={p} {mesh}", flush=True)
    rng = np.random.default_rng(p)
    E = n[0] * n[1] * n[2]
    vert = None
    if mesh == "hex":
        Z, Y, X = np.meshgrid(*[np.arange(n[a] + 1) / n[a] for a in (2, 1, 0)], indexing="ij")
        vert = np.stack([X, Y, Z], -1).reshape(-1, 3) + 0.01 * rng.uniform(-1, 1, (X.size, 3))
    op = H.Operator(n, p, rng.uniform(1e3, 2e3, E), rng.uniform(0.5, 2.0, E), pec_faces=0x13, vert=vert).setup(1.0)
    gids = np.array([np.asarray(elem_gids(n, p, ex, ey, ez)) for ez in range(n[2]) for ey in range(n[1]) for ex in range(n[0])])
    x = torch.from_numpy(rng.uniform(-1, 1, op.ndofs)).cuda()
    per = p * (p + 1) ** 2
    for (ex, ey, ez), loc in (((2, 1, 2), 0), ((1, 2, 3), per), ((3, 2, 0), 2 * per), ((3, 3, 5), 3 * per - 1)):
        dof = int(gids[(ez * n[1] + ey) * n[0] + ex][loc])
        away = torch.ones(op.ndofs, dtype=torch.bool, device="cuda")
        away[torch.from_numpy(np.unique(gids[(gids == dof).any(1)])).cuda()] = False
        for v in (float("nan"), float("inf"), 1.7e308):
            x0, xv = x.clone(), x.clone()
            x0[dof], xv[dof] = 0.0, v
            for f in (op.apply, op.apply_curl, lambda t: op.apply_f32(t.float())):
                y0, y = f(x0), f(xv)
                assert bool(torch.isfinite(y0).all())
                assert not bool(torch.isfinite(y).all())
                assert torch.equal(y[away], y0[away]), (dof, v, int((~torch.isfinite(y[away])).sum()))
    op.close()
