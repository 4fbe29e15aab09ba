"""GPU parity of the particle operations against the CPU oracle, through the C-ABI:
tree structure, fill_tree_mean, convolve_pencil / convolve, Richardson-Lucy,
reconstruct_constant, reconstruct_level and reconstruct_smooth.

The GPU sums in the reference's order (tree children: particles then tree nodes,
(z, x, y); convolution taps: (z, x, y)), so every float result is bit-equal to the
oracle, which is itself bit-equal to the reference build (test_oracle_numerics.py).
Larger volumes are checked through size-independent properties: a normalised
stencil maps a constant field to itself, tree means of a constant are constant,
Richardson-Lucy keeps a constant image, and sampling a reconstruction gives the
particles back.
"""
import numpy as np
import pytest
import torch

import libapr_amd as A

pytestmark = pytest.mark.gpu

CASES = [((32, 64, 64), 20, 0), ((29, 45, 61), 12, 3), ((16, 16, 130), 8, 4), ((64, 96, 128), 60, 5)]


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def _pair(O, ctx, shape, nb, seed):
    """oracle APR and the GPU APR built from the oracle's structure"""
    img = A.synth_blobs(shape, seed, nb)
    o = O.get_apr(img, O.params(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10), "oracle")
    g = A.APR.from_structure(o.dims, o.xz_end_vec, o.y_vec, ctx)
    print(f"case {shape} seed {seed} P={o.total}", flush=True)
    return img, o, g


def _stencils(O, kind, o):
    if kind == "mean3":
        st = np.full((3, 3, 3), 1.0 / 27, np.float32)
    elif kind == "gauss5":
        st = O.gaussian_stencil((1.0, 1.0, 1.0), (5, 5, 5), True)
    else:
        st = O.gaussian_stencil((1.0, 1.5, 2.0), (3, 5, 7), False)
    return st, O.downsampled_stencils(st, o.l_max - o.l_min, True, "oracle")


@pytest.mark.parametrize("shape,nb,seed", CASES)
def test_tree_and_tree_mean(oracle, ctx, shape, nb, seed):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    to, tg = o.tree(), g.tree()
    assert tg["total"] == to["total"] and tg["l_max"] == to["l_max"]
    for k in ("level_xz_vec", "xz_end_vec", "y_vec"):
        assert np.array_equal(tg[k], to[k]), k
    parts = o.sample(img)
    assert np.array_equal(_bits(A.APRTreeNumerics.fill_tree_mean(g, parts)), _bits(o.fill_tree_mean(parts)))
    pf = (parts.astype(np.float32) * np.float32(1.37)).astype(np.float32)
    assert np.array_equal(_bits(A.APRTreeNumerics.fill_tree_mean(g, pf)), _bits(o.fill_tree_mean(pf)))


@pytest.mark.parametrize("shape,nb,seed", [((3, 9, 511), 6, 1), ((5, 4, 513), 6, 2), ((18, 35, 129), 9, 3), ((4, 7, 1026), 9, 4), ((3, 5, 4133), 9, 5)])
def test_tree_mean_pieces(oracle, ctx, shape, nb, seed):
    """child rows of one piece and a cell more (512; 128 in the launch of the small levels), rows of several
    pieces, and odd dims, whose last children are scaled"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    for p in (parts, parts.astype(np.float32) * np.float32(0.83)):
        assert np.array_equal(_bits(A.APRTreeNumerics.fill_tree_mean(g, p)), _bits(o.fill_tree_mean(p)))


# y one short of, at and past a block's 64 and a row image's 1024; x about a block's 16; few and many planes
EDGES = [((8, 17, 63), 5, 1), ((7, 15, 65), 5, 2), ((41, 16, 64), 8, 3), ((9, 33, 129), 8, 4), ((8, 7, 1027), 9, 5)]


def _wide(o, stack):
    """particles of the levels whose lines are longer than half their stencil: in shorter ones the oracle's
    window holds what the level before left there"""
    y, x, z = o.dims
    keep = []
    for l, n in _particles_per_level(o):
        s, k = 1 << (o.l_max - l), stack[min(o.l_max - l, len(stack) - 1)].shape
        keep.append(np.full(n, all(-(-d // s) > m // 2 for d, m in zip((z, x, y), k))))
    return np.concatenate(keep)


@pytest.mark.parametrize("shape,nb,seed", EDGES)
@pytest.mark.parametrize("size", [3, 5, 7, 9])
@pytest.mark.parametrize("reflect", [True, False])
def test_convolve_cubic_edges(oracle, ctx, shape, nb, seed, size, reflect):
    """cubic stencils without symmetry in reference order; and one level's stencil of another form, which
    takes the list of all levels to the other kernels"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    rng = np.random.default_rng(seed)
    stack = oracle.downsampled_stencils(rng.uniform(-1, 1, (size,) * 3).astype(np.float32), o.l_max - o.l_min, False, "oracle")
    w = _wide(o, stack)
    assert w.mean() > 0.5
    for p in (parts, parts.astype(np.float32) * np.float32(0.83)):
        got = A.APRFilter.convolve_pencil(g, stack, p, reflect_boundary=reflect)
        assert np.array_equal(_bits(got)[w], _bits(o.convolve_pencil(stack, p, reflect))[w])
    stack[-1] = rng.uniform(-1, 1, (3, 1, 3)).astype(np.float32)
    got = A.APRFilter.convolve_pencil(g, stack, parts, reflect_boundary=reflect)
    assert np.array_equal(_bits(got)[w], _bits(o.convolve_pencil(stack, parts, reflect))[w])


@pytest.mark.parametrize("shape,nb,seed", CASES)
@pytest.mark.parametrize("kind", ["mean3", "gauss5", "aniso"])
@pytest.mark.parametrize("reflect", [True, False])
def test_convolve_pencil(oracle, ctx, shape, nb, seed, kind, reflect):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    st, stack = _stencils(oracle, kind, o)
    pf = parts.astype(np.float32)
    exp = o.convolve_pencil(stack, pf, reflect)
    got = A.APRFilter.convolve_pencil(g, stack, pf, reflect_boundary=reflect)
    nbad = int((_bits(got) != _bits(exp)).sum())
    assert nbad == 0, f"{nbad} of {got.size} differ; max abs {np.abs(got - exp).max()}"
    # u16 input, and the single-stencil form that prepares the stack itself
    assert np.array_equal(_bits(A.APRFilter.convolve(g, stack, parts, reflect_boundary=reflect)),
                          _bits(o.convolve_pencil(stack, parts, reflect)))
    assert np.array_equal(_bits(A.APRFilter.convolve_pencil(g, st, pf, reflect_boundary=reflect, normalize=True)), _bits(exp))


def test_convolve_unit_stencil_is_identity(oracle, ctx):
    img, o, g = _pair(oracle, ctx, *CASES[0])
    parts = o.sample(img).astype(np.float32)
    one = np.zeros((3, 3, 3), np.float32)
    one[1, 1, 1] = 1
    out = A.APRFilter.convolve_pencil(g, [one], parts)
    assert np.array_equal(out, parts)


@pytest.mark.parametrize("shape,nb,seed", CASES[:2])
def test_richardson_lucy(oracle, ctx, shape, nb, seed):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    psf = oracle.gaussian_stencil((1.0, 1.0, 2.0), (9, 9, 9), True)
    uo, it, rel_o = o.richardson_lucy(parts, psf, 3)
    ug, st = A.APRNumerics.richardson_lucy(g, parts, None, psf, 3, normalize=True)
    assert st["iterations"] == it == 3
    assert np.array_equal(_bits(ug), _bits(uo))
    assert abs(st["last_rel_update"] - rel_o) <= 1e-9 * max(rel_o, 1e-30)
    # resume continues from the estimate (APRNumerics.hpp:559-562)
    uo2, _, _ = o.richardson_lucy(parts, psf, 2, u=uo)
    ug2, _ = A.APRNumerics.richardson_lucy(g, parts, ug.copy(), psf, 2, normalize=True, resume=True)
    assert np.array_equal(_bits(ug2), _bits(uo2))
    # float input
    pf = parts.astype(np.float32)
    uo3, _, _ = o.richardson_lucy(pf, psf, 2)
    ug3, _ = A.APRNumerics.richardson_lucy(g, pf, None, psf, 2, normalize=True)
    assert np.array_equal(_bits(ug3), _bits(uo3))


@pytest.mark.parametrize("shape,nb,seed", CASES)
def test_richardson_lucy_tv(oracle, ctx, shape, nb, seed):
    """APRNumerics::richardson_lucy_tv: bit-equal to the oracle (whose restatement is bit-equal
    to the reference build), u16 and f32 input, fresh and resumed; reg = 0 is plain RL"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    psf = oracle.gaussian_stencil((1.0, 1.0, 1.5), (5, 5, 5), True)
    print(f"RL-TV {shape}: P={o.total}", flush=True)
    uo = o.richardson_lucy_tv(parts, psf, 3, 0.01)
    ug = A.APRNumerics.richardson_lucy_tv(g, parts, None, psf, 3, 0.01, normalize=True)
    assert np.array_equal(_bits(ug), _bits(uo))
    pf = parts.astype(np.float32) * np.float32(0.7)
    uo2 = o.richardson_lucy_tv(pf, psf, 2, 0.02, u=uo)
    ug2 = A.APRNumerics.richardson_lucy_tv(g, pf, ug.copy(), psf, 2, 0.02, normalize=True, resume=True)
    assert np.array_equal(_bits(ug2), _bits(uo2))
    plain, _ = A.APRNumerics.richardson_lucy(g, parts, None, psf, 2, normalize=True)
    assert np.array_equal(_bits(A.APRNumerics.richardson_lucy_tv(g, parts, None, psf, 2, 0.0, normalize=True)), _bits(plain))


def test_richardson_lucy_stopping_rule(oracle, ctx):
    img, o, g = _pair(oracle, ctx, *CASES[0])
    parts = o.sample(img)
    psf = oracle.gaussian_stencil((1.0, 1.0, 2.0), (9, 9, 9), True)
    uo, it, rel = o.richardson_lucy(parts, psf, 200, tol=1e-3)
    ug, st = A.APRNumerics.richardson_lucy(g, parts, None, psf, 200, normalize=True, tol=1e-3)
    assert st["iterations"] == it < 200 and st["last_rel_update"] < 1e-3
    assert np.array_equal(_bits(ug), _bits(uo))


@pytest.mark.parametrize("shape,nb,seed", CASES[:3])
@pytest.mark.parametrize("delta", [0, -1, -2])
def test_reconstruct_constant(oracle, ctx, shape, nb, seed, delta):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    for out_dtype in (np.uint16, np.float32):
        assert np.array_equal(A.APRReconstruction.reconstruct_constant(g, parts, delta, out_dtype),
                              o.reconstruct(parts, delta, out_dtype))
    pf = (parts * np.float32(0.73)).astype(np.float32)
    for out_dtype in (np.uint16, np.float32):
        got = A.APRReconstruction.reconstruct_constant(g, pf, delta, out_dtype)
        exp = o.reconstruct(pf, delta, out_dtype)
        assert np.array_equal(got.view(np.uint8), exp.view(np.uint8))


def test_gpu_apr_particle_ops(oracle, ctx):
    """the same operations on an APR made by the GPU converter"""
    img = A.synth_blobs((61, 63, 65), 1, 30)
    conv = A.APRConverter(ctx)
    conv.par = A.APRParameters(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10)
    g = conv.get_apr(img)
    o = oracle.get_apr(img, oracle.params(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10), "oracle")
    parts = A.ParticleData().sample_image(g, img)
    _, stack = _stencils(oracle, "gauss5", o)
    assert np.array_equal(_bits(A.APRFilter.convolve_pencil(g, stack, parts)), _bits(o.convolve_pencil(stack, parts, True)))
    assert np.array_equal(A.APRReconstruction.reconstruct_constant(g, parts), o.reconstruct(parts))


def test_malformed_structure_rejected(oracle, ctx):
    img = A.synth_blobs((32, 64, 64), 0, 20)
    o = oracle.get_apr(img, oracle.params(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10), "oracle")
    y = o.y_vec.copy()
    y[len(y) // 2] = 65000            # beyond y_num of any level
    with pytest.raises(A.AprhError):
        A.APR.from_structure(o.dims, o.xz_end_vec, y, ctx)
    x = o.xz_end_vec.copy()
    x[-1] += 1                        # total mismatch
    with pytest.raises(A.AprhError):
        A.APR.from_structure(o.dims, x, o.y_vec, ctx)
    with pytest.raises(A.AprhError):
        A.APR.from_structure(o.dims, o.xz_end_vec[:-1], o.y_vec, ctx)


def test_argument_errors(oracle, ctx):
    img, o, g = _pair(oracle, ctx, *CASES[0])
    parts = o.sample(img)
    with pytest.raises(A.AprhError):
        A.APRFilter.convolve_pencil(g, [np.ones((2, 3, 3), np.float32)], parts)          # even stencil
    with pytest.raises(A.AprhError):
        A.APRReconstruction.reconstruct_constant(g, parts, -(o.l_max))                # below l_min
    with pytest.raises(A.AprhError):
        A.APRNumerics.richardson_lucy(g, parts, None, np.ones((3, 3, 3), np.float32), -1)


def test_properties_at_size(ctx):
    """size-independent checks on a 512x512x256 volume (GPU only)"""
    shape = (256, 512, 512)
    img = A.synth_blobs(shape, 7, 3000, sigma=(1.5, 6.0), amp=(300.0, 4000.0))
    conv = A.APRConverter(ctx)
    conv.par = A.APRParameters(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10)
    g = conv.get_apr(img)
    parts = A.ParticleData().sample_image(g, img)
    print(f"P={g.total}", flush=True)
    # reconstruction then sampling returns the particles
    rec = A.APRReconstruction.reconstruct_constant(g, parts)
    assert np.array_equal(A.ParticleData().sample_image(g, rec), parts)
    # constant field: tree means, normalised convolution and RL keep it
    c = np.full(g.total, 7.0, np.float32)
    tm = A.APRTreeNumerics.fill_tree_mean(g, c)
    np.testing.assert_allclose(tm, 7.0, rtol=1e-6)
    st = A.APRStencil.create_gaussian_filter((1.0, 1.0, 1.0), (5, 5, 5), True)
    out = A.APRFilter.convolve_pencil(g, st, c, normalize=True)
    np.testing.assert_allclose(out, 7.0, rtol=1e-5)
    # u = 1 -> blur 1 -> ratio 7 -> u = 7, then ratio 1 keeps it
    u, s = A.APRNumerics.richardson_lucy(g, c, None, st, 3, normalize=True)
    np.testing.assert_allclose(u, 7.0, rtol=1e-4)
    assert s["iterations"] == 3


@pytest.fixture(scope="module")
def sep_ctx():
    c = A.Context(0)
    c.set_conv_mode(A.CONV_SEPARABLE)
    yield c
    c.close()


def _rel(got, exp):
    exp = exp.astype(np.float64)
    return np.abs(got.astype(np.float64) - exp) / np.maximum(np.abs(exp), 1e-3 * np.abs(exp).max())


@pytest.mark.parametrize("shape,nb,seed", CASES)
@pytest.mark.parametrize("kind", ["mean3", "gauss5", "aniso"])
@pytest.mark.parametrize("reflect", [True, False])
def test_convolve_separable_mode(oracle, sep_ctx, shape, nb, seed, kind, reflect):
    """CONV_SEPARABLE: rank-1 stencils as three 1-D passes; within 1e-5 relative of the
    reference-order result, and as close as it to the float64 ground truth"""
    img, o, g = _pair(oracle, sep_ctx, shape, nb, seed)
    parts = o.sample(img).astype(np.float32)
    st, stack = _stencils(oracle, kind, o)
    exp = o.convolve_pencil(stack, parts, reflect)
    got = A.APRFilter.convolve_pencil(g, stack, parts, reflect_boundary=reflect)
    r = _rel(got, exp).max()
    print(f"separable vs reference order: max rel {r:.2e}")
    assert r < 1e-5
    if shape == CASES[1][0]:
        from test_oracle_numerics import conv_gt
        t = o.tree()
        gt = conv_gt(o, stack, parts.astype(np.float64), o.fill_tree_mean(parts).astype(np.float64), t, reflect)
        e_exact, e_sep = _rel(exp, gt).max(), _rel(got, gt).max()
        print(f"vs float64 ground truth: reference order {e_exact:.2e}, separable {e_sep:.2e}")
        assert e_sep < 1e-5 and e_exact < 1e-5


@pytest.mark.parametrize("shape,nb,seed", EDGES)
@pytest.mark.parametrize("size", [1, 3, 5, 7, 9, 11, 13])
@pytest.mark.parametrize("reflect", [True, False])
def test_convolve_separable_edges(oracle, sep_ctx, shape, nb, seed, size, reflect):
    """every cubic size; weights and values are positive, so the reference order's size^3 roundings and the
    three passes' 3 size bound the difference, with 3 more for the factors"""
    img, o, g = _pair(oracle, sep_ctx, shape, nb, seed)
    parts = o.sample(img).astype(np.float32)
    stack = oracle.downsampled_stencils(oracle.gaussian_stencil((size / 4.0,) * 3, (size,) * 3, True), o.l_max - o.l_min, True, "oracle")
    exp = o.convolve_pencil(stack, parts, reflect)
    got = A.APRFilter.convolve_pencil(g, stack, parts, reflect_boundary=reflect)
    w = _wide(o, stack)
    assert w.mean() > 0.9   # the two finest levels at least
    assert _rel(got, exp)[w].max() <= 2 * (max(size, 3) ** 3 + 3 * max(size, 3) + 3) * 2.0 ** -24


@pytest.mark.parametrize("shape,nb,seed", EDGES)
@pytest.mark.parametrize("size", [1, 3, 5, 7, 9, 11, 13])
@pytest.mark.parametrize("reflect", [True, False])
def test_convolve_separable_lists(oracle, sep_ctx, shape, nb, seed, size, reflect):
    """lists of which one level's stencil is of another form: the cubic ones, the finest or the coarser, take the
    kernel with the z ring in registers (bound as above).  The finest level's stencil is the widest: the oracle's
    windows have its size"""
    img, o, g = _pair(oracle, sep_ctx, shape, nb, seed)
    wide = oracle.gaussian_stencil((1.0, 1.0, 1.0), (size + 2, size, size), True)
    narrow = oracle.gaussian_stencil((1.0, 1.0, 1.0), (min(size, 3), 1, min(size, 3)), True)
    stack = oracle.downsampled_stencils(oracle.gaussian_stencil((size / 4.0,) * 3, (size,) * 3, True), o.l_max - o.l_min, True, "oracle")
    for at, other in ((0, wide), (-1, narrow)):
        st = list(stack)
        st[at] = other
        w = _wide(o, st)
        assert w.mean() > 0.9
        for parts in (o.sample(img), o.sample(img).astype(np.float32) * np.float32(0.83)):
            exp = o.convolve_pencil(st, parts, reflect)
            got = A.APRFilter.convolve_pencil(g, st, parts, reflect_boundary=reflect)
            assert _rel(got, exp)[w].max() <= 2 * ((size + 2) ** 3 + 3 * (size + 2) + 3) * 2.0 ** -24


def test_richardson_lucy_wide_psf(oracle, sep_ctx):
    """a PSF of 15 taps a side: its finest level and the coarser ones (9, 5 and 3 taps) take different
    kernels, with the ratio and the update at their outputs"""
    img, o, g = _pair(oracle, sep_ctx, (40, 48, 66), 30, 6)
    psf = oracle.gaussian_stencil((2.0, 2.0, 2.5), (15, 15, 15), True)
    w = _wide(o, oracle.downsampled_stencils(psf, o.l_max - o.l_min, True, "oracle"))
    assert w.mean() > 0.9
    for parts in (o.sample(img), o.sample(img).astype(np.float32) * np.float32(0.83)):
        uo, _, _ = o.richardson_lucy(parts, psf, 2)
        ug, _ = A.APRNumerics.richardson_lucy(g, parts, None, psf, 2, normalize=True)
        assert _rel(ug, uo)[w].max() < 1e-5


@pytest.mark.parametrize("size", [5, 9])
@pytest.mark.parametrize("separable", [False, True])
def test_richardson_lucy_edges(oracle, ctx, sep_ctx, size, separable):
    """the ratio and the update, made where the convolutions write their results"""
    c = sep_ctx if separable else ctx
    img, o, g = _pair(oracle, c, (21, 33, 65), 20, 6)
    psf = oracle.gaussian_stencil((1.0, 1.0, 1.5), (size,) * 3, True)
    assert _wide(o, oracle.downsampled_stencils(psf, o.l_max - o.l_min, True, "oracle")).all()
    for parts in (o.sample(img), o.sample(img).astype(np.float32) * np.float32(0.83)):
        uo, _, _ = o.richardson_lucy(parts, psf, 2)
        ug, _ = A.APRNumerics.richardson_lucy(g, parts, None, psf, 2, normalize=True)
        if separable:
            assert _rel(ug, uo).max() < 1e-5
        else:
            assert np.array_equal(_bits(ug), _bits(uo))


def test_richardson_lucy_tv_separable_mode(oracle, sep_ctx):
    img, o, g = _pair(oracle, sep_ctx, *CASES[0])
    parts = o.sample(img)
    psf = oracle.gaussian_stencil((1.0, 1.0, 2.0), (9, 9, 9), True)
    uo = o.richardson_lucy_tv(parts, psf, 3, 0.01)
    ug = A.APRNumerics.richardson_lucy_tv(g, parts, None, psf, 3, 0.01, normalize=True)
    r = _rel(ug, uo).max()
    l2 = float(np.linalg.norm(ug.astype(np.float64) - uo) / np.linalg.norm(uo.astype(np.float64)))
    print(f"RL-TV 3 iterations, separable vs reference order: max rel {r:.2e}, rel L2 {l2:.2e}")
    # the normalised gradient turns where |grad u| is near zero, so single particles may differ
    # more than the convolutions do; the whole estimate stays within float rounding
    assert l2 < 1e-5


def test_richardson_lucy_separable_mode(oracle, sep_ctx):
    img, o, g = _pair(oracle, sep_ctx, *CASES[0])
    parts = o.sample(img)
    psf = oracle.gaussian_stencil((1.0, 1.0, 2.0), (9, 9, 9), True)
    uo, _, _ = o.richardson_lucy(parts, psf, 3)
    ug, st = A.APRNumerics.richardson_lucy(g, parts, None, psf, 3, normalize=True)
    r = _rel(ug, uo).max()
    print(f"RL 3 iterations, separable vs reference order: max rel {r:.2e}")
    assert st["iterations"] == 3 and r < 1e-5


def _level_image(o):
    """reconstruct_level restated from the structure (APRReconstruction.hpp:131-171): the
    particle of level l at row (z, x), position y covers the block [z, x, y] * 2^(l_max - l)"""
    y, x, z = o.dims
    img = np.zeros((z, x, y), np.uint16)
    lxz, xze, yv = o.level_xz_vec, o.xz_end_vec, o.y_vec
    for lev in range(o.l_min, o.l_max + 1):
        s = 2 ** (o.l_max - lev)
        xl, zl = -(-x // s), -(-z // s)
        for zi in range(zl):
            for xi in range(xl):
                r = int(lxz[lev]) + zi * xl + xi
                b = int(xze[r - 1]) if r > 0 else 0
                for yy in yv[b:int(xze[r])]:
                    img[zi * s:(zi + 1) * s, xi * s:(xi + 1) * s, int(yy) * s:(int(yy) + 1) * s] = lev
    return img


@pytest.mark.parametrize("shape,nb,seed", CASES[:3])
def test_reconstruct_level(oracle, ctx, shape, nb, seed):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    expect = _level_image(o)
    # the same image as the constant reconstruction of particles valued by their levels
    lev = np.zeros(o.total, np.uint16)
    for l in range(o.l_min, o.l_max + 1):
        r0 = int(o.level_xz_vec[l])
        b = int(o.xz_end_vec[r0 - 1]) if r0 > 0 else 0
        e = int(o.xz_end_vec[int(o.level_xz_vec[l + 1]) - 1])
        lev[b:e] = l
    assert np.array_equal(o.reconstruct(lev, 0, np.uint16), expect)
    assert int(expect.min()) >= o.l_min and int(expect.max()) == o.l_max
    for out_dtype in (np.uint16, np.float32):
        got = A.APRReconstruction.reconstruct_level(g, out_dtype)
        assert got.dtype == out_dtype and np.array_equal(got, expect.astype(out_dtype))


@pytest.mark.parametrize("shape,nb,seed,delta", [((3, 5, 1025), 6, 1, 0), ((5, 3, 2049), 6, 2, 0), ((4, 7, 4133), 9, 3, 0), ((5, 4, 4133), 9, 3, -1),
                                                 ((2, 9, 2050), 4, 4, 0)])
def test_reconstruct_long_rows(oracle, ctx, shape, nb, seed, delta):
    """rows of more than one 4096-byte piece (1024 f32, 2048 u16), whose levels' entries are found by
    search, at row starts of every alignment; and coarse cells wider than a piece"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    for out_dtype in (np.uint16, np.float32):
        assert np.array_equal(A.APRReconstruction.reconstruct_constant(g, parts, delta, out_dtype), o.reconstruct(parts, delta, out_dtype))
    if delta == 0:
        for out_dtype in (np.uint16, np.float32):
            assert np.array_equal(A.APRReconstruction.reconstruct_level(g, out_dtype), _level_image(o).astype(out_dtype))


def _level_image(o):
    lev = np.concatenate([np.full(n, l, np.uint16) for l, n in _particles_per_level(o)])
    return o.reconstruct(lev, 0, np.uint16)


def _particles_per_level(o):
    """(level, particles) of an oracle APR, from its row ends"""
    ends = o.xz_end_vec
    d = max(o.dims)
    out, row = [], 1
    for l in range(o.l_min, o.l_max + 1):
        s = 1 << (o.l_max - l)
        n = -(-o.dims[1] // s) * -(-o.dims[2] // s)
        out.append((l, int(ends[row + n - 1] - ends[row - 1])))
        row += n
    assert d <= 1 << o.l_max and sum(n for _, n in out) == o.total
    return out


@pytest.mark.parametrize("shape,nb,seed", [((3, 3, 6200), 5, 1), ((2, 3, 40001), 9, 2), ((90, 5, 70), 6, 3), ((5, 91, 67), 6, 4)])
def test_reconstruct_smooth_line_forms(oracle, ctx, shape, nb, seed):
    """one line of y in LDS, a line longer than LDS holds (marched), and x / z lines long and short
    against the ring of 42 sums"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    for out_dtype in (np.uint16, np.float32):
        for sc in ((2.0, 2.0, 2.0), (0.3, 0.5, 0.4)):
            exp = o.reconstruct_smooth(parts, scale=sc, out_dtype=out_dtype)
            got = A.APRReconstruction.reconstruct_smooth(g, parts, scale_d=sc, out_dtype=out_dtype)
            assert np.array_equal(got.view(np.uint8), exp.view(np.uint8)), (out_dtype, sc, int((got != exp).sum()))


@pytest.mark.parametrize("shape,nb,seed", CASES[:3] + [((3, 9, 40), 2, 8)])
def test_reconstruct_smooth(oracle, ctx, shape, nb, seed):
    """reconstruct_smooth bit-equal to the oracle: u16 and f32 particles into u16 and f32 images,
    the default scale and an anisotropic one, and a scale so large that no pixel is smoothed"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    pu = o.sample(img)
    pf = (pu.astype(np.float32) * np.float32(0.37)) + np.float32(1.5)
    for parts in (pu, pf):
        for out_dtype in (np.uint16, np.float32):
            for sc in ((2.0, 2.0, 2.0), (1.0, 0.7, 3.0), (1e6, 1e6, 1e6)):
                exp = o.reconstruct_smooth(parts, scale=sc, out_dtype=out_dtype)
                got = A.APRReconstruction.reconstruct_smooth(g, parts, scale_d=sc, out_dtype=out_dtype)
                assert got.dtype == exp.dtype
                if out_dtype == np.float32:
                    ok = np.array_equal(_bits(got), _bits(exp))
                else:
                    ok = np.array_equal(got, exp)
                assert ok, (parts.dtype, out_dtype, sc, int((got != exp).sum()))


def _patch_restated(o, values, tree_values, p, out_dtype):
    """the patch loop of APRReconstruction.hpp:296-394 (reconstruct_level :397-490 is the same
    loop with level-valued particles and the patch level for tree nodes), row by row"""
    y, x, z = o.dims
    max_level = o.l_max + p.level_delta
    img = np.zeros((p.z_end - p.z_begin, p.x_end - p.x_begin, p.y_end - p.y_begin), out_dtype)
    lxz, xze, yv = o.level_xz_vec, o.xz_end_vec, o.y_vec

    def row(lxz_, xze_, lev, zz, xx):
        xl = -(-x // 2 ** (o.l_max - lev))
        r = int(lxz_[lev]) + zz * xl + xx
        return (int(xze_[r - 1]) if r > 0 else 0), int(xze_[r])

    for xx in range(p.x_begin, p.x_end):
        for zz in range(p.z_begin, p.z_end):
            for lev in range(min(max_level, o.l_max), o.l_min - 1, -1):
                ylev = -(-y // 2 ** (o.l_max - lev))
                if lev == max_level:
                    b, e = row(lxz, xze, lev, zz, xx)
                    for i in range(b, e):
                        if p.y_begin <= yv[i] < p.y_end:
                            img[zz - p.z_begin, xx - p.x_begin, int(yv[i]) - p.y_begin] = values[i]
                else:
                    step = 2 ** (max_level - lev)
                    b, e = row(lxz, xze, lev, zz // step, xx // step)
                    ybl, yel = p.y_begin // step, min(-(-p.y_end // step), ylev)
                    for i in range(b, e):
                        if ybl <= yv[i] < yel:
                            lo = max(int(yv[i]) * step, p.y_begin) - p.y_begin
                            hi = min((int(yv[i]) + 1) * step, p.y_end) - p.y_begin
                            img[zz - p.z_begin, xx - p.x_begin, lo:hi] = values[i]
    if max_level < o.l_max:
        t = o.tree()
        for xx in range(p.x_begin, p.x_end):
            for zz in range(p.z_begin, p.z_end):
                b, e = row(t["level_xz_vec"], t["xz_end_vec"], max_level, zz, xx)
                for i in range(b, e):
                    yy = int(t["y_vec"][i])
                    if p.y_begin <= yy < p.y_end:
                        img[zz - p.z_begin, xx - p.x_begin, yy - p.y_begin] = tree_values[i]
    return img


def _levels_of(o):
    lev = np.zeros(o.total, np.uint16)
    for l in range(o.l_min, o.l_max + 1):
        r0 = int(o.level_xz_vec[l])
        b = int(o.xz_end_vec[r0 - 1]) if r0 > 0 else 0
        lev[b:int(o.xz_end_vec[int(o.level_xz_vec[l + 1]) - 1])] = l
    return lev


PATCHES = [dict(x_begin=3, x_end=40, y_begin=5, y_end=50, z_begin=2, z_end=20),
           dict(x_begin=-4, x_end=1000, y_begin=17, y_end=-1, z_begin=9, z_end=-1),
           dict(x_begin=1, x_end=12, y_begin=3, y_end=21, z_begin=0, z_end=7, level_delta=-1),
           dict(x_begin=2, x_end=9, y_begin=0, y_end=-1, z_begin=1, z_end=5, level_delta=-2),
           dict(x_begin=7, x_end=50, y_begin=11, y_end=90, z_begin=3, z_end=19, level_delta=1)]


@pytest.mark.parametrize("shape,nb,seed", CASES[:2])
@pytest.mark.parametrize("pi", range(len(PATCHES)))
def test_reconstruct_patch(oracle, ctx, shape, nb, seed, pi):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    p = A.ReconPatch(**PATCHES[pi])
    assert p.check_limits(g)
    d = p.level_delta
    # the restated loop against a cut of the oracle's whole-image reconstruction
    full = o.reconstruct(parts, min(d, 0), np.uint16)
    if d > 0:
        full = full.repeat(2 ** d, 0).repeat(2 ** d, 1).repeat(2 ** d, 2)
    cut = full[p.z_begin:p.z_end, p.x_begin:p.x_end, p.y_begin:p.y_end]
    tree = o.fill_tree_mean(parts) if d < 0 else None
    exp = _patch_restated(o, parts, tree, p, np.uint16)
    assert np.array_equal(exp, cut)
    got = A.APRReconstruction.reconstruct_constant(g, parts, patch=A.ReconPatch(**PATCHES[pi]))
    assert got.dtype == np.uint16 and np.array_equal(got, exp)
    gotf = A.APRReconstruction.reconstruct_constant(g, parts, out_dtype=np.float32, patch=A.ReconPatch(**PATCHES[pi]))
    expf = _patch_restated(o, parts.astype(np.float32), tree, p, np.float32)
    assert np.array_equal(_bits(gotf), _bits(expf))
    # levels: the particles' levels, capped at the patch level (tree nodes take the patch level)
    lev = _levels_of(o)
    maxl = o.l_max + d
    tl = np.full(o.tree()["total"], maxl, np.uint16) if d < 0 else None
    expl = _patch_restated(o, np.minimum(lev, maxl), tl, p, np.uint16)
    gotl = A.APRReconstruction.reconstruct_level(g, patch=A.ReconPatch(**PATCHES[pi]))
    assert np.array_equal(gotl, expl)
    if d == 0:
        assert np.array_equal(expl, _level_image(o)[p.z_begin:p.z_end, p.x_begin:p.x_end, p.y_begin:p.y_end])


def test_reconstruct_patch_limits(oracle, ctx):
    img, o, g = _pair(oracle, ctx, *CASES[1])
    y, x, z = o.dims
    p = A.ReconPatch(x_begin=-3, y_end=10 ** 6, z_begin=2, level_delta=-1)
    assert p.check_limits(g)
    assert (p.x_begin, p.x_end, p.y_begin, p.y_end, p.z_begin, p.z_end) == (0, -(-x // 2), 0, -(-y // 2), 2, -(-z // 2))
    for bad in (dict(x_begin=5, x_end=5), dict(y_begin=10 ** 6), dict(z_begin=3, z_end=2), dict(level_delta=40)):
        assert not A.ReconPatch(**bad).check_limits(g)
        with pytest.raises(ValueError):
            A.APRReconstruction.reconstruct_level(g, patch=A.ReconPatch(**bad))
    with pytest.raises(A.AprhError):
        A.APRReconstruction.reconstruct_level(g, patch=A.ReconPatch(level_delta=-(o.l_max - o.l_min) - 1))


def _gradient_stack(o, dim, delta, sobel):
    """APRNumerics::gradient_cfd / gradient_sobel's stencils (APRNumerics.hpp:165-213,
    APRStencil.hpp:135-152, :254-297) restated in float32, [z, x, y]"""
    y, x, z = o.dims
    nd = int(y > 1) + int(x > 1) + int(z > 1)
    h = np.float32(1.0) / (np.float32(2.0) * np.float32(delta))
    diff = np.array([-h, 0.0, h], np.float32)
    sm = np.array([0.25, 0.5, 0.25], np.float32)
    fy, fx, fz = (diff if dim == 0 else sm), (diff if dim == 1 else sm), (diff if dim == 2 else sm)
    if sobel and nd == 3:
        st = (fy[None, None, :] * fx[None, :, None]) * fz[:, None, None]
    elif sobel and nd == 2 and dim != 2:
        st = (fy[None, None, :] * fx[None, :, None]).astype(np.float32)
    else:
        st = diff.reshape([(3, 1, 1), (1, 3, 1), (1, 1, 3)][2 - dim])
    st = st.astype(np.float32)
    return [st / np.float32(2.0 ** d) for d in range(max(o.l_max - o.l_min, 1))]


@pytest.mark.parametrize("shape,nb,seed", CASES[:3])
@pytest.mark.parametrize("sobel", [False, True])
def test_gradients(oracle, ctx, shape, nb, seed, sobel):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    pf = (parts.astype(np.float32) * np.float32(0.731)).astype(np.float32)
    fn = A.APRNumerics.gradient_sobel if sobel else A.APRNumerics.gradient_cfd
    grads = []
    for dim, delta in ((0, 1.0), (1, 0.7), (2, 2.5)):
        stack = _gradient_stack(o, dim, delta, sobel)
        exp = o.convolve_pencil(stack, parts, True)
        got = fn(g, parts, dimension=dim, delta=delta)
        assert np.array_equal(_bits(got), _bits(exp)), (dim, int((_bits(got) != _bits(exp)).sum()))
        assert np.array_equal(_bits(fn(g, pf, dimension=dim, delta=delta)), _bits(o.convolve_pencil(stack, pf, True)))
        grads.append(exp)
    # the magnitude in the reference's order: g_y^2, + g_x^2, + g_z^2, sqrtf
    m = grads[0] * grads[0]
    m = (m + grads[1] * grads[1]).astype(np.float32)
    m = (m + grads[2] * grads[2]).astype(np.float32)
    m = np.sqrt(m).astype(np.float32)
    mfn = A.APRNumerics.gradient_magnitude_sobel if sobel else A.APRNumerics.gradient_magnitude_cfd
    assert np.array_equal(_bits(mfn(g, parts, deltas=(1.0, 0.7, 2.5))), _bits(m))
    # and against the reference's own APRNumerics, where its build is present
    if oracle.load("ref") is not None and hasattr(oracle.load("ref"), "orc_gradient_u16"):
        r = oracle.apr_from_structure(o.dims, o.xz_end_vec, o.y_vec, "ref")
        for dim, delta in ((0, 1.0), (1, 0.7), (2, 2.5)):
            for p in (parts, pf):
                assert np.array_equal(_bits(fn(g, p, dimension=dim, delta=delta)), _bits(r.gradient(p, sobel, dim, delta)))
        assert np.array_equal(_bits(mfn(g, pf, deltas=(1.0, 0.7, 2.5))), _bits(r.gradient_magnitude(pf, sobel, (1.0, 0.7, 2.5))))
    with pytest.raises(A.AprhError):
        fn(g, parts, dimension=3)


def test_gradient_of_a_constant_is_zero(oracle, ctx):
    img, o, g = _pair(oracle, ctx, *CASES[3])
    c = np.full(o.total, 1234, np.uint16)
    for fn in (A.APRNumerics.gradient_cfd, A.APRNumerics.gradient_sobel):
        for dim in range(3):
            assert np.all(fn(g, c, dimension=dim) == 0.0)
    assert np.all(A.APRNumerics.gradient_magnitude_sobel(g, c) == 0.0)


@pytest.mark.parametrize("shape,nb,seed", CASES[:3])
@pytest.mark.parametrize("size", [(3, 3, 3), (5, 3, 1)])
def test_local_std(oracle, ctx, shape, nb, seed, size):
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    assert np.array_equal(_bits(A.APRNumerics.local_std(g, parts, size=size)), _bits(o.local_std(parts, size)))
    pf = (parts.astype(np.float32) * np.float32(0.37)).astype(np.float32)
    assert np.array_equal(_bits(A.APRNumerics.local_std(g, pf, size=size)), _bits(o.local_std(pf, size)))


@pytest.mark.parametrize("shape,nb,seed", CASES + [((1, 70, 90), 6, 5), ((33, 17, 9), 5, 6)])
def test_face_neighbour_filters(oracle, ctx, shape, nb, seed):
    """APRNumerics::face_neighbour_filter / seperable_face_neighbour_filter, bit-equal to the
    oracle (itself bit-equal to the reference build), u16 and f32 input"""
    img, o, g = _pair(oracle, ctx, shape, nb, seed)
    parts = o.sample(img)
    pf = (parts.astype(np.float32) * np.float32(0.37)).astype(np.float32)
    f = np.array([0.25, 0.5, 0.3], np.float32)
    for p in (parts, pf):
        for dim in range(3):
            got = A.APRNumerics.face_neighbour_filter(g, p, f, dim)
            exp = o.face_neighbour_filter(p.astype(np.float32), f, dim)
            assert np.array_equal(_bits(got), _bits(exp)), (dim, int((_bits(got) != _bits(exp)).sum()))
    for rep in (0, 1, 2):
        got = A.APRNumerics.seperable_face_neighbour_filter(g, pf, f, rep)
        assert np.array_equal(_bits(got), _bits(o.face_neighbour_filter(pf, f, 0, rep))), rep



def _with_holes(oracle, shape, nb, seed, keep):
    """a converted APR's structure with only the particles that keep(level, z, x, y) wants: (dims, xz_end, y_vec)"""
    o = oracle.get_apr(A.synth_blobs(shape, seed, nb), oracle.params(rel_error=0.1, sigma_th=50, Ip_th=120, grad_th=10), "oracle")
    ends, yv = o.xz_end_vec.astype(np.int64), o.y_vec
    y, x, z = o.dims
    new, out, row = [0], [], 1
    for l in range(o.l_min, o.l_max + 1):
        s = 1 << (o.l_max - l)
        for zz in range(-(-z // s)):
            for xx in range(-(-x // s)):
                ys = yv[ends[row - 1]:ends[row]]
                out.append(np.array([v for v in ys if keep(l, zz, xx, int(v))], np.uint16))
                new.append(new[-1] + len(out[-1]))
                row += 1
    assert row == len(ends)
    return o.dims, np.array(new, np.uint64), np.concatenate(out)


def _images(apr, parts, tree_values):
    """per level (image of its particles, coarser ones and its tree nodes' values, with 0 where nothing is;
    the particles' (z, x, y)): what a convolution at that level reads"""
    y, x, z = apr.org_dims
    _, ends, yv = apr.structure()
    tree = apr.tree()
    tends, tyv, tlxz = tree["xz_end_vec"], tree["y_vec"], tree["level_xz_vec"]
    res, row, prev = {}, 1, None
    for l in range(apr.l_min, apr.l_max + 1):
        s = 1 << (apr.l_max - l)
        d = (-(-z // s), -(-x // s), -(-y // s))
        v = np.zeros(d, np.float32) if prev is None else prev.repeat(2, 0).repeat(2, 1).repeat(2, 2)[:d[0], :d[1], :d[2]].copy()
        at = []
        for r in range(d[0] * d[1]):
            for i in range(int(ends[row - 1]), int(ends[row])):
                at.append((r // d[1], r % d[1], int(yv[i])))
                v[at[-1]] = parts[i]
            row += 1
        if tree_values is not None and l < apr.l_max:
            for r in range(d[0] * d[1]):
                q = int(tlxz[l]) + r
                for i in range(int(tends[q - 1]), int(tends[q])):
                    v[r // d[1], r % d[1], int(tyv[i])] = tree_values[i]
        res[l] = (v, at)
        prev = v
    return res


@pytest.mark.parametrize("shape,nb,seed", [((9, 17, 70), 5, 1), ((20, 6, 33), 4, 2), ((3, 3, 2100), 9, 3)])
@pytest.mark.parametrize("what", ["scattered", "rows", "coarse", "nothing"])
def test_structure_with_uncovered_cells(oracle, ctx, shape, nb, seed, what):
    """a stored structure's particles need not cover the image: a cell without any reads the nearest tree node
    above it in a convolution, else 0, and is 0 in a reconstruction, whatever the memory held before"""
    keep = {"scattered": lambda l, z, x, y: (7 * y + 3 * x + z) % 5 != 0, "rows": lambda l, z, x, y: (x + z) % 3 != 0,
            "coarse": lambda l, z, x, y: l >= 5, "nothing": lambda l, z, x, y: False}[what]
    dims, xz, yv = _with_holes(oracle, shape, nb, seed, keep)
    A.APRReconstruction.reconstruct_constant(*(lambda i, o, g: (g, o.sample(i)))(*_pair(oracle, ctx, shape, nb, seed)))   # leaves values in LDS
    g = A.APR.from_structure(dims, xz, yv, ctx=ctx)
    parts = np.random.default_rng(seed).uniform(1, 100, len(yv)).astype(np.float32)
    tv = A.APRTreeNumerics.fill_tree_mean(g, parts) if what != "nothing" else np.zeros(0, np.float32)
    images = _images(g, parts, tv)
    nlev = g.l_max - g.l_min + 1
    for tap in ((0, 1, 2), (1, 1, 1), (2, 0, 1)):
        st = np.zeros((3, 3, 3), np.float32)
        st[tap] = 1.0
        exp = []
        for l in range(g.l_min, g.l_max + 1):
            v, at = images[l]
            w = np.pad(v, 1)
            exp += [w[z + tap[0], x + tap[1], y + tap[2]] for z, x, y in at]
        exp = np.array(exp, np.float32)
        got = A.APRFilter.convolve_pencil(g, [st] * nlev, parts, reflect_boundary=False)
        assert np.array_equal(got, exp)
        wide = np.zeros((3, 5, 3), np.float32)   # the same tap in a stencil that other kernels take
        wide[tap[0], tap[1] + 1, tap[2]] = 1.0
        assert np.array_equal(A.APRFilter.convolve_pencil(g, [wide] * nlev, parts, reflect_boundary=False), exp)
    plain = _images(g, parts, None)[g.l_max][0]
    for dt in (np.uint16, np.float32):
        assert np.array_equal(A.APRReconstruction.reconstruct_constant(g, parts, 0, dt), plain.astype(dt))
    levels = _images(g, np.concatenate([np.full(len(images[l][1]), l, np.float32) for l in images]), None)[g.l_max][0]
    assert np.array_equal(A.APRReconstruction.reconstruct_level(g), levels.astype(np.uint16))
    for dt in (np.uint16, np.float32):
        s0 = A.APRReconstruction.reconstruct_smooth(g, parts, out_dtype=dt)
        # half-widths of 0 everywhere leave the running sums' differences: the image up to their rounding
        s1 = A.APRReconstruction.reconstruct_smooth(g, parts, scale_d=(1e9,) * 3, out_dtype=dt)
        assert np.isfinite(s0.astype(np.float64)).all() and s0.max() <= 101
        tol = 3 * max(shape) * 100 * max(shape) * 2.0 ** -24 if dt == np.float32 else 3
        assert np.abs(s1.astype(np.float64) - plain.astype(dt)).max() <= tol
    g.close()


@pytest.mark.parametrize("y,left", [(4096, 12 << 30), (65535, None)])
def test_convolve_without_room_for_level_images(sep_ctx, y, left):
    """y x 1024 x 1024 with all particles at the level of 16-voxel cells, where the images of all levels would take
    19.6 GB of 12 that are left, or 314 GB.  The other kernels' two (4.3 GB, 69 GB) have room, and give what the same
    cells give as an APR of y / 16 x 64 x 64"""
    sep_ctx.release_cache()
    torch.cuda.empty_cache()
    free, total = torch.cuda.mem_get_info()
    if left is None and total > 4 * 8 * y * 1024 * 1024 // 7:
        pytest.skip("a device with room for the images")
    n, side = -(-y // 16), 64

    def one_level(dims, level):
        """(xz_end, y_vec) of particles in all cells of one level, n x 64 x 64 of them"""
        top = int(np.ceil(np.log2(max(dims))))
        rows = [-(-dims[1] // 2 ** (top - l)) * -(-dims[2] // 2 ** (top - l)) for l in range(1, top + 1)]
        assert rows[level - 1] == side * side and -(-dims[0] // 2 ** (top - level)) == n
        ends = np.concatenate([np.zeros(1 + sum(rows[:level - 1])), np.arange(1, side * side + 1) * n, np.full(sum(rows[level:]), side * side * n)])
        return ends.astype(np.uint64), np.tile(np.arange(n, dtype=np.uint16), side * side)

    top = int(np.ceil(np.log2(y)))
    parts = np.random.default_rng(0).uniform(50, 150, n * side * side).astype(np.float32)
    small = A.APR.from_structure((n, side, side), *one_level((n, side, side), top - 4), sep_ctx)
    big = A.APR.from_structure((y, 1024, 1024), *one_level((y, 1024, 1024), top - 4), sep_ctx)
    print("structures made", flush=True)
    g3 = A.APRStencil.create_gaussian_filter((0.75,) * 3, (3,) * 3, True)
    g5 = A.APRStencil.create_gaussian_filter((1.25,) * 3, (5,) * 3, True)
    taken = torch.empty(torch.cuda.mem_get_info()[0] - left, dtype=torch.uint8, device="cuda") if left else None
    got = A.APRFilter.convolve_pencil(big, [g3] * 4 + [g5], parts)
    ug, _ = A.APRNumerics.richardson_lucy(big, parts, None, g3, 1, use_stencil_downsample=False)
    print("done", flush=True)
    big.close()
    sep_ctx.release_cache()
    del taken
    torch.cuda.empty_cache()
    exp = A.APRFilter.convolve_pencil(small, [g5], parts)
    assert _rel(got, exp).max() <= 2 * (5 ** 3 + 3 * 5 + 3) * 2.0 ** -24
    us, _ = A.APRNumerics.richardson_lucy(small, parts, None, g3, 1, use_stencil_downsample=False)
    assert _rel(ug, us).max() < 1e-5
    small.close()
