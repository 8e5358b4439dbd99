"""The measurement pass against slice means in extended precision, on sides
where its tiles are ragged or a block takes several y tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    import langevina_amd
    langevina_amd.lib()
    return langevina_amd


def contract(n, A, V):
    return [-(n[1] * A[0]) - n[2] * A[1] - n[3] * A[2], n[0] * A[0] + n[3] * V[1] - n[2] * V[2],
            n[0] * A[1] - n[3] * V[0] + n[1] * V[2], n[0] * A[2] + n[2] * V[0] - n[1] * V[1]]


def observables(u):
    """The 25 observables of u[z, y, x, 10] (measurer.cxx:245-269, 351-392)."""
    f = np.moveaxis(u, 3, 0)
    phi2 = (f[:4] ** 2).sum(0)
    sigma = np.sqrt(phi2)
    ok = phi2 > 100 * np.finfo(float).tiny
    n = np.where(ok, f[:4] / np.where(ok, sigma, 1.), np.array([1., 0, 0, 0]).reshape(4, 1, 1, 1))
    A, V = f[4:7], f[7:]
    return [*f, phi2, sigma, *n, *contract(n, A, V), *contract(n, V, A), sigma * sigma]


# 4, 6, 10: one tile wraps the lattice, some lanes idle; 34, 50, 90: rows of one
# tile, short last y tile; 66, 130: rows split in two and three; 256: chunks of
# many planes
@pytest.mark.parametrize("N,prec", [(4, 0), (6, 1), (10, 0), (34, 0), (50, 1), (66, 0), (90, 0),
                                    (130, 1), (256, 1)])
def test_walls_are_the_slice_means(L, N, prec):
    print(f"[gpu-test] walls {N} {prec}", flush=True)
    u = np.random.default_rng(N).normal(size=(N, N, N, 10))
    u[0, 0, 0, :4] = 0.  # the |phi| = 0 branch
    if prec:
        u = u.astype(np.float32).astype(np.float64)
    ctx = L.Context(L.model_params(N), precision=prec)
    ctx.set_field(u)
    m = ctx.measure_full()
    wall, phase, oavg = ctx.measure()
    ctx.close()
    np.testing.assert_array_equal(wall, m["wall"])
    np.testing.assert_array_equal(phase, m["wallphase"])
    eps = np.finfo(float).eps
    walls = np.concatenate([wall, phase], axis=1)
    for o, f in enumerate(observables(u)):
        mag = np.abs(f)
        for d, axes in enumerate(((0, 1), (0, 2), (1, 2))):  # x, y, z walls of f[z, y, x]
            ref = f.sum(axis=axes, dtype=np.longdouble) / N ** 2
            # a site's value carries at most 8 roundings (n, A', V'), the
            # compensated sum and the division two more
            tol = 10 * eps * mag.mean(axis=axes) + 1e-300
            assert (np.abs(walls[d, o] - ref) <= tol).all(), (d, o)
    for w, wk in ((wall, m["wall_k"]), (phase, m["wallphase_k"])):
        ref = np.fft.rfft(w, axis=-1) / N
        assert np.abs(wk - ref).max() <= 8 * eps * np.abs(w).mean(-1).max() * np.log2(N)
    np.testing.assert_allclose(oavg, wall[0].mean(1), rtol=1e-13, atol=1e-15)


def test_walls_of_a_large_lattice(L):
    """N = 520: a block takes two y tiles one after the other and adds to its
    own z-wall sums.  phi_1 = g(x) + h(y) + k(z) with integer values, so every
    slice mean is known exactly."""
    print("[gpu-test] walls 520", flush=True)
    N = 520
    g, h, k = (np.random.default_rng(s).integers(-8, 8, N).astype(float) for s in (1, 2, 3))
    u = np.zeros((N, N, N, 10))
    u[..., 1] = g[None, None, :] + h[None, :, None] + k[:, None, None]
    u[..., 4] = 2.0
    ctx = L.Context(L.model_params(N), precision=L.FP32)
    ctx.set_field(u)
    wall, _, _ = ctx.measure()
    ctx.close()
    for d, (own, a, b) in enumerate(((g, h, k), (h, g, k), (k, g, h))):
        np.testing.assert_allclose(wall[d, 1], own + a.mean() + b.mean(), rtol=4e-16, atol=1e-14)
    np.testing.assert_array_equal(wall[:, 4], np.full((3, N), 2.0))


# Sides whose tiles and chunks are whole periods of the sign pattern below; 448:
# a wavefront takes four z tiles in turn
@pytest.mark.parametrize("N", [64, 128, 448])
def test_sums_are_compensated_whatever_the_first_row_holds(L, N):
    """Charges of +-2^16 that cancel in fours, plus noise of 2^-16, with rows
    y = 0, 4, ... (the first of every chunk) that hold the noise alone, or
    nothing: the walls in which the large values cancel inside a wavefront
    keep only the noise."""
    print(f"[gpu-test] compensated walls {N}", flush=True)
    M, quantum = 2.0 ** 16, 2.0 ** -36  # M + k quantum is exact for |k| <= 2^20
    i = np.arange(N)
    p = np.array([0, 1, -1, 0], np.int64)[i % 4]
    late = (i % 4 != 0).astype(np.int64)
    one = np.ones(N, np.int64)
    # sign(z) sign(y) sign(x) of component 4, 5, 6, 7, and whether its rows
    # y = 0, 4, ... hold noise
    signs = {4: (one, p, one, True), 5: (one, late, p, True), 6: (p, late, one, True),
             7: (one, late, p, False)}
    u = np.zeros((N, N, N, 10))
    u[..., 0] = 1.0  # n = (1, 0, 0, 0): the A' and V' are the charges
    rng = np.random.default_rng(N)
    hi, lo, mag = {}, {}, {}
    axes = ((0, 1), (0, 2), (1, 2))  # x, y, z walls of f[z, y, x]
    for o, (sz, sy, sx, noise) in signs.items():
        k = rng.integers(-2 ** 20, 2 ** 20 + 1, (N, N, N))
        if not noise:
            k *= late[None, :, None]
        u[..., o] = sz[:, None, None] * sy[None, :, None] * sx[None, None, :] * M + k * quantum
        for d, ax in enumerate(axes):
            lo[o, d] = k.sum(axis=ax).astype(np.longdouble) * quantum
            mag[o, d] = np.abs(k).sum(axis=ax) * quantum / N ** 2
        for d, (a, b, own) in enumerate(((sz, sy, sx), (sz, sx, sy), (sy, sx, sz))):
            hi[o, d] = (a.sum() * b.sum() * own).astype(np.longdouble) * M
    ctx = L.Context(L.model_params(N))
    ctx.set_field(u)
    wall, phase, _ = ctx.measure()
    ctx.close()
    x, y, z = 0, 1, 2
    cancels = {(4, x), (4, z), (5, y), (7, y)} | ({(6, y)} if N == 448 else set())
    unit = 2.0 ** -53
    for o in signs:
        for d in (x, y, z):
            ref = (hi[o, d] + lo[o, d]) / N ** 2
            # at most four roundings: a column's sum over a chunk, a tile's sum,
            # the wall's, and the division; the corrections themselves round
            # in second order (chunks and rows of at most 224 terms)
            tol = 4 * unit * mag[o, d] + unit ** 2 * N ** 2 * M
            if (o, d) not in cancels:
                tol = tol + 4 * unit * M
            assert (np.abs(wall[d, o] - ref) <= tol).all(), (o, d)
    np.testing.assert_array_equal(phase[:, 6:9], wall[:, 4:7])
    np.testing.assert_array_equal(phase[:, 10], wall[:, 7])


def test_walls_of_n_where_the_square_of_phi_overflows(L):
    """phi^2 = inf of finite phi: n = phi / inf = 0 there, and A', V' with it."""
    print("[gpu-test] walls, overflow", flush=True)
    N = 16
    u = np.random.default_rng(3).normal(size=(N, N, N, 10))
    for site in ((0, 0, 2), (3, 5, 7), (15, 15, 15)):
        u[site][:4] = [1e200, -1e200, 5e199, 1e-3]
    with np.errstate(over="ignore"):
        obs = observables(u)
    ctx = L.Context(L.model_params(N))
    ctx.set_field(u)
    wall, phase, _ = ctx.measure()
    ctx.close()
    walls = np.concatenate([wall, phase], axis=1)
    for o, f in enumerate(obs):
        if o in (10, 11, 24):  # phi^2, sigma: infinite
            continue
        for d, axes in enumerate(((0, 1), (0, 2), (1, 2))):
            ref = f.sum(axis=axes, dtype=np.longdouble) / N ** 2
            tol = 10 * np.finfo(float).eps * np.abs(f).mean(axis=axes) + 1e-300
            assert (np.abs(walls[d, o] - ref) <= tol).all(), (d, o)
