"""Whole fields across the C ABI: read-back, rewritten moments and initial
states go through device kernels that gather, scatter, decode and encode the
block layout. Each is compared, bit for bit, with node sampling or with the
storage conversion written out in numpy, at lattices of one tile, of extents
that are not powers of two, of one transfer slot and of several per worker."""
import math

import numpy as np
import pytest

import mrlbm

pytestmark = pytest.mark.gpu

SHAPES = [((8, 8, 8), {}), ((16, 8, 24), {}), ((40, 24, 56), {}), ((72, 64, 80), {}),
          ((32, 16, 64), dict(kernel=mrlbm.KERNEL_COLUMN))]
STORES = [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16]


def stored(m, storage):
    """The value the storage format holds for each moment (10, N)."""
    if storage == mrlbm.STORE_FP32:
        return m.astype(np.float32).astype(np.float64)
    if storage == mrlbm.STORE_FP16:
        s = np.full((10, 1), 4096.0)
        s[1:4] = 1024.0
        return (m * s).astype(np.float32).astype(np.float16).astype(np.float64) / s
    u = m.astype(np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)).astype(np.uint32) & np.uint32(0xFFFF0000)
    return u.view(np.float32).astype(np.float64)


def moments_of(rho, ux, uy, uz, q, mode, rho0=1.0):
    if mode == mrlbm.INIT_EQUILIBRIUM:
        p = [ux * ux, ux * uy, ux * uz, uy * uy, uy * uz, uz * uz]
    else:
        cx = [0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0]
        cy = [0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 1, -1]
        cz = [0, 0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 0, 0, -1, 1, -1, 1]
        w = (1 / 3, 1 / 18, 1 / 36) if q == 19 else (8 / 27, 2 / 27, 1 / 54)
        uu = ux * ux + uy * uy + uz * uz
        f = []
        for i in range(19):
            uc3 = 3.0 * (ux * cx[i] + uy * cy[i] + uz * cz[i])
            f.append((w[0 if i == 0 else 1 if i < 7 else 2] * rho0) * ((1.0 - 1.5 * uu) + uc3 * (1.0 + uc3 * 0.5)))
        ir, c = 1.0 / rho, 1.0 / 3.0

        def add(*ids):
            t = f[ids[0]]
            for i in ids[1:]:
                t = t + f[i]
            return t
        p = [add(1, 2, 7, 8, 9, 10, 13, 14, 15, 16) * ir - c, ((f[7] + f[8]) - (f[13] + f[14])) * ir,
             ((f[9] + f[10]) - (f[15] + f[16])) * ir, add(3, 4, 7, 8, 11, 12, 13, 14, 17, 18) * ir - c,
             ((f[11] + f[12]) - (f[17] + f[18])) * ir, add(5, 6, 9, 10, 11, 12, 15, 16, 17, 18) * ir - c]
    k = (4.5, 9.0, 9.0, 4.5, 9.0, 4.5)
    return np.stack([rho - rho0, 3.0 * ux, 3.0 * uy, 3.0 * uz] + [a * b for a, b in zip(k, p)])


def lattice(shape, kw, storage=mrlbm.STORE_FP32, q=19):
    if "kernel" in kw and storage != mrlbm.STORE_FP32:
        pytest.skip("the column kernel is built for FP32")
    return mrlbm.Lattice(shape, q=q, tau=0.57, storage=storage, seed=3, **kw)


@pytest.mark.parametrize("storage", STORES)
@pytest.mark.parametrize("shape,kw", SHAPES)
def test_read_back_equals_sampling(shape, kw, storage):
    print("case", shape, storage, flush=True)
    with lattice(shape, kw, storage) as lat:
        lat.init_taylor_green(0.05)
        lat.step(3)
        m = lat.moments()
        pts = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1)
        pts = pts.transpose(2, 1, 0, 3).reshape(-1, 3)  # x fastest
        assert np.array_equal(lat.sample(pts), m.T)


@pytest.mark.parametrize("storage", STORES)
@pytest.mark.parametrize("shape,kw", SHAPES)
def test_written_moments_and_fields(shape, kw, storage):
    print("case", shape, storage, flush=True)
    rng = np.random.default_rng(7)
    n = int(np.prod(shape))
    with lattice(shape, kw, storage) as lat:
        m = rng.normal(size=(10, n)) * 10.0 ** rng.uniform(-9, 0, (10, n))
        lat.write_moments(m)
        assert np.array_equal(lat.moments(), stored(m, storage))
        rho = 1.0 + 0.02 * rng.normal(size=n)
        u = 0.05 * rng.normal(size=(3, n))
        for mode in (mrlbm.INIT_EQUILIBRIUM, mrlbm.INIT_REFERENCE):
            lat.init_fields(rho, *u, mode)
            assert np.array_equal(lat.moments(), stored(moments_of(rho, *u, 19, mode), storage))


def test_reference_fields_d3q27():
    rng = np.random.default_rng(8)
    shape = (24, 16, 8)
    n = int(np.prod(shape))
    rho, u = 1.0 + 0.02 * rng.normal(size=n), 0.05 * rng.normal(size=(3, n))
    with lattice(shape, {}, q=27) as lat:
        lat.init_fields(rho, *u, mrlbm.INIT_REFERENCE)
        assert np.array_equal(lat.moments(),
                              stored(moments_of(rho, *u, 27, mrlbm.INIT_REFERENCE), mrlbm.STORE_FP32))


@pytest.mark.parametrize("storage", STORES)
def test_taylor_green_equals_its_formula(storage):
    shape, u0 = (16, 24, 40), 0.05
    k = [2.0 * math.pi / s for s in shape]
    f = np.zeros((4, int(np.prod(shape))))
    j = 0
    for z in range(shape[2]):
        for y in range(shape[1]):
            for x in range(shape[0]):
                f[0, j] = 1.0 + (3.0 / 16.0) * 1.0 * u0 * u0 * (math.cos(2 * k[0] * x) + math.cos(2 * k[1] * y)) * (
                    math.cos(2 * k[2] * z) + 2.0)
                f[1, j] = u0 * math.sin(k[0] * x) * math.cos(k[1] * y) * math.cos(k[2] * z)
                f[2, j] = -u0 * math.cos(k[0] * x) * math.sin(k[1] * y) * math.cos(k[2] * z)
                j += 1
    with lattice(shape, {}, storage) as a, lattice(shape, {}, storage) as b:
        a.init_taylor_green(u0)
        b.init_fields(*f)
        assert np.array_equal(a.moments(), b.moments())
        a.step(2)
        b.step(2)
        assert np.array_equal(a.moments(), b.moments())


def test_bad_density_changes_nothing():
    shape = (40, 64, 80)  # several check ranges
    n = int(np.prod(shape))
    with lattice(shape, {}) as lat:
        lat.init_taylor_green(0.05)
        before = lat.moments()
        for at in ((n - 1,), (n // 2, n - 3), (5,)):
            for v in (0.0, float("nan")):
                rho = np.ones(n)
                rho[list(at)] = v
                x, y, z = at[0] % 40, at[0] // 40 % 64, at[0] // (40 * 64)
                with pytest.raises(mrlbm.MrlbmError, match=rf"\({x},{y},{z}\)"):
                    lat.init_fields(rho, *np.zeros((3, n)))
        with pytest.raises(mrlbm.MrlbmError, match=r"\(0,0,"):
            lat.init_taylor_green(float("nan"))
        with pytest.raises(mrlbm.MrlbmError, match="non-positive density"):
            lat.init_taylor_green(4.0)
        assert np.array_equal(lat.moments(), before)


@pytest.mark.parametrize("storage", STORES)
@pytest.mark.parametrize("shape,kw", SHAPES)
def test_macroscopic_equals_moments(shape, kw, storage):
    print("case", shape, storage, flush=True)
    with lattice(shape, kw, storage) as lat:
        lat.init_taylor_green(0.05)
        lat.step(3)
        m = lat.moments()
        for rho0 in (1.0, 0.7):
            got = lat.macroscopic(rho0)
            want = [m[0] + rho0, m[1] / 3, m[2] / 3, m[3] / 3]
            for g, w in zip(got, want):
                assert g.shape == shape and np.array_equal(g.reshape(-1, order="F"), w)


def test_transfers_of_several_threads():
    """Threads move different lattices at the same time through the process's
    pinned slots; lattices come and go meanwhile."""
    import threading
    shapes = [(72, 64, 80), (40, 24, 56), (64, 64, 64), (16, 8, 24)]
    errors = []

    def work(i):
        try:
            rng = np.random.default_rng(i)
            for r in range(4):
                shape = shapes[(i + r) % len(shapes)]
                n = int(np.prod(shape))
                with mrlbm.Lattice(shape, q=19, tau=0.6) as lat:
                    m = rng.normal(size=(10, n)).astype(np.float32).astype(np.float64)
                    lat.write_moments(m)
                    if not np.array_equal(lat.moments(), m):
                        errors.append((i, r, shape))
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors


def test_macroscopic_adds_any_density():
    """rho0 as numpy takes it in a sum: arrays, lists and scalar types; what a
    sum refuses is refused."""
    shape = (24, 16, 8)
    n = int(np.prod(shape))
    with lattice(shape, {}) as lat:
        lat.init_taylor_green(0.05)
        lat.step(3)
        m = lat.moments()
        rng = np.random.default_rng(1)
        for rho0 in (rng.uniform(0.9, 1.1, n), rng.uniform(0.9, 1.1, n).astype(np.float32), np.array([0.8]), [0.5],
                     np.arange(n), np.float32(0.7), np.array(0.3), 1, True, -0.0, np.float64(1.0), 1.0 + 2.0j):
            rho, *u = lat.macroscopic(rho0)
            want = m[0] + rho0
            assert rho.shape == shape and rho.dtype == want.dtype
            assert np.array_equal(rho.reshape(-1, order="F"), want)
            for a in range(3):
                assert np.array_equal(u[a].reshape(-1, order="F"), m[1 + a] / 3)
        for rho0 in (None, "1.0", np.ones(n - 1)):
            with pytest.raises((TypeError, ValueError)):
                m[0] + rho0
            with pytest.raises((TypeError, ValueError)):
                lat.macroscopic(rho0)


def test_macroscopic_fields_own_their_memory():
    """A field that is kept does not keep the others; the C entry with one
    buffer gives the same values."""
    with lattice((40, 24, 56), {}) as lat:
        lat.init_taylor_green(0.05)
        lat.step(3)
        got = lat.macroscopic(0.9)
        for f in got:
            assert f.base is not None and f.base.nbytes == 8 * lat.n
        one = np.empty((4, lat.n))
        mrlbm._lib.check(mrlbm._lib.load().mrlbm_read_macroscopic(lat._h, 0.9, one.ctypes.data_as(mrlbm._lib._dp)))
        for f, w in zip(got, one):
            assert np.array_equal(f.reshape(-1, order="F"), w)


def test_lowest_bad_density_of_many_ranges():
    """Densities are checked in ranges of 2^17 nodes by as many threads as
    have a processor; the node that is reported is the lowest bad one."""
    shape = (160, 128, 104)  # 17 ranges
    n = int(np.prod(shape))
    per = 1 << 17
    rng = np.random.default_rng(5)
    rho, u = np.ones(n), np.zeros((3, n))
    with lattice(shape, {}) as lat:
        lat.init_uniform()
        cases = [[n - 1], [per - 1, per], [per, 9 * per + 3], [16 * per, 15 * per + 7, 14 * per + 99],
                 [3 * per + 100, 4 * per, 5 * per, 3 * per + 99]]
        cases += [list(rng.integers(0, n, 5)) for _ in range(12)]
        for at in cases:
            rho[at] = rng.choice([0.0, -1.0, np.nan], len(at))
            x, y, z = min(at) % 160, min(at) // 160 % 128, min(at) // (160 * 128)
            with pytest.raises(mrlbm.MrlbmError, match=rf"\({x},{y},{z}\)"):
                lat.init_fields(rho, *u)
            rho[at] = 1.0
        lat.init_fields(rho, *u)
        assert lat.reduce_checked() == (0.0, 0.0, 0)


@pytest.mark.parametrize("storage", STORES)
def test_many_chunks_both_ways(storage):
    """Transfers of up to 130 chunks with helpers joining in between."""
    shape = (128, 104, 128)
    n = int(np.prod(shape))
    with lattice(shape, {}, storage) as lat:
        m = stored(np.random.default_rng(7).normal(size=(10, n)) * 0.01, storage)
        for _ in range(3):
            lat.write_moments(m)
            assert np.array_equal(lat.moments(), m)
        rho, *u = lat.macroscopic()
        assert np.array_equal(rho.reshape(-1, order="F"), m[0] + 1.0)
        for a in range(3):
            assert np.array_equal(u[a].reshape(-1, order="F"), m[1 + a] / 3)
