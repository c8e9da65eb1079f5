"""Sums, running mean flow and node sampling at the edges of their kernels:
lattices of less than a workgroup and of many, rows of 2, 4 and 8 groups of
four nodes, every storage format, point counts around the pinned buffer's
capacity. The reference is numpy in 64 bits on the read-back moments; each
value is a sum of n terms, so it may be off by a few n eps of the sum of the
terms' magnitudes (a fixed tree of additions: far less)."""
import numpy as np
import pytest

import mrlbm

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8, 8), (16, 8, 24), (24, 16, 8), (40, 24, 16), (32, 8, 8), (128, 64, 40)]
EPS = 2.0 ** -52


@pytest.mark.parametrize("storage", [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16])
@pytest.mark.parametrize("shape", SHAPES)
def test_sums_equal_numpy(shape, storage):
    print("case", shape, storage, flush=True)
    with mrlbm.Lattice(shape, q=19, tau=0.55, storage=storage, seed=2) as lat:
        lat.init_taylor_green(0.05)
        lat.step(4)
        n = lat.n
        tol = 64 * EPS * np.sqrt(n)

        def close(got, terms):
            assert abs(got - terms.sum() / n) <= tol * np.abs(terms).sum() / n + 1e-300

        m = lat.moments()
        mass, ke, bad = lat.reduce_checked()
        close(mass, m[0])
        close(ke, (1.0 + m[0]) * (m[1:4] ** 2).sum(0) / 18.0)
        assert bad == 0
        for k, v in enumerate(lat.moment_means()):
            close(v, m[k])
        assert lat.velocity_residual() == -1.0
        f32 = np.float32
        u0 = (m[1:4].astype(f32) * f32(1.0 / 3.0)).astype(np.float64)
        lat.mean_flow_accumulate()
        lat.step(3)
        m1 = lat.moments()
        u1 = (m1[1:4].astype(f32) * f32(1.0 / 3.0)).astype(np.float64)
        res = np.sqrt(((u1 - u0) ** 2).sum() / (u1 ** 2).sum())
        assert lat.velocity_residual() == pytest.approx(res, rel=tol)
        lat.mean_flow_accumulate()
        (rho, *u), count = lat.mean_flow()
        assert count == 2
        flat = [f.reshape(-1, order="F") for f in (rho, *u)]
        assert np.allclose(flat[0], 1.0 + 0.5 * (m[0] + m1[0]), rtol=4 * EPS, atol=0)
        for a in range(3):
            mean = 0.5 * (m[1 + a] / 3.0 + m1[1 + a] / 3.0)
            assert np.allclose(flat[1 + a], mean, rtol=0, atol=4 * EPS * np.abs(m[1 + a]).max())
        e = (1.0 + m1[0]) * sum((m1[1 + a] / 3.0 - flat[1 + a]) ** 2 for a in range(3)) / 2.0
        assert lat.turbulent_ke() == pytest.approx(e.mean(), rel=max(tol, 1e-12))


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 711, 712, 713, 5000])
def test_sample_counts(n):
    shape = (32, 24, 16)
    with mrlbm.Lattice(shape, q=19, tau=0.56, storage=mrlbm.STORE_FP16) as lat:
        lat.init_taylor_green(0.05)
        lat.step(5)
        m = lat.moments()
        rng = np.random.default_rng(n)
        p = np.stack([rng.integers(0, s, n) for s in shape], axis=1)
        for _ in range(2):
            assert np.array_equal(lat.sample(p), m[:, p[:, 0] + 32 * (p[:, 1] + 24 * p[:, 2])].T)


@pytest.mark.parametrize("storage", [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16])
def test_non_finite_nodes_are_counted(storage):
    with mrlbm.Lattice((40, 16, 24), q=19, tau=0.6, storage=storage) as lat:
        lat.init_uniform(u=(0.01, 0.0, 0.0))
        m = lat.moments()
        for k, (row, v) in enumerate([(0, np.inf), (1, -np.inf), (2, np.inf), (3, -np.inf), (0, np.inf)]):
            m[row, 1000 * k + k] = v
        m[3, 0] = np.inf  # the node of the first one again
        m[5, 77] = np.inf  # a second moment does not count
        lat.write_moments(m)
        assert lat.reduce_checked()[2] == 5


@pytest.mark.parametrize("storage", [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16])
def test_infinite_velocities_stay_infinite_in_the_mean_flow(storage):
    with mrlbm.Lattice((40, 16, 24), q=19, tau=0.6, storage=storage) as lat:
        lat.init_uniform(u=(0.03, 0.0, 0.0))
        m = lat.moments()
        at = {(1, 0): np.inf, (2, 7): -np.inf, (3, 8191): np.inf, (1, lat.n - 1): -np.inf, (2, 500): np.nan}
        for (row, node), v in at.items():
            m[row, node] = v
        lat.write_moments(m)
        held = lat.moments()
        for key, v in at.items():
            assert np.array_equal(held[key], v, equal_nan=True)
        for _ in range(2):
            lat.mean_flow_accumulate()
        u = np.stack([f.reshape(-1, order="F") for f in lat.mean_flow()[0][1:]])
        assert np.array_equal(u, held[1:4] / 3.0, equal_nan=True)
        # against a finite mean an infinite velocity has infinite energy
        lat.mean_flow_reset()
        lat.init_uniform(u=(0.03, 0.0, 0.0))
        lat.mean_flow_accumulate()
        m = lat.moments()
        m[1, 77] = np.inf
        lat.write_moments(m)
        assert lat.turbulent_ke() == np.inf


def test_threads_read_one_lattice():
    """Sampling and sums of one lattice from several threads at a time share
    its result buffer: each call gets its own values."""
    import threading
    shape = (32, 24, 16)
    errors = []
    with mrlbm.Lattice(shape, q=19, tau=0.56) as lat:
        lat.init_taylor_green(0.05)
        lat.step(5)
        lat.mean_flow_accumulate()
        lat.step(2)
        m = lat.moments()
        sums = {"reduce_checked": lat.reduce_checked(), "moment_means": lat.moment_means(),
                "turbulent_ke": lat.turbulent_ke()}

        def sample(n):
            rng = np.random.default_rng(n)
            for _ in range(150):
                p = np.stack([rng.integers(0, s, n) for s in shape], axis=1)
                if not np.array_equal(lat.sample(p), m[:, p[:, 0] + 32 * (p[:, 1] + 24 * p[:, 2])].T):
                    errors.append(n)

        def total(name):
            for _ in range(150):
                if not np.array_equal(getattr(lat, name)(), sums[name]):
                    errors.append(name)

        def run(f, arg):
            try:
                f(arg)
            except Exception as e:  # noqa: BLE001
                errors.append(e)

        th = [threading.Thread(target=run, args=(sample, n)) for n in (1, 16, 300, 712)]
        th += [threading.Thread(target=run, args=(total, name)) for name in sums]
        for t in th:
            t.start()
        for t in th:
            t.join()
    assert not errors


@pytest.mark.parametrize("storage", [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16])
def test_sums_past_one_round_of_the_grid(storage):
    """More groups of four nodes than 1024 workgroups of 256 lanes, by a part
    of a round: the loop, its stride and the fold of 1024 records."""
    test_sums_equal_numpy((136, 104, 88), storage)
