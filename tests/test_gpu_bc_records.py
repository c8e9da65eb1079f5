"""Boundary solve with class records broadcast in a wave (one or two classes)
or read per lane (more): tile shapes put different nodes into a wave, so the
same lattice takes different paths with each of them and has to give the same
bits; the first case also against the FP64 oracle."""
import numpy as np
import pytest

import mrlbm
from mrlbm import geometry

pytestmark = pytest.mark.gpu

TILES = [(8, 8, 8), (16, 8, 4), (32, 4, 4), (64, 4, 2), (16, 8, 8)]


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("storage", [mrlbm.STORE_FP32, mrlbm.STORE_FP16, mrlbm.STORE_BF16])
@pytest.mark.parametrize("walls,spheres", [
    ((1, 1, 1), []),                                          # faces, edges, corners, a moving lid
    ((0, 1, 1), [((20, 8, 8), 3.2), ((41, 30, 17), 5.0)]),    # many patterns in one wave
    ((1, 0, 0), [((63, 12, 2), 0.4)]),                        # one solid voxel beside a wall
])
def test_same_bits_for_every_wave_composition(q, storage, walls, spheres):
    shape = (64, 32, 24)
    print("case", q, storage, walls, len(spheres), flush=True)
    solid = geometry.spheres(shape, [c for c, _ in spheres], [r for _, r in spheres]) if spheres else None
    moving = [(2, +1, 1)] if walls[2] and not spheres else []
    types = geometry.classify(shape, walls, solid, moving)
    ref = None
    for tile in TILES:
        with mrlbm.Lattice(shape, q=q, tau=0.58, walls=walls, force=(2e-5, 0, 0), tile=tile, storage=storage,
                           seed=9) as lat:
            lat.set_bc_velocity(1, (0.05, 0.01, 0.0))
            lat.set_node_types(types)
            lat.init_uniform(u=(0.02, 0.0, 0.0))
            lat.step(25)
            m = lat.moments()
        assert np.isfinite(m).all()
        if ref is None:
            ref = m
        assert np.array_equal(m, ref), tile


@pytest.mark.parametrize("n", [1, 2, 3])
def test_batch_of_walls_and_periodic_members(n):
    """One launch over members with and without a class map, D3Q27 included."""
    print("case", n, flush=True)
    specs = [((16, 16, 16), (1, 1, 1)), ((24, 8, 16), (0, 0, 0)), ((8, 8, 8), (0, 1, 1))][:n]
    for q in (19, 27):
        def make(shape, walls):
            lat = mrlbm.Lattice(shape, q=q, tau=0.6, walls=walls, force=(1e-5, 0, 0), tile=(8, 8, 8))
            if any(walls):
                lat.set_geometry()
            lat.init_uniform(u=(0.01, 0.0, 0.0))
            return lat
        lats = [make(*s) for s in specs]
        with mrlbm.Batch(q=q, tile=(8, 8, 8)) as b:
            for lat in lats:
                b.add(lat)
            b.step(20, graph_steps=5)
            got = [lat.moments() for lat in lats]
        for s, g, lat in zip(specs, got, lats):
            lat.close()
            with make(*s) as alone:
                alone.step(20)
                assert np.array_equal(alone.moments(), g)


@pytest.mark.parametrize("q", [19, 27])
def test_first_case_against_the_oracle(q):
    """Walls on all axes and a moving lid, FP32 moments against the FP64
    oracle, to the bar of the parity tests."""
    import _oracle
    from fields import rel_l2

    shape = (64, 32, 24)
    types = geometry.classify(shape, (1, 1, 1), None, [(2, +1, 1)])
    with mrlbm.Lattice(shape, q=q, tau=0.58, walls=(1, 1, 1), force=(2e-5, 0, 0), tile=(8, 8, 8)) as lat:
        lat.set_bc_velocity(1, (0.05, 0.01, 0.0))
        lat.set_node_types(types)
        lat.init_uniform(u=(0.02, 0.0, 0.0))
        lat.step(25)
        m = lat.moments()
    o = _oracle.Oracle(*shape, q=q, tau=0.58, walls=(1, 1, 1), force=(2e-5, 0, 0))
    o.set_bc_velocity(1, (0.05, 0.01, 0.0))
    o.set_node_types(types)
    o.init_uniform(u=(0.02, 0.0, 0.0))
    o.step(25)
    assert o.count_nan() == 0
    e = rel_l2(m, o.moments())
    print("case", q, e, flush=True)
    assert max(e.values()) <= 1e-5
