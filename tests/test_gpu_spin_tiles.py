"""The tiled spin chain product on long chains against the binary-search product, and ranges of few tiles, whose
tiles are shared by several workgroups, against the whole product to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(arch, L, sz, periodic, uniform):
    from diagham_amd import capi
    rng = np.random.default_rng(L)
    J = np.full(L, 0.7) if uniform else rng.uniform(0.5, 1.5, L)
    Jz = np.full(L, 1.3) if uniform else rng.uniform(0.5, 1.5, L)
    return capi.Problem.spin_chain(arch, L, sz, J, Jz, periodic)


# tiles of 14 sites (more than 26 sites), and the forms for two vectors with different couplings
@pytest.mark.parametrize("L,sz,periodic,uniform,k", [(28, 0, True, True, 1), (27, 1, False, False, 1),
                                                     (22, 0, True, False, 2), (22, 0, False, False, 2)])
def test_tiles_match_the_binary_search(arch, L, sz, periodic, uniform, k):
    from diagham_amd import capi
    p = chain(arch, L, sz, periodic, uniform)
    X = np.random.default_rng(k).standard_normal(p.dim * k)
    Y = p.hv(X, k)
    p.set_launch(1, 256, capi.INDEX_BSEARCH, 1)
    ref = p.hv(X, k)
    p.close()
    # at most 28 bonds a row
    assert np.max(np.abs(Y - ref)) <= 64 * 2.0 ** -53 * 28 * 1.5 * np.max(np.abs(X))


@pytest.mark.parametrize("L,sz,k,uniform", [(26, 0, 1, True), (26, 0, 1, False), (22, 0, 1, True), (22, 0, 2, True),
                                            (22, 0, 4, False), (22, 2, 8, True), (20, 0, 16, False)])
def test_ranges_of_few_tiles(arch, L, sz, k, uniform):
    from diagham_amd import capi
    p = chain(arch, L, sz, True, uniform)
    X = np.random.default_rng(L + k).standard_normal(p.dim * k)
    Y = p.hv(X, k).reshape(p.dim, k)
    dx = capi.DeviceBuffer.from_host(arch, X)
    base = np.random.default_rng(1).standard_normal(p.dim * k)
    # one row, odd ends inside a tile, part of a tile, several tiles
    for first, count in [(0, 1), (p.dim // 3, 777), (p.dim // 2 - 5, 1025), (p.dim // 5, 10001), (p.dim - 3000, 3000)]:
        dy = capi.DeviceBuffer.from_host(arch, base)
        p.hv_device(dx.ptr, dy.ptr, k, add=True, first=first, count=count)
        out = dy.download().reshape(p.dim, k)
        expect = base.reshape(p.dim, k).copy()
        expect[first:first + count] += Y[first:first + count]
        assert np.array_equal(out, expect), (first, count)
    p.close()
