"""Products of sector sets in the launch shapes that the sets choose by themselves and in the forms of the row
routine that such a choice reaches, every column of a block against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from test_gpu_sectors import SectorSet, coulomb

pytestmark = pytest.mark.gpu


def sphere_set_matches(S, n, lz_max, sectors, V, k, rows=None):
    """H of a set against the oracle in every column; rows: only that many rows of each sector, spread over it"""
    fac = O.Factors(lz_max, V)
    X = np.random.default_rng(lz_max + k).standard_normal((S.total, k))
    Y = S.hv(X.reshape(-1), k).reshape(S.total, k)
    for i, lz in enumerate(sectors):
        ref = O.FermionSphere(n, lz, lz_max)
        a, b = S.off[i], S.off[i + 1]
        assert b - a == ref.dim
        x = np.ascontiguousarray(X[a:b])
        if rows is None or ref.dim <= rows:
            y = np.stack([O.fs_hv(ref, fac, np.ascontiguousarray(x[:, v])) for v in range(k)], axis=1)
            got = Y[a:b]
        else:
            at = np.unique(np.linspace(0, ref.dim - 1, rows).astype(int))
            y = np.zeros((at.size, k))
            for j, r in enumerate(at):
                t, c = O.fs_row_elements(ref, fac, int(r))
                y[j] = c @ x[t]
            got = Y[a:b][at]
        for v in range(k):
            assert np.linalg.norm(got[:, v] - y[:, v]) <= 1e-12 * max(np.linalg.norm(y[:, v]), 1e-300), (lz, k, v)


# one lane per row on 64-bit words: the low rank table in LDS (34 orbitals) and both in global memory (36)
@pytest.mark.parametrize("n,lz_max,sectors", [(4, 33, [0, 2, 12, 90]), (4, 35, [0, 2, 10, 60])])
@pytest.mark.parametrize("k,row_mode", [(1, 1), (2, 1), (2, 3), (2, 4), (4, 3), (8, 1), (8, 3)])
@pytest.mark.parametrize("block", [256, 1024])
def test_sector_rows_on_one_lane_of_64_bit_words(arch, n, lz_max, sectors, k, row_mode, block):
    V = coulomb(lz_max)
    S = SectorSet(arch, n, lz_max, sectors, V)
    assert S.capi.gpu().dh_sector_set_row_mode(S.h, row_mode) == 0
    assert S.capi.gpu().dh_sector_set_launch(S.h, 1, block) == 0
    sphere_set_matches(S, n, lz_max, sectors, V, k)
    S.close()


# rank tables in LDS (26 to 28 orbitals, restaged from sector to sector; 29 never) in chosen shapes
@pytest.mark.parametrize("n,lz_max,lpr,block", [(4, 25, 1, 256), (4, 26, 2, 1024), (4, 27, 1, 1024), (4, 27, 1, 512),
                                                (4, 28, 1, 1024)])
@pytest.mark.parametrize("k", [2, 4, 16])
def test_every_column_with_rank_tables_in_lds(arch, n, lz_max, lpr, block, k):
    sectors = list(range((n * lz_max) % 2, 60, 2))
    V = coulomb(lz_max)
    S = SectorSet(arch, n, lz_max, sectors, V)
    assert S.capi.gpu().dh_sector_set_launch(S.h, lpr, block) == 0
    sphere_set_matches(S, n, lz_max, sectors, V, k, rows=40)
    S.close()


# a space in every branch of the rule below 256 rows per CU: few rows with small and large tables, from 64 and from
# 128 rows per CU, with the low rank table in LDS and in global memory; and one whose rank tables are both in LDS
@pytest.mark.parametrize("n,total_lz,lz_max", [(6, 0, 15), (3, 0, 26), (5, 0, 36), (6, 1, 31), (5, 0, 44), (7, 0, 30),
                                               (6, 0, 40), (10, 0, 27)])
@pytest.mark.parametrize("k", [1, 4, 8, 16])
def test_small_spaces_in_their_own_shape(arch, n, total_lz, lz_max, k):
    from diagham_amd import capi
    total_lz += (n * lz_max + total_lz) % 2
    V = coulomb(lz_max)
    p = capi.Problem.sphere(arch, n, total_lz, lz_max, V)
    X = np.random.default_rng(n + k).standard_normal((p.dim, k))
    Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
    p.close()
    space, fac = O.FermionSphere(n, total_lz, lz_max), O.Factors(lz_max, V)
    at = np.unique(np.linspace(0, space.dim - 1, 500).astype(int))
    y = np.zeros((at.size, k))
    for j, r in enumerate(at):
        t, c = O.fs_row_elements(space, fac, int(r))
        y[j] = c @ X[t]
    for v in range(k):
        assert np.linalg.norm(Y[at][:, v] - y[:, v]) <= 1e-12 * np.linalg.norm(y[:, v]), v


# every branch of the rule of sphere sets by rows per CU: few (with small and large tables), below 128, 128 to 2048 with
# workgroups that fit a CU many times and three times, above 2048 with both rank tables in LDS, one and none; 26 to
# 28 orbitals restage the high table from sector to sector
@pytest.mark.parametrize("n,lz_max,step", [(5, 13, 1), (3, 25, 1), (5, 23, 1), (7, 20, 1), (7, 25, 1), (6, 31, 1),
                                           (8, 24, 1), (7, 27, 1), (6, 35, 1)])
@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
def test_sphere_sets_in_their_own_shape(arch, n, lz_max, step, k):
    from diagham_amd import capi
    sectors = capi.sphere_sectors(n, lz_max)
    V = coulomb(lz_max)
    S = SectorSet(arch, n, lz_max, sectors, V)
    fac = O.Factors(lz_max, V)
    X = np.random.default_rng(lz_max + k).standard_normal((S.total, k))
    Y = S.hv(X.reshape(-1), k).reshape(S.total, k)
    active = np.zeros(len(sectors), np.uint8)
    active[[0, len(sectors) // 2, -1]] = 1
    Z = S.hv(X.reshape(-1), k, active, Y.reshape(-1).copy()).reshape(S.total, k)
    for i in sorted({0, 1, len(sectors) // 2, len(sectors) - 1}):
        ref = O.FermionSphere(n, sectors[i], lz_max)
        a, b = int(S.off[i]), int(S.off[i + 1])
        at = np.unique(np.linspace(0, ref.dim - 1, 60).astype(int))
        y = np.zeros((at.size, k))
        for j, r in enumerate(at):
            t, c = O.fs_row_elements(ref, fac, int(r))
            y[j] = c @ X[a:b][t]
        for v in range(k):
            for got in (Y, Z):  # all sectors, and three of them (the rest keep what was there)
                assert np.linalg.norm(got[a:b][at][:, v] - y[:, v]) <= 1e-12 * np.linalg.norm(y[:, v]), (i, k, v)
    keep = np.repeat(active == 0, np.diff(S.off))
    assert np.array_equal(Y[keep], Z[keep])
    S.close()


# the same for momentum sets: factors in LDS or not, the low rank table in LDS or not (35 sites and more)
@pytest.mark.parametrize("n,nx,ny", [(4, 4, 4), (5, 5, 4), (5, 6, 4), (6, 6, 5), (5, 8, 4), (4, 6, 6), (5, 7, 5), (4, 8, 6)])
@pytest.mark.parametrize("k", [1, 2, 4, 8])
def test_momentum_sets_in_their_own_shape(arch, n, nx, ny, k):
    from test_gpu_lattice import T1, T2, TPP, MomentumSet
    sectors = [(x, y) for x in range(nx) for y in range(ny)]
    S = MomentumSet(arch, n, nx, ny, sectors)
    c = S.capi
    u, _ = O.checkerboard_lower_band(nx, ny, T1, T2, TPP)
    fac = O.LatticeFactors(nx, ny, u)
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((S.total, k)) + 1j * rng.standard_normal((S.total, k))
    Y = S.hv(X, k)
    active = np.zeros(len(sectors), np.uint8)
    active[[0, len(sectors) // 2]] = 1
    dx = c.DeviceBuffer.from_host(arch, np.ascontiguousarray(X).view(np.float64).reshape(-1))
    dz = c.DeviceBuffer(arch, 2 * S.total * k)
    arch.check(c.gpu().dh_sectors_hv(S.h, dx.ptr, dz.ptr, k, 0, bytes(active)), "hv")
    Z = dz.download().view(np.complex128).reshape(S.total, k)
    for i in (0, len(sectors) // 2):
        ref = O.MomentumFermions(n, nx, ny, *sectors[i])
        a, b = int(S.off[i]), int(S.off[i + 1])
        at = np.unique(np.linspace(0, ref.dim - 1, 40).astype(int))
        y = np.zeros((at.size, k), complex)
        for j, r in enumerate(at):
            t, coef = O.fm_row_elements(ref, fac, int(r))
            y[j] = coef.conj() @ X[a:b][t]  # listed by source state: H[t, r]
        for v in range(k):
            for got in (Y, Z):
                assert np.linalg.norm(got[a:b][at][:, v] - y[:, v]) <= 1e-12 * np.linalg.norm(y[:, v]), (i, k, v)
    S.close()


# the most orbitals: rank tables of 2^31 words each (built on the host in about 40 s, 8 GiB each), where a byte
# offset into them does not fit 32 bits
def test_products_on_62_orbitals(arch):
    from diagham_amd import capi
    n, total_lz, lz_max = 3, 1, 61
    V = coulomb(lz_max)
    p = capi.Problem.sphere(arch, n, total_lz, lz_max, V)
    space, fac = O.FermionSphere(n, total_lz, lz_max), O.Factors(lz_max, V)
    assert p.dim == space.dim
    for k in (1, 2, 4, 8):
        X = np.random.default_rng(lz_max + k).standard_normal((p.dim, k))
        Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
        for v in range(k):
            y = O.fs_hv(space, fac, np.ascontiguousarray(X[:, v]))
            assert np.linalg.norm(Y[:, v] - y) <= 1e-12 * np.linalg.norm(y), (k, v)
    p.close()
