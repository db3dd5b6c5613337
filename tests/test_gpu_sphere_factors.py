"""Factor tables of the sphere products: whole matrices shared by mirrored orbital sums, or triangles.

The product kernels keep one matrix for the orbital sums S and 2 (M - 1) - S when the off-diagonal
factors are the same under the reflection of the orbitals, and a triangle per sum otherwise or when
the whole matrices would not fit.  Products against the matrix elements that the row listing gives
from the factors as they were handed over.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def factors(lz_max, mirrored, seed):
    """symmetric random factors in the per-pair layout; mirrored: off-diagonal ones unchanged under
    m -> lz_max - m, diagonal ones not"""
    rng = np.random.default_rng(seed)
    m = lz_max + 1
    mats = {}
    for s in range(1, 2 * lz_max):
        np_ = min(s, lz_max) - s // 2
        a = rng.uniform(-1, 1, (np_, np_))
        a = a + a.T
        if mirrored and s > lz_max:
            a = mats[2 * lz_max - s].copy()
            np.fill_diagonal(a, rng.uniform(-1, 1, np_))
        mats[s] = a
    f, off = [], []
    for m1 in range(m):
        for m2 in range(m1):
            off.append(len(f))
            f.extend(mats[m1 + m2][m1 - ((m1 + m2) // 2 + 1)])
    off.append(len(f))
    return np.array(f), np.array(off, dtype=np.int32)


@pytest.mark.parametrize("n,total_lz,lz_max,mirrored", [(4, 2, 9, True), (4, 2, 9, False), (5, 1, 15, False),
                                                        (4, 0, 31, True), (3, 1, 33, False), (3, 0, 50, True),
                                                        (3, 0, 52, True), (2, 0, 59, True)])
def test_products_match_row_listing(arch, n, total_lz, lz_max, mirrored):
    from diagham_amd import capi
    g = capi.gpu()
    f, off = factors(lz_max, mirrored, 10 * lz_max + n)
    basis, ham = ctypes.c_void_p(), ctypes.c_void_p()
    arch.check(g.dh_fermion_sphere_create(arch.ctx, ctypes.byref(basis), n, total_lz, lz_max), "basis")
    arch.check(g.dh_sphere_hamiltonian_create(arch.ctx, ctypes.byref(ham), basis, capi.dptr(f),
                                              off.ctypes.data_as(capi.P_I), f.size), "hamiltonian")
    dim = g.dh_basis_dimension(basis)
    dense = np.zeros((dim, dim))
    t, c, cnt = np.zeros(100000, np.int64), np.zeros(100000), ctypes.c_int64()
    for r in range(dim):
        arch.check(g.dh_hamiltonian_row_elements(ham, r, t.ctypes.data_as(capi.P_I64), capi.dptr(c), t.size,
                                                 ctypes.byref(cnt)), "row_elements")
        np.add.at(dense[r], t[:cnt.value], c[:cnt.value])
    rng = np.random.default_rng(1)
    for k in (1, 2, 8):
        x = rng.standard_normal((dim, k))
        dx = capi.DeviceBuffer.from_host(arch, x.reshape(-1))
        dy = capi.DeviceBuffer(arch, dim * k)
        ref = dense @ x
        # every term enters both sums once: a few hundred terms of rounding each
        bound = 1e-13 * np.abs(dense) @ np.abs(x) + 1e-300
        for mode in (1, 2, 3, 4):
            for lpr in (1, 2, 8):
                arch.check(g.dh_hamiltonian_set_launch(ham, lpr, 256, mode, 1), "set_launch")
                arch.check(g.dh_hv(ham, dx.ptr, dy.ptr, k, 0, 0, -1), "dh_hv")
                y = dy.download().reshape(dim, k)
                assert np.all(np.abs(y - ref) <= bound), (k, mode, lpr)
        dx.free()
        dy.free()
    g.dh_hamiltonian_destroy(ham)
    g.dh_basis_destroy(basis)
