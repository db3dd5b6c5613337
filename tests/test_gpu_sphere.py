"""GPU parity of the fermions-on-the-sphere path against the oracle (oracle/liboracle.so)
and the reference outputs in tests/golden.  Every call goes through the C ABI."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

SECTORS = [(4, 2, 8), (8, 0, 21), (8, 6, 21), (6, 4, 15), (10, 0, 27)]


def coulomb(lz_max):
    return O.round14(O.coulomb_pseudopotentials(lz_max))


@pytest.fixture(scope="module")
def n8_2s21(arch):
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, 8, 0, 21, coulomb(21))
    yield p
    p.close()


@pytest.mark.parametrize("n,total_lz,lz_max", SECTORS)
def test_basis_bit_exact(arch, n, total_lz, lz_max):
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, n, total_lz, lz_max, coulomb(lz_max))
    ref = O.FermionSphere(n, total_lz, lz_max)
    assert p.dim == ref.dim
    assert np.array_equal(p.states(), ref.states())
    p.close()


def test_doc_fixture_basis(arch, golden):
    from diagham_amd import capi
    g = golden["fermion_sphere_doc_basis_n4_2s8_lz1"]
    p = capi.Problem.sphere(arch, g["nbr_fermions"], g["total_lz"], g["lz_max"], coulomb(g["lz_max"]))
    expect = [sum(1 << i for i, o in enumerate(row) if o) for row in g["occupations"]]
    assert [int(s) for s in p.states()] == expect
    p.close()


@pytest.mark.parametrize("mode", [0, 1])
def test_find_state_index(n8_2s21, mode):
    states = n8_2s21.states()
    idx = n8_2s21.find_state_index(states, mode)
    assert np.array_equal(idx, np.arange(n8_2s21.dim))
    # states outside the sector (wrong particle number / wrong Lz / beyond lzMax) give dim
    s0 = int(states[0])
    bad = np.array([s0 | (1 << 30), s0 & (s0 - 1), 0], dtype=np.uint64)
    assert np.all(n8_2s21.find_state_index(bad, mode) == n8_2s21.dim)


def test_element_targets_bit_exact(n8_2s21):
    ref_space = O.FermionSphere(8, 0, 21)
    fac = O.Factors(21, coulomb(21))
    rows = list(range(0, n8_2s21.dim, 97)) + [n8_2s21.dim - 1]
    for r in rows:
        t_gpu, c_gpu = n8_2s21.row_elements(r)
        t_ref, c_ref = O.fs_row_elements(ref_space, fac, r)
        o_gpu = np.lexsort((c_gpu, t_gpu))
        o_ref = np.lexsort((c_ref, t_ref))
        assert np.array_equal(t_gpu[o_gpu], t_ref[o_ref]), r
        np.testing.assert_allclose(c_gpu[o_gpu], c_ref[o_ref], rtol=0, atol=1e-13)


def test_element_count(n8_2s21, golden):
    assert n8_2s21.count_elements() == golden["fermions_sphere_n8_2s21_lz0"]["full_matrix_elements"]


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("mode,lpr", [(1, 1), (1, 2), (1, 4), (0, 1), (0, 2), (2, 1), (2, 8), (3, 1), (3, 2), (3, 8),
                                      (4, 1), (4, 2)])
def test_hv_parity(n8_2s21, k, mode, lpr):
    """H.X (k vectors, [row][k] layout) vs the oracle, 1e-12 relative norm per vector."""
    ref_space = O.FermionSphere(8, 0, 21)
    fac = O.Factors(21, coulomb(21))
    X = np.stack([O.splitmix(100 + v, n8_2s21.dim) for v in range(k)], axis=1)
    n8_2s21.set_launch(lanes_per_row=lpr, block_size=256, index_mode=mode)
    Y = n8_2s21.hv(X.reshape(-1), k).reshape(n8_2s21.dim, k)
    for v in range(k):
        y_ref = O.fs_hv(ref_space, fac, X[:, v])
        err = np.linalg.norm(Y[:, v] - y_ref) / np.linalg.norm(y_ref)
        assert err < 1e-12, (k, mode, lpr, v, err)
    n8_2s21.set_launch(lanes_per_row=4, block_size=256, index_mode=1)


@pytest.mark.parametrize("k", [1, 2, 4])
@pytest.mark.parametrize("mode,lpr", [(1, 1), (1, 2), (2, 2), (0, 1), (3, 1), (3, 4), (4, 1)])
def test_hv_parity_beyond_32_orbitals(arch, k, mode, lpr):
    """36 orbitals: the rank kernels keep 64-bit state words for every k (the 32-bit form is for
    at most 32 orbitals)."""
    from diagham_amd import capi
    n, lz, lz_max = 4, 2, 35
    p = capi.Problem.sphere(arch, n, lz, lz_max, coulomb(lz_max))
    ref_space = O.FermionSphere(n, lz, lz_max)
    assert p.dim == ref_space.dim
    fac = O.Factors(lz_max, coulomb(lz_max))
    X = np.stack([O.splitmix(500 + v, p.dim) for v in range(k)], axis=1)
    p.set_launch(lanes_per_row=lpr, block_size=256, index_mode=mode)
    Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
    for v in range(k):
        y_ref = O.fs_hv(ref_space, fac, X[:, v])
        err = np.linalg.norm(Y[:, v] - y_ref) / np.linalg.norm(y_ref)
        assert err < 1e-12, (k, mode, lpr, v, err)
    p.close()


def test_hv_shift_add_and_range(n8_2s21, arch):
    from diagham_amd import capi
    ref_space = O.FermionSphere(8, 0, 21)
    fac = O.Factors(21, coulomb(21))
    x = O.splitmix(7, n8_2s21.dim)
    y0 = O.splitmix(8, n8_2s21.dim)
    shift = -0.5 * 64 / (0.5 * 21)  # FQHESphereFermionsTwoBodyGeneric.cc:320
    n8_2s21.set_shift(shift)
    dx = capi.DeviceBuffer.from_host(arch, x)
    dy = capi.DeviceBuffer.from_host(arch, y0)
    n8_2s21.hv_device(dx.ptr, dy.ptr, 1, add=True)
    got = dy.download()
    ref = y0 + O.fs_hv(ref_space, fac, x, shift=shift)
    assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < 1e-12
    # a row range writes only those rows
    dy.upload(y0)
    n8_2s21.hv_device(dx.ptr, dy.ptr, 1, add=False, first=100, count=1000)
    got = dy.download()
    full = O.fs_hv(ref_space, fac, x, shift=shift)
    assert np.array_equal(got[:100], y0[:100]) and np.array_equal(got[1100:], y0[1100:])
    assert np.linalg.norm(got[100:1100] - full[100:1100]) / np.linalg.norm(full[100:1100]) < 1e-12
    n8_2s21.set_shift(0.0)


def test_asymmetric_factors_are_refused(arch):
    """The kernels read one triangle of each pair-sum factor matrix: a table that is not symmetric
    must be refused, not silently symmetrised."""
    import ctypes
    from diagham_amd import capi
    lz = 9
    f, po = capi.sphere_factors(lz, coulomb(lz))
    basis = ctypes.c_void_p()
    arch.check(capi.gpu().dh_fermion_sphere_create(arch.ctx, ctypes.byref(basis), 4, 0, lz), "basis")
    ham = ctypes.c_void_p()
    rc = capi.gpu().dh_sphere_hamiltonian_create(arch.ctx, ctypes.byref(ham), basis, capi.dptr(f),
                                                 po.ctypes.data_as(capi.P_I), f.size)
    assert rc == 0
    capi.gpu().dh_hamiltonian_destroy(ham)
    bad = f.copy()
    # factor of pair (m1, m2) = (5, 2) towards the created pair m3 = 6 (sum 7): only one side changes
    bad[po[5 * 4 // 2 + 2] + (6 - 4)] += 0.1
    rc = capi.gpu().dh_sphere_hamiltonian_create(arch.ctx, ctypes.byref(ham), basis, capi.dptr(bad),
                                                 po.ctypes.data_as(capi.P_I), f.size)
    assert rc == capi.DH_E_ARG
    assert b"symmetric" in capi.gpu().dh_last_error(arch.ctx)
    capi.gpu().dh_basis_destroy(basis)


def test_autotune_keeps_parity(n8_2s21):
    """The autotuner sweeps the launch shapes of each block size, reports a consistent table and
    leaves a launch configured whose products still match the oracle."""
    rows, best = n8_2s21.autotune(ks=(1, 4, 8), repeats=2)
    assert [int(r["k"]) for r in rows] == [1, 4, 8]
    assert best in (1, 4, 8)
    for r in rows:
        assert r["lanes_per_row"] in (1, 2, 4, 8) and r["block_size"] in (128, 256, 512, 1024)
        assert r["index_mode"] in (0, 1, 2, 3, 4) and r["ms"] > 0
        assert r["elements_per_s"] > 0
    rates = {int(r["k"]): r["elements_per_s"] for r in rows}
    assert rates[best] == max(rates.values())
    ref_space = O.FermionSphere(8, 0, 21)
    fac = O.Factors(21, coulomb(21))
    X = np.stack([O.splitmix(300 + v, n8_2s21.dim) for v in range(best)], axis=1)
    Y = n8_2s21.hv(X.reshape(-1), best).reshape(n8_2s21.dim, best)
    for v in range(best):
        y_ref = O.fs_hv(ref_space, fac, X[:, v])
        assert np.linalg.norm(Y[:, v] - y_ref) <= 1e-12 * np.linalg.norm(y_ref)
    n8_2s21.set_launch(lanes_per_row=4, block_size=256, index_mode=1)


def test_stored_elements_match_on_the_fly(arch, golden):
    """EnableFastMultiplication form: the CSR of every element gives the same products (k = 1, 4,
    8, with shift and row ranges) and the same Lanczos eigenvalues; too small a budget is refused
    and leaves the on-the-fly product in place."""
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, 8, 0, 21, coulomb(21))
    ref_space = O.FermionSphere(8, 0, 21)
    fac = O.Factors(21, coulomb(21))
    nnz = p.count_elements()
    with pytest.raises(capi.DHError):
        p.precompute(max_bytes=1000)
    used = p.precompute()
    assert used == 8 * (p.dim + 1) + 12 * nnz
    for k in (1, 4, 8):
        X = np.stack([O.splitmix(500 + v, p.dim) for v in range(k)], axis=1)
        Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
        for v in range(k):
            y_ref = O.fs_hv(ref_space, fac, X[:, v])
            assert np.linalg.norm(Y[:, v] - y_ref) <= 1e-12 * np.linalg.norm(y_ref)
    p.set_shift(-1.5)
    x = O.splitmix(9, p.dim)
    assert np.linalg.norm(p.hv(x) - O.fs_hv(ref_space, fac, x, shift=-1.5)) <= 1e-12 * np.linalg.norm(x) * 100
    p.set_shift(0.0)
    r = p.lanczos(10, block_size=4)
    np.testing.assert_allclose(r["eigenvalues"], golden["fermions_sphere_n8_2s21_lz0"]["eigenvalues"], rtol=0,
                               atol=1e-10)
    p.release_precomputed()
    assert np.linalg.norm(p.hv(x) - O.fs_hv(ref_space, fac, x)) <= 1e-12 * np.linalg.norm(O.fs_hv(ref_space, fac, x))
    p.close()


def test_hermitian_reference_form_agrees(n8_2s21):
    """The reference's Hermitian-halved scatter (HermitianLowLevelAddMultiply) and the gather agree."""
    ref_space = O.FermionSphere(8, 0, 21)
    fac_h = O.Factors(21, coulomb(21), hermitian=True)
    x = O.splitmix(11, n8_2s21.dim)
    y_ref = O.fs_hv(ref_space, fac_h, x, hermitian=True)
    y = n8_2s21.hv(x)
    assert np.linalg.norm(y - y_ref) / np.linalg.norm(y_ref) < 1e-12


@pytest.mark.parametrize("block", [1, 4, 8])
def test_lanczos_reference_eigenvalues(n8_2s21, golden, block):
    ref = np.array(golden["fermions_sphere_n8_2s21_lz0"]["eigenvalues"])
    r = n8_2s21.lanczos(10, block_size=block)
    assert r["converged"]
    np.testing.assert_allclose(r["eigenvalues"], ref, rtol=0, atol=1e-10)


def test_lanczos_n10_2s27(arch, golden):
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, 10, 0, 27, coulomb(27))
    ref = np.array(golden["fermions_sphere_n10_2s27_lz0"]["eigenvalues"])
    assert p.dim == golden["fermions_sphere_n10_2s27_lz0"]["dimension"]
    r = p.lanczos(2, block_size=1)
    np.testing.assert_allclose(r["eigenvalues"], ref, rtol=0, atol=1e-10)
    p.close()


def test_l2_operator_on_gpu_labels_coulomb_states(arch):
    """L^2 through the product kernel: its expectation values on the Coulomb eigenvectors of
    N=6, 2S=15, Lz=0 are L(L+1) (the interaction conserves L), and with --l2-factor the
    L = 0 states stay put while the others move by factor * L(L+1)."""
    from diagham_amd import capi
    import torch
    n, tlz, lz = 6, 0, 15
    V = coulomb(lz)
    p = capi.Problem.sphere(arch, n, tlz, lz, V)
    vecs = torch.empty((6, p.dim), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    r = p.lanczos(6, block_size=1, d_vectors=vecs.data_ptr(), nbr_vectors=6)
    L2 = capi.Problem.sphere_l2(arch, n, tlz, lz, 1.0)
    Lvals = []
    for i in range(6):
        y = torch.empty_like(vecs[i])
        torch.cuda.synchronize()
        L2.hv_device(vecs[i].data_ptr(), y.data_ptr(), 1)
        arch.sync()
        l2 = torch.dot(vecs[i], y).item()
        L = (-1 + np.sqrt(1 + 4 * l2)) / 2
        assert abs(L - round(L)) < 1e-8, (i, l2)
        Lvals.append(int(round(L)))
    assert Lvals[0] == 0  # the Laughlin state at 2S = 3(N-1) is a singlet
    shifted = capi.Problem.sphere_l2(arch, n, tlz, lz, 0.5, pseudo=V)
    r2 = shifted.lanczos(6, block_size=1)
    # H + 0.5 L^2 keeps the L = 0 ground state and only raises the others
    assert abs(r2["eigenvalues"][0] - r["eigenvalues"][0]) < 1e-9
    for e, L in zip(r["eigenvalues"], Lvals):
        if L > 0:  # moved up by 0.5 L (L + 1): no longer in the spectrum at e
            assert np.min(np.abs(np.asarray(r2["eigenvalues"]) - e)) > 1e-6, (e, L)
    p.close()
    L2.close()
    shifted.close()


@pytest.mark.parametrize("block", [1, 4])
def test_laughlin_zero_mode_converges(arch, block):
    """V1 alone at 2S = 3(N - 1) has the Laughlin state at exactly zero energy.  Its Ritz value
    moves by rounding noise only, so the run stops by the near-zero rule of the strong convergence
    test (FullReorthogonalizedLanczosAlgorithm.cc:335-338), long before max_iter, here in a sector
    (8,512 states) larger than max_iter."""
    from diagham_amd import capi
    V = np.zeros(22)
    V[1] = 1.0
    p = capi.Problem.sphere(arch, 8, 0, 21, V)
    max_iter = 300
    r = p.lanczos(4, block_size=block, max_iter=max_iter)
    assert r["converged"] and r["products"] < max_iter, r
    ref_space, fac = O.FermionSphere(8, 0, 21), O.Factors(21, V)
    ev_ref, _ = O.fs_lanczos(ref_space, fac, 4, max_iter=max_iter, threads=8)
    assert abs(r["eigenvalues"][0]) < 1e-12
    np.testing.assert_allclose(r["eigenvalues"], ev_ref, rtol=0, atol=1e-10)
    p.close()


@pytest.mark.parametrize("nbr", [1, 3, 8, 13, 19])
@pytest.mark.parametrize("via_host", [False, True])
def test_hv_over_separate_vectors(arch, n8_2s21, nbr, via_host):
    """LowLevelMultipleAddMultiply over an array of separate vectors (dh_hv_vectors, and the host
    layer's MultipleVectorHamiltonianMultiplyOperation): every vector matches the oracle, a group of
    eight is bitwise the interleaved eight-vector product, and add / row ranges keep their meaning."""
    from diagham_amd import capi
    p = n8_2s21
    ref_space, fac = O.FermionSphere(8, 0, 21), O.Factors(21, coulomb(21))
    D = p.dim
    xs = [O.splitmix(500 + v, D) for v in range(nbr)]
    dx = [capi.DeviceBuffer.from_host(arch, x) for x in xs]
    dy = [capi.DeviceBuffer.from_host(arch, np.full(D, 0.5)) for _ in range(nbr)]
    p.hv_vectors_device([b.ptr for b in dx], [b.ptr for b in dy], via_host=via_host)
    ys = [b.download() for b in dy]
    for v in range(nbr):
        y_ref = O.fs_hv(ref_space, fac, xs[v])
        assert np.linalg.norm(ys[v] - y_ref) <= 1e-12 * np.linalg.norm(y_ref), v
    if nbr >= 8:
        X = np.stack(xs[:8], axis=1).reshape(-1)
        Y = p.hv(X, 8).reshape(D, 8)
        for v in range(8):
            assert np.array_equal(ys[v], Y[:, v])
    # add on a row range: rows outside keep their values
    a, b = 100, D - 300
    p.hv_vectors_device([b_.ptr for b_ in dx], [b_.ptr for b_ in dy], add=True, first=a, count=b - a,
                        via_host=via_host)
    for v in range(nbr):
        y2 = dy[v].download()
        assert np.array_equal(y2[:a], ys[v][:a]) and np.array_equal(y2[b:], ys[v][b:])
        assert np.allclose(y2[a:b], 2 * ys[v][a:b], rtol=1e-13, atol=0)
    for buf in dx + dy:
        buf.free()


def test_hv_over_separate_vectors_spin(arch):
    from diagham_amd import capi
    L = 16
    p = capi.Problem.spin_chain(arch, L, 0)
    ref = O.SpinChain(L, 0)
    J = np.ones(L)
    xs = [O.splitmix(600 + v, p.dim) for v in range(6)]
    dx = [capi.DeviceBuffer.from_host(arch, x) for x in xs]
    dy = [capi.DeviceBuffer(arch, p.dim) for _ in range(6)]
    p.hv_vectors_device([b.ptr for b in dx], [b.ptr for b in dy])
    for v in range(6):
        y_ref = np.zeros(p.dim)
        O.lib().or_spin_hv(ref.h, O.dptr(J), O.dptr(J), 1, O.dptr(xs[v]), O.dptr(y_ref))
        assert np.linalg.norm(dy[v].download() - y_ref) <= 1e-12 * np.linalg.norm(y_ref)
    for buf in dx + dy:
        buf.free()
    p.close()


@pytest.mark.parametrize("k,lpr", [(1, 1), (1, 2), (8, 2)])
def test_free_pair_rows_are_bitwise_the_range_rows(n8_2s21, k, lpr):
    """The free-pair iterator visits the terms of each row in the order of the range loop, so with
    the same lanes per row the products agree bit for bit."""
    X = np.stack([O.splitmix(700 + v, n8_2s21.dim) for v in range(k)], axis=1).reshape(-1)
    n8_2s21.set_launch(lanes_per_row=lpr, block_size=256, index_mode=4)
    Y1 = n8_2s21.hv(X, k)
    n8_2s21.set_launch(lanes_per_row=lpr, block_size=256, index_mode=3)
    Y3 = n8_2s21.hv(X, k)
    n8_2s21.set_launch(lanes_per_row=4, block_size=256, index_mode=1)
    if lpr == 1:
        assert np.array_equal(Y1, Y3)
    else:  # lanes take different terms, and their partial sums meet in another order
        assert np.linalg.norm(Y1 - Y3) <= 1e-14 * np.linalg.norm(Y1)



@pytest.mark.parametrize("n,total_lz,lz_max", [(4, 0, 8), (4, 2, 8), (5, 3, 9), (6, 0, 11)])
def test_l2_product_is_the_ladder_operator(arch, n, total_lz, lz_max):
    """The L^2 product on the device, column by column, equals L^- L^+ + Lz^2 + Lz built from
    Jordan-Wigner ladder operators (ParticleOnSphereL2Hamiltonian.cc:240 defines the operator)."""
    from diagham_amd import capi
    from test_l2_cpu import ladder_l2
    p = capi.Problem.sphere_l2(arch, n, total_lz, lz_max, 1.0)
    L2 = ladder_l2(n, total_lz, lz_max)
    assert p.dim == L2.shape[0]
    H = np.stack([p.hv(e) for e in np.eye(p.dim)], axis=1)
    assert np.max(np.abs(H - L2)) < 1e-12 * max(1.0, np.max(np.abs(L2)))
    p.close()


@pytest.mark.parametrize("n,total_lz,lz_max", [(4, 0, 28), (4, 2, 31), (5, 1, 33)])
@pytest.mark.parametrize("k", [1, 2, 8])
@pytest.mark.parametrize("launch", [None, (1, 1024, 1), (2, 256, 4), (1, 512, 3)])
def test_hv_parity_at_the_14_bit_rank_split(arch, n, total_lz, lz_max, k, launch):
    """29 to 34 orbitals: the rank tables split at 14 bits, the 16-bit low table staged in LDS and
    the high table (2^15 to 2^20 entries) read from global memory; the automatic launch and explicit
    shapes of each row routine, 32-bit (32 orbitals) and 64-bit state words."""
    from diagham_amd import capi
    p = capi.Problem.sphere(arch, n, total_lz, lz_max, coulomb(lz_max))
    ref_space = O.FermionSphere(n, total_lz, lz_max)
    assert p.dim == ref_space.dim
    assert np.array_equal(p.states(), ref_space.states())
    if launch:
        p.set_launch(lanes_per_row=launch[0], block_size=launch[1], index_mode=launch[2])
    fac = O.Factors(lz_max, coulomb(lz_max))
    X = np.stack([O.splitmix(900 + v, p.dim) for v in range(k)], axis=1)
    Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
    for v in range(k):
        y_ref = O.fs_hv(ref_space, fac, X[:, v])
        err = np.linalg.norm(Y[:, v] - y_ref) / np.linalg.norm(y_ref)
        assert err < 1e-12, (k, launch, v, err)
    p.close()


def test_basis_from_diagham_states(arch):
    """dh_fermion_sphere_from_states adopts a StateDescription built elsewhere (here the oracle's
    restatement of GenerateStates): the full sector in the reference's order is accepted and gives
    the products of the generated basis; a reordered array, or one that is not the full sector, is
    refused with the first differing index named."""
    import ctypes
    from diagham_amd import capi
    n, lz, lz_max = 6, 0, 15
    ref = O.FermionSphere(n, lz, lz_max)
    words = np.ascontiguousarray(ref.states(), dtype=np.uint64)
    h = ctypes.c_void_p()
    assert capi.gpu().dh_fermion_sphere_from_states(arch.ctx, ctypes.byref(h), n, lz, lz_max,
                                                    words.ctypes.data_as(capi.P_U64), words.size) == 0
    assert capi.gpu().dh_basis_dimension(h) == ref.dim
    back = np.zeros(ref.dim, np.uint64)
    assert capi.gpu().dh_basis_get_states(h, back.ctypes.data_as(capi.P_U64)) == 0
    assert np.array_equal(back, words)
    assert capi.gpu().dh_basis_destroy(h) == 0
    swapped = words.copy()
    swapped[[10, 11]] = swapped[[11, 10]]
    bad = ctypes.c_void_p()
    assert capi.gpu().dh_fermion_sphere_from_states(arch.ctx, ctypes.byref(bad), n, lz, lz_max,
                                                    swapped.ctypes.data_as(capi.P_U64), swapped.size) == capi.DH_E_ARG
    assert b"state 10 " in capi.gpu().dh_last_error(arch.ctx)
    assert capi.gpu().dh_fermion_sphere_from_states(arch.ctx, ctypes.byref(bad), n, lz, lz_max,
                                                    words.ctypes.data_as(capi.P_U64), words.size - 1) == capi.DH_E_ARG
    assert b"not the full sector" in capi.gpu().dh_last_error(arch.ctx)


@pytest.mark.parametrize("n,total_lz,lz", [(10, 0, 27), (10, 4, 26)])
@pytest.mark.parametrize("k", [1, 4])
def test_both_rank_tables_in_lds(arch, n, total_lz, lz, k):
    """27 and 28 orbitals with enough rows: 1024-thread workgroups hold both rank tables."""
    from diagham_amd import capi
    V = capi.coulomb_pseudopotentials(lz, True)
    p = capi.Problem.sphere(arch, n, total_lz, lz, V)
    assert p.dim >= 65536 * 2
    X = np.random.default_rng(k).standard_normal((p.dim, k))
    Y = p.hv(X.reshape(-1), k).reshape(p.dim, k)
    p.close()
    ref = O.fs_hv(O.FermionSphere(n, total_lz, lz), O.Factors(lz, V), np.ascontiguousarray(X[:, k - 1]))
    assert np.linalg.norm(Y[:, k - 1] - ref) <= 1e-12 * np.linalg.norm(ref)
