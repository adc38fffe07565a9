"""Device kernels at the sizes where their dispatch or their tiles can go
wrong: tile edges, remainders, the smallest sizes and both sides of a rule
(GPU).  Tolerances are forward-error bounds: unit roundoff times the number of
roundings an entry passes through times the sum of its absolute products."""
import ctypes

import numpy as np
import pytest

from gcge_old_amd import DeviceMatrix, DeviceMultiVec, _native, adjoint, problems
from oracle import adjoint as oadj

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def _corner_abs_sums(E, X):
    """sum of |x| over the 8 corners of every element, (E^3, k)"""
    N = E - 1
    full = np.zeros((E + 1, E + 1, E + 1, X.shape[1]))
    full[1:E, 1:E, 1:E] = np.abs(X).reshape(N, N, N, -1)
    s = sum(full[a:a + E, b:b + E, c:c + E] for a in (0, 1) for b in (0, 1) for c in (0, 1))
    return s.reshape(E ** 3, -1)


@pytest.mark.parametrize("permuted", [False, True])
@pytest.mark.parametrize("two_blocks", [False, True])
@pytest.mark.parametrize("E,k", [(2, 1), (3, 2), (9, 5), (17, 3), (33, 9), (92, 2)])
def test_element_gradient_sizes(E, k, two_blocks, permuted):
    """Four or eight node planes per thread (from E = 91), columns shared by
    four threads (k below, above and no multiple of four), planes cut off at
    the mesh end, one or two blocks, permuted rows."""
    rng = np.random.default_rng(E * 100 + k)
    n = (E - 1) ** 3
    X = rng.standard_normal((n, k))
    Y = rng.standard_normal((n, k)) if two_blocks else X
    w = rng.standard_normal(k)
    print(f"element gradient E={E} k={k} two={two_blocks} permuted={permuted}", flush=True)
    row = rng.permutation(n) if permuted else None
    Xr, Yr = np.empty_like(X), np.empty_like(Y)
    Xr[row if permuted else slice(None)], Yr[row if permuted else slice(None)] = X, Y
    dX = DeviceMultiVec.from_host(Xr)
    got = adjoint.q1_kappa_gradient(E, dX, w, Y=DeviceMultiVec.from_host(Yr) if two_blocks else None,
                                    node_row=row)
    want = oadj.q1_element_gradient(E, X, w, Y=Y if two_blocks else None)
    # 36 Khat has entries up to 12 in absolute value, and so have the products
    # of the transformed corner values; both sides round 16 + k times at most
    bound = (12.0 / 36.0 / E) * (_corner_abs_sums(E, X) * _corner_abs_sums(E, Y)) @ np.abs(w)
    assert np.all(np.abs(got - want) <= 2 * (16 + k) * EPS * bound)


@pytest.mark.parametrize("k", [1, 4, 5, 12, 13, 16, 20, 47, 80, 112, 113, 128, 129, 257])
@pytest.mark.parametrize("n,m", [(1, 1), (2, 3), (127, 4), (128, 33), (129, 16), (3000, 35)])
def test_linear_comb_tiles(n, m, k):
    """Quads and tiles of the output columns, one to three column groups,
    stages of four and eight steps with and without a rest, a single row and
    rows that end inside a pair, a wave and a workgroup; NaN in columns next to
    the ones that are read."""
    rng = np.random.default_rng(1000 * m + k + n)
    V = rng.standard_normal((n, m + 2))
    V[:, 0] = V[:, -1] = np.nan
    C = np.asfortranarray(rng.standard_normal((m, k)))
    Y0 = rng.standard_normal((n, k + 1))
    print(f"linear combination n={n} m={m} k={k}", flush=True)
    for beta in (0.0, -1.5):
        dV, dY = DeviceMultiVec.from_host(V), DeviceMultiVec.from_host(Y0)
        _native.hip().GCGE_HIP_LinearComb(dV.handle, 1, m, _native.as_dptr(C), m, beta, dY.handle, 0, k)
        got = dY.get()
        want = V[:, 1:-1] @ C + beta * Y0[:, :k]
        bound = np.abs(V[:, 1:-1]) @ np.abs(C) + abs(beta) * np.abs(Y0[:, :k])
        assert np.all(np.abs(got[:, :k] - want) <= 2 * (m + 2) * EPS * bound)
        np.testing.assert_array_equal(got[:, k:], Y0[:, k:])


@pytest.mark.parametrize("m,k", [(5, 3), (40, 20), (130, 100), (70, 128)])
def test_linear_comb_over_its_input(m, k):
    """Output columns that overlap the input columns (one block, up to 128
    output columns): the same bits as into another block."""
    n = 1003
    rng = np.random.default_rng(m + k)
    cols = max(m, k) + 2
    A = rng.standard_normal((n, cols))
    C = np.asfortranarray(rng.standard_normal((m, k)))
    dA, dY = DeviceMultiVec.from_host(A), DeviceMultiVec(n, k)
    lib = _native.hip()
    lib.GCGE_HIP_LinearComb(dA.handle, 0, m, _native.as_dptr(C), m, 0.0, dY.handle, 0, k)
    lib.GCGE_HIP_LinearComb(dA.handle, 0, m, _native.as_dptr(C), m, 0.0, dA.handle, 2, k)
    np.testing.assert_array_equal(dA.get(2, k), dY.get())


@pytest.mark.parametrize("m,k", [(9, 1), (1, 9), (17, 5), (16, 100), (48, 20), (129, 33), (113, 113),
                                 (300, 114), (257, 127), (400, 10), (30, 390), (130, 260)])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 65, 1000])
def test_gram_tiles(n, m, k):
    """One to three tiles of the wider block per wave with waves left over,
    tiles and quads of the other, several result blocks, fewer columns on
    either side; less than a stage of rows, whole stages and a rest; NaN in
    columns next to the ones that are read."""
    rng = np.random.default_rng(1000 * m + k + n)
    V, W = rng.standard_normal((n, m + 2)), rng.standard_normal((n, k + 2))
    V[:, 0] = V[:, -1] = W[:, 0] = W[:, -1] = np.nan
    dV, dW = DeviceMultiVec.from_host(V), DeviceMultiVec.from_host(W)
    print(f"Gram n={n} m={m} k={k}", flush=True)
    G = np.zeros((m, k), order="F")
    _native.hip().GCGE_HIP_Gram(dV.handle, 1, m, dW.handle, 1, k, _native.as_dptr(G), m)
    V, W = V[:, 1:-1], W[:, 1:-1]
    assert np.all(np.abs(G - V.T @ W) <= 2 * (n + 2) * EPS * (np.abs(V).T @ np.abs(W)))


def _permuted_q1(E, seed):
    K = problems.q1_fem_3d(E, problems.lognormal_kappa(E, seed))[0]
    return problems.symmetric_permutation(K, np.random.default_rng(seed).permutation(K.nrows))


@pytest.mark.parametrize("k", [11, 12, 13, 63, 64, 65, 127, 128, 129, 200])
def test_row_gather_product_widths(k):
    """Below and from the smallest width of the row gathers, one and two
    columns per lane, one and two passes, odd last columns; bit for bit the
    sums of the element gathers (the same order)."""
    A = DeviceMatrix(_permuted_q1(9, 3))
    assert A.storage_info()["storage"] == "rows"
    X = np.random.default_rng(k).standard_normal((A.nrows, k + 1))
    dX, dY, dZ = DeviceMultiVec.from_host(X), DeviceMultiVec(A.nrows, k + 1), DeviceMultiVec(A.nrows, k)
    lib = _native.hip()
    print(f"row gathers k={k}", flush=True)
    lib.GCGE_HIP_SpMM(A.handle, dX.handle, 1, dY.handle, 0, k)
    A.set_storage("sliced")
    lib.GCGE_HIP_SpMM(A.handle, dX.handle, 1, dZ.handle, 0, k)
    np.testing.assert_array_equal(dY.get(0, k), dZ.get())
    assert np.all(dY.get(k, 1) == 0.0)


@pytest.mark.parametrize("fp32,k,rtol", [(False, 70, 1e-10), (False, 131, 1e-10), (True, 70, 1e-4),
                                         (True, 131, 1e-4), (True, 20, 1e-4)])
def test_row_gather_block_cg(fp32, k, rtol):
    """p.w and p.p of the row gathers (one to four columns per lane, last pass
    partly filled) inside the block CG, against the element gathers."""
    A = DeviceMatrix(_permuted_q1(9, 4))
    rng = np.random.default_rng(k)
    b, x0 = rng.standard_normal((A.nrows, k)), np.zeros((A.nrows, k))
    lib = _native.hip()
    out = []
    for storage in ("rows", "sliced"):
        A.set_storage(storage)
        A.set_precision(fp32)
        R, X = DeviceMultiVec.from_host(b), DeviceMultiVec.from_host(x0)
        lib.GCGE_HIP_SetLinearSolverParams(8, 1e-30, 0, 0.0, None)
        lib.GCGE_HIP_MultiLinearSolve(A.handle, R.handle, 0, X.handle, 0, k)
        lib.GCGE_HIP_SetLinearSolverParams(20, 1e-2, 0, 0.0, None)
        out.append(X.get())
    assert np.linalg.norm(out[0] - out[1]) <= rtol * np.linalg.norm(out[1])


@pytest.mark.parametrize("n,m,k", [(1100007, 12, 20), (1060003, 17, 16), (600011, 50, 10), (240007, 140, 8),
                                   (200003, 140, 30), (27001, 200, 8), (17577, 128, 16), (42877, 256, 32)])
def test_gram_stage_lengths(n, m, k):
    """Stages of four and eight 16-row groups (blocks beyond 256 MiB, two tiles
    a wave on a small mesh) with a rest of rows, and one workgroup per CU."""
    rng = np.random.default_rng(n + m)
    V, W = rng.standard_normal((n, m)), rng.standard_normal((n, k))
    dV, dW = DeviceMultiVec.from_host(V), DeviceMultiVec.from_host(W)
    print(f"Gram n={n} m={m} k={k}", flush=True)
    G = np.zeros((m, k), order="F")
    _native.hip().GCGE_HIP_Gram(dV.handle, 0, m, dW.handle, 0, k, _native.as_dptr(G), m)
    assert np.all(np.abs(G - V.T @ W) <= 2 * (n + 2) * EPS * (np.abs(V).T @ np.abs(W)))


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("E,k,rows", [(42, 7, False), (42, 8, True), (42, 9, True), (42, 11, True), (32, 12, True),
                                      (26, 11, False), (26, 12, True), (24, 12, False), (24, 13, True),
                                      (9, 15, False), (9, 16, True), (9, 129, True), (33, 70, True)])
def test_row_gather_threshold(E, k, rows, fp32):
    """Both sides of the smallest width of the row gathers at each size of the
    rule, one-wave and four-wave workgroups: products bit for bit those of the
    element gathers; a float64 block CG gives their bits exactly where both
    storages run them (the forms add p.w up in different orders, which
    float32 directions round away)."""
    A = DeviceMatrix(_permuted_q1(E, 5))
    assert A.storage_info()["storage"] == "rows"
    rng = np.random.default_rng(100 * E + k)
    b, x0 = rng.standard_normal((A.nrows, k)), np.zeros((A.nrows, k))
    lib = _native.hip()
    print(f"row gathers E={E} k={k} fp32={fp32}", flush=True)
    out = []
    for storage in ("rows", "sliced"):
        A.set_storage(storage)
        X, Y = DeviceMultiVec.from_host(b), DeviceMultiVec(A.nrows, k)
        lib.GCGE_HIP_SpMM(A.handle, X.handle, 0, Y.handle, 0, k)
        A.set_precision(fp32)
        S = DeviceMultiVec.from_host(x0)
        lib.GCGE_HIP_SetLinearSolverParams(8, 1e-30, 0, 0.0, None)
        lib.GCGE_HIP_MultiLinearSolve(A.handle, X.handle, 0, S.handle, 0, k)
        lib.GCGE_HIP_SetLinearSolverParams(20, 1e-2, 0, 0.0, None)
        A.set_precision(False)
        out.append((Y.get(), S.get()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    assert np.linalg.norm(out[0][1] - out[1][1]) <= (1e-4 if fp32 else 1e-10) * np.linalg.norm(out[1][1])
    if not fp32:
        assert np.array_equal(out[0][1], out[1][1]) == (not rows)


@pytest.mark.parametrize("k", [1, 3, 4, 5, 8, 9, 33, 128, 129, 300])
@pytest.mark.parametrize("n,m", [(1, 1), (2, 2), (511, 3), (512, 4), (513, 5), (1025, 6), (1003, 7), (2049, 8),
                                 (140001, 1), (140001, 4)])
def test_linear_comb_few_inputs(n, m, k):
    """One to eight input columns (from five on few outputs only), column ranges
    on both sides of one workgroup per CU, rests of four columns, rows that end
    inside a pair and a workgroup; infinities stay in their rows; NaN in columns
    next to the ones that are read; over the input the same bits."""
    rng = np.random.default_rng(1000 * m + k + n)
    V = rng.standard_normal((n, m + 2))
    V[:, 0] = V[:, -1] = np.nan
    V[n // 2, m] = np.inf
    C = np.asfortranarray(rng.standard_normal((m, k)))
    Y0 = rng.standard_normal((n, k + 1))
    lib = _native.hip()
    print(f"linear combination n={n} m={m} k={k}", flush=True)
    rows = np.arange(n) != n // 2
    for beta in (0.0, -1.5):
        dV, dY = DeviceMultiVec.from_host(V), DeviceMultiVec.from_host(Y0)
        lib.GCGE_HIP_LinearComb(dV.handle, 1, m, _native.as_dptr(C), m, beta, dY.handle, 0, k)
        got = dY.get()
        want = V[rows, 1:-1] @ C + beta * Y0[rows, :k]
        bound = np.abs(V[rows, 1:-1]) @ np.abs(C) + abs(beta) * np.abs(Y0[rows, :k])
        assert np.all(np.abs(got[rows, :k] - want) <= 2 * (m + 2) * EPS * bound)
        np.testing.assert_array_equal(got[n // 2, :k], np.inf * C[m - 1])
        np.testing.assert_array_equal(got[:, k:], Y0[:, k:])
    if k <= 128:
        A = np.zeros((n, max(m, k) + 1))
        A[:, :m] = V[:, 1:-1]
        dA, dY = DeviceMultiVec.from_host(A), DeviceMultiVec(n, k)
        lib.GCGE_HIP_LinearComb(dA.handle, 0, m, _native.as_dptr(C), m, 0.0, dY.handle, 0, k)
        lib.GCGE_HIP_LinearComb(dA.handle, 0, m, _native.as_dptr(C), m, 0.0, dA.handle, 1, k)
        np.testing.assert_array_equal(dA.get(1, k), dY.get())


@pytest.mark.parametrize("two_blocks", [False, True])
def test_element_gradient_reported_bytes(two_blocks):
    """The gradient's recorded traffic: X once where Y is X, else both blocks."""
    E, k = 20, 7
    X = DeviceMultiVec.from_host(np.random.default_rng(0).standard_normal(((E - 1) ** 3, k)))
    Y = DeviceMultiVec.from_host(np.ones(((E - 1) ** 3, k))) if two_blocks else None
    lib = _native.hip()
    lib.GCGE_HIP_ProfileReset()
    lib.GCGE_HIP_ProfileEnable(1)
    adjoint.q1_kappa_gradient(E, X, np.ones(k), Y=Y)
    lib.GCGE_HIP_ProfileEnable(0)
    ms, count, moved = ctypes.c_double(), ctypes.c_int(), ctypes.c_double()
    lib.GCGE_HIP_KernelStats(b"q1_elem_grad", ctypes.byref(ms), ctypes.byref(count), ctypes.byref(moved))
    lib.GCGE_HIP_ProfileReset()
    assert count.value == 1
    assert moved.value == 8.0 * ((2 if two_blocks else 1) * k * (E - 1) ** 3 + E ** 3)


@pytest.mark.parametrize("n,m,k", [(1 << 20, 192, 9), (1048579, 193, 16), (1100001, 300, 13), ((1 << 20) - 1, 193, 12),
                                   (1048579, 191, 12)])
def test_linear_comb_tall(n, m, k):
    """Both sides of the sizes from which 9 to 16 columns have their own waves
    of 64 rows; a rest of rows and of input columns, beta, and over the input.
    Eight distinct input columns in turn, so the reference folds C."""
    rng = np.random.default_rng(m + k)
    base, C = rng.standard_normal((n, 8)), np.asfortranarray(rng.standard_normal((m, k)))
    Y0 = rng.standard_normal((n, k))
    fold = lambda M: np.stack([M[c::8].sum(0) for c in range(8)])
    bound = np.abs(base) @ fold(np.abs(C))
    dV, dY = DeviceMultiVec(n, m + 1), DeviceMultiVec.from_host(Y0)
    for c in range(0, m, 8):
        dV.set(np.ascontiguousarray(base[:, :min(8, m - c)]), c)
    dV.set(np.full((n, 1), np.nan), m)
    lib = _native.hip()
    print(f"linear combination n={n} m={m} k={k}", flush=True)
    lib.GCGE_HIP_LinearComb(dV.handle, 0, m, _native.as_dptr(C), m, -1.5, dY.handle, 0, k)
    got = dY.get()
    want = base @ fold(C) - 1.5 * Y0
    assert np.all(np.abs(got - want) <= 2 * (m + 2) * EPS * (bound + 1.5 * np.abs(Y0)))
    lib.GCGE_HIP_LinearComb(dV.handle, 0, m, _native.as_dptr(C), m, 0.0, dY.handle, 0, k)
    lib.GCGE_HIP_LinearComb(dV.handle, 0, m, _native.as_dptr(C), m, 0.0, dV.handle, 3, k)
    np.testing.assert_array_equal(dV.get(3, k), dY.get())
    assert np.all(np.abs(dY.get() - base @ fold(C)) <= 2 * (m + 2) * EPS * bound)
