"""bd_cholesky: the library's blocked factor on a caller's device matrix
(the replacement of cusolverDnDpotrf, func_cuda.cu:3513-3534), through the
C-ABI, against the compiled reference's factor (the |f| rule of
func.cpp:825-835), LAPACK, and the factor the step itself takes."""
import os
import threading

import numpy as np
import pytest

from brownian_dynamics_cuda_amd import engine as E
from brownian_dynamics_cuda_amd import fiber as Fb
from decks import rel_err

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def spd(m, seed):
    """A well-conditioned SPD matrix: RPY-like diagonal dominance."""
    g = np.random.default_rng(seed)
    X = g.standard_normal((m, m)) / np.sqrt(m)
    return X @ X.T + np.diag(g.uniform(1.0, 2.0, m))


def test_negative_pivots_against_reference():
    z = np.load(os.path.join(GOLDEN, "negative_pivot.npz"))
    L, neg = E.cholesky_device(z["D"])
    assert neg == int(z["neg"]) == 6
    assert rel_err(L, z["L"]) <= 1e-10


@pytest.mark.parametrize("m", [1, 3, 64, 65, 200, 1031])
def test_sizes_against_lapack(m):
    D = spd(m, m)
    L, neg = E.cholesky_device(D)
    assert neg == 0
    assert rel_err(L, np.linalg.cholesky(D)) <= 1e-12
    assert np.all(np.triu(L, 1) == 0)


@pytest.mark.parametrize("m", [2, 15, 16, 17, 33, 47, 63, 80, 127, 129])
def test_blocks_of_the_diagonal_tile(m):
    """Sizes around the 16x16 blocks of the diagonal tile's elimination, with
    the |f| rule in every block: D = U diag(s) U^T with U unit lower
    triangular and signs s, so pivot i is s_i and the factor the algorithm of
    func.cpp:806-836 gives, here in extended precision."""
    g = np.random.default_rng(m)
    U = np.tril(g.uniform(-0.5, 0.5, (m, m)) / np.sqrt(m), -1) + np.eye(m)
    s = np.where(g.random(m) < 0.3, -1.0, 1.0) * g.uniform(0.5, 2.0, m)
    s[0] = abs(s[0])
    D = (U * s) @ U.T
    D = np.tril(D) + np.tril(D, -1).T
    C = D.astype(np.longdouble)
    L = np.zeros_like(C)
    neg = 0
    for j in range(m):
        f = C[j, j]
        neg += int(f < 0)
        L[j:, j] = C[j:, j] / np.sqrt(abs(f))
        L[j, j] = np.sqrt(abs(f))
        C[j + 1:, j + 1:] -= np.outer(L[j + 1:, j], L[j + 1:, j])
    Lg, ng = E.cholesky_device(D)
    assert ng == neg
    assert rel_err(Lg, L.astype(np.float64)) <= 1e-12
    # a power of four in D is its root in L, exactly
    for k in (-600, 600):
        Ls, _ = E.cholesky_device(np.ldexp(D, k))
        assert np.array_equal(Ls, np.ldexp(Lg, k // 2))


@pytest.mark.parametrize("m", [3, 17, 64, 130])
@pytest.mark.parametrize("scale", [(-530,), (505,), (0, -530), (-530, 505, 0)])
def test_pivots_outside_the_normal_range(m, scale):
    """Pivots whose reciprocal is no FP64 number (below 2^-1024) or a subnormal
    one, alone and beside others: D = S T T^T S with T of small whole numbers
    and S powers of two, exact in FP64, has the factor S T.  T's diagonal of 16
    outweighs its other entries, so the factor is well conditioned."""
    g = np.random.default_rng(m)
    T = np.tril(g.integers(-1, 2, (m, m)) * (g.random((m, m)) < 4.0 / m), -1) + 16.0 * np.eye(m)
    k = np.resize(scale, m)
    D = np.ldexp(T @ T.T, k[:, None] + k[None, :])
    L, neg = E.cholesky_device(D)
    assert neg == 0
    assert rel_err(np.ldexp(L, -k[:, None]), T) <= 1e-12


@pytest.mark.parametrize("m", [2, 17, 64, 130, 200])
@pytest.mark.parametrize("mode", [E.CHOL_FP64, E.CHOL_FP32, E.CHOL_BF16])
def test_dependent_rows(m, mode):
    """Matrices with rows that are the same, a multiple of another or 0: the
    pivot is a rounding error or exactly 0, and the factor is finite with
    |L L^T - D| at most (m + 1) u |L| |L^T|, twice for the |f| of a pivot below
    0, u = 2^-53, and 2^-24 for the products of the reduced modes."""
    for j in [k for k in (0, 3, 15, 16, 40, 62, 63, 64, 100, 128) if k < m - 1]:
        for scale in (1.0, -1.0, 0.0):
            D = spd(m, m)
            D[j + 1, :] = scale * D[j, :]
            D[:, j + 1] = scale * D[:, j]
            D[j + 1, j + 1] = scale * scale * D[j, j]
            L, neg = E.cholesky_device(D, mode)
            assert np.all(np.isfinite(L)), (j, scale)
            assert neg <= 1
            A = np.abs(L) @ np.abs(L.T)
            u = 2.0 ** (-53 if mode == E.CHOL_FP64 else -24)
            assert np.all(np.abs(L @ L.T - D) <= (2 * m + 2) * u * A + (m + 1) * 2.0 ** -53 * np.abs(D)), (j, scale)


# In FP64 super-panels start at 60 block columns: 83 and 84 are panels with a
# last one of three and of four block columns, and the first sizes with and the
# last without are those of test_panels_solved_in_one_launch.
@pytest.mark.parametrize("m,mode", [(5312, E.CHOL_FP64), (5313, E.CHOL_FP64), (4033, E.CHOL_FP32), (4033, E.CHOL_BF16)])
def test_ends_of_the_super_panels(m, mode):
    """The first sizes with super-panels (84 and 64 block columns) and the last
    without: 64 = 7 8 + 8 and 84 = 10 8 + 4 block columns, whose trailing
    updates go on to factor the next panel's first tile.  |L L^T - D| is at
    most (m + 1) u |L| |L^T|, with u = 2^-53 in FP64 and 2^-24 for the products
    of the reduced modes."""
    D = spd(m, 3)
    L, neg = E.cholesky_device(D, mode)
    u = 2.0 ** (-53 if mode == E.CHOL_FP64 else -24)
    v = np.random.default_rng(1).standard_normal((m, 4))
    bound = (m + 1) * u * (np.abs(L) @ (np.abs(L.T) @ np.abs(v)))
    assert neg == 0
    assert np.all(np.abs(L @ (L.T @ v) - D @ v) <= bound + (m + 1) * 2.0 ** -53 * (np.abs(D) @ np.abs(v)))


@pytest.mark.parametrize("mode, nt", [(E.CHOL_FP64, 59), (E.CHOL_FP64, 60), (E.CHOL_FP64, 65), (E.CHOL_FP64, 71),
                                      (E.CHOL_FP64, 81), (E.CHOL_FP32, 63), (E.CHOL_FP32, 64), (E.CHOL_FP32, 73)])
def test_panels_solved_in_one_launch(mode, nt):
    """The first sizes whose super-panels factor their diagonal block beside
    the trailing update and solve their rows in one launch (60 and 64 block
    columns) and the last without; last panels of one (65, 73, 81), four and
    seven (71) block columns; 65 and more trailing block rows (two workgroups
    per CU) and more tiles than the steps take (71, 73, 81); two rows of padding.
    |L L^T - D| at most (m + 1) u |L| |L^T|, with u = 2^-53 in FP64 and 2^-24
    for the products of FP32."""
    m = 64 * nt - 2
    D = spd(m, 3)
    L, neg = E.cholesky_device(D, mode)
    u = 2.0 ** (-53 if mode == E.CHOL_FP64 else -24)
    v = np.random.default_rng(1).standard_normal((m, 4))
    bound = (m + 1) * u * (np.abs(L) @ (np.abs(L.T) @ np.abs(v)))
    assert neg == 0
    assert np.all(np.abs(L @ (L.T @ v) - D @ v) <= bound + (m + 1) * 2.0 ** -53 * (np.abs(D) @ np.abs(v)))


@pytest.mark.parametrize("m", [4030, 4032, 4094, 4542])
def test_super_panels_in_bf16(m):
    """The last sizes without super-panels in BF16 (63 block columns, with and
    without padding), the first with (64, a whole last panel) and 71 (a last one
    of seven).  |L L^T - D| at most (m + 1) u |L| |L^T|, u = 2^-24 for the
    three-slice products."""
    D = spd(m, 3)
    L, neg = E.cholesky_device(D, E.CHOL_BF16)
    v = np.random.default_rng(1).standard_normal((m, 4))
    bound = (m + 1) * 2.0 ** -24 * (np.abs(L) @ (np.abs(L.T) @ np.abs(v)))
    assert neg == 0
    assert np.all(np.abs(L @ (L.T @ v) - D @ v) <= bound + (m + 1) * 2.0 ** -53 * (np.abs(D) @ np.abs(v)))


# In FP64 too: from 60 block columns.
def test_super_panel_size_and_mixed_modes():
    """4500 rows: 71 block columns, super-panels of 8 in the reduced modes."""
    D = spd(4500, 7)
    L0 = np.linalg.cholesky(D)
    L, neg = E.cholesky_device(D)
    assert neg == 0 and rel_err(L, L0) <= 1e-12
    for mode in (E.CHOL_FP32, E.CHOL_BF16):
        Lm, neg = E.cholesky_device(D, mode)
        err = np.linalg.norm(Lm @ Lm.T - D) / np.linalg.norm(D)
        assert neg == 0 and err <= 1e-6, (mode, err)


@pytest.mark.parametrize("threads", [1, 3])
def test_kept_workspace(threads):
    """The workspace kept between calls: sizes that need a larger one, fit the
    kept one and leave most of it unused, from one thread and from three at
    once, with a release in between; each call's factor as the first one's."""
    lib = E.load_library()
    sizes = [65, 700, 130, 1, 700, 900, 64]
    mats = {m: spd(m, m) for m in sizes}
    assert lib.bd_cholesky_release() == 0
    ref = {m: np.linalg.cholesky(D) for m, D in mats.items()}
    bad = []

    def work(first):
        for rep in range(2):
            for m in sizes[first:] + sizes[:first]:
                L, neg = E.cholesky_device(mats[m])
                if neg != 0 or rel_err(L, ref[m]) > 1e-12:
                    bad.append((first, m))
            lib.bd_cholesky_release()

    ts = [threading.Thread(target=work, args=(2 * i,)) for i in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    assert lib.bd_cholesky_release() == 0 and lib.bd_cholesky_release() == 0


def test_same_factor_as_the_step():
    """The tensor of the 100-nucleosome fiber: bd_cholesky on it equals the
    factor the step forms in place (same kernels, same arithmetic)."""
    fib, st = Fb.make_config(2)
    with E.BDEngine(fib, use_graph=False) as eng:
        eng.set_state(st, rebuild=True)
        D = eng.get_tensor()
        eng.factor()
        L0, neg0 = eng.get_factor()
    L, neg = E.cholesky_device(D)
    assert neg == neg0 == 0
    assert np.array_equal(L, L0)


def test_in_place_and_argument_errors():
    lib = E.load_library()
    D = spd(130, 3)
    buf = E.DeviceBuffer(D.nbytes)
    try:
        buf.upload(D)
        import ctypes as C
        neg = C.c_int(-1)
        assert lib.bd_cholesky(130, buf.ptr, 130, buf.ptr, 130, E.CHOL_FP64, C.byref(neg), None) == 0
        L = buf.download((130, 130))
        assert neg.value == 0 and rel_err(L, np.linalg.cholesky(D)) <= 1e-12
        assert lib.bd_cholesky(0, buf.ptr, 130, buf.ptr, 130, 0, None, None) == -1
        assert lib.bd_cholesky(130, buf.ptr, 100, buf.ptr, 130, 0, None, None) == -1
        assert lib.bd_cholesky(130, buf.ptr, 130, buf.ptr, 130, 7, None, None) == -1
    finally:
        buf.free()
