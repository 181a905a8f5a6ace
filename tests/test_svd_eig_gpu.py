"""The eigenvector path of the sector SVD (blocks of 16 to 640 columns) at the
edges of its tiles, and blocks it has to leave to the Jacobi kernels, against
numpy's LAPACK.

Tolerances: a backward-stable SVD of an m x n block is the exact one of a block
within c max(m, n) eps ||M||; c = 4 covers both factorisations compared.
Factors: the pair test of either path accepts cosines up to max(m, n) eps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = {"D": 2.0 ** -52, "S": 2.0 ** -23}


def dense_svd(x, dtype):
    from tnsp_amd import TAT

    m, n = x.shape
    t = getattr(TAT.No, dtype).Tensor(["a", "b"], [m, n])
    t.storage = x.reshape(-1)
    u, s, v = t.svd({"a"}, "U", "V", "SU", "SV")
    k = s.edges[0].dimension()
    um = u.transpose(["a", "U"]).storage.numpy().reshape(m, k).astype(np.float64)
    sm = np.diag(s.transpose(["SU", "SV"]).storage.numpy().reshape(k, k)).astype(np.float64)
    vm = v.transpose(["V", "b"]).storage.numpy().reshape(k, n).astype(np.float64)
    return um, sm, vm


def check(x, dtype, factors=True):
    u, s, v = dense_svd(x, dtype)
    x = x.astype(np.float32).astype(np.float64) if dtype == "S" else x
    ref = np.linalg.svd(x, compute_uv=False)
    tol = 4 * max(x.shape) * EPS[dtype]
    assert np.all(np.diff(s) <= 0)
    assert np.max(np.abs(s - ref[:len(s)])) <= tol * ref[0]
    assert np.all(ref[len(s):] <= tol * ref[0])
    if factors:
        assert np.linalg.norm((u * s) @ v - x) <= tol * np.linalg.norm(x)
        assert np.max(np.abs(u.T @ u - np.eye(len(s)))) <= tol
        assert np.max(np.abs(v @ v.T - np.eye(len(s)))) <= tol


@pytest.mark.parametrize("m,n", [(16, 16), (17, 40), (100, 23), (32, 32), (33, 47), (64, 64), (65, 63), (100, 66), (128, 128), (129, 130), (192, 192),
                                 (193, 200), (64, 700), (1100, 40), (320, 320), (321, 333), (640, 640), (641, 645)])
def test_random_blocks(m, n):
    check(np.random.default_rng(m * 1000 + n).standard_normal((m, n)), "D")


@pytest.mark.parametrize("m,n", [(40, 50), (130, 129), (260, 210)])
def test_float32_blocks(m, n):
    check(np.random.default_rng(m + n).standard_normal((m, n)).astype(np.float32), "S")


@pytest.mark.parametrize("n", [48, 150, 210])
@pytest.mark.parametrize("kind", ["graded", "close", "isometry", "rank", "tiny", "huge", "split", "zero_columns"])
def test_special_spectra(n, kind):
    """Graded, close and equal singular values, rank deficiency, entries at
    the ends of the range, matrices whose tridiagonal form splits: taken or
    left, the singular values are right.  Factors only where the path takes
    the block: those of the others are the Jacobi kernels', whose V recovered
    from U is not backward stable to this tolerance (150 graded columns: 2.5e-13
    of rebuilding error, with and without this path)."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, n))
    u, s, v = np.linalg.svd(x)
    if kind == "graded":
        x = (u * np.logspace(0, -12, n)) @ v
    elif kind == "close":
        x = (u * (1 + 1e-11 * np.arange(n))) @ v
    elif kind == "isometry":
        x = u
    elif kind == "rank":
        x = x[:, :n // 2] @ rng.standard_normal((n // 2, n))
    elif kind == "tiny":
        x = x * 1e-200
    elif kind == "huge":
        x = x * 1e200
    elif kind == "split":
        x = np.diag(1.0 + np.arange(n))
    elif kind == "zero_columns":
        x[:, n // 3:] = 0.0
    check(x, "D", factors=kind in ("tiny", "huge"))


def test_batch_of_mixed_sectors():
    """Sectors of every size class in one launch, some of them singular."""
    from helpers import to_gpu
    from oracle import tat

    K = tat.KINDS["BoseU1"]
    rng = np.random.default_rng(5)
    a = tat.Tensor(K, ["a", "b"], [([(0, 33), (1, 70), (-1, 150), (2, 200), (-2, 5), (3, 90)], False),
                                   ([(0, 90), (-1, 66), (1, 140), (-2, 230), (2, 9), (-3, 100)], False)])
    a.data[:] = rng.standard_normal(a.size)
    blk = a.block((5, 5))
    blk[...] = np.outer(np.arange(90.0), np.arange(100.0))
    g = to_gpu(a)
    for cut in (-1, 100):
        u, s, v = a.svd({"a"}, "cu", "cv", "su", "sv", cut)
        gu, gs, gv = g.svd({"a"}, "cu", "cv", "su", "sv", cut)
        if cut > 0:
            assert np.max(np.abs(gs.storage.numpy() - s.data)) <= 1e-12 * np.max(s.data)
        r1 = gu.contract(gs, {("cu", "su")}).contract(gv, {("sv", "cv")})
        r0 = u.contract(s, {("cu", "su")}).contract(v, {("sv", "cv")})
        assert np.linalg.norm(r1.storage.numpy() - r0.data) <= 1e-12 * np.linalg.norm(r0.data)


def check_orthonormal(x, dtype):
    u, s, v = dense_svd(x, dtype)
    tol = 4 * max(x.shape) * EPS[dtype]
    ref = np.linalg.svd(x.astype(np.float64), compute_uv=False)
    assert np.max(np.abs(s - ref[:len(s)])) <= tol * ref[0]
    assert np.linalg.norm((u * s) @ v - x) <= tol * np.linalg.norm(x)
    assert np.max(np.abs(u.T @ u - np.eye(len(s)))) <= tol
    assert np.max(np.abs(v @ v.T - np.eye(len(s)))) <= tol


def with_null_values(m, n, null):
    rng = np.random.default_rng(m + n + null)
    u, s, v = np.linalg.svd(rng.standard_normal((m, n)), full_matrices=False)
    s[len(s) - null:] = 0.0
    return (u * s) @ v


@pytest.mark.parametrize("m,n,null", [(135, 47, 1), (64, 64, 2), (200, 210, 3), (48, 90, 8), (48, 48, 1), (64, 64, 1),
                                      (64, 66, 1), (128, 128, 1), (200, 200, 1), (300, 301, 2), (640, 640, 1)])
def test_null_columns_are_completed(m, n, null):
    """A few zero singular values, up to square blocks, whose null direction
    no unit vector comes near: U and V^T stay orthonormal.  (Blocks with more
    than eight, of at most 192 rows and beyond 76 KiB, end in the register
    kernel, which completes nothing.)"""
    check_orthonormal(with_null_values(m, n, null), "D")


@pytest.mark.parametrize("n", [48, 100, 200])
def test_equal_columns_float32(n):
    """An exact null vector in single precision."""
    x = np.random.default_rng(n).standard_normal((n, n)).astype(np.float32)
    x[:, 7] = x[:, 31]
    check_orthonormal(x, "S")


@pytest.mark.parametrize("first", [(24, 24), (23, 31), (16, 16), (16, 31), (15, 31), (15, 15), (31, 20),
                                   (8, 9)])
def test_sector_does_not_depend_on_its_company(first):
    """A sector alone and beside a larger one that takes the eigenvector path:
    the same bits."""
    from tnsp_amd import TAT

    m, n = first
    x = np.random.default_rng(m + n).standard_normal((m, n))
    alone = TAT.BoseU1.D.Tensor(["a", "b"], [[(0, m)], [(0, n)]])
    pair = TAT.BoseU1.D.Tensor(["a", "b"], [[(0, m), (1, 70)], [(0, n), (-1, 64)]])
    pair.storage = np.random.default_rng(1).standard_normal(pair.storage.size)
    pair.blocks[[("a", 0), ("b", 0)]] = x
    alone.blocks[[("a", 0), ("b", 0)]] = x
    for one, two in zip(alone.svd({"a"}, "U", "V", "SU", "SV"), pair.svd({"a"}, "U", "V", "SU", "SV")):
        key = [(name, 0) for name in one.names]
        assert np.array_equal(one.blocks[key], two.blocks[key])
