"""The LDS Householder QR on blocks of extreme range and structure, against
numpy's LAPACK, signs included.  (The blocked kernel, for blocks beyond LDS,
does not scale.)

Tolerances: both factorisations are backward stable, Q orthogonal and A - Q R
zero to c max(m, n) eps with c = 4; Q and R themselves differ between two such
factorisations by that times the condition number of the block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = {"D": 2.0 ** -52, "S": 2.0 ** -23}


def dense_qr(x, dtype, lq):
    from tnsp_amd import TAT

    m, n = x.shape
    t = getattr(TAT.No, dtype).Tensor(["a", "b"], [m, n])
    t.storage = x.reshape(-1)
    # the last edge decides between QR (it belongs to R) and LQ (to Q)
    q, r = t.qr("r", {"a"} if lq else {"b"}, "Q", "R")
    k = min(m, n)
    if lq:
        return (q.transpose(["b", "Q"]).storage.numpy().reshape(n, k).astype(np.float64),
                r.transpose(["R", "a"]).storage.numpy().reshape(k, m).astype(np.float64))
    return (q.transpose(["a", "Q"]).storage.numpy().reshape(m, k).astype(np.float64),
            r.transpose(["R", "b"]).storage.numpy().reshape(k, n).astype(np.float64))


def check(x, dtype, lq, same=True):
    q, r = dense_qr(x, dtype, lq)
    a = x.astype(np.float32).astype(np.float64) if dtype == "S" else x
    a = a.T if lq else a
    scale = np.max(np.abs(a)) or 1.0
    a, r = a / scale, r / scale
    tol = 4 * max(a.shape) * EPS[dtype]
    assert np.max(np.abs(q.T @ q - np.eye(q.shape[1]))) <= tol
    assert np.linalg.norm(q @ r - a) <= tol * np.linalg.norm(a)
    assert np.all(np.tril(r, -1) == 0)
    if same:
        q0, r0 = np.linalg.qr(a)
        tol *= np.linalg.cond(a)
        assert np.linalg.norm(q - q0) <= tol * np.linalg.norm(q0)
        assert np.linalg.norm(r - r0) <= tol * np.linalg.norm(r0)


@pytest.mark.parametrize("n", [20, 40, 100])
@pytest.mark.parametrize("kind", ["triangular", "identity", "diagonal", "rank", "zero_column", "graded_columns",
                                  "ill_conditioned", "tiny", "huge", "overflowing", "zero_rows"])
def test_special_blocks(n, kind):
    """The result is a QR; where Q and R are determined by the
    block (full rank, well conditioned) they have the Householder signs."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n + 30, n))
    same = True
    if kind == "triangular":
        x = np.triu(x)
    elif kind == "identity":
        x = np.eye(n + 30, n)
    elif kind == "diagonal":
        x = np.eye(n + 30, n) * rng.standard_normal(n)
    elif kind == "rank":
        x = x[:, :n // 2] @ rng.standard_normal((n // 2, n))
        same = False
    elif kind == "zero_column":
        x[:, n // 2] = 0.0
        same = False
    elif kind == "graded_columns":
        x = x * np.logspace(0, -6, n)
    elif kind == "ill_conditioned":
        u, s, v = np.linalg.svd(x, full_matrices=False)
        x = (u * np.logspace(0, -9, n)) @ v
    elif kind == "tiny":
        x = x * 1e-200
    elif kind == "huge":
        x = x * 1e150
    elif kind == "overflowing":
        x = x * 1e250
    elif kind == "zero_rows":
        x[n // 2:] = 0.0
        same = False
    check(x, "D", False, same)


@pytest.mark.parametrize("lq", [False, True])
def test_huge_block_keeps_its_tiny_columns(lq):
    """Columns of 1e145 and of 1e-150 side by side: the squares of both are
    finite, so the range scaling must not flush the small ones."""
    x = np.random.default_rng(3).standard_normal((50, 20))
    x[:, ::2] *= 1e145
    x[:, 1::2] *= 1e-150
    q, r = dense_qr(x.T if lq else x, "D", lq)
    tol = 4 * 50 * EPS["D"]
    assert np.max(np.abs(q.T @ q - np.eye(20))) <= tol
    q0, r0 = np.linalg.qr(x)
    # column by column: a column of R has the length of the block's
    for c in range(20):
        size = 1e145 if c % 2 == 0 else 1e-150
        small = np.abs(r0[:, c]) <= 10 * size
        assert np.all(small)
        assert np.linalg.norm((q @ (r[:, c] / size)) - x[:, c] / size) <= tol * np.linalg.norm(x[:, c] / size)
