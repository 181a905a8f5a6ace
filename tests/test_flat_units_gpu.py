"""Permute and fill launches at the edges of their chunks (2048 elements, one
workgroup) and units (the rest of a task, 512 per wave) against numpy.  Copies are exact, so results must be equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["D", "S"])
@pytest.mark.parametrize("shape", [(1, 1), (3, 21), (8, 8), (5, 13), (7, 73), (16, 32), (27, 19), (89, 23), (2, 1024, 1),
                                   (683, 3), (1449, 1449), (5, 29, 14465), (4099, 4097)])
def test_transpose_equals_numpy(shape, dtype):
    from tnsp_amd import TAT

    names = ["a", "b", "c"][:len(shape)]
    t = getattr(TAT.No, dtype).Tensor(names, list(shape))
    x = np.arange(int(np.prod(shape))).astype(np.float64 if dtype == "D" else np.float32)
    t.storage = x
    order = names[::-1]
    got = t.transpose(order).storage.numpy()
    ref = x.reshape(shape).transpose(*range(len(shape))[::-1]).reshape(-1)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("n", [1, 9, 23, 64])
def test_many_blocks_with_signs_equal_oracle(n):
    """Many tasks of different sizes in one launch, fermion signs included."""
    from helpers import to_gpu
    from oracle import tat

    K = tat.FermiU1
    segs = [[(q, d) for q, d in ((-1, 1 + (n + i) % 3), (0, 1 + n // (i + 1)), (1, 2))] for i in range(4)]
    t = tat.Tensor(K, ["i", "j", "k", "l"], [(s, bool(i % 2)) for i, s in enumerate(segs)])
    t.data[:] = np.random.default_rng(n).standard_normal(t.size)
    ref = t.transpose(["l", "j", "i", "k"]).data
    assert np.array_equal(to_gpu(t).transpose(["l", "j", "i", "k"]).storage.numpy(), ref)


@pytest.mark.parametrize("m,n", [(1, 1), (7, 9), (8, 64), (57, 9), (64, 32), (45, 47)])
def test_unmatched_sector_is_zero(m, n):
    """A sector the contraction leaves without a partner is filled with zeros."""
    from tnsp_amd import TAT

    a = TAT.BoseU1.D.Tensor(["i", "k"], [[(0, 3), (5, m)], [(0, 2)]])
    b = TAT.BoseU1.D.Tensor(["k", "j"], [[(0, 2)], [(0, 4), (-5, n)]])
    a.storage = np.ones(a.storage.size)
    b.storage = np.ones(b.storage.size)
    c = a.contract(b, {("k", "k")})
    assert np.array_equal(c.blocks[[("i", 5), ("j", -5)]], np.zeros((m, n)))
    assert np.array_equal(c.blocks[[("i", 0), ("j", 0)]], np.full((3, 4), 2.0))
