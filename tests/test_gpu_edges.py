"""Kernels at the edges of their tiles and chunks, against the oracle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from agipc_learning_amd import native  # noqa: E402

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def random_structure(n, per_row, hub, rng):
    """Upper structure: every diagonal block, about per_row others a row, and row 0 coupled to `hub` rows."""
    r = np.repeat(np.arange(n), per_row)
    c = rng.integers(0, n, len(r))
    pairs = np.concatenate([np.stack([np.arange(n)] * 2, 1), np.stack([np.minimum(r, c), np.maximum(r, c)], 1),
                            np.stack([np.zeros(hub, int), np.arange(hub)], 1)])
    pairs = np.unique(pairs, axis=0)
    return pairs[:, 0].astype(np.int32), pairs[:, 1].astype(np.int32)


@pytest.mark.parametrize("n,per_row,hub", [(1, 0, 0), (63, 3, 0), (64, 3, 0), (65, 9, 0), (340, 1, 340),
                                           (1100, 2, 1019), (1100, 2, 1100), (2300, 8, 2300)])
def test_spmv64_row_tiles_and_chunks(oracle, n, per_row, hub):
    """y = a A x + b y around the 64-row tiles and the 1,020-entry chunks (a
    tile of several chunks, a row of more than one), and x as its own output.
    Bound: each sum of m products errs by at most about m eps of the sum of
    magnitudes; m <= 3 (n + 1) here, and the result is compared in norm."""
    rng = np.random.default_rng(n + hub)
    rows, cols = random_structure(n, per_row, hub, rng)
    vals = rng.standard_normal((len(rows), 9))
    s = native.Solver()
    s.add_system(block_rows=n, rows=rows, cols=cols, use_mas=False, global_diag=True)
    s.setup()
    s.set_values(0, dev(vals))
    x, y = rng.standard_normal(3 * n), rng.standard_normal(3 * n)
    for a, b in ((1.0, 0.0), (-0.75, 1.5)):
        want = oracle.sym_spmv(vals, rows, cols, x, a, b, y)
        got = dev(y)
        s.spmv(dev(x), got, a=a, b=b)
        assert np.linalg.norm(host(got) - want) <= 1e-13 * np.linalg.norm(want)
    want = oracle.sym_spmv(vals, rows, cols, x)
    own = dev(x)
    s.spmv(own, own)
    assert np.linalg.norm(host(own) - want) <= 1e-13 * np.linalg.norm(want)
