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


@pytest.mark.parametrize("n_tets", [1, 63, 64, 65, 190])
def test_fem_assemble_tet_groups_and_chunks(oracle, n_tets):
    """Assembly around the 64-tet groups and 32-target tiles, and a tile whose
    contributions exceed a 252-entry chunk (every tet shares two vertices).
    Bound as in the other assembly tests (two routes of the same 64-bit
    projection, 1e-11 of the largest value)."""
    from agipc_learning_amd import adjoint

    rng = np.random.default_rng(n_tets)
    n = 2 + 2 * n_tets
    tets = np.stack([np.zeros(n_tets, int), 2 + 2 * np.arange(n_tets), np.full(n_tets, 1), 3 + 2 * np.arange(n_tets)],
                    1).astype(np.int32)
    rng.permuted(tets, axis=1, out=tets)  # both orientations of every pair
    dminv = rng.standard_normal((n_tets, 9))
    vol, mu, lam = rng.uniform(0.5, 1.5, n_tets), rng.uniform(1, 2, n_tets), rng.uniform(1, 2, n_tets)
    F = np.eye(3).reshape(9) + 0.4 * rng.standard_normal((n_tets, 9))
    rows, cols = adjoint.mesh_structure(n, tets)
    base = rng.standard_normal((len(rows), 9))
    fem = native.FemHessian(tets, rows, cols)
    args = [dev(a) for a in (dminv, vol, F, mu, lam)]
    got, plain = host(fem.assemble(*args, base=dev(base))), host(fem.assemble(*args))
    A = oracle.fem_assemble_dense(n, tets, dminv, vol, F, mu, lam)
    want = np.stack([A[3 * r:3 * r + 3, 3 * c:3 * c + 3].reshape(9, order="F") for r, c in zip(rows, cols)])
    assert np.abs(plain - want).max() <= 1e-11 * np.abs(want).max()
    assert np.abs(got - base - want).max() <= 1e-11 * np.abs(want).max()


@pytest.mark.parametrize("lengths,spread", [([1], 1), ([62, 63, 64, 65], 40), ([126, 127, 128, 129, 130], 9),
                                            ([63, 126, 189, 64, 0, 0, 70], 1), ([1024, 1025, 3, 1100], 7),
                                            ([90] * 70 + [0] * 3, 25)])
def test_converter_row_lengths(oracle, lengths, spread):
    """Rows around the register sort (64 and 128 triplets), the LDS sort (1,024)
    and the 63-triplet chunks of the sums, with runs that chunks cut; bit for
    bit as the oracle (sums in input order)."""
    rng = np.random.default_rng(len(lengths) + spread)
    r = np.repeat(np.arange(len(lengths)), lengths).astype(np.int32)
    r = rng.permutation(r).astype(np.int32)
    c = rng.integers(0, min(spread, len(lengths)), len(r)).astype(np.int32)
    v = rng.standard_normal((len(r), 9))
    conv = native.Converter()
    for drop_lower in (False, True):
        got = conv.convert(dev(r), dev(c), dev(v), len(lengths), drop_lower)
        want = oracle.convert_triplets(r, c, v, drop_lower)
        for a, b in zip(got, want):
            assert np.array_equal(host(a), b)


@pytest.mark.parametrize("n_rows", [2047, 2048, 2049, 4097, 2048 * 256 + 1, 2048 * 300])
def test_converter_scan_tiles(oracle, n_rows):
    """Row counts around the prefix scan's tiles of 2,048 rows and past the 256
    tiles that one pass over their totals takes; most rows are empty, the last one
    is not.  Bit for bit as the oracle."""
    rng = np.random.default_rng(n_rows)
    n = 3 * min(n_rows, 20000)
    r = rng.integers(0, n_rows, n).astype(np.int32)
    r[:4] = n_rows - 1
    c = np.minimum(r + rng.integers(0, 3, n), n_rows - 1).astype(np.int32)
    v = rng.standard_normal((n, 9))
    got = native.Converter().convert(dev(r), dev(c), dev(v), n_rows)
    for a, b in zip(got, oracle.convert_triplets(r, c, v, False)):
        assert np.array_equal(host(a), b)


def test_converter_many_long_rows(oracle):
    """More rows past the register sort than the lists' workgroups take at
    once (47 rows a list, 40 workgroups), so a workgroup sorts several, with
    rows past the LDS sort among them; bit for bit as the oracle."""
    rng = np.random.default_rng(5)
    lengths = 129 + np.arange(3000) % 7
    lengths[[0, 1, 1500, 2990, 2999]] = 1025
    r = rng.permutation(np.repeat(np.arange(3000), lengths)).astype(np.int32)
    c = rng.integers(0, 60, len(r)).astype(np.int32)
    v = rng.standard_normal((len(r), 9))
    conv = native.Converter()
    for _ in range(2):  # the counts are cleared between calls
        got = conv.convert(dev(r), dev(c), dev(v), 3000)
        for a, b in zip(got, oracle.convert_triplets(r, c, v, False)):
            assert np.array_equal(host(a), b)


def clustered_system(n_banks, per_vertex, seed):
    """Two slots to a level-1 node except the last 32 (all of one node, every
    pair coupled); the level-1 nodes of fine banks 2j and 2j + 1 pair up, those of
    banks 0 and 1 form one level-2 node, every pair coupled.  Besides, per_vertex
    random blocks a slot, most of them near the diagonal.  Vertices in random order."""
    n, rng = 32 * n_banks, np.random.default_rng(seed)
    edges = [(v, v + 1) for v in range(0, n, 2)] + [(v, v + 1) for v in range(n - 32, n - 1)]
    for j in range(0, n_banks, 2):
        edges += [(32 * j + 2 * k, 32 * j + 32 + 2 * k) for k in range(16)]
    edges += [(2 * k, 32 + 2 * ((k + 1) % 16)) for k in range(16)]
    part_to_real = rng.permutation(n)
    e = part_to_real[np.unique(np.array(edges), axis=0)]
    e = np.concatenate([e, e[:, ::-1]])
    e = e[np.lexsort((e[:, 1], e[:, 0]))]
    num = np.bincount(e[:, 0], minlength=n)
    start = np.concatenate([[0], np.cumsum(num)[:-1]])
    r = np.repeat(np.arange(n), per_vertex)
    c = np.where(rng.random(len(r)) < 0.75, r + rng.integers(-300, 301, len(r)), rng.integers(0, n, len(r)))
    c = np.clip(c, 0, n - 1)
    dense = [np.stack(np.triu_indices(m), 1) + o for m, o in ((64, 0), (32, n - 32))]
    p = part_to_real[np.concatenate([np.stack([np.arange(n)] * 2, 1), np.stack([r, c], 1)] + dense)]
    p = np.unique(np.sort(p, axis=1), axis=0)
    p = p[rng.permutation(len(p))]
    rows, cols = p[:, 0].astype(np.int32), p[:, 1].astype(np.int32)
    vals = 0.1 * rng.standard_normal((len(p), 9))
    d = rows == cols
    m = vals[d].reshape(-1, 3, 3)
    # diagonally dominant: every row's blocks are smaller in sum than its diagonal
    load = np.bincount(rows, minlength=n) + np.bincount(cols, minlength=n)
    vals[d] = (0.5 * (m + m.transpose(0, 2, 1)) + np.eye(3) * load[rows[d], None, None]).reshape(-1, 9)
    return n, rows, cols, vals, (start, num, e[:, 1]), part_to_real, np.argsort(part_to_real)


def test_galerkin_sums_of_large_levels(oracle):
    """Coarse levels of at least 65,536 entries (the sums that pass through LDS
    32 entries at a time) from fine and from coarse sources, as they are,
    transposed and doubled, with an entry of several 252-source chunks at both and
    counts that 32 does not divide: every bank's inverse equals the oracle's, which
    forms the coarse blocks from the fine ones.  Bound as in the other inverse
    tests, 2e-5 of a bank's largest value."""
    n, rows, cols, vals, nbr, p2r, r2p = clustered_system(600, 5, 13)
    s = native.Solver()
    s.add_system(block_rows=n, rows=rows, cols=cols)
    s.set_topology(0, *nbr, p2r, r2p)
    s.setup()
    s.set_values(0, dev(vals))
    s.build("fp32")
    mas = oracle.Mas(n, n, *nbr, p2r, r2p)
    mas.reorder()
    table = mas.hierarchy()["coarse_table"]
    I, J = table[rows, 0], table[cols, 0]
    for level in (1, 2):  # entries of the level and their sources
        lo, hi = np.minimum(I, J), np.maximum(I, J)
        pair, count = np.unique(np.stack([lo, hi], 1), axis=0, return_counts=True)
        assert len(pair) >= 65536 and len(pair) % 32 and count.max() > 252 and count.mean() <= 32
        if level == 1:
            assert 0.2 < np.mean(I > J) < 0.8
            up = dict(zip(table[:, 0], table[:, 1]))
            I, J = (np.array([up[a] for a in pair[:, k]]) for k in (0, 1))
            assert (I > J).any() and ((I == J) & (pair[:, 0] != pair[:, 1])).any()
    mas.assemble(vals, rows, cols)
    mas.invert(1)
    got = s.inverse()
    want = mas.inverse().reshape(got.shape[0], -1, 3, 3).transpose(0, 1, 3, 2).reshape(got.shape)
    assert s.factor_status() == 0
    scale = np.abs(want).max(axis=(1, 2), keepdims=True)
    assert (np.abs(got - want) <= 2e-5 * scale).all()


@pytest.mark.parametrize("bank", [32, 16])
@pytest.mark.parametrize("precision", ["fp32", "fp16", "bf16"])
@pytest.mark.parametrize("n,contacts", [(2, 0), (3, 4), (9, 150)])
def test_lane_tiles_agree_with_the_block_diagonal_layout(bank, precision, n, contacts):
    """The automatic local kernel (lane tiles) and the 4-wave kernel store the
    same inverse, value for value, and apply it alike (FP32 sums in other
    orders: within 1e-5 of each other, as the other variants' test), on one
    partly filled bank, a few, and with coarse levels; the setting changes
    between builds without a new one where it always did."""
    from agipc_learning_amd import session
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(n, n_contacts=contacts, seed=3, young_sigma=0.5)
    s = native.Solver()
    s.add_system(block_rows=w["block_rows"], rows=w["rows"], cols=w["cols"], bank=bank)
    nbr = W.neighbors(w["n_vertices"], w["tets"])
    s.set_topology_morton(0, *nbr, w["positions"])
    if contacts:
        s.set_contacts(0, w["pairs"])
    s.setup()
    s.set_values(0, dev(w["vals"]))
    s.build(precision)
    r = dev(np.random.default_rng(n).standard_normal(3 * w["block_rows"]))
    zs, invs = [], []
    for waves in (0, 4, 0, 8):
        s.set_mas_waves(waves)
        z = torch.zeros_like(r)
        s.apply_preconditioner(r, z)
        zs.append(host(z))
        invs.append(s.inverse())
    assert np.array_equal(invs[0], invs[1]) and np.array_equal(invs[0], invs[2])
    assert np.array_equal(zs[0], zs[2])
    for z in zs[1:]:
        assert np.linalg.norm(z - zs[0]) <= 1e-5 * np.linalg.norm(zs[0])
    if n == 9 or precision == "fp32":  # a 27-vertex inverse in 16 bits need not be positive definite
        s.set_mas_waves(0)
        b = dev(session.rhs_of(w))
        st = s.solve(b, torch.zeros_like(b), max_iter=200)[0]
        assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6)


@pytest.mark.parametrize("bank,precision", [(32, "fp32"), (32, "fp16"), (16, "fp32"), (16, "bf16")])
def test_inverse_is_read_in_the_layout_it_was_built_in(bank, precision):
    """New values ask for a build, and another local kernel set before it does
    not change how the inverses held are read (each kernel stores them in a
    layout of its own); set with a build in place, it builds them again from
    the same values."""
    from agipc_learning_amd import session
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(9, n_contacts=150, seed=3, young_sigma=0.5)
    s = session.solver_for(w, bank=bank)
    s.build(precision)
    inv = s.inverse()
    s.set_mas_waves(8)
    assert np.array_equal(s.inverse(), inv)
    s.set_mas_waves(0)
    s.set_values(0, dev(3.0 * w["vals"]))
    for waves in (4, 0, 8, 1):
        s.set_mas_waves(waves)
        assert np.array_equal(s.inverse(), inv), waves
    r = dev(np.ones(3 * w["block_rows"]))
    with pytest.raises(RuntimeError, match="build"):
        s.apply_preconditioner(r, torch.zeros_like(r))
    s.build(precision)
    assert not np.array_equal(s.inverse(), inv)


@pytest.mark.parametrize("bank,precision", [(32, "fp32"), (32, "fp16"), (16, "fp32"), (16, "bf16")])
def test_autotune_says_which_local_kernel_runs(bank, precision):
    """After the autotuner the solver is built and applies, bit for bit, as one
    set to the variant reported as used: the reported fastest or the automatic
    kernel, whatever was set before."""
    from agipc_learning_amd import session
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(9, n_contacts=150, seed=3, young_sigma=0.5)
    r = dev(np.random.default_rng(2).standard_normal(3 * w["block_rows"]))

    def applied(s):
        z = torch.zeros_like(r)
        s.apply_preconditioner(r, z)
        return host(z)

    for before in (0, 4, 8, 1):
        s = session.solver_for(w, bank=bank)
        s.set_mas_waves(before)
        s.build(precision)
        if before == 0:
            assert s.mas_waves_used() == 0
        best = s.autotune_mas(3)
        assert best["used"] == s.mas_waves_used() and best["used"] in (0, best["waves"])
        other = session.solver_for(w, bank=bank)
        other.set_mas_waves(best["used"])
        other.build(precision)
        assert other.mas_waves_used() == best["used"]
        assert np.array_equal(applied(s), applied(other))


def mas_object(w, m=None, levels=0):
    """A preconditioner object of the mesh of w (or m given that mesh)."""
    from agipc_learning_amd import workloads as W

    p2r, r2p = native.morton_partition(w["positions"])
    start, num, lst = W.neighbors(w["n_vertices"], w["tets"])
    m = native.MasPreconditioner(32) if m is None else m
    m.init_neighbor(w["n_vertices"], 0, len(lst), len(p2r))
    m.upload(lst, start, num, p2r, r2p)
    m.init_matrix(levels)
    return m


def test_mas_object_sees_a_structure_of_the_same_size():
    """A call with as many blocks and pairs as the last but another order of
    blocks, or other pairs, is not taken for the same structure: its apply
    equals a fresh object's bit for bit.  The selection may be null."""
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(9, n_contacts=120, seed=4, young_sigma=0.5)
    nv, nb = w["n_vertices"], len(w["rows"])
    rng = np.random.default_rng(8)
    R = dev(rng.standard_normal(3 * nv))

    def fresh():
        return mas_object(w)

    def apply(m, order, pairs, select=True):
        idx = dev(order.astype(np.int32)) if select else None
        vals, rows, cols = (w["vals"], w["rows"], w["cols"]) if select else (w["vals"][order], w["rows"][order], w["cols"][order])
        p = dev(np.ascontiguousarray(pairs, np.int32))
        m.set_preconditioner_bcoo(dev(vals), dev(rows), dev(cols), idx, 0, nb, pairs=p, cp_num=len(pairs))
        Z = torch.zeros_like(R)
        m.preconditioning(R, Z)
        return host(Z)

    plain, mixed = np.arange(nb), rng.permutation(nb)
    other = np.roll(np.asarray(w["pairs"]).reshape(-1, 4), 7, axis=1)
    other = (other + 13) % nv
    m = fresh()
    steps = [(plain, w["pairs"], True), (mixed, w["pairs"], True), (mixed, w["pairs"], False), (mixed, other, True),
             (plain, w["pairs"], True)]
    for order, pairs, select in steps:
        for _ in range(2):  # the second call keeps the structure
            assert np.array_equal(apply(m, order, pairs, select), apply(fresh(), order, pairs, select))
    with pytest.raises(RuntimeError):
        m.set_preconditioner_bcoo(dev(w["vals"]), dev(w["rows"]), dev(w["cols"]), dev(plain.astype(np.int32)), 1, nb,
                                  pairs=dev(np.asarray(w["pairs"], np.int32)), cp_num=len(w["pairs"]))


def test_mas_object_refuses_a_selection_outside_the_matrix():
    """After an accepted call, a call of the same counts whose indices, or whose
    count of indices or pairs, lead past the caller's arrays is refused on the
    host before anything reads there, and leaves the object as it was."""
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(9, n_contacts=120, seed=4, young_sigma=0.5)
    nv, nb = w["n_vertices"], len(w["rows"])
    vals, rows, cols, idx = dev(w["vals"]), dev(w["rows"]), dev(w["cols"]), dev(np.arange(nb, dtype=np.int32))
    # more pairs than a small tensor's allocation (2 MiB at most) can hold
    many = dev(np.tile(np.asarray(w["pairs"], np.int32).reshape(-1, 4), (1700, 1)))
    R = dev(np.random.default_rng(8).standard_normal(3 * nv))
    m = mas_object(w)
    m.set_preconditioner_bcoo(vals, rows, cols, idx, 0, nb, pairs=many, cp_num=len(many))
    want = torch.zeros_like(R)
    m.preconditioning(R, want)
    far = idx.clone()
    far[nb // 2] = 1 << 27
    with pytest.raises(RuntimeError, match="outside the matrix"):
        m.set_preconditioner_bcoo(vals, rows, cols, far, 0, nb, pairs=many, cp_num=len(many))
    with pytest.raises(RuntimeError, match="fewer contact pairs"):
        m.set_preconditioner_bcoo(vals, rows, cols, idx, 0, nb, pairs=many[:4].clone(), cp_num=len(many))
    with pytest.raises(RuntimeError, match="fewer indices"):
        m.set_preconditioner_bcoo(vals, rows, cols, idx, 0, 1 << 27, pairs=many, cp_num=len(many))
    got = torch.zeros_like(R)
    m.preconditioning(R, got)
    assert np.array_equal(host(got), host(want))
    m.set_preconditioner_bcoo(vals, rows, cols, idx, 0, nb, pairs=many, cp_num=len(many))
    m.preconditioning(R, got)
    assert np.array_equal(host(got), host(want))


@pytest.mark.parametrize("cp_num", [1 << 29, 1 << 30, 2**31 - 1])
def test_mas_object_counts_pairs_in_64_bits(cp_num):
    """Pair counts whose four indices a pair pass 2^31 are refused for an array
    that cannot hold them (in 32 bits 2^30 pairs count as none)."""
    from agipc_learning_amd import workloads as W

    w = W.fem_grid(4, n_contacts=10, seed=4, young_sigma=0.5)
    nb = len(w["rows"])
    m = mas_object(w)
    with pytest.raises(RuntimeError, match="fewer contact pairs"):
        m.set_preconditioner_bcoo(dev(w["vals"]), dev(w["rows"]), dev(w["cols"]), dev(np.arange(nb, dtype=np.int32)),
                                  0, nb, pairs=dev(np.asarray(w["pairs"], np.int32)), cp_num=cp_num)


def test_mas_object_takes_another_mesh():
    """One object given another partition, another level count, a smaller and
    a larger mesh applies as a fresh object does, bit for bit, and asks for the
    matrix before it applies anything; the same mesh again keeps its solver."""
    from agipc_learning_amd import workloads as W

    def matrix(m, w):
        nb = len(w["rows"])
        m.set_preconditioner_bcoo(dev(w["vals"]), dev(w["rows"]), dev(w["cols"]), dev(np.arange(nb, dtype=np.int32)),
                                  0, nb)

    def applied(m, w):
        R = dev(np.random.default_rng(3).standard_normal(3 * w["n_vertices"]))
        Z = torch.zeros_like(R)
        m.preconditioning(R, Z)
        return host(Z)

    w = W.fem_grid(9, seed=4, young_sigma=0.5)
    turned = dict(w, positions=np.ascontiguousarray(w["positions"][:, ::-1]) * [1.0, -2.0, 0.5])
    m = None
    for mesh, levels in ((w, 0), (turned, 0), (turned, 2), (W.fem_grid(5, seed=4), 0), (w, 0)):
        m = mas_object(mesh, m, levels)
        with pytest.raises(RuntimeError, match="set_preconditioner_bcoo must come first"):
            applied(m, mesh)
        matrix(m, mesh)
        fresh = mas_object(mesh, None, levels)
        matrix(fresh, mesh)
        got, want = applied(m, mesh), applied(fresh, mesh)
        assert np.array_equal(got, want)
        kept = m.L.masx_mas_solver(m.h)
        mas_object(mesh, m, levels)
        assert m.L.masx_mas_solver(m.h) == kept and np.array_equal(applied(m, mesh), want)
    small = W.fem_grid(5, seed=4)
    m.init_neighbor(small["n_vertices"], 0, 0, (small["n_vertices"] + 31) // 32 * 32)
    with pytest.raises(RuntimeError, match="upload must come first"):  # the arrays held are the other mesh's
        m.init_matrix()
    with pytest.raises(RuntimeError, match="init_matrix must come first"):
        matrix(m, small)


@pytest.mark.parametrize("sizes,per_row,hub", [((1,), 0, 0), ((256, 257), 0, 0), ((33100, 40), 0, 0), ((129, 127), 2, 90),
                                               ((700,), 24, 600), ((35000,), 2, 300)])
def test_device_structure_around_tile_ends(sizes, per_row, hub):
    """The device's SpMV tiles, entry lists and Galerkin maps equal the host's:
    tiles that end at 256 rows, at a system's end and at the entry cap, a chain
    of tiles longer than one staged window and than one of its segments, rows
    whose columns do not fit the staged ones, and a row of more than a tile."""
    rng = np.random.default_rng(sum(sizes) + hub)
    systems = [(n,) + random_structure(n, per_row, min(hub, n), rng) + (rng.random((n, 3)),) for n in sizes]
    solvers = []
    for on_device in (0, 1):
        s = native.Solver()
        for n, rows, cols, pos in systems:
            i = s.add_system(block_rows=n, rows=rows, cols=cols)
            s.set_topology_morton(i, np.zeros(n), np.zeros(n), [], pos)
        if not on_device:
            s.set_device_structure(0)
        s.setup()
        assert s.device_structure_used() == bool(on_device)
        solvers.append(s)
    want, got = solvers
    for entries in (2, 4, 8):
        for s in solvers:
            s.set_spmv_tiling(entries)
        for name in native.Solver.PLAN_ARRAYS:
            assert np.array_equal(want.plan_array(name), got.plan_array(name)), (entries, name)


@pytest.mark.parametrize("n", [1, 63, 65, 511, 513, 2047, 2049, 131072, 140000])
def test_device_morton_around_rounds_and_chunks(n):
    """The device partition equals the host's where waves, tiles and the scan's
    kept counts (64 tiles) end, with many equal codes (their order is the index order)."""
    rng = np.random.default_rng(n)
    pos = rng.integers(0, 9, (n, 3)).astype(np.float64)
    p2r, r2p = native.DeviceMorton().partition(dev(pos))
    want_p2r, want_r2p = native.morton_partition(pos)
    assert np.array_equal(host(p2r), want_p2r) and np.array_equal(host(r2p), want_r2p)
