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
