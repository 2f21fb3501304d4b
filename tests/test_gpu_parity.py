"""GPU parity: the HIP path through the C ABI against the CPU oracle.

Tolerances (floating point): the FP64 SpMV entry point matches to 1e-10
absolute on the reference KAT (the reference's own gate) and 1e-12 relative
elsewhere; the FP32 MAS apply matches the oracle's FP64 apply of the same
FP32-rounded inverse to 1e-4 relative (FP32 restriction/prolongation
arithmetic); PCG iteration counts are within 5% (at least +-1) of the oracle's
and the FP64 true relative residual meets the tolerance.  Integer work
(hierarchy) is compared bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from agipc_learning_amd import native
from agipc_learning_amd import session
from agipc_learning_amd import workloads as W
from chain_fixture import REFERENCE_ITERATIONS, padded_chain
from test_oracle import dense_sym, spmv_kat_system

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def oracle_mas(oracle, w, bank=32, levels=0, method=1):
    nv = w["n_vertices"]
    p2r, r2p = oracle.morton_partition(w["positions"], bank)
    st, nu, li = oracle.mesh_neighbors(nv, w["tets"])
    mas = oracle.Mas(nv, len(p2r), st, nu, li, p2r, r2p, bank=bank, levels=levels)
    mas.reorder(w["pairs"])
    fem = (w["rows"] >= w["fem_offset"]) & (w["cols"] >= w["fem_offset"])
    mas.assemble(w["vals"], w["rows"], w["cols"], indices=np.nonzero(fem)[0].astype(np.uint32),
                 offset=w["fem_offset"])
    mas.invert(method)
    return mas


def iters_close(a, b):
    return abs(a - b) <= max(1, int(0.05 * b + 0.5))


# ------------------------------------------------------------------ SpMV ----

def test_spmv64_reference_kat():
    vals, rows, cols, x, y0 = spmv_kat_system()
    s = native.Solver()
    s.add_system(block_rows=20, rows=rows, cols=cols, use_mas=False)
    s.setup()
    s.set_values(0, dev(vals))
    y = dev(y0)
    s.spmv(dev(x), y, a=1.25, b=-0.5)
    want = 1.25 * dense_sym(vals, rows, cols, 20) @ x - 0.5 * y0
    assert np.max(np.abs(host(y) - want)) <= 1e-10


def test_spmv64_grid_with_contacts(oracle):
    w = W.fem_grid(10, n_contacts=200, seed=3, young_sigma=0.5)
    s = session.solver_for(w)
    x = np.random.default_rng(0).standard_normal(3 * w["block_rows"])
    y = torch.zeros(3 * w["block_rows"], dtype=torch.float64, device="cuda")
    s.spmv(dev(x), y)
    want = oracle.sym_spmv(w["vals"], w["rows"], w["cols"], x)
    np.testing.assert_allclose(host(y), want, rtol=1e-12, atol=1e-12 * np.abs(want).max())


# ------------------------------------------------------------- hierarchy ----

def test_device_solver_hierarchy_equals_oracle(oracle):
    w = W.fem_grid(12, n_contacts=300, seed=1)
    s = session.solver_for(w)
    mas = oracle_mas(oracle, w)
    h, o = s.hierarchy(0), mas.hierarchy()
    assert h["total"] == mas.total_clusters
    assert np.array_equal(h["coarse_table"], o["coarse_table"])
    assert np.array_equal(h["fine_mask"], o["fine_mask"])


def test_new_contact_set_on_the_same_solver_is_reanalyzed(oracle):
    # contacts set after set-up mark the structure for re-analysis: the next
    # setup() rebuilds the hierarchy (on the device) with the new pairs, and
    # the solve on the rebuilt preconditioner converges
    w = W.fem_grid(10, n_contacts=0, seed=4, young_sigma=0.5)
    s = session.solver_for(w)
    rng = np.random.default_rng(3)
    pairs = np.sort(rng.choice(w["n_vertices"], size=(200, 4), replace=True), axis=1).astype(np.int32)
    pairs = pairs[(pairs[:, 0] != pairs[:, 1]) & (pairs[:, 1] != pairs[:, 2]) & (pairs[:, 2] != pairs[:, 3])]
    for contact_set in (pairs, pairs[:50]):
        s.set_contacts(0, contact_set)
        s.setup()
        s.set_values(0, dev(w["vals"]))
        s.build("fp32")
        wo = dict(w, pairs=contact_set)
        mas = oracle_mas(oracle, wo)
        h, o = s.hierarchy(0), mas.hierarchy()
        assert h["total"] == mas.total_clusters
        assert np.array_equal(h["coarse_table"], o["coarse_table"])
        assert np.array_equal(h["fine_mask"], o["fine_mask"])
        b = session.rhs_of(w)
        x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
        st = s.solve(dev(b), x, rule=1, tol=1e-4)[0]
        assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6)


def test_set_structure_on_the_same_solver_equals_a_fresh_solver():
    # a Newton step with a new contact set changes the upper structure: the
    # same solver takes it (masx_set_structure + contacts + setup, buffers
    # reused) and solves exactly as a solver built for it from scratch; then
    # back to the first structure (smaller), reusing the larger buffers
    w1 = W.fem_grid(10, n_contacts=100, seed=11, young_sigma=0.5)
    w2 = W.fem_grid(10, n_contacts=400, seed=12, young_sigma=0.5)
    assert len(w1["rows"]) != len(w2["rows"])

    def solve_with(s, w):
        s.set_values(0, dev(w["vals"]))
        s.build("fp32")
        b = session.rhs_of(w)
        x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
        st = s.solve(dev(b), x, rule=1, tol=1e-4)[0]
        torch.cuda.synchronize()
        return x.cpu().numpy(), st["iterations"]

    s = session.solver_for(w1)
    first = solve_with(s, w1)
    for w in (w2, w1):
        s.set_structure(0, w["rows"], w["cols"])
        s.set_contacts(0, w["pairs"])
        s.setup()
        got = solve_with(s, w)
        fresh = session.solver_for(w)
        ref = solve_with(fresh, w)
        fresh.close()
        assert got[1] == ref[1]
        assert np.array_equal(got[0], ref[0])
    assert np.array_equal(got[0], first[0])


# ------------------------------------------------------------------- MAS ----

@pytest.mark.parametrize("factor_waves", [1, 2])
@pytest.mark.parametrize("n,contacts", [(8, 0), (14, 400)])
def test_mas_inverse_and_apply_parity(oracle, n, contacts, factor_waves):
    """Both MAS factor kernels (one or two waves per bank) invert every bank
    to the oracle's inverse."""
    w = W.fem_grid(n, n_contacts=contacts, seed=n, young_sigma=0.5)
    s = session.solver_for(w)
    s.set_factor_waves(factor_waves)
    s.build("fp32")
    assert s.factor_status() == 0
    mas = oracle_mas(oracle, w)
    inv_gpu = s.inverse()                              # block row-major
    inv_orc = mas.inverse().reshape(inv_gpu.shape[0], -1, 3, 3).transpose(0, 1, 3, 2).reshape(inv_gpu.shape)
    scale = np.abs(inv_orc).max()
    assert np.max(np.abs(inv_gpu - inv_orc)) <= 2e-5 * scale
    r = np.random.default_rng(5).standard_normal(3 * w["block_rows"])
    z = torch.zeros_like(dev(r))
    s.apply_preconditioner(dev(r), z)
    want = mas.apply(r)
    got = host(z)
    assert np.linalg.norm(got - want) <= 1e-4 * np.linalg.norm(want)


@pytest.mark.parametrize("factor_waves", [1, 2])
def test_mas_bank16_apply_parity(oracle, factor_waves):
    w = W.fem_grid(9, n_contacts=50, seed=2)
    s = session.solver_for(w, bank=16)
    s.set_factor_waves(factor_waves)
    s.build("fp32")
    mas = oracle_mas(oracle, w, bank=16)
    r = np.random.default_rng(1).standard_normal(3 * w["block_rows"])
    z = torch.zeros_like(dev(r))
    s.apply_preconditioner(dev(r), z)
    want = mas.apply(r)
    assert np.linalg.norm(host(z) - want) <= 1e-4 * np.linalg.norm(want)


# ------------------------------------------------------------------- PCG ----

@pytest.mark.parametrize("n,contacts,rule", [(8, 0, 1), (8, 0, 0), (16, 600, 1), (16, 600, 0)])
def test_solve_parity_with_oracle(oracle, n, contacts, rule):
    w = W.fem_grid(n, n_contacts=contacts, seed=n, young_sigma=0.5 if contacts else 0.0)
    s = session.solver_for(w)
    s.build("fp32")
    b = session.rhs_of(w)
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    st = s.solve(dev(b), x, rule=rule, tol=1e-4)[0]
    mas = oracle_mas(oracle, w)
    xo, so = oracle.pcg(w["block_rows"], w["vals"], w["rows"], w["cols"], b, mas=mas, tol=1e-4, rule=rule)
    assert st["failure"] == 0 and st["status"] == 1
    assert iters_close(st["iterations"], so["iterations"]), (st, so)
    if rule == 1:
        assert st["rel_res_true"] <= 1e-4 * (1 + 1e-6)
        xr = host(x)
        assert np.linalg.norm(xr - xo) <= 1e-3 * np.linalg.norm(xo)
    else:
        assert abs(st["rel_res_true"] - so["true_rel_res"]) <= 0.05 * so["true_rel_res"]


def test_chain_reference_counts_on_gpu():
    d = padded_chain()
    rows, cols = d["rows"], d["cols"]
    # MAS32 over the identity partition, as the replay harness sets it up
    s = native.Solver()
    s.add_system(block_rows=d["n"], rows=rows, cols=cols, use_mas=True)
    s.set_topology(0, d["start"], d["num"], d["list"], d["part_to_real"], d["real_to_part"])
    s.setup()
    s.set_values(0, dev(d["vals"]))
    s.build("fp32")
    x = torch.zeros(3 * d["n"], dtype=torch.float64, device="cuda")
    st = s.solve(dev(d["rhs"]), x, rule=1, tol=1e-3, max_iter=512)[0]
    assert st["iterations"] == REFERENCE_ITERATIONS["mas32"], st
    # block-Jacobi
    j = native.Solver()
    j.add_system(block_rows=d["n"], rows=rows, cols=cols, use_mas=False, global_diag=True)
    j.setup()
    j.set_values(0, dev(d["vals"]))
    j.build("fp32")
    st = j.solve(dev(d["rhs"]), x, rule=1, tol=1e-3, max_iter=512)[0]
    assert st["iterations"] == REFERENCE_ITERATIONS["jacobi"], st


def test_hybrid_abd_fem_parity(oracle):
    w = W.hybrid(seed=4, n_bodies=60, n_body_pairs=400, fem_n=7, n_coupled=12)
    s = session.solver_for(w)
    s.build("fp32")
    b = session.rhs_of(w)
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    st = s.solve(dev(b), x, rule=1, tol=1e-4)[0]
    mas = oracle_mas(oracle, w)
    abd = oracle.abd_block_inverse(w["n_bodies"], w["vals"], w["rows"], w["cols"])
    xo, so = oracle.pcg(w["block_rows"], w["vals"], w["rows"], w["cols"], b, n_abd=w["n_bodies"], abd_inv=abd,
                        mas=mas, fem_offset=w["fem_offset"], tol=1e-4, rule=1)
    assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6)
    assert iters_close(st["iterations"], so["iterations"]), (st, so)


def test_set_values_many_equals_per_system_values():
    """masx_set_values_many (all systems in one call, on a stream) puts the
    same values in place as one masx_set_values per system: after the
    values are overwritten, it restores them and the solve is bit-identical."""
    ws = [W.fem_grid(n, n_contacts=c, seed=n, young_sigma=0.5) for n, c in ((6, 20), (9, 0), (7, 40))]
    s = session.solver_for(ws)
    vals = {i: dev(w["vals"]) for i, w in enumerate(ws)}
    b = dev(session.rhs_of(ws))

    def solve():
        s.build("fp32")
        x = torch.zeros_like(b)
        st = s.solve(b, x, rule=1, tol=1e-6)
        return [q["iterations"] for q in st], host(x)

    ref = solve()
    for i, v in vals.items():
        s.set_values(i, 2.0 * v)
    stream = torch.cuda.Stream()
    s.set_values_many(vals, stream=stream.cuda_stream)
    got = solve()
    assert got[0] == ref[0]
    assert np.array_equal(got[1], ref[1])
    with pytest.raises(ValueError):
        s.set_values_many({0: vals[1]})  # wrong length for system 0


def test_set_values_many_beyond_one_launch():
    """70 systems: more than one copy launch takes (64 arrays each); the
    values in place equal per-system copies, seen through a bit-identical
    solve of every system."""
    ws = [W.fem_grid(3 + i % 3, n_contacts=0, seed=i, young_sigma=0.5) for i in range(70)]
    s = session.solver_for(ws)
    vals = {i: dev(w["vals"]) for i, w in enumerate(ws)}
    b = dev(session.rhs_of(ws))

    def solve():
        s.build("fp32")
        x = torch.zeros_like(b)
        st = s.solve(b, x, rule=1, tol=1e-6)
        return [q["iterations"] for q in st], host(x)

    ref = solve()
    for i, v in vals.items():
        s.set_values(i, 0.5 * v)
    s.set_values_many(vals)
    got = solve()
    assert got[0] == ref[0]
    assert np.array_equal(got[1], ref[1])


def test_batched_equals_individual():
    ws = [W.fem_grid(n, n_contacts=c, seed=n, young_sigma=0.5) for n, c in ((6, 20), (11, 150), (9, 0))]
    batch = session.solver_for(ws)
    batch.build("fp32")
    b = session.rhs_of(ws)
    xb = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    stb = batch.solve(dev(b), xb, rule=1, tol=1e-4)
    off = 0
    for i, w in enumerate(ws):
        s = session.solver_for(w)
        s.build("fp32")
        xi = torch.zeros(3 * w["block_rows"], dtype=torch.float64, device="cuda")
        st = s.solve(dev(w["rhs"]), xi, rule=1, tol=1e-4)[0]
        assert st["iterations"] == stb[i]["iterations"]
        n = 3 * w["block_rows"]
        assert np.array_equal(host(xi), host(xb)[off:off + n])
        off += n


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
def test_mixed_precision_converges(precision):
    w = W.fem_grid(16, n_contacts=600, seed=16, young_sigma=0.5)
    s = session.solver_for(w)
    b = session.rhs_of(w)
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    s.build("fp32")
    ref = s.solve(dev(b), x, rule=1, tol=1e-4)[0]
    s.build(precision)
    st = s.solve(dev(b), x, rule=1, tol=1e-4)[0]
    assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6)
    assert st["iterations"] <= 1.5 * ref["iterations"] + 2


def half_ulp(y, precision):
    """Spacing of the FP16 / BF16 grid at |y| (subnormal FP16 spacing below 2^-14)."""
    a = np.abs(np.asarray(y, np.float64))
    if precision == "fp16":
        return 2.0 ** (np.floor(np.log2(np.maximum(a, 2.0 ** -14))) - 10)
    return 2.0 ** (np.floor(np.log2(np.maximum(a, 2.0 ** -126))) - 7)


@pytest.mark.parametrize("factor_waves,local", [(2, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("precision", ["fp16", "bf16"])
def test_half_inverse_and_apply_match_the_oracle(oracle, precision, factor_waves, local):
    """Each bank's inverse is stored as half(v / s) with s its largest entry in
    magnitude: every stored value lies within one half-precision ulp (at the
    bank scale) of the oracle's inverse, and the half apply (FP32
    accumulation) matches an FP64 apply of that stored inverse to 1e-4.  Both
    MAS factor kernels, in the block-diagonal layout and (local = 1) the MFMA
    local kernel's tile layout."""
    w = W.fem_grid(14, n_contacts=400, seed=14, young_sigma=0.5)
    s = session.solver_for(w)
    s.set_factor_waves(factor_waves)
    s.set_mas_waves(local)
    s.build(precision)
    assert s.factor_status() == 0
    mas = oracle_mas(oracle, w)
    got = s.inverse().astype(np.float64)  # banks x blocks x 9, block row-major
    nbk, nblk = got.shape[0], got.shape[1]
    ref = mas.inverse().reshape(nbk, nblk, 3, 3).transpose(0, 1, 3, 2).reshape(got.shape).astype(np.float64)
    scale = np.abs(ref).reshape(nbk, -1).max(axis=1)[:, None, None]
    tol = half_ulp(ref / scale, precision) * scale
    bad = np.abs(got - ref) > tol
    assert not bad.any(), (int(bad.sum()), float(np.abs(got - ref)[bad].max()))
    mas.set_inverse(got.reshape(nbk, nblk, 3, 3).transpose(0, 1, 3, 2).reshape(nbk, nblk, 9).astype(np.float32))
    r = np.random.default_rng(6).standard_normal(3 * w["block_rows"])
    z = torch.zeros_like(dev(r))
    s.apply_preconditioner(dev(r), z)
    want = mas.apply(r)
    assert np.linalg.norm(host(z) - want) <= 1e-4 * np.linalg.norm(want)


def test_graph_and_eager_agree_and_are_deterministic():
    w = W.fem_grid(12, n_contacts=200, seed=7, young_sigma=0.5)
    s = session.solver_for(w)
    s.build("fp32")
    b = dev(session.rhs_of(w))
    xs = []
    for use_graph in (True, True, False):
        x = torch.zeros_like(b)
        s.solve(b, x, rule=1, tol=1e-4, use_graph=use_graph)
        xs.append(host(x))
    assert np.array_equal(xs[0], xs[1]) and np.array_equal(xs[0], xs[2])


def test_zero_rhs_returns_zero():
    w = W.fem_grid(5)
    s = session.solver_for(w)
    s.build("fp32")
    b = torch.zeros(3 * w["block_rows"], dtype=torch.float64, device="cuda")
    x = torch.ones_like(b)
    st = s.solve(b, x, rule=1)[0]
    assert st["iterations"] == 0 and float(x.abs().max()) == 0.0


def test_mas_object_api_matches_oracle(oracle):
    """TraditionalMAS32Preconditioner-shaped calls on the FEM subset of a
    hybrid matrix (indices + block offset, as LocalPreconditioner passes them)."""
    w = W.hybrid(seed=9, n_bodies=20, n_body_pairs=50, fem_n=6, n_coupled=5)
    nv, foff = w["n_vertices"], w["fem_offset"]
    p2r, r2p = oracle.morton_partition(w["positions"])
    st, nu, li = oracle.mesh_neighbors(nv, w["tets"])
    m = native.MasPreconditioner(32)
    m.init_neighbor(nv, foff, len(li), len(p2r))
    m.upload(li, st, nu, p2r, r2p)
    m.init_matrix()
    fem = np.nonzero((w["rows"] >= foff) & (w["cols"] >= foff))[0].astype(np.int32)
    vals = dev(w["vals"])
    rows = torch.from_numpy(w["rows"]).cuda()
    cols = torch.from_numpy(w["cols"]).cuda()
    idx = torch.from_numpy(fem).cuda()
    m.set_preconditioner_bcoo(vals, rows, cols, idx, foff, len(fem))
    mas = oracle_mas(oracle, w)
    R = np.random.default_rng(3).standard_normal(3 * nv)
    Z = torch.zeros(3 * nv, dtype=torch.float64, device="cuda")
    m.preconditioning(dev(R), Z)
    want = mas.apply(R)
    assert np.linalg.norm(host(Z) - want) <= 1e-4 * np.linalg.norm(want)


TILINGS = [2, 4, 8]


def test_spmv_tilings_agree_and_autotune():
    """Every SpMV tiling (entries per thread) gives the same solve."""
    w = W.fem_grid(10, n_contacts=600, seed=5)
    s = session.solver_for(w)
    s.build("fp32")
    b = dev(session.rhs_of(w))
    ref = None
    for t in TILINGS:
        s.set_spmv_tiling(t)
        x = torch.zeros_like(b)
        st = s.solve(b, x, rule=1, tol=1e-6)[0]
        assert st["failure"] == 0 and st["rel_res_true"] <= 1e-6 * (1 + 1e-6), (t, st)
        if ref is None:
            ref = (st["iterations"], host(x))
        else:
            assert abs(st["iterations"] - ref[0]) <= 1, (t, st["iterations"], ref[0])
            assert np.linalg.norm(host(x) - ref[1]) <= 1e-5 * np.linalg.norm(ref[1]), t
    best = s.autotune(5)
    assert best["entries_per_thread"] in TILINGS
    x = torch.zeros_like(b)
    st = s.solve(b, x, rule=1, tol=1e-6)[0]
    assert st["failure"] == 0 and abs(st["iterations"] - ref[0]) <= 1


@pytest.mark.parametrize("kind", ["fem", "hybrid"])
def test_spmv_load_policies_identical(kind):
    """Nontemporal and ordinary SpMV matrix loads (masx_set_spmv_loads) give
    bit-identical solves at every tiling, FEM rows and affine-body couplings
    alike; the automatic policy keeps a matrix this small on ordinary loads."""
    w = (W.fem_grid(10, n_contacts=600, seed=5) if kind == "fem"
         else W.hybrid(seed=4, n_bodies=60, n_body_pairs=400, fem_n=7, n_coupled=12))
    s = session.solver_for(w)
    s.build("fp32")
    assert not s.spmv_nontemporal()
    b = dev(session.rhs_of(w))
    for t in TILINGS:
        s.set_spmv_tiling(t)
        out = {}
        for mode in (1, 2):
            s.set_spmv_loads(mode)
            assert s.spmv_nontemporal() == (mode == 1)
            x = torch.zeros_like(b)
            st = s.solve(b, x, rule=1, tol=1e-6)[0]
            assert st["failure"] == 0 and st["rel_res_true"] <= 1e-6 * (1 + 1e-6), (t, mode, st)
            out[mode] = (st["iterations"], host(x))
        assert out[1][0] == out[2][0], t
        assert np.array_equal(out[1][1], out[2][1]), t
    s.set_spmv_loads(0)
    assert not s.spmv_nontemporal()
    with pytest.raises(RuntimeError):
        s.set_spmv_loads(3)


@pytest.mark.parametrize("bank", [32, 16])
def test_mas_waves_agree_and_autotune(oracle, bank):
    """The FP32 MAS local kernel with 4 or 8 waves per workgroup, its inverse
    read by each lane or staged through LDS (variants 5 and 9), applies the
    same preconditioner (the FP32 sums of the waves' partials in another
    order: within 1e-6 of each other, 1e-4 of the oracle's apply; the staged
    form of a wave count bit for bit like the unstaged one) and gives the
    same solve; the autotuner reports one of them."""
    w = W.fem_grid(12, n_contacts=300, seed=21, young_sigma=0.5)
    s = session.solver_for(w, bank=bank)
    s.build("fp32")
    mas = oracle_mas(oracle, w, bank=bank)
    r = np.random.default_rng(4).standard_normal(3 * w["block_rows"])
    want = mas.apply(r)
    b = dev(session.rhs_of(w))
    its, zs = [], []
    for waves in (4, 8, 5, 9):
        s.set_mas_waves(waves)
        z = torch.zeros_like(dev(r))
        s.apply_preconditioner(dev(r), z)
        zs.append(host(z))
        assert np.linalg.norm(zs[-1] - want) <= 1e-4 * np.linalg.norm(want), waves
        x = torch.zeros_like(b)
        st = s.solve(b, x, rule=1, tol=1e-4)[0]
        assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6), (waves, st)
        its.append(st["iterations"])
    assert np.linalg.norm(zs[0] - zs[1]) <= 1e-6 * np.linalg.norm(zs[0])
    assert np.array_equal(zs[2], zs[0]) and np.array_equal(zs[3], zs[1])
    assert max(its) - min(its) <= 1
    best = s.autotune_mas(5)
    assert best["waves"] in (4, 8, 5, 9) and best["ms"] > 0


@pytest.mark.parametrize("precision", ["fp16", "bf16"])
def test_half_local_variants_agree_and_autotune(precision):
    """Half-precision 32-slot banks: the MFMA local kernel (tile layout) and
    the 4- and 8-wave VALU kernels (block-diagonal layout) apply the same
    stored inverse (FP32 accumulation in other orders: within 1e-5 of each
    other) and give the same solve; switching between the layouts asks for a
    new build; the autotuner reports one of the three."""
    w = W.fem_grid(12, n_contacts=300, seed=22, young_sigma=0.5)
    s = session.solver_for(w)
    r = dev(np.random.default_rng(5).standard_normal(3 * w["block_rows"]))
    b = dev(session.rhs_of(w))
    zs, its = [], []
    for waves in (1, 4, 8):
        s.set_mas_waves(waves)
        s.build(precision)
        z = torch.zeros_like(r)
        s.apply_preconditioner(r, z)
        zs.append(host(z))
        x = torch.zeros_like(b)
        st = s.solve(b, x, rule=1, tol=1e-4)[0]
        assert st["failure"] == 0 and st["rel_res_true"] <= 1e-4 * (1 + 1e-6), (waves, st)
        its.append(st["iterations"])
    for z in zs[1:]:
        assert np.linalg.norm(z - zs[0]) <= 1e-5 * np.linalg.norm(zs[0])
    assert max(its) - min(its) <= 1
    s.set_mas_waves(1)  # VALU layout -> MFMA layout: the built inverse no longer fits
    with pytest.raises(RuntimeError, match="build"):
        s.solve(b, torch.zeros_like(b), rule=1, tol=1e-4)
    s.build(precision)
    best = s.autotune_mas(5)
    assert best["waves"] in (1, 4, 8) and best["ms"] > 0
    x = torch.zeros_like(b)
    st = s.solve(b, x, rule=1, tol=1e-4)[0]
    assert st["failure"] == 0 and abs(st["iterations"] - its[0]) <= 1


def test_frozen_dump_replay_on_gpu(tmp_path):
    """A frozen system written in the reference's dump layout and read back
    solves with the reference-held counts (MAS32 over the identity partition)."""
    from agipc_learning_amd import frozen

    d = padded_chain()
    frozen.write_frozen(tmp_path, d["vals"], d["rows"], d["cols"], d["rhs"])
    r = frozen.read_frozen(tmp_path)
    s = native.Solver()
    s.add_system(block_rows=r["block_rows"], rows=r["rows"], cols=r["cols"], use_mas=True)
    s.set_topology(0, d["start"], d["num"], d["list"], d["part_to_real"], d["real_to_part"])
    s.setup()
    s.set_values(0, dev(r["vals"]))
    s.build("fp32")
    x = torch.zeros(3 * r["block_rows"], dtype=torch.float64, device="cuda")
    st = s.solve(dev(r["rhs"]), x, rule=1, tol=1e-3, max_iter=512)[0]
    assert st["iterations"] == REFERENCE_ITERATIONS["mas32"], st


@pytest.mark.parametrize("n,nr,drop_lower,long_row", [(5000, 50, False, False), (20000, 400, True, False),
                                                      (3000, 30, False, True), (1, 1, False, False)])
def test_converter_matches_oracle(oracle, n, nr, drop_lower, long_row):
    """Triplets -> BCOO on the GPU equals the oracle bit for bit (same sort
    order, duplicates summed in input order); a row of >1024 triplets takes
    the global-scratch sort."""
    rng = np.random.default_rng(n + nr)
    r = rng.integers(0, nr, n).astype(np.int32)
    c = rng.integers(0, nr, n).astype(np.int32)
    if long_row:
        r[: n // 2] = 7  # one row with 1500 triplets
    v = rng.standard_normal((n, 9))
    conv = native.Converter()
    ur, uc, uv = conv.convert(torch.from_numpy(r).cuda(), torch.from_numpy(c).cuda(), dev(v), nr, drop_lower)
    er, ec, ev = oracle.convert_triplets(r, c, v, drop_lower)
    assert np.array_equal(host(ur), er) and np.array_equal(host(uc), ec)
    assert np.array_equal(host(uv), ev)
    # a second call with other sizes reuses (and grows) the scratch
    ur2, _, _ = conv.convert(torch.from_numpy(r[:n // 3]).cuda(), torch.from_numpy(c[:n // 3]).cuda(),
                             dev(v[:n // 3]), nr, drop_lower)
    assert np.array_equal(host(ur2), oracle.convert_triplets(r[:n // 3], c[:n // 3], v[:n // 3], drop_lower)[0])


def test_converter_rejects_bad_index():
    conv = native.Converter()
    r = torch.tensor([0, 5], dtype=torch.int32, device="cuda")
    c = torch.tensor([0, 1], dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError):
        conv.convert(r, c, dev(np.zeros((2, 9))), 3)


def test_converter_feeds_the_solver(oracle):
    """Per-element triplets of a FEM system (every block split in random
    parts, shuffled) converted on the GPU solve like the assembled system."""
    w = W.fem_grid(8, n_contacts=100, seed=3)
    rng = np.random.default_rng(5)
    parts = rng.integers(1, 4, len(w["rows"]))
    idx = np.repeat(np.arange(len(w["rows"])), parts)
    frac = rng.random(len(idx))
    vals = w["vals"][idx] * frac[:, None]
    # make the parts sum exactly to the block: the last part takes the rest
    last = np.r_[np.nonzero(np.diff(idx))[0], len(idx) - 1]
    sums = np.zeros_like(w["vals"])
    np.add.at(sums, idx, vals)
    vals[last] += w["vals"] - sums
    perm = rng.permutation(len(idx))
    r, c, v = w["rows"][idx][perm].astype(np.int32), w["cols"][idx][perm].astype(np.int32), vals[perm]
    conv = native.Converter()
    ur, uc, uv = conv.convert(torch.from_numpy(r).cuda(), torch.from_numpy(c).cuda(), dev(v), w["block_rows"])
    er, ec, ev = oracle.convert_triplets(r, c, v)
    assert np.array_equal(host(uv), ev)
    s = native.Solver()
    s.add_system(block_rows=w["block_rows"], rows=host(ur), cols=host(uc), use_mas=False, global_diag=True)
    s.setup()
    s.set_values(0, uv.contiguous())
    s.build("fp32")
    b = session.rhs_of(w)
    x = torch.zeros(len(b), dtype=torch.float64, device="cuda")
    st = s.solve(dev(b), x, rule=1, tol=1e-6)[0]
    assert st["failure"] == 0 and st["rel_res_true"] <= 1e-6 * (1 + 1e-6)
    xo, so = oracle.pcg(w["block_rows"], w["vals"], w["rows"], w["cols"], b, global_diag=True, tol=1e-6, rule=1)
    assert np.linalg.norm(host(x) - xo) <= 1e-4 * np.linalg.norm(xo)


def test_spmv_row_longer_than_a_chunk(oracle):
    """Two hubs: block row 0 couples to 1500 rows after it (upper entries) and
    the last row to 1500 rows before it (lower entries), more than one SpMV
    chunk holds for every tiling (those rows' tiles loop over chunks)."""
    n = 1502
    rng = np.random.default_rng(2)
    rows, cols, vals = [], [], []
    for i in range(n):
        rows.append(i); cols.append(i)
        vals.append((np.eye(3) * (3000.0 if i in (0, n - 1) else 8.0)).T.reshape(9))
    for j in range(1, n - 1):
        for hub in (0, n - 1):
            B = rng.standard_normal((3, 3)) * 0.5
            r, c = (hub, j) if hub < j else (j, hub)
            rows.append(r); cols.append(c); vals.append(B.T.reshape(9))
    rows, cols, vals = np.array(rows, np.int32), np.array(cols, np.int32), np.array(vals)
    b = rng.standard_normal(3 * n)
    xo, so = oracle.pcg(n, vals, rows, cols, b, global_diag=True, tol=1e-6, rule=1)
    s = native.Solver()
    s.add_system(block_rows=n, rows=rows, cols=cols, use_mas=False, global_diag=True)
    s.setup()
    s.set_values(0, dev(vals))
    s.build("fp32")
    for t in TILINGS:
        s.set_spmv_tiling(t)
        x = torch.zeros(3 * n, dtype=torch.float64, device="cuda")
        st = s.solve(dev(b), x, rule=1, tol=1e-6)[0]
        assert st["failure"] == 0 and abs(st["iterations"] - so["iterations"]) <= max(1, round(0.05 * so["iterations"]))
        assert np.linalg.norm(host(x) - xo) <= 1e-4 * np.linalg.norm(xo), t
