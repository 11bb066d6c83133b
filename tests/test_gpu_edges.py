"""Kernels at the sizes where their tiles, passes and dispatch rules end:
row lengths around the entries loaded per pass, blocks that do not divide a
workgroup, vertex counts that leave partial tiles.  Compared with the CPU
oracle, bit for bit where the kernel keeps the oracle's order."""
import numpy as np
import pytest

import owtk
from oracle import gnn
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def ragged_pattern(rng, n, ghost, lengths):
    """Offsets and ascending columns with the given row lengths, diagonal left out."""
    offsets = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    columns = []
    for i in range(n):
        choice = np.setdiff1d(np.arange(n + ghost), [i])
        columns.append(np.sort(rng.choice(choice, lengths[i], replace=False)))
    return offsets, np.concatenate(columns).astype(np.int32)


@pytest.mark.parametrize("block", [5, 7, 36, 65, 300])
def test_row_component_spmv(ctx, block):
    """Blocks above four components: rows of 0 to 17 entries (8 per pass), rows that straddle waves and
    workgroups; split and CSR forms bitwise, FP32 storage bitwise, the residual vector."""
    rng = np.random.default_rng(block)
    n, ghost = 37, 3
    lengths = np.concatenate([[0, 1, 7, 8, 9, 15, 16, 17], rng.integers(0, 18, n - 8)])
    off, col = ragged_pattern(rng, n, ghost, lengths)
    val = rng.uniform(-1, 1, off[-1] * block)
    diag = rng.uniform(1, 2, n * block)
    x = rng.uniform(-1, 1, (n + ghost) * block)
    xd, yd = ctx.upload(x), ctx.empty(n * block)
    om = orc.OMatrix.split(n, ghost, block, off, col, diag, val)
    m = owtk.Matrix.split(ctx, n, ghost, block, off, col, diag, val)
    m.spmv(xd, yd)
    ref = om.spmv(x)
    assert np.array_equal(yd.download(), ref)
    b = rng.uniform(-1, 1, n * block)
    m.residual(ctx.upload(b), xd, yd)
    assert np.array_equal(yd.download(), b - ref)
    mc = owtk.Matrix.csr(ctx, n, ghost, block, off, col, val)
    mc.spmv(xd, yd)
    assert np.array_equal(yd.download(), orc.OMatrix.csr(n, ghost, block, off, col, val).spmv(x))
    m.add_storage(owtk.F32)
    yf = ctx.empty(n * block, np.float32)
    m.spmv(ctx.upload(x.astype(np.float32)), yf, owtk.F32)
    assert np.array_equal(yf.download(), om.spmv_f32(val, diag, x))


@pytest.mark.parametrize("nx,ny,block,degree", [(2, 2, 1, 1), (5, 3, 3, 9), (33, 2, 2, 3), (47, 31, 3, 4), (183, 180, 3, 4)])
def test_training_gradient_sizes(ctx, nx, ny, block, degree):
    """Vertex counts below one matrix-core step, odd, and beyond one pass of the gradient reduction's grid; 2 to 30
    outputs.  FP32 sums over at most n vertices of FP32 products: 2e-3 of a block's norm holds with the same margin
    as at the sizes of the other gradient test."""
    s = owtk.generate_split(nx, ny, block, 3, ordering=owtk.ORDER_HILBERT)
    m = owtk.Matrix.split(ctx, s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    g = gnn.Graph(s.nodes, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    rng = np.random.default_rng(nx)
    errs = [rng.uniform(-1, 1, (s.nodes, block)) for _ in range(2)]
    ress = [g.apply(e) for e in errs]
    lay = gnn.Layout(block, degree)
    p = lay.unpack(gnn.init_parameters(block, degree, 1))
    p["w_out"] = rng.normal(0, 0.3, p["w_out"].shape)
    for layer in range(gnn.LAYERS):
        p[f"b{layer}"] = rng.normal(0, 0.2, p[f"b{layer}"].shape)
    params = lay.pack(p).astype(np.float32)
    model = owtk.GnnModel(ctx, block, degree)
    model.set_parameters(params)
    prob = model.problem(m, ctx.upload(np.concatenate(ress).ravel()), ctx.upload(np.concatenate(errs).ravel()), 2)
    model.zero_grad()
    model.accumulate(prob, 1.0)
    loss, grad = model.read()
    ref_loss, ref_grad = gnn.loss_and_grad(g, gnn.bf16_round(params), degree, ress, errs)
    got, ref = lay.unpack(grad.astype(np.float64)), lay.unpack(ref_grad)
    assert abs(loss - ref_loss) <= 1e-4 * ref_loss
    for k in ref:
        assert np.linalg.norm(got[k] - ref[k]) <= 2e-3 * max(np.linalg.norm(ref[k]), 1e-6 * np.linalg.norm(ref_grad)), k


@pytest.mark.parametrize("block,pairs", [(1, 1), (4, 2), (2, 3), (3, 5), (1, 6), (3, 10), (2, 11), (1, 21)])
def test_training_loss_pairs(ctx, block, pairs):
    """Pair counts at and beyond every register width of the loss kernels (2, 5, 10), rows of unequal length, and a
    row count that leaves the last block ragged; bounds as in the test above."""
    s = owtk.generate_split(23, 17, block, 5, ordering=owtk.ORDER_RCM)
    m = owtk.Matrix.split(ctx, s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    g = gnn.Graph(s.nodes, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    rng = np.random.default_rng(pairs)
    errs = [rng.uniform(-1, 1, (s.nodes, block)) * 10.0 ** (p % 3) for p in range(pairs)]
    ress = [g.apply(e) for e in errs]
    lay = gnn.Layout(block, 2)
    params = gnn.init_parameters(block, 2, 4).astype(np.float32)
    model = owtk.GnnModel(ctx, block, 2)
    model.set_parameters(params)
    prob = model.problem(m, ctx.upload(np.concatenate(ress).ravel()), ctx.upload(np.concatenate(errs).ravel()), pairs)
    model.zero_grad()
    model.accumulate(prob, 0.75)
    loss, grad = model.read()
    ref_loss, ref_grad = gnn.loss_and_grad(g, gnn.bf16_round(params), 2, ress, errs)
    got, ref = lay.unpack(grad.astype(np.float64)), lay.unpack(0.75 * ref_grad)
    assert abs(loss - 0.75 * ref_loss) <= 1e-4 * ref_loss
    for k in ref:
        assert np.linalg.norm(got[k] - ref[k]) <= 2e-3 * max(np.linalg.norm(ref[k]), 1e-6 * np.linalg.norm(ref_grad)), k


def random_dominant(rng, n, block, low, high):
    """A diagonally dominant CSR matrix with low..high off-diagonal entries per row at random columns near the
    diagonal (no symmetric pattern)."""
    offsets, columns, values = [0], [], []
    for i in range(n):
        near = np.setdiff1d(np.arange(max(0, i - 40), min(n, i + 41)), [i])
        own = rng.choice(near, min(rng.integers(low, high + 1), near.size), replace=False)
        cols = np.sort(np.concatenate([own, [i]]))
        val = -rng.uniform(0.1, 1.0, (cols.size, block))
        val[cols == i] = np.abs(val).sum(0) + 0.5
        columns.append(cols)
        values.append(val)
        offsets.append(offsets[-1] + cols.size)
    return np.array(offsets, np.int32), np.concatenate(columns).astype(np.int32), np.concatenate(values).ravel()


@pytest.mark.parametrize("case", ["1-node", "grid-1", "grid-2", "grid-3", "grid-4-rcm", "sparse", "wide", "wider", "dense"])
def test_red_black_coarse_sweeps(ctx, case):
    """Red-black multigrid against the oracle after two V cycles: one-chunk and partial chunks, 1 to 4 components,
    black coarse rows of up to 3, 6 and 9 entries (the one-wave sweep with 4, 6 and 10 slots), of 18 to 28 and
    unsymmetric patterns (the workgroup sweep, several red levels).  The sweeps keep the oracle's operations and their order; the fine
    SpMV and the residual sums bound the difference: 1e-13, as for the other multigrid solves."""
    rng = np.random.default_rng(len(case))
    if case == "1-node":
        n, block, off, col, val = 1, 2, np.array([0, 1], np.int32), np.array([0], np.int32), np.array([2.0, 3.0])
    elif case.startswith("grid"):
        block = int(case[5])
        order = owtk.ORDER_RCM if case.endswith("rcm") else owtk.ORDER_HILBERT
        s = owtk.generate_split(61, 37, block, 2, ordering=order)
        n, (off, col, val) = s.nodes, s.csr()
    else:
        low, high = {"sparse": (0, 2), "wide": (4, 6), "wider": (6, 9), "dense": (20, 30)}[case]
        n, block = 500, 2
        off, col, val = random_dominant(rng, n, block, low, high)
    b = rng.uniform(-1, 1, n * block)
    kw = dict(relative_tolerance=1e-300, maximum_iterations=2)
    xo, _ = orc.OMultigrid(orc.OMatrix.csr(n, 0, block, off, col, val), smoother=1).solve(b, cycle=0, **kw)
    m = owtk.Matrix.csr(ctx, n, 0, block, off, col, val)
    x = ctx.empty(n * block)
    owtk.Multigrid(m, smoother=owtk.MG_RED_BLACK).solve(ctx.upload(b), x, owtk.SolverOptions(**kw))
    assert np.max(np.abs(x.download() - xo)) <= 1e-13 * np.max(np.abs(xo))


def banded(rng, n, block, reach, count):
    """Diagonally dominant split-form rows with up to `count` neighbours on each side, up to `reach` rows away (the
    farthest always among them), symmetric pattern."""
    pairs = set()
    for i in range(n):
        own = rng.choice(np.arange(1, reach + 1), min(count, reach), replace=False)
        for d in set(own[: rng.integers(0, count + 1)]) | {reach}:
            if i + d < n:
                pairs.add((i, i + int(d)))
    rows = [[] for _ in range(n)]
    for i, j in pairs:
        rows[i].append(j)
        rows[j].append(i)
    columns = np.concatenate([np.sort(r) for r in rows if r] or [np.zeros(0)]).astype(np.int32)
    offsets = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    off = -rng.uniform(0.1, 1.0, (columns.size, block))
    diag = np.add.reduceat(np.abs(np.vstack([off, np.zeros((1, block))])), offsets[:-1], axis=0) + 0.5
    diag[np.diff(offsets) == 0] = 1.0
    return offsets, columns, diag.ravel(), off.ravel()


@pytest.mark.parametrize("n,block,block_nodes,reach,count", [
    (1, 1, 0, 1, 1), (15, 2, 0, 3, 2), (16, 1, 0, 5, 2), (17, 3, 0, 5, 2), (65, 5, 16, 4, 2), (130, 3, 33, 9, 3),
    (700, 1, 0, 431, 2), (700, 2, 0, 449, 3), (900, 3, 0, 448, 3), (1300, 3, 640, 500, 4), (2100, 7, 0, 900, 5),
    (1100, 4, 550, 500, 8), (900, 1, 0, 433, 14), (3000, 1, 700, 650, 2)])
def test_chain_sweeps(ctx, n, block, block_nodes, reach, count):
    """Chain sweeps (one 16-row chunk after the other): partial chunks and blocks, 1 to 7 components (groups past the
    last chain), 2 to 15 entries per row (each slot count), entries at the ends of the near range (27 chunks) and
    beyond it, in place and not, FP64 and FP32 storage.  Backward in-chunk entries fold in the order they become
    available: 1e-14 of the largest value, as for the other chain sweeps; FP32 at 2^29 times that."""
    rng = np.random.default_rng(n + reach)
    off, col, diag, val = banded(rng, n, block, reach, count)
    om = orc.OMatrix.split(n, 0, block, off, col, diag, val)
    m = owtk.Matrix.split(ctx, n, 0, block, off, col, diag, val)
    m.add_storage(owtk.F32)
    x = rng.uniform(-1, 1, n * block)
    xd, yd = ctx.upload(x), ctx.empty(n * block)
    for kind, okind, omega in ((owtk.PC_ILU, 3, 1.0), (owtk.PC_SSOR, orc.OPreconditioner.SSOR, 1.0),
                               (owtk.PC_SSOR, orc.OPreconditioner.SSOR, 1.3)):
        opc = orc.OPreconditioner(om, okind, block_nodes=block_nodes, omega=omega)
        pc = owtk.Preconditioner(m, kind, block_nodes=block_nodes, omega=omega, schedule=2)
        ref = opc.apply(x)
        pc.apply(xd, yd)
        y = yd.download()
        assert np.max(np.abs(y - ref)) <= 1e-14 * np.max(np.abs(ref))
        zd = ctx.upload(x)
        pc.apply(zd, zd)
        assert np.array_equal(zd.download(), y)
        low = owtk.Preconditioner(m, kind, block_nodes=block_nodes, omega=omega, schedule=2, storage=owtk.F32)
        wd = ctx.empty(n * block, np.float32)
        low.apply(ctx.upload(x.astype(np.float32)), wd)
        assert np.max(np.abs(wd.download() - ref)) <= 2.0 ** 29 * 1e-14 * np.max(np.abs(ref))


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 6144, 128 * 1024, 128 * 1024 + 1, 300_001])
def test_reductions_around_the_fused_grid(ctx, n):
    """Reductions that end in the kernel itself (up to 128 blocks of 1,024 values) and in a finisher, several in a
    row on one counter.  Tree sums of n products: a few ulp of the sum of magnitudes, 1e-14 holds with room; the
    norms of extreme values take the scaled second pass."""
    rng = np.random.default_rng(n)
    a, b = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
    da, db, dy = ctx.upload(a), ctx.upload(b), ctx.upload(b)
    basis = [ctx.upload(rng.uniform(-1, 1, n)) for _ in range(9)]
    host = [v.download() for v in basis]
    for _ in range(3):
        assert abs(ctx.dot(da, db) - np.dot(a, b)) <= 1e-14 * np.sum(np.abs(a * b))
        assert abs(ctx.norm(da) - np.linalg.norm(a)) <= 1e-14 * np.linalg.norm(a)
        for k in (0, 1, 3, 7, 8, 9):
            got = ctx.multidot(basis[:k], da)
            ref = np.array([np.dot(a, v) for v in host[:k]] + [np.dot(a, a)])
            assert np.all(np.abs(got - ref) <= 1e-14 * n)
    y = b + 0.25 * a
    assert abs(ctx.axpy_dot(0.25, da, dy, db) - np.dot(b, y)) <= 1e-14 * np.sum(np.abs(b * y))
    assert np.allclose(dy.download(), y, rtol=0, atol=1e-15)
    for scale in (1e300, 1e-300):
        assert abs(ctx.norm(ctx.upload(a * scale)) - np.linalg.norm(a) * scale) <= 1e-13 * np.linalg.norm(a) * scale
    assert np.isnan(ctx.norm(ctx.upload(np.where(np.arange(n) == n // 2, np.nan, a))))
    assert np.isinf(ctx.norm(ctx.upload(np.where(np.arange(n) == n - 1, -np.inf, a))))


@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 8, 9, 15, 16, 30, 31, 32, 62])
def test_finisher_widths(ctx, k):
    """The finisher for every number of values, over the multi-dot's largest grid (1,024 blocks: one full pass of a
    wave above 8 values, part of one below); a NaN in one vector reaches only that vector's value.  Bounds as in the
    test above."""
    n = 1_700_001
    rng = np.random.default_rng(k)
    host = [rng.uniform(-1, 1, n) for _ in range(3)]
    host[1][n // 3] = np.nan
    vectors = [ctx.upload(v) for v in host]
    w = rng.uniform(-1, 1, n)
    got = ctx.multidot([vectors[i % 3] for i in range(k)], ctx.upload(w))
    exact = [np.dot(v, w) for v in host]
    for i in range(k):
        assert np.isnan(got[i]) if i % 3 == 1 else abs(got[i] - exact[i % 3]) <= 1e-14 * n
    assert abs(got[k] - np.dot(w, w)) <= 1e-14 * n


@pytest.mark.parametrize("nx,ny,block", [(5, 3, 1), (128, 128, 2), (128, 256, 1), (130, 255, 3), (130, 130, 5)])
def test_solvers_around_the_fused_grid(ctx, nx, ny, block):
    """BiCGSTAB, its pipelined and communication-hiding forms on grids below, at and above 128 SpMV blocks (256 rows)
    and vector blocks, against the oracle at rtol 1e-8.  The iteration counts agree to one there (near 1e-12, after
    twice the iterations, the sums' rounding has decoupled the recurrences and they drift by several).  A row's
    diagonal exceeds the sum of its other entries by 0.05, so |A^-1| <= 20 in the maximum norm and residuals of
    1e-8 |b| leave the two solutions at most 4e-7 |b| apart."""
    s = owtk.generate_split(nx, ny, block, 4, ordering=owtk.ORDER_RCM)
    om = orc.OMatrix.split(s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    m = owtk.Matrix.split(ctx, s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    pc, opc = owtk.Preconditioner(m, owtk.PC_JACOBI), orc.OPreconditioner(om, orc.OPreconditioner.JACOBI)
    b, x = ctx.upload(s.rhs), ctx.empty(s.nodes * block)
    ref, ro = orc.bicgstab(om, opc, s.rhs, relative_tolerance=1e-8, maximum_iterations=500)
    for solve in (owtk.bicgstab, owtk.pipelined_bicgstab, owtk.communication_hiding_bicgstab):
        x.zero()
        res = solve(m, pc, b, x, owtk.SolverOptions(relative_tolerance=1e-8, maximum_iterations=500))
        assert res["status_name"] == "converged"
        if solve is owtk.bicgstab:
            assert abs(res["iterations"] - ro["iterations"]) <= 1
        assert np.max(np.abs(x.download() - ref)) <= 4e-7 * np.linalg.norm(s.rhs)


@pytest.mark.parametrize("fill", [0, 1, 3])
@pytest.mark.parametrize("n,block,low,high,nodes", [(1, 1, 0, 0, 0), (63, 3, 1, 4, 0), (64, 1, 2, 6, 0),
                                                    (65, 2, 2, 6, 0), (200, 1, 0, 12, 0), (391, 2, 1, 5, 130),
                                                    (320, 1, 30, 40, 64)])
def test_ilu_factor_forms(ctx, n, block, low, high, nodes, fill):
    """Every form of the chunked factorization (records of 3 and 7 updates, the general one) and the kernel behind it
    (long rows), with chunks and blocks that end early: the operations are the oracle's in its order, so the factors
    are its bits."""
    offsets, columns, values = random_dominant(np.random.default_rng(n + fill), n, block, low, high)
    m = owtk.Matrix.csr(ctx, n, 0, block, offsets, columns, values)
    pc = owtk.Preconditioner(m, owtk.PC_ILU, fill_level=fill, block_nodes=nodes)
    opc = orc.OPreconditioner(orc.OMatrix.csr(n, 0, block, offsets, columns, values), 3, fill_level=fill,
                              block_nodes=nodes)
    for got, ref in zip(pc.ilu_factors(), opc.ilu_factors()):
        assert np.array_equal(got, ref)


@pytest.mark.parametrize("row", [0, 63, 64, 127, 199])
def test_ilu_small_pivot_anywhere(ctx, row):
    """A vanishing pivot in a chunk's first or last row, in an earlier chunk, or in the last row of all is reported,
    and a factorization after it succeeds."""
    n = 200
    d, e = np.full(n, 4.0), np.full(2 * (n - 1), -1.0)
    offsets = np.concatenate([[0], np.cumsum([1 + (1 if i in (0, n - 1) else 2) - 1 for i in range(n)])]).astype(np.int32)
    columns = np.concatenate([[j for j in (i - 1, i + 1) if 0 <= j < n] for i in range(n)]).astype(np.int32)
    m = owtk.Matrix.split(ctx, n, 0, 1, offsets, columns, d, e)
    pc = owtk.Preconditioner(m, owtk.PC_ILU)
    bad, cut = d.copy(), e.copy()
    bad[row] = 0.0
    cut[offsets[row]:offsets[row + 1]][columns[offsets[row]:offsets[row + 1]] < row] = 0.0
    m.update_values(bad, cut)
    with pytest.raises(owtk.ZeroPivotError):
        pc.update_values()
    m.update_values(d, e)
    pc.update_values()


@pytest.mark.parametrize("nx,ny,block", [(9, 7, 2), (128, 128, 3), (128, 256, 1), (60, 40, 5)])
def test_norms_of_vectors_written_by_their_own_kernel(ctx, nx, ny, block):
    """Right-hand sides scaled until the sum of squares leaves the range that the norm takes as it is (below 2^-960,
    or infinite), on grids of at most 128 blocks: the kernels that write s, r, q and b - A x then read them back for
    the scaled second pass, written by other waves and blocks.  The small scale is a power of two that leaves the
    products normal (above 1024 times the least normal number down to rtol 1e-5), so the solve is that of the
    unscaled right-hand side: the same iterations, norms to the rounding of their sums, solutions to 1e-8 (rounding
    near the subnormal range, grown over the iterations).  At the large one the products are infinite: the first
    residual's norm, and the status of the oracle."""
    s = owtk.generate_split(nx, ny, block, 4, ordering=owtk.ORDER_RCM)
    om = orc.OMatrix.split(s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    m = owtk.Matrix.split(ctx, s.nodes, 0, block, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    pc, opc = owtk.Preconditioner(m, owtk.PC_JACOBI), orc.OPreconditioner(om, orc.OPreconditioner.JACOBI)
    kw = dict(relative_tolerance=1e-5, maximum_iterations=200)
    norm = np.linalg.norm(s.rhs)
    small = 2.0 ** np.floor((-964 - np.log2(norm ** 2)) / 2)
    huge = 2.0 ** 700
    bs, bl = ctx.upload(s.rhs * small), ctx.upload(s.rhs * huge)
    b, x = ctx.upload(s.rhs), ctx.empty(s.nodes * block)
    for solve, oracle in ((owtk.bicgstab, orc.bicgstab), (owtk.pipelined_bicgstab, orc.pipelined_bicgstab),
                          (owtk.communication_hiding_bicgstab, orc.communication_hiding_bicgstab),
                          (owtk.fgmres, orc.fgmres)):
        x.zero()
        ref = solve(m, pc, b, x, owtk.SolverOptions(**kw))
        xr = x.download()
        assert ref["status_name"] == "converged"
        x.zero()
        res = solve(m, pc, bs, x, owtk.SolverOptions(**kw))
        assert res["status_name"] == "converged" and res["iterations"] == ref["iterations"]
        assert np.max(np.abs(x.download() / small - xr)) <= 1e-8 * np.max(np.abs(xr))
        for key in ("initial_residual_norm", "true_residual_norm"):
            assert abs(res[key] / small - ref[key]) <= (1e-13 if key[0] == "i" else 1e-6) * ref[key]
        x.zero()
        res = solve(m, pc, bl, x, owtk.SolverOptions(**kw))
        _, ro = oracle(om, opc, s.rhs * huge, **kw)
        assert res["status"] == ro["status"]
        assert abs(res["initial_residual_norm"] / huge - norm) <= 1e-13 * norm


@pytest.mark.parametrize("n", [1000, 6144, 128 * 1024, 128 * 1024 + 1])
def test_axpy_dot_vector_is_complete_on_return(ctx, n):
    """The vector that axpy_dot writes, read on another context's stream as soon as the call has returned, below, at
    and above the largest grid that ends its own reduction.  Every element changes each time, by the exact 1."""
    ones, y = ctx.upload(np.ones(n)), ctx.upload(np.zeros(n))
    with owtk.Context(0) as other:
        for k in range(1, 21):
            assert ctx.axpy_dot(1.0, ones, y, ones) == k * n
            assert other.dot(y, ones) == k * n


@pytest.mark.parametrize("n", [16384, 16385])
def test_chain_sweeps_largest_block(ctx, n):
    """The largest block that the chain sweeps take, and one row more: refused when asked for, level sets otherwise.
    Bound as for the other chain sweeps."""
    rng = np.random.default_rng(n)
    off, col, diag, val = banded(rng, n, 1, 500, 3)
    m = owtk.Matrix.split(ctx, n, 0, 1, off, col, diag, val)
    opc = orc.OPreconditioner(orc.OMatrix.split(n, 0, 1, off, col, diag, val), 3)
    x = rng.uniform(-1, 1, n)
    xd, yd, ref = ctx.upload(x), ctx.empty(n), opc.apply(x)
    for schedule in (0, 2):
        if n > 16384 and schedule == 2:
            with pytest.raises(owtk.OwtkError, match="16384 rows"):
                owtk.Preconditioner(m, owtk.PC_ILU, schedule=schedule)
            continue
        owtk.Preconditioner(m, owtk.PC_ILU, schedule=schedule).apply(xd, yd)
        assert np.max(np.abs(yd.download() - ref)) <= 1e-14 * np.max(np.abs(ref))


@pytest.mark.parametrize("schedule", [0, 1, 2])
@pytest.mark.parametrize("block,nodes", [(1, 0), (3, 50)])
def test_ssor_repeated_columns(ctx, schedule, block, nodes):
    """SSOR of CSR rows that name a column more than once (their products add up), near the row and farther off, by
    every schedule.  Bound as for the other sweeps."""
    rng = np.random.default_rng(7)
    n = 200
    offsets, columns, values = [0], [], []
    for i in range(n):
        near = np.array([j for j in (i - 70, i - 20, i - 3, i - 1, i + 1, i + 2, i + 33) if 0 <= j < n])
        twice = rng.choice(near, 2)
        cols = np.sort(np.concatenate([near, twice, [i]]))
        val = -rng.uniform(0.1, 1.0, (cols.size, block))
        val[cols == i] = np.abs(val).sum(0) + 0.5
        columns.append(cols)
        values.append(val)
        offsets.append(offsets[-1] + cols.size)
    args = (n, 0, block, np.array(offsets, np.int32), np.concatenate(columns).astype(np.int32), np.concatenate(values).ravel())
    x = rng.uniform(-1, 1, n * block)
    ref = orc.OPreconditioner(orc.OMatrix.csr(*args), orc.OPreconditioner.SSOR, block_nodes=nodes, omega=1.2).apply(x)
    yd = ctx.empty(n * block)
    owtk.Preconditioner(owtk.Matrix.csr(ctx, *args), owtk.PC_SSOR, block_nodes=nodes, omega=1.2,
                        schedule=schedule).apply(ctx.upload(x), yd)
    assert np.max(np.abs(yd.download() - ref)) <= 1e-14 * np.max(np.abs(ref))


@pytest.mark.parametrize("block,degree", [(1, 0), (2, 2), (3, 5), (2, 6), (1, 7), (3, 8), (1, 16), (1, 31)])
def test_training_gradient_degrees(ctx, block, degree):
    """Coefficient counts in one pass of every width, just beyond one pass, and up to the most outputs; the checks and
    bounds of the gradient test above."""
    test_training_gradient_sizes(ctx, 23, 17, block, degree)


@pytest.mark.parametrize("block", [5, 65])
def test_row_component_residual_norm(ctx, block):
    """The norm that the residual SpMV of blocks above four reduces, as a solver's first residual: rows of 0 to 17
    entries, a start vector that is not zero.  A sum of squares over n values: a few ulp."""
    rng = np.random.default_rng(block)
    n = 137
    off, col = ragged_pattern(rng, n, 0, rng.integers(0, 18, n))
    val, diag = rng.uniform(-1, 1, off[-1] * block), rng.uniform(1, 2, n * block)
    x, b = rng.uniform(-1, 1, n * block), rng.uniform(-1, 1, n * block)
    ref = np.linalg.norm(b - orc.OMatrix.split(n, 0, block, off, col, diag, val).spmv(x))
    m = owtk.Matrix.split(ctx, n, 0, block, off, col, diag, val)
    res = owtk.bicgstab(m, None, ctx.upload(b), ctx.upload(x), owtk.SolverOptions(maximum_iterations=1))
    assert abs(res["initial_residual_norm"] - ref) <= 1e-14 * ref


@pytest.mark.parametrize("n", [8192 * 1024 + 1, 9_000_001, 16384 * 1024 + 77])
def test_norm_of_more_partials_than_a_pass(ctx, n):
    """Two values of more than 8,192 blocks: the finisher's second pass, with one block in it, part of one, and at the
    largest grid.  The exact count: sums of small integers."""
    a = np.zeros(n)
    a[::3] = 2.0
    a[-1] = 5.0
    d = ctx.upload(a)
    exact = np.sum(a * a)
    assert ctx.norm(d) == np.sqrt(exact)
    assert ctx.dot(d, d) == exact
    a[-1] = np.inf
    assert np.isinf(ctx.norm(ctx.upload(a)))


def test_solvers_of_more_partials_than_a_pass(ctx):
    """Reductions of two to six values over 6,157 vector blocks and 8,209 SpMV blocks: the finisher's second and later
    passes for every width that the solvers use.  The first residual is the right-hand side, the last one is summed
    again on the host (a few ulp of n values, 1e-13 with room), and the two forms of one recurrence need the same
    number of iterations to a few."""
    s = owtk.generate_split(1500, 1401, 3, 4, ordering=owtk.ORDER_HILBERT)
    n = s.nodes * 3
    m = owtk.Matrix.split(ctx, s.nodes, 0, 3, s.offsets, s.columns, s.diagonal, s.off_diagonal)
    pc = owtk.Preconditioner(m, owtk.PC_JACOBI)
    b, x, r = ctx.upload(s.rhs), ctx.empty(n), ctx.empty(n)
    norm, counts = np.linalg.norm(s.rhs), []
    for solve in (owtk.bicgstab, owtk.pipelined_bicgstab, owtk.communication_hiding_bicgstab):
        x.zero()
        res = solve(m, pc, b, x, owtk.SolverOptions(relative_tolerance=1e-6, maximum_iterations=200))
        assert res["status_name"] == "converged"
        m.residual(b, x, r)
        assert abs(res["initial_residual_norm"] - norm) <= 1e-13 * norm
        true = np.linalg.norm(r.download())
        assert true <= 1e-6 * norm and abs(res["true_residual_norm"] - true) <= 1e-13 * true
        counts.append(res["iterations"])
    assert max(counts) - min(counts) <= 3


@pytest.mark.parametrize("seed,low,high,widest", [(1, 1, 3, 7), (2, 1, 3, 8), (2, 3, 4, 11), (1, 3, 4, 12), (1, 4, 4, 13),
                                                  (1, 3, 5, 16), (2, 5, 5, 17)])
def test_red_black_coarse_sweep_widths(ctx, seed, low, high, widest):
    """The one-wave sweep with 8, 12 and 16 slots at their fewest and most entries per black row, and one entry more
    (the workgroup sweep); the solve and bound of the test above."""
    n, block = 500, 2
    off, col, val = random_dominant(np.random.default_rng(seed), n, block, low, high)
    m = owtk.Matrix.csr(ctx, n, 0, block, off, col, val)
    om = orc.OMultigrid(orc.OMatrix.csr(n, 0, block, off, col, val), smoother=1)
    _, coff, ccol, _, _ = om.coarse()
    red, rows = set(), [set(ccol[coff[i]:coff[i + 1]]) - {i} for i in range(len(coff) - 1)]
    for i, row in enumerate(rows):
        if not row & red:
            red.add(i)
    assert max(len(row) for i, row in enumerate(rows) if i not in red) == widest
    b = np.random.default_rng(seed).uniform(-1, 1, n * block)
    kw = dict(relative_tolerance=1e-300, maximum_iterations=2)
    xo, _ = om.solve(b, cycle=0, **kw)
    x = ctx.empty(n * block)
    owtk.Multigrid(m, smoother=owtk.MG_RED_BLACK).solve(ctx.upload(b), x, owtk.SolverOptions(**kw))
    assert np.max(np.abs(x.download() - xo)) <= 1e-13 * np.max(np.abs(xo))
