"""Kernels whose split depends on the size, at the sizes where each split
starts, ends or has a remainder, against the oracle or a closed form."""
import ctypes as C

import numpy as np
import pytest

from neuronephys_clean_amd import _lib
from neuronephys_clean_amd.devmem import DeviceArray as DA

pytestmark = pytest.mark.gpu
DT = {np.float32: _lib.F32, np.float64: _lib.F64}


def say(*a):
    print(*a, flush=True)


def free_bytes(ctx):
    """Free device memory by the runtime that libnnx.so is linked to (its
    symbols resolve through the library's handle; another runtime in the same
    process, such as torch's own, may not get at the device any more)."""
    free, total = C.c_size_t(), C.c_size_t()
    assert ctx._l.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _time(ctx, call, reps=4):
    """Shortest of a few calls after one to warm up, in seconds."""
    import time
    ts = []
    for _ in range(reps + 1):
        ctx.synchronize()
        t = time.perf_counter()
        call()
        ctx.synchronize()
        ts.append(time.perf_counter() - t)
    return min(ts[1:])


def _csc(n, nnz, seed):
    """Random in-edges, sorted per target, with empty targets and one hub."""
    rng = np.random.default_rng(seed)
    deg = rng.multinomial(nnz - nnz // 8, np.full(n, 1.0 / n))
    deg[rng.integers(0, n, n // 16)] = 0
    deg[n // 3] += nnz - deg.sum()
    off = np.zeros(n + 1, np.int32)
    np.cumsum(deg, out=off[1:])
    return off, rng.integers(0, n, nnz, dtype=np.int32)


# lanes per target (few and many in-edges), slabs of 64 targets, and
# the bitmap in global memory; every residue of the CSC length mod 4
@pytest.mark.parametrize("n,nnz", [(130, 4), (1500, 45_001), (1500, 150_001), (1500, 150_002), (1500, 150_003),
                                   ((1 << 19) + 65, 2_000_002), ((1 << 19) + 1, 34_000_001),
                                   ((1 << 20) + 1, 3_000_003)])
def test_count_coupling_splits(ctx, n, nnz):
    """The sum of one 1.0 per spiking in-edge is the number of them, exactly."""
    off, src = _csc(n, nnz, n + nnz)
    d_off, d_src = DA.from_numpy(ctx, off), DA.from_numpy(ctx, src)
    g = _lib.Graph(n=n, nnz=nnz, in_offsets=d_off.ptr, in_sources=d_src.ptr)
    rng = np.random.default_rng(3)
    for T in (np.float32, np.float64):
        for frac in (0.0, 0.002, 0.6, 1.0):
            say("count", n, nnz, T.__name__, frac)
            fire = rng.random(n) < frac
            cum = np.concatenate([[0], np.cumsum(fire[src])])
            words = np.packbits(np.concatenate([fire, np.zeros(-n % 64, bool)]), bitorder="little").view(np.uint64)
            bits, out = DA.from_numpy(ctx, words), DA.from_numpy(ctx, np.full(n, np.nan, T))
            ctx.call("nnx_couple", C.byref(g), _lib.COUPLE_COUNT, DT[T], bits.ptr, None, None, None, out.ptr)
            assert np.array_equal(out.numpy(), (cum[off[1:]] - cum[off[:-1]]).astype(T))


def test_count_coupling_above_the_lds_bitmap(ctx):
    """Counting is no slower than the general kernel (which takes a source
    array off the 16-byte grid) where the spike bits are read from global
    memory and few neurons fire: 0.90 of its time; 1.065 when the bits of in-edges
    outside a target's range were read as well."""
    n, deg = (1 << 20) + 64, 200
    src = np.random.default_rng(1).integers(0, n, n * deg + 4, dtype=np.int32)
    d_src = DA.from_numpy(ctx, src)
    d_off = DA.from_numpy(ctx, np.arange(n + 1, dtype=np.int32) * deg)
    fire = np.random.default_rng(2).random(n) < 0.001
    bits, out = DA.from_numpy(ctx, np.packbits(fire, bitorder="little").view(np.uint64)), DA.zeros(ctx, n, np.float32)
    t = []
    for shift in (0, 1):
        g = _lib.Graph(n=n, nnz=n * deg, in_offsets=d_off.ptr, in_sources=d_src.ptr + 4 * shift)
        t.append(_time(ctx, lambda: ctx.call("nnx_couple", C.byref(g), _lib.COUPLE_COUNT, _lib.F32, bits.ptr, None,
                                             None, None, out.ptr)))
        assert np.array_equal(out.numpy(), fire[src[shift:shift + n * deg]].reshape(n, deg).sum(1).astype(np.float32))
    say("count above the LDS bitmap", t)
    assert t[0] <= 1.03 * t[1]


def _operator(ctx, nx, ny, nz, var, seed=6):
    """Device grid, oracle grid and the arrays to keep: constant c = 1.3, or
    random face coefficients."""
    import oracle
    if not var:
        return _lib.Grid(nx, ny, nz, 7, 1.3, 0.0, None, None, None), oracle.grid(nx, ny, nz, 7, 1.3), []
    rng = np.random.default_rng(seed)
    k = [rng.uniform(0.1, 5, s).astype(np.float32)
         for s in ((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx))]
    d = [DA.from_numpy(ctx, a) for a in k]
    return _lib.Grid(nx, ny, nz, 7, 0.0, 0.0, *(a.ptr for a in d)), oracle.grid(nx, ny, nz, 7, 0.0, 0.0, *k), d


# rows of 8, 16, 32 and 64 lanes with remainders in x, y and z; 2, 4 and 16
# planes a tile (variable coefficients: 2, 4, 8 and 16)
SHAPES = [(4, 3, 2), (20, 33, 7), (60, 50, 41), (100, 131, 22), (128, 130, 66), (152, 90, 97), (200, 120, 151)]
# more tiles than blocks: the first half's 2048 (variable coefficients), the
# second half's and the residual's 1024 (constant), in place and in padded rows
SHAPES += [(4, 1000, 600), (13, 1000, 600)]
# rows of every residue mod 4 (padded working rows), from the shortest padded
# row and one below it on, in every tile width
SHAPES += [(11, 9, 7), (12, 9, 5), (13, 9, 5), (31, 33, 8), (67, 40, 33), (102, 64, 21), (150, 131, 30), (201, 120, 150)]


@pytest.mark.parametrize("dims,var", [(d, v) for d in SHAPES for v in (False, True)] + [((276, 200, 190), True), ((250, 200, 215), True)])
def test_tiled_solve_shapes(ctx, dims, var):
    """The apply bit for bit; three CG iterations from zero against the
    oracle's (its sums taken in another order: alpha and beta are fp32 roundings
    of FP64 sums, each within 2^-23 of the oracle's, and the vectors' own
    roundings add a few 2^-24 an iteration: 1e-5 of the largest value); a
    refined solve to 1e-9 by its FP64 residual with the oracle's operator."""
    import oracle
    nx, ny, nz = dims
    say("tiles", dims, "var" if var else "const")
    g, og, keep = _operator(ctx, nx, ny, nz, var)
    n = nx * ny * nz
    b = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    db, dx = DA.from_numpy(ctx, b), DA.zeros(ctx, n, np.float32)
    ctx.call("nnx_stencil_apply", C.byref(g), db.ptr, dx.ptr)
    assert np.array_equal(dx.numpy(), oracle.apply(og, b))
    o = _lib.CgOpts(rtol=0.0, maxit=3, precond=_lib.PRECOND_JACOBI, check_every=1)
    assert ctx._l.nnx_cg_solve(ctx.h, C.byref(g), db.ptr, dx.ptr, C.byref(o), None) == 4  # NNX_ERR_NOCONV
    ref = oracle.cg(og, b, 0.0, maxit=3)[0]
    assert np.abs(dx.numpy() - ref).max() <= 1e-5 * np.abs(ref).max()
    b64, x64 = DA.from_numpy(ctx, b.astype(np.float64)), DA.zeros(ctx, n, np.float64)
    o = _lib.CgOpts(rtol=1e-9, maxit=500, precond=_lib.PRECOND_JACOBI, check_every=4)
    ctx.call("nnx_cg_solve_refine", C.byref(g), b64.ptr, x64.ptr, C.byref(o), 1e-6, 10, None)
    res = b.astype(np.float64) - oracle.apply(og, x64.numpy())
    assert np.linalg.norm(res) <= 1.001e-9 * np.linalg.norm(b.astype(np.float64))


@pytest.mark.parametrize("dims,var,shift", [((33, 21, 14), False, 0), ((33, 21, 14), True, 0), ((34, 21, 14), True, 0),
                                            ((35, 20, 9), False, 1), ((36, 20, 9), False, 1), ((36, 20, 9), True, 1),
                                            ((130, 131, 130), True, 0), ((147, 146, 146), False, 0)])
def test_padded_solvers_agree(ctx, dims, var, shift):
    """nnx_cg_solve, nnx_cg_solve_async and its allocation-free form on rows
    that are no multiple of 4 voxels, and on vectors off the 16-byte grid
    (shift), the last two grids of the sizes that the allocation-free form's
    array holds unpadded only (generic kernels in all three): the same bits, from zero and from a guess, and nothing written
    beside x."""
    nx, ny, nz = dims
    say("padded", dims, var, shift)
    g, og, keep = _operator(ctx, nx, ny, nz, var)
    n = nx * ny * nz
    rng = np.random.default_rng(n)
    b, x0 = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    db, res = DA.from_numpy(ctx, b), DA.zeros(ctx, 4, np.float64)
    for use_x0 in (0, 1):
        for maxit in (0, 1, 60):
            o = _lib.CgOpts(rtol=1e-6, maxit=maxit, precond=_lib.PRECOND_JACOBI, check_every=1, use_x0=use_x0)
            got = []
            for name in ("nnx_cg_solve", "nnx_cg_solve_async", "nnx_cg_solve_async_noalloc"):
                buf = np.full(n + 8, 7.0, np.float32)
                buf[4 + shift:4 + shift + n] = x0
                dx = DA.from_numpy(ctx, buf)
                last = C.byref(_lib.CgResult()) if name == "nnx_cg_solve" else res.ptr
                st = getattr(ctx._l, name)(ctx.h, C.byref(g), db.ptr, dx.ptr + 4 * (4 + shift), C.byref(o), last)
                assert st in (0, 4)
                got.append(dx.numpy())
            assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
            assert (got[0][:4 + shift] == 7.0).all() and (got[0][4 + shift + n:] == 7.0).all()
            if maxit == 0:
                assert np.array_equal(got[0][4 + shift:4 + shift + n], x0 if use_x0 else 0 * x0)


@pytest.mark.parametrize("var", [False, True])
def test_capturable_solve_allocates_once(var):
    """After a solve into an aligned x, one of the same grid into an x off the
    16-byte grid (as a capture may hold) allocates nothing: free device memory
    stays (a vector of this grid is 8 MiB)."""
    ctx = _lib.Context(0)
    n = 128 ** 3
    say("allocates once", var)
    g, og, keep = _operator(ctx, 128, 128, 128, var)
    db, res = DA.from_numpy(ctx, np.ones(n, np.float32)), DA.zeros(ctx, 4, np.float64)
    dx = DA.zeros(ctx, n + 4, np.float32)
    o = _lib.CgOpts(rtol=1e-3, maxit=4, precond=_lib.PRECOND_JACOBI, check_every=1)
    free = []
    for shift in (0, 1):
        ctx.call("nnx_cg_solve_async", C.byref(g), db.ptr, dx.ptr + 4 * shift, C.byref(o), res.ptr)
        ctx.synchronize()
        free.append(free_bytes(ctx))
    assert free[1] == free[0]


@pytest.mark.parametrize("var", [False, True])
@pytest.mark.parametrize("refine", [False, True])
def test_solves_on_one_long_row(ctx, var, refine):
    """Ten iterations and the closing FP64 residual on 1,000,000 x 1 x 1 cost a
    small multiple of the same voxels as 100 x 100 x 100: no pass leaves a row to
    one wavefront.  (A tile holds one row of its 4 to 32, and of its planes one:
    1.4-2.8 times the cube's; 22-64 with single-wavefront passes.)"""
    t = []
    for dims in ((100, 100, 100), (1_000_000, 1, 1)):
        g, og, keep = _operator(ctx, *dims, var)
        n = 1_000_000
        b = np.random.default_rng(1).standard_normal(n)
        if refine:
            db, dx = DA.from_numpy(ctx, b), DA.zeros(ctx, n, np.float64)
            o = _lib.CgOpts(rtol=1e-14, maxit=10, precond=_lib.PRECOND_JACOBI, check_every=5)
            t.append(_time(ctx, lambda: ctx._l.nnx_cg_solve_refine(ctx.h, C.byref(g), db.ptr, dx.ptr, C.byref(o), 1e-6,
                                                                   2, None)))
        else:
            db, dx = DA.from_numpy(ctx, b.astype(np.float32)), DA.zeros(ctx, n, np.float32)
            o = _lib.CgOpts(rtol=0.0, maxit=10, precond=_lib.PRECOND_JACOBI, check_every=5)
            res = _lib.CgResult()
            t.append(_time(ctx, lambda: ctx._l.nnx_cg_solve(ctx.h, C.byref(g), db.ptr, dx.ptr, C.byref(o),
                                                            C.byref(res))))
    say("one long row", var, refine, t, t[1] / t[0])
    assert t[1] <= 10 * t[0]


@pytest.mark.parametrize("call,vectors", [("solve", 5), ("refine", 8), ("fcg", 11), ("capturable", 6)])
def test_working_memory(call, vectors):
    """The device memory a new context's first solve on 128^3 with variable
    coefficients takes, in fp32 vectors of the grid (8 MiB): r, two directions,
    q and the inverse diagonal; a refinement's FP64 residual (two) and
    correction; flexible CG's seven and the residual's four; the capturable
    solve's vector for an unaligned x.  Reductions and state: under 4 MiB."""
    import gc
    gc.collect()  # (nothing of an earlier test is freed in between)
    ctx = _lib.Context(0)
    n = 128 ** 3
    g, og, keep = _operator(ctx, 128, 128, 128, True)
    T = np.float64 if call == "refine" else np.float32
    db, dx = DA.from_numpy(ctx, np.ones(n, T)), DA.zeros(ctx, n + 4, T)
    res = DA.zeros(ctx, 4, np.float64)
    o = _lib.CgOpts(rtol=1e-2, maxit=200, precond=_lib.PRECOND_JACOBI, check_every=4)
    ctx.synchronize()
    before = free_bytes(ctx)
    if call == "solve":
        ctx.call("nnx_cg_solve", C.byref(g), db.ptr, dx.ptr, C.byref(o), None)
    elif call == "refine":
        ctx.call("nnx_cg_solve_refine", C.byref(g), db.ptr, dx.ptr, C.byref(o), 1e-2, 5, None)
    elif call == "fcg":
        ctx.call("nnx_fcg_solve", C.byref(g), None, None, db.ptr, dx.ptr, C.byref(o), None)
    else:
        ctx.call("nnx_cg_solve_async", C.byref(g), db.ptr, dx.ptr, C.byref(o), res.ptr)
    ctx.synchronize()
    used = (before - free_bytes(ctx)) / 4.0 / n
    say("working memory", call, used, "vectors")
    assert vectors <= used <= vectors + 0.5


@pytest.mark.parametrize("dims,var", [((32, 32, 32), False), ((33, 20, 31), True)])
def test_converged_guess_enqueues_nothing(ctx, dims, var):
    """A solve whose start meets the tolerance (its own solution as the guess;
    a zero right-hand side; a refinement whose inner tolerance is 1) costs the
    same whatever check_every is: the iterations of a batch are not enqueued
    before the start is known.  (1000 of them past the end: 7.5 ms, the solve 50 us.)"""
    n = int(np.prod(dims))
    g, og, keep = _operator(ctx, *dims, var)
    b = np.random.default_rng(1).standard_normal(n).astype(np.float32)
    db, dx, zero = DA.from_numpy(ctx, b), DA.zeros(ctx, n, np.float32), DA.zeros(ctx, n, np.float32)
    o = _lib.CgOpts(rtol=1e-6, maxit=500, precond=_lib.PRECOND_JACOBI, check_every=1)
    ctx.call("nnx_cg_solve", C.byref(g), db.ptr, dx.ptr, C.byref(o), None)
    x = dx.numpy()
    b64, x64 = DA.from_numpy(ctx, b.astype(np.float64)), DA.zeros(ctx, n, np.float64)
    t = {}
    for every in (1, 1000):
        o = _lib.CgOpts(rtol=1e-5, maxit=2000, precond=_lib.PRECOND_JACOBI, check_every=every, use_x0=1)
        res = _lib.CgResult()
        t["guess", every] = _time(ctx, lambda: ctx.call("nnx_cg_solve", C.byref(g), db.ptr, dx.ptr, C.byref(o),
                                                        C.byref(res)))
        assert res.iters == 0 and res.converged and np.array_equal(dx.numpy(), x)
        o2 = _lib.CgOpts(rtol=1e-5, maxit=2000, precond=_lib.PRECOND_JACOBI, check_every=every)
        d0 = DA.from_numpy(ctx, b)
        t["zero", every] = _time(ctx, lambda: ctx.call("nnx_cg_solve", C.byref(g), zero.ptr, d0.ptr, C.byref(o2), None))
        assert not d0.numpy().any()
        t["inner", every] = _time(ctx, lambda: ctx._l.nnx_cg_solve_refine(ctx.h, C.byref(g), b64.ptr, x64.ptr,
                                                                          C.byref(o2), 1.0, 1, None))
        assert not x64.numpy().any()
    say("converged guess", dims, var, {k: f"{v * 1e6:.0f} us" for k, v in t.items()})
    for k in ("guess", "zero", "inner"):
        assert t[k, 1000] <= 5 * t[k, 1]


def _dst(b, c, axes=(0, 1, 2)):
    import scipy.fft
    lam = np.ones(b.shape)
    for ax in axes:
        s = [1] * b.ndim
        s[ax] = b.shape[ax]
        m = b.shape[ax]
        lam = lam + c * (2 - 2 * np.cos(np.pi * np.arange(1, m + 1) / (m + 1))).reshape(s)
    return scipy.fft.dstn(scipy.fft.dstn(b, type=1, norm="ortho", axes=axes) / lam, type=1, norm="ortho", axes=axes)


@pytest.mark.parametrize("dims", [(33, 35, 37), (34, 33, 40), (36, 33, 34), (64, 40, 36)])
def test_paracrine_step_on_ragged_grids(ctx, dims):
    """Two in-step solves on grids whose rows are and are not multiples of 4:
    the field against the exact solution of the release counts it consumed
    (solved to a true relative residual of 1e-8, condition number 13: 1.3e-7)."""
    from neuronephys_clean_amd import configs
    from neuronephys_clean_amd.sim import Simulation
    net = configs.c1(seed=0)
    net.grid, net.voxel = dims, None
    sim = Simulation(net, np.float32, couple="fused", record_cap=1 << 16, deposit=True, ctx=ctx)
    sim.set_paracrine(300, max_inner=48, max_outer=3)
    sim.run(300, use_graph=True, chunk=300)
    counts = sim.a["voxel_counts"].numpy()
    assert counts.sum() > 0
    sim.run(300, use_graph=True, chunk=300)
    ref = _dst(net.amount * counts.astype(np.float64).reshape(dims[::-1]), net.c).ravel()
    conc = sim.a["conc"].numpy()
    say("ragged in-step", dims, np.linalg.norm(conc - ref) / np.linalg.norm(ref), sim.paracrine_stats())
    assert np.linalg.norm(conc - ref) <= 1.3e-7 * np.linalg.norm(ref)
    assert sim.paracrine_stats()["unconverged"] == 0


# variable coefficients: rows of whole groups, with ky and kz off the 16-byte
# grid too (padded working rows), of each other residue, the shortest padded
# row, shorter ones (the generic kernels); and a constant field off 16 bytes
@pytest.mark.parametrize("dims,var,foff,coff", [((36, 33, 34), True, 0, 0), ((36, 33, 34), True, 1, 0),
                                                ((33, 35, 37), True, 0, 0), ((34, 33, 30), True, 0, 1),
                                                ((35, 34, 33), True, 3, 0), ((13, 40, 41), True, 0, 0),
                                                ((11, 40, 41), True, 0, 0), ((36, 33, 34), False, 0, 1),
                                                ((35, 33, 34), False, 0, 1)])
@pytest.mark.parametrize("graph", [False, True])
def test_paracrine_step_with_face_coefficients(ctx, dims, var, foff, coff, graph):
    """In-step solves, the first on a zero field without releases, the later
    ones from the field before, and between them one of another simulation on
    another grid in the same context (the inverse diagonal is kept per grid):
    each field by its FP64 residual with the oracle's operator on what it
    consumed, no neighbour of the field written, and a field that already meets
    the tolerance left as it is."""
    import oracle
    from neuronephys_clean_amd import configs
    from neuronephys_clean_amd.sim import Simulation
    nx, ny, nz = dims
    n = nx * ny * nz

    def start(dims, seed, foff, var=True):
        nx, ny, nz = dims
        k = [np.random.default_rng(seed + q).uniform(0.1, 2, sh).astype(np.float32)
             for q, sh in enumerate(((nz, ny, nx + 1), (nz, ny + 1, nx), (nz + 1, ny, nx)))]
        if not var:
            k = []
        d = [DA.from_numpy(ctx, np.concatenate([np.zeros(foff, np.float32), a.ravel()])) for a in k]
        f = [a.ptr + 4 * foff for a in d] if var else [None] * 3
        net = configs.c1(seed=0)
        net.grid, net.voxel = dims, None
        sim = Simulation(net, np.float32, couple="event", record_cap=1 << 16, deposit=True, ctx=ctx)
        sim.set_paracrine(20, max_inner=40, max_outer=3, grid=_lib.Grid(nx, ny, nz, 7, 0.0 if var else 1.3, 0.0, *f))
        sim.keep = d
        return sim, oracle.grid(nx, ny, nz, 7, 0.0 if var else 1.3, 0.0, *(k or [None] * 3))
    sim, og = start(dims, 1, foff, var)
    other, _ = start((nx + 4, ny, nz), 5, 0)
    field = DA.from_numpy(ctx, np.concatenate([np.full(coff, 7.0), np.zeros(n), [7.0]]))
    sim.plan.paracrine.conc = field.ptr + 8 * coff
    say("in-step faces", dims, var, foff, coff, graph)
    for w in range(5):
        before = field.numpy()[coff:coff + n]
        counts = np.random.default_rng(w).poisson(0.05 if 0 < w < 4 else 0.0, n).astype(np.int32)
        sim.a["voxel_counts"].upload(counts)
        if w == 4:  # nothing released, and any field will do
            sim.plan.paracrine.rtol = 1e9
        sim.run(20, use_graph=graph, chunk=20)
        after = field.numpy()
        assert (after[:coff] == 7.0).all() and after[coff + n] == 7.0
        after = after[coff:coff + n]
        st = sim.paracrine_stats()
        if w == 0 or w == 4:
            assert np.array_equal(after, before) and st["last_inner_iters"] == 0
            continue
        b = before + sim.net.amount * counts.astype(np.float64)
        rel = np.linalg.norm(b - oracle.apply(og, after)) / np.linalg.norm(b)
        say("  solve", w, int(counts.sum()), rel, st["last_inner_iters"], st["last_outer_steps"])
        assert rel <= 1e-8 and st["unconverged"] == 0 and st["last_outer_steps"] >= 2
        if w == 2:
            other.run(20, use_graph=graph, chunk=20)


@pytest.mark.parametrize("dims,block,off", [((64, 33, 20), 0, 1), ((50, 33, 20), 0, 1), ((32, 32, 16), 16, 1),
                                            ((32, 32, 16), 16, 0), ((256, 256, 208), 0, 0), ((8, 9, 10), 0, 1)])
def test_refinement_on_unaligned_fields(ctx, dims, block, off):
    """FP64 refinement to 1e-10 on fields at 8- and 16-byte addresses (off: 1,
    0), plain and on a block lattice, and on a grid of the 1024-thread tiles;
    the residual with the oracle's operator (block by block)."""
    import oracle
    nx, ny, nz = dims
    n = nx * ny * nz
    say("refine", dims, block, off)
    g = _lib.Grid(nx, ny, nz, 7, 1.3, 0.0, None, None, None, block)
    b = np.random.default_rng(n).standard_normal(n)
    db = DA.from_numpy(ctx, np.concatenate([np.zeros(off), b]))
    dx = DA.from_numpy(ctx, np.full(n + off, 3.0))
    o = _lib.CgOpts(rtol=1e-10, maxit=500, precond=_lib.PRECOND_JACOBI, check_every=4)
    ctx.call("nnx_cg_solve_refine", C.byref(g), db.ptr + 8 * off, dx.ptr + 8 * off, C.byref(o), 1e-6, 10, None)
    x = dx.numpy()
    assert (x[:off] == 3.0).all()
    X, B = x[off:].reshape(nz, ny, nx), b.reshape(nz, ny, nx)
    m = block or max(dims)
    res = 0.0
    for k in range(0, nz, m):
        for j in range(0, ny, m):
            for i in range(0, nx, m):
                s = np.s_[k:k + m, j:j + m, i:i + m]
                xs = np.ascontiguousarray(X[s])
                og = oracle.grid(xs.shape[2], xs.shape[1], xs.shape[0], 7, 1.3)
                res += ((B[s] - oracle.apply(og, xs.ravel()).reshape(xs.shape)) ** 2).sum()
    assert np.sqrt(res) <= 1.001e-10 * np.linalg.norm(b)


# small levels run by one workgroup: one, two and three of them, boxes long in
# each direction, 4096 cells exactly, and sizes above which another level goes
# by launches
@pytest.mark.parametrize("dims", [(8, 10, 12), (16, 16, 16), (32, 32, 32), (8, 8, 512), (8, 512, 8), (512, 8, 8),
                                  (48, 24, 16), (64, 32, 16), (40, 36, 28)])
@pytest.mark.parametrize("nu,smoother,cycle", [(3, 0, 2), (1, 1, 1), (5, 0, 1)])
def test_multigrid_small_levels(ctx, dims, nu, smoother, cycle):
    """One cycle against the numpy restatement in FP64: a cycle's fp32 sums
    carry a few hundred roundings of 2^-24 each, 1e-4 of the norm."""
    import mg_ref
    from neuronephys_clean_amd import host
    nx, ny, nz = dims
    say("mg small", dims, nu, smoother, cycle)
    rng = np.random.default_rng(nx + ny + nz)
    c = (20.0 * np.exp(0.5 * rng.standard_normal((nz, ny, nx)))).astype(np.float32)
    k = host.face_coefficients(c)
    d = [DA.from_numpy(ctx, a) for a in k]
    g = _lib.Grid(nx, ny, nz, 7, 0.0, 0.0, *(a.ptr for a in d))
    r = rng.standard_normal((nz, ny, nx)).astype(np.float32)
    dr, dz = DA.from_numpy(ctx, r.ravel()), DA.zeros(ctx, r.size, np.float32)
    ctx.call("nnx_mg_apply", C.byref(g), nu, smoother, cycle, dr.ptr, dz.ptr)
    ref = mg_ref.vcycle(r.astype(np.float64), *(a.astype(np.float64) for a in k), nu=nu,
                        smoother=("chebyshev", "jacobi")[smoother], gamma=cycle)
    got = dz.numpy().reshape(r.shape)
    assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref)


# levels above the one-workgroup ones: rows of whole 16-byte groups (fewer and
# more than a wavefront's 64, last workgroup partly empty, one coarse level
# off the rule) and rows that are not, every smoother, fields off 16 bytes
@pytest.mark.parametrize("dims", [(12, 40, 40), (20, 34, 22), (68, 20, 24), (260, 12, 10), (516, 8, 10), (18, 24, 24),
                                  (36, 24, 48)])
@pytest.mark.parametrize("nu,smoother,cycle,off", [(3, 0, 2, 0), (2, 1, 2, 1), (1, 0, 1, 3)])
def test_multigrid_row_groups(ctx, dims, nu, smoother, cycle, off):
    """One cycle against the numpy restatement in FP64, with the bound of
    test_multigrid_small_levels."""
    import mg_ref
    from neuronephys_clean_amd import host
    nx, ny, nz = dims
    say("mg rows", dims, nu, smoother, cycle, off)
    rng = np.random.default_rng(nx + ny + nz)
    c = (20.0 * np.exp(0.5 * rng.standard_normal((nz, ny, nx)))).astype(np.float32)
    k = host.face_coefficients(c)
    pad = np.zeros(off, np.float32)
    d = [DA.from_numpy(ctx, np.concatenate([pad, a.ravel()])) for a in k]
    g = _lib.Grid(nx, ny, nz, 7, 0.0, 0.0, *(a.ptr + 4 * off for a in d))
    r = rng.standard_normal((nz, ny, nx)).astype(np.float32)
    dr = DA.from_numpy(ctx, np.concatenate([pad, r.ravel(), pad]))
    dz = DA.from_numpy(ctx, np.full(r.size + 2 * off, 7.0, np.float32))
    ctx.call("nnx_mg_apply", C.byref(g), nu, smoother, cycle, dr.ptr + 4 * off, dz.ptr + 4 * off)
    ref = mg_ref.vcycle(r.astype(np.float64), *(a.astype(np.float64) for a in k), nu=nu,
                        smoother=("chebyshev", "jacobi")[smoother], gamma=cycle)
    z = dz.numpy()
    got = z[off:off + r.size].reshape(r.shape)
    assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref)
    assert (z[:off] == 7.0).all() and (z[off + r.size:] == 7.0).all()


# flexible CG's product: rows of whole 16-byte groups (eighths of the grid that
# start inside a row, fewer groups than lanes) and rows that are not
@pytest.mark.parametrize("dims", [(4, 4, 4), (12, 7, 5), (20, 33, 9), (260, 6, 7), (18, 9, 11)])
def test_flexible_cg_row_groups(ctx, dims):
    """The solution's residual against FP64 is what the solver reports:
    fp32 solves stop at 1e-5, so 2e-5 (the vectors' own roundings, 2^-24 per
    iteration, are far below)."""
    import mg_ref
    from neuronephys_clean_amd import host
    nx, ny, nz = dims
    say("fcg", dims)
    rng = np.random.default_rng(nx + ny + nz)
    c = (5.0 * np.exp(0.5 * rng.standard_normal((nz, ny, nx)))).astype(np.float32)
    k = host.face_coefficients(c)
    d = [DA.from_numpy(ctx, a) for a in k]
    g = _lib.Grid(nx, ny, nz, 7, 0.0, 0.0, *(a.ptr for a in d))
    b = rng.standard_normal((nz, ny, nx)).astype(np.float32)
    db, dx = DA.from_numpy(ctx, b.ravel()), DA.zeros(ctx, b.size, np.float32)
    o = _lib.CgOpts(rtol=1e-5, maxit=2000, precond=_lib.PRECOND_JACOBI, check_every=1, stall_iters=10)
    res = _lib.CgResult()
    ctx.call("nnx_fcg_solve", C.byref(g), None, None, db.ptr, dx.ptr, C.byref(o), C.byref(res))
    assert res.converged
    ax = mg_ref.apply(dx.numpy().reshape(b.shape).astype(np.float64), *(a.astype(np.float64) for a in k))
    assert np.linalg.norm(b - ax) <= 2e-5 * np.linalg.norm(b)


@pytest.mark.parametrize("n", [1, 64, 65, 4095, 4097, 262_145, (1 << 20) - 1, (1 << 20) + 1, 1_700_003, 1 << 22,
                               (1 << 22) + 1, 5_000_003])
def test_compaction_splits(ctx, n):
    """The ascending list and its length on bitmaps that are empty, sparse,
    full and mixed (full words among empty ones), at the block sizes' edges;
    nothing written past the list."""
    rng = np.random.default_rng(n)
    say("compact", n)
    d_list, d_count = DA(ctx, n + 8, np.int32), DA.zeros(ctx, 1, np.int32)
    for frac in (0.0, 0.0005, 0.02, 0.4, 1.0, -1.0):
        if frac < 0:
            fire = np.repeat(rng.random(-(-n // 64)) < 0.1, 64)[:n]
        else:
            fire = rng.random(n) < frac
        words = np.packbits(np.concatenate([fire, np.zeros(-n % 64, bool)]), bitorder="little").view(np.uint64)
        d_list.upload(np.full(n + 8, -7, np.int32))
        ctx.call("nnx_spike_compact", n, DA.from_numpy(ctx, words).ptr, d_list.ptr, d_count.ptr)
        want, got = np.flatnonzero(fire), d_list.numpy()
        assert int(d_count.numpy()[0]) == len(want)
        assert np.array_equal(got[:len(want)], want) and (got[len(want):] == -7).all()


def test_compaction_of_large_networks(ctx):
    """A spike list takes a time that grows with the network, not much faster:
    eight times the neurons, none firing, at most six times as long (4.5; 8 with
    a prefix over every 256 words), and at 5% firing at most twice as long as
    without spikes (1.2; 2.3 with the words emitted one by one)."""
    def words(n, frac):
        fire = np.random.default_rng(n).random(n, dtype=np.float32) < frac
        return DA.from_numpy(ctx, np.packbits(fire, bitorder="little").view(np.uint64))

    def seconds(n, frac):
        w, d_list, d_count = words(n, frac), DA(ctx, n, np.int32), DA.zeros(ctx, 1, np.int32)

        def many():
            for _ in range(50):
                ctx.call("nnx_spike_compact", n, w.ptr, d_list.ptr, d_count.ptr)
        return _time(ctx, many) / 50
    small, large, firing = seconds(1 << 21, 0.0), seconds(1 << 24, 0.0), seconds(1 << 21, 0.05)
    say("compact times", small, large, firing)
    assert large <= 6 * small and firing <= 2 * small


# the smoothed A-norm loss's operator: rows of 16, 32 and 80 lanes (a row's
# group in one wavefront, rows in one, a row over two), samples beside samples
@pytest.mark.parametrize("nx,batch,smooth", [(64, 3, 1), (128, 1, 2), (320, 2, 1), (576, 1, 0)])
def test_training_operator_rows(ctx, nx, batch, smooth):
    """With all-zero parameters the network's output is zero and the loss is
    (S^m t . A S^m t) / (t . A t).  Values carry a few dozen roundings of 2^-24
    of what S and A subtract, the quotient is some 0.05 of that: 1e-4."""
    import torch
    from test_gpu_unet import apply_A, diag_A

    from neuronephys_clean_amd.precond import UNet
    ny, nz = 32, 32
    rng = np.random.default_rng(nx)
    r = rng.standard_normal((batch, nz, ny, nx)).astype(np.float32)
    # the largest values where a row leaves a wavefront, and at the box's ends
    e = (0.05 * rng.standard_normal(r.shape)).astype(np.float32)
    for q in (0, nx - 1, min(255, nx - 1), min(256, nx - 1)):
        e[..., q] = rng.standard_normal(r.shape[:-1])
    faces = [rng.uniform(1, 60, sh).astype(np.float32) for sh in
             ((batch, nz, ny, nx + 1), (batch, nz, ny + 1, nx), (batch, nz + 1, ny, nx))]
    say("training operator", nx, batch, smooth)
    net = UNet(ctx, params=np.zeros_like(UNet(ctx, seed=1).params()))
    dr, de = DA.from_numpy(ctx, r), DA.from_numpy(ctx, e)
    loss = net.train_step((nx, ny, nz), batch, dr, dr, de, 0.0, faces=[DA.from_numpy(ctx, a) for a in faces],
                          smooth=smooth)
    K = [torch.from_numpy(a.astype(np.float64)) for a in faces]
    t = torch.from_numpy(e.astype(np.float64))
    u = t
    for _ in range(smooth):
        u = u - (2.0 / 3.0) * apply_A(u, *K) / diag_A(*K)
    ref = float(((u * apply_A(u, *K)).sum(dim=(1, 2, 3)) / (t * apply_A(t, *K)).sum(dim=(1, 2, 3))).mean())
    assert abs(loss - ref) <= 1e-4 * ref
