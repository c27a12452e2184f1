"""The work users of this framework have it do, as cases that can be timed.

Every case goes through the C ABI (include/nnx.h) as the package binds it,
on buffers that torch owns, and a pass starts from the same state each time:
what a step changes lies in one device block, and a pass first copies the
block's initial contents back.

  rk4    the benchmark network's loop: RK4 Hodgkin-Huxley neurons, weighted
         coupling, release and the paracrine solve on its cadence, replayed
         from step graphs (configs.c1, configs.c2)
  ens    the batched ensemble, every network with its own 64^3 grid
         (configs.c4_ensemble)
  leap   the reference's network: leapfrog with kinetic synapses and noise,
         count or signal coupling, electrodes read every print step
  scn    the reference's default program call by call: Diekman neurons, count
         coupling, release, and the reference's paracrine update
  pull   one dense weighted coupling over the transposed connectivity
  cg     one implicit diffusion step of a field, constant or variable
         diffusivity, to a true FP64 tolerance (Jacobi-CG or multigrid)
  train  one training step of the convolutional preconditioner
"""
import ctypes as C
import math

import numpy as np
import torch

from neuronephys_clean_amd import _lib, host

DEV = "cuda"
F64 = torch.float64


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # a small network on its own: 1,024 neurons with 100 edges each, launches and latency
        dict(name="loop_1k", kind="rk4", n=1024, topo="er", deg=100, f64=False, couple="fused", steps=400, chunk=100,
             every=100, hebbian=0),
        # the headline workload: a million neurons, ~210M distance-dependent edges, a 256^3 field; one cycle of its
        # synchronous firing
        dict(name="loop_1m", kind="rk4", n=1 << 20, topo="spatial", deg=200, f64=False, couple="fused", steps=1500,
             chunk=100, every=100, hebbian=0),
        # double precision, plain event coupling, Hebbian learning on every synapse, a ragged size whose field has
        # odd rows
        dict(name="loop_f64", kind="rk4", n=65_537, topo="spatial", deg=100, f64=True, couple="event", steps=400,
             chunk=50, every=50, hebbian=300),
        # the batched ensemble: 256 networks of 1,024 to 65,536 neurons
        dict(name="ensemble_256", kind="ens", count=256, lo=10.0, hi=16.0, deg=50, steps=500, chunk=100, every=100),
        # the reference's own network with its white noise and electrodes
        dict(name="reference_100k", kind="leap", n=100_003, deg=100, f64=False, couple="count", steps=250, chunk=125,
             every=40, regions=1000, k=50),
        # the reference's default program: 20,000 SCN neurons, each call issued by the caller
        dict(name="scn_20k", kind="scn", n=20_000, deg=30, steps=60, timescale=10, nx=60, ny=50, nz=41),
        # one dense coupling of the headline network at 1% of its neurons firing
        dict(name="pull_1m", kind="pull", n=1 << 20, deg=200, mode="weighted", f64=False, rate=0.01),
        # the headline field solved by itself
        dict(name="cg_256", kind="cg", nx=256, ny=256, nz=256, var=False, c=1.0, precond="jacobi", rtol=1e-8),
        # a ragged field
        dict(name="cg_ragged", kind="cg", nx=150, ny=131, nz=97, var=False, c=5.0, precond="jacobi", rtol=1e-8),
        # variable diffusivity with the plain solver
        dict(name="cgvar_128", kind="cg", nx=128, ny=128, nz=128, var=True, c=50.0, precond="jacobi", rtol=1e-8),
        # variable diffusivity with the multigrid solver
        dict(name="mg_256", kind="cg", nx=256, ny=256, nz=256, var=True, c=50.0, precond="mg", rtol=1e-8),
        # the preconditioner's training step, forward and backward (8 samples of 64^3)
        dict(name="train_64", kind="train", nx=64, ny=64, nz=64, batch=8, smooth=1),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rk4", "rk4", "ens", "leap", "scn", "pull", "cg", "cg", "cg", "train"])
    if kind == "rk4":
        f64 = rng.random() < 0.25
        n = _logint(rng, 256, 200_000 if f64 else 1 << 20)
        couple = rng.choice(["event", "pull"]) if f64 else rng.choice(["fused", "fused", "event"])
        chunk = rng.choice([20, 50, 100])
        steps = chunk * rng.randint(2, 4 if n > 100_000 else 8)
        return dict(kind=kind, n=n, topo=rng.choice(["er", "spatial"]) if n > 4096 else "er",
                    deg=rng.randint(20, 200), f64=f64, couple=couple, steps=steps, chunk=chunk, every=chunk,
                    hebbian=rng.choice([0, 0, 300]))
    if kind == "ens":
        lo = rng.uniform(8.0, 11.0)
        return dict(kind=kind, count=rng.randint(2, 160), lo=lo, hi=rng.uniform(lo + 1.0, 15.0),
                    deg=rng.randint(20, 60), steps=rng.choice([100, 200]), chunk=rng.choice([50, 100]),
                    every=rng.choice([50, 100]))
    if kind == "leap":
        return dict(kind=kind, n=_logint(rng, 500, 500_000), deg=rng.randint(20, 150), f64=rng.random() < 0.3,
                    couple=rng.choice(["count", "signal"]), steps=100, chunk=rng.choice([50, 100]),
                    every=rng.choice([10, 40]), regions=rng.randint(4, 1000), k=rng.randint(3, 60))
    if kind == "scn":
        return dict(kind=kind, n=_logint(rng, 1000, 300_000), deg=rng.randint(10, 60), steps=40,
                    timescale=rng.choice([5, 10, 20]), nx=rng.randint(20, 128), ny=rng.randint(20, 128),
                    nz=rng.randint(20, 128))
    if kind == "pull":
        return dict(kind=kind, n=_logint(rng, 5000, 1_500_000), deg=rng.randint(20, 120),
                    mode=rng.choice(["weighted", "count", "signal"]), f64=rng.random() < 0.3,
                    rate=math.exp(rng.uniform(math.log(0.0005), math.log(0.05))))
    if kind == "train":
        return dict(kind=kind, nx=64 * rng.randint(1, 2), ny=32 * rng.randint(1, 3), nz=32 * rng.randint(1, 3),
                    batch=rng.randint(1, 8), smooth=rng.randint(0, 2))
    if rng.random() < 0.4:
        mg = rng.random() < 0.6
        m = [2 * _logint(rng, 12, 96 if mg else 56) for _ in range(3)]
        if rng.random() < 0.5:
            m = [8 * max(2, v // 8) for v in m]
        return dict(kind=kind, nx=m[0], ny=m[1], nz=m[2], var=True, c=rng.uniform(5.0, 60.0 if mg else 30.0),
                    precond="mg" if mg else "jacobi", rtol=1e-8)
    return dict(kind=kind, nx=_logint(rng, 24, 288), ny=_logint(rng, 24, 288), nz=_logint(rng, 24, 200), var=False,
                c=rng.uniform(0.5, 20.0), precond="jacobi", rtol=1e-8)


# ---------------------------------------------------------------------------
# buffers
# ---------------------------------------------------------------------------
class _Block:
    """Named device arrays in one allocation (each 256-byte aligned), with a
    copy of their initial contents."""

    def __init__(self, ctx, items):
        self.ctx, self.t, at, spans = ctx, {}, 0, {}
        for k, v in items.items():
            b = max(v.numel() * v.element_size(), 8)
            spans[k] = (at, v.numel() * v.element_size())
            at += (b + 255) // 256 * 256
        self.buf = torch.zeros(at, dtype=torch.uint8, device=DEV)
        for k, v in items.items():
            o, b = spans[k]
            self.t[k] = self.buf[o:o + b].view(v.dtype)
            self.t[k].copy_(v.reshape(-1))
        self.init = self.buf.clone()

    def __getitem__(self, k):
        return self.t[k].data_ptr()

    def restore(self):
        self.ctx.call("nnx_memcpy_d2d", self.buf.data_ptr(), self.init.data_ptr(), C.c_size_t(self.buf.numel()))


class _Owner:
    """A state whose captured step graphs go when it goes."""

    def __init__(self, ctx, **kw):
        self.ctx = ctx
        self.__dict__.update(kw)

    def __del__(self):
        try:
            self.ctx.clear_graphs()
        except Exception:
            pass


def _gen(seed, k=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + k + 1)
    return g


def _uni(g, n, lo=0.0, hi=1.0, dtype=F64):
    return torch.rand(n, generator=g, device=DEV, dtype=dtype) * (hi - lo) + lo


def _nrm(g, n, mu=0.0, sd=1.0):
    return torch.randn(n, generator=g, device=DEV, dtype=F64) * sd + mu


def _zeros(n, dtype):
    return torch.zeros(n, dtype=dtype, device=DEV)


# ---------------------------------------------------------------------------
# networks
# ---------------------------------------------------------------------------
def _csr(rows, tgt, n):
    """offsets and targets of (row, target) pairs, targets ascending per row."""
    key, _ = torch.sort(rows * n + tgt)
    off = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(torch.div(key, n, rounding_mode="floor"), minlength=n), 0)
    return off.to(torch.int32), (key % n).to(torch.int32)


def _rows(deg):
    return torch.repeat_interleave(torch.arange(deg.numel(), device=DEV), deg)


def _spatial(g, n, mean):
    """Neurons at uniform positions in a box of 0.5 neurons per unit volume,
    log-normal out-degrees of the given mean, targets at distances with
    density exp(-d / 10) up to 60: the neuron of the displaced cell (or the
    next occupied one)."""
    box = 128.0 * (n / float(1 << 20)) ** (1.0 / 3.0)
    pos = _uni(g, 3 * n, 0.0, box).reshape(n, 3)
    # (the degrees are the network's, whatever the seed: as many synapses)
    deg = torch.exp(_nrm(_gen(0, 1), n, math.log(mean) - 0.125, 0.5)).round().clamp(1, 20000).long()
    nc = max(1, int(box))
    cell = (pos * (nc / box)).long().clamp(0, nc - 1)
    cid = cell[:, 0] + nc * (cell[:, 1] + nc * cell[:, 2])
    cs, order = torch.sort(cid)
    rows = _rows(deg)
    tgt = torch.empty_like(rows)
    for a in range(0, rows.numel(), 1 << 25):
        r = rows[a:a + (1 << 25)]
        m = r.numel()
        # a radius with density r^2 exp(-r / 10): the sum of three exponentials
        d = (-10.0 * torch.log(_uni(g, 3 * m).reshape(3, m).clamp_min(1e-300))).sum(0).clamp_max(min(60.0, box))
        w = _nrm(g, 3 * m).reshape(m, 3)
        p = pos[r] + w * (d / w.norm(dim=1).clamp_min(1e-30))[:, None]
        p = torch.where(p < 0, -p, p)
        p = torch.where(p >= box, 2 * box - p, p).clamp(0.0, box * (1 - 1e-9))
        q = (p * (nc / box)).long().clamp(0, nc - 1)
        at = torch.searchsorted(cs, q[:, 0] + nc * (q[:, 1] + nc * q[:, 2])) + (r % 2)
        tgt[a:a + m] = order[at.clamp_max(n - 1)]
    off, tg = _csr(rows, tgt, n)
    grid = max(8, int(round(2.0 * box)))
    v = (pos * (grid / box)).long().clamp(0, grid - 1)
    return off, tg, (v[:, 0] + grid * (v[:, 1] + grid * v[:, 2])).to(torch.int32), grid


def _transpose(ctx, off, tgt, w, deg=None):
    """The CSC side and its graph struct (nnx_graph_transpose)."""
    n, nnz = off.numel() - 1, tgt.numel()
    d = {"off": off, "tgt": tgt, "w": w, "in_off": _zeros(n + 1, torch.int32), "in_src": _zeros(nnz, torch.int32),
         "in_w": _zeros(nnz, torch.float32), "o2i": _zeros(nnz, torch.int32)}
    torch.cuda.synchronize()
    ctx.call("nnx_graph_transpose", n, nnz, off.data_ptr(), tgt.data_ptr(), w.data_ptr(), d["in_off"].data_ptr(),
             d["in_src"].data_ptr(), d["in_w"].data_ptr(), d["o2i"].data_ptr(),
             _lib.F64 if deg is not None and deg.dtype == F64 else _lib.F32,
             None if deg is None else deg.data_ptr())
    ctx.synchronize()
    return d, _lib.Graph(n=n, nnz=nnz, out_offsets=off.data_ptr(), out_targets=tgt.data_ptr(),
                         out_weights=w.data_ptr(), in_offsets=d["in_off"].data_ptr(),
                         in_sources=d["in_src"].data_ptr(), in_weights=d["in_w"].data_ptr(),
                         out_to_in=d["o2i"].data_ptr())


def _gates(V):
    u = V + 5.0
    a, b = 0.1 * u + 3.5, 0.1 * u + 5.0
    am, an = -a / torch.expm1(-a), -0.1 * b / torch.expm1(-b)
    bh = 1.0 / (torch.exp(-3.0 - 0.1 * u) + 1.0)
    w = u + 60.0
    return am, 4.0 * torch.exp(-w / 18.0), 0.07 * torch.exp(-u / 20.0 - 3.0), bh, an, 0.125 * torch.exp(-w / 80.0)


def _rk4_inputs(case, seed):
    """Connectivity, drive, initial state and field of an rk4 case (FP64
    values of what the network holds in its own type)."""
    g = _gen(seed)
    n = case["n"]
    if case["topo"] == "spatial":
        off, tgt, vox, grid = _spatial(g, n, case["deg"])
        w = torch.exp(_nrm(g, tgt.numel(), -3.0, 1.0)).float()
    else:
        rows = _rows(torch.full((n,), case["deg"], dtype=torch.int64, device=DEV))
        off, tgt = _csr(rows, torch.randint(n, rows.shape, generator=g, device=DEV), n)
        grid = 32
        vox = torch.randint(grid ** 3, (n,), generator=g, device=DEV, dtype=torch.int32)
        w = _uni(g, tgt.numel(), 0.0, 0.1).float()
    T = F64 if case["f64"] else torch.float32
    V = _uni(g, n, -70.0, -60.0)
    am, bm, ah, bh, an, bn = _gates(V)
    st = {"v": V, "m": am / (am + bm), "h": ah / (ah + bh), "ng": an / (an + bn), "s": torch.zeros_like(V),
          "i_ext": _nrm(g, n, 10.0, 2.0)}
    return off, tgt, w, vox, grid, {k: v.to(T) for k, v in st.items()}, T


def _hh_state(case_n, blk, iext, T, keys):
    return _lib.HHState(dtype=_lib.F64 if T == F64 else _lib.F32, n=case_n, i_ext=iext, **{k: blk[k] for k in keys})


STATE = ("v", "m", "h", "ng", "s")
COUPLE = {"fused": _lib.COUPLE_WEIGHTED_FUSED, "event": _lib.COUPLE_WEIGHTED_EVENT,
          "pull": _lib.COUPLE_WEIGHTED_PULL, "count": _lib.COUPLE_COUNT, "signal": _lib.COUPLE_SIGNAL}


def _set_paracrine(q, every, dims, c, blk, block=0):
    q.every = every
    q.grid = _lib.Grid(dims[0], dims[1], dims[2], _lib.STENCIL_7, c, 0.0, None, None, None, block)
    q.release, q.rtol, q.inner_rtol, q.max_inner, q.max_outer = 0.01, 1e-8, 1e-6, 32, 2
    q.conc, q.stats = blk["conc"], blk["stats"]


def _prepare_rk4(case, seed):
    ctx = _lib.context()
    off, tgt, w, vox, grid, st, T = _rk4_inputs(case, seed)
    n, nw, nnz = case["n"], (case["n"] + 63) // 64, tgt.numel()
    gd, graph = _transpose(ctx, off, tgt, w)
    items = {k: st[k] for k in STATE}
    items.update(bits0=_zeros(nw, torch.int64), bits1=_zeros(nw, torch.int64), list=_zeros(n, torch.int32),
                 count=_zeros(1, torch.int32), raster_len=_zeros(1, torch.int64),
                 voxel_counts=_zeros(grid ** 3, torch.int32), conc=_zeros(grid ** 3, F64), stats=_zeros(8, F64),
                 g_in=_zeros(n, T))
    cap = max(4 * n, 1 << 16)
    raster = _zeros(2 * cap, torch.int32)
    if case["hebbian"]:
        items.update(heb_w=w, armed=_zeros(nnz, torch.uint8), last_fire=_zeros(n, torch.int32),
                     ring=_zeros(case["hebbian"] * nw, torch.int64))
    o2i = torch.zeros(nnz, dtype=torch.int32, device=DEV)
    blk = _Block(ctx, items)
    p = _lib.StepPlan()
    p.state = _hh_state(n, blk, st["i_ext"].data_ptr(), T, STATE)
    p.params = _lib.params_squid()
    p.graph = graph
    p.integrator, p.spike_rule, p.couple_mode, p.record = _lib.INT_RK4, _lib.SPIKE_CROSSING, COUPLE[case["couple"]], 1
    p.dt = 0.01
    p.g_in, p.list, p.count = blk["g_in"], blk["list"], blk["count"]
    p.bits[0], p.bits[1] = blk["bits0"], blk["bits1"]
    p.voxel_of, p.voxel_counts = vox.data_ptr(), blk["voxel_counts"]
    p.raster, p.raster_len, p.raster_cap = raster.data_ptr(), blk["raster_len"], cap
    _set_paracrine(p.paracrine, case["every"], (grid,) * 3, 1.0, blk)
    if case["hebbian"]:
        h = p.hebbian
        h.window, h.heb_inc, h.weights = case["hebbian"], 0.1, blk["heb_w"]
        h.armed, h.last_fire, h.ring, h.in_to_out = blk["armed"], blk["last_fire"], blk["ring"], o2i.data_ptr()
        ctx.call("nnx_hebbian_init", C.byref(graph), C.byref(h))
        ctx.synchronize()
        blk.init.copy_(blk.buf)  # with the cleared learning state
    torch.cuda.synchronize()
    return _Owner(ctx, case=case, plan=p, blk=blk, keep=(gd, vox, raster, st, o2i), raster=raster)


def _run_rk4(s):
    case, blk = s.case, s.blk
    blk.restore()
    for at in range(0, case["steps"], case["chunk"]):
        s.ctx.call("nnx_run_steps", C.byref(s.plan), at, case["chunk"], 1)
    names = STATE + ("bits0", "bits1", "count", "raster_len", "voxel_counts", "conc")
    out = {k: blk.t[k] for k in names + (("heb_w", "armed") if case["hebbian"] else ())}
    if case["couple"] != "fused":  # (the fused step appends a step's spikes in no stated order)
        out["raster"] = s.raster
    return out


# ---------------------------------------------------------------------------
# the ensemble
# ---------------------------------------------------------------------------
def _ens_sizes(case):
    u = host.uniform(0, 106, case["count"], case["lo"], case["hi"])
    sizes = np.rint(2.0 ** u).astype(np.int64)
    begin = np.zeros(len(sizes), np.int64)
    begin[1:] = np.cumsum((sizes + 63) // 64 * 64)[:-1]
    return sizes, begin, int(begin[-1] + (sizes[-1] + 63) // 64 * 64)


def _lattice(count):
    a = max(1, min(4, count))
    b = max(1, min(4, -(-count // a)))
    return a, b, max(1, -(-count // (a * b)))


def _ens_inputs(case, seed):
    g = _gen(seed)
    sizes, begin, n = _ens_sizes(case)
    lat = _lattice(len(sizes))
    net = torch.zeros(n, dtype=torch.int64, device=DEV)
    live = torch.zeros(n, dtype=torch.bool, device=DEV)
    for i, (b, s) in enumerate(zip(begin, sizes)):
        net[b:b + (s + 63) // 64 * 64] = i
        live[b:b + s] = True
    sz, bg = torch.from_numpy(sizes).to(DEV), torch.from_numpy(begin).to(DEV)
    deg = torch.poisson(torch.full((n,), float(case["deg"]), device=DEV), generator=g).long() * live
    rows = _rows(deg)
    tgt = bg[net[rows]] + (_uni(g, rows.numel()) * sz[net[rows]]).long()
    off, tgt = _csr(rows, tgt, n)
    w = _uni(g, tgt.numel(), 0.0, 0.1).float()
    V = torch.where(live, _uni(g, n, -70.0, -60.0), torch.full((n,), -65.0, dtype=F64, device=DEV))
    am, bm, ah, bh, an, bn = _gates(V)
    mu = _uni(g, len(sizes), 6.0, 14.0)
    st = {"v": V, "m": am / (am + bm), "h": ah / (ah + bh), "ng": an / (an + bn), "s": torch.zeros_like(V),
          "i_ext": (_nrm(g, n, 0.0, 2.0) + mu[net]) * live}
    q = torch.randint(64, (3, n), generator=g, device=DEV)
    nx, ny = 64 * lat[0], 64 * lat[1]
    x = q[0] + 64 * (net % lat[0])
    y = q[1] + 64 * (torch.div(net, lat[0], rounding_mode="floor") % lat[1])
    z = q[2] + 64 * torch.div(net, lat[0] * lat[1], rounding_mode="floor")
    vox = (x + nx * (y + ny * z)).to(torch.int32)
    return sizes, begin, n, lat, off, tgt, w, vox, {k: v.float() for k, v in st.items()}, live


def _prepare_ens(case, seed):
    ctx = _lib.context()
    sizes, begin, n, lat, off, tgt, w, vox, st, _ = _ens_inputs(case, seed)
    gd, graph = _transpose(ctx, off, tgt, w)
    dims = tuple(64 * k for k in lat)
    nv = dims[0] * dims[1] * dims[2]
    items = {k: st[k] for k in STATE}
    items.update(bits0=_zeros(n // 64, torch.int64), bits1=_zeros(n // 64, torch.int64),
                 net_spikes=_zeros(len(sizes), torch.int32), voxel_counts=_zeros(nv, torch.int32),
                 conc=_zeros(nv, F64), stats=_zeros(8, F64))
    blk = _Block(ctx, items)
    p = _lib.EnsPlan()
    p.state = _hh_state(n, blk, st["i_ext"].data_ptr(), torch.float32, STATE)
    p.params = _lib.params_squid()
    p.graph = graph
    p.nnet, p.net_begin, p.net_size = len(sizes), begin.ctypes.data, sizes.ctypes.data
    p.dt = 0.01
    p.bits[0], p.bits[1], p.net_spikes = blk["bits0"], blk["bits1"], blk["net_spikes"]
    p.voxel_of, p.voxel_counts = vox.data_ptr(), blk["voxel_counts"]
    _set_paracrine(p.paracrine, case["every"], dims, 1.0, blk, block=64)
    torch.cuda.synchronize()
    return _Owner(ctx, case=case, plan=p, blk=blk, keep=(gd, vox, st, sizes, begin))


def _run_ens(s):
    case, blk = s.case, s.blk
    blk.restore()
    for at in range(0, case["steps"], case["chunk"]):
        s.ctx.call("nnx_ensemble_run", C.byref(s.plan), None, at, case["chunk"], 1)
    return {k: blk.t[k] for k in STATE + ("bits0", "bits1", "net_spikes", "voxel_counts", "conc")}


# ---------------------------------------------------------------------------
# the reference's network (leapfrog)
# ---------------------------------------------------------------------------
LEAP = ("v", "m", "h", "ng", "y_local", "y_i", "y_e", "out_local", "out_i", "out_e")


def _er(g, n, deg):
    rows = _rows(torch.full((n,), deg, dtype=torch.int64, device=DEV))
    return _csr(rows, torch.randint(n, rows.shape, generator=g, device=DEV), n)


def _prepare_leap(case, seed):
    ctx, g = _lib.context(), _gen(seed)
    n, nw, T = case["n"], (case["n"] + 63) // 64, F64 if case["f64"] else torch.float32
    off, tgt = _er(g, n, case["deg"])
    w = torch.ones(tgt.numel(), device=DEV)
    indeg = _zeros(n, T)
    gd, graph = _transpose(ctx, off, tgt, w, indeg)
    items = {k: _zeros(n, T) for k in LEAP + ("in_local",)}
    items["v"] = _nrm(g, n, -55.0, 25.0).to(T)
    rows = case["steps"] // case["every"] + 1
    items.update(bits0=_zeros(nw, torch.int64), bits1=_zeros(nw, torch.int64), list=_zeros(n, torch.int32),
                 count=_zeros(1, torch.int32), avg=_zeros(rows * case["regions"], T),
                 firing=_zeros(rows * case["regions"], torch.int32), mean=_zeros(rows, T))
    blk = _Block(ctx, items)
    const = {"appcur": _nrm(g, n, 0.0, 2.0).to(T), "zero": _zeros(n, T), "indeg": indeg}
    k = case["k"]
    r_off = torch.arange(0, k * case["regions"] + 1, k, dtype=torch.int32, device=DEV)
    r_idx = torch.randint(n, (k * case["regions"],), generator=g, device=DEV, dtype=torch.int32)
    z, ptr = const["zero"].data_ptr(), {m: const[m].data_ptr() for m in const}
    p = _lib.StepPlan()
    p.state = _lib.HHState(dtype=_lib.F64 if T == F64 else _lib.F32, n=n, appcur=ptr["appcur"],
                           in_local=blk["in_local"], count_local=ptr["indeg"], in_i=z, count_i=z, in_e=z, count_e=z,
                           **{m: blk[m] for m in LEAP})
    p.params = _lib.params_reference()
    p.params.noise_seed = seed + 1
    p.graph = graph
    p.integrator, p.spike_rule, p.couple_mode = _lib.INT_LEAPFROG, _lib.SPIKE_LEVEL, COUPLE[case["couple"]]
    p.dt = 0.4
    p.bits[0], p.bits[1], p.list, p.count = blk["bits0"], blk["bits1"], blk["list"], blk["count"]
    p.regions = _lib.Regions(n_regions=case["regions"], nnz=r_idx.numel(), offsets=r_off.data_ptr(),
                             idx=r_idx.data_ptr())
    p.readout_every, p.readout_cap = case["every"], rows
    p.readout_avg, p.readout_firing, p.readout_mean = blk["avg"], blk["firing"], blk["mean"]
    torch.cuda.synchronize()
    return _Owner(ctx, case=case, plan=p, blk=blk, keep=(gd, const, r_off, r_idx))


def _run_leap(s):
    case, blk = s.case, s.blk
    blk.restore()
    for at in range(0, case["steps"], case["chunk"]):
        s.ctx.call("nnx_run_steps", C.byref(s.plan), at, case["chunk"], 1)
    return {k: blk.t[k] for k in LEAP + ("in_local", "bits0", "bits1", "count", "avg", "firing", "mean")}


# ---------------------------------------------------------------------------
# the reference's default program (Diekman neurons, call by call)
# ---------------------------------------------------------------------------
DK = ("v", "m", "h", "ng", "rl", "rnl", "fnl", "s", "p", "y", "cas", "cac")
SCN = dict(h=1.0, D=0.5, decay=0.1, par_dt=0.4, coup=0.05)


def _scn_inputs(case, seed):
    g = _gen(seed)
    n, e = case["n"], torch.exp
    off, tgt = _er(g, n, case["deg"])
    V = _uni(g, n, -70.0, -40.0)
    V = torch.where(_uni(g, n) < 0.05, _uni(g, n, -20.0, 10.0), V)  # some are firing
    st = {"v": V, "m": 1 / (1 + e(-(V + 35.2) / 8.1)), "h": 1 / (1 + e((V + 62) / 2)),
          "ng": (1 + e((V - 14) / -17.0)) ** -0.25, "rl": 1 / (1 + e(-(V + 36) / 5.1)),
          "rnl": 1 / (1 + e(-(V + 21.6) / 6.7)), "fnl": 1 / (1 + e((V + 260) / 65)), "s": torch.zeros_like(V),
          "p": (1 + e(-(V + 25) / 7.4)) ** -1.5, "y": torch.zeros_like(V), "cas": torch.full_like(V, 1e-4),
          "cac": torch.full_like(V, 1e-4), "ioutput": 1 / (1 + e(-(V + 20) / 3.0))}
    const = {"egaba": torch.full_like(V, -60.0), "gkca": _nrm(g, n, 100.0, 0.5), "gkleak": _nrm(g, n, 0.12, 0.01)}
    dims = (case["nx"], case["ny"], case["nz"])
    # x / ((n - 1) h) + 0.5 in [0, 1]: positions centred on the grid
    pos = [(_uni(g, n, -0.5, 0.5) * ((m - 1) * SCN["h"])).float().cpu().numpy() for m in dims]
    return off, tgt, {k: v.float() for k, v in st.items()}, {k: v.float() for k, v in const.items()}, dims, pos


def _prepare_scn(case, seed):
    ctx = _lib.context()
    off, tgt, st, const, dims, pos = _scn_inputs(case, seed)
    n, nw = case["n"], (case["n"] + 63) // 64
    G = dims[0] * dims[1] * dims[2]
    w = torch.ones(tgt.numel(), device=DEV)
    indeg = _zeros(n, torch.float32)
    gd, graph = _transpose(ctx, off, tgt, w, indeg)
    wo, wc, wv, _ = host.trilinear_matrix(pos[0], pos[1], pos[2], *dims, SCN["h"])
    so, sc, sv = host.csr_transpose(n, G, wo, wc, wv)
    tri = [torch.from_numpy(np.ascontiguousarray(a)).to(DEV) for a in (wo, wc, wv, so, sc, sv)]
    items = dict(st)
    items.update(iin=_zeros(n, torch.float32), bits=_zeros(nw, torch.int64), list=_zeros(n, torch.int32),
                 count=_zeros(1, torch.int32), release=_zeros(n, torch.float32), density=_zeros(G, torch.float32),
                 at_neurons=_zeros(n, torch.float32))
    blk = _Block(ctx, items)
    dk = _lib.DiekmanState(dtype=_lib.F32, n=n, iin=blk["iin"], icount=indeg.data_ptr(), ioutput=blk["ioutput"],
                           **{k: const[k].data_ptr() for k in const}, **{k: blk[k] for k in DK})
    torch.cuda.synchronize()
    return _Owner(ctx, case=case, blk=blk, graph=graph, dk=dk, par=_lib.params_diekman(), res=_lib.CgResult(),
                  tri=[t.data_ptr() for t in tri], dims=dims, G=G, keep=(gd, indeg, const, tri))


def _run_scn(s):
    case, blk, call = s.case, s.blk, s.ctx.call
    n, t = case["n"], s.tri
    blk.restore()
    for i in range(case["steps"]):
        call("nnx_spike_threshold", _lib.F32, n, blk["ioutput"], s.par.out_thresh, blk["bits"])
        call("nnx_spike_compact", n, blk["bits"], blk["list"], blk["count"])
        call("nnx_couple", C.byref(s.graph), _lib.COUPLE_COUNT, _lib.F32, blk["bits"], blk["list"], blk["count"], None,
             blk["iin"])
        if i % case["timescale"] == 0:
            call("nnx_csr_spmv", s.G, t[3], t[4], t[5], blk["release"], blk["density"], 1)
            call("nnx_update_density_reference", *s.dims, SCN["h"], SCN["D"], SCN["decay"], SCN["par_dt"], 1e-6, 20,
                 blk["density"], C.byref(s.res))
            call("nnx_csr_spmv", n, t[0], t[1], t[2], blk["density"], blk["at_neurons"], 0)
            call("nnx_memset", blk["release"], 0, C.c_size_t(4 * n))
        call("nnx_release_add", blk["list"], blk["count"], SCN["coup"], blk["release"])
        call("nnx_diekman_step", C.byref(s.dk), C.byref(s.par), 0.1, blk["bits"])
    return {k: blk.t[k] for k in DK + ("ioutput", "iin", "bits", "count", "release", "density", "at_neurons")}


# ---------------------------------------------------------------------------
# one dense coupling
# ---------------------------------------------------------------------------
def _pull_inputs(case, seed):
    g = _gen(seed)
    n = case["n"]
    off, tgt = _er(g, n, case["deg"])
    w = torch.exp(_nrm(g, tgt.numel(), -3.0, 1.0)).float()
    fire = _uni(g, n) < case["rate"]
    out = _uni(g, n, 0.1, 1.0).to(F64 if case["f64"] else torch.float32)
    return off, tgt, w, fire, out


def _pack_bits(fire):
    n = fire.numel()
    f = torch.zeros((n + 63) // 64 * 64, dtype=torch.int64, device=DEV)
    f[:n] = fire
    return (f.reshape(-1, 64) << torch.arange(64, device=DEV)).sum(1)


def _prepare_pull(case, seed):
    ctx = _lib.context()
    off, tgt, w, fire, out = _pull_inputs(case, seed)
    gd, graph = _transpose(ctx, off, tgt, w)
    bits = _pack_bits(fire)
    lst = torch.nonzero(fire).flatten().to(torch.int32)
    lst = torch.cat([lst, _zeros(case["n"] - lst.numel(), torch.int32)])
    cnt = fire.sum().to(torch.int32).reshape(1)
    g_in = torch.zeros_like(out)
    mode = {"weighted": "pull"}.get(case["mode"], case["mode"])
    torch.cuda.synchronize()
    return _Owner(ctx, graph=graph, mode=COUPLE[mode], dt=_lib.F64 if case["f64"] else _lib.F32, bits=bits, lst=lst,
                  cnt=cnt, out=out, g_in=g_in, keep=gd)


def _run_pull(s):
    s.ctx.call("nnx_couple", C.byref(s.graph), s.mode, s.dt, s.bits.data_ptr(), s.lst.data_ptr(), s.cnt.data_ptr(),
               s.out.data_ptr(), s.g_in.data_ptr())
    return s.g_in


# ---------------------------------------------------------------------------
# one field
# ---------------------------------------------------------------------------
def _faces(c):
    """Harmonic-mean faces of a coefficient field [..., z, y, x] (fp32), the
    boundary faces at their voxel's value."""
    def along(ax):
        a, b = c.narrow(ax, 0, c.shape[ax] - 1).double(), c.narrow(ax, 1, c.shape[ax] - 1).double()
        return torch.cat([c.narrow(ax, 0, 1), (2 * a * b / (a + b)).float(), c.narrow(ax, c.shape[ax] - 1, 1)],
                         ax).contiguous()
    return along(c.dim() - 1), along(c.dim() - 2), along(c.dim() - 3)


def _coeff(g, shape, cbar, corr=8.0, sigma=1.0):
    """Log-normal coefficients: a unit Gaussian field of the given correlation length."""
    x = torch.randn(shape, generator=g, device=DEV, dtype=F64)
    f = torch.fft.fftn(x, dim=(-3, -2, -1))
    for ax in (-3, -2, -1):
        k = torch.fft.fftfreq(shape[ax], device=DEV, dtype=F64)
        v = [1] * len(shape)
        v[ax] = shape[ax]
        f = f * torch.exp(-(2 * math.pi * k * corr) ** 2 / 4.0).reshape(v)
    x = torch.fft.ifftn(f, dim=(-3, -2, -1)).real
    d = torch.exp(sigma * (x - x.mean()) / x.std())
    return (cbar * d / d.mean()).float(), x


def _cg_inputs(case, seed):
    g = _gen(seed)
    shape = (case["nz"], case["ny"], case["nx"])
    n = shape[0] * shape[1] * shape[2]
    # the releases of a few hundred steps: 0.01 at random voxels
    k = max(8, n // 16)
    b = 0.01 * torch.bincount(torch.randint(n, (k,), generator=g, device=DEV), minlength=n).double()
    return b, _faces(_coeff(g, shape, case["c"])[0]) if case["var"] else None


def _prepare_cg(case, seed):
    ctx = _lib.context()
    b, faces = _cg_inputs(case, seed)
    x = torch.zeros_like(b)
    k = [f.data_ptr() for f in faces] if faces else [None] * 3
    grid = _lib.Grid(case["nx"], case["ny"], case["nz"], _lib.STENCIL_7, 0.0 if faces else case["c"], 0.0, *k)
    o = _lib.CgOpts(rtol=case["rtol"], maxit=20000, check_every=8, stall_iters=10, smooth=1,
                    precond=_lib.PRECOND_MG if case["precond"] == "mg" else _lib.PRECOND_JACOBI)
    torch.cuda.synchronize()
    return _Owner(ctx, case=case, b=b, x=x, grid=grid, o=o, res=_lib.CgResult(), keep=faces)


def _run_cg(s):
    if s.case["precond"] == "mg":
        s.ctx.call("nnx_fcg_solve_refine", C.byref(s.grid), None, None, s.b.data_ptr(), s.x.data_ptr(), C.byref(s.o),
                   1e-6, 30, C.byref(s.res))
    else:
        s.ctx.call("nnx_cg_solve_refine", C.byref(s.grid), s.b.data_ptr(), s.x.data_ptr(), C.byref(s.o), 1e-6, 30,
                   C.byref(s.res))
    return s.x


# ---------------------------------------------------------------------------
# training step
# ---------------------------------------------------------------------------
LAYERS = ((2, 16), (16, 32), (32, 32), (32, 16), (16, 16))


def _train_inputs(case, seed):
    g = _gen(seed)
    shape = (case["batch"], case["nz"], case["ny"], case["nx"])
    c, x = _coeff(g, shape, 50.0)
    faces = _faces(c)
    feat = ((x - x.mean()) / x.std()).float()
    # what a smoother leaves of an error: smooth, with a rough remainder
    e = _coeff(g, shape, 1.0, corr=4.0)[1]
    e = (e / e.std() + 0.05 * torch.randn(shape, generator=g, device=DEV, dtype=F64)).float()
    r = _apply_var(e.double(), *(f.double() for f in faces)).float()
    w = []
    for ci, co in LAYERS:
        lim = math.sqrt(6.0 / (27 * ci))
        w += [_uni(g, co * 27 * ci, -lim, lim), _zeros(co, F64)]
    w += [_uni(g, 16, -0.5, 0.5), _zeros(1, F64)]
    return r, feat, e, faces, torch.cat(w).float()


class _Net(_Owner):
    def __del__(self):
        try:
            self.ctx.call("nnx_unet_destroy", self.h)
        except Exception:
            pass


def _prepare_train(case, seed):
    ctx = _lib.context()
    r, feat, e, faces, w = _train_inputs(case, seed)
    h, hw = C.c_void_p(), w.cpu().numpy()
    ctx.call("nnx_unet_create", hw.ctypes.data_as(C.c_void_p), 0, C.byref(h))
    torch.cuda.synchronize()
    return _Net(ctx, case=case, h=h, r=r, feat=feat, e=e, faces=faces, grad=np.empty(hw.size, np.float32),
                params=np.empty(hw.size, np.float32))


def _run_train(s):
    case = s.case
    loss = C.c_double()
    s.ctx.call("nnx_unet_train_step", s.h, case["nx"], case["ny"], case["nz"], case["batch"], s.r.data_ptr(),
               s.feat.data_ptr(), s.e.data_ptr(), *(f.data_ptr() for f in s.faces), case["smooth"], 1.5e-4,
               C.byref(loss))
    s.ctx.call("nnx_unet_get_grad", s.h, s.grad.ctypes.data_as(C.c_void_p))
    s.ctx.call("nnx_unet_get_params", s.h, s.params.ctypes.data_as(C.c_void_p))
    return {"grad": s.grad.copy(), "params": s.params.copy(), "loss": loss.value}


# ---------------------------------------------------------------------------
PREPARE = dict(rk4=_prepare_rk4, ens=_prepare_ens, leap=_prepare_leap, scn=_prepare_scn, pull=_prepare_pull,
               cg=_prepare_cg, train=_prepare_train)
RUN = dict(rk4=_run_rk4, ens=_run_ens, leap=_run_leap, scn=_run_scn, pull=_run_pull, cg=_run_cg, train=_run_train)


def prepare(case, seed):
    return case["kind"], PREPARE[case["kind"]](case, seed)


def run(state):
    return RUN[state[0]](state[1])


def work(case):
    k = case["kind"]
    if k in ("rk4", "ens"):
        if k == "rk4":
            n = case["n"]
            box = 128.0 * (n / float(1 << 20)) ** (1.0 / 3.0)
            nv = (max(8, int(round(2.0 * box))) if case["topo"] == "spatial" else 32) ** 3
            e = 8 if case["f64"] else 4
        else:
            _, _, n = _ens_sizes(case)
            lat = _lattice(case["count"])
            nv, e = 64 ** 3 * lat[0] * lat[1] * lat[2], 4
        steps = case["steps"]
        solves = steps // case["every"]
        # state in and out every step, one spike per neuron and 2,000 steps over its out-edges, and per solve the
        # field and its right-hand side in FP64 with 20 iterations over the unknown, direction and residual
        b = steps * (11.0 * e * n + n / 8.0 + n / 2000.0 * case["deg"] * 12.0) + solves * nv * (20.0 + 20 * 20.0)
        return {"bytes": b, "flops": steps * n * 500.0 + solves * nv * 20 * 20.0}
    if k == "leap":
        e, n = 8 if case["f64"] else 4, case["n"]
        return {"bytes": case["steps"] * (24.0 * e * n + 4.0 * n * case["deg"]), "flops": case["steps"] * n * 600.0}
    if k == "scn":
        G = case["nx"] * case["ny"] * case["nz"]
        ups = -(-case["steps"] // case["timescale"])
        return {"bytes": case["steps"] * (120.0 * case["n"] + 4.0 * case["n"] * case["deg"]) + ups * G * 4.0 * 30,
                "flops": case["steps"] * case["n"] * 700.0 + ups * G * 300.0}
    if k == "pull":
        E, n = case["n"] * case["deg"], case["n"]
        return {"bytes": 4.0 * E * (1.0 + case["rate"]) + n * ((8 if case["f64"] else 4) + 4.125),
                "flops": E * case["rate"]}
    if k == "cg":
        nv = case["nx"] * case["ny"] * case["nz"]
        # iterations to 1e-8 grow with the square root of the condition number
        it = 20.0 if case["precond"] == "mg" else 7.0 * math.sqrt(1.0 + 12.0 * case["c"] * (20.0 if case["var"] else 1))
        return {"bytes": nv * (16.0 + it * (32.0 if case["var"] else 20.0)), "flops": nv * it * 24.0}
    nv = case["nx"] * case["ny"] * case["nz"] * case["batch"]
    f = sum(54.0 * ci * co / s for (ci, co), s in zip(LAYERS, (1, 8, 64, 8, 1)))
    return {"bytes": nv * (4.0 * 6 + 32.0 * 2 * 2), "flops": 3.0 * nv * f}


def tolerance(case):
    k = case["kind"]
    if k in ("rk4", "ens"):
        # the trajectory is a fixed sequence of roundings and stays the same; the field is solved to a true relative
        # residual of 1e-8, and another solve that meets it is that far away
        return {"rel": 1e-7, "max": 1e-5}
    if k == "leap":
        return {"rel": 1e-12 if case["f64"] else 1e-6, "max": 1e-10 if case["f64"] else 1e-4}
    if k == "scn":
        # fp32 states; the update stops on its residual, a few 1e-5 of a small field
        return {"rel": 1e-4, "max": 1e-2}
    if k == "pull":
        return {"rel": 1e-12 if case["f64"] else 1e-6}
    if k == "cg":
        # two solves to a true 1e-8; the smooth parts of the error weigh up to the condition number
        return {"rel": 2e-6 if case["var"] else 2e-7, "max": 1e-3}
    # bf16 activations and weights, fp32 sums
    return {"rel": 1.5e-2, "max": 0.5}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _sine(n):
    i = torch.arange(1, n + 1, dtype=F64, device=DEV)
    S = math.sqrt(2.0 / (n + 1)) * torch.sin(math.pi * i[:, None] * i[None, :] / (n + 1))
    return S, 2.0 - 2.0 * torch.cos(math.pi * i / (n + 1))


def _along(x, S, ax):
    return torch.tensordot(x, S, dims=([ax], [0])).movedim(-1, ax)


def _dst_solve(b, c, axes):
    """(I - c L) x = b, Dirichlet 0 on the box spanned by `axes` (the other axes: independent boxes)."""
    lam = torch.ones([1] * b.dim(), dtype=F64, device=DEV)
    x = b
    mats = []
    for ax in axes:
        S, t = _sine(b.shape[ax])
        v = [1] * b.dim()
        v[ax] = b.shape[ax]
        lam = lam + c * t.reshape(v)
        mats.append(S)
        x = _along(x, S, ax)
    x = x / lam
    for ax, S in zip(axes, mats):
        x = _along(x, S, ax)
    return x


def _apply_var(x, kx, ky, kz):
    y = x * (1 + kx[..., 1:] + kx[..., :-1] + ky[..., 1:, :] + ky[..., :-1, :] + kz[..., 1:, :, :] + kz[..., :-1, :, :])
    f = kx[..., 1:-1]
    y[..., 1:] -= f * x[..., :-1]
    y[..., :-1] -= f * x[..., 1:]
    f = ky[..., 1:-1, :]
    y[..., 1:, :] -= f * x[..., :-1, :]
    y[..., :-1, :] -= f * x[..., 1:, :]
    f = kz[..., 1:-1, :, :]
    y[..., 1:, :, :] -= f * x[..., :-1, :, :]
    y[..., :-1, :, :] -= f * x[..., 1:, :, :]
    return y


def _exact_cg(case, seed):
    b, faces = _cg_inputs(case, seed)
    b = b.reshape(case["nz"], case["ny"], case["nx"])
    if not faces:
        return _dst_solve(b, case["c"], (0, 1, 2)).reshape(-1)
    k = [f.double() for f in faces]
    di = 1 / (1 + k[0][..., 1:] + k[0][..., :-1] + k[1][:, 1:] + k[1][:, :-1] + k[2][1:] + k[2][:-1])
    x, r = torch.zeros_like(b), b.clone()
    z = r * di
    p, rz, bb = z.clone(), (r * z).sum(), b.norm()
    for it in range(9000):
        q = _apply_var(p, *k)
        a = rz / (p * q).sum()
        x += a * p
        r -= a * q
        if it % 50 == 0 and float(r.norm()) <= 1e-12 * float(bb):
            break
        z = r * di
        new = (r * z).sum()
        p = z + (new / rz) * p
        rz = new
    return x.reshape(-1)


def _rk4_step(y, s0, sh, sf, iext):
    def f(V, m, h, n, s):
        am, bm, ah, bh, an, bn = _gates(V)
        i = iext - 120.0 * m ** 3 * h * (V - 50.0) - 36.0 * n ** 4 * (V + 77.0) - 0.3 * (V + 54.4) - s * V
        return i, am * (1 - m) - bm * m, ah * (1 - h) - bh * h, an * (1 - n) - bn * n
    dt = 0.01
    k1 = f(*y, s0)
    k2 = f(*(a + 0.5 * dt * b for a, b in zip(y, k1)), sh)
    k3 = f(*(a + 0.5 * dt * b for a, b in zip(y, k2)), sh)
    k4 = f(*(a + dt * b for a, b in zip(y, k3)), sf)
    return [a + dt / 6 * (p + 2 * q + 2 * r + t) for a, p, q, r, t in zip(y, k1, k2, k3, k4)]


def _exact_network(case, off, tgt, w, vox, st, shape, axes):
    n = off.numel() - 1
    off, tgt, w = off.long(), tgt.long(), w.double()
    st = {k: v.double() for k, v in st.items()}
    y, s = [st["v"], st["m"], st["h"], st["ng"]], st["s"]
    nv = math.prod(shape)
    counts, conc, spk = _zeros(nv, F64), _zeros(nv, F64), None
    eh, ef = math.exp(-0.01 / 4.0), math.exp(-0.01 / 2.0)
    for t in range(case["steps"]):
        g = _zeros(n, F64)
        if spk is not None and spk.numel():
            d = off[spk + 1] - off[spk]
            e = torch.repeat_interleave(off[spk] - torch.cumsum(d, 0) + d, d) + torch.arange(int(d.sum()), device=DEV)
            g.index_add_(0, tgt[e], w[e])
        if t % case["every"] == 0:
            conc = _dst_solve((conc + 0.01 * counts).reshape(shape), 1.0, axes).reshape(-1)
            counts.zero_()
        s0 = s + g
        v0 = y[0]
        y = _rk4_step(y, s0, s0 * eh, s0 * ef, st["i_ext"])
        s = s0 * ef
        spk = torch.nonzero((v0 < 0.0) & (y[0] >= 0.0)).flatten()
        counts.index_add_(0, vox[spk].long(), torch.ones_like(spk, dtype=F64))
    return dict(zip(STATE, y + [s]), conc=conc)


def _named(run_keys, got):
    return {k: got.get(k) for k in run_keys}


def _exact_rk4(case, seed):
    off, tgt, w, vox, grid, st, _ = _rk4_inputs(case, seed)
    got = _exact_network(case, off, tgt, w, vox, st, (grid,) * 3, (0, 1, 2))
    return _named(STATE + ("conc",), got)


def _exact_ens(case, seed):
    _, _, n, lat, off, tgt, w, vox, st, _ = _ens_inputs(case, seed)
    shape = (lat[2], 64, lat[1], 64, lat[0], 64)
    return _named(STATE + ("conc",), _exact_network(case, off, tgt, w, vox, st, shape, (1, 3, 5)))


def _exact_pull(case, seed):
    off, tgt, w, fire, out = _pull_inputs(case, seed)
    n = case["n"]
    rows = _rows((off[1:] - off[:-1]).long())
    on = fire[rows]
    v = {"weighted": w.double(), "count": torch.ones_like(w, dtype=F64), "signal": out.double()[rows]}[case["mode"]]
    return _zeros(n, F64).index_add_(0, tgt[on].long(), v[on])


def _sums27(u):
    """corner, edge and face neighbour sums, zero beyond the boundary."""
    p = torch.nn.functional.pad(u, (1, 1) * 3)
    m = [torch.zeros_like(u) for _ in range(4)]
    nz, ny, nx = u.shape
    for k in range(3):
        for j in range(3):
            for i in range(3):
                m[(i != 1) + (j != 1) + (k != 1)] += p[k:k + nz, j:j + ny, i:i + nx]
    return m


def _density_update(u):
    """The reference's Crank-Nicolson update: explicit guess, CG to ||r||^2 < 1e-6 or 20 iterations."""
    h, D, k, dt = SCN["h"], SCN["D"], SCN["decay"], SCN["par_dt"]
    c = dt * D / (h * h)

    def lap(v):
        m = _sums27(v)
        return m[3] + 3 * m[2] + 14 * m[1] - 128 * v
    L = lap(u) / (30 * h * h)
    x, b = (1 - dt * k) * u + dt * D * L, (1 - h * k / 2) * u + h * D / 2 * L
    A = lambda v: (1 + dt * k / 2) * v - c / 60 * lap(v)  # noqa: E731
    r = b - A(x)
    rr = (r * r).sum()
    if float(rr) < 1e-6:
        return u
    p = r.clone()
    for _ in range(20):
        q = A(p)
        a = rr / (p * q).sum()
        x = x + a * p
        r = r - a * q
        new = (r * r).sum()
        if float(new) < 1e-6:
            break
        p = r + new / rr * p
        rr = new
    return x


def _diekman(a, iin, icount, const, dt):
    e = torch.exp
    V, M, H, N, Rl, Rnl, Fnl, S, P, Y, Cas, Cac = (a[k] for k in DK)
    q = _lib.params_diekman()
    hdt = dt / 2

    def gate(tau, xinf, x):
        return (2 * dt * xinf + (2 * tau - dt) * x) / (2 * tau + dt)
    cas2 = 1e7 * Cas * Cas
    nM = gate(e(-(V + 286) / 160), 1 / (1 + e(-(V + 35.2) / 8.1)), M)
    nH = gate(0.51 + e(-(V + 26.6) / 7.1), 1 / (1 + e((V + 62) / 2)), H)
    nN = gate(e(-(V - 67) / 68), (1 + e((V - 14) / -17.0)) ** -0.25, N)
    nRl = gate(q.tau_rl, 1 / (1 + e(-(V + 36) / 5.1)), Rl)
    nRnl = gate(q.tau_rnl, 1 / (1 + e(-(V + 21.6) / 6.7)), Rnl)
    nFnl = gate(e(-(V - 444) / 220), 1 / (1 + e((V + 260) / 65)), Fnl)
    nP = gate(q.tau_p, (1 + e(-(V + 25) / 7.4)) ** -1.5, P)
    dV = V - q.eca
    ex = -q.kcas * (q.gcal * Rl * q.k1 / (q.k2 + Cas) + q.gcanl * Rnl * Fnl) * dV - Cas / q.taucas + q.bcas
    nl = hdt * q.kcas * q.gcanl * nRnl * nFnl * dV
    den = 1 + hdt / q.taucas
    B = (q.k2 - Cas - hdt * ex + nl + hdt / q.taucas * q.k2 - q.bcas * hdt) / den
    Cc = (-q.k2 * Cas - q.k2 * hdt * ex + hdt * q.kcas * q.gcal * nRl * q.k1 * dV + nl * q.k2 - q.bcas * hdt * q.k2) / den
    nCas = (torch.sqrt(B * B - 4 * Cc) - B) / 2
    n2 = 1e7 * nCas * nCas
    tS, tS2 = 500 / (cas2 + 5.6), 500 / (n2 + 5.6)
    nS = (S * (1 - dt / (2 * tS)) + hdt * (cas2 / (cas2 + 5.6) / tS + n2 / (n2 + 5.6) / tS2)) / (1 + dt / (2 * tS2))
    ca = q.gcal * nRl * (q.k1 / (q.k2 + Cac)) + q.gcanl * nRl * nFnl + q.gcal * Rl * (q.k1 / (q.k2 + Cas)) + \
        q.gcanl * Rnl * Fnl
    nCac = (Cac * (1 - dt / (2 * q.taucac)) + q.bcac * dt - dt * q.kcac / 2 * ca * dV) / (1 + dt / (2 * q.taucac))
    T = torch.where(icount == 0, torch.zeros_like(iin), iin / icount.clamp_min(1))
    ya = q.ar * T + q.ad
    nY = (q.ar * T * dt + (1 - hdt * ya) * Y) / (hdt * ya + 1)
    n4, fL, na = nN ** 4, q.k1 / (q.k2 + nCas), q.gna * nM ** 3 * nH
    kca = const["gkca"] * nS * nS
    ca = q.gcal * nRl * fL + q.gcanl * nRnl * nFnl
    G = na + q.gk * n4 + ca + kca + const["gkleak"] + q.gnaleak + q.gnap * nP + nY
    E = q.ena * (na + q.gnaleak + q.gnap * nP) + q.ek * (q.gk * n4 + kca + const["gkleak"]) + q.eca * ca + \
        q.g_gaba * nY * const["egaba"]
    nV = (q.appcur * dt + E * dt + (1 - hdt * G) * V) / (1 + hdt * G)
    return dict(zip(DK, (nV, nM, nH, nN, nRl, nRnl, nFnl, nS, nP, nY, nCas, nCac)),
                ioutput=q.tmax / (1 + e(-(nV - q.vt) / q.kp)))


def _exact_scn(case, seed):
    off, tgt, st, const, dims, pos = _scn_inputs(case, seed)
    n = case["n"]
    off, tgt = off.long(), tgt.long()
    a = {k: v.double() for k, v in st.items()}
    const = {k: v.double() for k, v in const.items()}
    ind = torch.bincount(tgt, minlength=n).double()
    # trilinear weights at x / ((m - 1) h) + 0.5 of each axis
    idx, wt = torch.zeros(n, 1, dtype=torch.int64, device=DEV), torch.ones(n, 1, dtype=F64, device=DEV)
    stride = 1
    for m, x in zip(dims, pos):
        u = (torch.from_numpy(x).to(DEV).double() / ((m - 1) * SCN["h"]) + 0.5) * (m - 1)
        i = torch.floor(u).clamp(0, m - 2)
        f = u - i
        i = i.long()
        idx = torch.cat([idx + (i * stride)[:, None], idx + ((i + 1) * stride)[:, None]], 1)
        wt = torch.cat([wt * (1 - f)[:, None], wt * f[:, None]], 1)
        stride *= m
    rel, dens, at = _zeros(n, F64), _zeros(stride, F64), _zeros(n, F64)
    iin = _zeros(n, F64)
    rows = _rows(off[1:] - off[:-1])
    for t in range(case["steps"]):
        fire = a["ioutput"] > 0.1
        iin = _zeros(n, F64).index_add_(0, tgt, fire[rows].double())
        if t % case["timescale"] == 0:
            dens = dens.index_add(0, idx.reshape(-1), (wt * rel[:, None]).reshape(-1))
            dens = _density_update(dens.reshape(dims[2], dims[1], dims[0])).reshape(-1)
            at = (wt * dens[idx]).sum(1)
            rel = torch.zeros_like(rel)
        rel = rel + SCN["coup"] * fire
        a = _diekman(a, iin, ind, const, 0.1)
    return _named(DK + ("ioutput", "iin", "release", "density", "at_neurons"),
                  dict(a, iin=iin, release=rel, density=dens, at_neurons=at))


def _conv3(x, w, ci, co):
    """3x3x3 convolution, channels last, weights [co][27][ci]."""
    p = torch.nn.functional.pad(x, (0, 0) + (1, 1) * 3)
    b, nz, ny, nx, _ = x.shape
    y = 0
    w = w.reshape(co, 27, ci)
    for t in range(27):
        i, j, k = t % 3, (t // 3) % 3, t // 9
        v = p[:, k:k + nz, j:j + ny, i:i + nx, :].reshape(-1, ci)
        y = y + v @ w[:, t, :].t()
    return y.reshape(b, nz, ny, nx, co)


def _pool(x):
    b, nz, ny, nx, c = x.shape
    return x.reshape(b, nz // 2, 2, ny // 2, 2, nx // 2, 2, c).mean((2, 4, 6))


def _up(x):
    return x.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)


def _exact_train(case, seed):
    r, feat, e, faces, w = _train_inputs(case, seed)
    r, feat, e, k = r.double(), feat.double(), e.double(), [f.double() for f in faces]
    w = w.double().requires_grad_(True)
    W, at = [], 0
    for ci, co in LAYERS:
        W.append((w[at:at + co * 27 * ci], w[at + co * 27 * ci:at + co * 27 * ci + co], ci, co))
        at += co * 27 * ci + co
    act = lambda v: torch.nn.functional.leaky_relu(v, 0.1)  # noqa: E731
    layer = lambda x, q: act(_conv3(x, W[q][0], W[q][2], W[q][3]) + W[q][1])  # noqa: E731
    s = r.square().mean((1, 2, 3), keepdim=True).sqrt()
    q, t = r / s, e / s
    e0 = layer(torch.stack([q, q * feat], -1), 0)
    e1 = layer(_pool(e0), 1)
    e2 = layer(_pool(e1), 2)
    d1 = layer(e1 + _up(e2), 3)
    d0 = layer(e0 + _up(d1), 4)
    d = d0 @ w[at:at + 16] + w[at + 16] - t
    dg = 1 + k[0][..., 1:] + k[0][..., :-1] + k[1][..., 1:, :] + k[1][..., :-1, :] + k[2][..., 1:, :, :] + \
        k[2][..., :-1, :, :]
    A = lambda v: _apply_var(v, *k)  # noqa: E731
    for _ in range(case["smooth"]):
        d = d - (2.0 / 3.0) * A(d) / dg
    loss = ((d * A(d)).sum((1, 2, 3)) / (t * A(t)).sum((1, 2, 3))).mean()
    loss.backward()
    return {"grad": w.grad.detach(), "params": None, "loss": float(loss)}


def exact(case, seed):
    k = case["kind"]
    f = dict(rk4=_exact_rk4, ens=_exact_ens, pull=_exact_pull, cg=_exact_cg, train=_exact_train,
             scn=_exact_scn).get(k)
    return f(case, seed) if f else None  # (the noise of the leapfrog network is the library's own stream)
