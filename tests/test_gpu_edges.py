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


def _csc(n, nnz, seed):
    """Random in-edges, sorted per target, with empty targets and one hub."""
    rng = np.random.default_rng(seed)
    deg = rng.multinomial(nnz - nnz // 8, np.full(n, 1.0 / n))
    deg[rng.integers(0, n, n // 16)] = 0
    deg[n // 3] += nnz - deg.sum()
    off = np.zeros(n + 1, np.int32)
    np.cumsum(deg, out=off[1:])
    return off, rng.integers(0, n, nnz, dtype=np.int32)


# lanes per target (few and many in-edges), slabs of 32 and 64 targets, and
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
