// mg.hip - geometric multigrid for the variable-coefficient 7-point
// backward-Euler operator, the preconditioner of flexible CG for the
// variable-diffusivity paracrine solve and the base the learned
// preconditioner corrects.
//
// Cell-centred coarsening by 2 x 2 x 2 blocks while every dimension is even
// and at least 8.  A coarse face carries 1/16 of the sum of the 4 fine faces
// it covers: the operator rediscretised on the coarse grid (a face twice as
// wide and a distance twice as long: (4 h^2 / (2h)) / h^3 per unit volume
// of the 8 times larger cell), with the 4 parallel fine conductances added.
// Restriction is the block mean of the residual, prolongation trilinear
// between cell centres with zero beyond the boundary (the fine operator's
// own boundary treatment), smoothing nu sweeps before and after (3 by
// default) of a Chebyshev polynomial in D^-1 A on [1/8, 2] (2 bounds the
// spectrum of D^-1 A for these diagonally dominant operators) or of damped
// Jacobi, the coarsest level 16 damped-Jacobi sweeps.  A W-cycle (each
// coarser level visited twice, the second time on the residual the first
// visit leaves) on the levels of more than 4096 cells, a V-cycle below.
// Block-mean restriction with trilinear prolongation is not a symmetric
// pair, so the cycle is used inside flexible CG.
//
// One generator produces the cycle as a sequence of steps (sweep, restrict,
// residual, prolong-add, add), each a kernel launch; a visit of the first
// level of <= 4096 cells and below is one step, run by a single workgroup
// (k_mg_sub).
//
// No counterpart in the reference, whose CG is unpreconditioned
// (src/paracrine.cu:106-129).
#include <algorithm>
#include <cstdio>
#include <vector>

#include "mg.h"

namespace nnx {

namespace {

unsigned grid_blocks(int64_t n) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 4096)); }
// row kernels: enough workgroups for one wavefront per x-row on small levels
unsigned row_blocks(int ny, int nz) { return (unsigned)std::max(1, std::min((ny * nz + 3) / 4, 4096)); }

__global__ __launch_bounds__(256) void k_mg_dinv(GridK g, float* __restrict__ dinv) {
    const int64_t n = (int64_t)g.nx * g.ny * g.nz;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dinv[i] = dinv_at(g, i);
}

// coarse face coefficients from the fine ones: x faces, then y, then z
__global__ __launch_bounds__(256) void k_mg_coarsen(GridK f, float* __restrict__ kx, float* __restrict__ ky,
                                                    float* __restrict__ kz, int NX, int NY, int NZ) {
    const int64_t nfx = (int64_t)(NX + 1) * NY * NZ, nfy = (int64_t)NX * (NY + 1) * NZ,
                  nfz = (int64_t)NX * NY * (NZ + 1);
    const int64_t nx = f.nx, ny = f.ny;
    for (int64_t q = blockIdx.x * 256ll + threadIdx.x; q < nfx + nfy + nfz; q += (int64_t)gridDim.x * 256) {
        float s;
        if (q < nfx) {
            const int64_t I = q % (NX + 1), J = (q / (NX + 1)) % NY, K = q / ((int64_t)(NX + 1) * NY);
            const float* a = f.kx + 2 * I + (nx + 1) * (2 * J + ny * 2 * K);
            s = (a[0] + a[nx + 1]) + (a[(nx + 1) * ny] + a[(nx + 1) * (ny + 1)]);
            kx[q] = s * (1.0f / 16.0f);
        } else if (q < nfx + nfy) {
            const int64_t r = q - nfx;
            const int64_t I = r % NX, J = (r / NX) % (NY + 1), K = r / ((int64_t)NX * (NY + 1));
            const float* a = f.ky + 2 * I + nx * (2 * J + (ny + 1) * 2 * K);
            s = (a[0] + a[1]) + (a[nx * (ny + 1)] + a[nx * (ny + 1) + 1]);
            ky[r] = s * (1.0f / 16.0f);
        } else {
            const int64_t r = q - nfx - nfy;
            const int64_t I = r % NX, J = (r / NX) % NY, K = r / ((int64_t)NX * NY);
            const float* a = f.kz + 2 * I + nx * (2 * J + ny * 2 * K);
            s = (a[0] + a[1]) + (a[nx] + a[nx + 1]);
            kz[r] = s * (1.0f / 16.0f);
        }
    }
}

// ---- the steps of a cycle, per cell ----
// (every load of a step precedes its stores: the buffers of one step never
// alias, but the compiler cannot know that)
__device__ __forceinline__ void op_cheb(const GridK& g, const MgOp& o, int i, int j, int k, int64_t id) {
    const float* __restrict__ xin = o.xin;
    const float xc = xin ? xin[id] : 0.0f;
    const float res = xin ? o.rhs[id] - apply_at<float, float>(xin, g, i, j, k) : o.rhs[id];
    const float dold = o.c1 != 0.0f ? o.dvec[id] : 0.0f;
    const float t = o.c2 * o.dinv[id] * res;
    const float dn = o.c1 != 0.0f ? o.c1 * dold + t : t;
    o.dvec[id] = dn;
    o.xout[id] = xin ? xc + dn : dn;
}
__device__ __forceinline__ void op_jac(const GridK& g, const MgOp& o, int i, int j, int k, int64_t id) {
    const float* __restrict__ xin = o.xin;
    o.xout[id] = xin ? xin[id] + o.c1 * o.dinv[id] * (o.rhs[id] - apply_at<float, float>(xin, g, i, j, k))
                     : o.c1 * o.dinv[id] * o.rhs[id];
}
// coarse cell (I, J, K): block mean of the fine residual over its 8 children
__device__ __forceinline__ void op_restrict(const GridK& g, const MgOp& o, int I, int J, int K, int64_t q) {
    const int64_t nx = g.nx, ny = g.ny;
    float s = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int i = 2 * I + (c & 1), j = 2 * J + ((c >> 1) & 1), k = 2 * K + (c >> 2);
        const int64_t id = i + nx * (j + ny * k);
        s = s + (o.rhs[id] - apply_at<float, float>(o.xin, g, i, j, k));
    }
    o.xout[q] = 0.125f * s;
}
__device__ __forceinline__ void op_resid(const GridK& g, const MgOp& o, int i, int j, int k, int64_t id) {
    o.xout[id] = o.xout[id] - apply_at<float, float>(o.xin, g, i, j, k);
}
// cell-centred linear weights along one axis: fine cell i sits at coarse
// coordinate i/2 - 1/4: 3/4 on its parent, 1/4 on the parent's neighbour
// toward it (none beyond the boundary)
__device__ __forceinline__ void lin_w(int i, int N, int& a, int& b, float& wb) {
    a = i >> 1;
    b = (i & 1) ? a + 1 : a - 1;
    wb = (b >= 0 && b < N) ? 0.25f : 0.0f;
    if (b < 0 || b >= N) b = a;
}
// x += P e (trilinear, zero outside); g fine, (NX, NY, NZ) coarse dims
__device__ __forceinline__ void op_prolong(const MgOp& o, int NX, int NY, int NZ, int i, int j, int k, int64_t id) {
    int ia, ib, ja, jb, ka, kb;
    float wi, wj, wk;
    lin_w(i, NX, ia, ib, wi);
    lin_w(j, NY, ja, jb, wj);
    lin_w(k, NZ, ka, kb, wk);
    const float* e = o.xin;
    auto E = [&](int I, int J, int K) { return e[I + (int64_t)NX * (J + (int64_t)NY * K)]; };
    const float ai = 0.75f, aj = 0.75f, ak = 0.75f;
    const float v0 = ai * E(ia, ja, ka) + wi * E(ib, ja, ka);
    const float v1 = ai * E(ia, jb, ka) + wi * E(ib, jb, ka);
    const float v2 = ai * E(ia, ja, kb) + wi * E(ib, ja, kb);
    const float v3 = ai * E(ia, jb, kb) + wi * E(ib, jb, kb);
    const float u0 = aj * v0 + wj * v1;
    const float u1 = aj * v2 + wj * v3;
    o.xout[id] = o.xout[id] + (ak * u0 + wk * u1);
}

template <int T> __device__ __forceinline__ void op_at(const GridK& g, const GridK& gc, const MgOp& o, int i, int j,
                                                       int k, int64_t id) {
    if (T == MG_CHEB) op_cheb(g, o, i, j, k, id);
    if (T == MG_JAC) op_jac(g, o, i, j, k, id);
    if (T == MG_RESTRICT) op_restrict(g, o, i, j, k, id);
    if (T == MG_RESID) op_resid(g, o, i, j, k, id);
    if (T == MG_PROLONG) op_prolong(o, gc.nx, gc.ny, gc.nz, i, j, k, id);
    if (T == MG_ADD) o.xout[id] = o.xout[id] + o.xin[id];
}

// one step over a large level: a wavefront per x-row (RESTRICT: per coarse row)
template <int T> __global__ __launch_bounds__(256) void k_mg_op(MgOp o, GridK g, GridK gc) {
    const GridK& d = T == MG_RESTRICT ? gc : g;
    for_rows(d.nx, d.ny, d.nz, [&](int i, int j, int k, int64_t id) { op_at<T>(g, gc, o, i, j, k, id); });
}

// ---- four cells of a row per lane ----
// The per-cell kernel asks for 13 words a cell one at a time, and consecutive
// workgroups - neighbouring rows - sit on different XCDs, so each of the
// eight L2s fetches its own copy of the rows above and below.  Here a lane
// takes 16 bytes of a row (any 4-byte alignment: the face rows have nx + 1),
// the x neighbours come from the lanes beside it, and each XCD (workgroups
// are dealt to the eight in turn) takes a contiguous eighth of the level.
// Bound by memory: a Chebyshev sweep moves 36 bytes a cell, 256^3 150 -> 118
// us (5.1 TB/s), 128^3 20 -> 11.6; the restricted residual 138 -> 87.
// CHEB, JAC, RESTRICT and RESID on a level whose rows are a multiple of four
// cells (row_quads); a lane takes four fine cells of a row (RESTRICT: of the
// four rows of two coarse cells).
template <int T> __global__ __launch_bounds__(256) void k_mg_op4(MgOp o, GridK g, GridK gc) {
    const int q8 = (int)(gridDim.x >> 3), r8 = (int)(gridDim.x & 7), xcd = (int)(blockIdx.x & 7);
    const int blk = xcd * q8 + min(xcd, r8) + (int)(blockIdx.x >> 3);
    const int rows = T == MG_RESTRICT ? gc.ny : g.ny, planes = T == MG_RESTRICT ? gc.nz : g.nz;
    const uint32_t nq = (uint32_t)g.nx >> 2, n4 = nq * (uint32_t)rows * (uint32_t)planes;
    const uint32_t mine = (uint32_t)blk * 256u + threadIdx.x, q = min(mine, n4 - 1u);
    const bool in = mine < n4;  // (lanes past the end repeat the last cells and store nothing)
    const uint32_t row = q / nq;
    const int i = 4 * (int)(q - row * nq), k = (int)(row / (uint32_t)rows), j = (int)(row - (uint32_t)k * rows);
    const float* __restrict__ xin = o.xin;
    f4_t xc;
    if (T == MG_RESTRICT) {
        const int64_t nx = g.nx, ny = g.ny;
        float s0 = 0.f, s1 = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int jj = 2 * j + (c & 1), kk = 2 * k + (c >> 1);
            const f4_t a = apply4(xin, g, i, jj, kk, xc), b = ld4(o.rhs + i + nx * (jj + ny * kk));
            s0 = s0 + (b[0] - a[0]);
            s0 = s0 + (b[1] - a[1]);
            s1 = s1 + (b[2] - a[2]);
            s1 = s1 + (b[3] - a[3]);
        }
        if (!in) return;
        float* __restrict__ out = o.xout + (i >> 1) + (int64_t)gc.nx * row;
        out[0] = 0.125f * s0;
        out[1] = 0.125f * s1;
        return;
    }
    const int64_t id = 4 * (int64_t)q;
    const f4_t rhs = ld4(T == MG_RESID ? o.xout + id : o.rhs + id);
    const bool from0 = T != MG_RESID && !xin;
    f4_t res = rhs;
    if (!from0) {
        const f4_t a = apply4(xin, g, i, j, k, xc);
#pragma unroll
        for (int e = 0; e < 4; ++e) res[e] = rhs[e] - a[e];
    }
    f4_t out, dn;
    if (T == MG_RESID) {
        out = res;
    } else {
        const f4_t di = ld4(o.dinv + id);
        f4_t dold = {0.f, 0.f, 0.f, 0.f};
        if (T == MG_CHEB && o.c1 != 0.0f) dold = ld4(o.dvec + id);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (T == MG_CHEB) {
                const float t = o.c2 * di[e] * res[e];
                dn[e] = o.c1 != 0.0f ? o.c1 * dold[e] + t : t;
            } else {
                dn[e] = o.c1 * di[e] * res[e];
            }
            out[e] = from0 ? dn[e] : xc[e] + dn[e];
        }
    }
    if (!in) return;
    if (T == MG_CHEB) st4(o.dvec + id, dn);
    st4(o.xout + id, out);
}

// One visit (a V-cycle) of the levels of at most kMgSubCells cells by one
// workgroup: a thread keeps its cells' operator, right-hand side, Chebyshev
// direction and value in registers (4 cells of the finest of the levels, one
// of the others), the values go through double-buffered LDS with a zero
// border, so a step costs LDS reads and one barrier.  The coarser levels of
// 4096 cells have at most 512 and 64 (a level is coarsened only while every
// dimension is at least 8), so three levels are the most.  Bound by the
// latency of its ~35 dependent steps: 16^3 with nu = 3 21.7 us where the same
// steps on buffers in global memory, interpreted from a list, took 91.
constexpr int kSubThreads = 1024, kSubCpt = kMgSubCells / kSubThreads;
// border included: the largest box of 4096 (512, 64) cells whose dimensions
// are all at least 4
constexpr int kSubBox0 = 6 * 6 * 258, kSubBox1 = 6 * 6 * 34, kSubBox2 = 6 * 6 * 6;

template <int CPT> struct SubLevel {
    GridK g;
    float *cur, *oth;  // LDS, border of one: the values, and the spare buffer
    int n, sy, sz;
    float k[CPT][6], dg[CPT], di[CPT], b[CPT], x[CPT], d[CPT];
    int pos[CPT];  // LDS index of the cell (0: none)

    __device__ __forceinline__ void load(const GridK& gk, const float* __restrict__ dinv,
                                         const float* __restrict__ rhs, float* b0, float* b1, int box) {
        g = gk, cur = b0, oth = b1;
        n = g.nx * g.ny * g.nz, sy = g.nx + 2, sz = sy * (g.ny + 2);
        for (int i = threadIdx.x; i < box; i += kSubThreads) b0[i] = 0.0f, b1[i] = 0.0f;
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            const int id = (int)threadIdx.x + q * kSubThreads;
            pos[q] = 0, x[q] = 0.0f, d[q] = 0.0f, b[q] = 0.0f, dg[q] = 0.0f, di[q] = 0.0f;
#pragma unroll
            for (int f = 0; f < 6; ++f) k[q][f] = 0.0f;
            if (id >= n) continue;
            const int i = id % g.nx, j = (id / g.nx) % g.ny, kk = id / (g.nx * g.ny);
            pos[q] = (i + 1) + sy * (j + 1) + sz * (kk + 1);
            const int fx = i + (g.nx + 1) * (j + g.ny * kk), fy = i + g.nx * (j + (g.ny + 1) * kk);
            k[q][0] = g.kx[fx], k[q][1] = g.kx[fx + 1];
            k[q][2] = g.ky[fy], k[q][3] = g.ky[fy + g.nx];
            k[q][4] = g.kz[id], k[q][5] = g.kz[id + g.nx * g.ny];
            dg[q] = 1.0f + k[q][0] + k[q][1] + k[q][2] + k[q][3] + k[q][4] + k[q][5];
            di[q] = dinv[id];
            if (rhs) b[q] = rhs[id];
        }
    }
    // b - A x at cell q (apply_at's operation order)
    __device__ __forceinline__ float resid(int q) const {
        const float* v = cur + pos[q];
        float s = k[q][0] * v[-1] + k[q][1] * v[1];
        s = s + k[q][2] * v[-sy];
        s = s + k[q][3] * v[sy];
        s = s + k[q][4] * v[-sz];
        s = s + k[q][5] * v[sz];
        return b[q] - (dg[q] * x[q] - s);
    }
    // the new values into the other buffer
    __device__ __forceinline__ void publish() {
#pragma unroll
        for (int q = 0; q < CPT; ++q)
            if (pos[q]) oth[pos[q]] = x[q];
        float* t = cur;
        cur = oth, oth = t;
        __syncthreads();
    }
    // zero: from x = 0 (nothing read)
    __device__ __forceinline__ void cheb(float c1, float c2, bool zero) {
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            if (!pos[q]) continue;
            const float t = c2 * di[q] * (zero ? b[q] : resid(q));
            const float dn = c1 != 0.0f ? c1 * d[q] + t : t;
            d[q] = dn;
            x[q] = zero ? dn : x[q] + dn;
        }
        publish();
    }
    __device__ __forceinline__ void jacobi(float w, bool zero) {
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            if (!pos[q]) continue;
            x[q] = zero ? w * di[q] * b[q] : x[q] + w * di[q] * resid(q);
        }
        publish();
    }
    __device__ __forceinline__ void sweeps(const MgSubArgs& a, bool zero) {
        for (int s = 0; s < a.nu; ++s) {
            if (a.jac) jacobi(a.w, zero && s == 0);
            else cheb(a.c1[s], a.c2[s], zero && s == 0);
        }
    }
    __device__ __forceinline__ void solve(const MgSubArgs& a) {
        for (int s = 0; s < a.coarse_sweeps; ++s) jacobi(a.w, s == 0);
    }
    // this level's residual into its spare buffer, its block means into c's b
    template <int C2> __device__ __forceinline__ void restrict_to(SubLevel<C2>& c) {
        float* o = oth;
#pragma unroll
        for (int q = 0; q < CPT; ++q)
            if (pos[q]) o[pos[q]] = resid(q);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < C2; ++q) {
            if (!c.pos[q]) continue;
            const int id = (int)threadIdx.x + q * kSubThreads;
            const int I = id % c.g.nx, J = (id / c.g.nx) % c.g.ny, K = id / (c.g.nx * c.g.ny);
            float s = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                s = s + o[(2 * I + (e & 1) + 1) + sy * (2 * J + ((e >> 1) & 1) + 1) + sz * (2 * K + (e >> 2) + 1)];
            c.b[q] = 0.125f * s;
        }
        __syncthreads();
    }
    // x += P (c's x): op_prolong's weights, its zeros outside from the border
    template <int C2> __device__ __forceinline__ void prolong_from(const SubLevel<C2>& c) {
        const float* e = c.cur;
#pragma unroll
        for (int q = 0; q < CPT; ++q) {
            if (!pos[q]) continue;
            const int id = (int)threadIdx.x + q * kSubThreads;
            const int i = id % g.nx, j = (id / g.nx) % g.ny, kk = id / (g.nx * g.ny);
            const int p = ((i >> 1) + 1) + c.sy * ((j >> 1) + 1) + c.sz * ((kk >> 1) + 1);
            const int di_ = (i & 1) ? 1 : -1, dj = (j & 1) ? c.sy : -c.sy, dk = (kk & 1) ? c.sz : -c.sz;
            const float v0 = 0.75f * e[p] + 0.25f * e[p + di_];
            const float v1 = 0.75f * e[p + dj] + 0.25f * e[p + dj + di_];
            const float v2 = 0.75f * e[p + dk] + 0.25f * e[p + dk + di_];
            const float v3 = 0.75f * e[p + dj + dk] + 0.25f * e[p + dj + dk + di_];
            const float u0 = 0.75f * v0 + 0.25f * v1;
            const float u1 = 0.75f * v2 + 0.25f * v3;
            x[q] = x[q] + (0.75f * u0 + 0.25f * u1);
        }
        publish();
    }
};

__global__ __launch_bounds__(kSubThreads) void k_mg_sub(MgSubArgs a) {
    __shared__ float s0[2][kSubBox0], s1[2][kSubBox1], s2[2][kSubBox2];
    SubLevel<kSubCpt> l0;
    SubLevel<1> l1, l2;
    l0.load(a.g[0], a.dinv[0], a.rhs, s0[0], s0[1], kSubBox0);
    if (a.nlev > 1) l1.load(a.g[1], a.dinv[1], nullptr, s1[0], s1[1], kSubBox1);
    if (a.nlev > 2) l2.load(a.g[2], a.dinv[2], nullptr, s2[0], s2[1], kSubBox2);
    __syncthreads();
    if (a.nlev == 1) {
        l0.solve(a);
    } else {
        l0.sweeps(a, true);
        l0.restrict_to(l1);
        if (a.nlev == 2) {
            l1.solve(a);
        } else {
            l1.sweeps(a, true);
            l1.restrict_to(l2);
            l2.solve(a);
            l1.prolong_from(l2);
            l1.sweeps(a, false);
        }
        l0.prolong_from(l1);
        l0.sweeps(a, false);
    }
#pragma unroll
    for (int q = 0; q < kSubCpt; ++q)
        if (l0.pos[q]) a.out[(int)threadIdx.x + q * kSubThreads] = l0.x[q];
}

// The steps of one visit of level l (right-hand side rhs, buffer set `set`),
// appended to ops; returns the buffer that holds the visit's result.  A
// visit of the level cycled in one workgroup is one marker (type -1, xout its
// result).  Level 0 starts its sweeps in t so that an even
// number of sweeps ends in `z0`.
float* gen_visit(const Mg& m, int l, const float* rhs, int set, std::vector<MgOp>& ops, float* z0) {
    if (l == m.sub) {
        MgOp o{};
        o.type = -1, o.level = l, o.rhs = rhs, o.xout = m.x[set][l];
        ops.push_back(o);
        return o.xout;
    }
    float* X = l == 0 ? z0 : m.x[set][l];
    float* T = m.t[set][l];
    float *cur = nullptr, *oth = nullptr;
    auto sweep = [&](int s, bool jacobi) {
        MgOp o{};
        o.level = l, o.rhs = rhs, o.dinv = m.dinv[l];
        if (!cur) {
            o.xin = nullptr;
            o.xout = l == 0 ? T : X;
            oth = l == 0 ? X : T;
        } else {
            o.xin = cur;
            o.xout = oth;
            oth = cur;
        }
        if (jacobi) {
            o.type = MG_JAC;
            o.c1 = m.w;
        } else {
            o.type = MG_CHEB;
            o.dvec = m.d[l];
            o.c1 = m.c1[s];
            o.c2 = m.c2[s];
        }
        ops.push_back(o);
        cur = o.xout;
    };
    if (l == m.nlev - 1) {
        for (int s = 0; s < m.coarse_sweeps; ++s) sweep(s, true);
        return cur;
    }
    const bool jac = m.smoother == NNX_MG_JACOBI;
    for (int s = 0; s < m.nu; ++s) sweep(s, jac);
    {
        MgOp o{};
        o.type = MG_RESTRICT, o.level = l, o.rhs = rhs, o.xin = cur, o.xout = m.b[l + 1];
        ops.push_back(o);
    }
    float* e = gen_visit(m, l + 1, m.b[l + 1], 0, ops, z0);
    // the W-cycle's second visit only for levels above the one-workgroup ones
    const int gam = (m.sub < 0 || l + 1 < m.sub) ? m.gamma : 1;
    for (int v = 1; v < gam; ++v) {
        MgOp r{};
        r.type = MG_RESID, r.level = l + 1, r.xin = e, r.xout = m.b[l + 1];
        ops.push_back(r);
        float* e2 = gen_visit(m, l + 1, m.b[l + 1], 1, ops, z0);
        MgOp a{};
        a.type = MG_ADD, a.level = l + 1, a.xin = e2, a.xout = e;
        ops.push_back(a);
    }
    {
        MgOp o{};
        o.type = MG_PROLONG, o.level = l, o.xin = e, o.xout = cur;
        ops.push_back(o);
    }
    for (int s = 0; s < m.nu; ++s) sweep(s, jac);
    return cur;
}

}  // namespace

nnx_status mg_setup(nnx_ctx* c, const GridK& g0, int nu, int smoother, int gamma, Mg* m) {
    NNX_CHECK(c, g0.kind == 1, "multigrid needs the variable-coefficient 7-point operator");
    NNX_CHECK(c, nu >= 0 && nu <= 16, "nu must be in [0, 16]");
    NNX_CHECK(c, smoother == NNX_MG_CHEBYSHEV || smoother == NNX_MG_JACOBI, "unknown smoother");
    NNX_CHECK(c, gamma >= 0 && gamma <= 2, "cycle must be 0 (W), 1 (V) or 2 (W)");
    m->nu = nu > 0 ? nu : 3;
    m->smoother = smoother;
    m->gamma = gamma > 0 ? gamma : 2;
    // Chebyshev polynomial on [lmax/16, lmax] with lmax = 2, the bound of
    // D^-1 A for these diagonally dominant operators (Gershgorin)
    {
        const double lmax = 2.0, lmin = lmax / 16.0;
        const double th = 0.5 * (lmax + lmin), de = 0.5 * (lmax - lmin), sig = th / de;
        double rho = 1.0 / sig;
        m->c1[0] = 0.0f;
        m->c2[0] = (float)(1.0 / th);
        for (int k = 1; k < 16; ++k) {
            const double r1 = 1.0 / (2.0 * sig - rho);
            m->c1[k] = (float)(r1 * rho);
            m->c2[k] = (float)(2.0 * r1 / de);
            rho = r1;
        }
    }
    m->g[0] = g0;
    int l = 0;
    while (l + 1 < kMgMaxLevels) {
        const GridK& f = m->g[l];
        if ((f.nx & 1) || (f.ny & 1) || (f.nz & 1) || std::min(f.nx, std::min(f.ny, f.nz)) < 8) break;
        GridK& g = m->g[l + 1];
        g = f;
        g.nx = g.nxr = f.nx / 2, g.ny = f.ny / 2, g.nz = f.nz / 2;
        const int64_t nfx = (int64_t)(g.nx + 1) * g.ny * g.nz, nfy = (int64_t)g.nx * (g.ny + 1) * g.nz,
                      nfz = (int64_t)g.nx * g.ny * (g.nz + 1);
        char name[32];
        void* p;
        std::snprintf(name, sizeof name, "mg_k%d", l + 1);
        NNX_TRY(scratch(c, name, (size_t)(nfx + nfy + nfz) * 4, false, &p));
        g.kx = (float*)p, g.ky = (float*)p + nfx, g.kz = (float*)p + nfx + nfy;
        ++l;
    }
    m->nlev = l + 1;
    auto n_of = [&](int q) { return (int64_t)m->g[q].nx * m->g[q].ny * m->g[q].nz; };
    for (int q = 0; q < m->nlev; ++q) {
        const int64_t n = n_of(q);
        char name[32];
        void* p;
        std::snprintf(name, sizeof name, "mg_v%d", q);
        NNX_TRY(scratch(c, name, (size_t)(q == 0 ? 3 : 7) * n * 4, false, &p));
        float* f = (float*)p;
        m->dinv[q] = f;
        m->d[q] = f + n;
        m->t[0][q] = f + 2 * n;
        m->x[0][q] = q ? f + 3 * n : nullptr;
        m->b[q] = q ? f + 4 * n : nullptr;
        m->x[1][q] = q ? f + 5 * n : nullptr;
        m->t[1][q] = q ? f + 6 * n : nullptr;
    }
    for (int q = 1; q < m->nlev; ++q) {
        const GridK& f = m->g[q - 1];
        GridK& g = m->g[q];
        const int64_t nf = (int64_t)(g.nx + 1) * g.ny * g.nz + (int64_t)g.nx * (g.ny + 1) * g.nz +
                           (int64_t)g.nx * g.ny * (g.nz + 1);
        k_mg_coarsen<<<grid_blocks(nf), 256, 0, c->stream>>>(f, (float*)g.kx, (float*)g.ky, (float*)g.kz, g.nx,
                                                             g.ny, g.nz);
        NNX_LAUNCHED(c);
    }
    for (int q = 0; q < m->nlev; ++q) {
        k_mg_dinv<<<grid_blocks(n_of(q)), 256, 0, c->stream>>>(m->g[q], m->dinv[q]);
        NNX_LAUNCHED(c);
    }
    // the small levels: the first level >= 1 with at most kMgSubCells cells
    m->sub = -1;
    for (int q = 1; q < m->nlev; ++q)
        if (n_of(q) <= kMgSubCells) {
            m->sub = q;
            break;
        }
    if (m->sub > 0) {
        NNX_CHECK(c, m->nlev - m->sub <= 3, "multigrid: more than three small levels");
        MgSubArgs& a = m->sub_args;
        a.nlev = m->nlev - m->sub;
        for (int q = 0; q < a.nlev; ++q) a.g[q] = m->g[m->sub + q], a.dinv[q] = m->dinv[m->sub + q];
        a.nu = m->nu, a.coarse_sweeps = m->coarse_sweeps, a.jac = m->smoother == NNX_MG_JACOBI, a.w = m->w;
        for (int q = 0; q < 16; ++q) a.c1[q] = m->c1[q], a.c2[q] = m->c2[q];
    }
    return NNX_OK;
}

nnx_status mg_vcycle(nnx_ctx* c, Mg& m, const float* r, float* z) {
    std::vector<MgOp> ops;
    ops.reserve(256);
    float* res = gen_visit(m, 0, r, 0, ops, z);
    for (const MgOp& o : ops) {
        if (o.type < 0) {
            MgSubArgs sa = m.sub_args;
            sa.rhs = o.rhs, sa.out = o.xout;
            k_mg_sub<<<1, kSubThreads, 0, c->stream>>>(sa);
            NNX_LAUNCHED(c);
            continue;
        }
        const GridK& g = m.g[o.level];
        const GridK& gc = m.g[o.level + 1 < m.nlev ? o.level + 1 : o.level];
        const GridK& d = o.type == MG_RESTRICT ? gc : g;
        const unsigned blocks = row_blocks(d.ny, d.nz);
        if (row_quads(g) && o.type <= MG_RESID) {
            const unsigned b4 = (unsigned)(((int64_t)(g.nx / 4) * d.ny * d.nz + 255) / 256);
            switch (o.type) {
                case MG_CHEB: k_mg_op4<MG_CHEB><<<b4, 256, 0, c->stream>>>(o, g, gc); break;
                case MG_JAC: k_mg_op4<MG_JAC><<<b4, 256, 0, c->stream>>>(o, g, gc); break;
                case MG_RESTRICT: k_mg_op4<MG_RESTRICT><<<b4, 256, 0, c->stream>>>(o, g, gc); break;
                default: k_mg_op4<MG_RESID><<<b4, 256, 0, c->stream>>>(o, g, gc); break;
            }
            NNX_LAUNCHED(c);
            continue;
        }
        switch (o.type) {
            case MG_CHEB: k_mg_op<MG_CHEB><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
            case MG_JAC: k_mg_op<MG_JAC><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
            case MG_RESTRICT: k_mg_op<MG_RESTRICT><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
            case MG_RESID: k_mg_op<MG_RESID><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
            case MG_PROLONG: k_mg_op<MG_PROLONG><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
            default: k_mg_op<MG_ADD><<<blocks, 256, 0, c->stream>>>(o, g, gc); break;
        }
        NNX_LAUNCHED(c);
    }
    if (res != z) NNX_HIP(c, hipMemcpyAsync(z, res, m.g[0].nx * (size_t)m.g[0].ny * m.g[0].nz * 4,
                                            hipMemcpyDeviceToDevice, c->stream));
    return NNX_OK;
}

}  // namespace nnx

using namespace nnx;

extern "C" nnx_status nnx_mg_apply(nnx_ctx* c, const nnx_grid* g, int nu, int smoother, int cycle,
                                   const float* d_r, float* d_z) {
    if (!c) return NNX_ERR_ARG;
    NNX_CHECK(c, g && d_r && d_z, "null argument");
    NNX_CHECK(c, g->stencil == NNX_STENCIL_7 && g->kx && g->ky && g->kz, "multigrid needs a 7-point grid with kx, ky, kz");
    NNX_CHECK(c, g->nx > 0 && g->ny > 0 && g->nz > 0, "bad dims");
    Mg m;
    NNX_TRY(mg_setup(c, make_grid(g), nu, smoother, cycle, &m));
    return mg_vcycle(c, m, d_r, d_z);
}
