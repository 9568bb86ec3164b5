// 2D ADI time step (the reference's FluidSolver2D path, CPU-only there).
//
// Semantics of AdiSolver2D (src/FluidSolver2D/AdiSolver2D.cpp:21-323,
// TimeLayer2D.h:88-172, Solver2D.cpp:48-85), kept exactly:
//   * one system per grid line (CreateSegments, :228-277): from the non-OUT
//     node before the first NODE_IN to the one after the last; obstacles inside
//     are solved through (BuildMatrix does not look at node types);
//   * rows 1/dt (not 3/dt), BC0 x0 = value or x0 - x1 = 0 (free), BC1 x = value
//     or x[n-2] - x[n-1] = 0 (:74-116), one BC kind per node for all fields;
//   * a direction copies the global Picard layer into a local one, copies the
//     first local solve into it and merges later ones, then copies the local
//     layer and the result out on NODE_IN (SolveDirection, :203-226);
//   * sweeps X then Y, the global loop while it < G or err > 0.1 with the
//     first iteration copying and later ones merging, and the exits above 100
//     iterations or err > 1.0 (TimeStep, :279-323);
//   * every copy and merge skips the last row and column (TimeLayer2D.h:104-172);
//   * the divergence error formula as written (TimeLayer2D.h:88-102).
// Layers other than the state start at zero; their last row and column are
// never written (the reference reads them from freshly allocated memory).
//
// Kernels: the Thomas recurrence of Algorithms.h:21-38 of a (line, field) in the
// reference's operation order.  The rows of a work-group's lines are built by all
// its threads at once into LDS; a line's recurrence and back substitution then
// run in chunks on the lanes of a wavefront, which start early and check one
// another (k2_sweep_chunks), or, for lines that this does not suit, on one lane
// (k2_sweep_lds; lines too long for the LDS keep c', d' in a global scratch,
// k2_sweep).  With one inner iteration a Picard iteration is the two sweeps,
// which write the directions' layers themselves, and one elementwise kernel for
// the merge, the next copies and the divergence sums (k2_merge_div).  The first G
// Picard iterations of a step, which run whatever their error, are queued back
// to back and their errors read once.
#pragma clang fp contract(off)

#include "cmcx_internal.h"
#include "line_solve.h"

#include <algorithm>
#include <cmath>
#include <memory>
#include <vector>

namespace cmcx {
namespace {

template <class T>
struct L3 {
    T* f[3];  // u, v, T
};

struct Sys2 {
    int a0, a1, b;  // X lines: (i_start, j, i_end); Y lines: (i, j_start, j_end)
};

struct P2 {
    double dt, dx, dy, v_T, v_vis, t_vis, t_phi;
};

constexpr int kBS2 = 256;

inline unsigned blocks2(int64_t n) { return (unsigned)((n + kBS2 - 1) / kBS2); }

// dst <- src on nodes (i < nx-1, j < ny-1) whose type bit is set in `mask`;
// merge: dst <- (dst + src) / 2 instead.
template <class T>
__global__ void k2_copy(int nx, int ny, const uint8_t* __restrict__ type, int mask, int merge,
                        L3<T> src, L3<T> dst) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const int i = (int)(q / ny), j = (int)(q % ny);
    if (i >= nx - 1 || j >= ny - 1 || !((mask >> type[q]) & 1)) return;
#pragma unroll
    for (int f = 0; f < 3; f++) dst.f[f][q] = merge ? (dst.f[f][q] + src.f[f][q]) / 2 : src.f[f][q];
}

// The step's copies of the state on nodes (i < nx-1, j < ny-1) as k2_copy, with
// both directions' first copies of the Picard layer: d0..d4 <- src (d4 unless null).
template <class T>
__global__ void k2_fan(int nx, int ny, L3<T> src, L3<T> d0, L3<T> d1, L3<T> d2, L3<T> d3, L3<T> d4) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const int i = (int)(q / ny), j = (int)(q % ny);
    if (i >= nx - 1 || j >= ny - 1) return;
#pragma unroll
    for (int f = 0; f < 3; f++) {
        const T v = src.f[f][q];
        d0.f[f][q] = v;
        d1.f[f][q] = v;
        d2.f[f][q] = v;
        d3.f[f][q] = v;
        if (d4.f[f]) d4.f[f][q] = v;
    }
}

// Solver2D::UpdateBoundaries: node values into the state on BOUND/VALVE, then
// state -> next on BOUND and VALVE (a copy that skips the last row and column).
template <class T>
__global__ void k2_update_boundaries(int nx, int ny, const uint8_t* __restrict__ type, L3<T> g,
                                     L3<T> cur, L3<T> next) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const uint8_t t = type[q];
    if (t != NODE_BOUND && t != NODE_VALVE) return;
    const int i = (int)(q / ny), j = (int)(q % ny);
    const bool inner = i < nx - 1 && j < ny - 1;
#pragma unroll
    for (int f = 0; f < 3; f++) {
        cur.f[f][q] = g.f[f][q];
        if (inner) next.f[f][q] = g.f[f][q];
    }
}

// End of a step: Solver2D::ClearOutterCells (Solver2D.cpp:75-85) on next, then
// state <- next (a copy that skips the last row and column).
template <class T>
__global__ void k2_end_step(int nx, int ny, const uint8_t* __restrict__ type, L3<T> next, L3<T> cur, T startT) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const int i = (int)(q / ny), j = (int)(q % ny);
    const bool outer = type[q] == NODE_OUT, inner = i < nx - 1 && j < ny - 1;
#pragma unroll
    for (int f = 0; f < 3; f++) {
        const T v = outer ? (f == 2 ? startT : (T)0) : next.f[f][q];
        if (outer) next.f[f][q] = v;
        if (inner) cur.f[f][q] = v;
    }
}

// Row t of a line system of n rows (BuildMatrix, AdiSolver2D.cpp:118-178, and
// ApplyBC0/1, :74-116): a, b, c, d of field `var` at cell ct.  Row 0 leaves a
// unset (the recurrence does not read it).
template <class T, bool DIRX>
__device__ __forceinline__ void row2(int t, int n, int var, int64_t ct, int64_t sxs,
                                     const uint8_t* __restrict__ bc, const L3<T>& g,
                                     const L3<T>& lc, const L3<T>& tl, const P2& prm, T& a, T& b,
                                     T& c, T& d) {
    const T dt = (T)prm.dt, hx = (T)prm.dx, hy = (T)prm.dy;
    const T v_T = (T)prm.v_T, t_phi = (T)prm.t_phi;
    const T v_vis = (T)prm.v_vis, t_vis = (T)prm.t_vis;
    const T vis = DIRX ? (var == 2 ? t_vis / (hx * hx) : v_vis / (hx * hx))
                       : (var == 2 ? t_vis / (hy * hy) : v_vis / (hy * hy));
    const T h = DIRX ? hx : hy;
    const T* U = tl.f[0];
    const T* V = tl.f[1];
    const T* TT = tl.f[2];
    if (t == 0) {
        // ApplyBC0
        if (bc[ct] == BC_NOSLIP) {
            b = 1; c = 0; d = g.f[var][ct];
        } else {
            b = 1; c = -1; d = 0;
        }
    } else if (t < n - 1) {
        const T w = DIRX ? U[ct] : V[ct];
        a = -w / (2 * h) - vis;
        b = 1 / dt + 2 * vis;
        c = w / (2 * h) - vis;
        const T lcv = lc.f[var][ct];
        if (DIRX) {
            if (var == 0) {
                const T Tx = (TT[ct + sxs] - TT[ct - sxs]) / (2 * hx);
                d = lcv / dt - v_T * Tx;
            } else if (var == 1) {
                d = lcv / dt;
            } else {
                const T ux = (U[ct + sxs] - U[ct - sxs]) / (2 * hx);
                const T vx = (V[ct + sxs] - V[ct - sxs]) / (2 * hx);
                const T uy = (U[ct + 1] - U[ct - 1]) / (2 * hy);
                d = lcv / dt + t_phi * (2 * ux * ux + vx * vx + uy * vx);
            }
        } else {
            if (var == 0) {
                d = lcv / dt;
            } else if (var == 1) {
                const T Ty = (TT[ct + 1] - TT[ct - 1]) / (2 * hy);
                d = lcv / dt - v_T * Ty;
            } else {
                const T vx = (V[ct + sxs] - V[ct - sxs]) / (2 * hx);
                const T uy = (U[ct + 1] - U[ct - 1]) / (2 * hy);
                const T vy = (V[ct + 1] - V[ct - 1]) / (2 * hy);
                d = lcv / dt + t_phi * (uy * uy + 2 * vy * vy + vx * uy);
            }
        }
    } else {
        // ApplyBC1
        c = 0;
        if (bc[ct] == BC_NOSLIP) {
            a = 0; b = 1; d = g.f[var][ct];
        } else {
            a = 1; b = -1; d = 0;
        }
    }
}

// One line system per thread (blockIdx.y = field): BuildMatrix, ApplyBC0/1,
// SolveTridiagonal (Algorithms.h:21-38), UpdateSegment.  c', d' in a global
// scratch; for systems too long for the LDS of k2_sweep_lds.
template <class T, bool DIRX>
__global__ void k2_sweep(int nsys, const Sys2* __restrict__ sys, int nx, int ny,
                         const uint8_t* __restrict__ bc, L3<T> g, L3<T> lc, L3<T> tl, L3<T> out,
                         P2 prm, T* __restrict__ sc, T* __restrict__ sd) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    const int var = blockIdx.y;
    const Sys2 q = sys[s];
    const int n = DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1;
    auto cell = [&](int t) -> int64_t {
        return DIRX ? (int64_t)(q.a0 + t) * ny + q.a1 : (int64_t)q.a0 * ny + q.a1 + t;
    };
    const int64_t sxs = ny;  // stride of i
    auto idx = [&](int t) { return ((int64_t)t * 3 + var) * nsys + s; };  // (row, field, line)
    T a = 0, b, c, d;
    row2<T, DIRX>(0, n, var, cell(0), sxs, bc, g, lc, tl, prm, a, b, c, d);
    // forward elimination, rows built on the fly (SolveTridiagonal with c[n-1] = 0)
    T cp = c / b, dp = d / b;
    sc[idx(0)] = cp;
    sd[idx(0)] = dp;
    for (int t = 1; t < n; t++) {
        row2<T, DIRX>(t, n, var, cell(t), sxs, bc, g, lc, tl, prm, a, b, c, d);
        const T den = b - a * cp;
        cp = c / den;
        dp = (d - dp * a) / den;
        sc[idx(t)] = cp;
        sd[idx(t)] = dp;
    }
    T x = dp;
    out.f[var][cell(n - 1)] = x;
    for (int t = n - 2; t >= 0; t--) {
        x = sd[idx(t)] - sc[idx(t)] * x;
        out.f[var][cell(t)] = x;
    }
}

// The same solve with the rows in LDS.  A work-group takes `spw` systems of
// one field (blockIdx.y): all its threads build the rows of all its systems
// at once into LDS ([row][system] of (a, b, c, d), and a flag byte per row),
// then thread s runs system s's recurrence from there, c' and d' overwriting
// c and d, and its back substitution.  The rows' global loads thus go out in
// parallel, and the serial chain holds no memory access: its rows come from
// LDS in register batches of kSweepBatch, each batch read while the one before
// is eliminated (a thread's global loads would instead queue behind its own
// scratch stores: one counter covers both on this architecture).
// mode 0: the solution on every row into `out` (the local result layer);
// mode 1 (a direction with one inner iteration): the solution into `lt` and
// `out` on NODE_IN rows off the grid's last row and column, which is what the
// direction's copies leave there (SolveDirection, AdiSolver2D.cpp:203-226:
// the local layer takes the first solve on NODE_IN, the layer and the result
// are copied out on NODE_IN, both copies skipping the last row and column);
// the other rows' stores go to `dm` (the local result layer, which such a
// direction does not read), so that no store waits on a branch.
constexpr int kSweepLdsThreads = 256;
constexpr int kSweepBatch = 8;

template <class T>
struct alignas(4 * sizeof(T)) Row4 {
    T a, b, c, d;
};

template <class T, bool DIRX>
__global__ void __launch_bounds__(kSweepLdsThreads) k2_sweep_lds(
    int nsys, int spw, int nmax, const Sys2* __restrict__ sys, int nx, int ny,
    const uint8_t* __restrict__ type, const uint8_t* __restrict__ bc, L3<T> g, L3<T> lc,
    L3<T> tl, L3<T> out, L3<T> lt, L3<T> dm, int mode, P2 prm) {
    extern __shared__ char smem2[];
    constexpr int R = kSweepBatch;
    const int rs = spw * nmax;  // rows in LDS
    Row4<T>* rw = reinterpret_cast<Row4<T>*>(smem2);
    uint8_t* sf = reinterpret_cast<uint8_t*>(rw + rs);
    const int var = blockIdx.y;
    const int s0 = blockIdx.x * spw;
    const int nloc = min(spw, nsys - s0);
    const int64_t sxs = ny;
    auto cell = [&](const Sys2& q, int t) -> int64_t {
        return DIRX ? (int64_t)(q.a0 + t) * ny + q.a1 : (int64_t)q.a0 * ny + q.a1 + t;
    };
    // rows: consecutive threads on neighbouring cells (X: the same row of
    // neighbouring lines, Y: neighbouring rows of a line)
    for (int e = threadIdx.x; e < rs; e += blockDim.x) {
        const int sl = DIRX ? e % spw : e / nmax;
        const int t = DIRX ? e / spw : e % nmax;
        if (sl >= nloc) continue;
        const Sys2 q = sys[s0 + sl];
        const int n = DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1;
        if (t >= n) continue;
        const int64_t ct = cell(q, t);
        Row4<T> r;
        r.a = 0;
        row2<T, DIRX>(t, n, var, ct, sxs, bc, g, lc, tl, prm, r.a, r.b, r.c, r.d);
        const int k = t * spw + sl;
        rw[k] = r;
        if (mode == 1) {
            const int i = DIRX ? q.a0 + t : q.a0;
            const int j = DIRX ? q.a1 : q.a1 + t;
            sf[k] = type[ct] == NODE_IN && i < nx - 1 && j < ny - 1;
        }
    }
    __syncthreads();
    const int sl = threadIdx.x;
    if (sl >= nloc) return;
    const Sys2 q = sys[s0 + sl];
    const int n = DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1;
    Row4<T>* my = rw + sl;  // row t at my[t * spw]
    const uint8_t* mf = sf + sl;

    // forward elimination (SolveTridiagonal with c[n-1] = 0); rows past the
    // end are read clamped to the last row and not used
    T cp, dp;
    {
        const Row4<T> r0 = my[0];
        cp = r0.c / r0.b;
        dp = r0.d / r0.b;
        my[0].c = cp;
        my[0].d = dp;
    }
    auto elim = [&](const Row4<T>& r, int t) {
        const T den = r.b - r.a * cp;
        cp = r.c / den;
        dp = (r.d - dp * r.a) / den;
        my[t * spw].c = cp;
        my[t * spw].d = dp;
    };
    int t = 1;
    Row4<T> cur[R];
#pragma unroll
    for (int k = 0; k < R; k++) cur[k] = my[min(t + k, n - 1) * spw];
    while (t + R <= n) {
        Row4<T> nxt[R];
#pragma unroll
        for (int k = 0; k < R; k++) nxt[k] = my[min(t + R + k, n - 1) * spw];
#pragma unroll
        for (int k = 0; k < R; k++) elim(cur[k], t + k);
#pragma unroll
        for (int k = 0; k < R; k++) cur[k] = nxt[k];
        t += R;
    }
#pragma unroll
    for (int k = 0; k < R; k++)
        if (t + k < n) elim(cur[k], t + k);

    // back substitution, rows n-2 down to 0 in batches read one batch ahead
    // (the flag bytes are read in mode 0 too, unused: no load under a branch)
    T* const o1 = out.f[var];
    T* const o2 = mode == 1 ? lt.f[var] : out.f[var];
    T* const od = dm.f[var];
    auto put = [&](int t, T v, uint8_t f) {
        const int64_t ct = cell(q, t);
        const bool w = mode == 0 || f != 0;
        (w ? o1 : od)[ct] = v;
        (w ? o2 : od)[ct] = v;
    };
    T x = dp;
    put(n - 1, x, mf[(n - 1) * spw]);
    T bc_[R], bd_[R];
    uint8_t bf_[R];
    t = n - 2;
#pragma unroll
    for (int k = 0; k < R; k++) {
        const int u = max(t - k, 0) * spw;
        bc_[k] = my[u].c;
        bd_[k] = my[u].d;
        bf_[k] = mf[u];
    }
    while (t - R + 1 >= 0) {
        T nc[R], nd[R];
        uint8_t nf[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            const int u = max(t - R - k, 0) * spw;
            nc[k] = my[u].c;
            nd[k] = my[u].d;
            nf[k] = mf[u];
        }
#pragma unroll
        for (int k = 0; k < R; k++) {
            x = bd_[k] - bc_[k] * x;
            put(t - k, x, bf_[k]);
        }
#pragma unroll
        for (int k = 0; k < R; k++) {
            bc_[k] = nc[k];
            bd_[k] = nd[k];
            bf_[k] = nf[k];
        }
        t -= R;
    }
#pragma unroll
    for (int k = 0; k < R; k++)
        if (t - k >= 0) {
            x = bd_[k] - bc_[k] * x;
            put(t - k, x, bf_[k]);
        }
}

// The same solve with a line's recurrences cut into chunks of CL rows, a lane
// each, and every value still the serial one's, bit for bit.  A row's c', d' (and
// x) depend on the rows before it less and less: an error in them shrinks by
// about |c'| per row, until rounding leaves none of it.  So each lane starts some
// rows early from zero: `wa` rows with an approximate reciprocal bring it within
// a few bits, kChunkExact rows with the exact operations to the value itself,
// as a rule.  Then it compares the values that it entered its chunk with to the
// lane before's at its end, and where they differ takes those and runs its chunk
// again, until no lane differs: then every chunk continues its predecessor's
// exactly, and the first one started the line.  One more chunk is settled each
// time, so it ends whatever the rows (infinite and NaN values too).  Back
// substitution likewise from the line's end (`wb` rows early).
// k2_sweep_lds is a chain of two FP64 divisions per row, some 220 ns each: lines
// of 256 rows took 58 us there and of 128 rows 31, and take 18.7 and 14.6 here (the
// slowest work-groups end after 15.1 and 13.3: their rows built in 6.4, elimination 6.1
// and 4.1, back substitution 3.9 and 2.3, results 1.5; the rest is launch and drain).
constexpr int kChunkExact = 12;
constexpr int kChunkMaxRows = 64 * 8;   // rows of a line at most
constexpr int kChunkMaxSystems = 2048;  // of one sweep at most: more of them fill the chip line by line

__device__ __forceinline__ float approx_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double approx_rcp(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}
__device__ __forceinline__ bool same_bits(float a, float b) { return __float_as_uint(a) == __float_as_uint(b); }
__device__ __forceinline__ bool same_bits(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
}

// Rows of a system in LDS: `w` = wa + kChunkExact before its first, its own up to
// whole chunks, wb after them, and one of padding per chunk (the lanes' rows are
// then on different banks); the rows that are not its own (a = 0, b = 1, c = d
// = 0) leave zero, so that the early starts need no conditions.
__host__ __device__ constexpr int chunk_rows(int nmax, int w, int wb, int cl) { return w + (nmax + cl - 1) / cl * cl + wb; }
__host__ __device__ constexpr int chunk_pitch(int rows, int cl) { return rows + rows / cl + 1; }

template <class T, bool DIRX, int CL>
__global__ void __launch_bounds__(kSweepLdsThreads) k2_sweep_chunks(
    int nsys, int spw, int nmax, const Sys2* __restrict__ sys, int nx, int ny,
    const uint8_t* __restrict__ type, const uint8_t* __restrict__ bc, L3<T> g, L3<T> lc,
    L3<T> tl, L3<T> out, L3<T> lt, L3<T> t2, int mode, P2 prm, int wa, int wb) {
    extern __shared__ __align__(16) char smem2[];
    Row4<T>* const rw = reinterpret_cast<Row4<T>*>(smem2);
    const int w = wa + kChunkExact, rows = chunk_rows(nmax, w, wb, CL), pitch = chunk_pitch(rows, CL);
    const int var = blockIdx.y;
    // neighbouring lines, which share cache lines, on one XCD
    const int s0 = (int)lsolve::xcd_remap(blockIdx.x, gridDim.x) * spw;
    const int nloc = min(spw, nsys - s0);
    auto cell = [&](const Sys2& q, int t) -> int64_t {
        return DIRX ? (int64_t)(q.a0 + t) * ny + q.a1 : (int64_t)q.a0 * ny + q.a1 + t;
    };
    // consecutive threads on neighbouring cells
    for (int e = threadIdx.x; e < spw * rows; e += blockDim.x) {
        const int sl = DIRX ? e % spw : e / rows, u = DIRX ? e / spw : e % rows;
        if (sl >= nloc) continue;
        const Sys2 q = sys[s0 + sl];
        const int n = DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1, t = u - w;
        Row4<T> r;
        r.a = r.c = r.d = 0;
        r.b = 1;
        if (t >= 0 && t < n) row2<T, DIRX>(t, n, var, cell(q, t), ny, bc, g, lc, tl, prm, r.a, r.b, r.c, r.d);
        rw[sl * pitch + u + u / CL] = r;
    }
    __syncthreads();

    for (int sl = threadIdx.x >> 6; sl < nloc; sl += kSweepLdsThreads / 64) {
        const Sys2 q = sys[s0 + sl];
        const int n = DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1;
        const int lane = threadIdx.x & 63, last = (n - 1) / CL;  // lanes past the last chunk repeat it
        const bool on = lane <= last;
        const int s = min(lane, last) * CL;  // first row of the lane's chunk
        // row s - w + i, i uniform
        Row4<T>* const my = rw + sl * pitch + s + s / CL;
        auto at = [&](int i) -> Row4<T>& { return my[i + i / CL]; };
        T cp = 0, dp = 0;
        Row4<T> A[4], B[4];
#pragma unroll
        for (int k = 0; k < 4; k++) A[k] = at(k);
        for (int i = 0; i < wa; i += 4) {
#pragma unroll
            for (int k = 0; k < 4; k++) B[k] = at(i + 4 + k);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const T iv = approx_rcp(__builtin_fma(-A[k].a, cp, A[k].b));
                cp = A[k].c * iv;
                dp = __builtin_fma(-A[k].a, dp, A[k].d) * iv;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) A[k] = B[k];
        }
        auto step = [&](const Row4<T>& r) {
            const T den = r.b - r.a * cp;
            cp = r.c / den;
            dp = (r.d - dp * r.a) / den;
        };
#pragma unroll
        for (int i = 0; i < kChunkExact; i += 4) {
#pragma unroll
            for (int k = 0; k < 4; k++) B[k] = at(wa + i + 4 + k);
#pragma unroll
            for (int k = 0; k < 4; k++) step(A[k]);
#pragma unroll
            for (int k = 0; k < 4; k++) A[k] = B[k];
        }
        Row4<T> own[CL];
#pragma unroll
        for (int k = 0; k < CL; k++) own[k] = k < 4 ? A[k] : at(w + k);
        // Row 0 takes no values from before it (a = 0).
        T cin = s == 0 ? (T)0 : cp, din = s == 0 ? (T)0 : dp, cv[CL], dv[CL], den[CL];
        bool quick = true;
        for (;;) {
            cp = cin;
            dp = din;
#pragma unroll
            for (int k = 0; k < CL; k++) {
                den[k] = own[k].b - own[k].a * cp;
                cp = own[k].c / den[k];
                dp = (own[k].d - dp * own[k].a) / den[k];
                cv[k] = cp;
                dv[k] = dp;
            }
            T pc = lsolve::lane_prev(cp), pd = lsolve::lane_prev(dp);
            bool bad = on && lane > 0 && !(same_bits(pc, cin) && same_bits(pd, din));
            if (!__any(bad)) break;
            const bool settled = !__any(on && lane > 0 && !same_bits(pc, cin));
            cin = bad ? pc : cin;
            din = bad ? pd : din;
            // Once c' is settled, d' goes on with its pivots' reciprocals and one
            // correction, a quotient as a rule, until no lane differs; the pass
            // above has the last word.  For lines where d' only decays (no
            // right-hand side left), whose bits depend on every row before: a
            // pass is then one chunk's progress, of 26 instructions instead of 200.
            if (quick && settled) {
                quick = false;
                T rden[CL];
#pragma unroll
                for (int k = 0; k < CL; k++) rden[k] = (T)1 / den[k];
                for (int pass = 0; pass < 64; pass++) {
                    dp = din;
#pragma unroll
                    for (int k = 0; k < CL; k++) {
                        const T num = own[k].d - dp * own[k].a, v = num * rden[k];
                        dp = __builtin_fma(__builtin_fma(-den[k], v, num), rden[k], v);
                    }
                    pd = lsolve::lane_prev(dp);
                    bad = on && lane > 0 && !same_bits(pd, din);
                    if (!__any(bad)) break;
                    din = bad ? pd : din;
                }
            }
        }
        // (the last row's x is its d'; rows past the end leave zero)
#pragma unroll
        for (int k = 0; k < CL; k++) {
            if (s + k >= n - 1) cv[k] = 0;
            if (s + k >= n) dv[k] = 0;
        }
        // c', d' over c, d: every lane of the system's wavefront has read its rows
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < CL; k++)
            if (on && s + k < n) {
                at(w + k).c = cv[k];
                at(w + k).d = dv[k];
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // x of the row after the chunk
        T x = 0, C[4], D[4];
        const int top = w + CL + wb - 1;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            C[k] = at(top - k).c;
            D[k] = at(top - k).d;
        }
        for (int i = 0; i < wb; i += 4) {
            T nc[4], nd[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                nc[k] = at(top - i - 4 - k).c;
                nd[k] = at(top - i - 4 - k).d;
            }
#pragma unroll
            for (int k = 0; k < 4; k++) x = D[k] - C[k] * x;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                C[k] = nc[k];
                D[k] = nd[k];
            }
        }
        T xin = x, xs[CL];
        for (;;) {
            x = xin;
#pragma unroll
            for (int k = CL - 1; k >= 0; k--) {
                x = dv[k] - cv[k] * x;
                xs[k] = x;
            }
            const T xn = lsolve::lane_next(xs[0]);
            const bool bad = lane < last && !same_bits(xn, xin);
            if (!__any(bad)) break;
            xin = bad ? xn : xin;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int k = 0; k < CL; k++)
            if (on && s + k < n) at(w + k).d = xs[k];
    }
    __syncthreads();
    T* const o1 = out.f[var];
    T* const o2 = mode == 1 ? lt.f[var] : o1;
    T* const o3 = mode == 1 ? t2.f[var] : nullptr;
    for (int e = threadIdx.x; e < spw * nmax; e += blockDim.x) {
        const int sl = DIRX ? e % spw : e / nmax, t = DIRX ? e / spw : e % nmax;
        if (sl >= nloc) continue;
        const Sys2 q = sys[s0 + sl];
        if (t >= (DIRX ? q.b - q.a0 + 1 : q.b - q.a1 + 1)) continue;
        const int64_t ct = cell(q, t);
        const int i = DIRX ? q.a0 + t : q.a0, j = DIRX ? q.a1 : q.a1 + t;
        if (mode == 0 || (type[ct] == NODE_IN && i < nx - 1 && j < ny - 1)) {
            const int u = t + w;
            const T v = rw[sl * pitch + u + u / CL].d;
            o1[ct] = v;
            o2[ct] = v;
            if (o3) o3[ct] = v;
        }
    }
}

// TimeLayer2D::EvalDivError: per-block partial sums of |tx + ty| in the field
// type and counts; the finish kernel adds them in block order.  The first
// kDiv2Blocks blocks of a launch take part, whatever its size.
constexpr int kDiv2Blocks = 256;

template <class T>
__device__ __forceinline__ void div_part(int nx, int ny, const uint8_t* __restrict__ type, const L3<T>& L,
                                         T dx, T dy, double* __restrict__ part) {
    __shared__ double ssum[kBS2], scnt[kBS2];
    double sum = 0, cnt = 0;
    const int64_t n = (int64_t)(nx - 1) * (ny - 1);
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (int64_t)kDiv2Blocks * blockDim.x) {
        const int i = (int)(q / (ny - 1)), j = (int)(q % (ny - 1));
        const int64_t c = (int64_t)i * ny + j;
        if (type[c] == NODE_IN && type[c + ny] == NODE_IN && type[c + 1] == NODE_IN &&
            type[c + ny + 1] == NODE_IN) {
            const T* U = L.f[0];
            const T* V = L.f[1];
            const T tx = dy * (U[c + ny] - U[c]) + (U[c + ny + 1] - U[c + 1]) / 2;
            const T ty = dx * (V[c + 1] - V[c]) + (V[c + ny + 1] - V[c + ny]) / 2;
            T e = tx + ty;
            sum += (double)(e < 0 ? -e : e);
            cnt += 1;
        }
    }
    ssum[threadIdx.x] = sum;
    scnt[threadIdx.x] = cnt;
    __syncthreads();
    for (int o = kBS2 / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            ssum[threadIdx.x] += ssum[threadIdx.x + o];
            scnt[threadIdx.x] += scnt[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = ssum[0];
        part[2 * blockIdx.x + 1] = scnt[0];
    }
}

template <class T>
__global__ void k2_div(int nx, int ny, const uint8_t* __restrict__ type, L3<T> L, T dx, T dy,
                       double* __restrict__ part) {
    div_part<T>(nx, ny, type, L, dx, dy, part);
}

// End of a Picard iteration of the one-iteration path: temp <- next on NODE_IN
// (merge: (temp + next) / 2), tl and tl2 <- temp everywhere (both directions'
// next copies of the Picard layer), on nodes (i < nx-1, j < ny-1) as k2_copy, and
// the partial sums of next's divergence error.  Apart, with the copy before the Y
// direction, these were four launches of about 4.5 us each.  A cell per thread, in
// as many blocks as that takes: in the sums' 256 blocks alone the merge of
// a 2000 x 2000 FP64 grid took 273 us (too few loads in flight), and takes 119 so, a
// 700 x 700 one 29 and 18.  Without tl2 (null) its cells are not written.
template <class T>
__global__ void __launch_bounds__(kBS2) k2_merge_div(int nx, int ny, const uint8_t* __restrict__ type,
                                                     int merge, L3<T> next, L3<T> temp, L3<T> tl, L3<T> tl2,
                                                     T dx, T dy, double* __restrict__ part) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // (the cells of a grid that fits the memory fit 32 bits)
    if (q < (int64_t)(nx - 1) * ny && (int)((uint32_t)q % (uint32_t)ny) < ny - 1) {
        const bool in = type[q] == NODE_IN;
#pragma unroll
        for (int f = 0; f < 3; f++) {
            T v = temp.f[f][q];
            if (in) {
                v = merge ? (v + next.f[f][q]) / 2 : next.f[f][q];
                temp.f[f][q] = v;
            }
            tl.f[f][q] = v;
            if (tl2.f[f]) tl2.f[f][q] = v;
        }
    }
    if (blockIdx.x < kDiv2Blocks) div_part<T>(nx, ny, type, next, dx, dy, part);
}

// One work-group of kDiv2Blocks threads per slot: its partials come into LDS in
// one parallel load, then thread 0 adds them in block order.
__global__ void __launch_bounds__(kDiv2Blocks) k2_div_finish(const double* __restrict__ part,
                                                             int nb, double* __restrict__ out) {
    __shared__ double sp[2 * kDiv2Blocks];
    for (int k = threadIdx.x; k < 2 * nb; k += blockDim.x) sp[k] = part[(int64_t)blockIdx.x * 2 * nb + k];
    __syncthreads();
    if (threadIdx.x != 0) return;
    double s = 0, c = 0;
    for (int b = 0; b < nb; b++) {
        s += sp[2 * b];
        c += sp[2 * b + 1];
    }
    out[2 * blockIdx.x] = s;
    out[2 * blockIdx.x + 1] = c;
}


// ---- StableSolver2D (StableSolver2D.cpp:21-234): explicit advection-diffusion,
// then a projection whose Poisson equation is relaxed cell by cell in place.

// SolveU / SolveV (StableSolver2D.cpp:55-81) on NODE_IN cells: the state plus
// dt times the advection-diffusion of the Picard layer `tl`, into w.
template <class T>
__global__ void k2s_solve_uv(int nx, int ny, const uint8_t* __restrict__ type, L3<T> cur, L3<T> tl,
                             L3<T> w, T dt, T dx, T dy, T v_vis) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny || type[q] != NODE_IN) return;
    const int64_t e = ny;
    const T* U = tl.f[0];
    const T* V = tl.f[1];
    const T u = U[q], v = V[q];
    const T ux = (U[q + e] - U[q - e]) / (2 * dx), uy = (U[q + 1] - U[q - 1]) / (2 * dy);
    const T uxx = (U[q + e] - 2 * U[q] + U[q - e]) / (dx * dx);
    const T uyy = (U[q + 1] - 2 * U[q] + U[q - 1]) / (dy * dy);
    const T vx = (V[q + e] - V[q - e]) / (2 * dx), vy = (V[q + 1] - V[q - 1]) / (2 * dy);
    const T vxx = (V[q + e] - 2 * V[q] + V[q - e]) / (dx * dx);
    const T vyy = (V[q + 1] - 2 * V[q] + V[q - 1]) / (dy * dy);
    w.f[0][q] = cur.f[0][q] + dt * (-u * ux - v * uy + v_vis * (uxx + uyy));
    w.f[1][q] = cur.f[1][q] + dt * (-u * vx - v * vy + v_vis * (vxx + vyy));
}

// Project's divergence field (StableSolver2D.cpp:85-97): w.Ux + w.Vy on NODE_IN
// cells, zero elsewhere, stored diagonal by diagonal (cell (i, j) at
// doff[i + j] + i - max(0, i + j - ny + 1)): the relaxation reads the cells of
// one anti-diagonal together, which then lie side by side.
template <class T>
__global__ void k2s_div(int nx, int ny, const uint8_t* __restrict__ type, L3<T> w, T dx, T dy,
                        const int32_t* __restrict__ doff, T* __restrict__ dvd) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const int i = (int)(q / ny), j = (int)(q % ny), d = i + j;
    const int64_t at = doff[d] + i - max(0, d - ny + 1);
    if (type[q] != NODE_IN) {
        dvd[at] = 0;
        return;
    }
    const T* U = w.f[0];
    const T* V = w.f[1];
    dvd[at] = (U[q + ny] - U[q - ny]) / (2 * dx) + (V[q + 1] - V[q - 1]) / (2 * dy);
}

// Project's last loop (StableSolver2D.cpp:153-164): w minus the gradient of q
// (ScalarField2D::grad, central differences in the field type) on NODE_IN cells.
template <class T>
__global__ void k2s_grad(int nx, int ny, const uint8_t* __restrict__ type, L3<T> w,
                         const T* __restrict__ qf, T dx, T dy, L3<T> proj) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny || type[q] != NODE_IN) return;
    const T gx = (qf[q + ny] - qf[q - ny]) / (2 * dx);
    const T gy = (qf[q + 1] - qf[q - 1]) / (2 * dy);
    proj.f[0][q] = w.f[0][q] - gx;
    proj.f[1][q] = w.f[1][q] - gy;
}

// The relaxation's stopping test folds the cells' relative changes
// |(qn - qo) / qn| in sweep order with std::max(cur, err) from err = 0, then
// continues while err >= tol: a NaN change (0/0) makes err NaN and the next
// cell's change replaces it, so the test depends only on the changes after
// the last NaN (none of them >= tol, or a NaN last, ends the loop).  A
// sequence's summary: kind 0 (empty), 1 (no NaN), 2 (a NaN, then ge counts
// only the changes after the last one); ge: some change >= tol.
struct ErrFold {
    int kind;
    int ge;
};

// One cell's change into the summary.  |qn - qo| against tol |qn| decides
// without dividing away from the threshold (the margin covers the rounding of
// both sides); close to it, and for zero or non-finite values, the change is
// divided out as the reference does, so the decision is the reference's.
__device__ inline void fold_cell(ErrFold& s, double qn, double qo, double tol) {
    const double d = qn - qo;
    const double a = fabs(d), m = fabs(qn), b = tol * m;
    // infinite or NaN values fail both tests below or decide them as the
    // division would (an infinite change is >= tol), so only tiny |qn| and
    // tiny tolerances need the division's exact rounding
    const bool plain = m >= 1e-290 && (b > 1e-300 || tol == 0.0);
    bool nan = false, ge;
    if (plain && a < b * (1.0 - 1e-12)) ge = false;
    else if (plain && a > b * (1.0 + 1e-12)) ge = true;
    else {
        const double ce = fabs(d / qn);
        nan = ce != ce;
        ge = ce >= tol;
    }
    if (nan) {
        s.kind = 2;
        s.ge = 0;
    } else {
        if (s.kind == 0) s.kind = 1;
        s.ge |= ge ? 1 : 0;
    }
}

// sequence a followed by sequence b
__device__ inline ErrFold fold_cat(ErrFold a, ErrFold b) {
    if (b.kind == 0) return a;
    if (a.kind == 0 || b.kind == 2) return b;
    return ErrFold{a.kind, a.ge | b.ge};
}

// Cell flags of the relaxation: kind in bits 0-1 (0 outside, 1 NODE_IN, 2
// NODE_BOUND or NODE_VALVE), then whether the neighbour (i-1, j), (i+1, j),
// (i, j-1), (i, j+1) is NODE_IN (bits 2-5; cells beyond the grid are not).
enum { PF_IN = 1, PF_BOUND = 2, PF_UP = 4, PF_DOWN = 8, PF_LEFT = 16, PF_RIGHT = 32 };

// Project's relaxation (StableSolver2D.cpp:99-151): sweeps over the boundary
// cells, then the inner cells, each list in (i, j) order, each cell's new value
// from its neighbours' current ones (those earlier in the order already
// relaxed in this sweep), until the stopping test passes.
//
// One work-group.  A sweep's step k relaxes the boundary cell (r, k - r) and
// the inner cell (r, k - 2 - r) of every row r: every value a cell reads is
// then the one the sequential order gives it (boundary cells read inner
// neighbours from the previous sweep and boundary neighbours from this one;
// inner cells read the boundary cells of this sweep, inner neighbours before
// them from this sweep and after them from the previous one), and the cells of
// one step touch no cell another cell of the step reads, so one barrier per
// step orders everything.
//
// Sweeps run in groups of up to D, member s starting LAG = 4 steps after
// member s - 1 in the same q: member s reads diagonals k - 3 .. k + 1 around
// its step k while member s - 1 writes k + 2 and k + 4 and member s + 1 writes
// k - 4 and k - 6, and every value a member reads from the previous sweep is
// final (its inner front passed it at least one step before), so the group
// gives exactly the values of its sweeps run one after the other.  The
// work-group holds D slices of rp threads (rp >= nx, a multiple of 64):
// thread r of a slice relaxes row r's boundary and inner cells for its member
// (a wave skips the boundary part when none of its rows has a boundary cell
// at the step); the members' waves share each SIMD and hide one another's
// latencies.  The stopping test of each
// member is known when the group ends: if member s passes it first, q goes
// back to the snapshot taken at the group's start (in global memory) and a
// group of s + 1 members runs again, which ends on member s's result.  The
// fold runs per row in the row's own order, then over a slice's threads in
// order: boundary rows, then inner rows.
//
// q lives per row over the row's span [lo, hi] of non-outside cells plus a
// zero guard cell at each end (row r at spans[3r]: column j at
// spans[3r] + 1 + j - lo); outside cells keep q = 0, and so do cells beyond the
// grid (the reference reads outside its arrays there, Grid2D.cpp:50-53 has no
// bounds check).  LDS holds q and the flags (QLDS) or they stay in global
// memory.  At most max_sweeps sweeps per launch; status = {sweeps so far,
// converged}; a launch with resume = 1 continues from qspan.
constexpr int kPoisLag = 4;

template <class T, bool QLDS>
__global__ void __launch_bounds__(1024) k2s_poisson(
    int nx, int ny, int S, int rp, int D, const int32_t* __restrict__ spans,
    const uint8_t* __restrict__ fspan, const int32_t* __restrict__ doff, const T* __restrict__ dvd,
    T* __restrict__ qspan, T* __restrict__ save, double dx2, double dy2, double rcp, double tol,
    int max_sweeps, int resume, int32_t* __restrict__ status) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ ErrFold sh[32];
    __shared__ int s_first;
    T* qs = QLDS ? reinterpret_cast<T*>(smem) : qspan;
    const uint8_t* fl = QLDS ? smem + (size_t)S * sizeof(T) : fspan;
    if (QLDS) {
        for (int c = threadIdx.x; c < S; c += blockDim.x) {
            qs[c] = resume ? qspan[c] : (T)0;
            smem[(size_t)S * sizeof(T) + c] = fspan[c];
        }
    } else if (!resume) {
        for (int c = threadIdx.x; c < S; c += blockDim.x) qs[c] = (T)0;
    }
    __syncthreads();
    const int mem = (int)threadIdx.x / rp;  // member slice, uniform per wave
    const int r = (int)threadIdx.x - mem * rp;
    const bool own = r < nx;
    // padded spans of rows r - 1, r, r + 1: storage [a, b] holds columns
    // lo - 1 .. hi + 1 (column j at base + j); a cell is inside for lo <= j <= hi
    int base[3], lo[3], hi[3], a[3], b[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int rd = r + d - 1;
        const bool ok = own && rd >= 0 && rd < nx;
        a[d] = ok ? spans[3 * rd] : 0;
        lo[d] = ok ? spans[3 * rd + 1] : 0;
        hi[d] = ok ? spans[3 * rd + 2] : -1;
        base[d] = a[d] + 1 - lo[d];
        // a row beyond the grid reads element 0, the first row's zero guard
        b[d] = ok ? a[d] + (hi[d] - lo[d] + 1) + 1 : 0;
    }
    auto clampi = [](int x, int lo_, int hi_) { return min(max(x, lo_), hi_); };
    auto inside = [&](int d, int j) -> bool { return j >= lo[d] && j <= hi[d]; };
    // A neighbour row's column j outside its span clamps onto one of that
    // row's zero guard cells (rows beyond the grid onto element 0, the first
    // row's guard), so the read gives the reference's q = 0 there unmasked.
    // The step's barrier: with q in LDS nothing global is shared between
    // threads within a group, so it waits for the LDS traffic only and the div
    // loads stay in flight across it.
    auto step_barrier = [&]() {
        if (QLDS) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else __syncthreads();
    };
    // div of (r, j), diagonal-major: the lanes of a wave read one diagonal's
    // consecutive cells
    auto dv_at = [&](int j) -> double {
        const bool ok = own && j >= 0 && j < ny;
        const int d = ok ? r + j : 0;  // every index stays inside its array
        const int at = ok ? doff[d] + r - max(0, d - ny + 1) : 0;
        return ok ? (double)dvd[at] : 0.0;
    };
    const int K = nx + ny + 1;
    const int wpm = rp / 64;  // waves per member slice
    int sweeps = resume ? status[0] : 0;
    int left = max_sweeps;
    bool converged = false;
    int rerun = 0;  // members of a group run again from the snapshot (uniform)
    while (left > 0) {
        const int g = rerun ? rerun : min(D, left);  // members of this group (uniform)
        if (!rerun && g > 1)
            for (int q = threadIdx.x; q < S; q += blockDim.x) save[q] = qs[q];
        ErrFold fb{0, 0}, fi{0, 0};
        const int steps = K + (g - 1) * kPoisLag;
        const int k0 = mem * kPoisLag;  // this member's first step
        double dA = dv_at(0 - k0 - 2 - r), dB = 0.0;
        for (int k2 = 0; k2 < steps; k2 += 2) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int kk = k2 + h;
                if (kk >= steps) break;  // uniform
                double& dcur = h == 0 ? dA : dB;
                double& dnxt = h == 0 ? dB : dA;
                const int k = kk - k0;
                const bool act = mem < g && k >= 0 && k < K;  // uniform per wave
                const int jb = k - r, ji = jb - 2;
                dnxt = dv_at(k + 1 - 2 - r);
                const int own_lo = a[1] + 1, own_hi = max(b[1] - 1, a[1] + 1);
                const int cb = clampi(base[1] + jb, own_lo, own_hi);
                const int ci = clampi(base[1] + ji, own_lo, own_hi);
                const int ub = clampi(base[0] + jb, a[0], b[0]), db = clampi(base[2] + jb, a[2], b[2]);
                const int ui = clampi(base[0] + ji, a[0], b[0]), di = clampi(base[2] + ji, a[2], b[2]);
                T bq = qs[cb], bl = qs[cb - 1], br = qs[cb + 1], bu = qs[ub], bd = qs[db];
                T iq = qs[ci], il = qs[ci - 1], ir = qs[ci + 1], iu = qs[ui], id = qs[di];
                int bf = fl[cb], jf = fl[ci];
                // the empty asm takes every read, so none is sunk into a branch
                asm volatile("" : "+v"(bq), "+v"(bl), "+v"(br), "+v"(bu), "+v"(bd), "+v"(bf));
                asm volatile("" : "+v"(iq), "+v"(il), "+v"(ir), "+v"(iu), "+v"(id), "+v"(jf));
                if (act) {
                    const int f = bf & (inside(1, jb) ? 0xff : 0);
                    if (f & PF_BOUND) {
                        const double up = (double)bu, dn = (double)bd;
                        const double lf_ = (double)bl, rt = (double)br;
                        const double i0 = (f & PF_UP) ? up : dn, i1 = (f & PF_DOWN) ? dn : up;
                        const double j0 = (f & PF_LEFT) ? lf_ : rt, j1 = (f & PF_RIGHT) ? rt : lf_;
                        // div is zero on boundary cells
                        const double qn = rcp * ((i0 + i1) * dy2 + (j0 + j1) * dx2 - 0.0 * dx2 * dy2);
                        qs[cb] = (T)qn;
                        fold_cell(fb, qn, (double)bq, tol);
                    }
                    const int g2 = jf & (inside(1, ji) ? 0xff : 0);
                    if (g2 & PF_IN) {
                        const double up = (double)iu, dn = (double)id;
                        const double qn =
                            rcp * ((up + dn) * dy2 + ((double)il + (double)ir) * dx2 - dcur * dx2 * dy2);
                        qs[ci] = (T)qn;
                        fold_cell(fi, qn, (double)iq, tol);
                    }
                }
                step_barrier();
            }
        }
        // each member's stopping test: an ordered fold over its slice's
        // waves, boundary rows then inner rows
        {
            const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
            ErrFold vb = fb, vi = fi;
            for (int off = 1; off < 64; off <<= 1) {
                ErrFold ob, oi;
                ob.kind = __shfl_down(vb.kind, off);
                ob.ge = __shfl_down(vb.ge, off);
                oi.kind = __shfl_down(vi.kind, off);
                oi.ge = __shfl_down(vi.ge, off);
                if (lane + off < 64) {
                    vb = fold_cat(vb, ob);
                    vi = fold_cat(vi, oi);
                }
            }
            if (lane == 0) {
                sh[wave] = vb;
                sh[16 + wave] = vi;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int first = -1;
            for (int m = 0; m < g && first < 0; m++) {
                ErrFold all{0, 0};
                for (int w = 0; w < wpm; w++) all = fold_cat(all, sh[m * wpm + w]);
                for (int w = 0; w < wpm; w++) all = fold_cat(all, sh[16 + m * wpm + w]);
                if (!(all.kind != 0 && all.ge)) first = m;
            }
            s_first = first;
        }
        __syncthreads();
        const int first = s_first;
        if (rerun || first + 1 == g) {  // a rerun ends on its last member
            sweeps += g;
            converged = true;
            break;
        }
        if (first >= 0) {
            for (int q = threadIdx.x; q < S; q += blockDim.x) qs[q] = save[q];
            __syncthreads();
            rerun = first + 1;
            continue;
        }
        sweeps += g;
        left -= g;
    }
    __syncthreads();
    if (QLDS)
        for (int q = threadIdx.x; q < S; q += blockDim.x) qspan[q] = qs[q];
    if (threadIdx.x == 0) {
        status[0] = sweeps;
        status[1] = converged ? 1 : 0;
    }
}

// The relaxation for grids whose q fits the LDS, the form that the solver
// picks whenever it does (the two fronts, the lag of kPoisLag steps between
// sweeps and the stopping test are those of k2s_poisson above, and so is every
// value).  Both run on one compute unit and are bound by the instructions that
// its wavefronts issue; k2s_poisson makes 10 reads, 6 clamped addresses and both
// fronts' arithmetic for every lane and step, half of its lanes outside the
// front (284 steps of 2700 cycles for 8 sweeps of a 120 x 135 grid).  Here:
//   * q lies in LDS by anti-diagonals: cell (r, j), x = j + 1, is element
//     ((x + r) mod P, r + 1) of P rows of nx + 2.  A front is one row, a lane's
//     neighbours are in the rows either side, and the lanes' accesses are
//     consecutive.  x = 0 and the first and last elements of a row hold zero;
//     P >= ny + 1, so that x = 0 also ends a grid row.
//   * slices of rp threads (rp >= nx) relax inner cells, lane r row r, for MW
//     sweeps each (D in all), one cell of each per step, and start their next
//     sweeps P steps after the last ones' start without waiting for the other
//     rows: no lane idles at the ends of a front.  Sweep n starts at step
//     (n mod D) kPoisLag + (n div D) P, at least kPoisLag after sweep n - 1
//     (P >= kPoisLag D), which is all that the order needs.  At residue
//     (x + r) mod P the rows r <= residue of a wavefront are in its newest
//     sweep, the others still in the one before: P >= nx, or P is a multiple
//     of 64 and each wavefront has its own delay.
//   * a cell's own value comes from the last step's right neighbour, its left
//     one from the last step's result.
//   * the few boundary cells of a front are relaxed for all D sweeps by bw
//     wavefronts of their own, from lists per residue.
//   * an inner cell's div dx2 dy2 comes from `dvs`, laid out like q, two steps
//     ahead; kNotInner marks the other cells, so that no flags are read.
//   * the stopping test works on lane masks, in scalar registers: per sweep and
//     row a NaN, and a change of tol or more since the row's last NaN.
// Per sweep of a 120 x 135 grid in FP64: 39.6 us before, 6.7 now; with one sweep
// per lane a sixth more, with four a fifth (scalar registers spill).  A first form with rows
// of q in LDS, where a lane moves on to its next sweep by itself in a branch
// that some lane takes on every step, took 7.7 to 8.6.
constexpr int kPoisGroup = 256;              // sweeps of a group at most
constexpr unsigned kNotInner = 0x7ff5a5a5u;  // high word of dvs off the inner cells (no result is this NaN)
constexpr int kDvRows = kPoisLag;            // rows of dvs repeated before the first
constexpr uint32_t kBValid = 1u << 28;
// Boundary list entry: x: place in sweep order (r P + x), selects << 16, kBValid;
// y: r, (x + r) / P << 16.

// Whether |(qn - qo) / qn| >= tol: the sign of |qn - qo| - tol |qn| away from
// zero (`eps` = tol times a margin far above the rounding of either side; the
// tiny constant keeps the margin where tol |qn| underflows): yes if t > b, no if
// t < -b, otherwise (infinite or NaN values too) change_divided decides.
__device__ __forceinline__ void change_sides(double qn, double qo, double tol, double eps, double& t, double& b) {
    const double m = fabs(qn);
    t = __builtin_fma(m, -tol, fabs(qn - qo));
    b = __builtin_fma(m, eps, 1e-300);
}
__device__ __forceinline__ bool change_divided(double qn, double qo, double tol, bool& nan) {
    const double ce = fabs((qn - qo) / qn);
    nan = ce != ce;
    return ce >= tol;
}

template <class T, int MW>
__global__ void __launch_bounds__(1024) k2s_poisson_lds(
    int nx, int ny, int P, int rp, int D, int bw, int cpad, const uint2* __restrict__ blist,
    const double* __restrict__ dvs, T* __restrict__ qgrid, T* __restrict__ save, double dx2,
    double dy2, double rcp, double tol, int max_sweeps, int resume, int32_t* __restrict__ status) {
    extern __shared__ __align__(16) unsigned char smem[];
    // per sweep: the last place in sweep order with a change >= tol, with a NaN
    // (0 = none)
    __shared__ int fold[2 * kPoisGroup];
    __shared__ int s_first;
    __shared__ T dump[64];  // stores of cells that are not inner ones
    using Lds = __attribute__((address_space(3))) T;
    using LdsByte = __attribute__((address_space(3))) char;
    T* const q = reinterpret_cast<T*>(smem);
    const int Q = nx + 2, S = P * Q;
    for (int c = threadIdx.x; c < S; c += blockDim.x) q[c] = resume ? qgrid[c] : (T)0;
    const double eps = tol * 2e-12;
    auto step_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    const int nin = D / MW * rp;                // threads of the inner slices
    const bool inner = (int)threadIdx.x < nin;  // uniform per wave
    // inner: row r of members mem .. mem + MW - 1; boundary: slot e0 of member mem
    const int epm = 64 * bw / D;
    const int lb = (int)threadIdx.x - nin;
    const int mem = inner ? (int)threadIdx.x / rp * MW : lb / epm;
    const int r = (int)threadIdx.x - mem / MW * rp, e0 = lb % epm;
    const int k0 = kPoisLag * mem;
    auto next = [&](int a) { return a + 1 == P ? 0 : a + 1; };

    int sweeps = resume ? status[0] : 0, left = max_sweeps, rerun = 0, gsize = resume ? kPoisGroup : 16;
    bool converged = false;
    __syncthreads();
    while (left > 0) {
        const int g = rerun ? rerun : min(gsize, left);  // sweeps of this group (uniform)
        if (!rerun && g > 1)
            for (int c = threadIdx.x; c < S; c += blockDim.x) save[c] = q[c];
        for (int c = threadIdx.x; c < 2 * kPoisGroup; c += blockDim.x) fold[c] = 0;
        if (threadIdx.x == 0) s_first = g;
        __syncthreads();
        // to the end of sweep g - 1: its start, rows, columns (x = 1 .. ny, not the whole
        // turn of P: of 12 x 10 cells 11 steps, not 60) and the inner front's two
        // steps, in whole turns of the loops' four steps
        const int steps = (((g - 1) / D) * P + ((g - 1) % D) * kPoisLag + nx + ny + 1 + 2 + 3) & ~3;
        if (inner) {
            // Branch-free but for the rare cases (a change too close to tol to
            // tell, the end of a turn), each tested once for the MW cells.
            const int w0 = __builtin_amdgcn_readfirstlane(r);  // the wavefront's first row
            const int late = __builtin_amdgcn_readfirstlane(w0 / P), wr = w0 - late * P;       // its delay in turns, its first row's residue at x = 0
            const uint64_t rows = nx - w0 >= 64 ? ~0ull : nx > w0 ? (1ull << (nx - w0)) - 1 : 0;
            const uint32_t qb = (uint32_t)Q * (uint32_t)sizeof(T), pb = (uint32_t)P * qb;  // bytes of a row, of q
            // lanes beyond the rows read the last one's cells and are never live
            Lds* const ql = (Lds*)(q + min(r, nx - 1));
            Lds* const pdump = (Lds*)&dump[threadIdx.x & 63];
            auto at = [&](uint32_t row) { return (Lds*)((LdsByte*)ql + row); };
            uint32_t voff[MW], rb[MW], rs[MW], rf[MW];  // rows of residues res - 1, res, res + 1
            int res[MW], n[MW];                         // per member: residue, newest sweep
            // lanes in the newest sweep; of these and of the others, those whose
            // sweep is one of the group's; rows with a change >= tol, with a NaN
            // in the newest sweep and in the one before
            uint64_t newest[MW], live1[MW], live0[MW], ge1[MW], ge0[MW], na1[MW], na0[MW];
            double lft[MW], cur[MW], dv[MW][2];
            auto set_live = [&](int u) {
                live1[u] = n[u] >= 0 && n[u] < g ? rows : 0;
                live0[u] = n[u] >= D && n[u] < g + D ? rows : 0;
            };
            // dvs two steps on, its row's residue the first member's
            const uint32_t db = (uint32_t)rp * (uint32_t)sizeof(double);
            const int res2 = __builtin_amdgcn_readfirstlane((P - (k0 + 2) % P) % P);
            uint32_t drow = (uint32_t)res2 * db;
            const uint32_t dend = (uint32_t)P * db;
            auto advance_dvs = [&] { drow = drow + db == dend ? 0 : drow + db; };
            auto dvs_at = [&](int u) {
                return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(dvs) + (voff[u] + drow));
            };
#pragma unroll
            for (int u = 0; u < MW; u++) {
                const int back = __builtin_amdgcn_readfirstlane(k0 + kPoisLag * u + 2), turns = (back + P - 1) / P;
                res[u] = turns * P - back;
                n[u] = __builtin_amdgcn_readfirstlane(mem + u - D * (turns + late));
                const int k1 = res[u] - wr;
                newest[u] = k1 >= 63 ? ~0ull : k1 >= 0 ? (2ull << k1) - 1 : 0;
                set_live(u);
                rs[u] = (uint32_t)res[u] * qb;
                rb[u] = rs[u] == 0 ? pb - qb : rs[u] - qb;
                rf[u] = rs[u] + qb == pb ? 0 : rs[u] + qb;
                voff[u] = (uint32_t)(kDvRows - kPoisLag * u) * db + (uint32_t)r * (uint32_t)sizeof(double);
                lft[u] = cur[u] = 0;
                ge1[u] = ge0[u] = na1[u] = na0[u] = 0;
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int u = 0; u < MW; u++) dv[u][h] = dvs_at(u);
                advance_dvs();
            }
            // (waited for here: loads outstanding at the loop's entry would make
            // every turn wait for its newest ones)
#pragma unroll
            for (int u = 0; u < MW; u++) asm volatile("" : "+v"(dv[u][0]), "+v"(dv[u][1]));
            // a finished sweep's last row with a change >= tol since its last NaN,
            // and its last NaN; inner cells follow the boundary cells in sweep order
            auto flush = [&](int m, uint64_t ge, uint64_t na) {
                if (m < 0 || m >= g || (threadIdx.x & 63) != 0) return;
                if (ge) atomicMax(&fold[2 * m], 0x10001 + 2 * (w0 + 63 - __builtin_clzll(ge)));
                if (na) atomicMax(&fold[2 * m + 1], 0x10000 + 2 * (w0 + 63 - __builtin_clzll(na)));
            };
            for (int k = 0; k < steps; k += 2) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    double rgt[MW], qn[MW], qo[MW];
                    uint64_t doubt[MW], any = 0;
#pragma unroll
                    for (int u = 0; u < MW; u++) {
                        Lds* const f = at(rf[u]);
                        const double up = (double)at(rb[u])[0], dn = (double)f[2];
                        rgt[u] = (double)f[1];
                        qn[u] = up + dn;
                    }
#pragma unroll
                    for (int u = 0; u < MW; u++) {
                        const double v = dv[u][h];
                        int mark = __double2hiint(v);
                        asm("" : "+v"(mark));
                        const uint64_t inm = __ballot((unsigned)mark != kNotInner) &
                                             ((newest[u] & live1[u]) | (~newest[u] & live0[u]));
                        const bool in = __builtin_amdgcn_inverse_ballot_w64(inm);
                        qn[u] = rcp * (qn[u] * dy2 + (lft[u] + rgt[u]) * dx2 - v);
                        qo[u] = cur[u];
                        *(in ? at(rs[u]) + 1 : pdump) = (T)qn[u];
                        lft[u] = in ? (double)(T)qn[u] : qo[u];
                        cur[u] = rgt[u];
                        double t, b;
                        change_sides(qn[u], qo[u], tol, eps, t, b);
                        const uint64_t ge = __ballot(t > b) & inm;
                        doubt[u] = inm & ~__ballot(fabs(t) > b);
                        any |= doubt[u];
                        ge1[u] |= ge & newest[u];
                        ge0[u] |= ge & ~newest[u];
                    }
                    if (any) {
#pragma unroll
                        for (int u = 0; u < MW; u++) {
                            bool nan;
                            const uint64_t ge = __ballot(change_divided(qn[u], qo[u], tol, nan)) & doubt[u];
                            const uint64_t na = __ballot(nan) & doubt[u];
                            ge1[u] = (ge1[u] & ~(na & newest[u])) | (ge & newest[u]);
                            ge0[u] = (ge0[u] & ~(na & ~newest[u])) | (ge & ~newest[u]);
                            na1[u] |= na & newest[u];
                            na0[u] |= na & ~newest[u];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < MW; u++) {
                        rb[u] = rs[u];
                        rs[u] = rf[u];
                        rf[u] = rf[u] + qb == pb ? 0 : rf[u] + qb;
                        res[u]++;
                        if (res[u] == P) {  // a new turn: every row is out of the last sweep
                            flush(n[u] - D, ge0[u], na0[u]);
                            ge0[u] = ge1[u];
                            na0[u] = na1[u];
                            ge1[u] = na1[u] = 0;
                            n[u] += D;
                            set_live(u);
                            res[u] = 0;
                            newest[u] = 0;
                        }
                        // (res >= wr as bit arithmetic: a comparison's result would go
                        // through the vector unit)
                        newest[u] = newest[u] << 1 | (uint64_t)((uint32_t)~(res[u] - wr) >> 31);
                        dv[u][h] = dvs_at(u);
                    }
                    advance_dvs();
                    step_barrier();
                }
            }
#pragma unroll
            for (int u = 0; u < MW; u++) {
                flush(n[u] - D, ge0[u], na0[u]);
                flush(n[u], ge1[u], na1[u]);
            }
        } else {
            __builtin_amdgcn_s_setprio(3);  // the longest chain of a step
            const bool mine = mem < D;
            // step - k0 = turn P + res (lanes beyond the last member's: any diagonal)
            int res = mine && k0 ? P - k0 : 0, turn = mine && k0 ? -1 : 0;
            const uint2* const bl = blist + (mine ? e0 : 0);
            uint2 w[4];
            int pre = res;
#pragma unroll
            for (int h = 0; h < 4; h++) {
                w[h] = bl[pre * cpad];
                pre = next(pre);
            }
            // relaxes the cell of a list entry, if its sweep is one of the group's
            auto relax = [&](uint2 e) {
                const int n = (turn - (int)(e.y >> 16)) * D + mem;
                if (!mine || !(e.x & kBValid) || n < 0 || n >= g) return;
                T* const c = q + (e.y & 0xffff);
                T* const b = c + (res == 0 ? P - 1 : res - 1) * Q;
                T* const s = c + res * Q + 1;
                const T* const f = c + next(res) * Q;
                const double qo = (double)s[0], lf = (double)b[1], rt = (double)f[1];
                const double up = (double)b[0], dn = (double)f[2];
                const double i0 = e.x & (1u << 16) ? up : dn, i1 = e.x & (1u << 17) ? dn : up;
                const double j0 = e.x & (1u << 18) ? lf : rt, j1 = e.x & (1u << 19) ? rt : lf;
                // div is zero on boundary cells
                const double qn = rcp * ((i0 + i1) * dy2 + (j0 + j1) * dx2 - 0.0);
                s[0] = (T)qn;
                double t, m;
                change_sides(qn, qo, tol, eps, t, m);
                bool nan = false, ge = t > m;
                if (!(fabs(t) > m)) ge = change_divided(qn, qo, tol, nan);
                if (ge) atomicMax(&fold[2 * n], (int)(e.x & 0xffff));
                if (nan) atomicMax(&fold[2 * n + 1], (int)(e.x & 0xffff));
            };
            for (int k = 0; k < steps; k += 4) {
#pragma unroll
                for (int h = 0; h < 4; h++) {
                    relax(w[h]);
                    w[h] = bl[pre * cpad];  // after its use: no wait for this load before the next step's
                    pre = next(pre);
                    for (int e = epm; e < cpad; e += epm) relax(bl[res * cpad + e]);
                    res = next(res);
                    if (res == 0) turn++;
                    step_barrier();
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        __syncthreads();
        for (int n = threadIdx.x; n < g; n += blockDim.x)
            if (fold[2 * n] <= fold[2 * n + 1]) atomicMin(&s_first, n);
        __syncthreads();
        const int first = s_first;
        if (rerun || first + 1 == g) {  // a rerun ends on its last sweep
            sweeps += g;
            converged = true;
            break;
        }
        if (first < g) {
            for (int c = threadIdx.x; c < S; c += blockDim.x) q[c] = save[c];
            rerun = first + 1;
            __syncthreads();
            continue;
        }
        sweeps += g;
        left -= g;
        gsize = min(2 * gsize, kPoisGroup);
        __syncthreads();
    }
    __syncthreads();
    for (int c = threadIdx.x; c < S; c += blockDim.x) qgrid[c] = q[c];
    if (threadIdx.x == 0) {
        status[0] = sweeps;
        status[1] = converged ? 1 : 0;
    }
}

// Project's divergence field as k2s_poisson_lds reads it (one thread per
// element of dvs): div in the field type, times dx2 and dy2.
template <class T>
__global__ void k2s_div_skew(int nx, int ny, int P, int rp, const uint8_t* __restrict__ type, L3<T> w,
                             T dx, T dy, double dx2, double dy2, double* __restrict__ dvs) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (P + kDvRows) * rp) return;
    const int res = t / rp - kDvRows, i = t % rp;
    int j = (res - i) % P - 1;
    if (j < -1) j += P;
    double v = __hiloint2double((int)kNotInner, 0);
    if (i < nx && j >= 0 && j < ny) {
        const int64_t c = (int64_t)i * ny + j;
        if (type[c] == NODE_IN) {
            const T* U = w.f[0];
            const T* V = w.f[1];
            const T dv = (U[c + ny] - U[c - ny]) / (2 * dx) + (V[c + 1] - V[c - 1]) / (2 * dy);
            v = (double)dv * dx2 * dy2;
        }
    }
    dvs[t] = v;
}

// q of the anti-diagonal layout over the whole grid for the gradient.
template <class T>
__global__ void k2s_undiag(int nx, int ny, int P, const T* __restrict__ qgrid, T* __restrict__ qf) {
    const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= (int64_t)nx * ny) return;
    const int i = (int)(c / ny), j = (int)(c % ny);
    qf[c] = qgrid[(int64_t)((i + j + 1) % P) * (nx + 2) + i + 1];
}

// q over the whole grid (zero outside the spans) for the gradient.
template <class T>
__global__ void k2s_unspan(int nx, int ny, const int32_t* __restrict__ spans,
                           const T* __restrict__ qspan, T* __restrict__ qf) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (int64_t)nx * ny) return;
    const int i = (int)(q / ny), j = (int)(q % ny);
    const int o = spans[3 * i], l = spans[3 * i + 1], h = spans[3 * i + 2];
    qf[q] = (j >= l && j <= h) ? qspan[o + 1 + j - l] : (T)0;
}
}  // namespace

struct ISolver2 {
    virtual ~ISolver2() {}
    virtual int update_boundaries() = 0;
    virtual int step(double dt, int G, int L, double* err, int* iters) = 0;
    virtual int get_fields(void* u, void* v, void* p, void* T) = 0;
    virtual int set_poisson(double tol, int64_t max_sweeps) = 0;
    virtual int set_grid(const uint8_t* t, const uint8_t* bc, const double* vx, const double* vy,
                         const double* T) = 0;
    virtual int poisson_sweeps(int32_t* out, int max) = 0;
};

template <class T>
class Solver2D final : public ISolver2 {
   public:
    int nx, ny;
    int64_t N;
    hipStream_t st;
    P2 prm{};
    double startT;
    uint8_t *d_type = nullptr, *d_bc = nullptr;
    T* buf = nullptr;  // 8 layers x 3 fields: g, cur, next, half, temp, tl, nl, tl2
    L3<T> g{}, cur{}, next{}, half{}, temp{}, tl{}, nl{}, tl2{};
    Sys2 *d_rows = nullptr, *d_cols = nullptr;
    int nrows = 0, ncols = 0;
    int rows_nmax = 0, cols_nmax = 0;  // longest system of each direction
    T* scratch = nullptr;
    int64_t sc_half = 0;
    double* d_part = nullptr;
    double* d_err = nullptr;  // kErrSlots (sum, count) pairs of the divergence error
    double* h_err = nullptr;  // their pinned host copy
    static constexpr int kErrSlots = 64;
    int method = CMCX2D_ADI;
    // Stable solver: next_w, q over the whole grid, the relaxation's status words;
    // of k2s_poisson div, q per row's span, the spans and their cells' flags
    L3<T> nw{};
    T *d_nw = nullptr, *d_dv = nullptr, *d_qf = nullptr, *d_qspan = nullptr;
    T* d_save = nullptr;  // q at the start of a relaxation group
    int32_t* d_spans = nullptr;
    int32_t* d_doff = nullptr;  // first cell of each anti-diagonal, diagonal-major
    uint8_t* d_fspan = nullptr;
    int32_t* d_pstat = nullptr;
    int S = 0;
    // k2s_poisson_lds (rl_P != 0: q fits the LDS): its P, the slice
    // length, members, boundary wavefronts, boundary list pitch
    int rl_P = 0, rl_rp = 0, rl_D = 0, rl_mw = 1, rl_bw = 0, rl_cpad = 0;
    uint2* d_blist = nullptr;
    size_t blist_cap = 0;         // its entries
    std::vector<uint2> h_blist;   // its host copy, read until the stream has passed its upload
    double* d_dvs = nullptr;
    T *d_qpad = nullptr, *d_qsave = nullptr;
    double ptol = 1e-2;            // POISSON_ERR_THRESHOLD (StableSolver2D.h:23)
    int64_t pcap = 1000000;        // the reference has no cap
    std::vector<int32_t> sweeps;   // relaxation sweeps of each project of the last step
    static constexpr int kPoisChunk = 2048;  // sweeps per launch

    Solver2D(const cmcx2d_domain* d, const cmcx_params* p, int meth, hipStream_t stream) {
        st = stream;
        method = meth;
        nx = d->dims[0];
        ny = d->dims[1];
        N = (int64_t)nx * ny;
        prm = {0.0, d->h[0], d->h[1], p->v_T, p->v_vis, p->t_vis, p->t_phi};
        startT = d->start_t;
        CMCX_HIP(hipMalloc((void**)&d_type, N));
        CMCX_HIP(hipMalloc((void**)&d_bc, N));
        CMCX_HIP(hipMalloc((void**)&buf, sizeof(T) * N * 24));
        CMCX_HIP(hipMemsetAsync(buf, 0, sizeof(T) * N * 24, st));
        L3<T>* Ls[8] = {&g, &cur, &next, &half, &temp, &tl, &nl, &tl2};
        for (int l = 0; l < 8; l++)
            for (int f = 0; f < 3; f++) Ls[l]->f[f] = buf + (int64_t)(l * 3 + f) * N;
        CMCX_HIP(hipMemcpyAsync(d_type, d->type, N, hipMemcpyHostToDevice, st));
        CMCX_HIP(hipMemcpyAsync(d_bc, d->bc, N, hipMemcpyHostToDevice, st));
        {
            std::vector<T> h(N);
            const double* src[3] = {d->v[0], d->v[1], d->T};
            for (int f = 0; f < 3; f++) {
                for (int64_t i = 0; i < N; i++) h[i] = (T)src[f][i];
                CMCX_HIP(hipMemcpyAsync(g.f[f], h.data(), sizeof(T) * N, hipMemcpyHostToDevice, st));
                // AdiSolver2D::Init: the state starts as the node values everywhere
                CMCX_HIP(hipMemcpyAsync(cur.f[f], h.data(), sizeof(T) * N, hipMemcpyHostToDevice, st));
                CMCX_HIP(hipStreamSynchronize(st));
            }
        }
        if (method == CMCX2D_STABLE) build_relaxation(d->type);
        else build_systems(d->type);
        CMCX_HIP(hipMalloc((void**)&d_part, sizeof(double) * 2 * kDiv2Blocks * kErrSlots));
        CMCX_HIP(hipMalloc((void**)&d_err, sizeof(double) * 2 * kErrSlots));
        CMCX_HIP(hipHostMalloc((void**)&h_err, sizeof(double) * 2 * kErrSlots, hipHostMallocDefault));
        if (method == CMCX2D_STABLE) {
            // StableSolver2D::Init (StableSolver2D.cpp:44-52): next and temp from
            // the state (copies that skip the last row and column)
            copy(cur, next, kAll, 0);
            copy(cur, temp, kAll, 0);
        }
        CMCX_HIP(hipStreamSynchronize(st));
    }

    // PrepareIndices (StableSolver2D.cpp:167-188) for the fixed mask: the lists of
    // the relaxation that runs on grids of this size (the stream is waited for
    // before the host's copies are used again, see h_blist).
    void build_relaxation(const uint8_t* t) {
        auto T_ = [&](int i, int j) -> int {
            return (i < 0 || j < 0 || i >= nx || j >= ny) ? (int)NODE_OUT : t[(int64_t)i * ny + j];
        };
        for (int i = 0; i < nx; i++)
            for (int j = 0; j < ny; j++)
                if (T_(i, j) == NODE_IN && (i == 0 || j == 0 || i == nx - 1 || j == ny - 1))
                    throw std::string("2D Stable: a NODE_IN cell on the grid's edge (" + std::to_string(i) +
                                      ", " + std::to_string(j) + ")");
        if (nx > 512) throw std::string("2D Stable: grids of more than 512 rows (dimx) are not supported");
        if (!d_pstat) {
            CMCX_HIP(hipMalloc((void**)&d_nw, sizeof(T) * N * 2));
            CMCX_HIP(hipMalloc((void**)&d_qf, sizeof(T) * N));
            CMCX_HIP(hipMemsetAsync(d_nw, 0, sizeof(T) * N * 2, st));
            nw.f[0] = d_nw;
            nw.f[1] = d_nw + N;
            nw.f[2] = temp.f[2];  // never read or written (the step solves u and v only)
            CMCX_HIP(hipMalloc((void**)&d_pstat, sizeof(int32_t) * 4));
        }
        // q in LDS by anti-diagonals where it fits there and a cell's place in
        // sweep order 16 bits
        const int rp = (nx + 63) / 64 * 64, smax = std::max(1, std::min(15, (1024 - 64) / rp));
        int P = std::max(ny + 1, kPoisLag * smax);
        if (nx > P) P = std::min(nx, (P + 63) / 64 * 64);
        const int64_t cells = (int64_t)(nx + 2) * P;
        if (cells * (int64_t)sizeof(T) + 3072 > 160 * 1024 || cells > 0xffff) build_spans(t);
        else build_fronts(t, P, rp, smax);
    }

    // k2s_poisson: per row the span of non-outside cells and the cells' flags.
    void build_spans(const uint8_t* t) {
        auto T_ = [&](int i, int j) -> int {
            return (i < 0 || j < 0 || i >= nx || j >= ny) ? (int)NODE_OUT : t[(int64_t)i * ny + j];
        };
        std::vector<int32_t> sp(3 * (size_t)nx);
        std::vector<uint8_t> fl;
        for (int i = 0; i < nx; i++) {
            int lo = 0, hi = -1;
            for (int j = 0; j < ny; j++)
                if (T_(i, j) != NODE_OUT) {
                    if (hi < lo) lo = j;
                    hi = j;
                }
            // storage: a zero guard cell, columns lo .. hi, a zero guard cell
            sp[3 * i] = (int32_t)fl.size();
            sp[3 * i + 1] = lo;
            sp[3 * i + 2] = hi;
            fl.push_back(0);
            for (int j = lo; j <= hi; j++) {
                const int ty = T_(i, j);
                int f = ty == NODE_IN ? PF_IN : (ty == NODE_BOUND || ty == NODE_VALVE) ? PF_BOUND : 0;
                if (T_(i - 1, j) == NODE_IN) f |= PF_UP;
                if (T_(i + 1, j) == NODE_IN) f |= PF_DOWN;
                if (T_(i, j - 1) == NODE_IN) f |= PF_LEFT;
                if (T_(i, j + 1) == NODE_IN) f |= PF_RIGHT;
                fl.push_back((uint8_t)f);
            }
            fl.push_back(0);
        }
        fl.push_back(0);  // one more guard: the last row's reads stay inside
        // the arrays once, for spans as long as they can be
        if (!d_save) {
            const size_t most = (size_t)nx * (ny + 2) + 1;
            std::vector<int32_t> doff(nx + ny);
            for (int d = 0, o = 0; d < nx + ny; d++) {
                doff[d] = o;
                if (d < nx + ny - 1) o += std::min(d, nx - 1) - std::max(0, d - ny + 1) + 1;
            }
            CMCX_HIP(hipMalloc((void**)&d_doff, sizeof(int32_t) * doff.size()));
            CMCX_HIP(hipMemcpy(d_doff, doff.data(), sizeof(int32_t) * doff.size(), hipMemcpyHostToDevice));
            CMCX_HIP(hipMalloc((void**)&d_dv, sizeof(T) * N));
            CMCX_HIP(hipMalloc((void**)&d_spans, sizeof(int32_t) * sp.size()));
            CMCX_HIP(hipMalloc((void**)&d_fspan, most));
            CMCX_HIP(hipMalloc((void**)&d_qspan, sizeof(T) * most));
            CMCX_HIP(hipMalloc((void**)&d_save, sizeof(T) * most));
        }
        S = (int)fl.size();
        CMCX_HIP(hipMemcpyAsync(d_spans, sp.data(), sizeof(int32_t) * sp.size(), hipMemcpyHostToDevice, st));
        CMCX_HIP(hipMemcpyAsync(d_fspan, fl.data(), S, hipMemcpyHostToDevice, st));
        CMCX_HIP(hipStreamSynchronize(st));
    }

    // k2s_poisson_lds: its layout and boundary lists.  The arrays are kept from
    // grid to grid: allocated anew for each, beside the spans that this relaxation
    // does not read, they took SetGrid on a 120 x 135 grid to 197 us; kept, it takes 92.
    void build_fronts(const uint8_t* t, int P, int rp, int smax) {
        auto T_ = [&](int i, int j) -> int {
            return (i < 0 || j < 0 || i >= nx || j >= ny) ? (int)NODE_OUT : t[(int64_t)i * ny + j];
        };
        std::vector<int> len(P, 0);
        auto each = [&](auto&& cell) {
            for (int i = 0; i < nx; i++)
                for (int j = 0; j < ny; j++) {
                    const int ty = t[(int64_t)i * ny + j];
                    if (ty == NODE_BOUND || ty == NODE_VALVE) cell(i, j);
                }
        };
        each([&](int i, int j) { len[(i + j + 1) % P]++; });
        const int cmax = std::max(1, *std::max_element(len.begin(), len.end()));
        // sweeps per slice as the row length allows; as many slices as leave the
        // boundary wavefronts a lane for every boundary cell of a front (at
        // least half of them otherwise)
        int D = 0, bw = 1, mw = 1;
        for (int sl = smax; sl >= std::max(1, smax / 2); sl--) {
            const int room = 16 - sl * rp / 64;
            mw = kPoisLag * 2 * sl <= P ? 2 : 1;
            D = mw * sl;
            bw = std::min(room, std::max((cmax * D + 63) / 64, 1));
            if (64 * bw / D >= cmax) break;
        }
        const int epm = 64 * bw / D, cpad = (cmax + epm - 1) / epm * epm;
        CMCX_HIP(hipStreamSynchronize(st));  // h_blist on its way, d_blist in use
        h_blist.assign((size_t)P * cpad, uint2{0, 0});
        std::fill(len.begin(), len.end(), 0);
        each([&](int i, int j) {
            const int x = j + 1, q = (i + x) % P;
            uint32_t w = kBValid | (uint32_t)(i * P + x);
            if (T_(i - 1, j) == NODE_IN) w |= 1u << 16;
            if (T_(i + 1, j) == NODE_IN) w |= 1u << 17;
            if (T_(i, j - 1) == NODE_IN) w |= 1u << 18;
            if (T_(i, j + 1) == NODE_IN) w |= 1u << 19;
            h_blist[(size_t)q * cpad + len[q]++] = uint2{w, (uint32_t)i | (uint32_t)((i + x) / P) << 16};
        });
        if (!d_qsave) {
            const int64_t cells = (int64_t)(nx + 2) * P;
            CMCX_HIP(hipMalloc((void**)&d_dvs, sizeof(double) * (P + kDvRows) * rp));
            CMCX_HIP(hipMalloc((void**)&d_qpad, sizeof(T) * cells));
            CMCX_HIP(hipMalloc((void**)&d_qsave, sizeof(T) * cells));
        }
        if (h_blist.size() > blist_cap) {
            uint2* p = nullptr;
            CMCX_HIP(hipMalloc((void**)&p, sizeof(uint2) * h_blist.size()));
            hipFree(d_blist);
            d_blist = p;
            blist_cap = h_blist.size();
        }
        CMCX_HIP(hipMemcpyAsync(d_blist, h_blist.data(), sizeof(uint2) * h_blist.size(), hipMemcpyHostToDevice, st));
        rl_P = P;
        rl_rp = rp;
        rl_D = D;
        rl_mw = mw;
        rl_bw = bw;
        rl_cpad = cpad;
    }

    // Grid2D::Prepare(t) between steps (FluidSolver2D.cpp:131): new cell types,
    // BC kinds and node values; the line systems (ADI) or the relaxation's
    // lists (Stable) follow the new types, as the reference rebuilds them
    // every step.
    int set_grid(const uint8_t* t, const uint8_t* bc, const double* vx, const double* vy,
                 const double* Tt) override {
        if (!t || !bc || !vx || !vy || !Tt) return CMCX_ERR_ARG;
        for (int64_t i = 0; i < N; i++)
            if (t[i] > 3 || bc[i] > 1) {
                set_error("node type or BC kind out of range at node " + std::to_string(i));
                return CMCX_ERR_ARG;
            }
        if (method == CMCX2D_STABLE) build_relaxation(t);
        else build_systems(t);
        CMCX_HIP(hipMemcpyAsync(d_type, t, N, hipMemcpyHostToDevice, st));
        CMCX_HIP(hipMemcpyAsync(d_bc, bc, N, hipMemcpyHostToDevice, st));
        std::vector<T> h(N);
        const double* src[3] = {vx, vy, Tt};
        for (int f = 0; f < 3; f++) {
            for (int64_t i = 0; i < N; i++) h[i] = (T)src[f][i];
            CMCX_HIP(hipMemcpyAsync(g.f[f], h.data(), sizeof(T) * N, hipMemcpyHostToDevice, st));
            CMCX_HIP(hipStreamSynchronize(st));
        }
        return CMCX_OK;
    }

    ~Solver2D() override {
        hipStreamSynchronize(st);
        hipFree(d_type);
        hipFree(d_bc);
        hipFree(buf);
        hipFree(d_rows);
        hipFree(d_cols);
        hipFree(scratch);
        hipFree(d_part);
        hipFree(d_err);
        hipHostFree(h_err);
        hipFree(d_nw);
        hipFree(d_dv);
        hipFree(d_qf);
        hipFree(d_qspan);
        hipFree(d_save);
        hipFree(d_blist);
        hipFree(d_dvs);
        hipFree(d_qpad);
        hipFree(d_qsave);
        hipFree(d_doff);
        hipFree(d_spans);
        hipFree(d_fspan);
        hipFree(d_pstat);
    }

    // AdiSolver2D::CreateSegments, for each new mask.  Types that are refused, or a
    // failed allocation, leave the lists there were.
    void build_systems(const uint8_t* t) {
        auto T_ = [&](int i, int j) { return t[(int64_t)i * ny + j]; };
        std::vector<Sys2> rows, cols;
        for (int j = 0; j < ny; j++) {
            int i = 0;
            while (i < nx && T_(i, j) == NODE_OUT) i++;
            while (i + 1 < nx && T_(i + 1, j) != NODE_IN) i++;
            if (i + 1 >= nx) continue;
            const int a = i;
            i = nx - 1;
            while (i >= 0 && T_(i, j) == NODE_OUT) i--;
            while (i - 1 >= 0 && T_(i - 1, j) != NODE_IN) i--;
            rows.push_back({a, j, i});
        }
        for (int i = 0; i < nx; i++) {
            int j = 0;
            while (j < ny && T_(i, j) == NODE_OUT) j++;
            while (j + 1 < ny && T_(i, j + 1) != NODE_IN) j++;
            if (j + 1 >= ny) continue;
            const int a = j;
            j = ny - 1;
            while (j >= 0 && T_(i, j) == NODE_OUT) j--;
            while (j - 1 >= 0 && T_(i, j - 1) != NODE_IN) j--;
            cols.push_back({i, a, j});
        }
        for (const Sys2& s : rows)
            if (s.b - s.a0 + 1 < 2) throw std::string("2D: a line system shorter than 2 nodes");
        for (const Sys2& s : cols)
            if (s.b - s.a1 + 1 < 2) throw std::string("2D: a line system shorter than 2 nodes");
        const int64_t nsys = std::max<int64_t>(std::max(rows.size(), cols.size()), 1);
        const int64_t half = (int64_t)std::max(nx, ny) * 3 * nsys;
        Sys2 *nr = nullptr, *nc = nullptr;
        T* ns = nullptr;
        try {
            if (!rows.empty()) {
                CMCX_HIP(hipMalloc((void**)&nr, sizeof(Sys2) * rows.size()));
                CMCX_HIP(hipMemcpy(nr, rows.data(), sizeof(Sys2) * rows.size(), hipMemcpyHostToDevice));
            }
            if (!cols.empty()) {
                CMCX_HIP(hipMalloc((void**)&nc, sizeof(Sys2) * cols.size()));
                CMCX_HIP(hipMemcpy(nc, cols.data(), sizeof(Sys2) * cols.size(), hipMemcpyHostToDevice));
            }
            if (half > sc_half) CMCX_HIP(hipMalloc((void**)&ns, sizeof(T) * 2 * half));
            CMCX_HIP(hipStreamSynchronize(st));  // the old lists' last reader
        } catch (...) {
            hipFree(nr);
            hipFree(nc);
            hipFree(ns);
            throw;
        }
        hipFree(d_rows);
        hipFree(d_cols);
        d_rows = nr;
        d_cols = nc;
        if (ns) {
            hipFree(scratch);
            scratch = ns;
            sc_half = half;
        }
        nrows = (int)rows.size();
        ncols = (int)cols.size();
        rows_nmax = cols_nmax = 0;
        for (const Sys2& s : rows) rows_nmax = std::max(rows_nmax, s.b - s.a0 + 1);
        for (const Sys2& s : cols) cols_nmax = std::max(cols_nmax, s.b - s.a1 + 1);
    }

    void copy(L3<T> src, L3<T> dst, int mask, int merge) {
        hipLaunchKernelGGL((k2_copy<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_type, mask,
                           merge, src, dst);
        CMCX_LAUNCH_CHECK();
    }

    static constexpr int kAll = 0xF, kIn = 1 << NODE_IN;

    // one inner iteration, and both directions' rows fit the LDS (sweep_lds)
    bool one_pass(int L) const { return L == 1 && nrows && ncols && lds_spw(true) && lds_spw(false); }

    // Systems per work-group of k2_sweep_lds for a direction (0: its rows do
    // not fit the LDS): a power of two, small enough that the launch spreads
    // over about 128 work-groups (the recurrences are serial; more systems per
    // work-group only lengthen its row-building phase), and within 150 KiB.
    int lds_spw(bool dirx) const {
        const int n = dirx ? nrows : ncols, nmax = dirx ? rows_nmax : cols_nmax;
        const int64_t per = (int64_t)nmax * (sizeof(Row4<T>) + 1);
        int spw = 1;
        while (spw < kSweepLdsThreads && (int64_t)(2 * spw) * per <= 150 * 1024 &&
               (int64_t)n * 3 / (2 * spw) >= 128)
            spw *= 2;
        return per <= 150 * 1024 ? spw : 0;
    }

    // Rows after which an error in c', d' or x has shrunk below the rounding of a
    // line's values, from the viscous part of the rows (its |c'| for constant
    // rows): the length of the chunks' early starts, at most the longest line.  0:
    // lines are solved serially (k2_sweep_lds): too many rows or systems, or so few
    // rows (under 22, stiff ones under 32) that the early starts (about 0.3 of a
    // serial row each) and the exact ones cost most of the line.
    // Longer lines stay with the chunks however little an error shrinks, by stiff
    // rows or by a flow of many cells per step, which the estimate does not see.
    // Chunks are then run again up to 64 times, which still costs less than one
    // lane's chain, as d' is settled by passes without divisions: at |c'| = 0.99, us
    // serially and in chunks, FP64 256 rows 58.2 / 39.9, 128 rows 30.9 / 26.3, 48 rows
    // 14.1 / 10.3; FP32 500 rows 95.9 / 67.0, 60 rows 16.5 / 17.6; at 20 cells per step
    // a step of a 500 x 60 FP64 grid 739 / 269.  Grids of 33^2 to 200^2 with dt nu / h^2 of
    // 0.01 to 5e4 and two local iterations take 0.42 to 0.86 of the serial steps' time.
    int early_rows(bool dirx) const {
        const int n = dirx ? nrows : ncols, nmax = dirx ? rows_nmax : cols_nmax;
        if (nmax > kChunkMaxRows || 3 * n > kChunkMaxSystems) return 0;
        const double h = dirx ? prm.dx : prm.dy, vis = std::max(prm.v_vis, prm.t_vis) / (h * h);
        const double b = 1.0 / prm.dt + 2 * vis;
        double w = 0;
        if (vis > 0) {
            const double c = (b - std::sqrt(b * b - 4 * vis * vis)) / (2 * vis);
            w = (sizeof(T) == 8 ? 56 : 27) / -std::log2(c);
        }
        const double rows = w + 4;
        if (!(rows >= 4) || 0.3 * std::min<double>(rows, nmax) + kChunkExact + 4 > 0.8 * nmax) return 0;
        return (int)std::min<double>(rows, nmax);
    }

    // mode 1: the solve writes lt, out and, where given, t2 (a copy of lt that is
    // kept up to date) on the NODE_IN rows (a direction with one inner iteration),
    // else the solution into out.  k2_sweep_lds leaves t2 to a copy: a third
    // store per row lengthens its serial back substitution (FP64 rows of 700: X 389
    // -> 413 us; of 2000: 4508 -> 4824, where the copy takes 36).
    void sweep_lds(bool dirx, int spw, int mode, L3<T> lc, L3<T> tlc, L3<T> out, L3<T> lt, L3<T> t2 = {}) {
        const int n = dirx ? nrows : ncols, nmax = dirx ? rows_nmax : cols_nmax;
        if (const int early = early_rows(dirx)) {
            // a wavefront per system
            const int cl = nmax <= 64 * 4 ? 4 : 8;
            const int w = (std::max(early, kChunkExact + 4) + cl - 1) / cl * cl, wa = w - kChunkExact;
            const int wb = (early + 3) / 4 * 4, pitch = chunk_pitch(chunk_rows(nmax, w, wb, cl), cl);
            int per = std::min(spw, kSweepLdsThreads / 64);
            while (per > 1 && per * pitch * sizeof(Row4<T>) > 150 * 1024) per /= 2;
            auto kern = dirx ? (cl == 4 ? k2_sweep_chunks<T, true, 4> : k2_sweep_chunks<T, true, 8>)
                             : (cl == 4 ? k2_sweep_chunks<T, false, 4> : k2_sweep_chunks<T, false, 8>);
            hipLaunchKernelGGL(kern, dim3((unsigned)((n + per - 1) / per), 3), dim3(kSweepLdsThreads),
                               (size_t)per * pitch * sizeof(Row4<T>), st, n, per, nmax, dirx ? d_rows : d_cols, nx, ny, d_type,
                               d_bc, g, lc, tlc, out, lt, t2, mode, prm, wa, wb);
            CMCX_LAUNCH_CHECK();
            return;
        }
        const size_t lds = (size_t)spw * nmax * (sizeof(Row4<T>) + 1);
        const dim3 grid((unsigned)((n + spw - 1) / spw), 3);
        if (dirx)
            hipLaunchKernelGGL((k2_sweep_lds<T, true>), grid, dim3(kSweepLdsThreads), lds, st, n,
                               spw, nmax, d_rows, nx, ny, d_type, d_bc, g, lc, tlc, out, lt, nl,
                               mode, prm);
        else
            hipLaunchKernelGGL((k2_sweep_lds<T, false>), grid, dim3(kSweepLdsThreads), lds, st, n,
                               spw, nmax, d_cols, nx, ny, d_type, d_bc, g, lc, tlc, out, lt, nl,
                               mode, prm);
        CMCX_LAUNCH_CHECK();
        if (t2.f[0]) copy(lt, t2, kAll, 0);
    }

    void sweep(bool dirx, L3<T> lc, L3<T> lt, L3<T> out) {
        const int n = dirx ? nrows : ncols;
        if (!n) return;
        if (const int spw = lds_spw(dirx)) {
            sweep_lds(dirx, spw, 0, lc, lt, out, L3<T>{});
            return;
        }
        // sc/sd indexing uses the launch's system count as the stride
        if (dirx)
            hipLaunchKernelGGL((k2_sweep<T, true>), dim3(blocks2(n), 3), dim3(kBS2), 0, st, n,
                               d_rows, nx, ny, d_bc, g, lc, lt, out, prm, scratch,
                               scratch + sc_half);
        else
            hipLaunchKernelGGL((k2_sweep<T, false>), dim3(blocks2(n), 3), dim3(kBS2), 0, st, n,
                               d_cols, nx, ny, d_bc, g, lc, lt, out, prm, scratch,
                               scratch + sc_half);
        CMCX_LAUNCH_CHECK();
    }

    // AdiSolver2D::SolveDirection
    void direction(bool dirx, int L, L3<T> lc, L3<T> lt, L3<T> out) {
        if (!(dirx ? nrows : ncols)) return;  // the reference reads list[0] unconditionally
        copy(lt, tl, kAll, 0);
        if (L == 1) {
            if (const int spw = lds_spw(dirx)) {
                // the solve writes what the copies below would leave on NODE_IN
                // (the local layer is read for the stencils, lt and out are not)
                sweep_lds(dirx, spw, 1, lc, tl, out, lt);
                return;
            }
        }
        for (int it = 0; it < L; it++) {
            sweep(dirx, lc, tl, nl);
            copy(nl, tl, kIn, it == 0 ? 0 : 1);
        }
        copy(tl, lt, kIn, 0);
        copy(nl, out, kIn, 0);
    }

    // The divergence error of Lr into slot `slot` (sum and count), no wait.
    void div_enqueue(L3<T> Lr, int slot) {
        hipLaunchKernelGGL((k2_div<T>), dim3(kDiv2Blocks), dim3(kBS2), 0, st, nx, ny, d_type, Lr,
                           (T)prm.dx, (T)prm.dy, d_part);
        CMCX_LAUNCH_CHECK();
        hipLaunchKernelGGL(k2_div_finish, dim3(1), dim3(kDiv2Blocks), 0, st, d_part, kDiv2Blocks,
                           d_err + 2 * slot);
        CMCX_LAUNCH_CHECK();
    }

    // The first n slots into h_err (waits for the stream).
    void read_errors(int n) {
        CMCX_HIP(hipMemcpyAsync(h_err, d_err, sizeof(double) * 2 * n, hipMemcpyDeviceToHost, st));
        CMCX_HIP(hipStreamSynchronize(st));
    }

    double div_error(L3<T> Lr) {
        div_enqueue(Lr, 0);
        read_errors(1);
        return h_err[0] / h_err[1];
    }

    void end_step() {
        hipLaunchKernelGGL((k2_end_step<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_type, next, cur,
                           (T)startT);
        CMCX_LAUNCH_CHECK();
    }

    int update_boundaries() override {
        hipLaunchKernelGGL((k2_update_boundaries<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny,
                           d_type, g, cur, next);
        CMCX_LAUNCH_CHECK();
        return CMCX_OK;
    }

    int set_poisson(double tol, int64_t max_sweeps) override {
        if (!(tol > 0) || max_sweeps < 1) return CMCX_ERR_ARG;
        ptol = tol;
        pcap = max_sweeps;
        return CMCX_OK;
    }

    int poisson_sweeps(int32_t* out, int max) override {
        for (int k = 0; k < max && k < (int)sweeps.size(); k++) out[k] = sweeps[k];
        return (int)sweeps.size();
    }

    // Sweeps in flight: as many member slices of rp threads as a 1024-thread
    // work-group holds, at most 8.
    template <bool QLDS>
    void launch_poisson_for(int rp, size_t lds, double dx2, double dy2, double rcp, int chunk, int resume) {
        const int D = std::min(8, 1024 / rp);
        hipLaunchKernelGGL((k2s_poisson<T, QLDS>), dim3(1), dim3(rp * D), lds, st, nx, ny, S, rp, D,
                           d_spans, d_fspan, d_doff, d_dv, d_qspan, d_save, dx2, dy2, rcp, ptol, chunk,
                           resume, d_pstat);
        CMCX_LAUNCH_CHECK();
    }

    // StableSolver2D::Project (StableSolver2D.cpp:83-165): w -> next on NODE_IN.
    // Returns false when the relaxation reached the sweep cap.
    bool project() {
        const double dx2 = prm.dx * prm.dx, dy2 = prm.dy * prm.dy, rcp = 0.5 / (dx2 + dy2);
        const bool fronts = rl_P != 0;
        if (fronts)
            hipLaunchKernelGGL((k2s_div_skew<T>), dim3(blocks2((int64_t)(rl_P + kDvRows) * rl_rp)), dim3(kBS2), 0,
                               st, nx, ny, rl_P, rl_rp, d_type, nw, (T)prm.dx, (T)prm.dy, dx2, dy2, d_dvs);
        else
            hipLaunchKernelGGL((k2s_div<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_type, nw,
                               (T)prm.dx, (T)prm.dy, d_doff, d_dv);
        CMCX_LAUNCH_CHECK();
        const int rp = std::max(64, (nx + 63) / 64 * 64);  // threads per set
        const size_t lds = (size_t)S * sizeof(T) + (size_t)S;
        const bool in_lds = lds + 2048 <= 160 * 1024;
        int64_t total = 0;
        bool done = false;
        for (int resume = 0; !done && total < pcap; resume = 1) {
            const int chunk = (int)std::min<int64_t>(kPoisChunk, pcap - total);
            if (fronts) {
                auto kern = rl_mw == 2 ? k2s_poisson_lds<T, 2> : k2s_poisson_lds<T, 1>;
                hipLaunchKernelGGL(kern, dim3(1), dim3(rl_D / rl_mw * rl_rp + 64 * rl_bw),
                                   sizeof(T) * (size_t)(nx + 2) * rl_P, st, nx, ny, rl_P, rl_rp, rl_D, rl_bw,
                                   rl_cpad, d_blist, d_dvs, d_qpad, d_qsave, dx2, dy2, rcp, ptol, chunk,
                                   resume, d_pstat);
                CMCX_LAUNCH_CHECK();
            } else if (in_lds) launch_poisson_for<true>(rp, lds, dx2, dy2, rcp, chunk, resume);
            else launch_poisson_for<false>(rp, 0, dx2, dy2, rcp, chunk, resume);
            int32_t h[2];
            CMCX_HIP(hipMemcpyAsync(h, d_pstat, sizeof(h), hipMemcpyDeviceToHost, st));
            CMCX_HIP(hipStreamSynchronize(st));
            total = h[0];
            done = h[1] != 0;
        }
        sweeps.push_back((int32_t)std::min<int64_t>(total, INT32_MAX));
        if (!done) return false;
        if (fronts)
            hipLaunchKernelGGL((k2s_undiag<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, rl_P, d_qpad, d_qf);
        else hipLaunchKernelGGL((k2s_unspan<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_spans, d_qspan,
                           d_qf);
        hipLaunchKernelGGL((k2s_grad<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_type, nw, d_qf,
                           (T)prm.dx, (T)prm.dy, next);
        CMCX_LAUNCH_CHECK();
        return true;
    }

    // StableSolver2D::TimeStep (StableSolver2D.cpp:190-234)
    int stable_step(double dt, int G, double* err_out, int* iters) {
        if (G < 0) return CMCX_ERR_ARG;
        prm.dt = dt;
        sweeps.clear();
        copy(cur, temp, kAll, 0);
        double err = div_error(next);
        int it;
        for (it = 0; it < G || err > 0.1; it++) {
            copy(cur, nw, kAll, 0);
            hipLaunchKernelGGL((k2s_solve_uv<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, d_type, cur,
                               temp, nw, (T)dt, (T)prm.dx, (T)prm.dy, (T)prm.v_vis);
            CMCX_LAUNCH_CHECK();
            if (!project()) {
                if (iters) *iters = it + 1;
                set_error("2D Stable: the Poisson relaxation did not converge within " +
                          std::to_string(pcap) + " sweeps");
                return CMCX_ERR_PICARD;
            }
            err = div_error(next);
            copy(next, temp, kIn, 1);
            if (it > 100 || err > 0.1 * 10) {
                if (err_out) *err_out = err;
                if (iters) *iters = it + 1;
                set_error(it > 100 ? "2D: Picard iterations exceeded 100" : "2D: divergence error above 1.0");
                return CMCX_ERR_PICARD;
            }
        }
        end_step();
        CMCX_HIP(hipStreamSynchronize(st));
        if (err_out) *err_out = err;
        if (iters) *iters = it;
        return CMCX_OK;
    }

    // AdiSolver2D::TimeStep (AdiSolver2D.cpp:279-323)
    int step(double dt, int G, int L, double* err_out, int* iters) override {
        if (method == CMCX2D_STABLE) return stable_step(dt, G, err_out, iters);
        if (G < 0 || L < 1) return CMCX_ERR_ARG;
        prm.dt = dt;
        const bool fused = one_pass(L);
        // the Picard layer's second copy, unless a copy makes it (sweep_lds)
        const L3<T> second = fused && early_rows(true) ? tl2 : L3<T>{};
        if (fused) {
            hipLaunchKernelGGL((k2_fan<T>), dim3(blocks2(N)), dim3(kBS2), 0, st, nx, ny, cur, next,
                               half, temp, tl, second);
            CMCX_LAUNCH_CHECK();
        } else {
            copy(cur, next, kAll, 0);
            copy(cur, half, kAll, 0);
            copy(cur, temp, kAll, 0);
        }
        // the error before the loop decides only whether a step with G = 0 iterates
        double err = G == 0 ? div_error(next) : 0.0;
        int it = 0;
        // Iterations below G run whatever their error (only an error above 1.0
        // ends them, with CMCX_ERR_PICARD and the state unchanged), so they are
        // queued back to back with their errors in slots that are read once.
        // Iterations queued after an erroring one change only working layers,
        // which the next step's copies overwrite before anything reads them.
        const int batch = std::min(G, (int)kErrSlots);
        for (int k = 0; k < batch; k++) {
            if (fused) {
                // tl and tl2 hold the Picard layer (k2_fan, k2_merge_div); the X
                // sweep brings tl2 up to date for the Y sweep
                sweep_lds(true, lds_spw(true), 1, cur, tl, half, temp, tl2);
                sweep_lds(false, lds_spw(false), 1, half, tl2, next, temp);
                hipLaunchKernelGGL((k2_merge_div<T>), dim3(std::max<unsigned>(kDiv2Blocks, blocks2(N))), dim3(kBS2), 0,
                                   st, nx, ny, d_type, k == 0 ? 0 : 1, next, temp, tl, second, (T)prm.dx, (T)prm.dy,
                                   d_part + (int64_t)k * 2 * kDiv2Blocks);
                CMCX_LAUNCH_CHECK();
            } else {
                direction(true, L, cur, temp, half);
                direction(false, L, half, temp, next);
                div_enqueue(next, k);
                copy(next, temp, kIn, k == 0 ? 0 : 1);
            }
        }
        if (fused && batch > 0) {
            hipLaunchKernelGGL(k2_div_finish, dim3(batch), dim3(kDiv2Blocks), 0, st, d_part, kDiv2Blocks, d_err);
            CMCX_LAUNCH_CHECK();
        }
        if (batch > 0) {
            read_errors(batch);
            for (int k = 0; k < batch; k++) {
                err = h_err[2 * k] / h_err[2 * k + 1];
                if (k > 100 || err > 0.1 * 10) {
                    if (err_out) *err_out = err;
                    if (iters) *iters = k + 1;
                    set_error(k > 100 ? "2D: Picard iterations exceeded 100"
                                      : "2D: divergence error above 1.0");
                    return CMCX_ERR_PICARD;
                }
            }
            it = batch;
        }
        for (; it < G || err > 0.1; it++) {
            direction(true, L, cur, temp, half);
            direction(false, L, half, temp, next);
            err = div_error(next);
            copy(next, temp, kIn, it == 0 ? 0 : 1);
            if (it > 100 || err > 0.1 * 10) {
                if (err_out) *err_out = err;
                if (iters) *iters = it + 1;
                set_error(it > 100 ? "2D: Picard iterations exceeded 100"
                                   : "2D: divergence error above 1.0");
                return CMCX_ERR_PICARD;
            }
        }
        end_step();
        CMCX_HIP(hipStreamSynchronize(st));
        if (err_out) *err_out = err;
        if (iters) *iters = it;
        return CMCX_OK;
    }

    int get_fields(void* u, void* v, void* p, void* Tt) override {
        void* dst[3] = {u, v, Tt};
        for (int f = 0; f < 3; f++)
            if (dst[f])
                CMCX_HIP(hipMemcpyAsync(dst[f], cur.f[f], sizeof(T) * N, hipMemcpyDeviceToHost, st));
        CMCX_HIP(hipStreamSynchronize(st));
        if (p) {
            std::vector<T> t(N);
            CMCX_HIP(hipMemcpy(t.data(), cur.f[2], sizeof(T) * N, hipMemcpyDeviceToHost));
            T* pp = (T*)p;
            const T vT = (T)prm.v_T;
            for (int64_t i = 0; i < N; i++) pp[i] = vT * t[i];
        }
        return CMCX_OK;
    }
};

}  // namespace cmcx

struct cmcx2d_solver {
    std::unique_ptr<cmcx::ISolver2> impl;
};

#define CMCX2_GUARD(body)                                                                       \
    try {                                                                                       \
        body                                                                                    \
    } catch (const cmcx::HipError& e) {                                                         \
        cmcx::set_error(std::string("HIP error ") + hipGetErrorString(e.code) + " in " + e.where); \
        return CMCX_ERR_HIP;                                                                    \
    } catch (const std::string& e) {                                                            \
        cmcx::set_error(e);                                                                     \
        return CMCX_ERR_ARG;                                                                    \
    } catch (const std::exception& e) {                                                         \
        cmcx::set_error(e.what());                                                              \
        return CMCX_ERR_ARG;                                                                    \
    }

extern "C" {

int cmcx2d_create(const cmcx2d_domain* d, const cmcx_params* p, int dtype, void* stream,
                  cmcx2d_solver** out) {
    return cmcx2d_create_method(d, p, CMCX2D_ADI, dtype, stream, out);
}

int cmcx2d_create_method(const cmcx2d_domain* d, const cmcx_params* p, int method, int dtype,
                         void* stream, cmcx2d_solver** out) {
    if (!d || !p || !out) return CMCX_ERR_ARG;
    *out = nullptr;
    if (dtype != CMCX_F32 && dtype != CMCX_F64) return CMCX_ERR_ARG;
    if (method != CMCX2D_ADI && method != CMCX2D_STABLE) {
        cmcx::set_error("cmcx2d_create_method: method must be CMCX2D_ADI or CMCX2D_STABLE");
        return CMCX_ERR_ARG;
    }
    if (d->dims[0] < 3 || d->dims[1] < 3 || !d->type || !d->bc || !d->v[0] || !d->v[1] || !d->T)
        return CMCX_ERR_ARG;
    const int64_t N = (int64_t)d->dims[0] * d->dims[1];
    for (int64_t i = 0; i < N; i++)
        if (d->type[i] > 3 || d->bc[i] > 1) {
            cmcx::set_error("node type or BC kind out of range at node " + std::to_string(i));
            return CMCX_ERR_ARG;
        }
    CMCX2_GUARD({
        auto* s = new cmcx2d_solver;
        try {
            if (dtype == CMCX_F32)
                s->impl.reset(new cmcx::Solver2D<float>(d, p, method, (hipStream_t)stream));
            else s->impl.reset(new cmcx::Solver2D<double>(d, p, method, (hipStream_t)stream));
        } catch (...) {
            delete s;
            throw;
        }
        *out = s;
        return CMCX_OK;
    })
}

int cmcx2d_update_boundaries(cmcx2d_solver* s) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD(return s->impl->update_boundaries();)
}

int cmcx2d_step(cmcx2d_solver* s, double dt, int G, int L, double* err, int* iters) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD(return s->impl->step(dt, G, L, err, iters);)
}

int cmcx2d_get_fields(cmcx2d_solver* s, void* u, void* v, void* p, void* T) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD(return s->impl->get_fields(u, v, p, T);)
}

int cmcx2d_set_grid(cmcx2d_solver* s, const uint8_t* type, const uint8_t* bc, const double* vx,
                    const double* vy, const double* T) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD(return s->impl->set_grid(type, bc, vx, vy, T);)
}

int cmcx2d_set_poisson(cmcx2d_solver* s, double tol, int64_t max_sweeps) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD(return s->impl->set_poisson(tol, max_sweeps);)
}

int cmcx2d_poisson_sweeps(cmcx2d_solver* s, int32_t* out, int max, int* count) {
    if (!s || !count || (max > 0 && !out)) return CMCX_ERR_ARG;
    CMCX2_GUARD({
        *count = s->impl->poisson_sweeps(out, max);
        return CMCX_OK;
    })
}

int cmcx2d_destroy(cmcx2d_solver* s) {
    if (!s) return CMCX_ERR_ARG;
    CMCX2_GUARD({
        delete s;
        return CMCX_OK;
    })
}

}  // extern "C"
