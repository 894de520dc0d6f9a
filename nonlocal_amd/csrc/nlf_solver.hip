// Krylov layer: CSR SpMV, CG (conjugate_gradient.hpp:48-79), Jacobi and ILLT preconditioners
// (eigen_preconditioner.hpp:50-57), FP32-inner / FP64-refinement mixed mode.
//
// The products read the upper triangle from slices (nlf_symv.inl), or the full (both-triangle) storage where
// that does not apply: every output row is a gather there (no scatter, no atomics, deterministic) and LPR
// lanes cooperate on one row.  CG keeps its scalars on the device in a state block; an iteration is the
// product with its dot, the update with the Jacobi preconditioner and its dot (or the two sweeps and their
// finish) and the p update, which form alpha and beta themselves, with no host synchronisation; the host
// reads the state every few iterations.
//
// ILLT: IC(0) of the local matrix, diagonal scaling s = 1/sqrt|a_ii| and shift retries (our choice:
// Eigen::IncompleteCholesky is not vendored, so its factor is not reproduced).  Rows are grouped by
// dependency level (computed once on the host from the pattern).  The factorisation and the triangular
// sweeps run as dataflows over chunks of rows (nlf_sweep.inl).  With more than 32 dependencies in a row the levels
// are taken one after the other with a barrier between them: the factorisation by a 1024-thread workgroup for each
// independent block, the sweeps by one workgroup for all rows.
#include "nlf_internal.hpp"

#include <mutex>

#include <algorithm>
#include <array>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <cmath>
#include <memory>
#include <numeric>
#include <type_traits>

namespace nlf {

constexpr int SPMV_THREADS = 256;
constexpr int SPMV_PAIRS_IN_FLIGHT = 4;  // nonzero pairs each lane of the pair kernel loads per step (8: no faster)
constexpr int LEVEL_THREADS = 1024;

struct CGState {
    double rz, rz_prev, pq, alpha, beta, bnorm, res, tol;
    int done, indefinite;                // indefinite: p'Ap < 0 is not a breakdown (bordered Neumann systems)
    i64 it, max_it;
    int breakdown, pad2;
};

template<class T> __device__ __forceinline__ T shfl_down_t(T v, int o) { return __shfl_down(v, o); }

template<class Acc>
__device__ __forceinline__ Acc block_sum(Acc v, Acc* sh) {
    // fixed-order tree reduction (deterministic)
    for (int o = 32; o > 0; o >>= 1) v += shfl_down_t(v, o);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    Acc s = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < int(blockDim.x >> 6); ++i) s += sh[i];
    __syncthreads();
    return s;
}

// y = A x (rows in [0, rows)), optionally partial[b] = sum_r x_r y_r over the block's rows.  LPR
// lanes per row, grid-stride over row groups (the grid is capped, so DOT partials stay few).
// Columns are absolute (cols) or, when off16 is given, 16-bit offsets from the row (col = r + off):
// 10 instead of 12 bytes per FP64 nonzero.  Each lane keeps four (value, column) pairs and then
// four x gathers in flight.
// (a template: with a bool argument the two loads are merged into a plain one before it is known)
template<bool NT, class T>
__device__ __forceinline__ T stream_load(const T* p) {
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// Split values: hi (FP32) + lo * 2^-16 ulp(hi), lo a 16-bit integer (40 significand bits).
__device__ __forceinline__ double split_value(float h, int16_t l) {
    unsigned e = (__float_as_uint(h) >> 23) & 0xffu;
    e = e ? e : 1u;
    return double(h) + double(l) * __longlong_as_double(static_cast<long long>(e + 857u) << 52);
}

// SPLIT (V = float): each value is split_value(val[p], lo[p]), summed in Acc.  NT (a variant for
// timing, per-nonzero offsets): the matrix stream is loaded non-temporally.
template<int LPR, class V, class X, class Acc, bool DOT, bool XCD = false, int UNROLL = 4, bool NT = false,
         bool SPLIT = false>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv(i64 rows, const i64* __restrict__ outer, const i32* __restrict__ cols,
                                                       const int16_t* __restrict__ off16, const i64* __restrict__ pstart,
                                                       const V* __restrict__ val, const int16_t* __restrict__ lo,
                                                       const X* __restrict__ x, X* __restrict__ y,
                                                       double* __restrict__ partial, const CGState* __restrict__ st) {
    __shared__ double sh[SPMV_THREADS / 64];
    if (st && st->done) return;
    constexpr int RPB = SPMV_THREADS / LPR;
    const int sub = threadIdx.x % LPR;
    double d = 0.0;
    // XCD: workgroups are dealt round-robin to the 8 XCDs; renumbering them so that each XCD sweeps
    // a contiguous range of row groups keeps the x window of neighbouring rows in one L2
    i64 lb = blockIdx.x;
    if (XCD && gridDim.x % 8 == 0) lb = i64(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
    const i64 rows_r = (rows + RPB - 1) / RPB * RPB;
    for (i64 r0 = lb * RPB; r0 < rows_r; r0 += i64(gridDim.x) * RPB) {
        const i64 r = r0 + threadIdx.x / LPR;
        Acc acc = 0;
        if (r < rows) {
            const i64 b = outer[r], e = outer[r + 1];
            // offsets of row r: off16[ob + p] (ob = 0 for per-nonzero offsets; with the row-pattern
            // dictionary ob moves p into the row's shared pattern, which stays in L2)
            const i64 ob = pstart ? pstart[r] : 0;
            i64 p = b + sub;
            for (; p + (UNROLL - 1) * LPR < e; p += UNROLL * LPR) {
                i64 c[UNROLL];
                V v[UNROLL];
                int16_t vl[UNROLL];
#pragma unroll
                for (int t = 0; t < UNROLL; ++t) {
                    c[t] = off16 ? r + i64(stream_load<NT>(off16 + ob + p + t * LPR))
                                 : i64(stream_load<NT>(cols + p + t * LPR));
                    v[t] = stream_load<NT>(val + p + t * LPR);
                    if constexpr (SPLIT) vl[t] = lo[p + t * LPR];
                }
                X xv[UNROLL];
#pragma unroll
                for (int t = 0; t < UNROLL; ++t) xv[t] = x[c[t]];
#pragma unroll
                for (int t = 0; t < UNROLL; ++t) {
                    if constexpr (SPLIT) acc += Acc(split_value(v[t], vl[t])) * Acc(xv[t]);
                    else acc += Acc(v[t]) * Acc(xv[t]);
                }
            }
            for (; p < e; p += LPR) {
                const i64 c = off16 ? r + i64(stream_load<NT>(off16 + ob + p)) : i64(stream_load<NT>(cols + p));
                if constexpr (SPLIT) acc += Acc(split_value(stream_load<NT>(val + p), lo[p])) * Acc(x[c]);
                else acc += Acc(stream_load<NT>(val + p)) * Acc(x[c]);
            }
        }
        for (int o = LPR / 2; o > 0; o >>= 1) acc += shfl_down_t(acc, o);   // lane sub==0 of each group holds the sum
        if (r < rows && sub == 0) {
            y[r] = X(acc);
            if (DOT) d += double(x[r]) * double(X(acc));
        }
    }
    if (DOT) {
        d = block_sum<double>(d, sh);
        if (threadIdx.x == 0) partial[blockIdx.x] = d;
    }
}

// Pair SpMV over 16-bit offsets (per nonzero, or the row-pattern dictionary whose row starts are
// even, see nlf_rowpat.hip): each lane takes two consecutive nonzeros per load, so one 2-value load
// and one 4-byte offset load replace two of each; two pairs stay in flight per lane.  A row that
// starts at an odd index handles its first nonzero apart, and an odd last one at the end, so
// every pair load is aligned.  The products are summed in the same order by every launch of a
// given LPR (results are reproducible, not bitwise equal to k_spmv's).
template<class V> struct Pair;
template<> struct Pair<double> { typedef double T __attribute__((ext_vector_type(2))); };
template<> struct Pair<float> { typedef float T __attribute__((ext_vector_type(2))); };

// XCD: each block takes a contiguous chunk of row groups, and the blocks that the hardware deals
// round-robin to one XCD take adjacent chunks, so each XCD's L2 holds the x window of its own
// eighth of the rows (without it, concurrently active rows span the whole matrix on every XCD).
// NT: the values are loaded non-temporally (the offsets are not: a row-pattern dictionary is read again).
template<int LPR, class V, class X, class Acc, bool DOT, bool SPLIT = false, bool XCD = false, int PF = SPMV_PAIRS_IN_FLIGHT,
         bool NT = false>
__global__ __launch_bounds__(SPMV_THREADS) void k_spmv2(i64 rows, const i64* __restrict__ outer,
                                                        const int16_t* __restrict__ off, const i64* __restrict__ pstart,
                                                        const V* __restrict__ val, const int16_t* __restrict__ lo,
                                                        const X* __restrict__ x, X* __restrict__ y,
                                                        double* __restrict__ partial, const CGState* __restrict__ st) {
    typedef typename Pair<V>::T V2;
    __shared__ double sh[SPMV_THREADS / 64];
    if (st && st->done) return;
    constexpr int RPB = SPMV_THREADS / LPR;
    const int sub = threadIdx.x % LPR;
    double d = 0.0;
    auto value = [&](V v, int16_t l) -> Acc {
        if constexpr (SPLIT) return Acc(split_value(v, l));
        else return Acc(v);
    };
    auto lo_pair = [&](i64 p) -> int {
        if constexpr (SPLIT) return *reinterpret_cast<const int*>(lo + p);
        else return 0;
    };
    const i64 groups = (rows + RPB - 1) / RPB;
    i64 g_begin = blockIdx.x, g_end = groups, g_step = gridDim.x;
    if (XCD) {
        const i64 lb = i64(blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
        const i64 per = (groups + gridDim.x - 1) / gridDim.x;
        g_begin = lb * per;
        g_end = std::min<i64>(groups, g_begin + per);
        g_step = 1;
    }
    for (i64 grp = g_begin; grp < g_end; grp += g_step) {
        const i64 r = grp * RPB + threadIdx.x / LPR;
        Acc acc = 0;
        if (r < rows) {
            const i64 b = outer[r], e = outer[r + 1];
            const int16_t* o = off + (pstart ? pstart[r] : 0);
            if ((b & 1) && sub == 0 && b < e)
                acc += value(val[b], SPLIT ? lo[b] : int16_t(0)) * Acc(x[r + o[b]]);
            i64 p = ((b + 1) & ~i64(1)) + 2 * sub;
            // PF pairs in flight per lane; a lane's pairs are summed in order whatever PF is
            for (; p + 2 * LPR * (PF - 1) + 1 < e; p += 2 * LPR * PF) {
                V2 v[PF];
                int cw[PF], lw[PF];
#pragma unroll
                for (int u = 0; u < PF; ++u) {
                    v[u] = stream_load<NT>(reinterpret_cast<const V2*>(val + p + 2 * LPR * u));
                    cw[u] = *reinterpret_cast<const int*>(o + p + 2 * LPR * u);
                    lw[u] = lo_pair(p + 2 * LPR * u);
                }
                X xs[2 * PF];
#pragma unroll
                for (int u = 0; u < PF; ++u) {
                    xs[2 * u] = x[r + int16_t(cw[u] & 0xffff)];
                    xs[2 * u + 1] = x[r + int16_t(cw[u] >> 16)];
                }
#pragma unroll
                for (int u = 0; u < PF; ++u) {
                    acc += value(v[u].x, int16_t(lw[u] & 0xffff)) * Acc(xs[2 * u]);
                    acc += value(v[u].y, int16_t(lw[u] >> 16)) * Acc(xs[2 * u + 1]);
                }
            }
            for (; p + 1 < e; p += 2 * LPR) {
                const V2 v0 = stream_load<NT>(reinterpret_cast<const V2*>(val + p));
                const int c0 = *reinterpret_cast<const int*>(o + p);
                const int l0 = lo_pair(p);
                acc += value(v0.x, int16_t(l0 & 0xffff)) * Acc(x[r + int16_t(c0 & 0xffff)]);
                acc += value(v0.y, int16_t(l0 >> 16)) * Acc(x[r + int16_t(c0 >> 16)]);
            }
            if (p < e) acc += value(val[p], SPLIT ? lo[p] : int16_t(0)) * Acc(x[r + o[p]]);
        }
        for (int k = LPR / 2; k > 0; k >>= 1) acc += shfl_down_t(acc, k);
        if (r < rows && sub == 0) {
            y[r] = X(acc);
            if (DOT) d += double(x[r]) * double(X(acc));
        }
    }
    if (DOT) {
        d = block_sum<double>(d, sh);
        if (threadIdx.x == 0) partial[blockIdx.x] = d;
    }
}

__global__ void k_sum_partials(const double* __restrict__ partial, int n, double* __restrict__ out) {
    __shared__ double sh[1024 / 64];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += partial[i];
    s = block_sum<double>(s, sh);
    if (threadIdx.x == 0) *out = s;
}

// The sum of n partials in every thread (the same in every block: all add in one order).
__device__ __forceinline__ double sum_partials(const double* __restrict__ partial, int n, double* sh) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += partial[i];
    s = block_sum<double>(s, sh);
    if (threadIdx.x == 0) sh[0] = s;
    __syncthreads();
    s = sh[0];
    __syncthreads();
    return s;
}

// st->done as one thread reads it: the first block may set it while this one starts
__device__ __forceinline__ bool stopped(const CGState* st) {
    __shared__ int done;
    if (threadIdx.x == 0) done = st->done;
    __syncthreads();
    return done != 0;
}

// alpha = rz / (p . A p); x += alpha p; r -= alpha q; z = M r (identity / Jacobi, or left for a separate
// apply); partial rz.  Every block sums the partials of p . A p itself, which costs a small system less than
// a launch for it does (40 x 40 nodes: a solve of 47
// iterations 4.86 -> 4.53 ms with k_update_p's); the first one
// keeps the state, of which the others read nothing that it writes but the stop, which all find alike.
template<class X, bool JACOBI, bool DOT>
__global__ __launch_bounds__(SPMV_THREADS) void k_update_xr(i64 n, X* __restrict__ x, X* __restrict__ r, const X* __restrict__ p,
                                                            const X* __restrict__ q, X* __restrict__ z,
                                                            const X* __restrict__ invd, const double* __restrict__ ppq, int npq,
                                                            double* __restrict__ partial, CGState* st) {
    __shared__ double sh[SPMV_THREADS / 64];
    if (stopped(st)) return;
    const double pq = sum_partials(ppq, npq, sh), rz = st->rz, alpha = rz / pq;
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (first) {
        st->pq = pq;
        st->alpha = alpha;
        st->rz_prev = rz;
    }
    const bool bad_curvature = st->indefinite ? pq == 0.0 : !(pq > 0.0);
    if (bad_curvature || !isfinite(alpha)) {
        if (first) { st->breakdown = 1; st->done = 1; }
        return;
    }
    const X a = X(alpha);
    double d = 0.0;
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) {
        x[i] += a * p[i];
        const X ri = r[i] - a * q[i];
        r[i] = ri;
        if (z) {
            const X zi = JACOBI ? invd[i] * ri : ri;
            z[i] = zi;
            if (DOT) d += double(ri) * double(zi);
        }
    }
    if (DOT) {
        d = block_sum<double>(d, sh);
        if (threadIdx.x == 0) partial[blockIdx.x] = d;
    }
}

template<class X>
__global__ __launch_bounds__(SPMV_THREADS) void k_dot(i64 n, const X* __restrict__ a, const X* __restrict__ b,
                                                      double* __restrict__ partial, const CGState* __restrict__ st) {
    __shared__ double sh[SPMV_THREADS / 64];
    if (st && st->done) return;
    double d = 0.0;
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x)
        d += double(a[i]) * double(b[i]);
    d = block_sum<double>(d, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = d;
}

// mu = rz_new / rz; p = z + mu p; residual = sqrt(rz)/||b||; stop test of the reference.  The partials of
// r.z are summed as in k_update_xr; a direction left half updated by the stop is not used again.
template<class X>
__global__ __launch_bounds__(SPMV_THREADS) void k_update_p(i64 n, X* __restrict__ p, const X* __restrict__ z,
                                                           const double* __restrict__ prz, int nrz, CGState* st) {
    __shared__ double sh[SPMV_THREADS / 64];
    if (stopped(st)) return;
    const double rz = sum_partials(prz, nrz, sh), beta = rz / st->rz_prev;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->beta = beta;
        st->rz = rz;
        st->it += 1;
        st->res = sqrt(fabs(rz)) / st->bnorm;
        if (!isfinite(st->res)) { st->breakdown = 1; st->done = 1; }
        if (st->res <= st->tol || st->it >= st->max_it) st->done = 1;
    }
    const X b = X(beta);
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) p[i] = z[i] + b * p[i];
}

// CG start: rz = r.z, bnorm from partials, residual, done.
__global__ void k_init_state(const double* __restrict__ prz, const double* __restrict__ pbb, int n, double tol, i64 max_it,
                             int indefinite, CGState* __restrict__ st) {
    __shared__ double sh[1024 / 64];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) { a += prz[i]; b += pbb[i]; }
    a = block_sum<double>(a, sh);
    b = block_sum<double>(b, sh);
    if (threadIdx.x == 0) {
        st->rz = a;
        st->bnorm = sqrt(b);
        st->tol = tol;
        st->it = 0;
        st->max_it = max_it;
        st->breakdown = 0;
        st->indefinite = indefinite;
        st->res = st->bnorm > 0.0 ? sqrt(fabs(a)) / st->bnorm : 0.0;
        st->done = (st->res <= tol || max_it <= 0) ? 1 : 0;
    }
}

template<class A, class B>
__global__ void k_axpby(i64 n, A alpha, const B* __restrict__ x, A beta, B* __restrict__ y) {   // y = alpha x + beta y
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x)
        y[i] = B(alpha * A(x[i]) + beta * A(y[i]));
}

// y += x (FP32 correction accumulated into the FP64 solution)
template<class S, class Y>
__global__ void k_add_to(i64 n, const S* __restrict__ x, Y* __restrict__ y) {
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) y[i] += Y(x[i]);
}

// rz from partial sums; `first` also initialises the state of a reliable-update solve (no
// convergence test inside: the host decides on the FP64 true residual).
__global__ void k_set_rz(const double* __restrict__ partial, int n, int first, i64 max_it, int indefinite,
                         CGState* __restrict__ st) {
    __shared__ double sh[1024 / 64];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += partial[i];
    s = block_sum<double>(s, sh);
    if (threadIdx.x == 0) {
        st->rz = s;
        st->done = 0;
        if (first) {
            st->it = 0;
            st->max_it = max_it;
            st->tol = -1.0;
            st->bnorm = 1.0;
            st->breakdown = 0;
            st->indefinite = indefinite;
        }
        st->res = sqrt(fabs(s));
    }
}

template<class A, class B>
__global__ void k_convert(i64 n, const A* __restrict__ x, B* __restrict__ y) {
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) y[i] = B(x[i]);
}

template<class X>
__global__ void k_scale(i64 n, const X* __restrict__ s, const X* __restrict__ x, X* __restrict__ y) {
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) y[i] = s[i] * x[i];
}

// r = b - A x (full storage, one wave per row) and partial sums of r.r and b.b.
template<class V, class X>
__global__ __launch_bounds__(SPMV_THREADS) void k_residual(i64 rows, const i64* __restrict__ outer, const i32* __restrict__ cols,
                                                           const V* __restrict__ val, const X* __restrict__ x,
                                                           const X* __restrict__ b, X* __restrict__ r,
                                                           double* __restrict__ prr, double* __restrict__ pbb) {
    __shared__ double sh[SPMV_THREADS / 64];
    const int lane = threadIdx.x & 63;
    constexpr int RPB = SPMV_THREADS / 64;
    double rr = 0.0, bb = 0.0;
    const i64 rows_r = (rows + RPB - 1) / RPB * RPB;
    for (i64 r0 = i64(blockIdx.x) * RPB; r0 < rows_r; r0 += i64(gridDim.x) * RPB) {     // one wave per row
        const i64 row = r0 + (threadIdx.x >> 6);
        double acc = 0.0;
        if (row < rows)
            for (i64 p = outer[row] + lane; p < outer[row + 1]; p += 64) acc += double(val[p]) * double(x[cols[p]]);
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o);
        if (row < rows && lane == 0) {
            const double ri = double(b[row]) - acc;
            r[row] = X(ri);
            rr += ri * ri;
            bb += double(b[row]) * double(b[row]);
        }
    }
    rr = block_sum<double>(rr, sh);
    bb = block_sum<double>(bb, sh);
    if (threadIdx.x == 0) { prr[blockIdx.x] = rr; pbb[blockIdx.x] = bb; }
}

// f -= K_bound x_D ; f[D] = x_D   (boundary_condition_first_kind_2d.hpp:50-59)
__global__ void k_first_kind(i64 rows, const i64* __restrict__ bo, const i32* __restrict__ bc, const double* __restrict__ bv,
                             const uint8_t* __restrict__ inner, const double* __restrict__ xD, double* __restrict__ f) {
    const i64 r = i64(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    double s = 0.0;
    for (i64 p = bo[r]; p < bo[r + 1]; ++p) s += bv[p] * xD[bc[p]];
    f[r] = inner[r] ? f[r] - s : xD[r];
}

__global__ void k_inv_diag(i64 rows, const i64* __restrict__ diag, const double* __restrict__ val, double* __restrict__ inv) {
    const i64 r = i64(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const double d = val[diag[r]];
    inv[r] = d != 0.0 ? 1.0 / d : 1.0;              // Eigen::DiagonalPreconditioner: 1 for zero diagonals
}

// ---- IC(0) ------------------------------------------------------------------------------------
// One independent diagonal block of a block-diagonal factor, factored by a workgroup of its own: its
// level count and first level offset (into the shared offsets).
struct SweepBlock {
    i32 levels, lptr_off;
};

struct LevelArgs {
    i64 rows;
    int levels;
    const i64* outer;
    const i32* cols;
    const i64* diag;
    const i64* tpos;       // position of the transposed entry
    const i32* lrows;      // rows sorted by level
    const i32* lptr;       // level offsets
};

__global__ void k_ic_init(i64 rows, const i64* __restrict__ outer, const i32* __restrict__ cols, const i64* __restrict__ diag,
                          const double* __restrict__ a, const double* __restrict__ s, double shift, double* __restrict__ F) {
    const i64 r = i64(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    for (i64 p = outer[r]; p < outer[r + 1]; ++p) F[p] = s[r] * a[p] * s[cols[p]];
    F[diag[r]] += shift;
}

__global__ void k_scale_from_diag(i64 rows, const i64* __restrict__ diag, const double* __restrict__ a, double* __restrict__ s) {
    const i64 r = i64(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const double d = fabs(a[diag[r]]);
    s[r] = d > 0.0 ? 1.0 / sqrt(d) : 1.0;
}

// Up-looking IC(0): for row k (all rows i < k it depends on are done and mirrored into row k's
// lower positions), U_kk = sqrt(a_kk - sum_i U_ik^2), U_kj = (a_kj - sum_{i<k} U_ik U_ij) / U_kk.
// blk: one workgroup per independent diagonal block, over the block's own levels (a.lrows block
// after block, a.lptr each block's level offsets from blk[b].lptr_off on).
__global__ __launch_bounds__(LEVEL_THREADS) void k_ic_factor(LevelArgs a, const SweepBlock* __restrict__ blk,
                                                             double* __restrict__ F, int* __restrict__ fail) {
    if (blk) {
        const SweepBlock b = blk[blockIdx.x];
        a.levels = b.levels;
        a.lptr += b.lptr_off;
    }
    for (int L = 0; L < a.levels; ++L) {
        for (i32 t = a.lptr[L] + threadIdx.x; t < a.lptr[L + 1]; t += blockDim.x) {
            const i64 k = a.lrows[t];
            const i64 b = a.outer[k], dk = a.diag[k], e = a.outer[k + 1];
            double d = F[dk];
            for (i64 p = b; p < dk; ++p) d -= F[p] * F[p];
            if (!(d > 0.0) || !isfinite(d)) { *fail = 1; d = 1.0; }
            const double ukk = sqrt(d);
            F[dk] = ukk;
            for (i64 p = dk + 1; p < e; ++p) {
                const i32 j = a.cols[p];
                double v = F[p];
                // intersection of lower(k) and lower(j) restricted to i < k
                i64 pj = a.outer[j];
                const i64 ej = a.diag[j];
                for (i64 pk = b; pk < dk; ++pk) {
                    const i32 i = a.cols[pk];
                    while (pj < ej && a.cols[pj] < i) ++pj;
                    if (pj < ej && a.cols[pj] == i) v -= F[pk] * F[pj];
                }
                v /= ukk;
                F[p] = v;
                F[a.tpos[p]] = v;
            }
        }
        __syncthreads();
    }
}

// One triangular sweep in level order, for rows with more dependencies than the chunked sweeps take.  Records (one per row) are stored contiguously in level
// order so a level's loads are coalesced; a dependency on a row solved at most K levels earlier is
// read from an LDS window of K x W slots (slot = (level mod K) * W + position in level), otherwise
// (dep < 0) from global memory.
struct PackedSweep {
    int levels, K, W;
    const i32* lptr;      // [levels+1] record offsets
    const i32* row;       // row of each record
    const i32* off;       // [records+1] entry offsets
    const i32* dep;       // window slot, or -(row+1)
    const double* val;         // factor entries
    const double* dinv;        // 1 / U_kk
    const double* scale;       // s_k
};

// z = S U^-1 U^-T S r : forward U^T y = S r, backward U z' = y, z = S z'.  One workgroup.
__global__ __launch_bounds__(LEVEL_THREADS) void k_ic_solve(PackedSweep fw, PackedSweep bw, const double* __restrict__ r,
                                                            double* __restrict__ y, double* __restrict__ z,
                                                            const CGState* __restrict__ st) {
    extern __shared__ unsigned char smem_raw[];
    double* win = reinterpret_cast<double*>(smem_raw);
    if (st && st->done) return;
    for (int L = 0; L < fw.levels; ++L) {
        const i32 b = fw.lptr[L], cnt = fw.lptr[L + 1] - b;
        for (i32 t = threadIdx.x; t < cnt; t += blockDim.x) {
            const i32 rec = b + t;
            const i32 k = fw.row[rec];
            double v = fw.scale[rec] * r[k];
            for (i32 e = fw.off[rec]; e < fw.off[rec + 1]; ++e) {
                const i32 d = fw.dep[e];
                v -= fw.val[e] * (d >= 0 ? win[d] : y[-d - 1]);
            }
            v *= fw.dinv[rec];
            if (fw.K) win[(L % fw.K) * fw.W + t] = v;
            y[k] = v;
        }
        __syncthreads();
    }
    for (int L = 0; L < bw.levels; ++L) {
        const i32 b = bw.lptr[L], cnt = bw.lptr[L + 1] - b;
        for (i32 t = threadIdx.x; t < cnt; t += blockDim.x) {
            const i32 rec = b + t;
            const i32 k = bw.row[rec];
            double v = y[k];
            for (i32 e = bw.off[rec]; e < bw.off[rec + 1]; ++e) {
                const i32 d = bw.dep[e];
                v -= bw.val[e] * (d >= 0 ? win[d] : y[-d - 1]);
            }
            v *= bw.dinv[rec];
            if (bw.K) win[(L % bw.K) * bw.W + t] = v;
            y[k] = v;                  // z' (row k of the backward sweep reads only its own y[k])
            z[k] = bw.scale[rec] * v;
        }
        __syncthreads();
    }
}

// Gathers the factor into the packed sweep layout (values by source position, per-record 1/U_kk, s_k).
__global__ void k_pack_entries(i64 n, const i64* __restrict__ src, const double* __restrict__ F, double* __restrict__ v) {
    for (i64 e = i64(blockIdx.x) * blockDim.x + threadIdx.x; e < n; e += i64(gridDim.x) * blockDim.x) v[e] = F[src[e]];
}

__global__ void k_pack_rows(i64 n, const i32* __restrict__ row, const i64* __restrict__ diag, const double* __restrict__ F,
                            const double* __restrict__ s, double* __restrict__ dinv, double* __restrict__ scale) {
    for (i64 t = i64(blockIdx.x) * blockDim.x + threadIdx.x; t < n; t += i64(gridDim.x) * blockDim.x) {
        const i32 k = row[t];
        dinv[t] = 1.0 / F[diag[k]];
        scale[t] = s[k];
    }
}

__global__ void k_transpose_pos(i64 rows, const i64* __restrict__ outer, const i32* __restrict__ cols, i64* __restrict__ tpos) {
    const i64 r = i64(blockIdx.x) * (blockDim.x / 64) + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    for (i64 p = outer[r] + lane; p < outer[r + 1]; p += 64) {
        const i32 c = cols[p];
        i64 lo = outer[c], hi = outer[c + 1];
        while (lo < hi) {
            const i64 mid = (lo + hi) >> 1;
            if (cols[mid] < r) lo = mid + 1; else hi = mid;
        }
        tpos[p] = (lo < outer[c + 1] && cols[lo] == r) ? lo : p;   // symmetric pattern: always found
    }
}

template<class X>
__global__ void k_zero(i64 n, X* __restrict__ x) {
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) x[i] = X(0);
}

unsigned grid_stride_blocks(i64 n) { return unsigned(std::min<i64>(std::max<i64>((n + 255) / 256, 1), 4096)); }

}  // namespace nlf

#include "nlf_sweep.inl"

// ---- preconditioner object ---------------------------------------------------------------------
struct nlf_precond_s {
    nlf_ctx ctx = nullptr;
    int kind = NLF_PRECOND_IDENTITY;
    nlf::i64 rows = 0;
    bool ok = true;
    double shift = 0.0;
    double setup_seconds = 0.0;
    // Jacobi
    nlf::DevBuf<double> invd;
    // ILLT
    int fw_levels = 0, bw_levels = 0;
    int blocks = 1;                      // independent diagonal blocks
    nlf::DevBuf<double> F, scale;
    // the chunked sweeps with their value buffers (by record) and tickets
    bool chunked = false;
    nlf::Sweep sw_fw, sw_bw;
    nlf::DevBuf<double> fw_lvl, bw_lvl;
    nlf::DevBuf<nlf::i32> ticket;
    // the packed sweeps (one workgroup)
    struct Packed {
        int levels = 0, K = 0, W = 0;
        nlf::DevBuf<nlf::i32> lptr, row, off, dep;
        nlf::DevBuf<double> val, dinv, scale;
        nlf::PackedSweep args() const { return {levels, K, W, lptr.p, row.p, off.p, dep.p, val.p, dinv.p, scale.p}; }
    } fw, bw;
    int solve_threads = 64;
    nlf::DevBuf<double> work;
    // learned (set by nlf_learned.hip)
    void* learned = nullptr;
    void (*learned_destroy)(void*) = nullptr;
    ~nlf_precond_s() {
        if (learned && learned_destroy) learned_destroy(learned);
    }
};

namespace nlf {

// Level sets of the lower (forward) and upper (backward) dependency DAGs of a symmetric pattern.
static void level_sets(const std::vector<i64>& outer, const std::vector<i32>& cols, const std::vector<i64>& diag,
                       std::vector<i32>& fr, std::vector<i32>& fp, std::vector<i32>& br, std::vector<i32>& bp) {
    const i64 n = i64(diag.size());
    std::vector<i32> lev(n, 0);
    int nl = 0;
    for (i64 k = 0; k < n; ++k) {
        int l = 0;
        for (i64 p = outer[k]; p < diag[k]; ++p) l = std::max(l, lev[cols[p]] + 1);
        lev[k] = l;
        nl = std::max(nl, l + 1);
    }
    auto bucket = [&](int levels, std::vector<i32>& rowsv, std::vector<i32>& ptr, bool ascending) {
        ptr.assign(levels + 1, 0);
        for (i64 k = 0; k < n; ++k) ptr[lev[k] + 1]++;
        for (int l = 0; l < levels; ++l) ptr[l + 1] += ptr[l];
        rowsv.assign(n, 0);
        std::vector<i32> fill(ptr.begin(), ptr.end() - 1);
        if (ascending) for (i64 k = 0; k < n; ++k) rowsv[fill[lev[k]]++] = i32(k);
        else for (i64 k = n - 1; k >= 0; --k) rowsv[fill[lev[k]]++] = i32(k);
    };
    bucket(nl, fr, fp, true);
    std::fill(lev.begin(), lev.end(), 0);
    nl = 0;
    for (i64 k = n - 1; k >= 0; --k) {
        int l = 0;
        for (i64 p = diag[k] + 1; p < outer[k + 1]; ++p) l = std::max(l, lev[cols[p]] + 1);
        lev[k] = l;
        nl = std::max(nl, l + 1);
    }
    bucket(nl, br, bp, false);
}

constexpr size_t IC_WINDOW_BYTES = 64 * 1024;

// Builds one packed sweep: records in level order, entries (lower part for the forward sweep,
// strict upper part for the backward one) with their dependency slots; values are gathered on the
// device from the factor by source position.
static void build_sweep(const std::vector<i64>& outer, const std::vector<i32>& cols, const std::vector<i64>& diag,
                        const std::vector<i32>& lrows, const std::vector<i32>& lptr, bool forward, const double* F,
                        const double* scale, const i64* d_diag, nlf_precond_s::Packed& sw, hipStream_t s) {
    const i64 n = i64(diag.size());
    const int levels = int(lptr.size()) - 1;
    std::vector<i32> level_of(n), pos_of(n);
    int W = 1;
    for (int L = 0; L < levels; ++L) {
        W = std::max(W, lptr[L + 1] - lptr[L]);
        for (i32 t = lptr[L]; t < lptr[L + 1]; ++t) { level_of[lrows[t]] = L; pos_of[lrows[t]] = t - lptr[L]; }
    }
    int K = 1;
    std::vector<i32> off(n + 1, 0);
    for (i64 t = 0; t < n; ++t) {
        const i32 k = lrows[t];
        const i64 b = forward ? outer[k] : diag[k] + 1, e = forward ? diag[k] : outer[k + 1];
        off[t + 1] = off[t] + i32(e - b);
        for (i64 p = b; p < e; ++p) K = std::max(K, level_of[k] - level_of[cols[p]]);
    }
    // K + 1 slot blocks: the level being written must not share its block with a dependency K
    // levels back that other threads of the same level are still reading
    K += 1;
    const bool window = size_t(K) * size_t(W) * sizeof(double) <= IC_WINDOW_BYTES;
    std::vector<i32> dep(off[n]);
    std::vector<i64> src(off[n]);
    for (i64 t = 0; t < n; ++t) {
        const i32 k = lrows[t];
        const i64 b = forward ? outer[k] : diag[k] + 1, e = forward ? diag[k] : outer[k + 1];
        i32 q = off[t];
        for (i64 p = b; p < e; ++p, ++q) {
            const i32 i = cols[p];
            dep[q] = window ? (level_of[i] % K) * W + pos_of[i] : -(i + 1);
            src[q] = p;
        }
    }
    sw.levels = levels;
    sw.K = window ? K : 0;
    sw.W = W;
    upload(sw.lptr, lptr.data(), lptr.size(), s);
    upload(sw.row, lrows.data(), lrows.size(), s);
    upload(sw.off, off.data(), off.size(), s);
    upload(sw.dep, dep.data(), std::max<size_t>(dep.size(), 1), s);
    DevBuf<i64> d_src;
    upload(d_src, src.data(), std::max<size_t>(src.size(), 1), s);
    const size_t ne = std::max<size_t>(src.size(), 1);
    sw.val.alloc(ne);
    sw.dinv.alloc(size_t(n)); sw.scale.alloc(size_t(n));
    if (!src.empty())
        hipLaunchKernelGGL(k_pack_entries, dim3(grid_stride_blocks(i64(src.size()))), dim3(256), 0, s, i64(src.size()),
                           d_src.p, F, sw.val.p);
    hipLaunchKernelGGL(k_pack_rows, dim3(grid_stride_blocks(n)), dim3(256), 0, s, n, sw.row.p, d_diag, F, scale,
                       sw.dinv.p, sw.scale.p);
    NLF_HIP(hipGetLastError());
    NLF_HIP(hipStreamSynchronize(s));
}

// Contiguous row ranges with no entry between them: the diagonal blocks of a block-diagonal pattern
// (a batch of independent instances), merged so that each holds at least min_rows rows; {0, n}
// for one block.  The pattern is symmetric, so no row after a boundary reaches back across it
// once no row before it reaches past it.
static std::vector<i64> independent_blocks(const std::vector<i64>& outer, const std::vector<i32>& cols, i64 min_rows) {
    const i64 n = i64(outer.size()) - 1;
    std::vector<i64> b(1, 0);
    i64 reach = -1;                 // the largest column of the rows so far
    for (i64 r = 0; r + 1 < n; ++r) {
        if (outer[r + 1] > outer[r]) reach = std::max<i64>(reach, cols[outer[r + 1] - 1]);
        if (reach <= r && r + 1 - b.back() >= min_rows) b.push_back(r + 1);
    }
    if (n - b.back() < min_rows && b.size() > 1) b.pop_back();    // a short tail joins the last block
    b.push_back(n);
    return b;
}

// The global levels restricted to each block, in order: rows block after block (level order within
// a block), the blocks' level offsets one after another (global record offsets; empty levels
// dropped, a row's dependencies stay at lower levels), seg[b] the index of block b's first offset.
struct BlockLevels {
    std::vector<i32> rows, ptr, blk;
    std::vector<i64> seg;
    std::vector<i32> levels;
};
static BlockLevels block_levels(const std::vector<i32>& lrows, const std::vector<i32>& level_ptr,
                                const std::vector<i64>& bounds) {
    const i64 n = bounds.back();
    const int B = int(bounds.size()) - 1;
    BlockLevels bl;
    bl.blk.resize(size_t(n));
    for (int b = 0; b < B; ++b)
        for (i64 r = bounds[b]; r < bounds[b + 1]; ++r) bl.blk[size_t(r)] = b;
    bl.rows.resize(size_t(n));
    std::vector<i64> pos(bounds.begin(), bounds.end() - 1);
    std::vector<std::vector<i32>> bptr(static_cast<size_t>(B));
    for (int b = 0; b < B; ++b) bptr[size_t(b)].push_back(i32(bounds[b]));
    std::vector<int> touched;
    std::vector<char> is_touched(static_cast<size_t>(B), 0);
    for (size_t L = 0; L + 1 < level_ptr.size(); ++L) {
        for (i32 t = level_ptr[L]; t < level_ptr[L + 1]; ++t) {
            const int b = bl.blk[size_t(lrows[t])];
            bl.rows[size_t(pos[size_t(b)]++)] = lrows[t];
            if (!is_touched[size_t(b)]) { is_touched[size_t(b)] = 1; touched.push_back(b); }
        }
        for (int b : touched) { bptr[size_t(b)].push_back(i32(pos[size_t(b)])); is_touched[size_t(b)] = 0; }
        touched.clear();
    }
    bl.seg.resize(size_t(B) + 1);
    bl.levels.resize(size_t(B));
    for (int b = 0; b < B; ++b) {
        bl.seg[size_t(b)] = i64(bl.ptr.size());
        bl.levels[size_t(b)] = i32(bptr[size_t(b)].size()) - 1;
        bl.ptr.insert(bl.ptr.end(), bptr[size_t(b)].begin(), bptr[size_t(b)].end());
    }
    bl.seg[size_t(B)] = i64(bl.ptr.size());
    return bl;
}

// Applies the preconditioner z = M^-1 r on the stream.  With `partial`, an ILLT also writes the partial
// sums of r.z in k_dot's blocks (`blocks` of them); returns whether it did.
bool precond_apply(const nlf_precond_s* P, i64 n, const double* r, double* z, const CGState* st, hipStream_t s,
                   double* partial = nullptr, unsigned blocks = 0) {
    if (P && P->kind == NLF_PRECOND_JACOBI)
        hipLaunchKernelGGL(k_scale<double>, dim3(grid_stride_blocks(n)), dim3(256), 0, s, n, P->invd.p, r, z);
    else if (P && P->kind == NLF_PRECOND_ILLT && P->chunked) {
        launch_sweep(P->sw_fw, r, P->fw_lvl.p, P->ticket.p, st, s);
        launch_sweep(P->sw_bw, P->fw_lvl.p, P->bw_lvl.p, P->ticket.p + 1, st, s);
        hipLaunchKernelGGL(k_sweep_finish, dim3(partial ? blocks : grid_stride_blocks(n)), dim3(SPMV_THREADS), 0, s, n,
                           P->sw_bw.pos.p, P->scale.p, P->fw_lvl.p, P->bw_lvl.p, P->ticket.p, r, z, partial, st);
        return partial != nullptr;
    } else if (P && P->kind == NLF_PRECOND_ILLT) {
        const size_t lds = size_t(std::max(P->fw.K * P->fw.W, P->bw.K * P->bw.W)) * sizeof(double);
        hipLaunchKernelGGL(k_ic_solve, dim3(1), dim3(P->solve_threads), lds, s, P->fw.args(), P->bw.args(), r, P->work.p, z, st);
    } else
        NLF_HIP(hipMemcpyAsync(z, r, size_t(n) * sizeof(double), hipMemcpyDeviceToDevice, s));
    return false;
}

// Lanes per row: the smallest power of two (4..64) giving each lane at most 16 nonzeros for the
// one-nonzero-per-load kernel, 64 for the pair kernel (16-bit offsets).  Measured on the 1000 x 1000
// composite (500 nonzeros per row, FP64): one-per-load 32 lanes 1.19 ms, 64 lanes 1.29 ms, 16 lanes
// 1.31 ms; pair kernel with the row-pattern dictionary 8 lanes 0.905 ms, 16 lanes 0.93 ms, 32 lanes
// 1.00 ms, 64 lanes 1.12 ms.
int pick_lpr(double avg, bool pairs = false) {
    const double per_lane = pairs ? 64.0 : 16.0;
    int l = 4;
    while (l < 64 && double(l) * per_lane < avg) l *= 2;
    return l;
}

int pick_lpr(const nlf_matrix_s* a) {
    ensure_spmv_storage(a);
    return pick_lpr(double(a->nnz_full) / double(std::max<i64>(a->rows, 1)), a->off16.p != nullptr);
}

// SpMV grid: one row group per block iteration, capped so that DOT partials stay <= SPMV_MAX_BLOCKS
constexpr i64 SPMV_MAX_BLOCKS = 4096;
unsigned spmv_blocks(int lpr, i64 rows) {
    return unsigned(std::min<i64>(std::max<i64>((rows + (SPMV_THREADS / lpr) - 1) / (SPMV_THREADS / lpr), 1), SPMV_MAX_BLOCKS));
}

// cs: column source (spmv_cols of the matrix, or plain offsets / columns with cs.pstart = null).
// lo: 16-bit remainders of split values (V = float, NLF_MODE_SPLIT), else null.  With 16-bit
// offsets (per nonzero or the dictionary) the pair kernel k_spmv2 runs unless pairs = false; xcd
// selects its XCD-contiguous row chunks (the one-nonzero-per-load kernel's XCD numbering when
// pairs = false).  nt: the pair kernel's values (not split ones) bypass the caches.
template<class V, class X, class Acc, bool DOT>
void launch_spmv(int lpr, i64 rows, const i64* outer, SpmvCols cs, const V* val, const X* x, X* y,
                 double* partial, const CGState* st, hipStream_t s, bool xcd = false, const int16_t* lo = nullptr,
                 bool pairs = true, int pf = SPMV_PAIRS_IN_FLIGHT, bool nt = false) {
    const i32* cols = cs.cols;
    const int16_t* off16 = cs.off;
    const i64* pstart = cs.pstart;
    const unsigned blocks = spmv_blocks(lpr, rows);
    if (off16 && pairs && xcd && blocks % 8 == 0 && !lo) {
#define NLF_SPMV2_XCASE(L)                                                                                         \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_spmv2<L, V, X, Acc, DOT, false, true>), dim3(blocks), dim3(SPMV_THREADS), 0, s, rows, outer, \
                           off16, pstart, val, static_cast<const int16_t*>(nullptr), x, y, partial, st);          \
        return;
        switch (lpr) {
            NLF_SPMV2_XCASE(4)
            NLF_SPMV2_XCASE(8)
            NLF_SPMV2_XCASE(16)
            NLF_SPMV2_XCASE(32)
            default: NLF_SPMV2_XCASE(64)
        }
#undef NLF_SPMV2_XCASE
    }
    if (off16 && pairs && !xcd) {
        if (lo) {
            if constexpr (sizeof(V) == sizeof(float)) {
#define NLF_SPMV2_SCASE(L)                                                                                         \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_spmv2<L, V, X, Acc, DOT, true>), dim3(blocks), dim3(SPMV_THREADS), 0, s, rows, outer, off16, \
                           pstart, val, lo, x, y, partial, st);                                                    \
        return;
                switch (lpr) {
                    NLF_SPMV2_SCASE(4)
                    NLF_SPMV2_SCASE(8)
                    NLF_SPMV2_SCASE(16)
                    NLF_SPMV2_SCASE(32)
                    default: NLF_SPMV2_SCASE(64)
                }
#undef NLF_SPMV2_SCASE
            }
        } else {
#define NLF_SPMV2_CASE(L)                                                                                          \
    case L:                                                                                                        \
        if (pf == 2)                                                                                               \
            hipLaunchKernelGGL((k_spmv2<L, V, X, Acc, DOT, false, false, 2>), dim3(blocks), dim3(SPMV_THREADS), 0, s, rows, \
                               outer, off16, pstart, val, static_cast<const int16_t*>(nullptr), x, y, partial, st);   \
        else if (nt)                                                                                               \
            hipLaunchKernelGGL((k_spmv2<L, V, X, Acc, DOT, false, false, SPMV_PAIRS_IN_FLIGHT, true>), dim3(blocks),  \
                               dim3(SPMV_THREADS), 0, s, rows, outer, off16, pstart, val,                           \
                               static_cast<const int16_t*>(nullptr), x, y, partial, st);                           \
        else                                                                                                       \
            hipLaunchKernelGGL((k_spmv2<L, V, X, Acc, DOT, false, false, SPMV_PAIRS_IN_FLIGHT>), dim3(blocks),        \
                               dim3(SPMV_THREADS), 0, s, rows, outer, off16, pstart, val,                           \
                               static_cast<const int16_t*>(nullptr), x, y, partial, st);                           \
        return;
            switch (lpr) {
                NLF_SPMV2_CASE(4)
                NLF_SPMV2_CASE(8)
                NLF_SPMV2_CASE(16)
                NLF_SPMV2_CASE(32)
                default: NLF_SPMV2_CASE(64)
            }
#undef NLF_SPMV2_CASE
        }
    }
    if constexpr (sizeof(V) == sizeof(float)) {
        if (lo) {
#define NLF_SPMV_SCASE(L)                                                                                          \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_spmv<L, V, X, Acc, DOT, false, 4, false, true>), dim3(blocks), dim3(SPMV_THREADS), 0, s,  \
                           rows, outer, cols, off16, pstart, val, lo, x, y, partial, st);                          \
        return;
            switch (lpr) {
                NLF_SPMV_SCASE(4)
                NLF_SPMV_SCASE(8)
                NLF_SPMV_SCASE(16)
                NLF_SPMV_SCASE(32)
                default: NLF_SPMV_SCASE(64)
            }
#undef NLF_SPMV_SCASE
        }
    }
    if (xcd) {
#define NLF_SPMV_XCASE(L)                                                                                          \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_spmv<L, V, X, Acc, DOT, true>), dim3(blocks), dim3(SPMV_THREADS), 0, s, rows, outer, cols, \
                           off16, pstart, val, static_cast<const int16_t*>(nullptr), x, y, partial, st);          \
        return;
        switch (lpr) {
            NLF_SPMV_XCASE(4)
            NLF_SPMV_XCASE(8)
            NLF_SPMV_XCASE(16)
            NLF_SPMV_XCASE(32)
            default: NLF_SPMV_XCASE(64)
        }
#undef NLF_SPMV_XCASE
    }
#define NLF_SPMV_CASE(L)                                                                                           \
    case L:                                                                                                        \
        hipLaunchKernelGGL((k_spmv<L, V, X, Acc, DOT>), dim3(blocks), dim3(SPMV_THREADS), 0, s, rows, outer, cols, off16, \
                           pstart, val, static_cast<const int16_t*>(nullptr), x, y, partial, st);                 \
        break;
    switch (lpr) {
        NLF_SPMV_CASE(4)
        NLF_SPMV_CASE(8)
        NLF_SPMV_CASE(16)
        NLF_SPMV_CASE(32)
        default: NLF_SPMV_CASE(64)
    }
#undef NLF_SPMV_CASE
}


// Pairs of HIP events around sampled kernel launches on the solver's stream (slot 0: SpMV, 1: preconditioner).
struct KernelTimer {
    std::vector<hipEvent_t> ev[2][2];
    double total_ms[2] = {0.0, 0.0};
    i64 count[2] = {0, 0};
    ~KernelTimer() {
        for (auto& a : ev)
            for (auto& b : a)
                for (hipEvent_t e : b) (void)hipEventDestroy(e);
    }
    void start(int slot, hipStream_t s) { record(slot, 0, s); }
    void stop(int slot, hipStream_t s) { record(slot, 1, s); }
    void record(int slot, int which, hipStream_t s) {
        hipEvent_t e;
        NLF_HIP(hipEventCreate(&e));
        NLF_HIP(hipEventRecord(e, s));
        ev[slot][which].push_back(e);
    }
    void collect() {
        for (int k = 0; k < 2; ++k)
            for (size_t i = 0; i < ev[k][1].size(); ++i) {
                float ms = 0.f;
                NLF_HIP(hipEventSynchronize(ev[k][1][i]));
                NLF_HIP(hipEventElapsedTime(&ms, ev[k][0][i], ev[k][1][i]));
                total_ms[k] += ms;
                count[k] += 1;
            }
        for (auto& a : ev)
            for (auto& b : a) {
                for (hipEvent_t e : b) (void)hipEventDestroy(e);
                b.clear();
            }
    }
    double avg(int k) const { return count[k] ? total_ms[k] / double(count[k]) : 0.0; }
};

// r = b - r (r holds A x on entry); per-block partials of r.r and b.b.
__global__ __launch_bounds__(SPMV_THREADS) void k_resid_finish(i64 n, const double* __restrict__ b, double* __restrict__ r,
                                                               double* __restrict__ prr, double* __restrict__ pbb) {
    __shared__ double sh[SPMV_THREADS / 64];
    double rr = 0.0, bb = 0.0;
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) {
        const double bi = b[i], ri = bi - r[i];
        r[i] = ri;
        rr += ri * ri;
        bb += bi * bi;
    }
    rr = block_sum<double>(rr, sh);
    __syncthreads();
    bb = block_sum<double>(bb, sh);
    if (threadIdx.x == 0) { prr[blockIdx.x] = rr; pbb[blockIdx.x] = bb; }
}

// FP64 true residual r = b - A x through the SpMV kernels, with nb partials of r.r and b.b
// (nb <= SPMV_MAX_BLOCKS; k_sum_partials reduces them).
void residual64(i64 n, const i64* outer, SpmvCols cs, const double* val, int lpr, const double* x, const double* b,
                double* r, double* prr, double* pbb, unsigned nb, hipStream_t s) {
    launch_spmv<double, double, double, false>(lpr, n, outer, cs, val, x, r, nullptr, nullptr, s);
    hipLaunchKernelGGL(k_resid_finish, dim3(nb), dim3(SPMV_THREADS), 0, s, n, b, r, prr, pbb);
}


// Work memory of one CG solve: the vectors r, z, p (n entries of X each, 256-byte aligned), five
// arrays of per-block partial sums (SPMV_MAX_BLOCKS doubles each: every launch of the solve writes at
// most that many), two reduced sums and the solver state.
struct CGWork {
    static size_t align(size_t b) { return (b + 255) & ~size_t(255); }
    template<class X>
    static size_t bytes(i64 n) {
        return 3 * align(size_t(n) * sizeof(X)) + 5 * align(SPMV_MAX_BLOCKS * sizeof(double)) + align(2 * sizeof(double)) +
               align(sizeof(CGState));
    }
};

}  // namespace nlf

#include "nlf_symv.inl"

nlf_matrix_s::~nlf_matrix_s() { delete symv; }

namespace nlf {
// residual64 from the matrix: the product from the symmetric storage when it is built (symv_prepare),
// else from the full storage.
void residual64(const nlf_matrix_s* a, const double* x, const double* b, double* r, double* prr, double* pbb, unsigned nb,
                hipStream_t s) {
    if (a->symv && a->symv->version == a->val_version && a->ctx->spmv_symmetric) {
        launch_symv<false>(a, x, r, nullptr, nullptr, s, SPMV_MAX_BLOCKS);
        hipLaunchKernelGGL(k_resid_finish, dim3(nb), dim3(SPMV_THREADS), 0, s, a->rows, b, r, prr, pbb);
    } else {
        residual64(a->rows, a->outer.p, spmv_cols(a), a->val.p, pick_lpr(a), x, b, r, prr, pbb, nb, s);
    }
}


// Blocks of CG's vector kernels and of the symmetric product's reduction: every block of the next kernel sums
// their partials.
constexpr unsigned CG_BLOCKS = 1024;
constexpr i64 SYMV_REDUCE_BLOCKS = 2048;

// Above this size the full storage's values bypass the caches in a solve with sweeps: the last-level cache
// holds 256 MB, a smaller matrix is read from it again, a larger one only drives out the factor that the
// sweeps read next, whose loads' latency bounds them.  Q8 sheets, us per iteration without / with: 31 000
// rows (112 MB) 259 / 271, 44 000 (204 MB) 352 / 363, 59 000 (352 MB) 550 / 447, 121 000 (1264 MB) 978 / 809; with
// FP32 values 77 000 (302 MB) 647 / 539, 98 000 (451 MB) 780 / 640, 121 000 (663 MB) 926 / 766.  Split values are not
// read so.
constexpr i64 SPMV_NT_BYTES = i64(256) << 20;

// Preconditioned CG on device vectors (conjugate_gradient::solve).  Vectors of type X, matrix values V.
// The work memory (CGWork) is allocated by the object, or given by the caller (no allocation then;
// `timed` = false also records no HIP events).
template<class V, class X>
struct CG {
    hipStream_t s;
    i64 n;
    int lpr;
    const i64* outer;
    const i32* cols;
    SpmvCols cs{};                      // column source of the SpMV (spmv_cols of the matrix)
    const V* val;
    const int16_t* lo = nullptr;        // split values: 16-bit remainders (NLF_MODE_SPLIT)
    const nlf_precond_s* P;
    DevBuf<unsigned char> own;
    DevBuf<double> r64;                 // solve_reliable: the FP64 residual and the increment of the solution
    DevBuf<X> xh;
    X *r = nullptr, *z = nullptr, *p = nullptr;
    double *part1 = nullptr, *part2 = nullptr, *pbb = nullptr, *prz = nullptr, *pb2 = nullptr, *sums = nullptr;
    CGState* st = nullptr;
    unsigned sblocks, vblocks;
    bool timed = true;
    bool indefinite = false;            // a bordered (Neumann) system: negative curvature allowed
    const nlf_matrix_s* sym = nullptr;  // products from the symmetric storage (symv_prepare done)
    bool nt = false;                    // the matrix values bypass the caches (see SPMV_NT_BYTES)
    KernelTimer timer;

    CG(hipStream_t s_, i64 n_, i64 nnz, const i64* o, const i32* c, const V* v, const nlf_precond_s* P_,
       void* work = nullptr)
        : s(s_), n(n_), outer(o), cols(c), val(v), P(P_) {
        cs.cols = c;
        nt = P && P->chunked && nnz * i64(sizeof(V)) > SPMV_NT_BYTES;
        lpr = pick_lpr(double(nnz) / double(std::max<i64>(n, 1)));
        if (!work) {
            own.alloc(CGWork::bytes<X>(n));
            work = own.p;
        } else {
            timed = false;
        }
        unsigned char* w = static_cast<unsigned char*>(work);
        auto take = [&](size_t b) { unsigned char* q = w; w += CGWork::align(b); return q; };
        r = reinterpret_cast<X*>(take(size_t(n) * sizeof(X)));
        z = reinterpret_cast<X*>(take(size_t(n) * sizeof(X)));
        p = reinterpret_cast<X*>(take(size_t(n) * sizeof(X)));
        double** parts[5] = {&part1, &part2, &pbb, &prz, &pb2};
        for (double** q : parts) *q = reinterpret_cast<double*>(take(SPMV_MAX_BLOCKS * sizeof(double)));
        sums = reinterpret_cast<double*>(take(2 * sizeof(double)));
        st = reinterpret_cast<CGState*>(take(sizeof(CGState)));
        sblocks = spmv_blocks(lpr, n);
        vblocks = std::min(grid_stride_blocks(n), CG_BLOCKS);
    }

    bool jacobi() const { return P && P->kind == NLF_PRECOND_JACOBI; }

    // Column source of the matrix; the lane count follows the kernel it selects.
    void set_cols(const nlf_matrix_s* a) {
        cs = spmv_cols(a);
        lpr = pick_lpr(a);
        sblocks = spmv_blocks(lpr, n);
    }

    // products from the symmetric storage (symv_prepare done): any number of partials
    void set_symmetric(const nlf_matrix_s* a) {
        sym = a;
        sblocks = unsigned(std::min<i64>((a->symv->ns + 3) / 4, SYMV_REDUCE_BLOCKS));
    }

    const X* invd() const;

    // the memory of solve_reliable
    void reserve_reliable() {
        r64.alloc(size_t(n));
        xh.alloc(size_t(n));
    }

    // x: initial guess in, solution out; b: right-hand side.  Returns iterations, sets residual.
    i64 solve(const X* b, X* x, double tol, i64 max_it, double* residual, int* breakdown, int check_every = 8) {
        // r = b - A x ; z = M r ; rz = r.z ; bnorm
        if (sym) residual64(sym, x, b, r, part1, part2, spmv_blocks(64, n), s);
        else
            hipLaunchKernelGGL((k_residual<V, X>), dim3(spmv_blocks(64, n)), dim3(SPMV_THREADS), 0, s, n, outer, cols, val, x, b,
                               r, part1, part2);
        const int nb_res = int(spmv_blocks(64, n));
        NLF_HIP(hipMemcpyAsync(pbb, part2, size_t(nb_res) * sizeof(double), hipMemcpyDeviceToDevice, s));
        precond_apply(P, n, r, p, nullptr, s);
        hipLaunchKernelGGL(k_dot<X>, dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, r, p, part1, (const CGState*)nullptr);
        // pad partial arrays: k_init_state sums vblocks of r.z and nb_res of b.b (cleared by a kernel,
        // not a memset, so that the sequence may be captured)
        const int npad = int(std::max<unsigned>(vblocks, unsigned(nb_res)));
        hipLaunchKernelGGL(k_zero<double>, dim3(grid_stride_blocks(npad)), dim3(256), 0, s, i64(npad), prz);
        hipLaunchKernelGGL(k_zero<double>, dim3(grid_stride_blocks(npad)), dim3(256), 0, s, i64(npad), pb2);
        NLF_HIP(hipMemcpyAsync(prz, part1, size_t(vblocks) * sizeof(double), hipMemcpyDeviceToDevice, s));
        NLF_HIP(hipMemcpyAsync(pb2, pbb, size_t(nb_res) * sizeof(double), hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_init_state, dim3(1), dim3(1024), 0, s, prz, pb2, npad, tol, max_it, indefinite ? 1 : 0, st);
        CGState hs{};
        NLF_HIP(hipMemcpyAsync(&hs, st, sizeof(CGState), hipMemcpyDeviceToHost, s));
        NLF_HIP(hipStreamSynchronize(s));
        while (!hs.done) {
            // the first iteration of each chunk starts with done == 0, so its kernels run in full:
            // HIP events around its SpMV and preconditioner give the live kernel timings
            for (int k = 0; k < check_every; ++k) iteration(x, timed && k == 0);
            NLF_HIP(hipMemcpyAsync(&hs, st, sizeof(CGState), hipMemcpyDeviceToHost, s));
            NLF_HIP(hipStreamSynchronize(s));
        }
        timer.collect();
        if (residual) *residual = hs.res;
        if (breakdown) *breakdown = hs.breakdown;
        return hs.it;
    }

    // Mixed precision with reliable updates: the CG recurrences run in X (FP32) on the X matrix;
    // whenever the recursive residual has dropped by `delta` since the last update, the FP32
    // solution increment is folded into the FP64 solution, the residual is recomputed in FP64 with
    // the FP64 matrix and replaces the recursive one (reserve_reliable first); the search direction is kept, so the
    // Krylov process is not restarted.  Stops on the FP64 true residual ||b - A x|| / ||b|| <= tol.
    i64 solve_reliable(const i64* o64, const i32* c64, const double* v64, const double* b, double* x, double tol,
                       i64 max_it, double delta, double* true_res, i64* updates, int* breakdown) {
        const unsigned rb = spmv_blocks(64, n);
        auto true_residual = [&]() {
            if (sym) residual64(sym, x, b, r64.p, part1, part2, rb, s);
            else residual64(n, o64, cs, v64, lpr, x, b, r64.p, part1, part2, rb, s);
            hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, part1, int(rb), sums);
            hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, part2, int(rb), sums + 1);
            double h[2];
            download(h, sums, 2, s);
            return h[1] > 0.0 ? std::sqrt(h[0] / h[1]) : 0.0;
        };
        // r = M^-1-preconditioned restart data from the FP64 residual: r32 = r64, z = M r32, rz = r32.z
        auto load_residual = [&](bool first) {
            hipLaunchKernelGGL((k_convert<double, X>), dim3(vblocks), dim3(256), 0, s, n, r64.p, r);
            precond_apply(P, n, r, z, nullptr, s);
            if (first) NLF_HIP(hipMemcpyAsync(p, z, size_t(n) * sizeof(X), hipMemcpyDeviceToDevice, s));
            hipLaunchKernelGGL(k_dot<X>, dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, r, z, part1,
                               (const CGState*)nullptr);
            hipLaunchKernelGGL(k_set_rz, dim3(1), dim3(1024), 0, s, part1, int(vblocks), first ? 1 : 0, max_it,
                               indefinite ? 1 : 0, st);
        };
        i64 nupd = 0;
        double rel = true_residual();
        hipLaunchKernelGGL(k_zero<X>, dim3(vblocks), dim3(256), 0, s, n, xh.p);
        CGState hs{};
        if (rel > tol && max_it > 0) {
            load_residual(true);
            NLF_HIP(hipMemcpyAsync(&hs, st, sizeof(CGState), hipMemcpyDeviceToHost, s));
            NLF_HIP(hipStreamSynchronize(s));
            double last = std::sqrt(std::fabs(hs.rz));
            // the recursive estimate sqrt(r'z) is preconditioned; q maps it to the relative true
            // residual as measured at the last update, so that the true residual is also checked
            // once it is predicted to meet tol (not only at the next tenfold drop)
            double q = last > 0.0 ? rel / last : 0.0;
            for (;;) {
                for (int k = 0; k < 8; ++k) iteration(xh.p, k == 0);
                NLF_HIP(hipMemcpyAsync(&hs, st, sizeof(CGState), hipMemcpyDeviceToHost, s));
                NLF_HIP(hipStreamSynchronize(s));
                const double est = std::sqrt(std::fabs(hs.rz));
                const bool stop = hs.it >= max_it || hs.breakdown;
                if (!(est < delta * last) && !(q * est <= tol) && !stop) continue;
                hipLaunchKernelGGL((k_add_to<X, double>), dim3(vblocks), dim3(256), 0, s, n, xh.p, x);
                hipLaunchKernelGGL(k_zero<X>, dim3(vblocks), dim3(256), 0, s, n, xh.p);
                ++nupd;
                rel = true_residual();
                if (rel <= tol || stop) break;
                load_residual(false);
                NLF_HIP(hipMemcpyAsync(&hs, st, sizeof(CGState), hipMemcpyDeviceToHost, s));
                NLF_HIP(hipStreamSynchronize(s));
                last = std::sqrt(std::fabs(hs.rz));
                q = last > 0.0 ? rel / last : 0.0;
            }
        }
        timer.collect();
        if (true_res) *true_res = rel;
        if (updates) *updates = nupd;
        if (breakdown) *breakdown = hs.breakdown;
        return hs.it;
    }

    void iteration(X* x, bool sample = false) {
        // z = A p with the partials of p.z
        if (sample) timer.start(0, s);
        if (sym) launch_symv<true>(sym, p, z, part1, st, s, sblocks, std::is_same_v<V, double> ? SYM_FP64 : lo ? SYM_SPLIT : SYM_FP32);
        else launch_spmv<V, X, double, true>(lpr, n, outer, cs, val, p, z, part1, st, s, false, lo, true, SPMV_PAIRS_IN_FLIGHT, nt);
        if (sample) timer.stop(0, s);
        if (!P || P->kind == NLF_PRECOND_IDENTITY || jacobi()) {
            // x += a p ; r -= a z ; z = M r ; partial r.z  (fused)
            if (jacobi())
                hipLaunchKernelGGL((k_update_xr<X, true, true>), dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, x, r, p, z,
                                   z, invd(), part1, int(sblocks), part2, st);
            else
                hipLaunchKernelGGL((k_update_xr<X, false, true>), dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, x, r, p,
                                   z, z, (const X*)nullptr, part1, int(sblocks), part2, st);
        } else {
            hipLaunchKernelGGL((k_update_xr<X, false, false>), dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, x, r, p, z,
                               (X*)nullptr, (const X*)nullptr, part1, int(sblocks), part2, st);
            if (sample) timer.start(1, s);
            const bool dotted = precond_apply(P, n, r, z, st, s, part2, vblocks);
            if (sample) timer.stop(1, s);
            if (!dotted) hipLaunchKernelGGL(k_dot<X>, dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, r, z, part2, st);
        }
        hipLaunchKernelGGL(k_update_p<X>, dim3(vblocks), dim3(SPMV_THREADS), 0, s, n, p, z, part2, int(vblocks), st);
    }
};

template<> const double* CG<double, double>::invd() const { return P->invd.p; }
template<> const double* CG<float, double>::invd() const { return P->invd.p; }

}  // namespace nlf

#include "nlf_learned.inl"
#include "nlf_batch.inl"

using namespace nlf;

namespace nlf {

// HBM bytes one SpMV streams: values, column source, row pointers, x once and y.  slices: it reads a->symv.
i64 spmv_stream_bytes(const nlf_matrix_s* a, size_t sv, size_t sx, bool slices) {
    const i64 n = a->rows;
    if (slices) {
        // slice values, the strips written and read, the direct sums written and read, x once and y
        const nlf_symv_s& v = *a->symv;
        return v.slots * 64 * i64(sv) + 2 * v.part_size * i64(sizeof(double)) + n * i64(4 * sizeof(double));
    }
    ensure_spmv_storage(a);
    i64 cols = a->nnz_full * i64(a->off16.p ? sizeof(int16_t) : sizeof(i32));
    if (a->pstart.p) cols = a->pat_size * i64(sizeof(int16_t)) + n * i64(sizeof(i64));
    return a->nnz_full * i64(sv) + cols + n * i64(sizeof(i64) + 2 * sx);
}

template<int LPR, int UNROLL, bool NT>
void launch_spmv_variant(nlf_matrix a, const double* x, double* y) {
    ensure_spmv_storage(a);
    hipLaunchKernelGGL((k_spmv<LPR, double, double, double, false, false, UNROLL, NT>), dim3(spmv_blocks(LPR, a->rows)),
                       dim3(SPMV_THREADS), 0, a->ctx->stream, a->rows, a->outer.p, a->cols.p, a->off16.p,
                       static_cast<const i64*>(nullptr), a->val.p, static_cast<const int16_t*>(nullptr), x, y, nullptr,
                       nullptr);
}

}  // namespace nlf

extern "C" {

// y = A x on the inner part (the reference's selfadjointView<Upper>() product), device vectors.
int nlf_spmv(nlf_matrix a, const double* x, double* y) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        if (symv_prepare(a, a->ctx->stream)) {
            launch_symv<false>(a, x, y, nullptr, nullptr, a->ctx->stream, SPMV_MAX_BLOCKS);
            NLF_HIP(hipGetLastError());
            return;
        }
        const int lpr = pick_lpr(a);
        launch_spmv<double, double, double, false>(lpr, a->rows, a->outer.p, spmv_cols(a), a->val.p, x, y, nullptr,
                                                   nullptr,
                                                   a->ctx->stream);
        NLF_HIP(hipGetLastError());
    });
}

int nlf_matrix_symv_info(nlf_matrix a, int64_t* slots, int64_t* strips) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        NLF_CHECK(symv_prepare(a, a->ctx->stream), NLF_ERR_STATE, "the symmetric SpMV storage does not apply");
        if (slots) *slots = a->symv->slots;
        if (strips) *strips = a->symv->part_size;
    });
}

// FP32 SpMV on the FP32 copy (nlf_matrix_make_fp32 first).
int nlf_spmv_fp32(nlf_matrix a, const float* x, float* y) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        NLF_CHECK(a->val32.p, NLF_ERR_STATE, "no FP32 copy");
        const int lpr = pick_lpr(a);
        launch_spmv<float, float, float, false>(lpr, a->rows, a->outer.p, spmv_cols(a), a->val32.p, x, y, nullptr,
                                                nullptr,
                                                a->ctx->stream);
        NLF_HIP(hipGetLastError());
    });
}


// Same SpMV with an explicit lanes-per-row choice (autotuning / benchmarking).  lpr bit 8 selects
// the XCD-contiguous workgroup numbering, bit 9 the 32-bit column indices instead of the offsets,
// bit 12 the per-nonzero 16-bit offsets instead of the row-pattern dictionary, bit 13 the split
// values (FP32 + 16-bit remainder, FP64 vectors; fp32 = 0), bit 14 the one-nonzero-per-load kernel
// instead of the pair kernel, bit 15 two nonzero pairs in flight per lane in the pair kernel instead of
// SPMV_PAIRS_IN_FLIGHT; bits 10 / 11 (FP64 only, LPR 32 or 64, per-nonzero offsets) select 8
// nonzeros in flight per lane / non-temporal loads of the matrix stream.
int nlf_spmv_lpr(nlf_matrix a, int lpr, int fp32, const void* x, void* y) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        const int variant = (lpr >> 10) & 3;
        if (variant && !fp32 && ((lpr & 0xff) == 32 || (lpr & 0xff) == 64)) {
            const double* xd = static_cast<const double*>(x);
            double* yd = static_cast<double*>(y);
            const bool l32 = (lpr & 0xff) == 32;
            if (variant == 1) l32 ? launch_spmv_variant<32, 8, false>(a, xd, yd) : launch_spmv_variant<64, 8, false>(a, xd, yd);
            else if (variant == 2) l32 ? launch_spmv_variant<32, 4, true>(a, xd, yd) : launch_spmv_variant<64, 4, true>(a, xd, yd);
            else l32 ? launch_spmv_variant<32, 8, true>(a, xd, yd) : launch_spmv_variant<64, 8, true>(a, xd, yd);
            NLF_HIP(hipGetLastError());
            return;
        }
        const bool xcd = (lpr & 0x100) != 0;
        const bool split = (lpr & 0x2000) != 0;
        const bool pairs = (lpr & 0x4000) == 0;
        const int pf = (lpr & 0x8000) ? 2 : SPMV_PAIRS_IN_FLIGHT;
        SpmvCols cs = spmv_cols(a);
        if (lpr & 0x1000) cs = SpmvCols{a->cols.p, a->off16.p, nullptr};
        if (lpr & 0x200) cs = SpmvCols{a->cols.p, nullptr, nullptr};
        lpr &= 0xff;
        if (split) {
            NLF_CHECK(a->split_ready, NLF_ERR_STATE, "no split values (nlf_matrix_make_split)");
            launch_spmv<float, double, double, false>(lpr, a->rows, a->outer.p, cs, a->val32.p,
                                                      static_cast<const double*>(x), static_cast<double*>(y), nullptr,
                                                      nullptr, a->ctx->stream, false, a->val_lo.p, pairs);
        } else if (fp32) {
            NLF_CHECK(a->val32.p, NLF_ERR_STATE, "no FP32 values");
            launch_spmv<float, float, float, false>(lpr, a->rows, a->outer.p, cs, a->val32.p, static_cast<const float*>(x),
                                                    static_cast<float*>(y), nullptr, nullptr, a->ctx->stream, xcd, nullptr,
                                                    pairs, pf);
        } else {
            launch_spmv<double, double, double, false>(lpr, a->rows, a->outer.p, cs, a->val.p, static_cast<const double*>(x),
                                                       static_cast<double*>(y), nullptr, nullptr, a->ctx->stream, xcd, nullptr,
                                                       pairs, pf);
        }
        NLF_HIP(hipGetLastError());
    });
}

// f -= K_bound x_D; f[D] = x_D  (boundary_condition_first_kind_2d), device vectors.
int nlf_apply_first_kind(nlf_matrix a, const double* xD, double* f) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        hipLaunchKernelGGL(k_first_kind, dim3(blocks_for(a->rows, 256)), dim3(256), 0, a->ctx->stream, a->rows,
                           a->b_outer.p, a->b_cols.p, a->b_val.p, a->inner.p, xD, f);
        NLF_HIP(hipGetLastError());
    });
}

// init_preconditioner<...> (iterative_solver_base.hpp:203-207): JACOBI from A's diagonal, ILLT from
// the matrix passed (the reference factors the LOCAL matrix, stationary_heat_equation_solver_2d.hpp:91-96).
int nlf_precond_create(nlf_matrix a, int kind, nlf_precond* out) {
    if (!out) return NLF_ERR_ARGUMENT;
    nlf_ctx ctx = a ? a->ctx : nullptr;
    return guarded(ctx, [&] {
        const auto t0 = std::chrono::steady_clock::now();
        auto P = std::make_unique<nlf_precond_s>();
        P->ctx = ctx;
        P->kind = kind;
        if (kind == NLF_PRECOND_IDENTITY) { P->rows = a ? a->rows : 0; *out = P.release(); return; }
        NLF_CHECK(a, NLF_ERR_ARGUMENT, "matrix required");
        hipStream_t s = ctx->stream;
        P->rows = a->rows;
        const i64 n = a->rows;
        if (kind == NLF_PRECOND_JACOBI) {
            P->invd.alloc(size_t(n));
            hipLaunchKernelGGL(k_inv_diag, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, a->diag.p, a->val.p, P->invd.p);
            NLF_HIP(hipGetLastError());
        } else if (kind == NLF_PRECOND_ILLT) {
            // pattern copy + level sets (host analysis of the pattern only)
            std::vector<i64> outer(n + 1), diag(n);
            std::vector<i32> cols(size_t(a->nnz_full));
            download(outer.data(), a->outer.p, outer.size(), s);
            download(diag.data(), a->diag.p, diag.size(), s);
            download(cols.data(), a->cols.p, cols.size(), s);
            std::vector<i32> fr, fp, br, bp;
            level_sets(outer, cols, diag, fr, fp, br, bp);
            P->fw_levels = int(fp.size()) - 1;
            P->bw_levels = int(bp.size()) - 1;
            // independent row blocks (a batch's instances) end a chunk, or get a workgroup of their own
            const std::vector<i64> bounds = independent_blocks(outer, cols, std::max<i64>(1024, n / 2048));
            P->blocks = int(bounds.size()) - 1;
            const i64 *d_outer = a->outer.p, *d_diag = a->diag.p;
            const i32* d_cols = a->cols.p;
            DevBuf<i64> tpos{cols.size()};
            hipLaunchKernelGGL(k_transpose_pos, dim3(blocks_for(n, 4)), dim3(256), 0, s, n, d_outer, d_cols, tpos.p);
            P->scale.alloc(size_t(n));
            P->F.alloc(cols.size());
            hipLaunchKernelGGL(k_scale_from_diag, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, d_diag, a->val.p, P->scale.p);
            DevBuf<int> fail{1};
            // factorisation with growing shift until no pivot fails
            auto factor = [&](auto&& attempt_with) {
                double shift = 0.0;
                P->ok = false;
                for (int attempt = 0; attempt < 40; ++attempt) {
                    attempt_with(shift);
                    NLF_HIP(hipGetLastError());
                    int f = 0;
                    download(&f, fail.p, 1, s);
                    if (!f) { P->ok = true; P->shift = shift; break; }
                    shift = shift == 0.0 ? 1e-3 : 2 * shift;
                }
            };
            SweepPlan pf, pb, pi;                        // forward, backward; the factorisation's where rows merge
            std::vector<uint8_t> mf, mb;
            std::vector<i32> mrows, mptr;
            auto plan = [&](bool forward, std::vector<uint8_t>& merged, SweepPlan& q) {
                if (merged_levels(outer, cols, diag, forward, merged, mrows, mptr))
                    return plan_sweep(outer, cols, diag, mrows, mptr, bounds, forward, merged, false, q);
                merged.clear();
                return plan_sweep(outer, cols, diag, forward ? fr : br, forward ? fp : bp, bounds, forward, merged, false, q);
            };
            // level by level, a workgroup per independent block
            auto factor_levels = [&] {
                DevBuf<i32> lrows, lptr;
                DevBuf<SweepBlock> blk;
                LevelArgs la{n, P->fw_levels, d_outer, d_cols, d_diag, tpos.p, nullptr, nullptr};
                BlockLevels bl;
                std::vector<SweepBlock> bd;
                if (P->blocks > 1) {
                    bl = block_levels(fr, fp, bounds);
                    for (int b = 0; b < P->blocks; ++b) bd.push_back(SweepBlock{bl.levels[size_t(b)], i32(bl.seg[size_t(b)])});
                    upload(blk, bd.data(), bd.size(), s);
                    upload(lrows, bl.rows.data(), bl.rows.size(), s);
                    upload(lptr, bl.ptr.data(), bl.ptr.size(), s);
                } else {
                    upload(lrows, fr.data(), fr.size(), s);
                    upload(lptr, fp.data(), fp.size(), s);
                }
                la.lrows = lrows.p;
                la.lptr = lptr.p;
                factor([&](double shift) {
                    NLF_HIP(hipMemsetAsync(fail.p, 0, sizeof(int), s));
                    hipLaunchKernelGGL(k_ic_init, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, d_outer, d_cols, d_diag, a->val.p,
                                       P->scale.p, shift, P->F.p);
                    hipLaunchKernelGGL(k_ic_factor, dim3(unsigned(P->blocks)), dim3(LEVEL_THREADS), 0, s, la,
                                       P->blocks > 1 ? (const SweepBlock*)blk.p : nullptr, P->F.p, fail.p);
                });
            };
            // over the chunks; false where there is no memory for its lists (up to 4 KB a row)
            auto factor_chunks = [&] {
                try {
                    Sweep own;                           // a merged pair's rows are factored one after the other
                    if (!mf.empty()) {
                        plan_sweep(outer, cols, diag, fr, fp, bounds, true, {}, true, pi);
                        upload_plan(pi, own, s);
                    }
                    const Sweep& sw = mf.empty() ? P->sw_fw : own;
                    DevBuf<i32> list;
                    const int W = std::max(P->sw_fw.WE, P->sw_bw.WE);
                    ic_lists(sw, W, n, d_outer, d_cols, d_diag, list, s);
                    factor([&](double shift) {
                        launch_ic(sw, W, P->ticket.p, d_outer, d_cols, d_diag, tpos.p, list.p, a->val.p, P->scale.p, shift,
                                  i64(cols.size()), P->F.p, fail.p, s);
                    });
                    return true;
                } catch (const OutOfMemory&) {
                    return false;
                }
            };
            P->chunked = cols.size() < (size_t(1) << 31) && plan(true, mf, pf) && plan(false, mb, pb);
            if (P->chunked) {
                upload_plan(pf, P->sw_fw, s);
                upload_plan(pb, P->sw_bw, s);
                P->ticket.alloc(2);
                if (!factor_chunks()) factor_levels();
                pack_sweep(pf, true, d_outer, d_diag, P->F.p, P->scale.p, nullptr, P->sw_fw, s);
                pack_sweep(pb, false, d_outer, d_diag, P->F.p, P->scale.p, P->sw_fw.pos.p, P->sw_bw, s);
                P->fw_lvl.alloc(size_t(n));
                P->bw_lvl.alloc(size_t(n));
                hipLaunchKernelGGL(k_sweep_empty, dim3(grid_stride_blocks(n)), dim3(256), 0, s, n, P->fw_lvl.p, P->bw_lvl.p,
                                   P->ticket.p);
                NLF_HIP(hipGetLastError());
            } else {
                // rows with more dependencies than the chunked sweeps take
                factor_levels();
                build_sweep(outer, cols, diag, fr, fp, true, P->F.p, P->scale.p, d_diag, P->fw, s);
                build_sweep(outer, cols, diag, br, bp, false, P->F.p, P->scale.p, d_diag, P->bw, s);
                const int widest = std::max(P->fw.W, P->bw.W);
                P->solve_threads = std::min(LEVEL_THREADS, std::max(64, (widest + 63) / 64 * 64));
                P->work.alloc(size_t(n));
            }
        } else {
            throw Error(NLF_ERR_UNSUPPORTED, "use nlf_learned_precond_create for the learned preconditioner");
        }
        NLF_HIP(hipStreamSynchronize(s));
        P->setup_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        *out = P.release();
    });
}

int nlf_precond_destroy(nlf_precond p) {
    if (!p) return NLF_OK;
    CtxScope scope(live_ctx(p->ctx));
    delete p;
    return NLF_OK;
}

// computation_info(): ok = 1 on success; shift used; number of forward / backward levels.
int nlf_precond_info(nlf_precond p, int* ok, double* shift, int* fw_levels, int* bw_levels, double* setup_seconds) {
    if (!p) return NLF_ERR_ARGUMENT;
    if (ok) *ok = p->ok;
    if (shift) *shift = p->shift;
    if (fw_levels) *fw_levels = p->fw_levels;
    if (bw_levels) *bw_levels = p->bw_levels;
    if (setup_seconds) *setup_seconds = p->setup_seconds;
    return NLF_OK;
}

int nlf_precond_sweep_info(nlf_precond p, int32_t out[8]) {
    if (!p || !out) return NLF_ERR_ARGUMENT;
    for (int i = 0; i < 8; ++i) out[i] = 0;
    if (p->kind != NLF_PRECOND_ILLT) return NLF_ERR_ARGUMENT;
    for (int k = 0; k < 2; ++k) {
        if (p->chunked) {
            const Sweep& w = k ? p->sw_bw : p->sw_fw;
            out[4 * k] = w.levels;
            out[4 * k + 1] = w.width;
            out[4 * k + 2] = SWEEP_K;
            out[4 * k + 3] = 2;
        } else {
            const auto& w = k ? p->bw : p->fw;
            out[4 * k] = w.levels;
            out[4 * k + 1] = p->solve_threads;
            out[4 * k + 2] = w.K;
            out[4 * k + 3] = 0;
        }
    }
    return NLF_OK;
}

int nlf_precond_blocks(nlf_precond p, int32_t* blocks) {
    if (!p || !blocks || p->kind != NLF_PRECOND_ILLT) return NLF_ERR_ARGUMENT;
    *blocks = p->blocks;
    return NLF_OK;
}

// preconditioner_base::solve: z = M^-1 r on device vectors.
int nlf_precond_apply(nlf_precond p, const double* r, double* z) {
    if (!p) return NLF_ERR_ARGUMENT;
    return guarded(p->ctx, [&] {
        NLF_CHECK(p->rows > 0, NLF_ERR_STATE, "preconditioner has no size");
        if (p->kind == NLF_PRECOND_LEARNED) {
            LearnedGraph& g = *learned_of(p);
            learned_apply<double>(g, g.w.p, r, z, p->ctx->stream);
        } else {
            precond_apply(p, p->rows, r, z, nullptr, p->ctx->stream);
        }
        NLF_HIP(hipGetLastError());
    });
}

// Host export of the ILLT factor in full storage (upper: U, lower: U^T) and the scaling.
int nlf_precond_export_factor(nlf_precond p, double* values, double* scale) {
    if (!p || p->kind != NLF_PRECOND_ILLT) return NLF_ERR_ARGUMENT;
    return guarded(p->ctx, [&] {
        if (values) download(values, p->F.p, p->F.n, p->ctx->stream);
        if (scale) download(scale, p->scale.p, p->scale.n, p->ctx->stream);
    });
}

// conjugate_gradient::solve on device vectors.  mode NLF_MODE_FP64: the reference's PCG with its
// stopping rule sqrt(r'z)/||b|| <= tol.  NLF_MODE_MIXED: FP64 iterative refinement around FP32 PCG
// (x += A32^-1 (b - A x)) until the FP64 true residual ||b - Ax||/||b|| <= tol.  NLF_MODE_SPLIT: the
// same with the values read as FP32 + 16-bit remainder.  x holds the initial guess on entry.
// ---- CG with no allocation -------------------------------------------------------------------
// The work memory of nlf_cg_solve_noalloc: one file-scope device array (every GPU the library runs
// on holds its own copy until the process ends).  Host code never passes the array's name to a
// kernel: its device address, per device, comes from hipGetSymbolAddress at context creation
// (noalloc_scratch_init) and is kept in g_scratch_ptr.
constexpr size_t NOALLOC_SCRATCH_BYTES = 3 * (size_t(NLF_NOALLOC_MAX_ROWS) * sizeof(double)) +
                                         5 * (SPMV_MAX_BLOCKS * sizeof(double)) + 3 * 256;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static void* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
static std::mutex g_scratch_mu;

}  // extern "C"

namespace nlf {
// Called by nlf_ctx_create with `device` current: looks up this device's copy of the scratch array once.
int noalloc_scratch_init(int device) {
    if (device < 0 || device >= NOALLOC_MAX_DEVICES) return NLF_ERR_ARGUMENT;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return NLF_OK;
    void* ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return NLF_ERR_HIP;
    g_scratch_ptr[device] = ptr;
    return NLF_OK;
}
}  // namespace nlf

extern "C" {

int nlf_cg_solve_noalloc(nlf_matrix a, nlf_precond p, const double* b, double* x, double tol, int64_t max_it,
                         nlf_solve_stats* stats) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        NLF_CHECK(b && x, NLF_ERR_ARGUMENT, "null vector");
        NLF_CHECK(!p || p->kind != NLF_PRECOND_LEARNED, NLF_ERR_ARGUMENT, "the learned preconditioner needs nlf_fcg_solve");
        NLF_CHECK(a->rows <= NLF_NOALLOC_MAX_ROWS, NLF_ERR_ARGUMENT,
                  "nlf_cg_solve_noalloc: the matrix has more rows than its fixed work memory holds (NLF_NOALLOC_MAX_ROWS = "
                  "2097152); use nlf_cg_solve");
        NLF_CHECK(CGWork::bytes<double>(a->rows) <= NOALLOC_SCRATCH_BYTES, NLF_ERR_ARGUMENT, "work memory too small");
        const int dev = a->ctx->device;
        void* work = (dev >= 0 && dev < NOALLOC_MAX_DEVICES) ? g_scratch_ptr[dev] : nullptr;
        NLF_CHECK(work, NLF_ERR_STATE, "the fixed work memory of this device was not set up (nlf_ctx_create)");
        hipStream_t s = a->ctx->stream;
        const auto t0 = std::chrono::steady_clock::now();
        const i64 n = a->rows;
        nlf_solve_stats out{};
        out.preconditioner = p ? p->kind : NLF_PRECOND_IDENTITY;
        int breakdown = 0;
        CG<double, double> cg(s, n, a->nnz_full, a->outer.p, a->cols.p, a->val.p, p, work);
        cg.set_cols(a);
        cg.indefinite = a->neumann;
        out.iterations = cg.solve(b, x, tol, max_it, &out.residual, &breakdown);
        out.spmv_bytes = spmv_stream_bytes(a, sizeof(double), sizeof(double), false);
        // FP64 true residual ||b - A x|| / ||b||, with z and the partial arrays of the work memory
        const unsigned rb = spmv_blocks(64, n);
        residual64(n, a->outer.p, spmv_cols(a), a->val.p, pick_lpr(a), x, b, cg.z, cg.part1, cg.part2, rb, s);
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, cg.part1, int(rb), cg.sums);
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, cg.part2, int(rb), cg.sums + 1);
        double h[2];
        download(h, cg.sums, 2, s);
        out.true_residual = h[1] > 0 ? std::sqrt(h[0]) / std::sqrt(h[1]) : 0.0;
        out.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        if (stats) *stats = out;
        NLF_CHECK(!breakdown, NLF_ERR_NUMERIC, "CG breakdown (non-positive curvature or non-finite residual)");
    });
}

int nlf_cg_solve(nlf_matrix a, nlf_precond p, const double* b, double* x, double tol, int64_t max_it, int mode,
                 nlf_solve_stats* stats) {
    if (!a) return NLF_ERR_ARGUMENT;
    return guarded(a->ctx, [&] {
        NLF_CHECK(b && x, NLF_ERR_ARGUMENT, "null vector");
        NLF_CHECK(!p || p->kind != NLF_PRECOND_LEARNED, NLF_ERR_ARGUMENT, "the learned preconditioner needs nlf_fcg_solve");
        hipStream_t s = a->ctx->stream;
        const auto t0 = std::chrono::steady_clock::now();
        const i64 n = a->rows;
        nlf_solve_stats out{};
        out.preconditioner = p ? p->kind : NLF_PRECOND_IDENTITY;
        int breakdown = 0;
        auto timings = [&](const KernelTimer& t, size_t sv, size_t sx, bool slices) {
            out.spmv_ms = t.avg(0);
            out.precond_ms = t.avg(1);
            out.spmv_samples = t.count[0];
            out.spmv_bytes = spmv_stream_bytes(a, sv, sx, slices);
        };
        if (mode == NLF_MODE_FP64) {
            CG<double, double> cg(s, n, a->nnz_full, a->outer.p, a->cols.p, a->val.p, p);
            cg.indefinite = a->neumann;
            if (symv_prepare(a, s)) cg.set_symmetric(a);
            else cg.set_cols(a);
            out.iterations = cg.solve(b, x, tol, max_it, &out.residual, &breakdown);
            timings(cg.timer, sizeof(double), sizeof(double), cg.sym != nullptr);
        } else {
            NLF_CHECK(mode == NLF_MODE_MIXED || mode == NLF_MODE_SPLIT, NLF_ERR_ARGUMENT, "unknown mode");
            NLF_CHECK(a->val32.p, NLF_ERR_STATE, "mixed mode needs nlf_matrix_make_fp32 first");
            NLF_CHECK(mode != NLF_MODE_SPLIT || a->split_ready, NLF_ERR_STATE, "split mode needs nlf_matrix_make_split first");
            // FP32 matrix values (the bytes that bound the SpMV) with FP64 vectors and recurrences: FP32
            // CG recurrences lose orthogonality at the conditioning of these operators (kappa ~ 1e6)
            // and need several times the iterations, while FP32 storage costs none; the FP64 true
            // residual with the FP64 matrix replaces the recursive one at every reliable update.
            CG<float, double> cg(s, n, a->nnz_full, a->outer.p, a->cols.p, a->val32.p, p);
            cg.indefinite = a->neumann;
            if (mode == NLF_MODE_SPLIT) cg.lo = a->val_lo.p;
            cg.reserve_reliable();
            const SymSolve sym(a, cg.lo ? SYM_SPLIT : SYM_FP32, s);
            if (sym.on) cg.set_symmetric(a);
            else cg.set_cols(a);
            out.iterations = cg.solve_reliable(a->outer.p, a->cols.p, a->val.p, b, x, tol, max_it, 0.1,
                                               &out.true_residual, &out.outer_iterations, &breakdown);
            out.residual = out.true_residual;
            timings(cg.timer, mode == NLF_MODE_SPLIT ? sizeof(float) + sizeof(int16_t) : sizeof(float), sizeof(double), sym.on);
        }
        // FP64 true residual ||b - A x|| / ||b||
        {
            const unsigned rb = spmv_blocks(64, n);
            DevBuf<double> r{size_t(n)}, prr{rb}, pbb{rb}, sums{2};
            residual64(a, x, b, r.p, prr.p, pbb.p, rb, s);
            hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, prr.p, int(rb), sums.p);
            hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(1024), 0, s, pbb.p, int(rb), sums.p + 1);
            double h[2];
            download(h, sums.p, 2, s);
            out.true_residual = h[1] > 0 ? std::sqrt(h[0]) / std::sqrt(h[1]) : 0.0;
        }
        out.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        if (stats) *stats = out;
        NLF_CHECK(!breakdown, NLF_ERR_NUMERIC, "CG breakdown (non-positive curvature or non-finite residual)");
    });
}

}  // extern "C"
