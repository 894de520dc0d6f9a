// Triangular sweeps of the ILLT as a dataflow over chunks of rows.  Compiled as part of nlf_solver.hip.
//
// The rows are cut into contiguous chunks in the order of the sweep, so a row depends only on rows of
// its own chunk and of earlier chunks.  One workgroup sweeps one chunk, level by level in steps of at
// most 64 independent records (a record is a row); the chunks run side by side, each a little behind
// the one before it, and pass values on through memory.  What bounds a sweep is the serial chain of
// levels: with one workgroup for all rows a level cost a barrier among ten waves and all record traffic
// went through one compute unit; a chunk's level is one wave's work with no barrier.  One apply (both
// sweeps, one workgroup against chunks): 500 x 500 Q4 nodes 1.14 -> 0.34 ms, 1000 x 1000 2.41 -> 0.71 ms,
// 220 x 220 plane stress 3.07 -> 0.50 ms, 200 x 200 Q8 3.77 -> 0.62 ms, 40 x 40 Q4 67 -> 33 us
// (before rows were merged, see merged_levels).
//
// A workgroup is four waves, one per SIMD, that talk through LDS counters:
//   compute  holds the next records (factor values, dependency addresses) in a register ring and has no
//            store to memory, so it waits for exactly the loads it needs; dependencies come from LDS.  A
//            step of 4 entries takes 190 cycles, 160 of them the LDS write, read and FMA chain; one of
//            12 entries 400 (270 the chain; the rest is the ring of 6 steps, all that 256 registers hold);
//   rhs      gathers the right-hand sides of coming steps into an LDS ring;
//   ext      reads the values of other chunks (and of steps too old for the window) into an LDS ring;
//   store    copies finished steps from the window to memory, in record order.  It loads from LDS only: a
//            load from memory would wait for the stores before it (300 cycles per step instead of 190).
// A value in memory is its own flag: the buffer holds SWEEP_EMPTY, a NaN pattern that no sweep stores,
// until the value is there, and the ext wave reads again until it is (about 2.5 us from one chunk to the
// next).  k_sweep_finish empties both buffers after the backward sweep.  Chunks are handed out in order
// by a ticket, so whoever waits waits for a workgroup that is already running.

#include "nlf_sweep_flow.hpp"

namespace nlf {

constexpr int SWEEP_LEVEL_CAP = 512;     // records of a level before it is split into several
constexpr int SWEEP_EXT = 1024;          // slots of the external values' ring
constexpr int SWEEP_EXT_STEP = 256;      // most new external values of a step
constexpr int SWEEP_EXT_REUSE = 256;     // how far back (in values) a step may use an external value again
constexpr int SWEEP_EB = 1;              // external values per lane of the ext wave
constexpr int SWEEP_MAX_WE = 32;         // most dependencies of a record
constexpr i64 SWEEP_CHUNK_ROWS = 1 << 23;   // most rows of a chunk (32-bit byte offsets into its records)
// LDS: a zero (dependency of the padding entries), the counters, a dump for idle lanes (ctl_store), the
// first records of coming steps, window, right-hand sides, external values
constexpr int SWEEP_CTL = 16, SWEEP_IDLE = 64, SWEEP_SP = 320, SWEEP_WIN = 832, SWEEP_RHS = SWEEP_WIN + SWEEP_K * 512, SWEEP_XV = SWEEP_RHS + SWEEP_R * 512,
              SWEEP_LDS = SWEEP_XV + SWEEP_EXT * 8;
static_assert(SWEEP_SP + 4 * SWEEP_FIRST <= SWEEP_WIN, "the ring of first records lies before the window");
constexpr int SWEEP_ALL = 1 << 30;       // a helper wave has staged every step
constexpr unsigned long long SWEEP_EMPTY = 0xfff8dead0badc0deull;
constexpr int SWEEP_EMPTY_HI = int(SWEEP_EMPTY >> 32), SWEEP_NAN_HI = 0x7ff80000;

struct SweepChunk {
    i32 steps, step0;                    // steps, and the chunk's first offset in sptr / eptr (steps + 1 each)
    i64 ext0;                            // its first external value in esrc
};

struct SweepArgs {
    i32 chunks;
    const SweepChunk* chunk;
    const i32* sptr;                     // first record of each step
    const i32* eptr;                     // external values before each step (from the chunk's first)
    const i32* esrc;                     // record of each external value
    const i32* rsrc;                     // where a record's right-hand side is read
    const double* rcoef;                 // its factor
    // WE factor entries per record, divided by the diagonal, and their LDS byte offsets, in planes of 16 bytes per
    // record (two values or four offsets), so that a wave's load of one plane is one contiguous kilobyte: with a
    // record's bytes together each load touches 64 lines, and 9 such loads took the step of 12 entries 490 cycles
    const unsigned char* rec;
    i64 plane;                           // bytes of a plane
    i64 wait;                            // most reads of a missing value (sweep_wait_reads)
};

// Register-ring depth: the steps whose records are in flight, as many as 256 registers hold (3 per entry
// and step; a wave has the SIMD to itself).  It divides SWEEP_K and SWEEP_R.  At 12 entries 4 steps in
// flight took 510 cycles per step and 6 take 400: the loads' latency.
template<int WE> constexpr int sweep_depth() { return WE <= 4 ? 16 : WE <= 8 ? 8 : WE <= 12 ? 6 : WE <= 16 ? 4 : WE <= 24 ? 3 : 2; }

// LDS counters: one wave's LDS accesses are carried out in order, so a counter stored after the data
// is seen after the data; only the compiler has to keep the order.
__device__ __forceinline__ i32 ctl_load(const i32* p) {
    const i32 v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
    return __builtin_amdgcn_readfirstlane(v);
}
// `p`: the counter in lane 0, a dump elsewhere (no branch on the lane in the chain of steps)
__device__ __forceinline__ void ctl_store(i32* p, i32 v) {
    asm volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template<int WE>
__global__ __launch_bounds__(256) void k_sweep(SweepArgs a, const double* __restrict__ src, double* lvl, i32* ticket,
                                               const CGState* __restrict__ st) {
    __shared__ __align__(64) unsigned char lds[SWEEP_LDS];
    if (st && st->done) return;
    i32* const ctl = reinterpret_cast<i32*>(lds + SWEEP_CTL);    // rhs staged, ext staged, computed, stored, chunk
    double* const win = reinterpret_cast<double*>(lds + SWEEP_WIN);
    double* const rhs = reinterpret_cast<double*>(lds + SWEEP_RHS);
    double* const xv = reinterpret_cast<double*>(lds + SWEEP_XV);
    if (threadIdx.x == 0) {
        *reinterpret_cast<double*>(lds) = 0.0;
        for (int k = 0; k < 4; ++k) ctl[k] = 0;
        ctl[4] = atomicAdd(ticket, 1);
    }
    __syncthreads();
    const i32 c = __builtin_amdgcn_readfirstlane(ctl[4]);
    if (c < 0 || c >= a.chunks) return;
    const SweepChunk ch = a.chunk[c];
    const int n = __builtin_amdgcn_readfirstlane(ch.steps), lane = threadIdx.x & 63;
    const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const i32* __restrict__ sp = a.sptr + ch.step0;
    // this wave's counter
    i32* const mine = reinterpret_cast<i32*>(lds + (lane ? SWEEP_IDLE + 4 * lane : SWEEP_CTL + 4 * (role == 0 ? 2 : role == 3 ? 3 : role - 1)));

    if (role == 0) {
        constexpr int D = sweep_depth<WE>();
        double v[D][WE];
        i32 d[D][WE];
        // Lanes past a step's width take the records that follow (the planes end in 64 spare ones): what
        // they compute goes to window slots that nobody reads.
        const i32 rec0 = __builtin_amdgcn_readfirstlane(sp[0]);
        const unsigned char* const rb = a.rec + i64(rec0) * 16;
        const u32 at = u32(lane - rec0) * 16;
        auto load = [&](i32 first, int u) {
            const u32 o = u32(first) * 16 + at;
#pragma unroll
            for (int k = 0; k < WE / 2; ++k) {
                const uint4 w = *reinterpret_cast<const uint4*>(rb + k * a.plane + o);
                __builtin_memcpy(&v[u][2 * k], &w, 16);
            }
#pragma unroll
            for (int k = 0; k < WE / 4; ++k) {
                const uint4 w = *reinterpret_cast<const uint4*>(rb + (WE / 2 + k) * a.plane + o);
                __builtin_memcpy(&d[u][4 * k], &w, 16);
            }
        };
        i32 spv = sp[min(lane, n)], spf = spv;
        spv = sp[min(D - 1 + lane, n)];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < D; ++u) {
            load(__builtin_amdgcn_readlane(spf, u), u);
            __builtin_amdgcn_sched_barrier(0);
        }
        int avail = 0;
        // whole trips of D steps (the steps past the last compute what follows its records into window
        // slots that nobody reads): no exit inside the unrolled trip, where it would drain the ring
        for (int s0 = 0; s0 < n; s0 += D) {
            const i32 spn = sp[min(s0 + 2 * D - 1 + lane, n)];
            const double* const rs = rhs + (s0 % SWEEP_R) * 64 + lane;
            double* const ws = win + (s0 % SWEEP_K) * 64 + lane;
#pragma unroll
            for (int u = 0; u < D; ++u) {
                const int s = s0 + u;
                while (s >= avail)
                    avail = min(min(ctl_load(ctl), ctl_load(ctl + 1)), sweep_window_end(ctl_load(ctl + 3)));
                double x = rs[u * 64];
                double dv[WE];
#pragma unroll
                for (int j = 0; j < WE; ++j) dv[j] = *reinterpret_cast<const double*>(lds + d[u][j]);
                __builtin_amdgcn_sched_barrier(0);
                // while they are on the way: the slot of the step before is free, refill it
                if (u > 0 || s0 > 0) load(__builtin_amdgcn_readlane(spv, u), (u + D - 1) % D);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < WE; ++j) x -= v[u][j] * dv[j];
                ws[u * 64] = x;
                ctl_store(mine, s + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            spv = spn;
        }
    } else if (role == 1) {
        // three stages, SWEEP_RB steps each: addresses, gathers, LDS.  The steps' first records go to LDS too,
        // for the store wave: that wave must not load, a load behind its stores would wait for them.
        constexpr int B = SWEEP_RB;
        const i32 rec0 = __builtin_amdgcn_readfirstlane(sp[0]);
        const i32* __restrict__ rsrc = a.rsrc + rec0 + lane;
        const double* __restrict__ rcoef = a.rcoef + rec0 + lane;
        i32 ix[B], spa, spb, spc;                // first records of the steps in the LDS, gather and address stages
        double cf[B], x[B], y[B];
        auto addresses = [&](i32 spv) {          // past a step's width: the records that follow (64 spare ones)
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const u32 k = u32(__builtin_amdgcn_readlane(spv, u) - rec0);
                ix[u] = rsrc[k];
                cf[u] = rcoef[k];
            }
        };
        auto gather = [&]() {
#pragma unroll
            for (int u = 0; u < B; ++u) { x[u] = src[ix[u]]; y[u] = cf[u]; }
        };
        spa = sp[min(lane, n)];
        spb = sp[min(B + lane, n)];
        spc = sp[min(2 * B + lane, n)];
        addresses(spa);
        gather();
        addresses(spb);
        for (int s0 = 0; s0 < n; s0 += B) {
            const i32 spn = sp[min(s0 + 3 * B + lane, n)];
            double w[B];
#pragma unroll
            for (int u = 0; u < B; ++u) w[u] = y[u] * x[u];
            gather();
            addresses(spc);
            while (!sweep_rhs_free(s0, ctl_load(ctl + 2), ctl_load(ctl + 3))) __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int u = 0; u < B; ++u) rhs[((s0 + u) % SWEEP_R) * 64 + lane] = w[u];
            if (lane <= B) reinterpret_cast<u32*>(lds + SWEEP_SP)[(s0 + lane) % SWEEP_FIRST] = u32(spa - rec0) * 8;
            ctl_store(mine, s0 + B >= n ? SWEEP_ALL : s0 + B);
            spa = spb;
            spb = spc;
            spc = spn;
        }
    } else if (role == 2) {
        const i32* __restrict__ ep = a.eptr + ch.step0;
        const i32* __restrict__ es = a.esrc + ch.ext0;
        const int total = ep[n];
        constexpr int B = 64 * SWEEP_EB;
        int ready = 0, limit = 0, blk = 0;
        i32 epv = ep[min(1 + lane, n)];              // values needed by the steps of this block of 64
        auto publish = [&](int have) {
            for (;;) {
                const int k = __popcll(__ballot(64 * blk + lane < n && epv <= have));
                ready = 64 * blk + k;
                if (k < 64 || ready >= n) break;
                ++blk;
                epv = ep[min(64 * blk + 1 + lane, n)];
            }
            ctl_store(mine, ready >= n ? SWEEP_ALL : ready);
        };
        for (int e0 = 0; e0 < total; e0 += B) {
            i32 at[SWEEP_EB];
            bool got[SWEEP_EB];
#pragma unroll
            for (int k = 0; k < SWEEP_EB; ++k) {
                const int e = e0 + 64 * k + lane;
                at[k] = es[min(e, total - 1)];
                got[k] = e >= total;
            }
            for (i64 spin = 0;; ++spin) {
                // a slot is free once no step at or after the next one uses the value it holds
                if (limit < min(e0 + B, total)) limit = ep[min(ctl_load(ctl + 2), n)] + SWEEP_EXT - SWEEP_EXT_REUSE;
                unsigned long long w[SWEEP_EB];
#pragma unroll
                for (int k = 0; k < SWEEP_EB; ++k)
                    w[k] = got[k] ? 0 : __hip_atomic_load(reinterpret_cast<unsigned long long*>(lvl) + at[k],
                                                          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                int have = e0;
                bool run = true;
#pragma unroll
                for (int k = 0; k < SWEEP_EB; ++k) {
                    const int e = e0 + 64 * k + lane;
                    if (!got[k] && e < limit && (w[k] != SWEEP_EMPTY || spin >= a.wait)) {
                        xv[e % SWEEP_EXT] = __longlong_as_double(static_cast<long long>(w[k]));
                        got[k] = true;
                    }
                    const unsigned long long miss = __ballot(!got[k]);
                    if (run) have += miss ? __ffsll(miss) - 1 : 64;
                    run = run && !miss;
                }
                have = min(have, total);
                publish(have);
                if (run) break;
                __builtin_amdgcn_s_sleep(1);
            }
        }
        publish(total);
    } else {
        // Finished steps, eight at a time so that their LDS reads overlap.  Past the last finished one the
        // width is 0: nothing is stored.  The only loads are from LDS.
        constexpr int B = 8;
        const u32* const first = reinterpret_cast<const u32*>(lds + SWEEP_SP);
        unsigned char* const out = reinterpret_cast<unsigned char*>(lvl + __builtin_amdgcn_readfirstlane(sp[0]));
        const u32 at = u32(lane) * 8;
        int done = 0;
        while (done < n) {
            const int to = min(ctl_load(ctl + 2), n);
            if (to == done) { __builtin_amdgcn_s_sleep(1); continue; }
            const int m = min(to - done, B);
            u32 b[B + 1];
            int lo[B], hi[B];
#pragma unroll
            for (int k = 0; k <= B; ++k) b[k] = first[(done + min(k, m)) % SWEEP_FIRST];
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const double w = win[((done + min(k, m - 1)) % SWEEP_K) * 64 + lane];
                lo[k] = __double2loint(w);
                hi[k] = __double2hiint(w);
            }
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const u32 o = b[k] + at;
                if (hi[k] == SWEEP_EMPTY_HI) hi[k] = SWEEP_NAN_HI;
                if (o < b[k + 1])
                    __hip_atomic_store(reinterpret_cast<double*>(out + o), __hiloint2double(hi[k], lo[k]), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
            done += m;
            ctl_store(mine, done);
        }
    }
}

// z = S z' in row order from the backward sweep's records, with the partial sums of r.z (k_dot's blocks
// and order) where `partial` is given; empties both sweeps' buffers and resets the tickets.
__global__ __launch_bounds__(SPMV_THREADS) void k_sweep_finish(i64 n, const i32* __restrict__ pos, const double* __restrict__ scale,
                                                               double* __restrict__ fw, double* __restrict__ bw,
                                                               i32* __restrict__ ticket, const double* __restrict__ r,
                                                               double* __restrict__ z, double* __restrict__ partial,
                                                               const CGState* __restrict__ st) {
    __shared__ double sh[SPMV_THREADS / 64];
    if (st && st->done) return;
    const double empty = __longlong_as_double(static_cast<long long>(SWEEP_EMPTY));
    double d = 0.0;
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) {
        const i32 k = pos[i];
        const double zi = scale[i] * bw[k];
        z[i] = zi;
        if (partial) d += r[i] * zi;
        bw[k] = empty;
        fw[i] = empty;
    }
    if (blockIdx.x == 0 && threadIdx.x < 2) ticket[threadIdx.x] = 0;
    if (partial) {
        d = block_sum<double>(d, sh);
        if (threadIdx.x == 0) partial[blockIdx.x] = d;
    }
}

__global__ void k_sweep_empty(i64 n, double* __restrict__ fw, double* __restrict__ bw, i32* __restrict__ ticket) {
    const double empty = __longlong_as_double(static_cast<long long>(SWEEP_EMPTY));
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += i64(gridDim.x) * blockDim.x) { fw[i] = empty; bw[i] = empty; }
    if (blockIdx.x == 0 && threadIdx.x < 2) ticket[threadIdx.x] = 0;
}

// The records' values from the factor.  Entry j of a record is its row's j-th entry below (forward) or above
// (backward) the diagonal over the diagonal; of a row merged with the one before it in the sweep (see
// merged_levels) it is the entry at src[2 t] less m times that row's at src[2 t + 1] (-1: none), m the
// coefficient between the two, and m itself for src[2 t + 1] = -2.  The right-hand side's factor is s_k / U_kk
// and the row (forward) or 1 / U_kk and the row's record in the forward sweep (backward).
__global__ void k_sweep_pack(i64 n, int WE, int forward, const i32* __restrict__ row, const i64* __restrict__ outer,
                             const i64* __restrict__ diag, const double* __restrict__ F, const double* __restrict__ scale,
                             const i32* __restrict__ fw_pos, const i32* __restrict__ dep, const i32* __restrict__ src,
                             unsigned char* __restrict__ out, double* __restrict__ rcoef, i32* __restrict__ rsrc) {
    for (i64 t = i64(blockIdx.x) * blockDim.x + threadIdx.x; t < (n + 64) * WE; t += i64(gridDim.x) * blockDim.x) {
        const i64 rec = t / WE;
        const int j = int(t - rec * WE);
        double* const v = reinterpret_cast<double*>(out + (j / 2) * (n + 64) * 16 + rec * 16) + j % 2;
        i32* const d = reinterpret_cast<i32*>(out + (WE / 2 + j / 4) * (n + 64) * 16 + rec * 16) + j % 4;
        if (rec >= n) {
            *v = 0.0;
            *d = 0;
            if (j == 0) { rcoef[rec] = 0.0; rsrc[rec] = 0; }
            continue;
        }
        const i64 k = row[rec], dk = diag[k];
        const double inv = 1.0 / F[dk];
        if (src) {
            const i32 pk = src[2 * t], pa = src[2 * t + 1];
            double x = pk >= 0 ? F[pk] * inv : 0.0;
            if (pa != -1) {
                const double m = F[forward ? dk - 1 : dk + 1] * inv;
                x = pa < 0 ? m : x - m * (F[pa] / F[diag[forward ? k - 1 : k + 1]]);
            }
            *v = x;
        } else {
            const i64 p = (forward ? outer[k] : dk + 1) + j, e = forward ? dk : outer[k + 1];
            *v = p < e ? F[p] * inv : 0.0;
        }
        *d = dep[t];
        if (j == 0) {
            rcoef[rec] = forward ? scale[k] * inv : inv;
            rsrc[rec] = forward ? i32(k) : fw_pos[k];
        }
    }
}

// ---- plan (host) ---------------------------------------------------------------------------------------
struct SweepPlan {
    int WE = 4, levels = 0, width = 64;
    std::vector<SweepChunk> chunk;
    std::vector<i32> sptr, eptr, esrc;
    std::vector<i32> row, pos;           // row of each record, record of each row
    std::vector<i32> dep;
    std::vector<i32> src;                // with merged rows: two factor positions per entry (k_sweep_pack)
};

static int sweep_width(i64 entries) { return entries <= 4 ? 4 : entries <= 8 ? 8 : entries <= 12 ? 12 : entries <= 16 ? 16 : entries <= 24 ? 24 : 32; }

// Levels with rows merged in pairs: row k takes the place of its dependency a on the row right before it in the
// sweep, y_a = b_a - sum c_ad y_d, into its own sum, so that both are solved at once: b_k - m b_a and the
// coefficients c_kd - m c_ad over the union of the two rows' dependencies (and m for b_a).  A pair is merged
// where that union still fits the entries a record has anyway, so a step costs the same and there are fewer:
// plane stress 2 levels a node less one (1320 -> 660 at 220 x 220), Q8 1600 -> 1000 at 200 x 200; never on Q4
// heat rows, whose unions have 6 entries.  One apply: plane stress 500 -> 280 us, Q8 617 -> 484 us.
// False where too few pairs merge to matter.
static bool merged_levels(const std::vector<i64>& outer, const std::vector<i32>& cols, const std::vector<i64>& diag,
                          bool forward, std::vector<uint8_t>& merged, std::vector<i32>& lrows, std::vector<i32>& lptr) {
    const i64 n = i64(diag.size());
    auto begin = [&](i64 k) { return forward ? outer[k] : diag[k] + 1; };
    auto end = [&](i64 k) { return forward ? diag[k] : outer[k + 1]; };
    i64 widest = 0;
    for (i64 k = 0; k < n; ++k) widest = std::max(widest, end(k) - begin(k));
    if (widest > SWEEP_MAX_WE) return false;
    const int cap = sweep_width(widest);
    // whether row k's entries with those of the row before it fit a record (a itself among them: the entry of b_a)
    auto fits = [&](i64 k) {
        const i64 a = forward ? k - 1 : k + 1;
        const i64 b = begin(k), e = end(k);
        if (e == b || i64(cols[size_t(forward ? e - 1 : b)]) != a) return false;
        i64 p = b, q = begin(a), count = 0;
        const i64 ea = end(a);
        while (p < e || q < ea) {
            const i32 cp = p < e ? cols[size_t(p)] : INT32_MAX, cq = q < ea ? cols[size_t(q)] : INT32_MAX;
            p += cp <= cq;
            q += cq <= cp;
            ++count;
        }
        return count <= cap;
    };
    // a look at some rows first: of those that fit, every second one is merged
    const i64 every = std::max<i64>(1, n / 1024);
    i64 seen = 0, fit = 0;
    for (i64 k = every / 2; k < n; k += every, ++seen) fit += fits(k);
    if (8 * fit < seen) return false;
    merged.assign(size_t(n), 0);
    std::vector<i32> lev(static_cast<size_t>(n));
    i32 levels = 0;
    i64 pairs = 0;
    for (i64 o = 0; o < n; ++o) {
        const i64 k = forward ? o : n - 1 - o, a = forward ? k - 1 : k + 1;
        const i64 b = begin(k), e = end(k);
        const bool linked = e > b && i64(cols[size_t(forward ? e - 1 : b)]) == a;
        const bool join = linked && !merged[size_t(a)] && fits(k);
        i32 l = linked ? lev[size_t(a)] + (join ? 0 : 1) : 0;
        for (i64 p = b; p < e; ++p)
            if (i64(cols[size_t(p)]) != a) l = std::max(l, lev[size_t(cols[size_t(p)])] + 1);
        if (join) {
            merged[size_t(k)] = 1;
            ++pairs;
            lev[size_t(a)] = l;                              // nothing but k depends on a yet
        }
        lev[size_t(k)] = l;
        levels = std::max(levels, l + 1);
    }
    if (8 * pairs < n) return false;
    lptr.assign(size_t(levels) + 1, 0);
    for (i64 k = 0; k < n; ++k) lptr[size_t(lev[size_t(k)]) + 1]++;
    for (i32 l = 0; l < levels; ++l) lptr[size_t(l) + 1] += lptr[size_t(l)];
    lrows.resize(size_t(n));
    std::vector<i32> at(lptr.begin(), lptr.end() - 1);
    for (i64 o = 0; o < n; ++o) {
        const i64 k = forward ? o : n - 1 - o;
        lrows[size_t(at[size_t(lev[size_t(k)])]++)] = i32(k);
    }
    return true;
}

// Chunks, steps and dependencies of one sweep; false when a row has more than SWEEP_MAX_WE dependencies.
// lrows / lptr: the rows by level, in sweep order within a level.  bounds: independent row blocks, whose
// boundaries end a chunk.  merged: rows merged with the one before them in the sweep (merged_levels; empty:
// none), kept in one step with it.  steps_only: no dependencies (for the factorisation).
//
// A chunk grows while its steps stay few more than its levels: each level of the chunk then fits the
// wave, so a longer chunk would only lengthen the chain and a shorter one would add a hand-over between
// workgroups (about 2.5 us).  On a grid of n x n nodes in row order that is 64 rows of nodes.
static bool plan_sweep(const std::vector<i64>& outer, const std::vector<i32>& cols, const std::vector<i64>& diag,
                       const std::vector<i32>& lrows, const std::vector<i32>& lptr, const std::vector<i64>& bounds,
                       bool forward, const std::vector<uint8_t>& merged, bool steps_only, SweepPlan& P) {
    const i64 n = i64(diag.size());
    i64 widest = 0;
    for (i64 k = 0; k < n; ++k) widest = std::max(widest, forward ? diag[k] - outer[k] : outer[k + 1] - diag[k] - 1);
    if (widest > SWEEP_MAX_WE) return false;
    P.WE = sweep_width(widest);
    auto is_merged = [&](i64 k) { return !merged.empty() && merged[size_t(k)]; };
    // levels wider than the cap (often level 0, the first-kind rows) are split: their records are independent
    std::vector<i32> lev(static_cast<size_t>(n));
    int levels = 0;
    i64 w = 1;
    for (size_t L = 0; L + 1 < lptr.size(); ++L)
        for (i32 t = lptr[L], e; t < lptr[L + 1]; t = e, ++levels) {
            e = std::min(t + SWEEP_LEVEL_CAP, lptr[L + 1]);
            if (e < lptr[L + 1] && is_merged(lrows[size_t(e)])) --e;           // not between a pair
            w = std::max<i64>(w, e - t);
            for (i32 i = t; i < e; ++i) lev[size_t(lrows[size_t(i)])] = levels;
        }
    P.levels = levels;
    P.width = int((w + 63) / 64 * 64);
    // chunks of consecutive rows in sweep order
    std::vector<i32> chunk_of(static_cast<size_t>(n)), cnt(static_cast<size_t>(levels), 0), stamp(static_cast<size_t>(levels), -1);
    std::vector<i64> first;                              // records before each chunk
    {
        int c = -1;
        i64 steps = 0, distinct = 0;
        size_t b = 0;
        for (i64 o = 0; o < n; ++o) {
            const i64 k = forward ? o : n - 1 - o;
            const bool edge = b + 1 < bounds.size() && k == (forward ? bounds[b] : bounds[bounds.size() - 1 - b] - 1);
            if (edge) ++b;
            if (c < 0 || edge || (!is_merged(k) && (steps - distinct > std::max<i64>(4, distinct / 64) || o - first.back() >= SWEEP_CHUNK_ROWS))) {
                ++c;
                first.push_back(o);
                steps = distinct = 0;
            }
            const size_t l = size_t(lev[size_t(k)]);
            if (stamp[l] != c) { stamp[l] = c; cnt[l] = 0; ++distinct; }
            if (cnt[l]++ % 64 == 0) ++steps;
            chunk_of[size_t(k)] = c;
        }
        first.push_back(n);
    }
    const int C = int(first.size()) - 1;
    P.row.resize(size_t(n));
    P.pos.resize(size_t(n));
    {
        std::vector<i64> at(first.begin(), first.end() - 1);
        for (i64 t = 0; t < n; ++t) {
            const i32 k = lrows[size_t(t)];
            const i64 rec = at[size_t(chunk_of[size_t(k)])]++;
            P.row[size_t(rec)] = k;
            P.pos[size_t(k)] = i32(rec);
        }
    }
    if (!steps_only) P.dep.assign(size_t(P.WE) * size_t(n), 0);
    if (!merged.empty()) P.src.assign(2 * size_t(P.WE) * size_t(n), -1);
    P.chunk.resize(size_t(C));
    std::vector<i32> step_of(static_cast<size_t>(n)), lane_of(static_cast<size_t>(n));
    std::vector<i32> x_chunk(static_cast<size_t>(n), -1), x_idx(static_cast<size_t>(n), 0);     // last external slot of a row
    for (int c = 0; c < C; ++c) {
        SweepChunk& ch = P.chunk[size_t(c)];
        ch.step0 = i32(P.sptr.size());
        ch.ext0 = i64(P.esrc.size());
        int step = -1, lane = 64, in_step = 0;
        i32 level = -1, ext = 0, ext_begin = 0;
        for (i64 rec = first[size_t(c)]; rec < first[size_t(c) + 1]; ++rec) {
            const i32 k = P.row[size_t(rec)];
            const i64 pb = forward ? outer[k] : diag[k] + 1, pe = forward ? diag[k] : outer[k + 1];
            // a pair's records lie side by side: the later one reads the earlier one's right-hand side
            const bool joined = is_merged(k);
            const bool pair = rec + 1 < first[size_t(c) + 1] && is_merged(P.row[size_t(rec) + 1]) && !joined &&
                              P.row[size_t(rec) + 1] == (forward ? k + 1 : k - 1);
            if (!joined && (lev[size_t(k)] != level || lane + int(pair) >= 64 ||
                            in_step + (pair ? 2 : 1) * P.WE > SWEEP_EXT_STEP)) {
                ++step;
                lane = in_step = 0;
                level = lev[size_t(k)];
                ext_begin = ext;
                P.sptr.push_back(i32(rec));
                P.eptr.push_back(ext);
            }
            step_of[size_t(k)] = step;
            lane_of[size_t(k)] = lane++;
            if (steps_only) continue;
            i32* dep = &P.dep[size_t(P.WE) * size_t(rec)];
            auto depend = [&](i32 i) {
                if (chunk_of[size_t(i)] == c && step - step_of[size_t(i)] <= SWEEP_K) {
                    *dep++ = SWEEP_WIN + ((step_of[size_t(i)] % SWEEP_K) * 64 + lane_of[size_t(i)]) * 8;
                    return;
                }
                if (x_chunk[size_t(i)] != c || ext_begin - x_idx[size_t(i)] > SWEEP_EXT_REUSE) {
                    x_chunk[size_t(i)] = c;
                    x_idx[size_t(i)] = ext++;
                    P.esrc.push_back(P.pos[size_t(i)]);
                    ++in_step;
                }
                *dep++ = SWEEP_XV + (x_idx[size_t(i)] % SWEEP_EXT) * 8;
            };
            if (merged.empty()) {
                for (i64 p = pb; p < pe; ++p) depend(cols[size_t(p)]);
                continue;
            }
            i32* src = &P.src[2 * size_t(P.WE) * size_t(rec)];
            const i32 a = forward ? k - 1 : k + 1;
            i64 p = pb, q = joined ? (forward ? outer[a] : diag[a] + 1) : 0;
            const i64 qe = joined ? (forward ? diag[a] : outer[a + 1]) : 0;
            while (p < pe || q < qe) {
                const i32 cp = p < pe ? cols[size_t(p)] : INT32_MAX, cq = q < qe ? cols[size_t(q)] : INT32_MAX;
                const i32 i = std::min(cp, cq);
                if (joined && i == a) {
                    src[0] = i32(p);
                    src[1] = -2;
                    *dep++ = SWEEP_RHS + ((step % SWEEP_R) * 64 + lane_of[size_t(a)]) * 8;
                } else {
                    src[0] = cp == i ? i32(p) : -1;
                    src[1] = cq == i ? i32(q) : -1;
                    depend(i);
                }
                src += 2;
                p += cp == i;
                q += cq == i;
            }
        }
        P.sptr.push_back(i32(first[size_t(c) + 1]));
        P.eptr.push_back(ext);
        ch.steps = step + 1;
    }
    return true;
}

// ---- factorisation --------------------------------------------------------------------------------------
// IC(0) over the forward sweep's chunks and steps.  A row takes GL lanes, one per entry: lane l holds entry l
// below the diagonal and computes entry l above it.  What bounds it is the chain of levels again, here with
// a memory round trip per level: with one workgroup and one thread per row, a row's entries and merges were
// serial loads (30 us per level at 200 x 200 Q8).  No barrier: like the sweeps, a value is its own flag and
// is read again until it is there, each wave going through the steps by itself.  Whole set-up of the
// preconditioner, host analysis included, before and after: 200 x 200 Q8 59 -> 25 ms, 220 x 220 plane
// stress 49 -> 19.5 ms (of these two, 11 and 7 ms are the host's, for merging rows and for a plan of the
// factorisation without merged ones), 500 x 500 Q4 26 -> 15 ms, 1000 x 1000 Q4 154 -> 106 ms, 40 x 40 Q4
// 1.2 -> 0.6 ms.
//
// Entry m of lane l's list: the position in row j (the column of entry l above the diagonal) of column
// cols[outer[k] + m], -1 where row j lacks it.
template<int M> constexpr int ic_lanes() { return M <= 4 ? 4 : M <= 8 ? 8 : M <= 16 ? 16 : 32; }
// rows a workgroup takes at a time: a whole step, or what 256 registers a lane allow
template<int M> constexpr int ic_rows() { return M <= 12 ? 64 : M <= 16 ? 32 : 16; }

__global__ void k_ic_lists(i64 n, int M, int GL, const i32* __restrict__ row, const i64* __restrict__ outer,
                           const i32* __restrict__ cols, const i64* __restrict__ diag, i32* __restrict__ list) {
    for (i64 t = i64(blockIdx.x) * blockDim.x + threadIdx.x; t < n * M * GL; t += i64(gridDim.x) * blockDim.x) {
        const i64 rec = t / (M * GL), k = row[rec], b = outer[k], dk = diag[k];
        const int m = int(t / GL % M), l = int(t % GL);
        i32 at = -1;
        if (b + m < dk && dk + 1 + l < outer[k + 1]) {
            const i32 i = cols[b + m], j = cols[dk + 1 + l];
            i64 lo = outer[j], hi = diag[j];
            while (lo < hi) {
                const i64 mid = (lo + hi) >> 1;
                if (cols[mid] < i) lo = mid + 1; else hi = mid;
            }
            if (lo < diag[j] && cols[lo] == i) at = i32(lo);
        }
        list[t] = at;
    }
}

__device__ __forceinline__ double ic_load(const double* F, i64 p) {
    return __hip_atomic_load(F + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ic_store(double* F, i64 p, double v) {
    if (__double2hiint(v) == SWEEP_EMPTY_HI) v = __hiloint2double(SWEEP_NAN_HI, 0);
    __hip_atomic_store(F + p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template<int M>
__global__ __launch_bounds__(ic_lanes<M>() * ic_rows<M>()) void k_ic_chunks(SweepArgs s, i32* ticket, const i32* __restrict__ row,
                                                   const i64* __restrict__ outer, const i32* __restrict__ cols,
                                                   const i64* __restrict__ diag, const i64* __restrict__ tpos,
                                                   const i32* __restrict__ list, const double* __restrict__ a,
                                                   const double* __restrict__ scale, double shift, double* F, int* fail) {
    constexpr int GL = ic_lanes<M>(), G = ic_rows<M>();
    __shared__ i32 sh_c;
    if (threadIdx.x == 0) sh_c = atomicAdd(ticket, 1);
    __syncthreads();
    const i32 c = __builtin_amdgcn_readfirstlane(sh_c);
    if (c < 0 || c >= s.chunks) return;
    const SweepChunk ch = s.chunk[c];
    const i32* __restrict__ sp = s.sptr + ch.step0;
    const int g = threadIdx.x / GL, l = threadIdx.x % GL;
    // what does not depend on the factor, one step ahead of its use
    struct Row {
        i64 b, dk;
        int nl, nu;
        i32 at[M];
        i64 tp;
        double av, ad;
    };
    const int slots = ch.steps * (64 / G);
    auto fetch = [&](int t) {
        Row r;
        const int st = t / (64 / G), rec = sp[st] + t % (64 / G) * G + g;
        const bool on = rec < sp[st + 1];
        const i64 k = row[on ? rec : sp[st]], e = outer[k + 1];
        r.b = outer[k];
        r.dk = diag[k];
        r.nl = on ? int(r.dk - r.b) : -1;
        r.nu = on ? int(e - r.dk - 1) : 0;
        const bool up = l < r.nu;
        const i64 p = up ? r.dk + 1 + l : r.dk;
#pragma unroll
        for (int m = 0; m < M; ++m) r.at[m] = up ? list[(i64(rec) * M + m) * GL + l] : -1;
        r.tp = tpos[p];
        r.av = scale[k] * a[p] * scale[cols[p]];
        r.ad = scale[k] * a[r.dk] * scale[k] + shift;
        return r;
    };
    Row next = fetch(0);
    for (int t = 0; t < slots; ++t) {
        const Row r = next;
        if (t + 1 < slots) next = fetch(t + 1);
        // the entries below the diagonal and the other rows' entries, until all are there
        double low = 0.0, fj[M];
        bool got = !(l < r.nl);
#pragma unroll
        for (int m = 0; m < M; ++m) fj[m] = 0.0;
        u32 want = 0;
#pragma unroll
        for (int m = 0; m < M; ++m) want |= r.at[m] >= 0 ? 1u << m : 0u;
        for (i64 spin = 0;; ++spin) {
            if (!got) low = ic_load(F, r.b + l);
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (want >> m & 1) fj[m] = ic_load(F, r.at[m]);
            const bool give_up = spin >= s.wait;
            if (!got && (__double2hiint(low) != SWEEP_EMPTY_HI || give_up)) got = true;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if ((want >> m & 1) && (__double2hiint(fj[m]) != SWEEP_EMPTY_HI || give_up)) want &= ~(1u << m);
            if (!__ballot(!got || want)) break;
        }
        double d = r.ad, v = r.av;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const double x = __shfl(low, m, GL);
            if (m < r.nl) d -= x * x;
            if (r.at[m] >= 0) v -= x * fj[m];
        }
        if (r.nl >= 0) {
            if (!(d > 0.0) || !isfinite(d)) {
                if (l == 0) *fail = 1;
                d = 1.0;
            }
            const double ukk = sqrt(d);
            if (l == 0) ic_store(F, r.dk, ukk);
            if (l < r.nu) {
                v /= ukk;
                ic_store(F, r.dk + 1 + l, v);
                if (r.tp != r.dk + 1 + l) ic_store(F, r.tp, v);
            }
        }
    }
}

// F emptied, the ticket and the failure flag cleared
__global__ void k_ic_empty(i64 nnz, double* __restrict__ F, i32* __restrict__ ticket, int* __restrict__ fail) {
    const double empty = __longlong_as_double(static_cast<long long>(SWEEP_EMPTY));
    for (i64 i = i64(blockIdx.x) * blockDim.x + threadIdx.x; i < nnz; i += i64(gridDim.x) * blockDim.x) F[i] = empty;
    if (blockIdx.x == 0 && threadIdx.x == 0) { *ticket = 0; *fail = 0; }
}

// One sweep on the device.
struct Sweep {
    int chunks = 0, WE = 4, levels = 0, width = 64;
    DevBuf<SweepChunk> chunk;
    DevBuf<i32> sptr, eptr, esrc, rsrc, pos, row;
    DevBuf<double> rcoef;
    DevBuf<unsigned char> rec;
    i64 plane = 0, steps = 0;            // steps of all chunks
    SweepArgs args() const { return {chunks, chunk.p, sptr.p, eptr.p, esrc.p, rsrc.p, rcoef.p, rec.p, plane, sweep_wait_reads(steps)}; }
};

// The plan without the factor's values.
static void upload_plan(const SweepPlan& P, Sweep& sw, hipStream_t s) {
    sw.chunks = int(P.chunk.size());
    sw.WE = P.WE;
    sw.levels = P.levels;
    sw.width = P.width;
    sw.steps = i64(P.sptr.size()) - sw.chunks;
    upload(sw.chunk, P.chunk.data(), P.chunk.size(), s);
    upload(sw.sptr, P.sptr.data(), P.sptr.size(), s);
    upload(sw.eptr, P.eptr.data(), P.eptr.size(), s);
    const i32 none = 0;
    upload(sw.esrc, P.esrc.empty() ? &none : P.esrc.data(), std::max<size_t>(P.esrc.size(), 1), s);
    upload(sw.pos, P.pos.data(), P.pos.size(), s);
    upload(sw.row, P.row.data(), P.row.size(), s);
    NLF_HIP(hipStreamSynchronize(s));                   // `none`
}

// The records, from the factor.
static void pack_sweep(const SweepPlan& P, bool forward, const i64* d_outer, const i64* d_diag, const double* F,
                       const double* scale, const i32* fw_pos, Sweep& sw, hipStream_t s) {
    const i64 n = i64(P.row.size());
    DevBuf<i32> dep, src;
    upload(dep, P.dep.data(), P.dep.size(), s);
    if (!P.src.empty()) upload(src, P.src.data(), P.src.size(), s);
    sw.plane = 16 * (n + 64);
    sw.rec.alloc(size_t(12 * P.WE) * size_t(n + 64));
    sw.rcoef.alloc(size_t(n + 64));
    sw.rsrc.alloc(size_t(n + 64));
    hipLaunchKernelGGL(k_sweep_pack, dim3(grid_stride_blocks((n + 64) * P.WE)), dim3(256), 0, s, n, P.WE, int(forward), sw.row.p,
                       d_outer, d_diag, F, scale, fw_pos, dep.p, src.p, sw.rec.p, sw.rcoef.p, sw.rsrc.p);
    NLF_HIP(hipGetLastError());
    NLF_HIP(hipStreamSynchronize(s));                   // the plan's host arrays are released
}

// The lists of k_ic_chunks (by record); 32-bit positions.
// W: the width class of the rows' entries on either side of the diagonal, whichever has more (a lane computes an
// entry above it, and the lists run over those below).
static void ic_lists(const Sweep& w, int W, i64 n, const i64* outer, const i32* cols, const i64* diag, DevBuf<i32>& list, hipStream_t s) {
    const int GL = W <= 4 ? 4 : W <= 8 ? 8 : W <= 16 ? 16 : 32;
    list.alloc(size_t(n) * size_t(W) * size_t(GL));
    hipLaunchKernelGGL(k_ic_lists, dim3(grid_stride_blocks(n * W * GL)), dim3(256), 0, s, n, W, GL, w.row.p, outer, cols,
                       diag, list.p);
}

static void launch_ic(const Sweep& w, int W, i32* ticket, const i64* outer, const i32* cols, const i64* diag, const i64* tpos,
                      const i32* list, const double* a, const double* scale, double shift, i64 nnz, double* F, int* fail,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_ic_empty, dim3(grid_stride_blocks(nnz)), dim3(256), 0, s, nnz, F, ticket, fail);
#define NLF_IC_CASE(C)                                                                                                   \
    hipLaunchKernelGGL((k_ic_chunks<C>), dim3(unsigned(w.chunks)), dim3(unsigned(ic_lanes<C>() * ic_rows<C>())), 0, s,         \
                       w.args(), ticket, w.row.p, outer, cols, diag, tpos, list, a, scale, shift, F, fail)
    switch (W) {
        case 4: NLF_IC_CASE(4); break;
        case 8: NLF_IC_CASE(8); break;
        case 12: NLF_IC_CASE(12); break;
        case 16: NLF_IC_CASE(16); break;
        case 24: NLF_IC_CASE(24); break;
        default: NLF_IC_CASE(32); break;
    }
#undef NLF_IC_CASE
}

static void launch_sweep(const Sweep& w, const double* src, double* lvl, i32* ticket, const CGState* st, hipStream_t s) {
    const dim3 g(unsigned(w.chunks)), b(256);
    switch (w.WE) {
        case 4: hipLaunchKernelGGL((k_sweep<4>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
        case 8: hipLaunchKernelGGL((k_sweep<8>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
        case 12: hipLaunchKernelGGL((k_sweep<12>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
        case 16: hipLaunchKernelGGL((k_sweep<16>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
        case 24: hipLaunchKernelGGL((k_sweep<24>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
        default: hipLaunchKernelGGL((k_sweep<32>), g, b, 0, s, w.args(), src, lvl, ticket, st); break;
    }
}

}  // namespace nlf
