// resident.hpp -- Krylov iterations in one launch, the system on the chip.
//
// A system of up to a few hundred thousand rows spends a Krylov iteration in
// the dispatch of its three (CG) or five (BiCGStab) dependent launches: on
// 200 x 200 quads each takes 3.5-4 us, of which the work itself is well
// under one.  A resident launch keeps one workgroup per few row chunks on
// the chip for a whole batch of iterations; a thread owns one row and holds
// its matrix entries, its x, r, p and the direction values of its columns in
// registers.  What the workgroups exchange -- one double per chunk and dot
// product, and one vector entry per row -- goes through relaxed agent-scope
// atomics (sc1 accesses: stores written through, loads served past the
// non-coherent caches), so no barrier writes back or invalidates an L2: a
// release / acquire pair per barrier costs 10 us over 256 workgroups, an
// exchange by atomics 1.4-2.0 us.
//
// The exchange of a dot product is also the barrier: every workgroup posts
// its partial sums and waits for those of all others.  A CG iteration needs
// two of them.  z = r / d is published before the second, and each thread
// forms p = z + beta p for its own columns from the z it gathers and the p
// it kept, so the new direction needs no barrier of its own.
//
// Arithmetic: rows, threads, partial sums and their order of addition are
// those of the separate launches (row_chunk, store_partials,
// finish_partials), so iterates agree with them bit for bit.
//
// Waiting: a launch first counts its workgroups in (res_census).  Only when
// all of them are resident does any of them enter the iterations; when that
// takes too long (another launch holds the chip) all leave, nothing has
// changed, and the host takes the separate launches.  After the census every
// workgroup runs until the batch ends, so each wait is for a workgroup that
// is running; the waits are bounded all the same.
#pragma once

#include "kernels.hpp"

namespace ogsx {

// A slot that holds no partial sum yet: a NaN no dot product yields (a sum
// with these bits is posted as the default NaN).
constexpr unsigned long long kSlotEmpty = 0xFFF8DEADBEEF0001ull;
constexpr int kSlotSets = 3;    // rotating sets of slots
constexpr int kSlotVals = 3;    // values of one exchange
// Copies of each slot: workgroup w reads copy w % 8, so that a line is
// polled by an eighth of the workgroups (256 workgroups: 3.2 -> 2.0 us per
// exchange; 16: 1.5 -> 1.4 us).
constexpr int kSlotCopies = 8;
constexpr int kResMaxSlots = kBlock;          // slots per value and copy
constexpr int kResMaxRows = 1 << 18;          // rows of a resident system
// Larger systems whose vectors fit the LDS of 256 workgroups (k_cg_stream):
// 1024 chunks, four to a workgroup, of up to 9 rows per thread.
constexpr int kStreamVb = 4;
constexpr int kStreamBlocks = 1024;
constexpr int kStreamSlots = 9;
constexpr int kStreamMaxRows = kStreamBlocks * kStreamSlots * kBlock;
constexpr int kFirstPoll = 12;                // 64-clock units before the first poll
constexpr unsigned kResPolls = 1u << 21;      // polls of one wait (seconds)
constexpr long long kCensusTicks = 20000;     // 100 MHz: 200 us
constexpr int kCensusRing = 64;

// Exchange buffers of one system, kept between launches.
struct ResSync {
    int phase;  // set of the next exchange (its slots are empty)
    int pad[31];
    unsigned long long slot[1];  // [set][value][copy][slots]
};

__host__ __device__ constexpr int res_slots(int G)
{
    return ((G + part_q(G) - 1) / part_q(G) + 15) / 16 * 16;
}
__host__ __device__ constexpr size_t res_slot_count(int G)
{
    return (size_t)kSlotSets * kSlotVals * kSlotCopies * res_slots(G);
}
constexpr size_t res_sync_bytes(int G) { return sizeof(int) * 32 + 8 * res_slot_count(G); }

// Arrival count and decision of one launch (0 open, 1 go, 2 leave).
struct ResCensus {
    unsigned arrived;
    int decision;
    int pad[14];
};

// One resident launch: its census entry, the workgroups to count and
// iterations.  A launch clears the entry half a ring ahead for a later one, so
// only launches that take the census may be numbered through the ring: one
// that does not (k_cg_one, k_bi_one) would leave the entry it skips with an
// old count and decision, and the launch that takes that entry next would go
// on, or leave, without counting anyone in.
struct ResLaunch {
    ResCensus* ring;
    int entry;
    int wgs;
    int iters;
    bool expire = false;  // its first waits count as run out (ogsx_resident_fail)
};

template <typename T>
__device__ __forceinline__ T agent_load(const OGSX_GL T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(OGSX_GL T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A pointer that is the same for the whole wave, kept in scalar registers (a
// pointer read from a descriptor is not known to be, and each of a thread's
// gathers would hold a 64-bit address of its own).
template <typename T>
__device__ __forceinline__ OGSX_GL T* wave_uniform(OGSX_GL T* p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (OGSX_GL T*)(((unsigned long long)hi << 32) | lo);
}
// The wave's loads have returned and its stores have reached the memory that
// other workgroups read.
__device__ __forceinline__ void wait_memory() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Empties the exchange buffers and the phase.
__global__ __launch_bounds__(kBlock) void k_res_clear(ResSync* rs, size_t count)
{
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < count;
         i += (size_t)gridDim.x * kBlock)
        rs->slot[i] = kSlotEmpty;
    if (blockIdx.x == 0 && threadIdx.x == 0) rs->phase = 0;
}

// After a wait that ran out: empties the exchange buffers, whose slots and
// phase the workgroups no longer agree on, and stops the solve, so that no later
// launch goes on from its vectors.
__global__ __launch_bounds__(kBlock) void k_res_stop(const SysDev* sys)
{
    const size_t count = res_slot_count(sys->G);
    for (size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x; i < count;
         i += (size_t)gridDim.x * kBlock)
        sys->rs->slot[i] = kSlotEmpty;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sys->rs->phase = 0;
        sys->st->done = 4;
        sys->st->pend = 0;
        sys->st->expired = 0;
        if (sys->irs) {
            sys->irs->status = 0;
            sys->irs->action = 0;
        }
    }
}

// Counts the launch's workgroups in; true when all of them are resident.  A
// workgroup that has nothing to do (its solve stopped earlier) only counts.
__device__ __forceinline__ bool res_census(const ResLaunch& L, bool idle, int* flag)
{
    // the workgroup has read the state before it counts: another may end the
    // batch, and write the state, once all have counted
    wait_memory();
    __syncthreads();
    if (threadIdx.x == 0) {
        OGSX_GL ResCensus* c = (OGSX_GL ResCensus*)(L.ring + L.entry);
        const unsigned before =
            __hip_atomic_fetch_add(&c->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int d = 0;
        auto decide = [&](int want) {
            int open = 0;
            const bool mine = __hip_atomic_compare_exchange_strong(
                &c->decision, &open, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                __HIP_MEMORY_SCOPE_AGENT);
            d = mine ? want : open;
        };
        if (before + 1 == (unsigned)L.wgs) {
            decide(1);
        } else if (!idle) {
            const long long t0 = wall_clock64();
            for (unsigned polls = 0; d == 0; polls++) {
                d = agent_load(&c->decision);
                if (d == 0 && (wall_clock64() - t0 > kCensusTicks || polls > kResPolls)) decide(2);
            }
        }
        if (blockIdx.x == 0) {  // an entry no launch uses now, for a later one
            OGSX_GL ResCensus* f =
                (OGSX_GL ResCensus*)(L.ring + (L.entry + kCensusRing / 2) % kCensusRing);
            agent_store(&f->arrived, 0u);
            agent_store(&f->decision, 0);
        }
        *flag = d == 1;
    }
    __syncthreads();
    return *flag != 0 && !idle;
}

// Exchange of NV dot products among the workgroups of one system (VB chunks
// of 256 threads each per workgroup, q chunks to a slot).
template <int VB, bool STREAM = false>
struct ResExchange {
    OGSX_GL unsigned long long* slot;
    int slots, q, w, set, nwg;
    double (*sw)[4 * VB];  // [kSlotVals] wave sums
    double (*sm)[4];       // [kSlotVals] sums of the waves that poll
    int* ok;

    __device__ __forceinline__ OGSX_GL unsigned long long* at(int s, int k, int copy) const
    {
        return slot + ((size_t)(s * kSlotVals + k) * kSlotCopies + copy) * slots;
    }

    // Waits for every workgroup of the system (an exchange of nothing):
    // vector entries published before it can be read after it.
    template <typename F>
    __device__ __forceinline__ bool barrier(F&& meanwhile)
    {
        const double none[1] = {0.0};
        double out[1];
        return sum<1, false>(none, out, meanwhile);
    }

    template <int NV>
    __device__ __forceinline__ bool sum(const double (&v)[NV], double (&out)[NV])
    {
        return sum<NV, true>(v, out, [] {});
    }

    // meanwhile(): loads to issue once this workgroup has posted its sums
    template <int NV, bool VALUES, typename F>
    __device__ __forceinline__ bool sum(const double (&v)[NV], double (&out)[NV], F&& meanwhile)
    {
        const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
        const int per = VB / q;  // slots this workgroup posts per value
        if constexpr (VALUES) {
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const double s = wave_sum(v[k]);
                if (lane == 0) sw[k][wave] = s;
            }
        }
        wait_memory();  // vector entries published before this exchange
        __syncthreads();
        const int copy = t % kSlotCopies, j = t / kSlotCopies % per, kk = t / kSlotCopies / per;
        if (kk < NV) {
            double s = 0.0;
            if constexpr (VALUES) {
                // (all of the sums read before the first is added)
                double c[VB][4];
#pragma unroll
                for (int i = 0; i < VB; i++)
#pragma unroll
                    for (int x = 0; x < 4; x++) c[i][x] = sw[kk][4 * min(j * q + i, VB - 1) + x];
#pragma unroll
                for (int i = 0; i < VB; i++)
                    if (i < q) s += ((c[i][0] + c[i][1]) + c[i][2]) + c[i][3];
            }
            unsigned long long bits = (unsigned long long)__double_as_longlong(s);
            if (bits == kSlotEmpty) bits = 0x7FF8000000000000ull;
            agent_store(at(set, kk, copy) + w * per + j, bits);
        }
        meanwhile();
        if (wave < 4) {
            // the others' sums arrive no sooner: polls before then only slow
            // the stores they wait for (200 x 200 quads FP64 4.40 -> 4.08 ms;
            // a pause twice as long, pauses between polls, or several polls
            // under way at once are slower again)
            __builtin_amdgcn_s_sleep(kFirstPoll);
            unsigned long long got[NV];
#pragma unroll
            for (int k = 0; k < NV; k++) got[k] = 0;
            if (t < nwg * per) {
                unsigned polls = 0, limit = kResPolls;
                if constexpr (STREAM) asm("" : "+s"(limit));
#pragma nounroll
                for (bool wait = true; wait;) {
                    wait = false;
#pragma unroll
                    for (int k = 0; k < NV; k++) got[k] = agent_load(at(set, k, w % kSlotCopies) + t);
#pragma unroll
                    for (int k = 0; k < NV; k++) wait = wait || got[k] == kSlotEmpty;
                    // (a constant the compiler sees in the thread-per-row kernels,
                    // one it does not in the streaming ones: it hoists more out
                    // of the loop with the first, 0.1 us per iteration faster in
                    // those and 0.7 us slower, by its spills, in these)
                    if (wait && ++polls > limit) {
                        *ok = 0;
                        break;
                    }
                }
            }
            if constexpr (VALUES) {
#pragma unroll
                for (int k = 0; k < NV; k++) {
                    const double s = wave_sum(__longlong_as_double((long long)got[k]));
                    if (lane == 0) sm[k][wave] = s;
                }
            }
        }
        __syncthreads();
        if constexpr (VALUES) {
#pragma unroll
            for (int k = 0; k < NV; k++) out[k] = ((sm[k][0] + sm[k][1]) + sm[k][2]) + sm[k][3];
        }
        // every workgroup has read the previous set: empty this one's slots
        // there (it is used again two exchanges on)
        const int prev = set == 0 ? kSlotSets - 1 : set - 1;
        if (t < kSlotVals * per * kSlotCopies)
            agent_store(at(prev, t / kSlotCopies / per, copy) + w * per + j, kSlotEmpty);
        set = set == kSlotSets - 1 ? 0 : set + 1;
        return *ok != 0;
    }
};

// A row's entries in the order of its sum, padded to NE with zeros: the CRS
// row, or the symmetric diagonal copy -- in CRS column order (FP64), or as
// spmv_symdia_k takes it (FP32, PAIR: the diagonal, then each offset's upper
// and lower entry).  col holds byte offsets into a T vector.
template <typename T, int NE, bool PAIR>
__device__ __forceinline__ void load_row(const SysDev& S, bool dia, int row, T (&a)[NE],
                                         unsigned (&col)[NE])
{
    constexpr int KM = (NE - 1) / 2;
    const int n = S.n;
#pragma unroll
    for (int e = 0; e < NE; e++) {
        a[e] = 0;
        col[e] = (unsigned)row * sizeof(T);
    }
    if (PAIR || dia) {
        const MatView<T>& M = mv_of<T>(S);
        const OGSX_GL T* dv = gl(M.dia_val);
        const OGSX_GL int* off = gl(M.dia_off);
        const int K = M.dia_k;
        a[PAIR ? 0 : KM] = dv[row];
#pragma unroll
        for (int k = 0; k < KM; k++) {
            if (k >= K) continue;
            const int o = off[k], up = min(row + o, n - 1), lo = max(row - o, 0);
            const OGSX_GL T* u = dv + (int64_t)(k + 1) * n;
            const int eu = PAIR ? 1 + 2 * k : KM + 1 + k, el = PAIR ? 2 + 2 * k : KM - 1 - k;
            a[eu] = u[row];
            col[eu] = (unsigned)up * sizeof(T);
            a[el] = row - o >= 0 ? u[lo] : (T)0;
            col[el] = (unsigned)lo * sizeof(T);
        }
    } else {
        const OGSX_GL int* ptr = gl(S.m64.ptr);
        const OGSX_GL int* cols = gl(S.m64.col);
        const OGSX_GL double* A = gl(S.A);
        const int k0 = ptr[row], k1 = ptr[row + 1];
#pragma unroll
        for (int e = 0; e < NE; e++)
            if (k0 + e < k1) {
                a[e] = (T)A[k0 + e];
                col[e] = (unsigned)cols[k0 + e] * sizeof(T);
            }
    }
}

template <typename T, int NE, bool PAIR>
__device__ __forceinline__ T row_sum(const T (&a)[NE], const T (&v)[NE])
{
    if constexpr (PAIR) {
        T s = a[0] * v[0];
#pragma unroll
        for (int e = 1; e < NE; e++) s = fma(a[e], v[e], s);
        return s;
    } else {
#pragma clang fp contract(off)
        T s = 0;
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const T prod = a[e] * v[e];
            s = s + prod;
        }
        return s;
    }
}

template <typename T>
__device__ __forceinline__ T at_byte(const OGSX_GL T* base, unsigned off)
{
    return *(const OGSX_GL T*)((const OGSX_GL char*)base + off);
}

// Row `row` of the FP64 matrix times the FP64 vector that the workgroups have
// published in x, as k_ir_residual sums it (the symmetric diagonal copy in CRS
// order, or the CRS row).
__device__ __forceinline__ double row_times_published(const SysDev& S, int row,
                                                      const OGSX_GL double* x)
{
#pragma clang fp contract(off)
    double s = 0.0;
    if (gl(S.prm)->dia) {
        const OGSX_GL double* dv = gl(S.m64.dia_val);
        const OGSX_GL int* off = gl(S.m64.dia_off);
        const int K = S.m64.dia_k, n = S.n;
#pragma unroll 4
        for (int k = K - 1; k >= 0; k--) {
            const int lo = max(row - off[k], 0);
            const double a = dv[(int64_t)(k + 1) * n + lo], xl = agent_load(x + lo);
            const double prod = (row >= off[k] ? a : 0.0) * xl;
            s = s + prod;
        }
        const double prod = dv[row] * agent_load(x + row);
        s = s + prod;
#pragma unroll 4
        for (int k = 0; k < K; k++) {
            const double a = dv[(int64_t)(k + 1) * n + row];
            const double prod = a * agent_load(x + min(row + off[k], n - 1));
            s = s + prod;
        }
    } else {
        const OGSX_GL int* cols = gl(S.m64.col);
        const OGSX_GL double* A = gl(S.A);
        const int k1 = gl(S.m64.ptr)[row + 1];
#pragma unroll 4
        for (int k = gl(S.m64.ptr)[row]; k < k1; k++) {
            const double prod = A[k] * agent_load(x + cols[k]);
            s = s + prod;
        }
    }
    return s;
}

// A batch of Jacobi-CG iterations (k_cg_spmv, k_cg_update, k_cg_direction)
// of the members of `g`, one row per thread.  What bounds it: the two
// exchanges, 1.4-2 us each, and one gather of z.
//
// FP32 (inside FP64 refinement with reliable updates): a recurrence that stops
// for an update or at its target goes through the refinement step right here
// (k_ir_fold, k_ir_residual, k_ir_decide, k_ir_prepare, k_cg_rescan,
// k_cg_resume, in their arithmetic) and runs on; only a finished solve or the
// batch's end leaves the launch.
template <typename T, int NE, bool PAIR, int VB>
__global__ __launch_bounds__(kBlock * VB) void k_cg_resident(Grp g, ResLaunch L)
{
    // gathers in flight: all of a row's, where the registers allow it
    constexpr int kBatch = NE * (int)sizeof(T) / 4 * 3 + NE + 28 <= 512 / VB ? NE : (NE + 1) / 2;
    __shared__ double sw[kSlotVals][4 * VB];
    __shared__ double sm[kSlotVals][4];
    __shared__ int flag, ok;
    const int si = g.blk2sys ? g.blk2sys[blockIdx.x] : 0;
    const int w = (int)blockIdx.x - (g.blk2sys ? g.blk0[si] : 0);
    const SysDev& S = g.sys[si];
    OGSX_GL KrylovState* st = gl(S.st);
    const bool idle = st->done != 0;
    const int G = S.G, n = S.n, tid = threadIdx.x;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    double tol = gl(S.prm)->tol, upd_thresh = gl(S.prm)->upd_thresh;
    constexpr bool IR = sizeof(T) == 4;
    const bool reliable = IR && gl(S.prm)->ir_reliable;
    int updates = 0, status = -1;
    double ir_error = 0.0, maxr = 0.0;
    double rr = st->rr;
    ResExchange<VB> ex{gl(S.rs->slot), res_slots(G), part_q(G), w, S.rs->phase, G / VB,
                       sw, sm, &ok};
    if (tid == 0) ok = !L.expire;
    if (!res_census(L, idle, &flag)) {
        if (!idle && w == 0 && tid == 0) st->resident = 1;
        return;
    }
    const GVec<T> v = gvec(kv_of<T>(S));
    // chunk c = w VB + tid / 256, its row tid % 256
    const int c = w * VB + tid / kBlock, ns = (n + 63) / 64;
    const int sb = (int)((int64_t)ns * c / G), se = (int)((int64_t)ns * (c + 1) / G);
    const int mine = sb * 64 + tid % kBlock;
    const bool have = mine < min(se * 64, n);
    const int row = have ? mine : n - 1;
    T a[NE], pj[NE];
    unsigned col[NE];
    load_row<T, NE, PAIR>(S, sizeof(T) == 8 && gl(S.prm)->dia, row, a, col);
    OGSX_GL T* z = wave_uniform(v.s);  // A p stays in registers: its vector carries z
#pragma unroll
    for (int e = 0; e < NE; e++) pj[e] = at_byte(v.p, col[e]);
    T x = v.x[row], r = v.r[row], p = v.p[row];
    const T d = v.d[row];
    double error = st->error, alpha_d = st->alpha, rr_old = st->rr_old;
    int it = it0, done = 0;
    bool good = true;
    for (int k = 0; k < L.iters; k++) {
        const T s = row_sum<T, NE, PAIR>(a, pj);
        double dot[1] = {have ? (double)p * (double)s : 0.0}, ps[1];
        good = ex.sum(dot, ps);
        if (!good) break;
        alpha_d = rr / ps[0];
        rr_old = rr;
        const T alpha = (T)alpha_d;
        x = x + alpha * p;
        r = r - alpha * s;
        T zi = r / d;
        bool limit = true;  // (k_cg_direction tests the limit, k_cg_resume does not)
        if (have) agent_store(z + row, zi);
        double two[2] = {have ? (double)r * (double)r : 0.0, have ? (double)zi * (double)r : 0.0};
        double res[2];
        good = ex.sum(two, res);
        if (!good) break;
        const double rnorm = sqrt(res[0]);
        error = rnorm / bnorm;
        it++;
        if (error < tol || rnorm < upd_thresh) {
            done = error < tol ? 1 : 5;
            if constexpr (!IR) break;
            if (!reliable) break;
            // x64 += unscale x32; r64 = b - A x64
            const OGSX_GL KrylovParams* P = gl(S.prm);
            OGSX_GL double* x64 = wave_uniform(gl(S.v64.x));
            const double bi = gl(S.v64.b)[row];
            if (have) agent_store(x64 + row, agent_load(x64 + row) + P->unscale * (double)x);
            good = ex.barrier([] {});
            if (!good) break;
            const double ri = bi - row_times_published(S, row, x64);
            double norms[1] = {have ? ri * ri : 0.0}, rs[1];
            good = ex.sum(norms, rs);
            if (!good) break;
            // the decision of k_ir_decide, in every workgroup
            const double rn = sqrt(rs[0]);
            updates++;
            ir_error = rn / gl(S.irs)->bnorm;
            if (ir_error < P->ir_tol) {
                status = 1;
                break;
            }
            if (it >= P->ir_max_iter) {
                status = 0;
                break;
            }
            maxr = rn * P->scale;
            upd_thresh = P->ir_delta * maxr;
            tol = P->ir_tol * gl(S.irs)->bnorm * P->scale * (rn / rn);
            // the recurrence resumes from the true residual
            done = 0;
            r = (T)(ri * P->scale);
            x = 0;
            zi = r / d;
            if (have) agent_store(z + row, zi);
            two[0] = have ? (double)r * (double)r : 0.0;
            two[1] = have ? (double)zi * (double)r : 0.0;
            good = ex.sum(two, res);
            if (!good) break;
            limit = false;
        }
        const T beta = (T)(res[1] / rr_old);
#pragma unroll
        for (int e0 = 0; e0 < NE; e0 += kBatch) {
            T zj[kBatch];
#pragma unroll
            for (int e = 0; e < kBatch && e0 + e < NE; e++) {
                // (opaque: keeps one 32-bit offset per entry in registers, not
                // the 64-bit address the compiler would compute before the loop)
                asm("" : "+v"(col[e0 + e]));
                zj[e] = agent_load((const OGSX_GL T*)((const OGSX_GL char*)z + col[e0 + e]));
            }
#pragma unroll
            for (int e = 0; e < kBatch && e0 + e < NE; e++)
                pj[e0 + e] = zj[e] + beta * pj[e0 + e];
        }
        p = zi + beta * p;
        rr = res[1];
        if (limit && it >= max_iter) {
            done = 2;
            break;
        }
    }
    if (have) {
        v.x[row] = x;
        v.r[row] = r;
        v.p[row] = p;
    }
    // (by any workgroup: the others may have had their sums and gone on)
    if (!good && tid == 0) agent_store(&st->expired, 1);
    if (w == 0 && tid == 0) {
        st->error = error;
        st->rr = rr;
        st->rr_old = rr_old;
        st->alpha = alpha_d;
        st->iter = it;
        st->done = done;
        st->resident = 0;
        S.rs->phase = ex.set;
        if (IR && updates > 0) {
            OGSX_GL IRState* R = gl(S.irs);
            R->error = ir_error;
            R->total = it;
            R->updates = R->updates + updates;
            R->status = status;
            R->action = status < 0 ? 2 : 0;
            if (status < 0) {  // (a finished solve's last decision leaves these)
                R->maxr = maxr;
                gl(S.prm)->upd_thresh = upd_thresh;
                gl(S.prm)->tol = tol;
            }
        }
    }
}

// A batch of right-preconditioned Jacobi-BiCGStab iterations (k_bi_dir,
// k_bi_spmv_v, k_bi_s, k_bi_spmv_t, k_bi_update) of the members of `g`, one row
// per thread.  Three exchanges per iteration instead of five launches:
//   (r0, v), with v published;
//   (s, s), (t, t), (t, s) -- t is formed before the test on s, which discards
//     it where it stops the solve;
//   (r, r), (r0, r), with r published.
// A thread forms p and s of its columns itself, from the r and v it gathers
// and the p it keeps, so neither needs to be exchanged.  173 x 118 quads
// (FP64): 8 us per iteration, 24 with five launches; bound by the exchanges
// (5 us), then by the divisions of a row's columns (exact ones, twice).
//
// Five values per entry of a row are more registers than a thread of 512 has for
// 15 entries in FP64 or 27 in FP32: p and d of the columns are then in LDS.
template <typename T, int NE, int VB>
constexpr bool bi_lds()
{
    return VB == 2 && NE * sizeof(T) >= 108;
}

template <typename T, int NE, bool PAIR, int VB>
__global__ __launch_bounds__(kBlock * VB) void k_bi_resident(Grp g, ResLaunch L)
{
    constexpr bool kLds = bi_lds<T, NE, VB>();
    constexpr int NT = kBlock * VB, NR = kLds ? 1 : NE;
    extern __shared__ __align__(16) char stream_lds[];
    __shared__ double sw[kSlotVals][4 * VB];
    __shared__ double sm[kSlotVals][4];
    __shared__ int flag, ok;
    const int si = g.blk2sys ? g.blk2sys[blockIdx.x] : 0;
    const int w = (int)blockIdx.x - (g.blk2sys ? g.blk0[si] : 0);
    const SysDev& S = g.sys[si];
    OGSX_GL KrylovState* st = gl(S.st);
    const bool idle = st->done != 0 || st->pend != 0;
    const int G = S.G, n = S.n, tid = threadIdx.x;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    const double tol = gl(S.prm)->tol;
    double rho0 = st->rho0, rho1 = st->rho1, alpha_d = st->alpha, omega_d = st->omega;
    double error = st->error;
    ResExchange<VB> ex{gl(S.rs->slot), res_slots(G), part_q(G), w, S.rs->phase, G / VB,
                       sw, sm, &ok};
    if (tid == 0) ok = !L.expire;
    if (!res_census(L, idle, &flag)) {
        if (!idle && w == 0 && tid == 0) st->resident = 1;
        return;
    }
    const GVec<T> v = gvec(kv_of<T>(S));
    const int c = w * VB + tid / kBlock, ns = (n + 63) / 64;
    const int sb = (int)((int64_t)ns * c / G), se = (int)((int64_t)ns * (c + 1) / G);
    const int mine = sb * 64 + tid % kBlock;
    const bool have = mine < min(se * 64, n);
    const int row = have ? mine : n - 1;
    T a[NE], rj[NE], vj[NE], preg[NR], dreg[NR];
    T* const pl = (T*)stream_lds + tid;
    T* const dl = pl + NE * NT;
    const auto pj = [&](int e) -> T& {
        if constexpr (kLds) return pl[e * NT];
        else return preg[e];
    };
    const auto dj = [&](int e) -> T& {
        if constexpr (kLds) return dl[e * NT];
        else return dreg[e];
    };
    unsigned col[NE];
    load_row<T, NE, PAIR>(S, sizeof(T) == 8 && gl(S.prm)->dia, row, a, col);
    OGSX_GL T* const rg = wave_uniform(v.r);
    OGSX_GL T* const vg = wave_uniform(v.v);
#pragma unroll
    for (int e = 0; e < NE; e++) {
        pj(e) = at_byte(v.p, col[e]);
        rj[e] = at_byte(rg, col[e]);
        vj[e] = at_byte(vg, col[e]);
        dj(e) = at_byte(v.d, col[e]);
    }
    auto gather = [&](const OGSX_GL T* from, T (&to)[NE]) {
#pragma unroll
        for (int e = 0; e < NE; e++) {
            asm("" : "+v"(col[e]));  // (as in k_cg_resident)
            to[e] = agent_load((const OGSX_GL T*)((const OGSX_GL char*)from + col[e]));
        }
    };
    T x = v.x[row], r = rg[row], p = v.p[row], vi = vg[row];
    const T d = v.d[row], r0 = v.r0[row];
    int it = it0, done = 0, pend = 0;
    // the sums the next direction starts from
    double rr[2] = {have ? (double)r * (double)r : 0.0, have ? (double)r0 * (double)r : 0.0};
    double res[2];
    bool good = ex.sum(rr, res);
    for (int k = 0; good && k < L.iters; k++) {
        T beta = 0, omega = 0;
        if (it > 0) {
            const double err = sqrt(res[0]) / bnorm;
            if (err < tol || fabs(omega_d) < DBL_MIN || it >= max_iter) {
                error = err;
                done = err < tol ? 1 : fabs(omega_d) < DBL_MIN ? 3 : 2;
                break;
            }
        }
        if (fabs(res[1]) < DBL_MIN) {
            done = 6;
            break;
        }
        rho1 = res[1];
        if (it > 0) {
            beta = (T)((rho1 / rho0) * (alpha_d / omega_d));
            omega = (T)omega_d;
        }
        T h[NE];  // the preconditioned p, then s, of the row's columns
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const T pe = it == 0 ? rj[e] : bi_p(rj[e], beta, pj(e), omega, vj[e]);
            pj(e) = pe;
            h[e] = pe / dj(e);
        }
        p = it == 0 ? r : bi_p(r, beta, p, omega, vi);
        const T ph = p / d;
        vi = row_sum<T, NE, PAIR>(a, h);
        if (have) agent_store(vg + row, vi);
        it++;
        double one[1] = {have ? (double)r0 * (double)vi : 0.0}, rv[1];
        good = ex.sum(one, rv);
        if (!good) break;
        alpha_d = rho1 / rv[0];
        rho0 = rho1;
        const T alpha = (T)alpha_d;
        gather(vg, vj);
        const T s = r - alpha * vi;
        const T sh = s / d;
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const T sj = rj[e] - alpha * vj[e];
            h[e] = sj / dj(e);
        }
        const T t = row_sum<T, NE, PAIR>(a, h);
        double three[3] = {have ? (double)s * (double)s : 0.0, have ? (double)t * (double)t : 0.0,
                           have ? (double)t * (double)s : 0.0};
        double sums[3];
        good = ex.sum(three, sums);
        if (!good) break;
        const double err = sqrt(sums[0]) / bnorm;
        if (err < tol) {
            x = x + alpha * ph;
            error = err;
            pend = 1;
            break;
        }
        omega_d = (sums[1] > DBL_MIN) ? sums[2] / sums[1] : 1.0;
        omega = (T)omega_d;
        x = bi_x(x, alpha, ph, omega, sh);
        r = s - omega * t;
        if (have) agent_store(rg + row, r);
        rr[0] = have ? (double)r * (double)r : 0.0;
        rr[1] = have ? (double)r0 * (double)r : 0.0;
        good = ex.sum(rr, res);
        if (!good) break;
        gather(rg, rj);
    }
    if (have) {  // (r and v are up to date where they were published)
        v.x[row] = x;
        v.p[row] = p;
    }
    // (r, r) and (r0, r) of the last update, for a direction launched separately
    OGSX_GL double* part = gl(S.part);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double s = wave_sum(rr[k]);
        if ((tid & 63) == 0) sw[k][tid >> 6] = s;
    }
    __syncthreads();
    if (tid % kBlock == 0) {
        const int q = part_q(G), vb = tid / kBlock;
#pragma unroll
        for (int k = 0; k < 2; k++)
            part[k * part_stride(G) + kBlock * (c % q) + c / q] =
                ((sw[k][4 * vb] + sw[k][4 * vb + 1]) + sw[k][4 * vb + 2]) + sw[k][4 * vb + 3];
    }
    // (by any workgroup: the others may have had their sums and gone on)
    if (!good && tid == 0) agent_store(&st->expired, 1);
    if (w == 0 && tid == 0) {
        st->error = error;
        st->rho0 = rho0;
        st->rho1 = rho1;
        st->alpha = alpha_d;
        st->omega = omega_d;
        st->iter = it;
        st->pend = pend;
        st->done = done;
        st->resident = 0;
        S.rs->phase = ex.set;
    }
}

// ---- Systems of one workgroup -------------------------------------------------
// The smallest systems (FP64, up to 2048 rows) fit one workgroup of W waves:
// wave i takes the 64-row slices i, i + W, ..., up to ROWS of them, with their
// matrix entries in registers and every vector in LDS.  Nothing is exchanged
// through memory; a dot product costs one workgroup barrier (0.1 us instead of
// 1.4-2).  Instruction issue bounds these kernels, so the waves are few and the
// rows per thread several.  Chunks of these sizes have one row per thread, so a
// slice's sum is one wave's sum of store_partials, and the sums below add up in
// its order.
constexpr int kOneMaxSlices = 32;

struct OneSums {
    double (*ws)[kSlotVals][kOneMaxSlices];  // [2]: slice sums, by turns
    int turn, G, ns;

    template <int W, int NV, int ROWS>
    __device__ __forceinline__ void sum(const double (&v)[ROWS][NV], double (&out)[NV])
    {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (int j = 0; j < ROWS; j++)
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const double s = wave_sum(v[j][k]);
                if (lane == 0) ws[turn][k][wave + W * j] = s;
            }
        __syncthreads();
        // chunk `lane`: its slices' sums, then the sum over the chunks
        const int sb = lane < G ? ns * lane / G : 0, se = lane < G ? ns * (lane + 1) / G : 0;
#pragma unroll
        for (int k = 0; k < NV; k++) {
            double c[4];
#pragma unroll
            for (int i = 0; i < 4; i++) c[i] = ws[turn][k][min(sb + i, kOneMaxSlices - 1)];
            double s = sb < se ? c[0] : 0.0;
#pragma unroll
            for (int i = 1; i < 4; i++) s += sb + i < se ? c[i] : 0.0;
            const double t = wave_sum(s);
            const long long b = __double_as_longlong(t);
            const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
            const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
            out[k] = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
        }
        turn ^= 1;  // (a wave is at most one sum ahead of another)
    }
};

// A thread's rows: entries, and their columns' byte offsets into an LDS vector
// two to a register (up to 16 KB a vector).
template <int NE, int ROWS, int W>
struct OneRows {
    double a[ROWS][NE];
    unsigned col[ROWS][(NE + 1) / 2];

    __device__ __forceinline__ void load(const SysDev& S)
    {
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = (int)threadIdx.x + 64 * W * j;
            unsigned c[NE];
            load_row<double, NE, false>(S, gl(S.prm)->dia, min(row, S.n - 1), a[j], c);
#pragma unroll
            for (int e = 0; e < (NE + 1) / 2; e++)
                col[j][e] = c[2 * e] | (2 * e + 1 < NE ? c[2 * e + 1] << 16 : 0u);
        }
    }
    __device__ __forceinline__ double sum(int j, const double* x) const
    {
        double v[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const unsigned off = e & 1 ? col[j][e / 2] >> 16 : col[j][e / 2] & 0xffffu;
            v[e] = *(const double*)((const char*)x + off);
        }
        return row_sum<double, NE, false>(a[j], v);
    }
};

// Jacobi-CG of one-workgroup members (the recurrence of k_cg_resident).
template <int NE, int ROWS, int W>
__global__ __launch_bounds__(64 * W) void k_cg_one(Grp g, ResLaunch L)
{
    extern __shared__ __align__(16) char stream_lds[];
    __shared__ double ws[2][kSlotVals][kOneMaxSlices];
    const SysDev& S = g.sys[g.blk2sys ? g.blk2sys[blockIdx.x] : 0];
    OGSX_GL KrylovState* st = gl(S.st);
    if (st->done) return;
    const int n = S.n, tid = threadIdx.x;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    const double tol = gl(S.prm)->tol, upd_thresh = gl(S.prm)->upd_thresh;
    double rr = st->rr, error = st->error, alpha = st->alpha, rr_old = st->rr_old;
    OneSums sums{ws, 0, S.G, (n + 63) / 64};
    const GVec<double> v = gvec(S.v64);
    constexpr int N = 64 * W * ROWS;
    double* const pl = (double*)stream_lds;  // by row; the others by thread
    double* const xl = pl + N;
    double* const rl = xl + N;
    double* const dl = rl + N;
    OneRows<NE, ROWS, W> rows;
    rows.load(S);
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int row = tid + 64 * W * j;
        const bool have = row < n;
        pl[row] = have ? v.p[row] : 0.0;
        xl[row] = have ? v.x[row] : 0.0;
        rl[row] = have ? v.r[row] : 0.0;
        dl[row] = have ? v.d[row] : 1.0;
    }
    int it = it0, done = 0;
    for (int k = 0; k < L.iters; k++) {
        __syncthreads();  // p is written
        double s[ROWS], dot[ROWS][1], ps[1];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            s[j] = rows.sum(j, pl);
            dot[j][0] = row < n ? pl[row] * s[j] : 0.0;
        }
        sums.sum<W, 1, ROWS>(dot, ps);
        alpha = rr / ps[0];
        rr_old = rr;
        double z[ROWS], two[ROWS][2], res[2];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            xl[row] = xl[row] + alpha * pl[row];
            const double r = rl[row] - alpha * s[j];
            rl[row] = r;
            z[j] = r / dl[row];
            two[j][0] = row < n ? r * r : 0.0;
            two[j][1] = row < n ? z[j] * r : 0.0;
        }
        sums.sum<W, 2, ROWS>(two, res);
        const double rnorm = sqrt(res[0]);
        error = rnorm / bnorm;
        it++;
        if (error < tol || rnorm < upd_thresh) {
            done = error < tol ? 1 : 5;
            break;
        }
        const double beta = res[1] / rr_old;
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            pl[row] = z[j] + beta * pl[row];
        }
        rr = res[1];
        if (it >= max_iter) {
            done = 2;
            break;
        }
    }
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int row = tid + 64 * W * j;
        if (row < n) {
            v.x[row] = xl[row];
            v.r[row] = rl[row];
            v.p[row] = pl[row];
        }
    }
    if (tid == 0) {
        st->error = error;
        st->rr = rr;
        st->rr_old = rr_old;
        st->alpha = alpha;
        st->iter = it;
        st->done = done;
        st->resident = 0;
    }
}

// BiCGStab of one-workgroup members (the recurrence of k_bi_resident).
template <int NE, int ROWS, int W>
__global__ __launch_bounds__(64 * W) void k_bi_one(Grp g, ResLaunch L)
{
    extern __shared__ __align__(16) char stream_lds[];
    __shared__ double ws[2][kSlotVals][kOneMaxSlices];
    const SysDev& S = g.sys[g.blk2sys ? g.blk2sys[blockIdx.x] : 0];
    OGSX_GL KrylovState* st = gl(S.st);
    if (st->done != 0 || st->pend != 0) return;
    const int n = S.n, tid = threadIdx.x, G = S.G, ns = (n + 63) / 64;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    const double tol = gl(S.prm)->tol;
    double rho0 = st->rho0, rho1 = st->rho1, alpha = st->alpha, omega = st->omega;
    double error = st->error;
    OneSums sums{ws, 0, G, ns};
    const GVec<double> v = gvec(S.v64);
    constexpr int N = 64 * W * ROWS;
    double* const hl = (double*)stream_lds;  // preconditioned p, by row
    double* const tl = hl + N;               // preconditioned s, by row
    double* const xl = tl + N;               // the others by thread
    double* const rl = xl + N;
    double* const pl = rl + N;
    double* const vl = pl + N;
    double* const ol = vl + N;
    double* const dl = ol + N;
    OneRows<NE, ROWS, W> rows;
    rows.load(S);
    double rr[ROWS][2], res[2];
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int row = tid + 64 * W * j;
        const bool have = row < n;
        xl[row] = have ? v.x[row] : 0.0;
        rl[row] = have ? v.r[row] : 0.0;
        pl[row] = have ? v.p[row] : 0.0;
        vl[row] = have ? v.v[row] : 0.0;
        ol[row] = have ? v.r0[row] : 0.0;
        dl[row] = have ? v.d[row] : 1.0;
        rr[j][0] = rl[row] * rl[row];
        rr[j][1] = ol[row] * rl[row];
    }
    int it = it0, done = 0, pend = 0;
    sums.sum<W, 2, ROWS>(rr, res);
    for (int k = 0; k < L.iters; k++) {
        if (it > 0) {
            const double err = sqrt(res[0]) / bnorm;
            if (err < tol || fabs(omega) < DBL_MIN || it >= max_iter) {
                error = err;
                done = err < tol ? 1 : fabs(omega) < DBL_MIN ? 3 : 2;
                break;
            }
        }
        if (fabs(res[1]) < DBL_MIN) {
            done = 6;
            break;
        }
        rho1 = res[1];
        const double beta = it > 0 ? (rho1 / rho0) * (alpha / omega) : 0.0;
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            const double p = it == 0 ? rl[row] : bi_p(rl[row], beta, pl[row], omega, vl[row]);
            pl[row] = p;
            hl[row] = p / dl[row];
        }
        it++;
        __syncthreads();
        double one[ROWS][1], rv[1];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            const double vi = row < n ? rows.sum(j, hl) : 0.0;
            vl[row] = vi;
            one[j][0] = ol[row] * vi;
        }
        sums.sum<W, 1, ROWS>(one, rv);
        alpha = rho1 / rv[0];
        rho0 = rho1;
        double s[ROWS], t[ROWS], three[ROWS][3], out[3];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            s[j] = rl[row] - alpha * vl[row];
            tl[row] = s[j] / dl[row];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            t[j] = row < n ? rows.sum(j, tl) : 0.0;
            three[j][0] = s[j] * s[j];
            three[j][1] = t[j] * t[j];
            three[j][2] = t[j] * s[j];
        }
        sums.sum<W, 3, ROWS>(three, out);
        const double err = sqrt(out[0]) / bnorm;
        if (err < tol) {
#pragma unroll
            for (int j = 0; j < ROWS; j++) {
                const int row = tid + 64 * W * j;
                xl[row] = xl[row] + alpha * hl[row];
            }
            error = err;
            pend = 1;
            break;
        }
        omega = (out[1] > DBL_MIN) ? out[2] / out[1] : 1.0;
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int row = tid + 64 * W * j;
            xl[row] = bi_x(xl[row], alpha, hl[row], omega, tl[row]);
            const double r = s[j] - omega * t[j];
            rl[row] = r;
            rr[j][0] = row < n ? r * r : 0.0;
            rr[j][1] = row < n ? ol[row] * r : 0.0;
        }
        sums.sum<W, 2, ROWS>(rr, res);
    }
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int row = tid + 64 * W * j;
        if (row < n) {
            v.x[row] = xl[row];
            v.r[row] = rl[row];
            v.p[row] = pl[row];
            v.v[row] = vl[row];
        }
    }
    // (r, r) and (r0, r) of the last update, for a direction launched separately
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ROWS; j++)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const double w = wave_sum(rr[j][k]);
            if ((tid & 63) == 0) ws[0][k][(tid >> 6) + W * j] = w;
        }
    __syncthreads();
    if (tid < G) {
        const int sb = ns * tid / G, se = ns * (tid + 1) / G;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            double s = 0.0;
            for (int i = sb; i < se; i++) s = i == sb ? ws[0][k][i] : s + ws[0][k][i];
            gl(S.part)[k * part_stride(G) + tid] = s;  // (G is 8: q = 1)
        }
    }
    if (tid == 0) {
        st->error = error;
        st->rho0 = rho0;
        st->rho1 = rho1;
        st->alpha = alpha;
        st->omega = omega;
        st->iter = it;
        st->pend = pend;
        st->done = done;
        st->resident = 0;
    }
}

// The symmetric diagonal copy as k_cg_stream reads it: KC offsets and every
// array's base in scalar registers.
template <int KC, typename T>
struct DiaRows {
    const OGSX_GL T* dv;
    int off[KC];
    int n;

    __device__ __forceinline__ explicit DiaRows(const MatView<T>& m)
    {
        dv = wave_uniform(gl(const_cast<T*>(m.dia_val)));
        n = __builtin_amdgcn_readfirstlane(m.n);
#pragma unroll
        for (int k = 0; k < KC; k++) off[k] = __builtin_amdgcn_readfirstlane(gl(m.dia_off)[k]);
    }

    // The products' factors of entries e0 .. e1 of row r: matrix value and x.
    // Entries are in CRS column order: KC - 1 - k the lower entry of offset k,
    // KC the diagonal, KC + 1 + k the upper.  EDGE: the row may reach past the
    // first or last one (indices clamped, such a value taken as 0).
    template <bool EDGE, int E0, int E1, bool A = true, bool X = true>
    __device__ __forceinline__ void load(const OGSX_GL T* x, int r, T* a, T* xv) const
    {
        const unsigned sz = sizeof(T), at = (unsigned)r * sz;
#pragma unroll
        for (int e = E0; e < E1; e++) {
            const int k = e < KC ? KC - 1 - e : e > KC ? e - KC - 1 : 0;
            const int o = e < KC ? -off[k] : e > KC ? off[k] : 0;
            const unsigned dia = e == KC ? 0u : (unsigned)((k + 1) * n);  // its array
            if constexpr (EDGE) {
                const int j = min(max(r + o, 0), n - 1);
                if constexpr (A) a[e - E0] = at_byte(dv, sz * (dia + (unsigned)(e < KC ? j : r)));
                if constexpr (X) xv[e - E0] = at_byte(x, sz * (unsigned)j);
            } else {
                // 32-bit offsets from two bases: (KC + 1) n values are under 4 GB
                if constexpr (A) a[e - E0] = at_byte(dv, at + sz * (dia + (unsigned)(e < KC ? o : 0)));
                if constexpr (X) xv[e - E0] = at_byte(x, at + sz * (unsigned)o);
            }
        }
    }

    // The loads above are issued before anything below uses one (left alone,
    // the compiler takes the row two loads and one round trip at a time).
    static __device__ __forceinline__ void issued() { asm volatile("" ::: "memory"); }

    // Matrix values of the entries a row sum takes first (FP32 all of them).
    static constexpr int kFirst = sizeof(T) == 4 ? 2 * KC + 1 : KC;
    __device__ __forceinline__ bool inner(int r) const
    {
        // the wave's 64 rows are consecutive: one test for all of them
        const int lead = __builtin_amdgcn_readfirstlane(r);
        return lead - off[KC - 1] >= 0 && lead + 63 + off[KC - 1] < n;
    }
    __device__ __forceinline__ void prefetch(int r, T* a) const
    {
        if (inner(r))
            load<false, 0, kFirst, true, false>(nullptr, r, a, nullptr);
        else
            load<true, 0, kFirst, true, false>(nullptr, r, a, nullptr);
    }

    // Lower entries of a row that reaches past the first one are 0 (upper
    // ones past the last are stored so).
    template <bool EDGE>
    __device__ __forceinline__ void mask(int r, T* a) const
    {
        if constexpr (EDGE) {
#pragma unroll
            for (int e = 0; e < KC; e++) a[e] = r >= off[KC - 1 - e] ? a[e] : (T)0;
        }
    }

    // Row sum of row r in the order of spmv_symdia_k (FP32) or
    // spmv_symdia_crs_k (FP64).  FP32 takes the row's 2 x 27 loads at once,
    // FP64 (twice the registers) its lower and its upper half.
    // PRE: its first values are in `a` already.
    template <bool EDGE, bool PRE>
    __device__ __forceinline__ T sum(const OGSX_GL T* x, int r, T* a) const
    {
        constexpr int NE = 2 * KC + 1;
        if constexpr (sizeof(T) == 4) {
            T xv[NE];
            load<EDGE, 0, NE, !PRE>(x, r, a, xv);
            issued();
            mask<EDGE>(r, a);
            T s = a[KC] * xv[KC];
#pragma unroll
            for (int k = 0; k < KC; k++) {
                s = fma(a[KC + 1 + k], xv[KC + 1 + k], s);
                s = fma(a[KC - 1 - k], xv[KC - 1 - k], s);
            }
            return s;
        } else {
#pragma clang fp contract(off)
            T xv[KC], a2[KC + 1], xv2[KC + 1];
            load<EDGE, 0, KC, !PRE>(x, r, a, xv);
            issued();
            mask<EDGE>(r, a);
            T s = 0;
#pragma unroll
            for (int e = 0; e < KC; e++) {
                const T prod = a[e] * xv[e];
                s = s + prod;
            }
            load<EDGE, KC, NE>(x, r, a2, xv2);
            issued();
#pragma unroll
            for (int e = 0; e <= KC; e++) {
                const T prod = a2[e] * xv2[e];
                s = s + prod;
            }
            return s;
        }
    }

    // epi(row, sum) of the thread's rows r, r + 256, ... < end; pre holds the
    // first row's first values.
    template <typename Epi>
    __device__ __forceinline__ void rows(const OGSX_GL T* x, int r, int end, const T (&pre)[kFirst],
                                         Epi&& epi) const
    {
        if (r >= end) return;
        asm("" : "+v"(r));
        T a[kFirst];
#pragma unroll
        for (int e = 0; e < kFirst; e++) a[e] = pre[e];
        epi(r, inner(r) ? sum<false, true>(x, r, a) : sum<true, true>(x, r, a));
#pragma nounroll
        for (r += kBlock; r < end; r += kBlock) {
            asm("" : "+v"(r));  // opaque: no induction variable, hence register, per load
            T b[kFirst];
            epi(r, inner(r) ? sum<false, false>(x, r, b) : sum<true, false>(x, r, b));
        }
    }
};

// A batch of Jacobi-CG iterations of one system too large for a thread per
// row: 256 workgroups hold its vectors in LDS (a thread's rows are those of
// the separate launches, up to 9) and stream the symmetric diagonal copy of
// the matrix (KC offsets) from memory.  p is gathered through the caches: it is published into one of
// four vectors in turn, and once in four iterations one wave per workgroup
// invalidates its compute unit's and XCD's caches (0.25 us an iteration; every
// iteration 1.6 us, by every wave 28 us), so that no gather finds a line of
// that vector's previous use.  Three exchanges per iteration: (p, s), then
// (r, r) and (z, r), then the new p.
//
// Per iteration on 128^3 hexes (FP32): 39 us, 61 with three launches (the
// time is the matrix, 23 us, then the exchanges); on 85 x 64 x 53 (FP64) 19
// and 31 us (the latency of two rows of loads and of the exchanges).
//
// XL, PL: x and p in LDS too; without, x stays in memory (read and written
// by its row's thread alone) and a row's own p is read back from where it was
// published.  LDS sets which: 160 KB hold 9 rows per thread of four FP32
// vectors, or 4, 6 or 9 of four, three or two FP64 ones.
template <int KC, typename T, bool XL, bool PL>
__global__ __launch_bounds__(kBlock * kStreamVb) void k_cg_stream(Grp g, ResLaunch L)
{
    constexpr int VB = kStreamVb, NT = kBlock * VB;
    extern __shared__ __align__(16) char stream_lds[];
    __shared__ double sw[kSlotVals][4 * VB];
    __shared__ double sm[kSlotVals][4];
    __shared__ int flag, ok;
    const int si = g.blk2sys ? g.blk2sys[blockIdx.x] : 0;
    const int launched = (int)blockIdx.x - (g.blk2sys ? g.blk0[si] : 0);
    const SysDev& S = g.sys[si];
    OGSX_GL KrylovState* st = gl(S.st);
    const bool idle = st->done != 0;
    const int G = S.G, n = S.n, tid = threadIdx.x, nwg = G / VB;
    // workgroups are dealt to the XCDs in turn: each XCD gets neighbouring chunks
    const int w = nwg % kNumXcd ? launched
                                : (launched % kNumXcd) * (nwg / kNumXcd) + launched / kNumXcd;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    const double tol = gl(S.prm)->tol, upd_thresh = gl(S.prm)->upd_thresh;
    double rr = st->rr;
    ResExchange<VB, true> ex{gl(S.rs->slot), res_slots(G), part_q(G), w, S.rs->phase, nwg, sw, sm, &ok};
    if (tid == 0) ok = !L.expire;
    if (!res_census(L, idle, &flag)) {
        if (!idle && w == 0 && tid == 0) st->resident = 1;
        return;
    }
    const DiaRows<KC, T> m(mv_of<T>(S));
    const GVec<T> v = gvec(kv_of<T>(S));
    OGSX_GL T* const vd = wave_uniform(v.d);
    OGSX_GL T* const vx = wave_uniform(v.x);
    const int c = w * VB + tid / kBlock, ns = (n + 63) / 64;
    const int beg = (int)((int64_t)ns * c / G) * 64;
    const int end = min((int)((int64_t)ns * (c + 1) / G) * 64, n);
    const int first = beg + chunk_thread();
    // row first + 256 j lives at [1024 j + tid] of each vector in LDS
    const int stride = ((ns + G - 1) / G * 64 + kBlock - 1) / kBlock * NT;
    T* const rl = (T*)stream_lds + tid;
    T* const sl = rl + stride;
    T* const pl = sl + stride;
    T* const xl = pl + stride;
    auto at = [&](int row) { return (row - first) * VB; };
    for (int i = first; i < end; i += kBlock) {
        rl[at(i)] = v.r[i];
        if constexpr (PL) pl[at(i)] = v.p[i];
        if constexpr (XL) xl[at(i)] = v.x[i];
    }
    // (CG leaves these vectors unused)
    OGSX_GL T* const ring[4] = {wave_uniform(v.r0), wave_uniform(v.v), wave_uniform(v.t),
                                wave_uniform(v.ph)};
    const OGSX_GL T* src = wave_uniform(v.p);
    // the first row's first matrix values, loaded while the exchange before
    // their use waits; likewise the rows' diagonal entries
    T pre[DiaRows<KC, T>::kFirst];
    // (opaque row numbers: nothing of a row is computed ahead of the loop and
    // kept in registers)
    auto ahead = [&] {
        int i = min(first, end - 1);
        asm("" : "+v"(i));
        m.prefetch(i, pre);
    };
    T dj[kStreamSlots];
    auto diagonal = [&] {
        int i = first;
        asm("" : "+v"(i));
#pragma unroll
        for (int j = 0; j < kStreamSlots; j++) dj[j] = 1;
#pragma unroll
        for (int j = 0; j < kStreamSlots; j++)
            if (i + j * kBlock < end) dj[j] = at_byte(vd, (unsigned)(i + j * kBlock) * sizeof(T));
    };
    ahead();
    double error = st->error, alpha_d = st->alpha, rr_old = st->rr_old;
    int it = it0, done = 0;
    bool good = true;
    for (int k = 0; k < L.iters; k++) {
        double dot[1] = {0.0}, ps[1];
        m.rows(src, first, end, pre, [&](int row, T ax) {
            T pi;
            if constexpr (PL)
                pi = pl[at(row)];
            else
                pi = src[row];
            sl[at(row)] = ax;
            dot[0] = fma((double)pi, (double)ax, dot[0]);
        });
        good = ex.template sum<1, true>(dot, ps, diagonal);
        if (!good) break;
        alpha_d = rr / ps[0];
        rr_old = rr;
        const T alpha = (T)alpha_d;
        double two[2] = {0.0, 0.0}, res[2];
        int start = first;
        asm("" : "+v"(start));
#pragma unroll
        for (int j = 0; j < kStreamSlots; j++) {
            const int i = start + j * kBlock;
            if (i >= end) break;
            T pi;
            if constexpr (PL)
                pi = pl[at(i)];
            else
                pi = src[i];
            if constexpr (XL)
                xl[at(i)] = xl[at(i)] + alpha * pi;
            else
                vx[i] = vx[i] + alpha * pi;
            const T rn = rl[at(i)] - alpha * sl[at(i)];
            rl[at(i)] = rn;
            const T zi = rn / dj[j];
            sl[at(i)] = zi;  // A p is done with
            two[0] = fma((double)rn, (double)rn, two[0]);
            two[1] = fma((double)zi, (double)rn, two[1]);
        }
        good = ex.sum(two, res);
        if (!good) break;
        const double rnorm = sqrt(res[0]);
        error = rnorm / bnorm;
        it++;
        if (error < tol || rnorm < upd_thresh) {
            done = error < tol ? 1 : 5;
            break;
        }
        const T beta = (T)(res[1] / rr_old);
        OGSX_GL T* to = k & 2 ? (k & 1 ? ring[3] : ring[2]) : (k & 1 ? ring[1] : ring[0]);
        for (int i = first; i < end; i += kBlock) {
            T pi;
            if constexpr (PL)
                pi = pl[at(i)];
            else
                pi = src[i];
            pi = sl[at(i)] + beta * pi;
            if constexpr (PL) pl[at(i)] = pi;
            agent_store(to + i, pi);
        }
        src = to;
        rr = res[1];
        if (it >= max_iter) {
            done = 2;
            break;
        }
        good = ex.barrier(ahead);
        if (!good) break;
        if ((k & 3) == 0) {
            if (tid < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            __syncthreads();
        }
    }
    const GVec<T> out = gvec(kv_of<T>(S));
    for (int i = first; i < end; i += kBlock) {
        out.r[i] = rl[at(i)];
        if constexpr (PL)
            out.p[i] = pl[at(i)];
        else
            out.p[i] = agent_load(src + i);
        if constexpr (XL) out.x[i] = xl[at(i)];
    }
    // (by any workgroup: the others may have had their sums and gone on)
    if (!good && tid == 0) agent_store(&st->expired, 1);
    if (w == 0 && tid == 0) {
        st->error = error;
        st->rr = rr;
        st->rr_old = rr_old;
        st->alpha = alpha_d;
        st->iter = it;
        st->done = done;
        st->resident = 0;
        S.rs->phase = ex.set;
    }
}

// A SELL-64 matrix with a stencil dictionary as k_bi_stream reads it: the
// dictionary in LDS, a row's pattern kept by its thread.
template <typename T>
struct DictRows {
    const OGSX_GL T* val;
    const OGSX_GL int* ptr;
    const OGSX_GL int* width;
    const int* delta;

    // Row sum of the thread's row in slice `slice`, in CRS order, U entries at
    // a time: their loads are issued together, those past the row's width read
    // its last entry again and are not added (the width is the wave's).
    __device__ __forceinline__ T sum(const OGSX_GL T* x, int slice, int row, int pat, int n) const
    {
#pragma clang fp contract(off)
        constexpr int U = sizeof(T) == 4 ? 16 : 8;
        const int w = __builtin_amdgcn_readfirstlane(width[slice]);
        const int base = __builtin_amdgcn_readfirstlane(ptr[slice]);
        const int lane = (int)threadIdx.x & 63;
        T s = 0;
        for (int e0 = 0; e0 < w; e0 += U) {
            T a[U], xv[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int e = min(e0 + u, w - 1);
                a[u] = at_byte(val, (unsigned)(base + e * 64 + lane) * sizeof(T));
                xv[u] = at_byte(x, (unsigned)(min(row, n - 1) + delta[pat + e]) * sizeof(T));
            }
            asm volatile("" ::: "memory");
#pragma unroll
            for (int u = 0; u < U; u++)
                if (e0 + u < w) {
                    const T prod = a[u] * xv[u];
                    s = s + prod;
                }
        }
        return s;
    }
};

// BiCGStab of one system too large for a thread per row (the recurrence of
// k_bi_resident, the layout of k_cg_stream: vectors in LDS, up to ROWS rows per
// thread, the matrix streamed).  The preconditioned p and s are published into
// four vectors in turn and gathered through the caches, which are invalidated
// once in two iterations.  Five exchanges per iteration: the new p (a barrier),
// (r0, v), (s, s) with the new s, (t, t) and (t, s), (r, r) and (r0, r).
// The matrix read twice per iteration and the five exchanges bound it: the
// FP32 steps of 80x72x64 hexes cut into tets (385,000 rows, 15 entries) take
// 25 us per iteration, 37 us with a launch per phase; a time step of it 4.31 ->
// 2.56 ms.
template <typename T, int ROWS>
__global__ __launch_bounds__(kBlock * kStreamVb) void k_bi_stream(Grp g, ResLaunch L)
{
    constexpr int VB = kStreamVb, NT = kBlock * VB;
    extern __shared__ __align__(16) char stream_lds[];
    __shared__ double sw[kSlotVals][4 * VB];
    __shared__ double sm[kSlotVals][4];
    __shared__ int flag, ok;
    const int si = g.blk2sys ? g.blk2sys[blockIdx.x] : 0;
    const int launched = (int)blockIdx.x - (g.blk2sys ? g.blk0[si] : 0);
    const SysDev& S = g.sys[si];
    OGSX_GL KrylovState* st = gl(S.st);
    const bool idle = st->done != 0 || st->pend != 0;
    const int G = S.G, n = S.n, tid = threadIdx.x, nwg = G / VB;
    const int w = nwg % kNumXcd ? launched
                                : (launched % kNumXcd) * (nwg / kNumXcd) + launched / kNumXcd;
    const int it0 = st->iter, max_iter = st->max_iter;
    const double bnorm = st->bnorm;
    const double tol = gl(S.prm)->tol;
    double rho0 = st->rho0, rho1 = st->rho1, alpha_d = st->alpha, omega_d = st->omega;
    double error = st->error;
    ResExchange<VB, true> ex{gl(S.rs->slot), res_slots(G), part_q(G), w, S.rs->phase, nwg, sw, sm, &ok};
    if (tid == 0) ok = !L.expire;
    if (!res_census(L, idle, &flag)) {
        if (!idle && w == 0 && tid == 0) st->resident = 1;
        return;
    }
    const MatView<T>& M = mv_of<T>(S);
    const GVec<T> v = gvec(kv_of<T>(S));
    OGSX_GL T* const vd = wave_uniform(v.d);
    const int c = w * VB + tid / kBlock, ns = (n + 63) / 64;
    const int beg = (int)((int64_t)ns * c / G) * 64;
    const int end = min((int)((int64_t)ns * (c + 1) / G) * 64, n);
    const int first = beg + chunk_thread();
    // vector q of row first + 256 j at [(q ROWS + j) 1024 + tid]; then the
    // dictionary
    T* const rl = (T*)stream_lds + tid;  // r, and s
    T* const pl = rl + ROWS * NT;
    T* const vl = pl + ROWS * NT;
    T* const xl = vl + ROWS * NT;
    T* const ol = xl + ROWS * NT;        // r0
    T* const hl = ol + ROWS * NT;        // preconditioned p
    T* const kl = hl + ROWS * NT;        // preconditioned s
    T* const tl = kl + ROWS * NT;        // t
    int* const delta = (int*)((T*)stream_lds + 8 * ROWS * NT);
    for (int i = tid; i < M.pat_cnt * M.pat_w; i += NT) delta[i] = gl(M.pat_delta)[i];
    const DictRows<T> m{wave_uniform(gl(const_cast<T*>(M.sval))),
                        wave_uniform(gl(const_cast<int*>(M.sell_ptr))),
                        wave_uniform(gl(const_cast<int*>(M.sell_w))), delta};
    int pat[ROWS];
    T dj[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int i = first + j * kBlock;
        pat[j] = 0;
        dj[j] = 1;
        if (i < end) {
            pat[j] = (int)gl(M.sell_pid)[i] * M.pat_w;
            dj[j] = vd[i];
            rl[j * NT] = v.r[i];
            pl[j * NT] = v.p[i];
            vl[j * NT] = v.v[i];
            xl[j * NT] = v.x[i];
            ol[j * NT] = v.r0[i];
        }
    }
    OGSX_GL T* const ring[4] = {wave_uniform(v.ph), wave_uniform(v.sh), wave_uniform(v.s),
                                wave_uniform(v.t)};
    auto row_sums = [&](const OGSX_GL T* x, T* to) {
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            int i = first + j * kBlock;
            asm("" : "+v"(i));
            if (i < end) to[j * NT] = m.sum(x, __builtin_amdgcn_readfirstlane(i >> 6), i, pat[j], n);
        }
    };
    int it = it0, done = 0, pend = 0;
    double rr[2] = {0.0, 0.0}, res[2];
#pragma unroll
    for (int j = 0; j < ROWS; j++)
        if (first + j * kBlock < end) {
            const double r = (double)rl[j * NT];
            rr[0] = fma(r, r, rr[0]);
            rr[1] = fma((double)ol[j * NT], r, rr[1]);
        }
    bool good = ex.sum(rr, res);
    for (int k = 0; good && k < L.iters; k++) {
        if (it > 0) {
            const double err = sqrt(res[0]) / bnorm;
            if (err < tol || fabs(omega_d) < DBL_MIN || it >= max_iter) {
                error = err;
                done = err < tol ? 1 : fabs(omega_d) < DBL_MIN ? 3 : 2;
                break;
            }
        }
        if (fabs(res[1]) < DBL_MIN) {
            done = 6;
            break;
        }
        rho1 = res[1];
        T beta = 0, omega = 0;
        if (it > 0) {
            beta = (T)((rho1 / rho0) * (alpha_d / omega_d));
            omega = (T)omega_d;
        }
        OGSX_GL T* const hp = k & 1 ? ring[2] : ring[0];
        OGSX_GL T* const hs = k & 1 ? ring[3] : ring[1];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int i = first + j * kBlock;
            if (i < end) {
                const T p = it == 0 ? rl[j * NT]
                                    : bi_p(rl[j * NT], beta, pl[j * NT], omega, vl[j * NT]);
                pl[j * NT] = p;
                const T h = p / dj[j];
                hl[j * NT] = h;
                agent_store(hp + i, h);
            }
        }
        it++;
        good = ex.barrier([] {});
        if (!good) break;
        if ((k & 1) == 0) {
            if (tid < 64) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            __syncthreads();
        }
        row_sums(hp, vl);
        double one[1] = {0.0}, rv[1];
#pragma unroll
        for (int j = 0; j < ROWS; j++)
            if (first + j * kBlock < end) one[0] = fma((double)ol[j * NT], (double)vl[j * NT], one[0]);
        good = ex.sum(one, rv);
        if (!good) break;
        alpha_d = rho1 / rv[0];
        rho0 = rho1;
        const T alpha = (T)alpha_d;
        double ss[1] = {0.0}, norm[1];
#pragma unroll
        for (int j = 0; j < ROWS; j++) {
            const int i = first + j * kBlock;
            if (i < end) {
                const T s = rl[j * NT] - alpha * vl[j * NT];
                tl[j * NT] = s;  // (t's place until r has been tested and replaced)
                const T h = s / dj[j];
                kl[j * NT] = h;
                agent_store(hs + i, h);
                ss[0] = fma((double)s, (double)s, ss[0]);
            }
        }
        good = ex.sum(ss, norm);
        if (!good) break;
        const double err = sqrt(norm[0]) / bnorm;
        if (err < tol) {
#pragma unroll
            for (int j = 0; j < ROWS; j++)
                if (first + j * kBlock < end) xl[j * NT] = xl[j * NT] + alpha * hl[j * NT];
            error = err;
            pend = 1;
            break;
        }
#pragma unroll
        for (int j = 0; j < ROWS; j++) rl[j * NT] = tl[j * NT];  // s
        row_sums(hs, tl);
        double two[2] = {0.0, 0.0}, sums[2];
#pragma unroll
        for (int j = 0; j < ROWS; j++)
            if (first + j * kBlock < end) {
                const T t = tl[j * NT];
                two[0] = fma((double)t, (double)t, two[0]);
                two[1] = fma((double)t, (double)rl[j * NT], two[1]);
            }
        good = ex.sum(two, sums);
        if (!good) break;
        omega_d = (sums[0] > DBL_MIN) ? sums[1] / sums[0] : 1.0;
        omega = (T)omega_d;
        rr[0] = rr[1] = 0.0;
#pragma unroll
        for (int j = 0; j < ROWS; j++)
            if (first + j * kBlock < end) {
                xl[j * NT] = bi_x(xl[j * NT], alpha, hl[j * NT], omega, kl[j * NT]);
                const T r = rl[j * NT] - omega * tl[j * NT];
                rl[j * NT] = r;
                rr[0] = fma((double)r, (double)r, rr[0]);
                rr[1] = fma((double)ol[j * NT], (double)r, rr[1]);
            }
        good = ex.sum(rr, res);
    }
    const GVec<T> out = gvec(kv_of<T>(S));
#pragma unroll
    for (int j = 0; j < ROWS; j++) {
        const int i = first + j * kBlock;
        if (i < end) {
            out.x[i] = xl[j * NT];
            out.r[i] = rl[j * NT];
            out.p[i] = pl[j * NT];
            out.v[i] = vl[j * NT];
        }
    }
    // (r, r) and (r0, r) of the last update, for a direction launched separately
    OGSX_GL double* part = gl(S.part);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double s = wave_sum(rr[k]);
        if ((tid & 63) == 0) sw[k][tid >> 6] = s;
    }
    __syncthreads();
    if (tid % kBlock == 0) {
        const int q = part_q(G), vb = tid / kBlock;
#pragma unroll
        for (int k = 0; k < 2; k++)
            part[k * part_stride(G) + kBlock * (c % q) + c / q] =
                ((sw[k][4 * vb] + sw[k][4 * vb + 1]) + sw[k][4 * vb + 2]) + sw[k][4 * vb + 3];
    }
    // (by any workgroup: the others may have had their sums and gone on)
    if (!good && tid == 0) agent_store(&st->expired, 1);
    if (w == 0 && tid == 0) {
        st->error = error;
        st->rho0 = rho0;
        st->rho1 = rho1;
        st->alpha = alpha_d;
        st->omega = omega_d;
        st->iter = it;
        st->pend = pend;
        st->done = done;
        st->resident = 0;
        S.rs->phase = ex.set;
    }
}

// Bytes of LDS that one vector of k_cg_stream takes.
constexpr size_t stream_vec_bytes(int n, int G, size_t size)
{
    const int ns = (n + 63) / 64;
    return (size_t)(((ns + G - 1) / G * 64 + kBlock - 1) / kBlock) * kBlock * kStreamVb * size;
}
constexpr int kCuLds = 160 * 1024;             // LDS of a compute unit
constexpr size_t kStreamLds = kCuLds - 1024;  // ... less the exchange's

}  // namespace ogsx
