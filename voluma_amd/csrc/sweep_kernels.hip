// Triangular sweeps: the DIC/DILU preconditioner (factor, forward and backward
// substitution, LinearSolver.cpp:56-105), the Gauss–Seidel solver sweeps
// (LinearSolver.cpp:238-264) and the Gauss–Seidel GAMG smoother (GAMG.cpp:363-384).
//
// The reference runs these loops one cell (or one face) at a time. A cell's update reads
// the new values of its neighbours on one side (smaller indices forward, larger ones
// backward), so cells are grouped into levels: the forward level of a cell is one more
// than the largest forward level among its lower-numbered neighbours, and no two cells of
// one level are neighbours. A level's cells are updated at once, each with the same
// operands, in the same order, as in the sequential loop: the results are its bits.
//
// What bounds a sweep is the chain of levels (10²–10³ of 10¹–10⁴ cells), i.e. the time of
// one level's dependence: from a value to its neighbours' values. That is shortest through
// LDS, so a sweep keeps x there: the cells are cut into chunks of consecutive indices
// (SweepPlanHost), a workgroup takes a chunk and works through its rows in level order,
// 64 rows of a level (a step) per wavefront, the steps dealt to the wavefronts in turn.
// While one wavefront computes, the others load the entries and operands of their next
// steps, so their memory latency is hidden behind as many steps as there are wavefronts;
// a wavefront then waits for a count of finished steps in LDS, gathers from LDS, and adds
// to the count. No barrier, no launch and no memory round trip lies between two levels of
// a chunk. Between chunks the new values travel through memory and are their own flags:
// a published value replaces a sentinel, and a wavefront whose step needs it polls for it
// before its turn. Chunks are handed out by a ticket counter in sweep order, so a value
// is only ever waited for from a workgroup that has started (and waits itself only for
// earlier ones): whichever workgroups are resident, the earliest unfinished chunk
// proceeds. A wait past the plan's limit (sweepPolls) sets *fault and every later wait
// gives up at once.
//
// Measured (MI355X): handing a step over through LDS takes 0.14 µs and a value handed to
// another workgroup through memory 0.6 µs plus the polling; one CU streams rows at about
// 30 GB/s. Levels cost 0.4 µs in one chunk and about 0.9 µs across chunks, against 4–5 µs
// for a launch per level or a barrier per level in one workgroup. Two Gauss–Seidel sweeps,
// forward and backward: 373,920 tets (158 levels) 163 and 149 µs, 64³ hexes (190 levels)
// 150 and 141. What a step does after its turn counts fully, what a poll does between two
// looks counts where chunks wait for each other: with a division after the sum, a wait for
// the stores before the count, an add per LDS address, branches per entry in the polls and
// the first look at other chunks' values one round trip each, these took 205 and 185 µs
// (24,000 agglomerated cells of up to 20 entries 310, now 170). PCG with GAMG smoothed by
// Gauss–Seidel on these meshes: 228 → 53 and 66 → 18 ms; DIC-PCG on 24,273 hexes 34.6 → 7.6
// ms; three momentum components by PBiCGStab + DILU on 839,664 tets, assembly and factor
// included, 28.8 → 6.3 ms.
#include "device_common.hpp"
#include "vol_internal.hpp"

#include <atomic>

namespace vol {

namespace {
constexpr int SWEEP_THREADS = 256;
inline dim3 sweep_grid(size_t cnt) { return dim3(unsigned((cnt + SWEEP_THREADS - 1) / SWEEP_THREADS)); }
}  // namespace

// Row operations (T: double, or float in the mixed-precision inner solve):
//   SW_GS   Gauss–Seidel (LinearSolver.cpp:247-262, GAMG.cpp:368-379):
//           x_c = (b_c − Σ coef·x_nb) / diag_c, entries in ascending face order
//   SW_FWD  DILU forward substitution (LinearSolver.cpp:93-98):
//           w_u = rD_u·r_u − Σ (rD_u·A_ul)·w_l, entries in ascending (l, face) order
//   SW_BWD  DILU backward substitution (LinearSolver.cpp:99-103):
//           w_l = w_l − Σ (rD_l·A_lu)·w_u, entries in descending (u, face) order
//   SW_FAC  DIC/DILU factor (LinearSolver.cpp:67-74):
//           d_u = diag_u − Σ (A_lu·A_ul) / d_l, entries in ascending (l, face) order
// Except in GS the row's start value lies in its own slot of x when the sweep starts.
template <int OP, class T> __device__ __forceinline__ T row_term(T cf, T x) {
    if constexpr (OP == SW_FAC) return cf / x;
    else return cf * x;
}

// A value not published yet: a signalling NaN, which arithmetic does not produce (a value
// that is one, copied from the caller's data, is published as the quiet NaN).
template <class T> struct Sentinel;
template <> struct Sentinel<double> {
    static constexpr unsigned long long bits = 0x7FF4A5A5DEAD0001ull;
    __device__ static bool is(double v) { return (unsigned long long)__double_as_longlong(v) == bits; }
    __device__ static double value() { return __longlong_as_double((long long)bits); }
    __device__ static double quiet() { return __longlong_as_double((long long)(bits | (1ull << 51))); }
};
template <> struct Sentinel<float> {
    static constexpr unsigned bits = 0x7FA5DEADu;
    __device__ static bool is(float v) { return (unsigned)__float_as_uint(v) == bits; }
    __device__ static float value() { return __uint_as_float(bits); }
    __device__ static float quiet() { return __uint_as_float(bits | (1u << 22)); }
};

template <class T> __device__ __forceinline__ T peek(const T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T> __device__ __forceinline__ void publish_value(T* p, T v) {
    if (Sentinel<T>::is(v)) v = Sentinel<T>::quiet();
    // a read-modify-write is performed where every XCD sees it
    (void)__hip_atomic_exchange(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Whether a wait ends without its value after `spins` polls, looked at every 64: past its
// limit (sweepPolls; it reports that), or because another wait has.
__device__ __forceinline__ bool given_up(unsigned spins, unsigned limit, int* fault) {
    if ((spins & 63) != 63) return false;
    if (spins > limit) {
        __hip_atomic_fetch_or(fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return true;
    }
    return __hip_atomic_load(fault, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}
// Finished steps of the chunk.
__device__ __forceinline__ int finished(int* cnt) {
    return __hip_atomic_load(cnt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// One more, by one lane (the compiler would first add up over the wavefront's lanes).
__device__ __forceinline__ void count_step(int* cnt) {
    using Count = __attribute__((address_space(3))) int;
    asm volatile("ds_add_u32 %0, %1" ::"v"((Count*)cnt), "v"(1) : "memory");
}
// Steps before its turn that a wavefront starts to watch closely: 2, 4, 8 and 12 make two
// forward sweeps over 373,920 tets 255, 188, 163 and 159 µs.
constexpr int SWEEP_NEAR = 8;
// LDS-only ordering. A wavefront's LDS instructions are performed in the order in which it
// issues them, so its stores are there for whoever reads its later addition to the count:
// the compiler's order is all that a release needs (waiting for the stores would put one
// more LDS round trip into every dependence).
__device__ __forceinline__ void lds_release() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local"); }
__device__ __forceinline__ void lds_acquire() { __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local"); }

// A step's division a / d, the same bits as `/` in fewer dependent operations: everything
// that needs only d is done before the step's turn. With y = 1/d correctly rounded and e
// the next digits of 1/d, q = a·y + a·e is off by less than one unit in the last place, and
// then q + y·(a − d·q) with fused operations is the correctly rounded quotient (Markstein,
// Computation of elementary functions on the IBM RISC System/6000 processor, 1990), as long
// as nothing leaves the normal range: exponents past half of it take `/`.
template <class T> struct RowDivide {
    static constexpr T HI = sizeof(T) == 8 ? T(0x1p400) : T(0x1p48f), LO = sizeof(T) == 8 ? T(0x1p-400) : T(0x1p-48f);
    T d, y, e;
    bool plain;  // wave-uniform
    __device__ __forceinline__ static bool outside(T v) { return !(fabs(v) <= HI && fabs(v) >= LO); }
    __device__ __forceinline__ explicit RowDivide(T dg) : d(dg), y(T(1) / dg) {
        e = fma(-d, y, T(1)) * y;
        plain = __any(outside(d));
    }
    __device__ __forceinline__ T operator()(T a) const {
        const T z = a * y, q = fma(a, y, a * e);
        T x = a == T(0) ? z : fma(fma(-d, q, a), y, q);
        asm volatile("" : "+v"(x));  // computed beside the test, not after it
        if (__builtin_expect(plain || __any(a != T(0) && outside(a)), 0)) x = a / d;
        return x;
    }
};

// Steps s0 .. s1 of a chunk from cell c0, its slots of x in xs (pad: the padding slot, whose
// value has a term of 0), by a workgroup of WAVES wavefronts; *cnt counts finished steps
// from 0. Everything that does not depend on the step's turn is done before it: the row's
// first PF entries (later ones are loaded after the turn), their LDS addresses, the
// division by the diagonal but for its last four operations, and (MULTI) the terms of the
// values that come by mail. After the turn a step gathers from LDS, subtracts in order, stores
// and adds to the count; the code for that exists once per number of entry groups, so
// that every LDS read is in flight before the first is waited for. Lanes past the step's
// rows repeat its last row. MULTI: every value goes to the mailbox of this sweep.
template <int OP, bool MULTI, int PF, int WAVES, class T>
__device__ __forceinline__ void sweep_steps(const SweepPlan& P, const SweepArgs<T>& a, T* xs, int pad, int* cnt, int c0,
                                            int s0, int s1, int sweep) {
    constexpr int GRP = SWEEP_GROUP;
    static_assert(PF % GRP == 0 && PF <= 24);
    const int lane = threadIdx.x % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / WAVE);
    using Lds = __attribute__((address_space(3))) T;
    const unsigned lds = unsigned(uintptr_t((Lds*)xs));  // an LDS address is a 32-bit integer
    const auto value = [](unsigned addr) { return *(const Lds*)uintptr_t(addr); };
    // past the last step a wavefront loads the last one's data again (unused)
    const auto stepAt = [&](int s) { return P.steps[s < s1 ? s : s1 - 1]; };
    const auto rowOf = [&](const SweepStep& d) {
        const int rows = d.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1);
        return lane < rows ? lane : rows - 1;
    };
    // MULTI: an entry at < 0 is a value in the mailbox (from mail), or x before the sweep
    const T* const mail = MULTI ? a.mail + (sweep - 1) * ptrdiff_t(P.n) : nullptr;
    const auto mailed = [&](int at) { return unsigned(~at) < 2u * unsigned(P.n); };
    const auto initial = [&](int at) {
        const T x = a.zero ? T(0) : a.x[~at - 2 * P.n];
        return Sentinel<T>::is(x) ? Sentinel<T>::quiet() : x;
    };
    const int* const places = MULTI && sweep > 0 ? P.col2 : P.col;
    int s = s0 + wave;
    if (s >= s1) return;
    SweepStep d = stepAt(s), dn = stepAt(s + WAVES);
    int c = P.cell[d.pos + rowOf(d)];
    for (; s < s1; s += WAVES) {
        const int rows = __builtin_amdgcn_readfirstlane(d.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1));
        const int need = __builtin_amdgcn_readfirstlane(d.rowsNeed >> SWEEP_ROWS_BITS);
        const int width = __builtin_amdgcn_readfirstlane(d.width), base = __builtin_amdgcn_readfirstlane(d.base);
        const int pos = __builtin_amdgcn_readfirstlane(d.pos);
        const unsigned t = unsigned(lane < rows ? lane : rows - 1);
        const int* const ecol = places + base;  // uniform: the loads take 32-bit offsets
        const T* const ecoef = a.coef + base;
        T acc = T(0), dg = T(1);
        if constexpr (OP == SW_GS) {
            acc = a.b[unsigned(c)];
            dg = a.diag[unsigned(c)];
        }
        const int cn = P.cell[unsigned(dn.pos + rowOf(dn))];
        const SweepStep dnn = stepAt(s + 2 * WAVES);
        int at[PF];
        T cf[PF];
#pragma unroll
        for (int g = 0; g < PF; g += GRP) {
            if (g < width) {
#pragma unroll
                for (int k = g; k < g + GRP; ++k) at[k] = ecol[unsigned(k * rows) + t];
#pragma unroll
                for (int k = g; k < g + GRP; ++k) cf[k] = ecoef[unsigned(k * rows) + t];
            } else {
#pragma unroll
                for (int k = g; k < g + GRP; ++k) at[k] = 0;
            }
        }
        // as loaded, so that no use of them waits between one group's loads and the next
#pragma unroll
        for (int k = 0; k < PF; ++k) asm volatile("" : "+v"(at[k]));
        unsigned slot = lds + unsigned(c - c0) * unsigned(sizeof(T));
        if constexpr (OP != SW_GS) acc = value(slot);  // only this step writes it
        RowDivide<T> div(dg);
        unsigned addr[PF];
#pragma unroll
        for (int k = 0; k < PF; ++k) {
            addr[k] = lds + unsigned(MULTI && at[k] < 0 ? pad : at[k]) * unsigned(sizeof(T));
            asm volatile("" : "+v"(addr[k]));
        }
        // MULTI: the term of another chunk's value is put into add, and what is gathered for
        // it is a product of −0 (the padding's); a value in LDS has −0 there, which leaves
        // its product as it is: the term is the sum of both. Only one product per entry is
        // left to do when the values arrive.
        T add[MULTI ? PF : 1];
        if constexpr (MULTI) {
            int lowest = 0;
#pragma unroll
            for (int k = 0; k < PF; ++k) {
                lowest = min(lowest, at[k]);
                add[k] = -T(0);
            }
            if (__any(lowest < 0)) {
                T v[PF], own[PF];
                bool inf = false;
#pragma unroll
                for (int k = 0; k < PF; ++k) {
                    own[k] = at[k] < 0 ? -T(0) : cf[k];
                    v[k] = OP == SW_FAC ? T(1) : copysign(T(0), -cf[k]);  // cf·v = −0
                    if (OP != SW_FAC) inf = inf | __builtin_isinf(own[k]);
                    asm volatile("" : "+v"(own[k]), "+v"(v[k]));
                }
                const bool infinite = __any(inf);
                // all of them in one round trip; then, once the turn is near (asking
                // earlier only loads the fabric), the ones not yet published again,
                // together, until they are
#pragma unroll
                for (int k = 0; k < PF; ++k)
                    if (mailed(at[k])) v[k] = peek(&mail[~at[k]]);
                if (__any(lowest < 0 && !mailed(lowest))) {
#pragma unroll
                    for (int k = 0; k < PF; ++k)
                        if (at[k] < 0 && !mailed(at[k])) v[k] = initial(at[k]);
                }
                for (unsigned spins = 0;;) {
                    bool miss = false;
#pragma unroll
                    for (int k = 0; k < PF; ++k) miss = miss | Sentinel<T>::is(v[k]);
                    if (!__any(miss)) break;
                    if (need - finished(cnt) > SWEEP_NEAR) {
                        __builtin_amdgcn_s_sleep(2);
                        continue;
                    }
                    if (given_up(++spins, a.polls, a.fault)) break;
#pragma unroll
                    for (int k = 0; k < PF; ++k) {
                        asm volatile("" : "+v"(at[k]));  // no address kept over the loop
                        if (Sentinel<T>::is(v[k])) v[k] = peek(&mail[~at[k]]);
                    }
                }
#pragma unroll
                for (int k = 0; k < PF; ++k) {
                    const T f = OP != SW_FAC || at[k] < 0 ? cf[k] : -T(0);
                    add[k] = row_term<OP>(f, v[k]);
                    cf[k] = own[k];
                }
                if (infinite) {  // ∞·0 is no −0 (a select in every step would come after the values)
#pragma unroll
                    for (int k = 0; k < PF; ++k)
                        if (at[k] >= 0) add[k] = -T(0);
                }
            }
        }
        // keep all of the above before the turn
#pragma unroll
        for (int k = 0; k < PF; ++k) {
            asm volatile("" : "+v"(addr[k]), "+v"(cf[k]));
            if constexpr (MULTI) asm volatile("" : "+v"(add[k]));
        }
        asm volatile("" : "+v"(slot), "+v"(acc));
        if constexpr (OP == SW_GS) asm volatile("" : "+v"(div.y), "+v"(div.e));
        // the step's turn: every step of the chunk's earlier levels is done
        for (;;) {
            const int got = finished(cnt);
            if (got >= need) break;
            if (need - got > SWEEP_NEAR) __builtin_amdgcn_s_sleep(1);
        }
        lds_acquire();
        __builtin_amdgcn_s_setprio(3);  // ahead of the wavefronts that prepare later steps
        const auto rowSum = [&](auto groups) {
            constexpr int N = decltype(groups)::value * GRP;
            T xv[N];
#pragma unroll
            for (int k = 0; k < N; ++k) xv[k] = value(addr[k]);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                if constexpr (!MULTI) acc = acc - row_term<OP>(cf[k], xv[k]);
                else if constexpr (OP == SW_FAC) acc = acc - (row_term<OP>(cf[k], xv[k]) + add[k]);
                else acc = acc - fma(cf[k], xv[k], add[k]);
            }
        };
        const int ng = width / GRP;
        if (ng >= 6 && PF >= 24) rowSum(std::integral_constant<int, PF >= 24 ? 6 : 1>{});
        else if (ng >= 5 && PF >= 20) rowSum(std::integral_constant<int, PF >= 20 ? 5 : 1>{});
        else if (ng >= 4 && PF >= 16) rowSum(std::integral_constant<int, PF >= 16 ? 4 : 1>{});
        else if (ng >= 3 && PF >= 12) rowSum(std::integral_constant<int, PF >= 12 ? 3 : 1>{});
        else if (ng >= 2 && PF >= 8) rowSum(std::integral_constant<int, PF >= 8 ? 2 : 1>{});
        else if (ng >= 1) rowSum(std::integral_constant<int, 1>{});
        for (int k0 = PF; k0 < width; k0 += GRP) {
            int j[GRP];
            T f[GRP], xt[GRP];
#pragma unroll
            for (int q = 0; q < GRP; ++q) j[q] = ecol[unsigned((k0 + q) * rows) + t];
#pragma unroll
            for (int q = 0; q < GRP; ++q) f[q] = ecoef[unsigned((k0 + q) * rows) + t];
#pragma unroll
            for (int q = 0; q < GRP; ++q) {
                xt[q] = value(lds + unsigned(MULTI && j[q] < 0 ? 0 : j[q]) * unsigned(sizeof(T)));
                if (MULTI && j[q] < 0) {
                    xt[q] = mailed(j[q]) ? Sentinel<T>::value() : initial(j[q]);
                    for (unsigned spins = 0; Sentinel<T>::is(xt[q]) && !given_up(spins, a.polls, a.fault); ++spins)
                        xt[q] = peek(&mail[~j[q]]);
                }
            }
#pragma unroll
            for (int q = 0; q < GRP; ++q) acc = acc - row_term<OP>(f[q], xt[q]);
        }
        if constexpr (OP == SW_GS) acc = div(acc);
        *(Lds*)uintptr_t(slot) = acc;
        lds_release();
        if (lane == 0) count_step(cnt);
        __builtin_amdgcn_s_setprio(0);
        if constexpr (MULTI) {
            if (lane < rows) publish_value(&a.mail[sweep * ptrdiff_t(P.n) + pos + lane], acc);
        }
        c = cn;
        d = dn;
        dn = dnn;
    }
}

// The chunk's slots at the start of a sweep: start values or x before the sweep, the
// halo's x before the sweep, and the padding.
template <int OP, class T>
__device__ __forceinline__ void sweep_fill(const SweepPlan& P, const SweepArgs<T>& a, T* xs, int c0, int nc, int h0,
                                           int nh) {
    constexpr int SB = 8;  // loads in flight per thread
    for (int i0 = threadIdx.x; i0 < nc; i0 += SB * int(blockDim.x)) {
        T v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) {
            const int i = i0 + u * int(blockDim.x), q = c0 + (i < nc ? i : 0);
            if constexpr (OP == SW_GS || OP == SW_BWD) v[u] = a.zero ? T(0) : a.x[q];
            else if constexpr (OP == SW_FWD) v[u] = a.rD[q] * a.b[q];
            else v[u] = a.diag[q];
        }
#pragma unroll
        for (int u = 0; u < SB; ++u)
            if (i0 + u * int(blockDim.x) < nc) xs[i0 + u * int(blockDim.x)] = v[u];
    }
    for (int i0 = threadIdx.x; i0 < nh; i0 += SB * int(blockDim.x)) {
        int q[SB];
        T v[SB];
#pragma unroll
        for (int u = 0; u < SB; ++u) q[u] = P.halo[h0 + (i0 + u * int(blockDim.x) < nh ? i0 + u * int(blockDim.x) : 0)];
#pragma unroll
        for (int u = 0; u < SB; ++u) v[u] = a.zero ? T(0) : a.x[q[u]];
#pragma unroll
        for (int u = 0; u < SB; ++u)
            if (i0 + u * int(blockDim.x) < nh) xs[nc + i0 + u * int(blockDim.x)] = v[u];
    }
    if (threadIdx.x == 0) xs[nc + nh] = OP == SW_FAC ? T(1) : T(0);
}

// Sweeps over more than one chunk: one workgroup per chunk and sweep, by ticket, the
// chunks of the first sweep first: a chunk's next sweep runs while the first one is still
// under way further on. The last sweep writes x, in place: whatever reads a cell's x
// before the first sweep (its own chunk, or a halo) does so when its workgroup starts,
// and every value of a chunk's last sweep comes after the first-sweep values of its
// cells' neighbours, so after those workgroups' starts.
template <int OP, bool BACK, int PF, int WAVES, class T>
__global__ __launch_bounds__(WAVES* WAVE) void k_sweep_chunks(SweepPlan P, SweepArgs<T> a, int sweeps,
                                                              const int* done) {
    if (done && *done) return;
    extern __shared__ double sweepLds[];
    T* xs = reinterpret_cast<T*>(sweepLds);
    __shared__ int cnt, mine;
    if (threadIdx.x == 0) {
        cnt = 0;
        mine = __hip_atomic_fetch_add(a.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const int sweep = mine / P.nChunks;
    if (sweep >= sweeps) return;
    const int i = mine - sweep * P.nChunks, k = BACK ? P.nChunks - 1 - i : i;
    const int c0 = P.chunkOff[k], nc = P.chunkOff[k + 1] - c0;
    const int h0 = P.haloOff[k], nh = P.haloOff[k + 1] - h0;
    if (sweep == 0) sweep_fill<OP>(P, a, xs, c0, nc, h0, nh);
    else if (threadIdx.x == 0) xs[nc + nh] = T(0);  // the others are written before they are read
    __syncthreads();
    sweep_steps<OP, true, PF, WAVES, T>(P, a, xs, nc + nh, &cnt, c0, P.stepOff[k], P.stepOff[k + 1], sweep);
    if (sweep + 1 < sweeps) return;
    __syncthreads();
    for (int q = threadIdx.x; q < nc; q += blockDim.x) a.x[c0 + q] = xs[q];
}

// A sweep (or a schedule of several) over one chunk that holds every cell.
template <int OP, int PF, int WAVES, class T>
__global__ __launch_bounds__(WAVES* WAVE) void k_sweep_one(SweepPlan P, SweepArgs<T> a, const int* done) {
    if (done && *done) return;
    extern __shared__ double sweepLds[];
    T* xs = reinterpret_cast<T*>(sweepLds);
    __shared__ int cnt;
    if (threadIdx.x == 0) cnt = 0;
    sweep_fill<OP>(P, a, xs, 0, P.n, 0, 0);
    __syncthreads();
    sweep_steps<OP, false, PF, WAVES, T>(P, a, xs, P.n, &cnt, 0, 0, P.nSteps, 0);
    __syncthreads();
    for (int i = threadIdx.x; i < P.n; i += blockDim.x) a.x[i] = xs[i];
}

// Both DIC/DILU substitutions over one chunk, w staying in LDS between them.
template <int PF, int WAVES, class T>
__global__ __launch_bounds__(WAVES* WAVE) void k_dilu_one(SweepPlan F, SweepPlan B, SweepArgs<T> a, const T* eb,
                                                          const int* done) {
    if (done && *done) return;
    extern __shared__ double sweepLds[];
    T* xs = reinterpret_cast<T*>(sweepLds);
    __shared__ int cnt[2];
    if (threadIdx.x < 2) cnt[threadIdx.x] = 0;
    sweep_fill<SW_FWD>(F, a, xs, 0, F.n, 0, 0);
    __syncthreads();
    sweep_steps<SW_FWD, false, PF, WAVES, T>(F, a, xs, F.n, &cnt[0], 0, 0, F.nSteps, 0);
    __syncthreads();
    a.coef = eb;
    sweep_steps<SW_BWD, false, PF, WAVES, T>(B, a, xs, B.n, &cnt[1], 0, 0, B.nSteps, 0);
    __syncthreads();
    for (int i = threadIdx.x; i < F.n; i += blockDim.x) a.x[i] = xs[i];
}

// Mailbox values ← sentinel and tickets ← 0.
template <class T> __global__ void k_sweep_prepare(size_t m, T* mail, int* tickets, const int* done) {
    if (done && *done) return;
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < m) mail[i] = Sentinel<T>::value();
    if (i < SWEEP_TICKETS) tickets[i] = 0;
}

template <class T> void launch_sweep_prepare(hipStream_t st, size_t m, T* mail, int* tickets, const int* done) {
    hipLaunchKernelGGL(k_sweep_prepare<T>, sweep_grid(std::max<size_t>(m, SWEEP_TICKETS)), dim3(SWEEP_THREADS), 0, st,
                       m, mail, tickets, done);
}
template void launch_sweep_prepare<double>(hipStream_t, size_t, double*, int*, const int*);
template void launch_sweep_prepare<float>(hipStream_t, size_t, float*, int*, const int*);

// Launch with dynamic LDS beyond the default limit, which is raised once per device.
template <auto Kernel, class... A>
static hipError_t launch_lds(int blocks, int threads, size_t lds, hipStream_t st, A... args) {
    static std::atomic<unsigned long long> raised{0};  // a bit per device
    const void* const f = reinterpret_cast<const void*>(Kernel);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    if (!(raised.load(std::memory_order_relaxed) & bit)) {
        e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                int((SWEEP_MAX_SLOTS + 1) * sizeof(double)));
        if (e != hipSuccess) return e;
        raised.fetch_or(bit, std::memory_order_relaxed);
    }
    void* p[] = {&args...};
    return hipLaunchKernel(f, dim3(blocks), dim3(threads), p, lds, st);
}

// Rows of at most 8 entries (mesh cells) run 16 wavefronts; longer ones (coarse GAMG
// levels) 8, whose registers hold up to 24 entries each (20 with the values of other
// chunks beside them; entries past that cost a memory round trip inside the dependence:
// a level of 5,739 cells with up to 24 took 365 µs with 16 held and 220 with 20). The
// widest row decides for its whole level, and through sweepChunks' longRows for its chunks:
// a 64³ box with one cell of 18 faces takes 25.7 ms per PCG + Gauss–Seidel GAMG solve, the
// plain box 16.9.
template <int OP, bool BACK, class T>
static hipError_t launch_sweep_t(hipStream_t st, const SweepPlan& P, const SweepArgs<T>& a, int sweeps,
                                 const int* done) {
    const size_t lds = (size_t(P.maxSlots) + 1) * sizeof(T);
    const int blocks = P.nChunks * sweeps;
    if (P.nChunks > 1) {
        if (P.maxWidth <= 8)
            return launch_lds<k_sweep_chunks<OP, BACK, 8, 16, T>>(blocks, 16 * WAVE, lds, st, P, a, sweeps, done);
        if (P.maxWidth <= 12)
            return launch_lds<k_sweep_chunks<OP, BACK, 12, 8, T>>(blocks, 8 * WAVE, lds, st, P, a, sweeps, done);
        return launch_lds<k_sweep_chunks<OP, BACK, 20, 8, T>>(blocks, 8 * WAVE, lds, st, P, a, sweeps, done);
    }
    if (P.maxWidth <= 8) return launch_lds<k_sweep_one<OP, 8, 16, T>>(1, 16 * WAVE, lds, st, P, a, done);
    return launch_lds<k_sweep_one<OP, 24, 8, T>>(1, 8 * WAVE, lds, st, P, a, done);
}

template <class T>
hipError_t launch_sweep(hipStream_t st, int op, bool backward, const SweepPlan& P, const SweepArgs<T>& a, int sweeps,
                        const int* done) {
    if (P.n <= 0) return hipSuccess;
    switch (op) {
    case SW_GS:
        return backward ? launch_sweep_t<SW_GS, true, T>(st, P, a, sweeps, done)
                        : launch_sweep_t<SW_GS, false, T>(st, P, a, sweeps, done);
    case SW_FWD: return launch_sweep_t<SW_FWD, false, T>(st, P, a, sweeps, done);
    case SW_BWD: return launch_sweep_t<SW_BWD, true, T>(st, P, a, sweeps, done);
    default:
        if constexpr (std::is_same_v<T, double>) return launch_sweep_t<SW_FAC, false, T>(st, P, a, sweeps, done);
        return hipErrorInvalidValue;
    }
}
template hipError_t launch_sweep<double>(hipStream_t, int, bool, const SweepPlan&, const SweepArgs<double>&, int,
                                         const int*);
template hipError_t launch_sweep<float>(hipStream_t, int, bool, const SweepPlan&, const SweepArgs<float>&, int,
                                        const int*);

template <class T>
hipError_t launch_dilu_one(hipStream_t st, const SweepPlan& F, const SweepPlan& B, const SweepArgs<T>& a, const T* eb,
                           const int* done) {
    if (F.n <= 0) return hipSuccess;
    const size_t lds = (size_t(F.n) + 1) * sizeof(T);
    if (std::max(F.maxWidth, B.maxWidth) <= 8)
        return launch_lds<k_dilu_one<8, 16, T>>(1, 16 * WAVE, lds, st, F, B, a, eb, done);
    return launch_lds<k_dilu_one<24, 8, T>>(1, 8 * WAVE, lds, st, F, B, a, eb, done);
}
template hipError_t launch_dilu_one<double>(hipStream_t, const SweepPlan&, const SweepPlan&, const SweepArgs<double>&,
                                            const double*, const int*);
template hipError_t launch_dilu_one<float>(hipStream_t, const SweepPlan&, const SweepPlan&, const SweepArgs<float>&,
                                           const float*, const int*);

// Entries of the DIC/DILU factor and substitutions, a wavefront per step. src[e] is a
// face with its side of the row's own cell (f << 1 | side, 0: upper, 1: lower holds the
// row's coefficient). rD null: A_lu·A_ul (factor), else rD_row times the row's own.
__global__ void k_dilu_entries(SweepPlan P, const int* src, const double* upper, const double* lower, const double* rD,
                               double* out) {
    const int s = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE, lane = threadIdx.x % WAVE;
    if (s >= P.nSteps) return;
    const SweepStep d = P.steps[s];
    const int rows = d.rowsNeed & ((1 << SWEEP_ROWS_BITS) - 1);
    if (lane >= rows) return;
    const double r = rD ? rD[P.cell[d.pos + lane]] : 0.0;
    for (int k = 0; k < d.width; ++k) {
        const int e = d.base + k * rows + lane, q = src[e], f = q >> 1;
        double v = 0.0;
        if (q >= 0) {
            const double own = (q & 1) ? lower[f] : upper[f];
            v = rD ? r * own : ((q & 1) ? upper[f] : lower[f]) * own;
        }
        out[e] = v;
    }
}
void launch_dilu_entries(hipStream_t st, const SweepPlan& P, const int* src, const double* upper, const double* lower,
                         const double* rD, double* out) {
    if (P.nSteps > 0)
        hipLaunchKernelGGL(k_dilu_entries, sweep_grid(size_t(P.nSteps) * WAVE), dim3(SWEEP_THREADS), 0, st, P, src,
                           upper, lower, rD, out);
}

// Per-entry coefficients of a sweep plan from their source array: out[e] = from[src[e]]
// (0 for padding, src < 0).
template <class T>
__global__ void k_gather_entries(size_t n, const int* src, const T* from, T* out) {
    const size_t e = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e < n) {
        const int s = src[e];
        out[e] = s >= 0 ? from[s] : T(0);
    }
}
template <class T> void launch_gather_entries(hipStream_t st, size_t n, const int* src, const T* from, T* out) {
    if (n > 0)
        hipLaunchKernelGGL(k_gather_entries<T>, dim3(unsigned((n + SWEEP_THREADS - 1) / SWEEP_THREADS)),
                           dim3(SWEEP_THREADS), 0, st, n, src, from, out);
}
template void launch_gather_entries<double>(hipStream_t, size_t, const int*, const double*, double*);
template void launch_gather_entries<float>(hipStream_t, size_t, const int*, const float*, float*);

// Coarsest-level solve in the reference's order (GAMG.cpp:406-421): forward substitution
// (rows ascending, each subtracting in ascending k: done column by column by all lanes,
// which keeps every row's order), then backward substitution row by row from the last,
// each row subtracting in ascending k before its division. A row's sum starts with the
// value the previous row just produced, so the backward pass is one dependent chain,
// run by lane 0 with the factors in LDS when they fit (n ≤ 64).
template <class T>
__global__ __launch_bounds__(64) void k_coarse_solve_rows(int n, const double* lu, const T* r, T* x,
                                                          const int* done) {
    if (done && *done) return;
    extern __shared__ double sh[];  // g (n), then the factors (n·n) when n ≤ 64
    const bool small = n <= 64;
    double* gv = sh;
    double* f = sh + n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) gv[i] = double(r[i]);
    if (small) {  // 16 loads in flight per lane, then their stores
        constexpr int SB = 16;
        for (int i0 = threadIdx.x; i0 < n * n; i0 += SB * 64) {
            double v[SB];
#pragma unroll
            for (int u = 0; u < SB; ++u) v[u] = i0 + u * 64 < n * n ? lu[i0 + u * 64] : 0.0;
#pragma unroll
            for (int u = 0; u < SB; ++u)
                if (i0 + u * 64 < n * n) f[i0 + u * 64] = v[u];
        }
    }
    __syncthreads();
    const double* a = small ? f : lu;
    for (int k = 0; k < n; ++k) {
        const double gk = gv[k];
        for (int i = k + 1 + threadIdx.x; i < n; i += blockDim.x) gv[i] -= a[size_t(i) * n + k] * gk;
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        for (int i = n - 1; i >= 0; --i) {
            double acc = gv[i];
            const double* row = a + size_t(i) * n;
            for (int k = i + 1; k < n; ++k) acc -= row[k] * gv[k];
            gv[i] = acc / row[i];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) x[i] = T(gv[i]);
}

template <class T>
void launch_coarse_solve_rows(hipStream_t st, int n, const double* lu, const T* r, T* x, const int* done) {
    const size_t lds = sizeof(double) * (size_t(n) + (n <= 64 ? size_t(n) * n : 0));
    hipLaunchKernelGGL(k_coarse_solve_rows<T>, dim3(1), dim3(64), lds, st, n, lu, r, x, done);
}
template void launch_coarse_solve_rows<double>(hipStream_t, int, const double*, const double*, double*, const int*);
template void launch_coarse_solve_rows<float>(hipStream_t, int, const double*, const float*, float*, const int*);

// x = 0 and x[i] += xc[agg[i]] (GAMG.cpp:423,438) for the Gauss–Seidel V-cycle.
template <class T>
__global__ void k_fill_zero(int n, T* x, const int* done) {
    if (done && *done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = T(0);
}
template <class T>
__global__ void k_prolong(int n, const int* agg, const T* xc, T* x, const int* done) {
    if (done && *done) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + xc[agg[i]];
}

template <class T>
void launch_fill_zero(hipStream_t st, int n, T* x, const int* done) {
    if (n > 0) hipLaunchKernelGGL(k_fill_zero<T>, sweep_grid(n), dim3(SWEEP_THREADS), 0, st, n, x, done);
}
template void launch_fill_zero<double>(hipStream_t, int, double*, const int*);
template void launch_fill_zero<float>(hipStream_t, int, float*, const int*);

template <class T>
void launch_prolong(hipStream_t st, int n, const int* agg, const T* xc, T* x, const int* done) {
    if (n > 0) hipLaunchKernelGGL(k_prolong<T>, sweep_grid(n), dim3(SWEEP_THREADS), 0, st, n, agg, xc, x, done);
}
template void launch_prolong<double>(hipStream_t, int, const int*, const double*, double*, const int*);
template void launch_prolong<float>(hipStream_t, int, const int*, const float*, float*, const int*);

}  // namespace vol
