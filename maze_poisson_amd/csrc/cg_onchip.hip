// cg_onchip.hip -- a whole FP64 CG solve in one launch, its vectors on the chip.
//
// The sweeps of the single-reduction CG iteration (k_cg1_dir, k_cg1_update,
// grid_kernels.hip) move 64 B per point and iteration through the memory
// hierarchy and pay two kernel boundaries (32 us at 128^3, 14 us at 64^3 and
// 32^3), although x, r, p and A p of a 128^3 grid (67 MB) fit the chip's
// registers and LDS (128 + 40 MB).  9.7, 5.0 and 3.7 us here, of which the
// exchange of the sums takes 2.3.  Here one
// work-group per CU keeps its share of the grid for the whole solve: x, r and
// A p in registers, p (with its in-plane halo) and the halo's r in LDS.  Per
// iteration it exchanges one set of sums with all work-groups and the halo of
// A p with its neighbours.
//
// A work-group owns two neighbouring 256-point plane chunks of one slab -- two
// of the tiles that `march` (stencil.hpp) gives one work-group each -- and a
// thread owns one column of the slab.  The partial sums are formed per tile,
// added per pair and folded in the same order as k_cg1_dir does, so the two
// forms give the same bits, and either may run a solve.
//
// Exchange.  A work-group's sums go to its slot (a cache line of its own) as two
// 64-bit words each, 32 bits of the value beside the exchange's epoch, so a word
// is valid by itself and needs no flag or counter.  One wave per 64 slots folds
// them and publishes the group's sums the same way, and every work-group adds
// the groups' sums.  Measured on the exchange of one sum alone: 1.3 us between
// two work-groups, 2.3 us between 256 (3.1 us where every work-group reads all
// slots, 2.7 and 3.2 us with several slots to a line).  A p values that
// neighbours need are stored device-wide before (vmcnt(0), work-group barrier)
// the work-group's sums are; a work-group that sees a neighbour's epoch may
// read them, while the sums are on their way.  Values and words alternate between
// two buffers: the next but one exchange overwrites them, by when every work-group
// has published the next exchange and so has seen this one (exchange_set).
//
// Every wait ends: a poll that lasts longer than kWaitTicks marks the solve as
// abandoned (kPoison in ctl), which every other wait sees.  x is written only
// after all work-groups have met once more at the end (counted in the same
// word, so that all of them see the same outcome), hence an abandoned solve
// leaves x and the solver state as they were and the caller runs the sweeps.
#include <algorithm>

#include "stencil.hpp"

namespace maze {

namespace {

using u64 = unsigned long long;
constexpr unsigned int kPoison = 1u << 10;  // over the count of arrivals
constexpr long long kWaitTicks = 20000000;  // 0.2 s of the 100 MHz clock
constexpr size_t kLdsMax = 160 * 1024 - 1024;
constexpr int kThreads = 2 * kBlock;
constexpr int kMaxWg = 256;
constexpr int kMaxGroups = kMaxWg / kWave;
// Marks by every thread of a launch at once neither overflow nor look like arrivals.
static_assert(kPoison > kMaxWg && (u64)kPoison * kMaxWg * 1024 <= 0xffffffffull, "marks overflow");
constexpr int kVals = kCg1Sums + 1;  // the sums and max|r|
constexpr int kLine = 16;            // words per 128-byte line
constexpr int kHalo = 8;             // in-plane halo entries per thread, at most
constexpr int kSlot = kExchangeSets * kLine;  // words per work-group or group: a line per set
constexpr int kSumsAt = kSlot * kMaxWg;       // the groups' slots

struct OnchipArgs {
    GridDims d;
    int groups, nwg;  // work-groups per slab, all of them
    u64* words;       // a slot per work-group, per line a pair per value; at kSumsAt the
                      // same per group of 64 work-groups
    double *h0, *h1;  // A p values for the neighbours, by grid index, alternating
    unsigned int* ctl;
    unsigned int epoch;
};

__device__ __forceinline__ void put(u64* w, double v, unsigned int e) {
    const u64 b = __double_as_longlong(v), t = (u64)e << 32;
    __hip_atomic_store(w, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(w + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ u64 word(const u64* w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One look at a wait that may have to be given up: false once the solve is
// abandoned, by this call if it has lasted kWaitTicks.
__device__ __forceinline__ bool keep_waiting(int spin, long long& t0, unsigned int* ctl) {
    if ((spin & 63) != 63) return true;
    if (__hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= kPoison) return false;
    const long long now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (now - t0 <= kWaitTicks) return true;
    __hip_atomic_fetch_add(ctl, kPoison, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return false;
}

// The meeting of all work-groups (one thread of each): true once all `n` have
// come, false if the solve was or is now abandoned.  All see the same outcome.
__device__ bool meet(unsigned int* ctl, unsigned int n) {
    __hip_atomic_fetch_add(ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    long long t0 = 0;
    for (;;) {
        const unsigned int v = __hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (v == n) return true;
        if (v >= kPoison) return false;
        const long long now = wall_clock64();
        if (t0 == 0) t0 = now;
        // Given up, unless another one arrived just now (the next look tells).
        unsigned int seen = v;
        if (now - t0 > kWaitTicks &&
            __hip_atomic_compare_exchange_strong(ctl, &seen, v + kPoison, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return false;
    }
}

// The values at C word pairs, `stride` words apart, once all carry the epoch.
// false: abandoned.
template <int C>
__device__ __forceinline__ bool poll(const u64* w, int stride, unsigned int e, unsigned int* ctl,
                                     double (&v)[C]) {
    long long t0 = 0;
    for (int spin = 0;; spin++) {
        u64 a[C], b[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            a[c] = word(w + c * stride);
            b[c] = word(w + c * stride + 1);
        }
        unsigned int off = 0;  // (no short cuts: every load is waited for here)
#pragma unroll
        for (int c = 0; c < C; c++) {
            off |= ((unsigned int)(a[c] >> 32) ^ e) | ((unsigned int)(b[c] >> 32) ^ e);
            v[c] = __longlong_as_double((b[c] << 32) | (a[c] & 0xffffffffull));
        }
        if (off == 0) return true;
        if (!keep_waiting(spin, t0, ctl)) return false;
    }
}

// One value of the slots at, at + 8, ..., at + 56 (0 past the last slot).
__device__ __forceinline__ bool poll_slots(const u64* slots, int at, int cnt, unsigned int e,
                                           unsigned int* ctl, double (&v)[8]) {
    long long t0 = 0;
    for (int spin = 0;; spin++) {
        u64 a[8], b[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const u64* w = slots + kSlot * min(at + 8 * i, cnt - 1);
            a[i] = word(w);
            b[i] = word(w + 1);
        }
        unsigned int off = 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            off |= ((unsigned int)(a[i] >> 32) ^ e) | ((unsigned int)(b[i] >> 32) ^ e);
            v[i] = at + 8 * i < cnt ? __longlong_as_double((b[i] << 32) | (a[i] & 0xffffffffull))
                                    : 0.0;
        }
        if (off == 0) return true;
        if (!keep_waiting(spin, t0, ctl)) return false;
    }
}

// The values at the word offsets off[0 .. C) (0 where negative).
template <int C, int N>
__device__ __forceinline__ bool poll_at(const u64* base, const int (&off)[N], unsigned int e,
                                        unsigned int* ctl, double (&v)[N]) {
    long long t0 = 0;
    for (int spin = 0;; spin++) {
        u64 a[C], b[C];
#pragma unroll
        for (int c = 0; c < C; c++) {
            const u64* w = base + max(off[c], 0);
            a[c] = word(w);
            b[c] = word(w + 1);
        }
        unsigned int bad = 0;
#pragma unroll
        for (int c = 0; c < C; c++) {
            const unsigned int d = ((unsigned int)(a[c] >> 32) ^ e) | ((unsigned int)(b[c] >> 32) ^ e);
            bad |= off[c] < 0 ? 0u : d;
            v[c] = off[c] < 0 ? 0.0 : __longlong_as_double((b[c] << 32) | (a[c] & 0xffffffffull));
        }
        if (bad == 0) return true;
        if (!keep_waiting(spin, t0, ctl)) return false;
    }
}

// The value, opaque to the compiler: keeps it from forming every plane's
// addresses and masks ahead of the iteration loop, where they would be held in
// (and spill) the registers that the vectors need.
__device__ __forceinline__ int vopaque(int v) {
    __asm__ volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int sopaque(int v) {
    __asm__ volatile("" : "+s"(v));
    return v;
}

// SLAB: planes per work-group (d.slab <= SLAB).
template <bool PB, int SLAB>
__global__ __launch_bounds__(kThreads) void k_cg_onchip(OnchipArgs A, PBCoef pb, double* x,
                                                        const double* r, CGState* st) {
    extern __shared__ double lds[];
    __shared__ double shw[kVals][kThreads / kWave], sha[4];
    __shared__ double stops[2];  // what the decisions need of the state
    __shared__ int modes[3], bad, ended, result;
    // Written by earlier kernels only: this one's store follows the meeting at
    // its end.
    if (st->done) return;
    constexpr int nt = kThreads;
    const int n = A.d.n, n2 = A.d.n2, t = threadIdx.x;
    const int lane = t & (kWave - 1), wv = t / kWave;
    const int sl = blockIdx.x / A.groups, g0 = blockIdx.x - sl * A.groups;
    const int base = g0 * nt, cnt = min(nt, n2 - base);
    const int i0 = sl * A.d.slab, ni = min(n, i0 + A.d.slab) - i0;
    const int W = nt + 2 * n;  // window of one plane in LDS: n points before, n after the own
    double* const rh = lds + A.d.slab * W;  // r on the in-plane halo
    const bool act = t < cnt;
    const int pl = act ? base + t : base;
    const int idx = n + pl - base;
    const int k = pl % n;
    const int okm = k == 0 ? n - 1 : -1, okp = k == n - 1 ? 1 - n : 1;
    const int im = (i0 == 0 ? n - 1 : i0 - 1) * n2 + pl;
    const int ip = (i0 + ni == n ? 0 : i0 + ni) * n2 + pl;
    // Points within n of the own range's ends, and the first and last plane,
    // are neighbours of other work-groups' points.
    const bool edge = t < n || t >= cnt - n;
    const int J = (A.nwg + kWave - 1) / kWave;
    // The in-plane halo: 2 n values per plane, at window offsets [0, n) and
    // [n + cnt, cnt + 2 n); the window is contiguous in the plane modulo n2.
    // A thread takes entries t, t + nt, ...: plane u, entry h of the plane.
    const int n2h = 2 * n, nh = n2h * ni, du = nt / n2h, dh = nt - du * n2h;
    const int u_t = t / n2h, h_t = t - u_t * n2h;
    auto halo_at = [&](int h, int& o, int& p) {
        o = h < n ? h : cnt + h;
        p = base - n + o;
        if (p < 0) p += n2;
        if (p >= n2) p -= n2;
    };
    auto next = [&](int& u, int& h) {
        u += du;
        h += dh;
        if (h >= n2h) {
            h -= n2h;
            u++;
        }
    };
    const double cr = st->plain ? -1.0 : 1.0 / 6.0;
    int iter = 0;
    unsigned int e = A.epoch;
    if (t == 0) {
        bad = ended = 0;
        stops[0] = st->tol;
        stops[1] = st->rtol * st->r0;
        modes[0] = st->limit;
        modes[1] = st->count_mode;
        modes[2] = st->plain;
    }

    double X[SLAB], R[SLAB], Q[SLAB], P[SLAB];
#pragma unroll
    for (int u = 0; u < SLAB; u++) {
        const int c = (i0 + min(u, ni - 1)) * n2 + pl;
        X[u] = x[c];
        R[u] = r[c];
    }
    double rim = r[im], rip = r[ip], pim = rim * cr, pip = rip * cr;
#pragma unroll
    for (int u = 0; u < SLAB; u++) {
        P[u] = R[u] * cr;
        if (act && u < ni) lds[u * W + idx] = P[u];
        __asm__ volatile("" : "+v"(X[u]));  // arrived, as the halo values below
    }
#pragma unroll 1
    for (int q = t, u = u_t, h = h_t; q < nh; q += nt, next(u, h)) {
        int o, p;
        halo_at(h, o, p);
        const double v = r[(i0 + u) * n2 + p];
        rh[q] = v;
        lds[u * W + o] = v * cr;
    }
    __syncthreads();

    for (;;) {
        // A p of the own column; the iteration's sums.
        double s[kCg1Sums] = {0.0, 0.0, 0.0, 0.0}, m = 0.0;
        double* const hq = (e & 1) ? A.h1 : A.h0;
        if (act) {
            const int nu = sopaque(ni), w = sopaque(W);
            const double* L = lds + vopaque(idx);
            int b0 = sopaque(i0) * n2;
            double vm = pim;
            double exm = PB ? pb.ex[im] : 0.0;
#pragma unroll
            for (int u = 0; u < SLAB; u++, L += w, b0 += n2) {
                if (u < nu) {
                    const double vc = P[u];
                    const double vp = u + 1 < nu ? P[u + 1 < SLAB ? u + 1 : u] : pip;
                    const double vjm = L[-n], vjp = L[n], vkm = L[okm], vkp = L[okp];
                    double lap;
                    if (!PB) {
                        lap = vp + vm + vjp + vjm + vkp + vkm - vc * 6.0;
                    } else {
                        const int c = b0 + pl;
                        const int jm = pl - n < 0 ? pl - n + n2 : pl - n;
                        const double exc = pb.ex[c], eyc = pb.ey[c], ezc = pb.ez[c];
                        const double eym = pb.ey[b0 + jm], ezm = pb.ez[c + okm], k2c = pb.k2[c];
                        lap = vp * exc + vm * exm + vjp * eyc + vjm * eym + vkp * ezc +
                              vkm * ezm - vc * (exc + exm + eyc + eym + ezc + ezm + k2c);
                        exm = exc;
                    }
                    Q[u] = lap;
                    if (edge || u == 0 || u == nu - 1) store_partial(hq, b0 + pl, lap);
                    cg1_terms(vc, R[u], lap, s, m);
                    vm = vc;
                }
            }
        }
        e++;
        u64* const slots = A.words + exchange_set(e) * kLine;
        u64* const sums = slots + kSumsAt;
        // The tiles' sums and their pair's, published once the work-group's
        // A p values have arrived.
#pragma unroll
        for (int c = 0; c < kCg1Sums; c++) s[c] = wave_sum_dpp(s[c]);
        m = wave_max_dpp(m);
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < kCg1Sums; c++) shw[c][wv] = s[c];
            shw[kCg1Sums][wv] = m;
        }
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        bool ok = true;
        const int val = lane & 7, sub = lane / 8;  // a lane's value and place among 8 slots
        if (wv == 0) {
            if (lane < kVals)
                put(slots + kSlot * blockIdx.x + 2 * lane,
                    lane < kCg1Sums ? cg1_pair(shw[lane], shw[lane] + 4)
                                    : cg1_pair_max(shw[lane], shw[lane] + 4),
                    e);
        } else if (wv == 1) {
            // The work-groups that hold the halo: those of the planes before and
            // after, those that the window's two sides begin and end in.
            const int q = vopaque(lane);
            int p = q == 2 ? base - n : q == 3 ? base - 1 : q == 4 ? base + cnt : base + cnt + n - 1;
            if (p < 0) p += n2;
            if (p >= n2) p -= n2;
            const int s_ = q == 0 ? (sl == 0 ? A.d.slabs - 1 : sl - 1)
                                  : q == 1 ? (sl == A.d.slabs - 1 ? 0 : sl + 1) : sl;
            const int slot = s_ * A.groups + (q < 2 ? g0 : p / nt);
            if (q < 6) {
                double v[1];
                ok = poll<1>(slots + kSlot * slot, 0, e, A.ctl, v);
            }
        } else if (wv == 2) {
            // Group g of 64 slots is folded by work-group g.
#pragma unroll 1
            for (int g = blockIdx.x; g < J; g += A.nwg) {
                const int at = vopaque(g * kWave + sub);
                double v[8];
                ok = poll_slots(slots + 2 * (val < kVals ? val : 0), at, A.nwg, e, A.ctl, v);
                const double f = cg1_fold(v, val == kCg1Sums);
                if (sub == 0 && val < kVals) put(sums + kSlot * g + 2 * val, f, e);
            }
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) return;
        // The halo of A p.
        const double qim = load_partial(hq, im), qip = load_partial(hq, ip);
        constexpr int HB = SLAB < kHalo ? SLAB : kHalo;
        double qh[HB];  // held until alpha is known
        {
            int u = vopaque(u_t), h = vopaque(h_t), q = vopaque(t);
#pragma unroll
            for (int c = 0; c < HB; c++, q += nt, next(u, h)) {
                int o, p;
                halo_at(h, o, p);
                qh[c] = load_partial(hq, q < nh ? (i0 + u) * n2 + p : im);
            }
        }
        if (wv == 0) {
            const int g = min(sub, J - 1);
            double v[1];
            ok = poll<1>(sums + kSlot * g + 2 * (val < kVals ? val : 0), 0, e, A.ctl, v);
            double S[kVals];
#pragma unroll
            for (int c = 0; c < kVals; c++) {
                S[c] = lane_value(v[0], c);
                for (int q = 1; q < J; q++) {
                    const double w = lane_value(v[0], 8 * q + c);
                    S[c] = c < kCg1Sums ? S[c] + w : fmax(S[c], w);
                }
            }
            Cg1 cg;
            int res = -1;
            const bool end = cg.decide(S, S[kCg1Sums], iter, modes[0], modes[1], modes[2],
                                       stops[0], stops[1], res);
            if (lane == 0) {
                ended = end ? 1 : 0;
                result = res;
                sha[0] = cg.alpha;
                sha[1] = cg.beta;
                sha[2] = cg.rr;
                sha[3] = cg.rmax;
            }
            if (!ok) bad = 1;
        }
        // The halo values have arrived before any branch: on a way to the loop's
        // head with loads still pending (the compiler joins the exits below with
        // it), the waits for them there would also be waits for the stencil's own
        // stores (3.4 times its time at 128^3).  The polls wait for all their
        // loads for the same reason.
        __asm__ volatile("" ::"v"(qim), "v"(qip));
#pragma unroll
        for (int c = 0; c < HB; c++) __asm__ volatile("" : "+v"(qh[c]));
        __syncthreads();
        if (bad) return;
        if (ended) break;
        // x += alpha p, r += alpha A p, p = beta p + cr r; the halo likewise.
        const double alpha = sha[0], beta = sha[1];
        iter++;
        if (act) {
            const int nu = sopaque(ni), w = sopaque(W);
            double* L = lds + vopaque(idx);
#pragma unroll
            for (int u = 0; u < SLAB; u++, L += w) {
                if (u < nu) {
                    const double v = P[u];
                    X[u] = X[u] + alpha * v;
                    R[u] = R[u] + alpha * Q[u];
                    P[u] = v * beta + cr * R[u];
                    L[0] = P[u];
                }
            }
        }
        rim = rim + alpha * qim;
        rip = rip + alpha * qip;
        pim = pim * beta + cr * rim;
        pip = pip * beta + cr * rip;
        // The loads of a batch go before its stores (the compiler cannot tell
        // them apart).
        constexpr int UB = HB < 4 ? HB : SLAB > 12 ? 2 : 4;
        int u = vopaque(u_t), h = vopaque(h_t), q = vopaque(t);
#pragma unroll
        for (int c0 = 0; c0 < HB; c0 += UB) {
            double rv[UB], pv[UB];
            int at[UB];
            const int qb = q;
#pragma unroll
            for (int c = 0; c < UB; c++, q += nt, next(u, h)) {
                int o, p;
                halo_at(h, o, p);
                at[c] = q < nh ? u * W + o : 0;
                rv[c] = rh[min(q, nh - 1)];
                pv[c] = lds[at[c]];
            }
#pragma unroll
            for (int c = 0; c < UB; c++) {
                if (qb + c * nt < nh) {
                    const double rn = rv[c] + alpha * qh[c0 + c];
                    rh[qb + c * nt] = rn;
                    lds[at[c]] = pv[c] * beta + cr * rn;
                }
            }
        }
        __syncthreads();
    }
    // All work-groups meet; then, and only then, x and the state are written.
    if (t == 0 && !meet(A.ctl, A.nwg)) bad = 1;
    __syncthreads();
    if (bad) return;
    if (act) {
        const int nu = sopaque(ni);
        int c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll
        for (int u = 0; u < SLAB; u++, c += n2)
            if (u < nu) x[c] = X[u];
    }
    if (blockIdx.x == 0 && t == 0) {
        st->rr = sha[2];
        st->rmax = sha[3];
        st->iter = iter;
        st->first = 0;
        st->res = result;
        st->done = 1;
    }
}

// ---- two reductions per iteration ------------------------------------------------
// The iteration of k_cg_dir and k_cg_update with their bits: <p, A p>, then the
// update and <r, r>, max|r|.  For FP64 modes above 128^3 (Sim::cg_two) and for the
// cold solves of the mixed precisions: their FP32 inner solves turn a last-bit
// difference of the start into 2.6e-9 of the forces after 200 steps at 4096 ions /
// 128^3, so a trajectory stays what it was.
// Two exchanges an iteration, of the sums of each tile of `march` (grid_dims_for)
// in the order of block_sum and reduce_partials_sum; the halo is that of r.
struct Onchip2Args {
    GridDims d;
    int T, groups, nwg;  // tiles per work-group, work-groups per slab, all of them
    u64* words;          // a slot per work-group, per line a pair per tile, then max|r|; at
                         // kSumsAt per group of 64 slots the sum and max
    double* h;           // r values for the neighbours, by grid index
    unsigned int* ctl;
    unsigned int epoch;
};
constexpr int kMaxTiles = 4;        // per work-group
constexpr int kFoldSlots = 1024;    // 4 per lane and group

// wave_sum's tree with DPP moves for the exchanges inside a row.
__device__ __forceinline__ double wave_sum_rows(double v) {
    v += __shfl_xor(v, 32);
    v += __shfl_xor(v, 16);
    v += dpp_move<kDppRor8>(v);
    v += dpp_move<kDppReverse4>(dpp_move<kDppHalfMirror>(v));
    v += dpp_move<kDppXor2>(v);
    v += dpp_move<kDppXor1>(v);
    return v;
}

template <bool PB, int SLAB, int NT>
__global__ __launch_bounds__(NT) void k_cg_onchip2(Onchip2Args A, PBCoef pb, double* x, const double* r,
                                                   CGState* st) {
    extern __shared__ double lds[];
    __shared__ double shw[2][NT / kWave], sha[4], stops[2];
    __shared__ int modes[3], bad, ended, result;
    if (st->done) return;
    const int n = A.d.n, n2 = A.d.n2, t = threadIdx.x, nt = blockDim.x;
    const int lane = t & (kWave - 1), wv = t / kWave;
    const int sl = blockIdx.x / A.groups, g0 = blockIdx.x - sl * A.groups;
    const int base = g0 * nt, cnt = min(nt, n2 - base);
    const int i0 = sl * A.d.slab, ni = min(n, i0 + A.d.slab) - i0;
    const int W = nt + 2 * n;
    const bool act = t < cnt;
    const int pl = act ? base + t : base;
    const int idx = n + pl - base;
    const int k = pl % n;
    const int okm = k == 0 ? n - 1 : -1, okp = k == n - 1 ? 1 - n : 1;
    const int im = (i0 == 0 ? n - 1 : i0 - 1) * n2 + pl;
    const int ip = (i0 + ni == n ? 0 : i0 + ni) * n2 + pl;
    const bool edge = t < n || t >= cnt - n;
    const int nb = A.d.blocks;
    // Tiles of this work-group (the last of a slab may hold fewer).
    const int tiles = min(A.T, A.d.chunks - g0 * A.T);
    const int n2h = 2 * n, nh = n2h * ni, du = nt / n2h, dh = nt - du * n2h;
    const int u_t = t / n2h, h_t = t - u_t * n2h;
    auto halo_at = [&](int h, int& o, int& p) {
        o = h < n ? h : cnt + h;
        p = base - n + o;
        if (p < 0) p += n2;
        if (p >= n2) p -= n2;
    };
    auto next = [&](int& u, int& h) {
        u += du;
        h += dh;
        if (h >= n2h) {
            h -= n2h;
            u++;
        }
    };
    const double cr = st->plain ? -1.0 : 1.0 / 6.0;
    double rdv = st->rdv;
    int iter = 0;
    unsigned int e = A.epoch;
    if (t == 0) {
        bad = ended = 0;
        stops[0] = st->tol;
        stops[1] = st->rtol * st->r0;
        modes[0] = st->limit;
        modes[1] = st->count_mode;
        modes[2] = st->plain;
    }

    double X[SLAB], R[SLAB], Q[SLAB];
#pragma unroll
    for (int u = 0; u < SLAB; u++) {
        const int c = (i0 + min(u, ni - 1)) * n2 + pl;
        X[u] = x[c];
        R[u] = r[c];
    }
    double pim = r[im] * cr, pip = r[ip] * cr;
#pragma unroll
    for (int u = 0; u < SLAB; u++) {
        if (act && u < ni) lds[u * W + idx] = R[u] * cr;
        __asm__ volatile("" : "+v"(X[u]));  // arrived, as the halo values below
    }
#pragma unroll 1
    for (int q = t, u = u_t, h = h_t; q < nh; q += nt, next(u, h)) {
        int o, p;
        halo_at(h, o, p);
        lds[u * W + o] = r[(i0 + u) * n2 + p] * cr;
    }
    __syncthreads();

    auto slots = [&]() { return A.words + exchange_set(e) * kLine; };
    // This work-group's tile sums (and max) to its line, as block_sum forms them.
    auto publish = [&](double s, double m, bool with_max) {
        s = wave_sum_rows(s);
        if (with_max) m = wave_max_dpp(m);
        if (lane == 0) {
            shw[0][wv] = s;
            shw[1][wv] = m;
        }
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (wv == 0 && lane < tiles) {
            double v = 0.0;
            for (int w = 0; w < kBlock / kWave; w++) v += shw[0][lane * (kBlock / kWave) + w];
            put(slots() + kSlot * blockIdx.x + 2 * lane, v, e);
        }
        if (with_max && wv == 0 && lane == kMaxTiles) {
            double v = 0.0;
            for (int w = 0; w < nt / kWave; w++) v = fmax(v, shw[1][w]);
            put(slots() + kSlot * blockIdx.x + 2 * kMaxTiles, v, e);
        }
    };
    // Lanes of group g hold the partials 64 g + lane + 256 u in the sweeps' order
    // of work-groups and add them over u, as reduce_partials_sum does; the groups
    // are its waves.  Wave 2 of work-group g (mod nwg).
    // The word offsets of a lane's partials and of one work-group's max (-1: none).
    auto offsets = [&](int g, int (&off)[kFoldSlots / kBlock + 1]) {
#pragma unroll
        for (int u = 0; u < kFoldSlots / kBlock; u++) {
            const int xs = g * kWave + lane + u * kBlock;
            const int tile = xcd_tile(min(xs, nb - 1), nb);
            const int ts = tile / A.d.chunks, ch = tile - ts * A.d.chunks, gg = ch / A.T;
            off[u] = xs < nb ? kSlot * (ts * A.groups + gg) + 2 * (ch - gg * A.T) : -1;
        }
        const int wg = g * kWave + lane;
        off[kFoldSlots / kBlock] = wg < A.nwg ? kSlot * wg + 2 * kMaxTiles : -1;
    };
    int mine[kFoldSlots / kBlock + 1];
    offsets(blockIdx.x, mine);
    auto fold_groups = [&](bool with_max) {
        bool ok = true;
        if (wv != 2) return ok;
#pragma unroll 1
        for (int g = blockIdx.x; g < kBlock / kWave; g += A.nwg) {
            if (g != (int)blockIdx.x) offsets(g, mine);
            double v[kFoldSlots / kBlock + 1];
            if (with_max) {
                ok = poll_at<kFoldSlots / kBlock + 1>(slots(), mine, e, A.ctl, v) && ok;
            } else {
                ok = poll_at<kFoldSlots / kBlock>(slots(), mine, e, A.ctl, v) && ok;
                v[kFoldSlots / kBlock] = 0.0;
            }
            double s = 0.0;
#pragma unroll
            for (int u = 0; u < kFoldSlots / kBlock; u++) s += v[u];
            s = wave_sum_rows(s);
            const double m = wave_max_dpp(v[kFoldSlots / kBlock]);
            if (lane == 0) put(slots() + kSumsAt + kSlot * g, s, e);
            if (with_max && lane == 1) put(slots() + kSumsAt + kSlot * g + 2, m, e);
        }
        if (A.nwg < kBlock / kWave) offsets(blockIdx.x, mine);
        return ok;
    };
    // The totals (wave 0): lane 8 g + c holds value c of group g.
    auto totals = [&](bool with_max, double& S, double& M) {
        const int g = min(lane / 8, kBlock / kWave - 1), c = with_max ? min(lane & 7, 1) : 0;
        double v[1];
        const bool ok = poll<1>(slots() + kSumsAt + kSlot * g + 2 * c, 0, e, A.ctl, v);
        S = M = 0.0;
#pragma unroll
        for (int q = 0; q < kBlock / kWave; q++) {
            S += lane_value(v[0], 8 * q);
            M = fmax(M, with_max ? lane_value(v[0], 8 * q + 1) : 0.0);
        }
        return ok;
    };

    for (;;) {
        // A p of the own column and <p, A p>.
        double s = 0.0;
        if (act) {
            const int nu = sopaque(ni), w = sopaque(W);
            const double* L = lds + vopaque(idx);
            int b0 = sopaque(i0) * n2;
            double vm = pim, vc = L[0];
            double exm = PB ? pb.ex[im] : 0.0;
#pragma unroll
            for (int u = 0; u < SLAB; u++, L += w, b0 += n2) {
                if (u < nu) {
                    const double vp = u + 1 < nu ? L[w] : pip;
                    const double vjm = L[-n], vjp = L[n], vkm = L[okm], vkp = L[okp];
                    double lap;
                    if (!PB) {
                        lap = vp + vm + vjp + vjm + vkp + vkm - vc * 6.0;
                    } else {
                        const int c = b0 + pl;
                        const int jm = pl - n < 0 ? pl - n + n2 : pl - n;
                        const double exc = pb.ex[c], eyc = pb.ey[c], ezc = pb.ez[c];
                        const double eym = pb.ey[b0 + jm], ezm = pb.ez[c + okm], k2c = pb.k2[c];
                        lap = vp * exc + vm * exm + vjp * eyc + vjm * eym + vkp * ezc +
                              vkm * ezm - vc * (exc + exm + eyc + eym + ezc + ezm + k2c);
                        exm = exc;
                    }
                    Q[u] = lap;
                    s += vc * lap;
                    vm = vc;
                    vc = vp;
                }
            }
        }
        e++;
        publish(s, 0.0, false);
        bool ok = fold_groups(false);
        if (wv == 0) {
            double S, M;
            ok = totals(false, S, M) && ok;
            const bool end = fabs(S) < 1e-300;  // breakdown guard, as BodyDir
            if (lane == 0) {
                sha[0] = end ? 0.0 : rdv / S;
                if (end) {
                    ended = 1;
                    result = iter;
                    sha[2] = sha[3] = 0.0;
                }
            }
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) return;
        if (ended) break;
        // x += alpha p, r += alpha A p, <r, r>, max|r|.
        const double alpha = sha[0];
        double m = 0.0;
        s = 0.0;
        if (act) {
            const int nu = sopaque(ni), w = sopaque(W);
            const double* L = lds + vopaque(idx);
            int c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll
            for (int u = 0; u < SLAB; u++, L += w, c += n2) {
                if (u < nu) {
                    X[u] = X[u] + alpha * L[0];
                    const double rn = R[u] + alpha * Q[u];
                    R[u] = rn;
                    s += rn * rn;
                    m = fmax(m, fabs(rn));
                    if (edge || u == 0 || u == nu - 1) store_partial(A.h, c, rn);
                }
            }
        }
        e++;
        publish(s, m, true);
        ok = true;
        if (wv == 1) {
            // The work-groups that hold the halo, as in k_cg_onchip.
            const int q = vopaque(lane);
            int p = q == 2 ? base - n : q == 3 ? base - 1 : q == 4 ? base + cnt : base + cnt + n - 1;
            if (p < 0) p += n2;
            if (p >= n2) p -= n2;
            const int s_ = q == 0 ? (sl == 0 ? A.d.slabs - 1 : sl - 1)
                                  : q == 1 ? (sl == A.d.slabs - 1 ? 0 : sl + 1) : sl;
            const int slot = s_ * A.groups + (q < 2 ? g0 : p / nt);
            if (q < 6) {
                double v[1];
                ok = poll<1>(slots() + kSlot * slot, 0, e, A.ctl, v);
            }
        }
        ok = fold_groups(true) && ok;
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) return;
        const double rim = load_partial(A.h, im), rip = load_partial(A.h, ip);
        constexpr int HB = SLAB < kHalo ? SLAB : kHalo;
        double rh[HB];
        {
            int u = vopaque(u_t), h = vopaque(h_t), q = vopaque(t);
#pragma unroll
            for (int c = 0; c < HB; c++, q += nt, next(u, h)) {
                int o, p;
                halo_at(h, o, p);
                rh[c] = load_partial(A.h, q < nh ? (i0 + u) * n2 + p : im);
            }
        }
        if (wv == 0) {
            // The decisions of BodyUpdate::finalize.
            double S, M, beta = 0.0;
            if (!totals(true, S, M)) bad = 1;
            const int limit = modes[0], count = modes[1];
            int end = 0, res = -1;
            if (M <= stops[count ? 1 : 0]) {
                end = 1;
                res = count ? iter + 1 : iter;
            } else {
                const double rn_dot_vn = modes[2] ? S : -S / 6.0;
                beta = rn_dot_vn / rdv;
                rdv = rn_dot_vn;
                if (iter + 1 >= limit) {
                    end = 1;
                    res = count ? limit : -1;
                }
            }
            if (lane == 0) {
                ended = end;
                result = res;
                sha[1] = beta;
                sha[2] = S;
                sha[3] = M;
            }
        }
        // Arrived before any branch (see k_cg_onchip).
        __asm__ volatile("" ::"v"(rim), "v"(rip));
#pragma unroll
        for (int c = 0; c < HB; c++) __asm__ volatile("" : "+v"(rh[c]));
        __syncthreads();
        if (bad) return;
        if (ended) break;
        iter++;
        // p = beta p + cr r on the own points and the halo.
        const double beta = sha[1];
        pim = pim * beta + cr * rim;
        pip = pip * beta + cr * rip;
        {
            const int nu = sopaque(ni), w = sopaque(W);
            double* L = lds + vopaque(idx);
            constexpr int UB = SLAB < 4 ? SLAB : 4;
#pragma unroll
            for (int u0 = 0; u0 < SLAB; u0 += UB, L += UB * w) {
                double v[UB];
#pragma unroll
                for (int u = 0; u < UB; u++) v[u] = L[u0 + u < nu ? u * w : 0];
#pragma unroll
                for (int u = 0; u < UB; u++)
                    if (act && u0 + u < nu) L[u * w] = v[u] * beta + cr * R[u0 + u];
            }
        }
        constexpr int UB = HB < 4 ? HB : 4;
        int u = vopaque(u_t), h = vopaque(h_t), q = vopaque(t);
#pragma unroll
        for (int c0 = 0; c0 < HB; c0 += UB) {
            double pv[UB];
            int at[UB];
            const int qb = q;
#pragma unroll
            for (int c = 0; c < UB; c++, q += nt, next(u, h)) {
                int o, p;
                halo_at(h, o, p);
                at[c] = q < nh ? u * W + o : 0;
                pv[c] = lds[at[c]];
            }
#pragma unroll
            for (int c = 0; c < UB; c++)
                if (qb + c * nt < nh) lds[at[c]] = pv[c] * beta + cr * rh[c0 + c];
        }
        __syncthreads();
    }

    if (t == 0 && !meet(A.ctl, A.nwg)) bad = 1;
    __syncthreads();
    if (bad) return;
    if (act) {
        const int nu = sopaque(ni);
        int c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll
        for (int u = 0; u < SLAB; u++, c += n2)
            if (u < nu) x[c] = X[u];
    }
    if (blockIdx.x == 0 && t == 0) {
        st->rr = sha[2];
        st->rmax = sha[3];
        st->iter = iter;
        st->first = 0;
        st->res = result;
        st->done = 1;
    }
}

// ---- larger grids: x and the halo stay in memory -----------------------------------
// The two-reduction solve of grids whose vectors do not fit whole: r and A p in
// registers, the own p in LDS without the halo in j and i, which is read from its
// owner's copy in memory after a third, neighbours-only exchange.  x streams through
// memory while the sums of the second exchange are on their way.  A work-group holds
// two tiles of one slab, of the last two slabs where the last is a short one.  The
// slabs are the sweeps' (the sums keep their order), so not every size fits 256 CUs:
// 130 to 135, 140, 141, 143 to 146, 160 and 161 do, the others run as sweeps.
//
// An iteration moves x (16 B per point), the edges of p (10 B) and the PB
// coefficients (32 B), where the sweeps move 64 and 128 B: at 160^3 27.6 against
// 73 us (Poisson) and 44.7 against 117 us (PB; 5.3 TB/s).  The vectors take 144
// of a thread's 256 registers; batches of more planes than 2 (PB) or 6 (Poisson),
// whose operands are requested together, spill or give nothing.  Updating x before the second exchange instead of during it costs
// 2.5 us, half the halo's points in k in registers instead of LDS 4 us (Poisson).
constexpr int kStreamPlanes = 36;
constexpr int kStreamStride = kThreads + 4;  // a plane in LDS: p, then the ends of cut rows

struct StreamArgs {
    GridDims d;
    int groups, slabs, nwg;  // work-groups per slab, slabs of work-groups, all of them
    u64* words;              // as Onchip2Args, per line: up to four tiles' sums, max|r|, p ready
    double* h;               // p on the edges, by grid index
    double* xs;              // x after the first update (x itself is written at the end)
    unsigned int* ctl;
    unsigned int epoch;
};
constexpr int kReadyWord = 2 * kMaxTiles + 2;

template <bool PB>
__global__ __launch_bounds__(kThreads) void k_cg_stream(StreamArgs A, PBCoef pb, double* x,
                                                        const double* r, CGState* st) {
    constexpr int SLAB = kStreamPlanes, nt = kThreads, LP = kStreamStride, NW = kThreads / kWave;
    extern __shared__ double lds[];
    __shared__ double shw[3][NW], sha[4], stops[2];
    __shared__ int modes[3], bad, ended, result;
    if (st->done) return;
    const int n = A.d.n, n2 = A.d.n2, t = threadIdx.x;
    const int lane = t & (kWave - 1), wv = t / kWave;
    const int sl = blockIdx.x / A.groups, g0 = blockIdx.x - sl * A.groups;
    const int base = g0 * nt, cnt = min(nt, n2 - base);
    const int i0 = sl * A.d.slab, i1 = sl == A.slabs - 1 ? n : i0 + A.d.slab, ni = i1 - i0;
    const int split = min(ni, A.d.slab);  // planes of the first of up to two slabs
    const bool act = t < cnt;
    const int pl = act ? base + t : base;
    const int idx = pl - base;
    const int k = pl % n;
    auto wrap = [n2](int q) { return q < 0 ? q + n2 : q >= n2 ? q - n2 : q; };
    // Neighbours in j outside the own range come from memory; those in k lie in the
    // rows the range cuts: its first row's point before the range (LDS entry nt) and
    // first point (nt + 1), its last row's point after the range and last point.
    const bool jl = idx < n, jh = idx >= cnt - n;
    const int jm = wrap(pl - n), jp = wrap(pl + n);
    const int km = pl + (k == 0 ? n - 1 : -1);
    const int first = base - base % n, last = base + cnt - 1 - (base + cnt - 1) % n + n - 1;
    int okm = k == 0 ? n - 1 : -1, okp = k == n - 1 ? 1 - n : 1;
    if (idx + okm < 0) okm = nt - idx;
    if (idx + okm >= cnt && k == 0) okm = nt + 3 - idx;
    if (idx + okp >= cnt) okp = nt + 2 - idx;
    if (idx + okp < 0) okp = nt + 1 - idx;
    const int im = (i0 == 0 ? n - 1 : i0 - 1) * n2 + pl;
    const int ip = (i1 == n ? 0 : i1) * n2 + pl;
    const bool edge = jl || jh;  // is a neighbour of other work-groups' points
    const int nb = A.d.blocks;
    const double cr = st->plain ? -1.0 : 1.0 / 6.0;
    double rdv = st->rdv;
    int iter = 0;
    unsigned int e = A.epoch;
    if (t == 0) {
        bad = ended = 0;
        stops[0] = st->tol;
        stops[1] = st->rtol * st->r0;
        modes[0] = st->limit;
        modes[1] = st->count_mode;
        modes[2] = st->plain;
    }

    const double* xin = x;
    double R[SLAB], Q[SLAB];
#pragma unroll
    for (int u = 0; u < SLAB; u++) {
        R[u] = r[(i0 + min(u, ni - 1)) * n2 + pl];
        if (act && u < ni) lds[u * LP + idx] = R[u] * cr;
    }

    // The words of an iteration's first and second exchange; those that tell that p is
    // ready are written once an iteration, with both exchanges between, and need one set.
    auto slots = [&](bool second) { return A.words + exchange_set(second ? 1 : 0) * kLine; };
    // Tile sums (of two slabs' parts) and max to this work-group's line.
    auto publish = [&](double s0, double s1, double m, bool with_max) {
        s0 = wave_sum_rows(s0);
        s1 = wave_sum_rows(s1);
        if (with_max) m = wave_max_dpp(m);
        if (lane == 0) {
            shw[0][wv] = s0;
            shw[1][wv] = s1;
            shw[2][wv] = m;
        }
        __syncthreads();
        if (wv == 0 && lane < kMaxTiles) {
            const double* w = &shw[lane >> 1][(lane & 1) * (kBlock / kWave)];
            double v = 0.0;
            for (int q = 0; q < kBlock / kWave; q++) v += w[q];
            put(slots(with_max) + kSlot * blockIdx.x + 2 * lane, v, e);
        }
        if (with_max && wv == 0 && lane == kMaxTiles) {
            double v = 0.0;
            for (int w = 0; w < NW; w++) v = fmax(v, shw[2][w]);
            put(slots(with_max) + kSlot * blockIdx.x + 2 * kMaxTiles, v, e);
        }
    };
    // As in k_cg_onchip2; tile (slab, chunk) is part 2 (slab past the last
    // work-group slab) + chunk & 1 of its work-group.
    auto offsets = [&](int g, int (&off)[kFoldSlots / kBlock + 1]) {
#pragma unroll
        for (int u = 0; u < kFoldSlots / kBlock; u++) {
            const int xs = g * kWave + lane + u * kBlock;
            const int tile = xcd_tile(min(xs, nb - 1), nb);
            const int ts = tile / A.d.chunks, ch = tile - ts * A.d.chunks;
            const int ws = min(ts, A.slabs - 1);
            off[u] = xs < nb ? kSlot * (ws * A.groups + ch / 2) + 2 * (2 * (ts - ws) + (ch & 1)) : -1;
        }
        const int wg = g * kWave + lane;
        off[kFoldSlots / kBlock] = wg < A.nwg ? kSlot * wg + 2 * kMaxTiles : -1;
    };
    int mine[kFoldSlots / kBlock + 1];
    offsets(blockIdx.x, mine);
    auto fold_groups = [&](bool with_max) {
        if (wv != 2 || blockIdx.x >= kBlock / kWave) return true;  // (nwg is over 4)
        double v[kFoldSlots / kBlock + 1];
        bool ok;
        if (with_max) {
            ok = poll_at<kFoldSlots / kBlock + 1>(slots(with_max), mine, e, A.ctl, v);
        } else {
            ok = poll_at<kFoldSlots / kBlock>(slots(with_max), mine, e, A.ctl, v);
            v[kFoldSlots / kBlock] = 0.0;
        }
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < kFoldSlots / kBlock; u++) s += v[u];
        s = wave_sum_rows(s);
        const double m = wave_max_dpp(v[kFoldSlots / kBlock]);
        if (lane == 0) put(slots(with_max) + kSumsAt + kSlot * blockIdx.x, s, e);
        if (with_max && lane == 1) put(slots(with_max) + kSumsAt + kSlot * blockIdx.x + 2, m, e);
        return ok;
    };
    auto totals = [&](bool with_max, double& S, double& M) {
        const int g = min(lane / 8, kBlock / kWave - 1), c = with_max ? min(lane & 7, 1) : 0;
        double v[1];
        const bool ok = poll<1>(slots(with_max) + kSumsAt + kSlot * g + 2 * c, 0, e, A.ctl, v);
        S = M = 0.0;
#pragma unroll
        for (int q = 0; q < kBlock / kWave; q++) {
            S += lane_value(v[0], 8 * q);
            M = fmax(M, with_max ? lane_value(v[0], 8 * q + 1) : 0.0);
        }
        return ok;
    };
    // The edges of the new p to memory, and the neighbours' (wave 1 waits for the
    // six work-groups that hold the halo).
    auto share_p = [&]() {
        if (act) {
            const int nu = sopaque(ni);
            const double* L = lds + vopaque(idx);
            int c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll 4
            for (int u = 0; u < nu; u++, L += LP, c += n2)
                if (edge || u == 0 || u == nu - 1) store_partial(A.h, c, L[0]);
        }
        __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        bool ok = true;
        if (wv == 0 && lane == 0) put(A.words + kSlot * blockIdx.x + kReadyWord, 0.0, e);
        if (wv == 1) {
            const int q = vopaque(lane);
            const int p = wrap(q == 2 ? base - n : q == 3 ? base - 1 : q == 4 ? base + cnt
                                                                              : base + cnt + n - 1);
            const int s_ = q == 0 ? (sl == 0 ? A.slabs - 1 : sl - 1)
                                  : q == 1 ? (sl == A.slabs - 1 ? 0 : sl + 1) : sl;
            const int slot = s_ * A.groups + (q < 2 ? g0 : p / nt);
            if (q < 6) {
                double v[1];
                ok = poll<1>(A.words + kSlot * slot + kReadyWord, 0, e, A.ctl, v);
            }
        }
        // Waves 2 to 4: the ends of cut rows (nothing that is used where a row starts
        // or ends with the range).
        const int h = t - 2 * kWave, u = h >> 2;
        if (h >= 0 && u < ni) {
            const int q = h & 3, g = q < 2 ? max(g0 - 1, 0) : min(g0 + 1, A.groups - 1);
            const int p = q == 0 ? max(base - 1, 0) : q == 1 ? first : q == 2 ? min(base + cnt, n2 - 1)
                                                                              : last;
            double v[1];
            ok = poll<1>(A.words + kSlot * (sl * A.groups + g) + kReadyWord, 0, e, A.ctl, v);
            lds[u * LP + nt + q] = load_partial(A.h, (i0 + u) * n2 + p);
        }
        if (!ok) bad = 1;
        __syncthreads();
    };

    __syncthreads();
    e++;
    share_p();
    if (bad) return;
    for (;;) {
        // A p of the own column and <p, A p>, in batches of planes whose memory
        // operands are requested together.
        double s0 = 0.0, s1 = 0.0;
        {
            constexpr int UB = PB ? 2 : 6;
            const int nu = sopaque(ni);
            const double* L = lds + vopaque(idx);
            int b0 = sopaque(i0) * n2;
            double vm = load_partial(A.h, im), vc = L[0];
            const double vip = load_partial(A.h, ip);
            double exm = PB ? pb.ex[im] : 0.0;
#pragma unroll
            for (int u0 = 0; u0 < SLAB; u0 += UB) {
                double hjm[UB], hjp[UB];
                double cx[UB], cy[UB], cz[UB], my[UB], mz[UB], ck[UB];
                if (u0 < nu) {
#pragma unroll
                    for (int u = 0; u < UB; u++) {
                        const int b = b0 + min(u, nu - 1 - u0) * n2;
                        hjm[u] = hjp[u] = 0.0;
                        if (jl) hjm[u] = load_partial(A.h, b + jm);
                        if (jh) hjp[u] = load_partial(A.h, b + jp);
                        if (PB) {
                            cx[u] = pb.ex[b + pl];
                            cy[u] = pb.ey[b + pl];
                            cz[u] = pb.ez[b + pl];
                            my[u] = pb.ey[b + jm];
                            mz[u] = pb.ez[b + km];
                            ck[u] = pb.k2[b + pl];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < UB; u++) {
                        if (u0 + u < nu) {
                            const double vp = u0 + u + 1 < nu ? L[LP] : vip;
                            const double vjm = jl ? hjm[u] : L[jl ? 0 : -n];
                            const double vjp = jh ? hjp[u] : L[jh ? 0 : n];
                            const double vkm = L[okm], vkp = L[okp];
                            double lap;
                            if (!PB) {
                                lap = vp + vm + vjp + vjm + vkp + vkm - vc * 6.0;
                            } else {
                                lap = vp * cx[u] + vm * exm + vjp * cy[u] + vjm * my[u] +
                                      vkp * cz[u] + vkm * mz[u] -
                                      vc * (cx[u] + exm + cy[u] + my[u] + cz[u] + mz[u] + ck[u]);
                                exm = cx[u];
                            }
                            Q[u0 + u] = lap;
                            const double w = act ? vc * lap : 0.0;
                            if (u0 + u < split) s0 += w;
                            else s1 += w;
                            vm = vc;
                            vc = vp;
                        }
                        L += LP;
                    }
                }
                b0 += UB * n2;
            }
        }
        e++;
        publish(s0, s1, 0.0, false);
        // The first planes of x, while the sums are on their way.
        constexpr int XB = 12;
        double xv[XB];
        {
            const int nu = sopaque(ni), c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll
            for (int u = 0; u < XB; u++) xv[u] = xin[c + min(u, nu - 1) * n2];
        }
        bool ok = fold_groups(false);
        if (wv == 0) {
            double S, M;
            ok = totals(false, S, M) && ok;
            const bool end = fabs(S) < 1e-300;  // breakdown guard, as BodyDir
            if (lane == 0) {
                sha[0] = end ? 0.0 : rdv / S;
                if (end) {
                    ended = 1;
                    result = iter;
                    sha[2] = sha[3] = 0.0;
                }
            }
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) return;
        if (ended) break;
        // r += alpha A p, <r, r>, max|r|.
        const double alpha = sha[0];
        double m = 0.0;
        s0 = s1 = 0.0;
        {
            const int nu = sopaque(ni);
#pragma unroll
            for (int u = 0; u < SLAB; u++) {
                if (act && u < nu) {
                    const double rn = R[u] + alpha * Q[u];
                    R[u] = rn;
                    if (u < split) s0 += rn * rn;
                    else s1 += rn * rn;
                    m = fmax(m, fabs(rn));
                }
            }
        }
        e++;
        publish(s0, s1, m, true);
        ok = fold_groups(true);
        // x += alpha p, while the sums are on their way.
        {
            const int nu = sopaque(ni);
            const double* L = lds + vopaque(idx);
            int c = sopaque(i0) * n2 + vopaque(pl);
#pragma unroll
            for (int u0 = 0; u0 < SLAB; u0 += XB, c += XB * n2, L += XB * LP) {
                if (u0 < nu) {
                    if (u0 > 0) {
#pragma unroll
                        for (int u = 0; u < XB; u++) xv[u] = xin[c + min(u, nu - 1 - u0) * n2];
                    }
#pragma unroll
                    for (int u = 0; u < XB; u++)
                        if (act && u0 + u < nu) A.xs[c + u * n2] = xv[u] + alpha * L[u * LP];
                }
            }
        }
        xin = A.xs;
        if (wv == 0) {
            // The decisions of BodyUpdate::finalize.
            double S, M, beta = 0.0;
            ok = totals(true, S, M) && ok;
            const int limit = modes[0], count = modes[1];
            int end = 0, res = -1;
            if (M <= stops[count ? 1 : 0]) {
                end = 1;
                res = count ? iter + 1 : iter;
            } else {
                const double rn_dot_vn = modes[2] ? S : -S / 6.0;
                beta = rn_dot_vn / rdv;
                rdv = rn_dot_vn;
                if (iter + 1 >= limit) {
                    end = 1;
                    res = count ? limit : -1;
                }
            }
            if (lane == 0) {
                ended = end;
                result = res;
                sha[1] = beta;
                sha[2] = S;
                sha[3] = M;
            }
        }
        if (!ok) bad = 1;
        __syncthreads();
        if (bad) return;
        if (ended) break;
        iter++;
        const double beta = sha[1];
        {
            constexpr int UB = 4;
            const int nu = sopaque(ni);
            double* L = lds + vopaque(idx);
#pragma unroll
            for (int u0 = 0; u0 < SLAB; u0 += UB, L += UB * LP) {
                if (u0 < nu) {
                    double v[UB];
#pragma unroll
                    for (int u = 0; u < UB; u++) v[u] = L[min(u, nu - 1 - u0) * LP];
#pragma unroll
                    for (int u = 0; u < UB; u++)
                        if (act && u0 + u < nu) L[u * LP] = v[u] * beta + cr * R[u0 + u];
                }
            }
        }
        e++;
        share_p();
        if (bad) return;
    }

    if (t == 0 && !meet(A.ctl, A.nwg)) bad = 1;
    __syncthreads();
    if (bad) return;
    if (act && xin != x) {
        int c = i0 * n2 + pl;
#pragma unroll 4
        for (int u = 0; u < ni; u++, c += n2) x[c] = xin[c];
    }
    if (blockIdx.x == 0 && t == 0) {
        st->rr = sha[2];
        st->rmax = sha[3];
        st->iter = iter;
        st->first = 0;
        st->res = result;
        st->done = 1;
    }
}

int slab_class(int slab) {
    return slab <= 1 ? 1 : slab <= 2 ? 2 : slab <= 4 ? 4 : slab <= 8 ? 8 : slab <= 12 ? 12 : 16;
}

size_t lds_bytes(const GridDims& d) {
    return sizeof(double) * (size_t)d.slab * (kThreads + 4 * d.n);
}

int groups_of(const GridDims& d) { return (d.chunks + 1) / 2; }

int work_groups() { return std::min(compute_units(), kMaxWg); }

// Halo entries a thread of k_cg_onchip / k_cg_onchip2 holds, at most.
int held(int slab) {
    const int c = slab_class(slab);
    return c < kHalo ? c : kHalo;
}

size_t lds2_bytes(const GridDims& d, int T) {
    return sizeof(double) * (size_t)d.slab * (T * kBlock + 2 * d.n);
}

// Tiles per work-group of k_cg_onchip2 so that one work-group per CU covers the
// sweeps' tiles; 0: they do not fit the chip.
int tiles_per_wg(const GridDims& d, int cus) {
    if (d.slab > 16 || d.blocks > kFoldSlots) return 0;
    for (int T = 1; T <= kMaxTiles; T++) {
        if (T == 4 && d.slab > 4) break;  // 1024 threads leave 128 registers each
        if ((d.chunks + T - 1) / T * d.slabs <= cus && lds2_bytes(d, T) <= kLdsMax &&
            2 * d.n * d.slab <= held(d.slab) * T * kBlock)
            return T;
    }
    return 0;
}

template <bool PB, int SLAB>
void launch2_slab(hipStream_t s, const Onchip2Args& a, const PBCoef& pb, double* x, const double* r,
                  CGState* st) {
    const size_t lds = lds2_bytes(a.d, a.T);
    const dim3 g(a.nwg), b(a.T * kBlock);
    // Up to 512 threads leave 256 registers each, 768 leave 168, 1024 128.
    if (a.T <= 2)
        MAZE_LAUNCH((k_cg_onchip2<PB, SLAB, 512>), g, b, lds, s, a, pb, x, r, st);
    else if (SLAB > 4 || a.T == 3)
        MAZE_LAUNCH((k_cg_onchip2<PB, SLAB, 768>), g, b, lds, s, a, pb, x, r, st);
    else if constexpr (SLAB <= 4)
        MAZE_LAUNCH((k_cg_onchip2<PB, SLAB, 1024>), g, b, lds, s, a, pb, x, r, st);
}

template <bool PB>
void launch2_any(hipStream_t s, const Onchip2Args& a, const PBCoef& pb, double* x, const double* r,
                 CGState* st) {
    switch (slab_class(a.d.slab)) {
        case 1: return launch2_slab<PB, 1>(s, a, pb, x, r, st);
        case 2: return launch2_slab<PB, 2>(s, a, pb, x, r, st);
        case 4: return launch2_slab<PB, 4>(s, a, pb, x, r, st);
        case 8: return launch2_slab<PB, 8>(s, a, pb, x, r, st);
        case 12: return launch2_slab<PB, 12>(s, a, pb, x, r, st);
        default: return launch2_slab<PB, 16>(s, a, pb, x, r, st);
    }
}

// The work-group slabs of k_cg_stream: the sweeps' own, the last two as one
// where the chip has no room for a short last one.  0: the grid does not fit.
int stream_slabs(const GridDims& d, int cus) {
    const int groups = groups_of(d), last = d.n - (d.slabs - 1) * d.slab;
    if (d.blocks > kFoldSlots || d.slab > kStreamPlanes) return 0;
    const bool merge = groups * d.slabs > cus;
    if (merge && (d.slabs < 2 || d.slab + last > kStreamPlanes)) return 0;
    const int slabs = d.slabs - (merge ? 1 : 0), nwg = groups * slabs;
    return nwg <= cus && nwg >= kBlock / kWave ? slabs : 0;
}

template <bool PB>
void launch_any(hipStream_t s, const OnchipArgs& a, const PBCoef& pb, double* x, const double* r,
                CGState* st) {
    const size_t lds = lds_bytes(a.d);
    const dim3 g(a.nwg), b(kThreads);
    switch (slab_class(a.d.slab)) {
        case 1: MAZE_LAUNCH((k_cg_onchip<PB, 1>), g, b, lds, s, a, pb, x, r, st); break;
        case 2: MAZE_LAUNCH((k_cg_onchip<PB, 2>), g, b, lds, s, a, pb, x, r, st); break;
        case 4: MAZE_LAUNCH((k_cg_onchip<PB, 4>), g, b, lds, s, a, pb, x, r, st); break;
        case 8: MAZE_LAUNCH((k_cg_onchip<PB, 8>), g, b, lds, s, a, pb, x, r, st); break;
        case 12: MAZE_LAUNCH((k_cg_onchip<PB, 12>), g, b, lds, s, a, pb, x, r, st); break;
        default: MAZE_LAUNCH((k_cg_onchip<PB, 16>), g, b, lds, s, a, pb, x, r, st); break;
    }
}

}  // namespace

int compute_units() {
    int dev = 0, cus = 0;
    MAZE_HIP(hipGetDevice(&dev));
    MAZE_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    return cus;
}

// The vectors of a work-group's share fit it.
static bool share_fits(const GridDims& d) {
    return d.slab <= 16 && groups_of(d) * d.slabs <= kMaxWg && lds_bytes(d) <= kLdsMax &&
           2 * d.n * d.slab <= held(d.slab) * kThreads;
}

bool cg_one_reduction(const GridDims& d) { return share_fits(d); }

// The flattest slabs that leave at most one work-group per CU, where the grid
// then fits (up to 128^3).
GridDims cg_dims_for(int n) {
    const GridDims d = grid_dims_for(n);
    const int per_slab = groups_of(d);
    if (per_slab > kMaxWg) return d;
    const int slabs = std::min(n, kMaxWg / per_slab);
    const GridDims c = make_dims(n, (n + slabs - 1) / slabs);
    return share_fits(c) ? c : d;
}

bool cg_onchip_fits(const GridDims& d) {
    return share_fits(d) && groups_of(d) * d.slabs <= work_groups();
}

long cg_onchip_words() { return kSlot * (kMaxWg + kMaxGroups); }

void launch_cg_onchip(hipStream_t s, const GridDims& d, const PBCoef& pb, double* x, double* r,
                      double* h0, double* h1, CGState* st, const CgOnchip& w) {
    OnchipArgs a;
    a.d = d;
    a.groups = groups_of(d);
    a.nwg = a.groups * d.slabs;
    a.words = w.words;
    a.h0 = h0;
    a.h1 = h1;
    a.ctl = w.ctl;
    a.epoch = w.epoch;
    if (pb.ex) launch_any<true>(s, a, pb, x, r, st);
    else launch_any<false>(s, a, pb, x, r, st);
}

bool cg_onchip2_fits(const GridDims& d) {
    const int cus = work_groups();
    return tiles_per_wg(d, cus) > 0 || stream_slabs(d, cus) > 0;
}

void launch_cg_onchip2(hipStream_t s, const GridDims& d, const PBCoef& pb, double* x, double* r,
                       double* h, double* xs, CGState* st, const CgOnchip& w) {
    Onchip2Args a;
    a.d = d;
    a.T = tiles_per_wg(d, work_groups());
    if (!a.T) {
        StreamArgs b;
        b.d = d;
        b.groups = groups_of(d);
        b.slabs = stream_slabs(d, work_groups());
        b.nwg = b.groups * b.slabs;
        b.words = w.words;
        b.h = h;
        b.xs = xs;
        b.ctl = w.ctl;
        b.epoch = w.epoch;
        const size_t lds = sizeof(double) * (size_t)kStreamPlanes * kStreamStride;
        if (pb.ex) MAZE_LAUNCH(k_cg_stream<true>, dim3(b.nwg), dim3(kThreads), lds, s, b, pb, x, r, st);
        else MAZE_LAUNCH(k_cg_stream<false>, dim3(b.nwg), dim3(kThreads), lds, s, b, pb, x, r, st);
        return;
    }
    a.groups = (d.chunks + a.T - 1) / a.T;
    a.nwg = a.groups * d.slabs;
    a.words = w.words;
    a.h = h;
    a.ctl = w.ctl;
    a.epoch = w.epoch;
    if (pb.ex) launch2_any<true>(s, a, pb, x, r, st);
    else launch2_any<false>(s, a, pb, x, r, st);
}

}  // namespace maze
