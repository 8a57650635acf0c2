// Wavefront-level tracking shared by the tracking kernels (single tracker and
// batched jobs): a wavefront's particles advanced for a number of turns with
// the table record in scalar registers, loss kept as lane masks, and the
// survivors appended to the next live list. Replaces the per-turn launches of
// src/henon.cu:636-691 / :3155-3185 and the host loop :2701-2752.
#pragma once
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdint>

#include "hm_device.h"

namespace hm {

constexpr uint32_t kFlagRange = 1u;

// Lanes whose v is not below s (NaN included), as a mask.
__device__ __forceinline__ uint64_t not_below(double v, double s)
{
    constexpr int kUnorderedOrGE = 11;
    return __builtin_amdgcn_fcmp(v, s, kUnorderedOrGE);
}

// Whether both pairs of a record are the sine and cosine of one angle, to 2^-40 (a
// table of hm_build_table keeps to about 2^-52; records that are not finite do not).
// Turns that do not rotate may take a point out from anywhere, or bring it down to
// where products leave the normal range.
__device__ __forceinline__ bool rotates(const TabEntry &t)
{
    return fabs(fma(t.sx, t.sx, fma(t.cx, t.cx, -1.0))) < 0x1p-40 &&
           fabs(fma(t.sy, t.sy, fma(t.cy, t.cy, -1.0))) < 0x1p-40;
}

// Per-lane fallback used when the live lanes of a wavefront do not share one
// turn index (particles reset while others were not) or when that index range
// leaves the table: each lane reads its own table record, and a lane whose
// index would leave [0, tab_len) stops unchanged and raises kFlagRange.
template <int MODE, bool INV, bool OCT>
__device__ __forceinline__ void track_lanes(double &x, double &px, double &y, double &py, bool &alive,
                                            uint32_t &done, uint32_t s, const TabEntry *__restrict__ tab,
                                            uint32_t tab_len, uint32_t n_turns, double mu, double b2, uint32_t *status)
{
    const double m3mu = -3.0 * mu;
    for (uint32_t k = 0; k < n_turns; ++k) {
        if (alive) {
            const int64_t ti = INV ? (int64_t)s - 1 - (int64_t)k : (int64_t)s + (int64_t)k;
            if (ti < 0 || ti >= (int64_t)tab_len) {
                atomicOr(status, kFlagRange);
                alive = false;
                done = k;
            } else {
                const TabEntry t = tab[ti];
                map_step<MODE, INV, OCT>(x, px, y, py, mu, m3mu, t);
                if (!(radius2<MODE>(x, px, y, py) < b2)) {
                    x = px = y = py = __builtin_nan("");
                    alive = false;
                    done = k;
                }
            }
        }
        if (!__any(alive)) break;
    }
}

// One particle per lane, n_turns turns in registers. Wavefront w owns the 64
// consecutive entries [64 w, 64 (w + 1)) of the particle list (or of the
// live-index list `idx_in`). The particle count is read from device memory
// (`count_in`) when given, so a launch can be sized from an upper bound without a
// host round trip.
//
// The first live lane's turn index s0 is read into a scalar register; when every
// live particle of the wavefront shares it (the normal case: all particles of a
// tracker advance together), the table record of turn s0+k is the same for the
// whole wavefront and is fetched with a scalar load, ahead of its use, straight
// into SGPR operands of the VALU ops. Losses are kept as wave-uniform lane masks.
struct TrackArgs {
    double *gx, *gpx, *gy, *gpy;
    uint32_t *gsteps;
    const uint32_t *idx_in, *count_in;
    uint32_t n_arg;
    const TabEntry *tab;
    uint32_t tab_len, n_turns;
    double mu, b2;
    double safe1;  // squared radius below which the next turn cannot lose a point (safe_radius2)
    uint32_t *idx_out, *count_out, *status;
};

// How much of a turn's octupole kick is fused (fwd_exact_fused): 0 without
// octupole, 2 in exact mode when mu is a power of two, else 1.
inline int octupole_kind(int mode, double mu)
{
    if (mu == 0.0) return 0;
    if (mode != kExact) return 1;
    int e = 0;
    const double m = std::frexp(std::fabs(mu), &e);
    return m == 0.5 && e >= -63 && e <= 65 ? 2 : 1;
}

// Squared radius R^2 such that a point with r < R is inside the barrier b and stays
// inside for one turn of the map or of its inverse: the kick moves (px, py) by at
// most rho^2 + |mu| rho^3, rho = |(x, y)| <= r, and the rotations keep r, so a turn
// takes r to at most r + r^2 + |mu| r^3; R takes that to b, less a margin far above
// the roundings. 0 (never inside) where no such radius exists: a barrier or a mu that
// is NaN (no point is inside the one, the other has no bound), a mu beyond 1e100.
inline double safe_radius2(double barrier, double mu)
{
    const double m = std::fabs(mu);
    if (!(std::fabs(barrier) > 0.0) || !(m < 1e100)) return 0.0;
    const double b = std::fmin(std::fabs(barrier), 1e100);
    const auto reach = [m](double r) { return r * (1.0 + r * (1.0 + m * r)); };
    // Newton's steps from above (the function is convex), from where one of the terms
    // alone reaches b (none overflows there): at most six of them, 0.07 us a call, where
    // 60 bisections took 0.6
    double r = std::fmin(b, std::fmin(std::sqrt(b), std::cbrt(b / m)));
    for (int i = 0; i < 1100; ++i) {
        const double next = r - (reach(r) - b) / (1.0 + r * (2.0 + 3.0 * m * r));
        if (!(next < r * (1.0 - 1e-9))) break;
        r = next;
    }
    r *= 1.0 - 1e-6;
    return reach(r) < b * (1.0 - 1e-7) ? r * r : 0.0;
}

// What a wavefront writes at the end of its turns. Read again then (see
// track_wave): kept through the turn loop, these pointers would take 14 of its
// scalar registers.
struct TrackOut {
    double *gx, *gpx, *gy, *gpy;
    uint32_t *gsteps, *idx_out, *count_out;
};

constexpr uint32_t kBlock = 8;  // turns per pass of the turn loop
// out(): the TrackOut of this wavefront, called after the turns.
template <int MODE, bool INV, int OCT, class Out>
__device__ __forceinline__ void track_wave(const TrackArgs &A, uint32_t base, uint32_t n, Out out)
{
    constexpr bool EXACT = MODE == kExact;
    const TabEntry *__restrict__ tab = A.tab;
    const uint32_t tab_len = A.tab_len, n_turns = A.n_turns;
    const double mu = A.mu, b2 = A.b2, m3mu = -3.0 * mu;
    const uint32_t lane = __lane_id(), i = base + lane;
    const uint64_t my_bit = 1ull << lane;
    const bool in_range = i < n;
    uint32_t j = 0, s = 0, done = n_turns;
    double x = __builtin_nan(""), px = x, y = x, py = x;
    if (in_range) {
        j = A.idx_in ? A.idx_in[i] : i;
        x = A.gx[j];
        px = A.gpx[j];
        y = A.gy[j];
        py = A.gpy[j];
        s = A.gsteps[j];
    }
    // henon.cu:431-434: a particle with a NaN coordinate is not stepped
    const bool alive0 = in_range && !any_nan(x, px, y, py);
    uint64_t live = __ballot(alive0);
    if (!live) return;
    const uint32_t s0 = __builtin_amdgcn_readlane(s, __builtin_ctzll(live));
    const bool same = __all(!alive0 || s == s0);
    // forward reads records s0 .. s0+n_turns-1, inverse s0-1 down to s0-n_turns:
    // both ends must lie inside [0, tab_len), else the per-lane path flags it
    const bool in_table = INV ? (s0 >= n_turns && s0 <= tab_len) : ((uint64_t)s0 + n_turns <= (uint64_t)tab_len);

    if (same && in_table && n_turns > 0) {
        // the table is read-only for the whole launch: reading it through the
        // constant address space lets wave-uniform records come in by scalar
        // loads even when the table pointer itself was loaded from memory
        const ConstPtr<TabEntry> tp = as_const(INV ? tab + (s0 - 1) : tab + s0);
        auto rec = [&](uint32_t k) -> TabEntry {
            const ConstPtr<TabEntry> r = INV ? tp - k : tp + k;
            return load_record(r);
        };
        double xx = x * x, yy = y * y, r2 = 0.0;
        // exact mode screens losses with a fused radius (screen_radius2) and
        // confirms candidates with the reference's expression
        const double b2s = EXACT ? screen_bound(b2) : b2;
        auto radius = [&] {
            r2 = EXACT ? fma(px, px, xx) + fma(py, py, yy) : radius2<MODE>(x, px, y, py);
        };
        auto turn = [&](const TabEntry &t) {
            if (EXACT && INV) inv_exact_fused<OCT>(x, px, y, py, xx, yy, mu, t);
            else if (EXACT) fwd_exact_fused<OCT>(x, px, y, py, xx, yy, mu, t);
            else map_step<MODE, INV, OCT != 0>(x, px, y, py, mu, m3mu, t);
        };
        // The losses of turn kk (the exact confirmation, the loss turn, the live
        // mask): the rare path of a checked turn.
        auto settle = [&](uint32_t kk) {
            uint64_t lost = live & not_below(r2, b2s);
            if (EXACT && lost) lost &= not_below(exact_radius2(x * x, px, y * y, py), b2);
            if (lost & my_bit) done = kk;
            live &= ~lost;
        };
        // The fused forms need every coordinate zero or at least kTinyCoord.
        bool plain = true;
        if (EXACT) {
            auto small = [](double v) { return v != 0.0 && fabs(v) < kTinyCoord; };
            plain = !__any(alive0 && (small(x) || small(px) || small(y) || small(py)));
        }
        uint32_t k = 0;
        if (plain && n_turns >= kBlock) {
            // Turns go in pairs with one test: a point below safe1 after the first
            // turn is inside the barrier after the second, whatever it is, as far as
            // the records rotate. A turn is then 30 to 32 operations and half a test
            // (4 operations and a branch), where every turn had one: 1e6 particles on
            // the 1000 x 1000 grid, 3e4 turns, mu = 0.5: 21.7 -> 19.1 ms (exact), 15.7
            // -> 14.1 ms (fast).
            const double safe1 = A.safe1;
            auto pair = [&](const TabEntry &t0, const TabEntry &t1, uint32_t kk) {
                turn(t0);
                radius();
                if (__builtin_expect((live & not_below(r2, safe1)) == 0, 1)) {
                    turn(t1);
                } else {
                    if (live & not_below(r2, b2s)) settle(kk);
                    turn(t1);
                    radius();
                    if (live & not_below(r2, b2s)) settle(kk + 1);
                }
            };
            // Two pairs of records: while one pair's turns run, the other is
            // requested (one 64-byte scalar load), into the registers the pair
            // before last used.
            const uint32_t last = n_turns - 2;
            TabEntry a0 = rec(0), a1 = rec(1), b0, b1;
            ConstPtr<TabEntry> tp_next = tp - 1;
            if (INV) asm("" : "+s"(tp_next));  // kept, not formed again at each use
            // At every 64th turn each lane takes one of the 64 records from 64 turns
            // ahead on: to see that all rotate before the turns get there, and so that
            // the scalar loads find the table in L2 also the first time it is read (64
            // particles, 1e4 turns: 0.79 ms; the first call 1.0 ms longer without).
            auto ahead = [&](uint32_t from) {
                const uint32_t kk = min(from + lane, n_turns - 1);
                return INV ? tab[s0 - 1 - kk] : tab[s0 + kk];
            };
            uint32_t blocks = n_turns / kBlock;
            bool rotating = !__any(!rotates(ahead(0)));
            while (rotating && blocks && live) {
                const TabEntry later = ahead(k + 64);
                uint32_t m = min(blocks, 64 / kBlock);
                blocks -= m;
                do {
                    // (from the lowest address of the block's records on, for fixed offsets)
                    const ConstPtr<TabEntry> p = INV ? tp - (k + (kBlock - 1)) : tp + k;
#pragma unroll
                    for (uint32_t q = 0; q < kBlock; q += 4) {
                        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): a0, a1 are there
                        __builtin_amdgcn_sched_barrier(0);
                        b0 = load_record(p + (INV ? kBlock - 1 - (q + 2) : q + 2));
                        b1 = load_record(p + (INV ? kBlock - 1 - (q + 3) : q + 3));
                        // (keeps the loads ahead of the first turn)
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_sched_barrier(0);
                        pair(a0, a1, k + q);
                        const uint32_t nx = min(k + q + 4, last);
                        __builtin_amdgcn_s_waitcnt(0xC07F);
                        __builtin_amdgcn_sched_barrier(0);
                        const ConstPtr<TabEntry> pn = INV ? tp_next - nx : tp + nx;
                        a0 = load_record(INV ? pn + 1 : pn);
                        a1 = load_record(INV ? pn : pn + 1);
                        __builtin_amdgcn_sched_barrier(0);
                        pair(b0, b1, k + q + 2);
                    }
                    k += kBlock;
                    m = __builtin_amdgcn_readfirstlane(m - 1);  // (kept in a scalar register)
                } while (m && live);
                rotating = !__any(!rotates(later));
            }
        }
        // What is left (fewer than kBlock turns, all of them for tiny coordinates, all
        // from a window of records on that do not all rotate): the map's own
        // operations and a test every turn.
        TabEntry next = rec(min(k, n_turns - 1));
        for (; k < n_turns && live; ++k) {
            const TabEntry t = next;
            next = rec(min(k + 1, n_turns - 1));
            map_step<MODE, INV, OCT != 0>(x, px, y, py, mu, m3mu, t);
            r2 = EXACT ? screen_radius2(x, px, y, py) : radius2<MODE>(x, px, y, py);
            if (live & not_below(r2, b2s)) settle(k);
        }
        if (alive0 && !(live & my_bit)) x = px = y = py = __builtin_nan("");
    } else if (n_turns > 0) {
        bool a = alive0;
        track_lanes<MODE, INV, OCT != 0>(x, px, y, py, a, done, s, tab, tab_len, n_turns, mu, b2, A.status);
        live = __ballot(a);
    }

    const TrackOut o = out();
    if (alive0) {
        o.gx[j] = x;
        o.gpx[j] = px;
        o.gy[j] = y;
        o.gpy[j] = py;
        o.gsteps[j] = INV ? s - done : s + done;
    }
    if (o.idx_out && live) {
        // wavefront-aggregated append of the survivors to the next live list
        const int leader = __builtin_ctzll(live);
        uint32_t slot = 0;
        if ((int)lane == leader) slot = atomicAdd(o.count_out, (uint32_t)__popcll(live));
        slot = __builtin_amdgcn_readlane(slot, leader);
        if (live & my_bit) o.idx_out[slot + __popcll(live & (my_bit - 1ull))] = j;
    }
}

}  // namespace hm
