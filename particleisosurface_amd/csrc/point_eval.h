// Neighbour sums for a wave's points, one point after another (any points, in any order).
#pragma once
#include "pisurf_internal.h"

#include <algorithm>
#include <type_traits>

namespace pisurf {

// SingleEval / SingleEvalWithGrad at points in any order: a wave takes m points (points_per_wave at most) one after another.
// Lanes 0 - 8 look up the nine rows of a point's window, the lanes test 64 candidates at a time (consecutive
// records of a row: coalesced reads, where threads with a point each gather from windows of their own), the
// passing ones are listed in order in LDS and evaluated 64 at a time, and their terms wait in LDS until one lane
// per sum adds them in the reference's order, the sums of all the wave's points side by side. Terms, order and
// roundings are those of field_sum.
//
// What bounds it: the latency of a point's dependent reads, 16 waves per CU side by side (a thread per point's
// window reads gathered a line per candidate: 1 M shuffled points with gradients on 1.6 M particles, compensated
// FP32, 2216 -> 1157 us), and for a few points the latency of one: 1000 points 88 -> 8.4 us, as each point's
// candidates are tested side by side instead of one by one.
// (gradients in FP64 keep four points' terms: with eight, LDS leaves two workgroups per CU)
constexpr int points_per_wave(bool fp64, bool grad) { return fp64 && grad ? 4 : 8; }

template <class R, bool GRAD> struct PointLds {
    static constexpr int C = GRAD ? 4 : 1;
    static constexpr int kStride = kWave + 1;  // (a stride of 64 would put every sum's terms in one bank)
    R term[points_per_wave(sizeof(R) == 8, GRAD) * C * kStride];
    int list[2 * kWave];
};

// Points i0 .. i0 + np - 1 of src (np <= points_per_wave; i0 and np uniform over the wave): bool point(i, p) gives a
// point's position (R or float) or says that there is none, the same in every lane; store(i, c, v) takes its sum c (field, then gradient). Returns the
// candidates visited and adds the points evaluated to evals.
template <class R, bool K, bool GRAD, int MODE, class Src>
__device__ __forceinline__ unsigned long long point_eval(const GridDev& g, const Recs<R>& rec, const FieldConst& fc,
                                                         const Src& src, int64_t i0, int np, PointLds<R, GRAD>& L,
                                                         int& evals) {
    constexpr int C = PointLds<R, GRAD>::C, kStride = PointLds<R, GRAD>::kStride;
    const int lane = threadIdx.x & (kWave - 1);
    R* const term = L.term;
    int* const list = L.list;
    const R inv_h2 = R(fc.inv_h2), h2 = R(fc.h2);
    Acc<R, K> sum;    // lane k C + c: sum c of point k
    int waiting = 0;  // its terms not added yet
    auto add_terms = [&]() {
        int most = waiting;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, kWave));
        for (int t = 0; t < most; t++)
            if (t < waiting) sum.add_unfused(term[lane * kStride + t]);
        waiting = 0;
        wave_sync();
    };
    unsigned long long vis = 0;
    for (int k = 0; k < np; k++) {
        R p[3];
        if (!src.point(i0 + k, p)) continue;
        evals++;
        const R px = p[0], py = p[1], pz = p[2];
        int ix, iy, iz, lo = 0, hi = 0;
        cell_of(g, float(px), float(py), float(pz), ix, iy, iz);
        if (lane >= 9 || !row_range(g, ix, iy, iz, lane, lo, hi)) lo = hi = 0;
        int end = hi - lo;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int t = __shfl_up(end, o, kWave);
            end += lane >= o ? t : 0;
        }
        // row r holds positions [first[r], first[r + 1]) of the window, position t being sorted particle t + d[r]
        const int begin = end - (hi - lo);
        int first[9], d[9];
#pragma unroll
        for (int r = 0; r < 9; r++) {
            first[r] = __builtin_amdgcn_readlane(begin, r);
            d[r] = __builtin_amdgcn_readlane(lo - begin, r);
        }
        const int total = __builtin_amdgcn_readlane(end, 8);
        vis += (unsigned long long)total;
        int have = 0;  // listed candidates
        auto evaluate = [&](int cnt) {
            if (__any(waiting && lane / C == k)) add_terms();  // the point's earlier terms come first
            if (lane < cnt) {
                const int j = list[lane];
                const auto a = rec.a[j];
                const float4 l4 = (K && sizeof(R) == 4) ? fc.lo[j] : make_float4(0.f, 0.f, 0.f, 0.f);
                const R dx = px - a.x, dy = py - a.y, dz = pz - a.z;
                Acc<R, K> v, gv[3];
                field_contrib<R, K, GRAD, MODE>(fc, inv_h2, h2, dx, dy, dz, dist2(dx, dy, dz), rec.g[2 * j],
                                                rec.g[2 * j + 1], l4, v, gv);
                term[(k * C) * kStride + lane] = v.get();
                if (GRAD)
#pragma unroll
                    for (int c = 0; c < 3; c++) term[(k * C + (GRAD ? 1 + c : 0)) * kStride + lane] = gv[c].get();
            }
            wave_sync();
            if (lane / C == k) waiting = cnt;
        };
        for (int t0 = 0; t0 < total; t0 += kWave) {
            const int t = t0 + lane;
            int dt = d[0];
#pragma unroll
            for (int r = 1; r < 9; r++) dt = t >= first[r] ? d[r] : dt;
            bool pass = false;
            if (t < total) {
                const auto a = rec.a[t + dt];
                pass = !(dist2(px - a.x, py - a.y, pz - a.z) >= a.w);
            }
            const unsigned long long pm = __ballot(pass);
            if (pass) list[have + __builtin_popcountll(pm & ((1ull << lane) - 1ull))] = t + dt;
            have += __builtin_popcountll(pm);
            wave_sync();
            if (have >= kWave) {
                evaluate(kWave);
                // the rest moves to the front
                const int rest = lane + kWave < have ? list[kWave + lane] : 0;
                wave_sync();
                if (lane + kWave < have) list[lane] = rest;
                have -= kWave;
                wave_sync();
            }
        }
        if (have) evaluate(have);
    }
    add_terms();
    if (lane < np * C) src.store(i0 + lane / C, lane % C, sum.get());
    return vis;
}

// go(mode) with the kernel mode as a compile-time constant
template <class Go> inline void point_dispatch(int mode, Go&& go) {
    if (mode == kModeAniBspline) go(std::integral_constant<int, kModeAniBspline>());
    else go(std::integral_constant<int, kModeAny>());
}

// Points per wave for n points, at most most: one as long as the waves fit the chip at once (256 CUs x 16), for the
// latency of few points, then as many as share their sums' additions
inline int point_share(int64_t n, int most) { return (int)std::max<int64_t>(1, std::min<int64_t>(most, (n + 4095) / 4096)); }

}  // namespace pisurf
