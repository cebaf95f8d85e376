// Neighbour sums for the 64 points of one wave, culled on the matrix cores.
//
// Every lane holds one query point. The wave takes the points of one (y, z) row of hash cells at a
// time (points in cell order: nearly always all of them, or two rows' ends), stages the candidates of the
// union of their windows (nine neighbour rows, each one contiguous range of sorted particles) in its own
// piece of LDS, finds for every lane the candidates that can contribute, and lets each lane sum its
// own in order. A point sees its 27-cell candidates in the reference's order (rows z-outer, then y, each row's
// cells x-ascending, sorted particles within a cell), so sums are those of the per-point kernels bit for bit. No
// workgroup barrier is used: the waves of a workgroup are independent.
//
// What bounds it: vector issue (0.95 vector instructions per CU and cycle). As runs of cells with a distance test
// per candidate and thread (run_eval.h), half of a wave's instructions tested candidates of which six in seven
// fail, and a third of the lanes idled in runs that did not fill their workgroup. Here
//  - every wave is full: it takes 64 consecutive points whatever their cells;
//  - the test is a product on the matrix cores: with the point p and the candidate a relative to the wave,
//      |p - a|^2 - R^2 = |p|^2 + (-2 a.x, -2 a.y, -2 a.z, |a|^2 - R^2) . (p.x, p.y, p.z, 1),
//    K = 4, one v_mfma_f32_16x16x4 for 16 candidates x 16 points, and one instruction per candidate
//    and wave gathers the sign bits;
//  - each lane walks its own pass bits over the whole chunk, so a wave takes as many steps as its busiest point has
//    passing candidates in the chunk (52 at the crown splash's deepest level; word by word it is 70).
// Deepest sampled level of the crown splash, its 11.9 M distinct points sorted by cell over the level (as leaf centres and a
// caller's many points come): 1.20 ms, 60 vector instructions per point, against 1.5 ms and 90 as runs. Its 14.7 M
// records as the tiles of nodes list them, without that sort: 1.5 ms.
// A chunk of 224 candidates takes a tenth fewer instructions, but its LDS leaves two waves per SIMD instead of
// four, and the kernel 1.5 times as long. Sorting the points by their passing candidates before dealing them to
// the lanes saves a tenth of the instructions (two points per lane) and loses as much to the occupancy.
#pragma once
#include "pisurf_internal.h"

#include <type_traits>

namespace pisurf {

constexpr int kWaveBatch = 112;  // candidates per round of products: four words of at most 28 pass bits
constexpr int kWaveCells = 16;   // cells of a row taken together at most

// The sign test's slack. A pass is only a promise that the candidate may contribute (R is a radius
// beyond which its contribution is exactly zero), so the radius may be enlarged freely. Rounding moves the
// tested value by at most 32 * 2^-24 * max(|a|, |p|)^2 (in cells squared: the rounding of the relative
// positions, of the four products and of their sums), and a pair that has to pass has |p| < |a| + R:
// kWaveSlack (|a|^2 + R^2) is more than twice that.
constexpr float kWaveSlack = 1e-5f;

typedef float wave_acc __attribute__((ext_vector_type(4)));

// Policy interface of wave_visit:
//   Pol::kChunk                                         candidates staged at a time (1 - 4 batches)
//   typename Pol::Real                                  type of the staged positions
//   typename Pol::Lds                                   staging buffers for kChunk candidates
//   typename Pol::State                                 per-point accumulators
//   void stage(Lds&, int t, int j, Real a[4]) const     candidate j -> slot t; a: its position and
//                                                       squared radius
//   void take(State&, const Lds&, int t) const          contribution of slot t
template <class Pol> struct WaveLds {
    typename Pol::Lds rec;
    float4 cull[Pol::kChunk];           // (-2 a, |a|^2 - R^2) of the staged candidates
    // per lane, its words with a bit set, one after another: pass bits | word number << 28 (one more is read)
    unsigned word[(4 * Pol::kChunk / kWaveBatch + 1) * kWave];
    int raw[9 * (kWaveCells + 3)];      // sorted position of cell boundary x0 - 1 + i of row r at 9 i + r
};

// after: r[i] of lane group g (16 lanes each) = the former r[g] of lane group i
__device__ __forceinline__ void wave_transpose4(unsigned r[4]) {
    auto s32 = [](unsigned& a, unsigned& b) {
        const auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        a = v[0];
        b = v[1];
    };
    auto s16 = [](unsigned& a, unsigned& b) {
        const auto v = __builtin_amdgcn_permlane16_swap(a, b, false, false);
        a = v[0];
        b = v[1];
    };
    s32(r[0], r[2]);
    s32(r[1], r[3]);
    s16(r[0], r[1]);
    s16(r[2], r[3]);
}

// The wave's points as the cull's right-hand operand: b[k] holds points 16 k .. 16 k + 15, component
// l / 16 of (x, y, z, 1) in lane l; sq[k] their squared lengths.
struct WavePoints {
    float b[4], sq[4];
    __device__ __forceinline__ void set(float x, float y, float z) {
        unsigned v[4] = {__float_as_uint(x), __float_as_uint(y), __float_as_uint(z), __float_as_uint(1.0f)};
        const unsigned q = __float_as_uint(x * x + y * y + z * z);
        unsigned w[4] = {q, q, q, q};
        wave_transpose4(v);
        wave_transpose4(w);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            b[k] = __uint_as_float(v[k]);
            sq[k] = __uint_as_float(w[k]);
        }
    }
};

// Pass words of the lane's own point: bit u of s[k] is set when slot 4 nb k + u (u < 4 nb) can contribute.
// In the products, row 4 k + i of block rb is slot 4 nb k + 4 rb + i, so lane l ends up with segment
// l / 16 for point l % 16 of each of the four point blocks; the transpose gives every lane its own
// point's four words.
__device__ __forceinline__ void wave_cull(const float4* cull, const WavePoints& pt, int nb, unsigned s[4]) {
    const int lane = threadIdx.x & (kWave - 1);
    const float* a = (const float*)&cull[4 * nb * ((lane >> 2) & 3) + (lane & 3)] + (lane >> 4);
    float next = a[16 * (nb - 1)];
#pragma unroll
    for (int k = 0; k < 4; k++) s[k] = 0;
#pragma unroll 1
    for (int rb = nb - 1; rb >= 0; rb--) {
        const float av = next;
        next = a[16 * max(rb - 1, 0)];
        wave_acc d[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const wave_acc c0 = {pt.sq[k], pt.sq[k], pt.sq[k], pt.sq[k]};
            d[k] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, pt.b[k], c0, 0, 0, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);   // the four products first,
        __builtin_amdgcn_sched_group_barrier(0x2, 16, 0);  // then their sign bits: no wait in between
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int i = 3; i >= 0; i--) s[k] = __builtin_amdgcn_alignbit(s[k], __float_as_uint(d[k][i]), 31);
    }
    wave_transpose4(s);
}

// Adds to st the contributions of the candidates of point p (act: the lane has a point) and returns
// their number, passing or not. Every lane of the wave calls it. Neighbouring lanes should lie close
// together; any order is right unless kWaveSorted is given, which says that the points come in cell order,
// active lanes first. BACK: cells before the first lane's that its row piece may take. p is the position that picks the
// cell, q the one that distances are taken from (the same, or p before it was rounded to float).
constexpr int kWaveSorted = -1;
template <int BACK, class Pol>
__device__ __forceinline__ int wave_visit(const GridDev& g, const Pol& pol, typename Pol::State& st, bool act,
                                          const float p[3], const typename Pol::Real q[3], WaveLds<Pol>& L) {
    typedef typename Pol::Real Real;
    const int lane = threadIdx.x & (kWave - 1);
    int ix, iy, iz;
    cell_of(g, p[0], p[1], p[2], ix, iy, iz);
    // a cell more than one off the grid has no neighbour in it
    const bool in = act && ix >= -1 && ix <= g.n[0] && iy >= -1 && iy <= g.n[1] && iz >= -1 && iz <= g.n[2];
    const float ic = 1.0f / g.cell;
    int ncand = 0;
    unsigned long long rem = __ballot(in);
    while (rem) {
        const int lead = __builtin_ctzll(rem);
        const int lx = __builtin_amdgcn_readlane(ix, lead), ly = __builtin_amdgcn_readlane(iy, lead),
                  lz = __builtin_amdgcn_readlane(iz, lead);
        // the lanes taken with the leader: its row, and at most kWaveCells cells
        constexpr bool SORTED = BACK == kWaveSorted;
        constexpr int kBack = SORTED ? 0 : BACK;
        const bool mem = ((rem >> lane) & 1) && iy == ly && iz == lz && (unsigned)(ix - lx + kBack) < (unsigned)kWaveCells;
        const unsigned long long mm = __ballot(mem);
        rem &= ~mm;
        int x0 = lx, x1 = lx;
        if (SORTED) {
            x1 = __builtin_amdgcn_readlane(ix, 63 - __builtin_clzll(mm));
        } else {
            int lo = mem ? ix : lx, hi = lo;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                lo = min(lo, __shfl_xor(lo, o, kWave));
                hi = max(hi, __shfl_xor(hi, o, kWave));
            }
            x0 = __builtin_amdgcn_readfirstlane(lo);
            x1 = __builtin_amdgcn_readfirstlane(hi);
        }
        const int nc = x1 - x0 + 1;  // <= kWaveCells
        const int rel = mem ? ix - x0 : 0;
        // cell boundaries of the nine neighbour rows (a row outside the grid is empty)
        for (int e = lane; e < 9 * (nc + 3); e += kWave) {
            const int i = e / 9, r = e - 9 * i;
            const int yy = ly + (r % 3) - 1, zz = lz + (r / 3) - 1;
            int v = 0;
            if (yy >= 0 && yy < g.n[1] && zz >= 0 && zz < g.n[2])
                v = g.off[(zz * g.n[1] + yy) * g.n[0] + min(max(x0 - 1 + i, 0), g.n[0])];
            L.raw[e] = v;
        }
        wave_sync();
        // the rows' candidates concatenated in row order: row r holds positions [roff[r], roff[r + 1]),
        // sorted position = concatenated position - dl[r]
        const int r9 = min(lane, 8);
        const int first = L.raw[r9], len = L.raw[9 * (nc + 2) + r9] - first;
        int end = lane < 9 ? len : 0;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) {
            const int t = __shfl_up(end, o, kWave);
            end += lane >= o ? t : 0;
        }
        int roff[10], dl[9];
        roff[0] = 0;
#pragma unroll
        for (int r = 0; r < 9; r++) {
            roff[r + 1] = __builtin_amdgcn_readlane(end, r);
            dl[r] = roff[r] - __builtin_amdgcn_readlane(first, r);
        }
        const int total = roff[9];
        if (nc == 1) {
            ncand = mem ? total : ncand;
        } else {
            // candidates of cells up to each boundary; a window is three cells wide
            int below = 0;
            const int col = 9 * min(lane, nc + 2);
#pragma unroll
            for (int r = 0; r < 9; r++) below += L.raw[col + r];
            const int win = __shfl(below, rel + 3, kWave) - __shfl(below, rel, kWave);
            ncand = mem ? win : ncand;
        }
        if (total == 0) continue;
        // the cull works in cells about the middle of the row piece
        const float ox = g.b0[0] + 0.5f * float(x0 + x1 + 1) * g.cell, oy = g.b0[1] + (float(ly) + 0.5f) * g.cell,
                    oz = g.b0[2] + (float(lz) + 0.5f) * g.cell;
        WavePoints pt;
        pt.set(float(q[0] - Real(ox)) * ic, float(q[1] - Real(oy)) * ic, float(q[2] - Real(oz)) * ic);
        for (int cb = 0; cb < total; cb += Pol::kChunk) {
            const int n = min((int)Pol::kChunk, total - cb);
            // batches of 16 nb slots, four words of wl = 4 nb each
            const int nbatch = (n + kWaveBatch - 1) / kWaveBatch;
            const int nb = (n + 16 * nbatch - 1) / (16 * nbatch), wl = 4 * nb;
            for (int t = lane; t < n; t += kWave) {
                const int c = cb + t;
                int d = dl[0];
#pragma unroll
                for (int r = 1; r < 9; r++) d = c >= roff[r] ? dl[r] : d;  // the row holding position c
                Real a[4];
                pol.stage(L.rec, t, c - d, a);
                const float x = float(a[0] - Real(ox)) * ic, y = float(a[1] - Real(oy)) * ic,
                            z = float(a[2] - Real(oz)) * ic;
                // (in cells before it is narrowed: a small radius' square is no normal float)
                const float a2 = x * x + y * y + z * z, r2 = float(a[3] * Real(ic) * Real(ic));
                const float w = a2 - r2 - kWaveSlack * (a2 + r2);
                // a NaN or unbounded record always passes: it reaches every sum of its window
                const bool fin = fabsf(w) < 1e30f;
                L.cull[t] = fin ? make_float4(-2.0f * x, -2.0f * y, -2.0f * z, w) : make_float4(0.f, 0.f, 0.f, -1e30f);
            }
            wave_sync();
            unsigned* wp = L.word + lane;
            int left = 0;  // passing candidates of this lane
            for (int b = 0; b < nbatch; b++) {
                // the slots of each lane's own window, as words of wl bits
                const int s0 = 4 * b * wl;
                unsigned w[4];
                if (nc == 1) {
#pragma unroll
                    for (int k = 0; k < 4; k++) w[k] = mem ? (1u << min(max(n - s0 - k * wl, 0), wl)) - 1u : 0u;
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++) w[k] = 0;
#pragma unroll
                    for (int r = 0; r < 9; r++) {
                        const int lo = roff[r] - cb - s0, hi = roff[r + 1] - cb - s0;
                        if (hi <= 0 || lo >= 4 * wl || lo == hi) continue;
                        const int d = dl[r] - cb - s0;
                        int clo = mem ? L.raw[9 * rel + r] + d : 0;
                        const int chi = mem ? min(L.raw[9 * (rel + 3) + r] + d, n - s0) : 0;
                        clo = min(clo, chi);  // (the chunk may end below the window)
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            if (hi <= k * wl || lo >= (k + 1) * wl) continue;
                            const int b0 = min(max(clo - k * wl, 0), wl), b1 = min(max(chi - k * wl, 0), wl);
                            w[k] |= (1u << b1) - (1u << b0);  // bits b0 .. b1 - 1 (wl < 32)
                        }
                    }
                }
                unsigned s[4];
                wave_cull(L.cull + s0, pt, nb, s);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    w[k] &= s[k];
                    left += __builtin_popcount(w[k]);
                    *wp = w[k] | ((unsigned)(4 * b + k) << 28);
                    wp += w[k] ? kWave : 0;
                }
            }
            // Each lane takes its own passing candidates, in order, whatever word they are in: the wave
            // takes as many steps as its busiest lane has candidates.
            wp = L.word + lane;
            unsigned next = *wp, m = 0;
            int base = 0;
            while (left > 0) {
                const bool z = m == 0;
                m = z ? next & 0x0fffffffu : m;
                base = z ? (int)(next >> 28) * wl : base;
                wp += z ? kWave : 0;
                next = *wp;
                const int t = base + __builtin_ctz(m);
                m &= m - 1;
                left--;
                pol.take(st, L.rec, t);
            }
            wave_sync();  // the slots are free again
        }
    }
    return ncand;
}

// ---- field sums (SingleEval / SingleEvalWithGrad) ----
// Staged records: the values a contribution needs, packed into 16-byte reads (FP32: mean and G; compensated
// FP32 adds the mean's residual; FP64 in pairs of doubles).
template <class R, bool LO, int N> struct WaveRec;
template <int N> struct WaveRec<float, false, N> {
    float4 q0[N], q1[N];
    float2 q2[N];
    __device__ __forceinline__ void put(int t, const float4& a, const float4& g0, const float4& g1, const float4&) {
        q0[t] = make_float4(a.x, a.y, a.z, g0.x);
        q1[t] = make_float4(g0.y, g0.z, g0.w, g1.x);
        q2[t] = make_float2(g1.y, g1.z);
    }
    __device__ __forceinline__ void get(int t, float a[3], float4& g0, float4& g1, float4& lo) const {
        const float4 u = q0[t], v = q1[t];
        const float2 w = q2[t];
        a[0] = u.x;
        a[1] = u.y;
        a[2] = u.z;
        g0 = make_float4(u.w, v.x, v.y, v.z);
        g1 = make_float4(v.w, w.x, w.y, 0.f);
        lo = make_float4(0.f, 0.f, 0.f, 0.f);
    }
};
template <int N> struct WaveRec<float, true, N> {
    float4 q0[N], q1[N], q2[N];
    float q3[N];
    __device__ __forceinline__ void put(int t, const float4& a, const float4& g0, const float4& g1, const float4& lo) {
        q0[t] = make_float4(a.x, a.y, a.z, lo.x);
        q1[t] = make_float4(lo.y, lo.z, g0.x, g0.y);
        q2[t] = make_float4(g0.z, g0.w, g1.x, g1.y);
        q3[t] = g1.z;
    }
    __device__ __forceinline__ void get(int t, float a[3], float4& g0, float4& g1, float4& lo) const {
        const float4 u = q0[t], v = q1[t], w = q2[t];
        a[0] = u.x;
        a[1] = u.y;
        a[2] = u.z;
        lo = make_float4(u.w, v.x, v.y, 0.f);
        g0 = make_float4(v.z, v.w, w.x, w.y);
        g1 = make_float4(w.z, w.w, q3[t], 0.f);
    }
};
template <int N> struct WaveRec<double, false, N> {
    double2 q0[N], q1[N], q2[N], q3[N], q4[N];
    __device__ __forceinline__ void put(int t, const double4& a, const double4& g0, const double4& g1, const float4&) {
        q0[t] = make_double2(a.x, a.y);
        q1[t] = make_double2(a.z, g0.x);
        q2[t] = make_double2(g0.y, g0.z);
        q3[t] = make_double2(g0.w, g1.x);
        q4[t] = make_double2(g1.y, g1.z);
    }
    __device__ __forceinline__ void get(int t, double a[3], double4& g0, double4& g1, float4& lo) const {
        const double2 u = q0[t], v = q1[t], w = q2[t], x = q3[t], y = q4[t];
        a[0] = u.x;
        a[1] = u.y;
        a[2] = v.x;
        g0 = make_double4(v.y, w.x, w.y, x.x);
        g1 = make_double4(x.y, y.x, y.y, 0.0);
        lo = make_float4(0.f, 0.f, 0.f, 0.f);
    }
};

template <class R, bool K, bool GRAD, int MODE> struct WaveField {
    static constexpr bool LO = K && sizeof(R) == 4;
    static constexpr int kChunk = kWaveBatch;
    typedef R Real;
    typedef WaveRec<R, LO, kChunk> Lds;
    struct State {
        R px, py, pz;
        Acc<R, K> acc, ga[3];
        __device__ __forceinline__ State(R x, R y, R z) : px(x), py(y), pz(z) {}
    };
    Recs<R> rec;
    FieldConst fc;
    R inv_h2, h2;
    __device__ __forceinline__ WaveField(const Recs<R>& r, const FieldConst& f)
        : rec(r), fc(f), inv_h2(R(f.inv_h2)), h2(R(f.h2)) {}
    __device__ __forceinline__ void stage(Lds& l, int t, int j, R a4[4]) const {
        const typename Vec4<R>::T a = rec.a[j];
        l.put(t, a, rec.g[2 * j], rec.g[2 * j + 1], LO ? fc.lo[j] : make_float4(0.f, 0.f, 0.f, 0.f));
        a4[0] = a.x;
        a4[1] = a.y;
        a4[2] = a.z;
        a4[3] = a.w;
    }
    __device__ __forceinline__ void take(State& s, const Lds& l, int t) const {
        typename Vec4<R>::T g0, g1;
        R a[3];
        float4 lo;
        l.get(t, a, g0, g1, lo);
        const R dx = s.px - a[0], dy = s.py - a[1], dz = s.pz - a[2];
        field_contrib<R, K, GRAD, MODE>(fc, inv_h2, h2, dx, dy, dz, dist2(dx, dy, dz), g0, g1, lo, s.acc, s.ga);
    }
};

// Points h = blockIdx.x * T + threadIdx.x < n of src evaluated by the waves of a block of T threads; returns the
// candidates of this thread's point. bool src.point(h, p) gives a point or says that there is none.
template <int T, class R, bool K, bool GRAD, int MODE, int BACK = kWaveSorted, class Src>
__device__ __forceinline__ int wave_eval(const GridDev& g, const Recs<R>& rec, const FieldConst& fc, const Src& src,
                                         int n, WaveLds<WaveField<R, K, GRAD, MODE>>* lds) {
    const WaveField<R, K, GRAD, MODE> pol(rec, fc);
    const int h = (int)blockIdx.x * T + (int)threadIdx.x;
    float p[3] = {0.f, 0.f, 0.f};
    const bool act = h < n && src.point(h, p);
    const R q[3] = {R(p[0]), R(p[1]), R(p[2])};
    typename WaveField<R, K, GRAD, MODE>::State st{q[0], q[1], q[2]};
    const int ncand = wave_visit<BACK>(g, pol, st, act, p, q, lds[threadIdx.x / kWave]);
    if (act) {
        const R gr[3] = {st.ga[0].get(), st.ga[1].get(), st.ga[2].get()};
        src.store(h, st.acc.get(), gr);
    }
    return ncand;
}

// The sum at one position q per lane (act: the lane has one); neighbouring lanes should lie close together. Returns the
// candidates of this lane's point.
template <class R, bool K, int MODE>
__device__ __forceinline__ int wave_sum(const GridDev& g, const Recs<R>& rec, const FieldConst& fc, bool act,
                                        const R q[3], WaveLds<WaveField<R, K, false, MODE>>& lds, R& sum) {
    const WaveField<R, K, false, MODE> pol(rec, fc);
    const float p[3] = {float(q[0]), float(q[1]), float(q[2])};
    typename WaveField<R, K, false, MODE>::State st{q[0], q[1], q[2]};
    const int ncand = wave_visit<kWaveCells / 2>(g, pol, st, act, p, q, lds);
    sum = st.acc.get();
    return ncand;
}

// go(block size, kernel mode) with both as compile-time constants
template <class Go> inline void wave_dispatch(int T, int mode, Go&& go) {
    using M0 = std::integral_constant<int, kModeAny>;
    using M1 = std::integral_constant<int, kModeAniBspline>;
    auto with = [&](auto tag) { mode == kModeAniBspline ? go(tag, M1()) : go(tag, M0()); };
    if (T == 256) with(std::integral_constant<int, 256>());
    else if (T == 128) with(std::integral_constant<int, 128>());
    else with(std::integral_constant<int, 64>());
}

}  // namespace pisurf
