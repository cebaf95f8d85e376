// Vertex placement: edge bisection (VisitorExtract::calc_vertices, src/visitorextract.cpp:47-84)
// and the per-leaf QEF solve (TNode::NodeCalcNode, src/iso_method_ours.cpp:101-174).
#include "pisurf_internal.h"
#include "point_eval.h"
#include "qef_device.h"

#include <type_traits>

namespace pisurf {

// An edge under bisection. Endpoints are (x, y, z, f) with f of opposite signs (f > 0 is +1).
// The midpoint replaces the endpoint of equal sign and the length is halved (not recomputed)
// until it is at most r/2; then the zero crossing is interpolated, snapping to an endpoint
// when the ratio is below 0.1 or above 0.9. The edge length and the interpolation round every
// operation as the reference does.
template <class R> struct Edge {
    R v1[4], v2[4], d;
    int nev = 0;
    __device__ __forceinline__ void load(const double* ends, int64_t i) {
#pragma clang fp contract(off)
        for (int a = 0; a < 4; a++) {
            v1[a] = R(ends[8 * i + a]);
            v2[a] = R(ends[8 * i + 4 + a]);
        }
        const R ex = v1[0] - v2[0], ey = v1[1] - v2[1], ez = v1[2] - v2[2];
        const R e2 = ex * ex + ey * ey + ez * ez;
        d = (sizeof(R) == 4) ? R(__builtin_sqrtf(float(e2))) : R(sqrt(double(e2)));
    }
    // (the reference loop has no cap; 256 halvings bound it for any finite input)
    __device__ __forceinline__ bool open(float half_r) const { return nev < 256 && d > R(half_r); }
    __device__ __forceinline__ void middle(R m[4]) const {
        for (int a = 0; a < 3; a++) m[a] = (v1[a] + v2[a]) / R(2);
    }
    __device__ __forceinline__ void step(R m[4], R iso, R sigma, R sum) {
#pragma clang fp contract(off)
        nev++;
        m[3] = iso - sigma * sum;
        const int sm = m[3] > R(0) ? 1 : -1, s1 = v1[3] > R(0) ? 1 : -1;
        if (sm == s1)
            for (int a = 0; a < 4; a++) v1[a] = m[a];
        else
            for (int a = 0; a < 4; a++) v2[a] = m[a];
        d /= R(2);
    }
    __device__ __forceinline__ void store(double* out, int64_t i) const {
#pragma clang fp contract(off)
        const R ratio = (R(0) - v1[3]) / (v2[3] - v1[3]);
        R o[3];
        if (ratio < R(0.1))
            for (int a = 0; a < 3; a++) o[a] = v1[a];
        else if (ratio > R(0.9))
            for (int a = 0; a < 3; a++) o[a] = v2[a];
        else
            for (int a = 0; a < 3; a++) o[a] = v1[a] + (v2[a] - v1[a]) * ratio;
        for (int a = 0; a < 3; a++) out[3 * i + a] = double(o[a]);
    }
};

// One thread per edge
template <class R, bool K, int MODE>
__global__ void __launch_bounds__(256) k_bisect(GridDev g, Recs<R> rec, FieldConst fc, float half_r,
                                                const double* __restrict__ ends, int64_t n, double* __restrict__ out,
                                                int* __restrict__ nev_out, Counters* ctr) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int vis = 0;
    Edge<R> e;
    if (i < n) {
        e.load(ends, i);
        while (e.open(half_r)) {
            R m[4], sum, g3[3];
            e.middle(m);
            vis += field_sum<R, K, false, MODE, true>(g, rec, fc, float(m[0]), float(m[1]), float(m[2]), m[0], m[1],
                                                      m[2], sum, g3);
            e.step(m, R(fc.iso), out_sigma<R, K>(fc), sum);
        }
        e.store(out, i);
        if (nev_out) nev_out[i] = e.nev;
    }
    wave_count(&ctr_stripe(ctr)->field_evals, (unsigned long long)e.nev);
    wave_count(&ctr_stripe(ctr)->candidates, (unsigned long long)vis);
}

// A wave per m edges, for few edges: lane k holds edge k and the wave sums the open edges' midpoints one after another
// (point_eval.h). A thread per edge sums two or three midpoints' 200 candidates in a chain of dependent reads
// that takes 115 us for the 16 k edges of a 14 k-particle frame (FP32); this way it is 42 us. With the chip full of
// edges a thread per edge is ahead: 202 k edges in FP64 0.22 against 0.44 ms. (64 edges to a wave in mesh order
// share too few windows: 1.27 -> 1.45 ms for 1.75 M edges.)
template <class R> struct EdgeSrc {
    const R* m;  // this lane's midpoint
    bool open;
    int64_t i0;
    R* sum;
    __device__ __forceinline__ bool point(int64_t i, R p[3]) const {
        const int k = (int)(i - i0);
        if (!((__ballot(open) >> k) & 1)) return false;
        for (int a = 0; a < 3; a++) p[a] = __shfl(m[a], k, kWave);
        return true;
    }
    __device__ __forceinline__ void store(int64_t, int, R v) const { *sum = v; }
};
template <class R, bool K, int MODE>
__global__ void __launch_bounds__(256) k_point_bisect(GridDev g, Recs<R> rec, FieldConst fc, float half_r,
                                                      const double* __restrict__ ends, int64_t n, int m,
                                                      double* __restrict__ out, int* __restrict__ nev_out,
                                                      Counters* ctr) {
    __shared__ PointLds<R, false> lds[4];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int64_t i0 = ((int64_t)blockIdx.x * 4 + w) * m, i = i0 + lane;
    const int np = (int)max((int64_t)0, min((int64_t)m, n - i0));
    unsigned long long vis = 0;
    int evals = 0;
    Edge<R> e;
    if (lane < np) e.load(ends, i);
    for (bool open = lane < np && e.open(half_r); __any(open); open = open && e.open(half_r)) {
        R mid[4] = {R(0), R(0), R(0), R(0)}, sum = R(0);
        if (open) e.middle(mid);
        vis += point_eval<R, K, false, MODE>(g, rec, fc, EdgeSrc<R>{mid, open, i0, &sum}, i0, np, lds[w], evals);
        if (open) e.step(mid, R(fc.iso), out_sigma<R, K>(fc), sum);
    }
    if (lane < np) {
        e.store(out, i);
        if (nev_out) nev_out[i] = e.nev;
    }
    if (lane == 0 && evals > 0) {
        Counters* c = ctr_stripe(ctr);
        atomicAdd(&c->field_evals, (unsigned long long)evals);
        atomicAdd(&c->candidates, vis);
    }
}

constexpr int64_t kPointEdges = 1 << 16;
void launch_bisect(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, float half_r, const double* ends,
                   int64_t n, double* out, int* nev, Counters* ctr, hipStream_t s) {
    if (n <= 0) return;
    const unsigned nb = (unsigned)((n + 255) / 256);
    const int m = point_share(n, points_per_wave(prec == 2, false));
    auto go = [&](auto mode) {
        constexpr int M = decltype(mode)::value;
        if (n < kPointEdges) {
            const unsigned np = (unsigned)((n + 4 * m - 1) / (4 * m));
            if (prec == 2) {
                Recs<double> r{(const double4*)ra, (const double4*)rg};
                k_point_bisect<double, false, M><<<np, 256, 0, s>>>(g, r, fc, half_r, ends, n, m, out, nev, ctr);
            } else {
                Recs<float> r{(const float4*)ra, (const float4*)rg};
                if (prec == 1)
                    k_point_bisect<float, true, M><<<np, 256, 0, s>>>(g, r, fc, half_r, ends, n, m, out, nev, ctr);
                else k_point_bisect<float, false, M><<<np, 256, 0, s>>>(g, r, fc, half_r, ends, n, m, out, nev, ctr);
            }
            return;
        }
        if (prec == 2) {
            Recs<double> r{(const double4*)ra, (const double4*)rg};
            k_bisect<double, false, M><<<nb, 256, 0, s>>>(g, r, fc, half_r, ends, n, out, nev, ctr);
        } else {
            Recs<float> r{(const float4*)ra, (const float4*)rg};
            if (prec == 1) k_bisect<float, true, M><<<nb, 256, 0, s>>>(g, r, fc, half_r, ends, n, out, nev, ctr);
            else k_bisect<float, false, M><<<nb, 256, 0, s>>>(g, r, fc, half_r, ends, n, out, nev, ctr);
        }
    };
    if (field_mode(fc) == kModeAniBspline) go(std::integral_constant<int, kModeAniBspline>());
    else go(std::integral_constant<int, kModeAny>());
}

// Standalone QEF over given samples (n x 27 x 4) and gradients (n x 27 x 3).
template <class R, bool K>
__global__ void __launch_bounds__(64) k_qef(GridDev g, Recs<R> rec, FieldConst fc, TreeParams tp,
                                            const float4* __restrict__ cen, const double* __restrict__ samples,
                                            const double* __restrict__ grads, int64_t n, int mode,
                                            double4* __restrict__ out, Counters* ctr) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int vis = 0;
    if (i < n) {
        const float4 c = cen[i];
        float pts[27][3];
        R f[27], gr[27][3];
        for (int s = 0; s < 27; s++) {
            for (int a = 0; a < 3; a++) {
                pts[s][a] = float(samples[(i * 27 + s) * 4 + a]);
                gr[s][a] = R(grads[(i * 27 + s) * 3 + a]);
            }
            f[s] = R(samples[(i * 27 + s) * 4 + 3]);
        }
        R pc[4], err;
        R vx = R(c.x), vy = R(c.y), vz = R(c.z);
        if (qef_solve<R>(c, pts, f, gr, mode, tp.qef_svd_tol, pc, err)) {
            vx = pc[0];
            vy = pc[1];
            vz = pc[2];
        }
        R sum, g3[3];
        vis = field_sum<R, K, false>(g, rec, fc, float(vx), float(vy), float(vz), vx, vy, vz, sum, g3);
        R fv = field_value(R(fc.iso), out_sigma<R, K>(fc), sum);
        if (err / R(__fmul_rn(2.0f, c.w)) < R(0.0001)) fv = R(0);
        out[i] = make_double4(double(vx), double(vy), double(vz), double(fv));
    }
    wave_count(&ctr_stripe(ctr)->qef_solves, i < n ? 1ull : 0ull);
    wave_count(&ctr_stripe(ctr)->field_evals, i < n ? 1ull : 0ull);
    wave_count(&ctr_stripe(ctr)->candidates, (unsigned long long)vis);
}

void launch_qef(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, TreeParams tp, const float4* cen,
                const double* samples, const double* grads, int64_t n, int mode, double4* out, Counters* ctr,
                hipStream_t s) {
    if (n <= 0) return;
    const unsigned nb = (unsigned)((n + 63) / 64);
    if (prec == 2) {
        Recs<double> r{(const double4*)ra, (const double4*)rg};
        k_qef<double, false><<<nb, 64, 0, s>>>(g, r, fc, tp, cen, samples, grads, n, mode, out, ctr);
    } else {
        Recs<float> r{(const float4*)ra, (const float4*)rg};
        if (prec == 1) k_qef<float, true><<<nb, 64, 0, s>>>(g, r, fc, tp, cen, samples, grads, n, mode, out, ctr);
        else k_qef<float, false><<<nb, 64, 0, s>>>(g, r, fc, tp, cen, samples, grads, n, mode, out, ctr);
    }
}

}  // namespace pisurf
