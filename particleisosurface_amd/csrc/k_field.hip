// Field evaluation at arbitrary points (Evaluator::SingleEval / SingleEvalWithGrad,
// src/evaluator.cpp:60-125) and particle normals (CalcParticlesNormal, :363-375).
#include "pisurf_internal.h"
#include "point_eval.h"
#include "run_eval.h"
#include "run_tuner.h"
#include "wave_eval.h"

#include <cmath>
#include <type_traits>

namespace pisurf {

// SingleEval / SingleEvalWithGrad, a wave per m points
template <class R> struct PointSrc {
    const float* q;
    double* f;
    double* grad;
    R iso, sigma;
    __device__ __forceinline__ bool point(int64_t i, R p[3]) const {
        for (int a = 0; a < 3; a++) p[a] = R(q[3 * i + a]);
        return true;
    }
    __device__ __forceinline__ void store(int64_t i, int c, R v) const {
        if (c == 0) f[i] = double(field_value(iso, sigma, v));
        else grad[3 * i + c - 1] = double(sigma * v);
    }
};
template <class R, bool K, bool GRAD, int MODE>
__global__ void __launch_bounds__(256) k_eval_points(GridDev g, Recs<R> rec, FieldConst fc, const float* __restrict__ q,
                                                     int64_t n, int m, double* __restrict__ f,
                                                     double* __restrict__ grad, Counters* ctr) {
    __shared__ PointLds<R, GRAD> lds[4];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int64_t i0 = ((int64_t)blockIdx.x * 4 + w) * m;
    const int np = (int)max((int64_t)0, min((int64_t)m, n - i0));
    const PointSrc<R> src{q, f, grad, R(fc.iso), out_sigma<R, K>(fc)};
    int evals = 0;
    const unsigned long long vis = point_eval<R, K, GRAD, MODE>(g, rec, fc, src, i0, np, lds[w], evals);
    Counters* ct = ctr_stripe(ctr);
    if (lane == 0 && np > 0) {
        atomicAdd(GRAD ? &ct->grad_evals : &ct->field_evals, (unsigned long long)np);
        atomicAdd(&ct->candidates, vis);
    }
}

// per-particle form for grids that leave particles outside (shifted cell windows, no runs)
template <class R, bool K>
__global__ void __launch_bounds__(256) k_normals_pt(GridDev g, Recs<R> rec, FieldConst fc, const float4* __restrict__ spos,
                                                 int64_t n, float4* __restrict__ nrm, Counters* ctr) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int vis = 0;
    if (p < n) {
        const float4 pp = spos[p];
        R s, gr[3];
        vis = field_sum<R, K, true>(g, rec, fc, pp.x, pp.y, pp.z, R(pp.x), R(pp.y), R(pp.z), s, gr);
        const R sigma = out_sigma<R, K>(fc);
        nrm[p] = make_float4(float(sigma * gr[0]), float(sigma * gr[1]), float(sigma * gr[2]), 0.0f);
    }
    wave_count(&ctr_stripe(ctr)->grad_evals, p < n ? 1ull : 0ull);
    wave_count(&ctr_stripe(ctr)->candidates, (unsigned long long)vis);
}

// CalcParticlesNormal over runs: the particles of kx consecutive cells of one (y, z) row of the
// grid (their sorted range is contiguous), candidates staged through LDS
template <class R> struct ParticleSrc {
    const float4* spos;
    float4* nrm;
    R sigma;
    __device__ __forceinline__ void point(int h, float p[3]) const {
        const float4 q = spos[h];
        p[0] = q.x;
        p[1] = q.y;
        p[2] = q.z;
    }
    __device__ __forceinline__ void store(int h, R, const R* gr) const {
        nrm[h] = make_float4(float(sigma * gr[0]), float(sigma * gr[1]), float(sigma * gr[2]), 0.0f);
    }
};

template <class R, bool K, int T, int MODE>
__global__ void __launch_bounds__(T) k_run_normals(GridDev g, Recs<R> rec, FieldConst fc,
                                                   const float4* __restrict__ spos, int kx,
                                                   const uint8_t* __restrict__ mark, bool count,
                                                   float4* __restrict__ nrm, Counters* ctr) {
    __shared__ RunLds<R, K && sizeof(R) == 4> lds;
    int h0, h1;
    const int cell = particle_run(g, kx, h0, h1);
    if (h0 >= h1) return;  // uniform over the block
    // (the count is the reference's, which takes every particle's normal)
    if (count && threadIdx.x == 0) atomicAdd(&ctr_stripe(ctr)->grad_evals, (unsigned long long)(h1 - h0));
    if (mark) {
        const int nc = min(kx, g.n[0] - cell % g.n[0]);
        bool any = false;
        for (int x = threadIdx.x; x < nc; x += T) any = any || mark[cell + x] == 1;
        if (!__syncthreads_or(any)) return;
    }
    ParticleSrc<R> src{spos, nrm, out_sigma<R, K>(fc)};
    const unsigned long long vis = run_eval<T, R, K, true, MODE>(g, rec, fc, src, h0, h1, lds);
    wave_count(&ctr_stripe(ctr)->candidates, vis);
}

void launch_eval_points(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, const float* q, int64_t n,
                        double* f, double* grad, Counters* ctr, hipStream_t s) {
    if (n <= 0) return;
    const int m = point_share(n, points_per_wave(prec == 2, grad != nullptr));
    // 8 or 16 threads a point, and a launch holds fewer than 2^32: slices of 2^27 points (a multiple of a workgroup's 4 m)
    constexpr int64_t kSlice = int64_t(1) << 27;
    auto go = [&](auto gr, auto mode) {
        constexpr bool G = decltype(gr)::value;
        constexpr int M = decltype(mode)::value;
        for (int64_t i = 0; i < n; i += kSlice) {
            const int64_t k = std::min(kSlice, n - i);
            const unsigned nb = (unsigned)((k + 4 * m - 1) / (4 * m));
            const float* qi = q + 3 * i;
            double* fi = f + i;
            double* gi = grad ? grad + 3 * i : nullptr;
            if (prec == 2) {
                Recs<double> r{(const double4*)ra, (const double4*)rg};
                k_eval_points<double, false, G, M><<<nb, 256, 0, s>>>(g, r, fc, qi, k, m, fi, gi, ctr);
            } else {
                Recs<float> r{(const float4*)ra, (const float4*)rg};
                if (prec == 1) k_eval_points<float, true, G, M><<<nb, 256, 0, s>>>(g, r, fc, qi, k, m, fi, gi, ctr);
                else k_eval_points<float, false, G, M><<<nb, 256, 0, s>>>(g, r, fc, qi, k, m, fi, gi, ctr);
            }
        }
    };
    point_dispatch(field_mode(fc), [&](auto mode) {
        if (grad) go(std::true_type(), mode);
        else go(std::false_type(), mode);
    });
}

// Many points: sorted by hash cell, then 64 to a wave (wave_eval.h)
__global__ void k_point_keys(GridDev g, const float* __restrict__ q, int64_t n, int vbits, uint64_t* __restrict__ key,
                             int* __restrict__ val) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t k = cell_group(g, q[3 * i], q[3 * i + 1], q[3 * i + 2]);
    if (vbits) {
        key[i] = (k << vbits) | (uint64_t)i;
    } else {
        key[i] = k;
        val[i] = (int)i;
    }
}
template <class R> struct QuerySrc {
    const float* q;
    SortedKV kv;
    double* f;
    double* grad;
    R iso, sigma;
    __device__ __forceinline__ bool point(int h, float p[3]) const {
        const float* x = q + 3 * (int64_t)kv.val(h);
        p[0] = x[0];
        p[1] = x[1];
        p[2] = x[2];
        return true;
    }
    __device__ __forceinline__ void store(int h, R sum, const R* gr) const {
        const int64_t i = kv.val(h);
        f[i] = double(field_value(iso, sigma, sum));
        if (grad)
            for (int a = 0; a < 3; a++) grad[3 * i + a] = double(sigma * gr[a]);
    }
};
template <class R, bool K, bool GRAD, int T, int MODE>
__global__ void __launch_bounds__(T) k_wave_points(GridDev g, Recs<R> rec, FieldConst fc, const float* __restrict__ q,
                                                   SortedKV kv, int n, double* __restrict__ f,
                                                   double* __restrict__ grad, Counters* ctr) {
    __shared__ WaveLds<WaveField<R, K, GRAD, MODE>> lds[T / kWave];
    const QuerySrc<R> src{q, kv, f, GRAD ? grad : nullptr, R(fc.iso), out_sigma<R, K>(fc)};
    const int vis = wave_eval<T, R, K, GRAD, MODE>(g, rec, fc, src, n, lds);
    Counters* c = ctr_stripe(ctr);
    wave_count(&c->candidates, (unsigned long long)vis);
    if (threadIdx.x == 0)
        atomicAdd(GRAD ? &c->grad_evals : &c->field_evals, (unsigned long long)min(T, n - (int)blockIdx.x * T));
}

// Sorting costs about 0.1 ms per million points and a dozen launches, and pays in shared windows: from 2^18 points and
// a point for four particles on (particles at rest lie 8 to a cell: two points to a cell of the fluid). 1 M
// shuffled points with gradients on 1.6 M particles, compensated FP32: 0.60 ms sorted, 1.16 ms a wave per
// eight points, 2.2 ms a thread per point; 70 k points on 200 k particles: the whole call takes 0.43 ms sorted
// and 0.30 ms unsorted; from 200 k to 500 k points the two are within 5 %.
bool eval_points_sorts(int64_t n, int64_t particles) {
    return n >= (1 << 18) && n < (1 << 30) && 4 * n >= particles;
}
void launch_eval_points_sorted(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, const float* q,
                               int64_t n, double* f, double* grad, uint64_t* key, int* val, uint64_t* key2, int* val2,
                               int* tmp, Counters* ctr, hipStream_t s) {
    const int bits = cell_group_bits(g), vbits = pack_vbits(bits, n);
    k_point_keys<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(g, q, n, vbits, key, val);
    const SortedKV kv = radix_sort_entries(key, val, key2, val2, n, bits, vbits, tmp, s);
    constexpr int T = 128;
    const unsigned nb = (unsigned)((n + T - 1) / T);
    auto go = [&](auto gr, auto mode) {
        constexpr bool G = decltype(gr)::value;
        constexpr int M = decltype(mode)::value;
        if (prec == 2) {
            Recs<double> r{(const double4*)ra, (const double4*)rg};
            k_wave_points<double, false, G, T, M><<<nb, T, 0, s>>>(g, r, fc, q, kv, (int)n, f, grad, ctr);
        } else {
            Recs<float> r{(const float4*)ra, (const float4*)rg};
            if (prec == 1) k_wave_points<float, true, G, T, M><<<nb, T, 0, s>>>(g, r, fc, q, kv, (int)n, f, grad, ctr);
            else k_wave_points<float, false, G, T, M><<<nb, T, 0, s>>>(g, r, fc, q, kv, (int)n, f, grad, ctr);
        }
    };
    auto with = [&](auto gr) {
        if (field_mode(fc) == kModeAniBspline) go(gr, std::integral_constant<int, kModeAniBspline>());
        else go(gr, std::integral_constant<int, kModeAny>());
    };
    if (grad) with(std::true_type());
    else with(std::false_type());
}

void launch_normals(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, const float4* spos, int64_t n,
                    int64_t n_invalid, const uint8_t* mark, bool count, float4* nrm, Counters* ctr,
                    Counters* trial_ctr, hipStream_t s) {
    if (n <= 0) return;
    if (n_invalid > 0) {
        const unsigned nb = (unsigned)((n + 255) / 256);
        if (prec == 2) {
            Recs<double> r{(const double4*)ra, (const double4*)rg};
            k_normals_pt<double, false><<<nb, 256, 0, s>>>(g, r, fc, spos, n, nrm, ctr);
        } else {
            Recs<float> r{(const float4*)ra, (const float4*)rg};
            if (prec == 1) k_normals_pt<float, true><<<nb, 256, 0, s>>>(g, r, fc, spos, n, nrm, ctr);
            else k_normals_pt<float, false><<<nb, 256, 0, s>>>(g, r, fc, spos, n, nrm, ctr);
        }
        return;
    }
    // runs of kx cells of a grid row, one workgroup each (empty runs end at once); the shape is
    // tuned per precision and average particles per cell
    const double p = (double)n / std::max<int64_t>((int64_t)g.n[0] * g.n[1] * g.n[2], 1);
    tuned_run_launch(
        prec, mark ? kRunMarkedNormals : kRunNormals, p, false, trial_ctr, s,
        [&](RunShape c) { return (int64_t)((g.n[0] + c.kx - 1) / c.kx) * g.n[1] * g.n[2] <= INT32_MAX; },
        [&](RunShape c, bool trial) {
            Counters* cc = trial ? trial_ctr : ctr;
            const unsigned nb = (unsigned)((int64_t)((g.n[0] + c.kx - 1) / c.kx) * g.n[1] * g.n[2]);
            auto go = [&](auto tag, auto mode) {
                constexpr int TT = decltype(tag)::value, M = decltype(mode)::value;
                if (prec == 2) {
                    Recs<double> r{(const double4*)ra, (const double4*)rg};
                    k_run_normals<double, false, TT, M><<<nb, TT, 0, s>>>(g, r, fc, spos, c.kx, mark, count, nrm, cc);
                } else {
                    Recs<float> r{(const float4*)ra, (const float4*)rg};
                    if (prec == 1) k_run_normals<float, true, TT, M><<<nb, TT, 0, s>>>(g, r, fc, spos, c.kx, mark, count, nrm, cc);
                    else k_run_normals<float, false, TT, M><<<nb, TT, 0, s>>>(g, r, fc, spos, c.kx, mark, count, nrm, cc);
                }
            };
            using M0 = std::integral_constant<int, kModeAny>;
            using M1 = std::integral_constant<int, kModeAniBspline>;
            const bool m1 = field_mode(fc) == kModeAniBspline;
            if (c.T == 256) m1 ? go(std::integral_constant<int, 256>(), M1()) : go(std::integral_constant<int, 256>(), M0());
            else m1 ? go(std::integral_constant<int, 128>(), M1()) : go(std::integral_constant<int, 128>(), M0());
        });
}

// UniformGrid::gridSampling (src/marching.cpp:72-91): point i = x + dims0 * (y + dims1 * z) at
// float(steps - x) / float(steps) * min + float(x) / float(steps) * max per axis, each operation
// rounded on its own (the reference is built without FMA contraction)
__device__ __forceinline__ void lattice_point(const UniformBox& ub, const int ix[3], float p[3]) {
#pragma unroll
    for (int a = 0; a < 3; a++) {
        // plain operators with contraction off in this scope: the *_rn helpers are inlined as
        // contractable operations, and a fused product would round differently
#pragma clang fp contract(off)
        const float st = (float)ub.steps[a];
        const float u = (float)(ub.steps[a] - ix[a]) / st;
        const float v = (float)ix[a] / st;
        p[a] = u * ub.lo[a] + v * ub.hi[a];
    }
}

// One thread per point, for hash cells too small to hold several
template <class R, bool K>
__global__ void __launch_bounds__(256) k_uniform_grid(GridDev g, Recs<R> rec, FieldConst fc, UniformBox ub,
                                                      int64_t total, float* __restrict__ out, Counters* ctr) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int vis = 0;
    if (i < total) {
        const int64_t plane = (int64_t)ub.dims[0] * ub.dims[1];
        const int z = (int)(i / plane);
        const int64_t rem = i - (int64_t)z * plane;
        const int y = (int)(rem / ub.dims[0]);
        const int ix[3] = {(int)(rem - (int64_t)y * ub.dims[0]), y, z};
        float p[3];
        lattice_point(ub, ix, p);
        R s, gr[3];
        vis = field_sum<R, K, false>(g, rec, fc, p[0], p[1], p[2], R(p[0]), R(p[1]), R(p[2]), s, gr);
        out[i] = float(field_value(R(fc.iso), out_sigma<R, K>(fc), s));
    }
    wave_count(&ctr_stripe(ctr)->field_evals, i < total ? 1ull : 0ull);
    wave_count(&ctr_stripe(ctr)->candidates, (unsigned long long)vis);
}

// A wave per block of 4 x 4 x 4 points. The lattice has four points to a hash cell's width (spacing r, cells of 4 r), and
// the blocks start where cells do (shift), so a wave's points nearly always share one window: 216 candidates staged
// and tested once for 64 points (wave_eval.h). Four blocks side by side along x per workgroup.
// 2 M points around 120 k particles, FP32: 260 us, a thread per point 426.
struct LatticeBlocks {
    int shift[3];  // points of the first block along an axis that lie before the lattice
    int n[3];      // blocks (x: groups of four)
};
template <class R, bool K, int MODE>
__global__ void __launch_bounds__(256) k_wave_lattice(GridDev g, Recs<R> rec, FieldConst fc, UniformBox ub,
                                                      LatticeBlocks lb, float* __restrict__ out, Counters* ctr) {
    __shared__ WaveLds<WaveField<R, K, false, MODE>> lds[4];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int b = blockIdx.x, bx = b % lb.n[0], by = (b / lb.n[0]) % lb.n[1], bz = b / lb.n[0] / lb.n[1];
    const int ix[3] = {16 * bx + 4 * w + (lane & 3) - lb.shift[0], 4 * by + ((lane >> 2) & 3) - lb.shift[1],
                       4 * bz + (lane >> 4) - lb.shift[2]};
    bool act = true;
#pragma unroll
    for (int a = 0; a < 3; a++) act = act && ix[a] >= 0 && ix[a] < ub.dims[a];
    float p[3] = {0.f, 0.f, 0.f};
    if (act) lattice_point(ub, ix, p);
    const R q[3] = {R(p[0]), R(p[1]), R(p[2])};
    R sum;
    const int vis = wave_sum<R, K, MODE>(g, rec, fc, act, q, lds[w], sum);
    if (act)
        out[((int64_t)ix[2] * ub.dims[1] + ix[1]) * ub.dims[0] + ix[0]] =
            float(field_value(R(fc.iso), out_sigma<R, K>(fc), sum));
    wave_count(&ctr_stripe(ctr)->field_evals, act ? 1ull : 0ull);
    wave_count(&ctr_stripe(ctr)->candidates, (unsigned long long)vis);
}

void launch_uniform_grid(int prec, GridDev g, const void* ra, const void* rg, FieldConst fc, UniformBox ub,
                         int64_t total, float* out, Counters* ctr, hipStream_t s) {
    if (total <= 0) return;
    LatticeBlocks lb;
    double per_cell = 1;
    int64_t blocks = 1;
    for (int a = 0; a < 3; a++) {
        const double h = ((double)ub.hi[a] - ub.lo[a]) / ub.steps[a];
        per_cell *= g.cell / h;
        const double at = ((double)g.b0[a] - ub.lo[a]) / h;  // lattice position of a cell's first point, modulo 4
        const double first = std::ceil(at - 4 * std::floor(at / 4) - 1e-3);
        lb.shift[a] = std::isfinite(first) ? (4 - (int)first) & 3 : 0;
        const int width = a == 0 ? 16 : 4;
        lb.n[a] = (ub.dims[a] + lb.shift[a] + width - 1) / width;
        blocks *= lb.n[a];
    }
    // (cells of another size: 64 points in more than 16 cells share too little; a sheet fills as little as a third
    // of its blocks, and a launch holds fewer than 2^32 threads)
    const bool waves = per_cell >= kWaveDensity && blocks < (1 << 24);
    const unsigned nb = (unsigned)((total + 255) / 256);
    auto go = [&](auto mode) {
        constexpr int M = decltype(mode)::value;
        if (prec == 2) {
            Recs<double> r{(const double4*)ra, (const double4*)rg};
            if (waves) k_wave_lattice<double, false, M><<<(unsigned)blocks, 256, 0, s>>>(g, r, fc, ub, lb, out, ctr);
            else k_uniform_grid<double, false><<<nb, 256, 0, s>>>(g, r, fc, ub, total, out, ctr);
        } else {
            Recs<float> r{(const float4*)ra, (const float4*)rg};
            if (prec == 1 && waves)
                k_wave_lattice<float, true, M><<<(unsigned)blocks, 256, 0, s>>>(g, r, fc, ub, lb, out, ctr);
            else if (prec == 1) k_uniform_grid<float, true><<<nb, 256, 0, s>>>(g, r, fc, ub, total, out, ctr);
            else if (waves) k_wave_lattice<float, false, M><<<(unsigned)blocks, 256, 0, s>>>(g, r, fc, ub, lb, out, ctr);
            else k_uniform_grid<float, false><<<nb, 256, 0, s>>>(g, r, fc, ub, total, out, ctr);
        }
    };
    point_dispatch(field_mode(fc), go);
}

}  // namespace pisurf
