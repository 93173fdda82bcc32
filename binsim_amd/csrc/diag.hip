// Davidson inner-loop kernels (libdiag on the GPU).
//
// Same entry points and arithmetic as src/include/diag/davidson.hpp:31-272 (C ABI
// src/include/diag/declare.hpp:4-75); state vectors are device pointers, the small arrays
// (Ritz coefficients, heff) stay on the host as in jl/davidson.jl.  Reductions are two-stage
// (per-block partials, then one block) so results are deterministic run to run.
#include "hipotf.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace hipotf {

constexpr int DMAX = 64;  // subspace cap, as local_V[64] in davidson.hpp:41-43

struct VecPack {
    const double *v[DMAX];
    double c[DMAX];
};

__device__ __forceinline__ double block_sum_d(double v) {
    __shared__ double red[16];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)((blockDim.x + 63) >> 6); ++i) t += red[i];
    return t;
}

static int nblk(i64 n) { return (int)std::max<i64>(1, std::min<i64>((n + 255) / 256, 2048)); }

// f(std::integral_constant<int, c>) for c = k in 1..8 (k > 8 -> 8)
template <typename F>
static void dispatch_m8(int k, F &&f) {
    switch (k) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    case 6: f(std::integral_constant<int, 6>{}); break;
    case 7: f(std::integral_constant<int, 7>{}); break;
    default: f(std::integral_constant<int, 8>{}); break;
    }
}

// Streaming kernels keep several independent loads in flight per thread: the vector loops load
// 4 vectors' elements before using them, the single-vector loops 4 elements (256 apart) per step.
constexpr int VU = 4;

// y = sum_j c_j V_j ; with RES: r = sum_j c_j AV_j - e y (written to y), partial |r|^2
// (the sum runs over j in order, as before the loads were batched)
template <bool RES>
__global__ __launch_bounds__(256) void k_combine(VecPack V, VecPack AV, int dim, double e, double *__restrict__ out,
                                                 double *__restrict__ partial, i64 n) {
    double acc = 0.0;
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        double x = 0.0, ax = 0.0;
        int j = 0;
        for (; j + VU <= dim; j += VU) {
            double xv[VU], av[VU];
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                xv[u] = V.v[j + u][i];
                if (RES) av[u] = AV.v[j + u][i];
            }
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                x += V.c[j + u] * xv[u];
                if (RES) ax += V.c[j + u] * av[u];
            }
        }
        for (; j < dim; ++j) {
            x += V.c[j] * V.v[j][i];
            if (RES) ax += V.c[j] * AV.v[j][i];
        }
        const double r = RES ? ax - e * x : x;
        out[i] = r;
        acc += r * r;
    }
    const double t = block_sum_d(acc);
    if (threadIdx.x == 0 && partial) partial[blockIdx.x] = t;
}

// Calls f(i) for every i < n, VU indices per thread and step: the full steps are unrolled so
// their loads issue together, the last partial step is checked per index.
template <typename F>
__device__ __forceinline__ void stream_for(i64 n, F &&f) {
    const i64 step = (i64)gridDim.x * blockDim.x * VU;
    for (i64 base = (i64)blockIdx.x * blockDim.x * VU + threadIdx.x; base < n; base += step) {
        if (base + (i64)(VU - 1) * blockDim.x < n) {
#pragma unroll
            for (int u = 0; u < VU; ++u) f(base + (i64)u * blockDim.x);
        } else {
            for (int u = 0; u < VU; ++u)
                if (base + (i64)u * blockDim.x < n) f(base + (i64)u * blockDim.x);
        }
    }
}

__global__ __launch_bounds__(256) void k_reduce(const double *__restrict__ partial, int n,
                                                double *__restrict__ out, int mode) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
    const double t = block_sum_d(acc);
    if (threadIdx.x == 0) *out = mode == 1 ? sqrt(t) : t;
}

__global__ __launch_bounds__(256) void k_precond(double *__restrict__ axt, const double *__restrict__ diags,
                                                 double e, double shift, i64 n) {
    const double as = fabs(shift);
    stream_for(n, [&](i64 i) {
        double d = diags[i] - e;
        if (fabs(d) < as) d = d >= 0 ? as : -as;
        axt[i] = axt[i] / d;
    });
}

__global__ __launch_bounds__(256) void k_dotp(const double *__restrict__ a, const double *__restrict__ b,
                                              double *__restrict__ partial, i64 n) {
    double acc = 0.0;
    stream_for(n, [&](i64 i) { acc += a[i] * b[i]; });
    const double t = block_sum_d(acc);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// One modified Gram-Schmidt step in one pass: y -= p x, with p the sum of the nin partials of the
// step before (added by every workgroup in the order k_reduce adds them), then the partials of
// z . y (NORM: y . y) for the next; the rounding of every operation is that of a dot, a sum and a
// subtraction done one after the other.  Those moved five vectors per step in three launches, this
// moves four in one, at 6.2 TB/s (x was the z of the step before, and partly still in the Infinity
// Cache): 20 steps on 10.3M elements 1.34 -> 1.07 ms.  z may be y itself (a subspace that holds the
// vector): then, as everywhere, its new values count.
template <bool NORM>
__global__ __launch_bounds__(256) void k_mgs_step(double *__restrict__ y, const double *__restrict__ x,
                                                  const double *__restrict__ z, const double *__restrict__ pin,
                                                  int nin, double *__restrict__ pout, i64 n) {
    __shared__ double ps;
    double s = 0.0;
    for (int i = threadIdx.x; i < nin; i += blockDim.x) s += pin[i];
    s = block_sum_d(s);
    if (threadIdx.x == 0) ps = s;
    __syncthreads();
    const double p = ps;
    const bool own = NORM || z == y;
    double acc = 0.0;
    stream_for(n, [&](i64 i) {
        const double zv = NORM ? 0.0 : z[i], v = y[i] - p * x[i];
        y[i] = v;
        acc += (own ? v : zv) * v;
    });
    const double t = block_sum_d(acc);
    if (threadIdx.x == 0) pout[blockIdx.x] = t;
}

// y *= s
__global__ __launch_bounds__(256) void k_scale(double *__restrict__ y, double s, i64 n) {
    stream_for(n, [&](i64 i) { y[i] *= s; });
}

// y *= 1 / *nrm
__global__ __launch_bounds__(256) void k_scale_inv(double *__restrict__ y, const double *__restrict__ nrm,
                                                   i64 n) {
    const double s = 1.0 / *nrm;
    stream_for(n, [&](i64 i) { y[i] *= s; });
}

struct DiagScratch {
    DevBuf partial, scal;
    DiagScratch() {
        partial.alloc(8 * 2048 * sizeof(double));
        scal.alloc(128 * sizeof(double));
    }
};

static DiagScratch &scratch() {
    static thread_local std::unique_ptr<DiagScratch> s;
    if (!s) s.reset(new DiagScratch());
    return *s;
}

static double d2h(const double *d, hipStream_t st) {
    double h = 0.0;
    HIPOTF_CHECK(hipMemcpyAsync(&h, d, sizeof(double), hipMemcpyDeviceToHost, st));
    HIPOTF_CHECK(hipStreamSynchronize(st));
    return h;
}

static void pack(VecPack &P, const double *const *V, const double *coeffs, int dim) {
    HIPOTF_REQUIRE(dim >= 0 && dim <= DMAX, "subspace dimension must be in [0, 64]");
    for (int j = 0; j < dim; ++j) {
        HIPOTF_REQUIRE(V[j] != nullptr, "NULL subspace vector");
        P.v[j] = V[j];
        P.c[j] = coeffs ? coeffs[j] : 0.0;
    }
}

double ritz_and_residual(i64 N, int dim, const double *coeffs, double min_e, const double *const *V,
                         const double *const *AV, double *axt, hipStream_t st) {
    VecPack P{}, Q{};
    pack(P, V, coeffs, dim);
    pack(Q, AV, coeffs, dim);
    auto &S = scratch();
    const int nb = nblk(N);
    hipLaunchKernelGGL(k_combine<true>, dim3(nb), dim3(256), 0, st, P, Q, dim, min_e, axt,
                       S.partial.as<double>(), N);
    HIPOTF_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, st, S.partial.as<double>(), N > 0 ? nb : 0,
                       S.scal.as<double>(), 1);
    HIPOTF_CHECK(hipGetLastError());
    return d2h(S.scal.as<double>(), st);
}

void ritz_vector(i64 N, int dim, const double *coeffs, const double *const *V, double *xt,
                 hipStream_t st) {
    VecPack P{}, Q{};
    pack(P, V, coeffs, dim);
    hipLaunchKernelGGL(k_combine<false>, dim3(nblk(N)), dim3(256), 0, st, P, Q, dim, 0.0, xt,
                       (double *)nullptr, N);
    HIPOTF_CHECK(hipGetLastError());
}

void precondition(i64 N, double *axt, const double *diags, double min_e, double shift, hipStream_t st) {
    hipLaunchKernelGGL(k_precond, dim3(nblk(N)), dim3(256), 0, st, axt, diags, min_e, shift, N);
    HIPOTF_CHECK(hipGetLastError());
}

// dot into device scalar dres
void dot_dev(i64 N, const double *a, const double *b, double *dres, hipStream_t st) {
    auto &S = scratch();
    const int nb = nblk(N);
    hipLaunchKernelGGL(k_dotp, dim3(nb), dim3(256), 0, st, a, b, S.partial.as<double>(), N);
    HIPOTF_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, st, S.partial.as<double>(), N > 0 ? nb : 0,
                       dres, 0);
    HIPOTF_CHECK(hipGetLastError());
}

double mgs(i64 N, int dim, const double *const *V, double *vt, hipStream_t st) {
    auto &S = scratch();
    for (int j = 0; j < dim; ++j) HIPOTF_REQUIRE(V[j] != nullptr, "NULL subspace vector");
    double *nrm = S.scal.as<double>() + 9;
    if (dim <= 0) {
        dot_dev(N, vt, vt, nrm, st);
        return std::sqrt(d2h(nrm, st));
    }
    const int nb = nblk(N);
    double *part[2] = {S.partial.as<double>(), S.partial.as<double>() + 2048};
    hipLaunchKernelGGL(k_dotp, dim3(nb), dim3(256), 0, st, V[0], vt, part[0], N);
    HIPOTF_CHECK(hipGetLastError());
    for (int j = 0; j < dim; ++j) {
        const double *pin = part[j & 1];
        double *pout = part[(j + 1) & 1];
        if (j + 1 < dim)
            hipLaunchKernelGGL(k_mgs_step<false>, dim3(nb), dim3(256), 0, st, vt, V[j], V[j + 1], pin, nb, pout, N);
        else
            hipLaunchKernelGGL(k_mgs_step<true>, dim3(nb), dim3(256), 0, st, vt, V[j], (const double *)nullptr, pin,
                               nb, pout, N);
        HIPOTF_CHECK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, st, part[dim & 1], N > 0 ? nb : 0, nrm, 0);
    HIPOTF_CHECK(hipGetLastError());
    return std::sqrt(d2h(nrm, st));
}

double normalize(i64 N, double *vec, hipStream_t st) {
    auto &S = scratch();
    const int nb = nblk(N);
    double *nrm = S.scal.as<double>() + 10;
    hipLaunchKernelGGL(k_dotp, dim3(nb), dim3(256), 0, st, vec, vec, S.partial.as<double>(), N);
    HIPOTF_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, st, S.partial.as<double>(), N > 0 ? nb : 0, nrm, 1);
    HIPOTF_CHECK(hipGetLastError());
    hipLaunchKernelGGL(k_scale_inv, dim3(nb), dim3(256), 0, st, vec, nrm, N);
    HIPOTF_CHECK(hipGetLastError());
    return d2h(nrm, st);  // (waits for the scaling too)
}

// vec /= nrm for a norm the caller already has (mgs returns it): no further dot product or wait
void scale_inv(i64 N, double *vec, double nrm, hipStream_t st) {
    hipLaunchKernelGGL(k_scale, dim3(nblk(N)), dim3(256), 0, st, vec, 1.0 / nrm, N);
    HIPOTF_CHECK(hipGetLastError());
}

// out[j] = |T_j|, j < k <= 8, with one synchronisation
void norms(i64 N, int k, double *const *T, double *out, hipStream_t st) {
    HIPOTF_REQUIRE(k >= 0 && k <= 8, "norms: at most 8 vectors");
    if (k == 0) return;
    auto &S = scratch();
    double *d = S.scal.as<double>() + 16;
    for (int j = 0; j < k; ++j) dot_dev(N, T[j], T[j], d + j, st);
    double h[8];
    HIPOTF_CHECK(hipMemcpyAsync(h, d, k * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPOTF_CHECK(hipStreamSynchronize(st));
    for (int j = 0; j < k; ++j) out[j] = std::sqrt(h[j]);
}

double dot(i64 N, const double *a, const double *b, hipStream_t st) {
    auto &S = scratch();
    double *d = S.scal.as<double>() + 12;
    dot_dev(N, a, b, d, st);
    return d2h(d, st);
}

void block_dots(i64 N, int na, const double *const *A, int nbv, const double *const *B, double *G, hipStream_t st);
// out[j] = <V_j, a>, j < dim (any number), written to host memory
void multidot(i64 N, int dim, const double *const *V, const double *a, double *out_host, hipStream_t st) {
    HIPOTF_REQUIRE(dim >= 0, "subspace dimension must not be negative");
    for (int j = 0; j < dim; ++j) HIPOTF_REQUIRE(V[j] != nullptr, "NULL subspace vector");
    for (int j = 0; j < dim; j += DMAX) block_dots(N, std::min(DMAX, dim - j), V + j, 1, &a, out_host + j, st);
}

// ------------------------------------------------------------------------------------------
// Block subspace operations of the mixed-precision block Davidson (no reference counterpart:
// jl/davidson.jl works one vector at a time).  Each reads every subspace vector once per call
// instead of once per (root, vector) pair; reductions stay two-stage and deterministic.
// ------------------------------------------------------------------------------------------
constexpr int BK = 8;  // outputs per launch
constexpr int DOT_BLOCKS = 1024;  // workgroups of the dot products

struct Ptr64 { const double *p[DMAX]; };
struct Out8 { double *p[BK]; };

// out_r = sum_j C[j*ldc + r] X_j  (r < nout <= BK); with Y: out_r = sum_j C[j*ldc+r] (Y_j - w_r X_j)
// and partial[r * nblk + b] = block sums of out_r^2
// (the sums run over j in order; the loads of VU vectors are issued together)
template <int KO, bool HY>
__global__ __launch_bounds__(256) void k_block_combo(Ptr64 X, Ptr64 Y, int m, const double *__restrict__ C, int ldc,
                                                     const double *__restrict__ w, Out8 out,
                                                     double *__restrict__ partial, i64 n) {
    double nrm[KO];
#pragma unroll
    for (int r = 0; r < KO; ++r) nrm[r] = 0.0;
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        double x[KO], y[KO];
#pragma unroll
        for (int r = 0; r < KO; ++r) x[r] = y[r] = 0.0;
        auto step = [&](int j, double xv, double yv) {
#pragma unroll
            for (int r = 0; r < KO; ++r) {
                const double c = C[j * ldc + r];
                x[r] += c * xv;
                if (HY) y[r] += c * yv;
            }
        };
        int j = 0;
        for (; j + VU <= m; j += VU) {
            double xv[VU], yv[VU];
#pragma unroll
            for (int u = 0; u < VU; ++u) {
                xv[u] = X.p[j + u][i];
                yv[u] = HY ? Y.p[j + u][i] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < VU; ++u) step(j + u, xv[u], yv[u]);
        }
        for (; j < m; ++j) step(j, X.p[j][i], HY ? Y.p[j][i] : 0.0);
#pragma unroll
        for (int r = 0; r < KO; ++r) {
            const double o = HY ? y[r] - w[r] * x[r] : x[r];
            out.p[r][i] = o;
            nrm[r] += o * o;
        }
    }
    if (partial) {
#pragma unroll
        for (int r = 0; r < KO; ++r) {
            const double t = block_sum_d(nrm[r]);
            if (threadIdx.x == 0) partial[r * gridDim.x + blockIdx.x] = t;
        }
    }
}

// T_j -= sum_i P[i*ldp + j] V_i   (j < nt <= BK, i < m <= DMAX)
template <int KO>
__global__ __launch_bounds__(256) void k_block_subtract(Ptr64 V, int m, const double *__restrict__ P, int ldp,
                                                        Out8 T, i64 n) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        double acc[KO];
#pragma unroll
        for (int r = 0; r < KO; ++r) acc[r] = 0.0;
        int j = 0;
        for (; j + VU <= m; j += VU) {
            double v[VU];
#pragma unroll
            for (int u = 0; u < VU; ++u) v[u] = V.p[j + u][i];
#pragma unroll
            for (int u = 0; u < VU; ++u)
#pragma unroll
                for (int r = 0; r < KO; ++r) acc[r] += P[(j + u) * ldp + r] * v[u];
        }
        for (; j < m; ++j) {
            const double v = V.p[j][i];
#pragma unroll
            for (int r = 0; r < KO; ++r) acc[r] += P[j * ldp + r] * v;
        }
#pragma unroll
        for (int r = 0; r < KO; ++r) T.p[r][i] -= acc[r];
    }
}

// Sums of A_a . B_b over the elements, for all a < na <= DMAX and NB vectors B in one pass: a thread
// holds DOT_EL elements of every B and streams the A through; per a, the wave adds its NB sums
// up with VALU moves (wave_sum4) into its own row of LDS, so no accumulator lives across vectors.
// (One launch per 8 x 4 sums re-read the B and added each sum up over the block with two barriers:
// 8 launches of 55 us at 854,000 elements, 64 x 4 sums, bound by those reductions.)  HBM bound:
// 8 N (na + NB) bytes.
// partial[(a * NB + b) * gridDim.x + block]
constexpr int DOT_THREADS = 256;
template <int NB>
constexpr int dot_el() { return NB <= 4 ? 8 : 4; }

// sums over the wave of four values: lanes 12..15 end with those of a[0..3]
__device__ __forceinline__ double dot_wave_sum4(const double (&a)[4]) {
    const int lane = threadIdx.x & 63;
    auto dpp = [](double v, auto ctrl) {
        constexpr int CT = decltype(ctrl)::value;
        const long long b = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CT, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CT, 0xf, 0xf, false);
        return __longlong_as_double(((long long)hi << 32) | (u32)lo);
    };
    const bool o1 = lane & 1, o2 = lane & 2;
    const double u = (o1 ? a[1] : a[0]) + dpp(o1 ? a[0] : a[1], std::integral_constant<int, 0xb1>{});
    const double v = (o1 ? a[3] : a[2]) + dpp(o1 ? a[2] : a[3], std::integral_constant<int, 0xb1>{});
    double w = (o2 ? v : u) + dpp(o2 ? u : v, std::integral_constant<int, 0x4e>{});
    w += dpp(w, std::integral_constant<int, 0x114>{});
    w += dpp(w, std::integral_constant<int, 0x118>{});
    w += __shfl_xor(w, 16, 64);
    w += __shfl_xor(w, 32, 64);
    return w;
}

template <int NB>
__global__ __launch_bounds__(DOT_THREADS) void k_dots(Ptr64 A, int na, Out8 B, double *__restrict__ partial, i64 n) {
    constexpr int EL = dot_el<NB>(), NQ = (NB + 3) / 4, W = DOT_THREADS / 64;
    extern __shared__ double sums[];  // [W][na * NB]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, no = na * NB;
    for (int i = tid; i < W * no; i += DOT_THREADS) sums[i] = 0.0;
    __syncthreads();
    double *mine = sums + wave * no;
    for (i64 base = (i64)blockIdx.x * DOT_THREADS * EL + tid; base - tid < n; base += (i64)gridDim.x * DOT_THREADS * EL) {
        double bv[NB][EL];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int q = 0; q < EL; ++q) {
                const i64 i = base + q * DOT_THREADS;
                bv[b][q] = i < n ? B.p[b][i] : 0.0;
            }
        double av[EL], nx[EL];
        auto load = [&](double (&d)[EL], int a) {
            const double *p = A.p[a];
#pragma unroll
            for (int q = 0; q < EL; ++q) {
                const i64 i = base + q * DOT_THREADS;
                d[q] = i < n ? p[i] : 0.0;
            }
        };
        load(av, 0);
        for (int a = 0; a < na; ++a) {
            load(nx, a + 1 < na ? a + 1 : a);
#pragma unroll
            for (int g = 0; g < NQ; ++g) {
                double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (g * 4 + b < NB)
#pragma unroll
                        for (int q = 0; q < EL; ++q) s[b] += av[q] * bv[g * 4 + b < NB ? g * 4 + b : 0][q];
                const double t = dot_wave_sum4(s);
                const int b = g * 4 + lane - 12;
                if (lane >= 12 && lane < 16 && b < NB) mine[a * NB + b] += t;
            }
#pragma unroll
            for (int q = 0; q < EL; ++q) av[q] = nx[q];
        }
    }
    __syncthreads();
    for (int o = tid; o < no; o += DOT_THREADS) {
        double t = 0.0;
        for (int w = 0; w < W; ++w) t += sums[w * no + o];
        partial[(i64)o * gridDim.x + blockIdx.x] = t;
    }
}

// out[o] = sum of partial[o * nparts .. + nparts) for o = blockIdx.x
__global__ __launch_bounds__(256) void k_multi_reduce(const double *__restrict__ partial, int nparts,
                                                      double *__restrict__ out) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) acc += partial[(i64)blockIdx.x * nparts + i];
    const double t = block_sum_d(acc);
    if (threadIdx.x == 0) out[blockIdx.x] = t;
}

struct BlockScratch {
    DevBuf partial, coef, small;
    BlockScratch() {
        partial.alloc((size_t)DMAX * BK * DOT_BLOCKS * sizeof(double));
        coef.alloc((size_t)DMAX * DMAX * sizeof(double));
        small.alloc((size_t)4 * DMAX * BK * sizeof(double));
    }
};
static BlockScratch &bscratch() {
    static thread_local std::unique_ptr<BlockScratch> s;
    if (!s) s.reset(new BlockScratch());
    return *s;
}
static int nblk_block(i64 n) { return (int)std::max<i64>(1, std::min<i64>((n + 255) / 256, 2048)); }

template <int KO>
static void launch_combo(i64 N, const double *const *X, const double *const *Y, int m, const double *Cdev, int ldc,
                         const double *wdev, double *const *out, double *partial, hipStream_t st) {
    Ptr64 PX{}, PY{};
    for (int j = 0; j < m; ++j) {
        PX.p[j] = X[j];
        PY.p[j] = Y ? Y[j] : nullptr;
    }
    Out8 O{};
    for (int r = 0; r < KO; ++r) O.p[r] = out[r];
    if (Y)
        hipLaunchKernelGGL((k_block_combo<KO, true>), dim3(nblk_block(N)), dim3(256), 0, st, PX, PY, m, Cdev, ldc,
                           wdev, O, partial, N);
    else
        hipLaunchKernelGGL((k_block_combo<KO, false>), dim3(nblk_block(N)), dim3(256), 0, st, PX, PY, m, Cdev, ldc,
                           wdev, O, partial, N);
    HIPOTF_CHECK(hipGetLastError());
}

// out_r = sum_j C[j][r] X_j (Y == nullptr) or residuals sum_j C[j][r] (Y_j - w_r X_j) with their
// norms in norms[r] (host); C is host row-major [m][k]; k may exceed BK (done in slices)
void block_combine(i64 N, int m, int k, const double *C, const double *w, const double *const *X,
                   const double *const *Y, double *const *out, double *norms, hipStream_t st) {
    HIPOTF_REQUIRE(m >= 1 && m <= DMAX && k >= 1 && k <= DMAX, "block_combine: bad sizes");
    auto &S = bscratch();
    std::vector<double> cw((size_t)m * BK + BK);
    const int nb = nblk_block(N);
    for (int r0 = 0; r0 < k; r0 += BK) {
        const int kk = std::min(BK, k - r0);
        for (int j = 0; j < m; ++j)
            for (int r = 0; r < BK; ++r) cw[(size_t)j * BK + r] = r < kk ? C[(size_t)j * k + r0 + r] : 0.0;
        for (int r = 0; r < BK; ++r) cw[(size_t)m * BK + r] = (w && r < kk) ? w[r0 + r] : 0.0;
        HIPOTF_CHECK(hipMemcpyAsync(S.coef.p, cw.data(), cw.size() * sizeof(double), hipMemcpyHostToDevice, st));
        const double *Cd = S.coef.as<double>();
        const double *wd = Cd + (size_t)m * BK;
        double *part = norms ? S.partial.as<double>() : nullptr;
        dispatch_m8(kk, [&](auto kc) {
            constexpr int KO = decltype(kc)::value;
            launch_combo<KO>(N, X, Y, m, Cd, BK, wd, out + r0, part, st);
        });
        if (norms) {
            hipLaunchKernelGGL(k_multi_reduce, dim3(kk), dim3(256), 0, st, S.partial.as<double>(), nb,
                               S.small.as<double>());
            HIPOTF_CHECK(hipGetLastError());
            std::vector<double> h(kk);
            HIPOTF_CHECK(hipMemcpyAsync(h.data(), S.small.p, kk * sizeof(double), hipMemcpyDeviceToHost, st));
            HIPOTF_CHECK(hipStreamSynchronize(st));
            for (int r = 0; r < kk; ++r) norms[r0 + r] = std::sqrt(h[r]);
        }
        // the next slice rewrites the coefficient buffer: let this one finish reading it
        HIPOTF_CHECK(hipStreamSynchronize(st));
    }
}

// In place X_r <- sum_j C[j][r] X_j for r < keep <= m <= DMAX: the subspace restart without a
// second copy of the kept vectors.  Each thread loads all m elements of its index before it
// writes any, and no two threads share an index, so reading and writing the same vectors is
// safe.  C is [keep][M], read by scalar loads (from LDS, 64 broadcast reads per output and thread
// were the bound: 669 us at 854,000 elements, 64 -> 32 vectors).  M = m rounded up to a multiple of 8.
struct PtrMut64 { double *p[DMAX]; };

template <int M>
__global__ __launch_bounds__(256) void k_rotate_inplace(PtrMut64 X, int m, int keep, const double *__restrict__ C,
                                                        i64 n) {
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        double x[M];
#pragma unroll
        for (int j = 0; j < M; ++j) x[j] = j < m ? X.p[j][i] : 0.0;
        for (int r = 0; r < keep; ++r) {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < M; ++j) acc += C[r * M + j] * x[j];
            X.p[r][i] = acc;
        }
    }
}

// X_r <- sum_j C[j*keep + r] X_j in place (C host row-major [m][keep])
void rotate_inplace(i64 N, int m, int keep, const double *C, double *const *X, hipStream_t st) {
    HIPOTF_REQUIRE(m >= 1 && m <= DMAX && keep >= 1 && keep <= m, "rotate_inplace: bad sizes");
    auto &S = bscratch();
    PtrMut64 P{};
    for (int j = 0; j < m; ++j) P.p[j] = X[j];
    const int mm = (m + 7) / 8 * 8;
    std::vector<double> Ct((size_t)keep * mm, 0.0);
    for (int j = 0; j < m; ++j)
        for (int r = 0; r < keep; ++r) Ct[(size_t)r * mm + j] = C[(size_t)j * keep + r];
    HIPOTF_CHECK(hipMemcpyAsync(S.coef.p, Ct.data(), Ct.size() * sizeof(double), hipMemcpyHostToDevice, st));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(nblk_block(N)), dim3(256), 0, st, P, m, keep, S.coef.as<double>(), N);
    };
    switch (mm) {
    case 8: go(k_rotate_inplace<8>); break;
    case 16: go(k_rotate_inplace<16>); break;
    case 24: go(k_rotate_inplace<24>); break;
    case 32: go(k_rotate_inplace<32>); break;
    case 40: go(k_rotate_inplace<40>); break;
    case 48: go(k_rotate_inplace<48>); break;
    case 56: go(k_rotate_inplace<56>); break;
    default: go(k_rotate_inplace<64>); break;
    }
    HIPOTF_CHECK(hipGetLastError());
    // the coefficient buffer is rewritten by the next block call: let this one finish reading it
    HIPOTF_CHECK(hipStreamSynchronize(st));
}

__global__ __launch_bounds__(256) void k_scatter(double *__restrict__ v, const i64 *__restrict__ idx,
                                                 const double *__restrict__ val, int count) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) v[idx[i]] = val[i];
}

// v[idx[i]] = val[i], i < count (host arrays)
void scatter_values(double *v, const i64 *idx, const double *val, int count, hipStream_t st) {
    if (count <= 0) return;
    DevBuf di((size_t)count * sizeof(i64)), dv((size_t)count * sizeof(double));
    HIPOTF_CHECK(hipMemcpyAsync(di.p, idx, (size_t)count * sizeof(i64), hipMemcpyHostToDevice, st));
    HIPOTF_CHECK(hipMemcpyAsync(dv.p, val, (size_t)count * sizeof(double), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_scatter, dim3((count + 255) / 256), dim3(256), 0, st, v, di.as<i64>(), dv.as<double>(),
                       count);
    HIPOTF_CHECK(hipGetLastError());
    HIPOTF_CHECK(hipStreamSynchronize(st));
}

// G[a][b] = A_a . B_b into host row-major [na][nb] (na <= DMAX, nb <= BK)
void block_dots(i64 N, int na, const double *const *A, int nbv, const double *const *B, double *G,
                hipStream_t st) {
    HIPOTF_REQUIRE(na >= 0 && na <= DMAX && nbv >= 1 && nbv <= BK, "block_dots: bad sizes");
    if (na == 0) return;
    auto &S = bscratch();
    Ptr64 PA{};
    Out8 PB{};
    for (int a = 0; a < na; ++a) PA.p[a] = A[a];
    for (int b = 0; b < nbv; ++b) PB.p[b] = const_cast<double *>(B[b]);
    const int no = na * nbv;
    std::vector<double> h((size_t)no, 0.0);
    if (N > 0) {
        int nb = 1;
        dispatch_m8(nbv, [&](auto bc) {
            constexpr int NB = decltype(bc)::value;
            const i64 per = (i64)DOT_THREADS * dot_el<NB>();
            nb = (int)std::max<i64>(1, std::min<i64>((N + per - 1) / per, DOT_BLOCKS));
            hipLaunchKernelGGL(k_dots<NB>, dim3(nb), dim3(DOT_THREADS), (size_t)(DOT_THREADS / 64) * no * sizeof(double),
                               st, PA, na, PB, S.partial.as<double>(), N);
        });
        HIPOTF_CHECK(hipGetLastError());
        hipLaunchKernelGGL(k_multi_reduce, dim3(no), dim3(256), 0, st, S.partial.as<double>(), nb, S.small.as<double>());
        HIPOTF_CHECK(hipGetLastError());
        HIPOTF_CHECK(hipMemcpyAsync(h.data(), S.small.p, (size_t)no * sizeof(double), hipMemcpyDeviceToHost, st));
        HIPOTF_CHECK(hipStreamSynchronize(st));
    }
    std::copy(h.begin(), h.end(), G);
}

// T_j -= sum_i P[i][j] V_i  (P host row-major [m][nt], nt <= BK)
void block_subtract(i64 N, int m, const double *const *V, const double *P, int nt, double *const *T,
                    hipStream_t st) {
    HIPOTF_REQUIRE(m >= 0 && m <= DMAX && nt >= 1 && nt <= BK, "block_subtract: bad sizes");
    if (m == 0) return;
    auto &S = bscratch();
    std::vector<double> pw((size_t)m * BK, 0.0);
    for (int i = 0; i < m; ++i)
        for (int j = 0; j < nt; ++j) pw[(size_t)i * BK + j] = P[(size_t)i * nt + j];
    HIPOTF_CHECK(hipMemcpyAsync(S.coef.p, pw.data(), pw.size() * sizeof(double), hipMemcpyHostToDevice, st));
    Ptr64 PV{};
    for (int i = 0; i < m; ++i) PV.p[i] = V[i];
    Out8 O{};
    for (int j = 0; j < nt; ++j) O.p[j] = T[j];
    dispatch_m8(nt, [&](auto kc) {
        constexpr int KO = decltype(kc)::value;
        hipLaunchKernelGGL(k_block_subtract<KO>, dim3(nblk_block(N)), dim3(256), 0, st, PV, m,
                           S.coef.as<double>(), BK, O, N);
    });
    HIPOTF_CHECK(hipGetLastError());
    HIPOTF_CHECK(hipStreamSynchronize(st));
}

}  // namespace hipotf
