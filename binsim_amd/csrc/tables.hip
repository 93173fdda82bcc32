// Same-spin operator tables built on the device (the host build in ham.cpp stays for rows longer
// than the in-LDS sort takes).
//
// For each string I of one spin: the row G[I, .] of the same-spin operator (the diagonal, the
// k (n-k) single and C(k,2) C(n-k,2) double excitations, coefficients as ham.cpp's
// build_same_spin forms them from h_pq and (pq|rs)), its source strings as colex ranks, the row
// sorted by source in LDS; then the row-block tables of the same-spin SpMM -- per block of rb
// consecutive strings the ascending union of their sources and an rb-wide coefficient column per
// union entry -- with the union as a bit set in LDS.  Replaces the host construction of
// src/include/ham/ham.hpp:635-996 / :998-1069 (JW terms and SVD groups) with a direct build.
#include "hipotf.hpp"

#include <algorithm>
#include <climits>

namespace hipotf {

constexpr int TB_LP = 2048;  // padded row length of the in-LDS row sort
constexpr int TB_BW = 33;    // binomial table C(a, b), a, b <= 32

__device__ __forceinline__ u32 tb_binom(int a, int b) {
    if (b < 0 || b > a) return 0u;
    u64 c = 1;
    for (int i = 0; i < b; ++i) c = c * (u64)(a - i) / (u64)(i + 1);
    return (u32)c;
}

// ascending bitonic sort of key[0..LP) (with val when V) by nt threads
template <bool V, typename VT>
__device__ void tb_bitonic(int *key, VT *val, int LP, int tid, int nt) {
    for (int size = 2; size <= LP; size <<= 1)
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            for (int i = tid; i < LP; i += nt) {
                const int j = i ^ stride;
                if (j > i) {
                    const bool up = (i & size) == 0;
                    const int ki = key[i], kj = key[j];
                    if ((ki > kj) == up) {
                        key[i] = kj;
                        key[j] = ki;
                        if constexpr (V) {
                            const VT t = val[i];
                            val[i] = val[j];
                            val[j] = t;
                        }
                    }
                }
            }
            __syncthreads();
        }
}

// first index in sorted a[0..m) whose value is >= x
__device__ __forceinline__ int tb_lower(const int *a, int m, i64 x) {
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((i64)a[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// one workgroup per string I: row I of the same-spin table, sorted by source
__global__ __launch_bounds__(256) void k_ss_rows(const u64 *__restrict__ strs, i64 N, int n, int k, int L,
                                                 const double *__restrict__ h, const double *__restrict__ eri,
                                                 int32_t *__restrict__ J, double *__restrict__ c64,
                                                 float *__restrict__ c32, int32_t *__restrict__ P,
                                                 double *__restrict__ gdiag) {
    __shared__ int key[TB_LP];
    __shared__ double val[TB_LP];
    __shared__ u32 bn[TB_BW * TB_BW];
    __shared__ int occ[32], vir[32];
    const int tid = threadIdx.x, nt = blockDim.x;
    const i64 I = blockIdx.x;
    const u64 s = strs[I];
    for (int t = tid; t < TB_BW * TB_BW; t += nt) bn[t] = tb_binom(t / TB_BW, t % TB_BW);
    if (tid == 0) {
        int no = 0, nv = 0;
        for (int p = 0; p < n; ++p) {
            if ((s >> p) & 1) occ[no++] = p;
            else vir[nv++] = p;
        }
    }
    __syncthreads();
    const int nv = n - k;
    const i64 n2 = (i64)n * n;
    auto E = [&](int p, int q, int r, int t) { return eri[((i64)p * n + q) * n2 + (i64)r * n + t]; };
    auto rank = [&](u64 x) {
        u32 r = 0;
        int j = 0;
        while (x) {
            r += bn[__builtin_ctzll(x) * TB_BW + j + 1];
            x &= x - 1;
            ++j;
        }
        return (int)r;
    };
    auto between = [](int a, int b) {
        const int lo = a < b ? a : b, hi = a < b ? b : a;
        return ((1ull << hi) - 1) & ~((1ull << (lo + 1)) - 1);
    };
    // (the index of pair e of m items in lexicographic (i < j) order)
    auto pair_of = [](int e, int m, int &i, int &j) {
        i = 0;
        while (e >= m - 1 - i) {
            e -= m - 1 - i;
            ++i;
        }
        j = i + 1 + e;
    };
    const int ns = k * nv, np = nv * (nv - 1) / 2;
    for (int e = tid; e < TB_LP; e += nt) {
        int kk = INT_MAX;
        double v = 0.0;
        if (e == 0) {
            for (int a = 0; a < k; ++a) {
                const int p = occ[a];
                v += h[p * n + p];
                for (int b = 0; b < k; ++b) {
                    const int q = occ[b];
                    v += 0.5 * (E(p, p, q, q) - E(p, q, q, p));
                }
            }
            kk = (int)I;
            gdiag[I] = v;
        } else if (e <= ns) {
            const int io = (e - 1) / nv, iv = (e - 1) % nv;
            const int r = occ[io], t = vir[iv];
            v = h[r * n + t];
            for (int a = 0; a < k; ++a) {
                const int j = occ[a];
                if (j == r) continue;
                v += E(r, t, j, j) - E(r, j, j, t);
            }
            if (__popcll(s & between(r, t)) & 1) v = -v;
            kk = rank(s ^ (1ull << r) ^ (1ull << t));
        } else if (e < L) {
            const int q = e - 1 - ns;
            int a1, a2, b1, b2;
            pair_of(q / np, k, a1, a2);
            pair_of(q % np, nv, b1, b2);
            const int r1 = occ[a1], r2 = occ[a2], s1 = vir[b1], s2 = vir[b2];
            const u64 js = s ^ (1ull << r1) ^ (1ull << r2) ^ (1ull << s1) ^ (1ull << s2);
            const int g1 = __popcll(js & between(r1, s1)) & 1;
            const u64 j1 = js ^ (1ull << s1) ^ (1ull << r1);
            const int g2 = __popcll(j1 & between(r2, s2)) & 1;
            v = E(r1, s1, r2, s2) - E(r1, s2, r2, s1);
            if (g1 ^ g2) v = -v;
            kk = rank(js);
        }
        key[e] = kk;
        val[e] = v;
    }
    __syncthreads();
    tb_bitonic<true>(key, val, TB_LP, tid, nt);
    for (int e = tid; e < L; e += nt) {
        J[I * L + e] = key[e];
        c64[I * L + e] = val[e];
        c32[I * L + e] = (float)val[e];
    }
    if (tid <= SS_RANGES)
        P[I * (SS_RANGES + 1) + tid] = tid == SS_RANGES ? L : tb_lower(key, L, (i64)tid * N / SS_RANGES);
}

// The set of sources of a block of rows, in LDS: a bit per string, and the count of bits before each
// 256 (ascending order and positions come from the bits: no sort)
struct TbSet {
    u32 *bits;   // [8 groups]
    int *pre;    // [groups + 1]
    int groups;
};
static int tb_groups(i64 N) { return (int)((N + 255) / 256); }
static size_t tb_set_bytes(i64 N) { return ((size_t)tb_groups(N) * 9 + 1 + 16) * 4; }

// number of members below x
__device__ __forceinline__ int tb_below(const TbSet &s, i64 x) {
    if (x >= (i64)s.groups * 256) return s.pre[s.groups];
    const int g = (int)(x >> 8), w1 = (int)(x >> 5);
    int p = s.pre[g];
    for (int w = g * 8; w < w1; ++w) p += __popc(s.bits[w]);
    return p + __popc(s.bits[w1] & ((1u << (x & 31)) - 1));
}

// the set of J[0..m), by the whole workgroup
__device__ TbSet tb_union(u32 *lds, const int32_t *__restrict__ J, int m, i64 N) {
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, G = (int)((N + 255) / 256);
    TbSet s{lds, reinterpret_cast<int *>(lds + 8 * G), G};
    int *wsum = s.pre + G + 1;  // up to 16 waves
    for (int i = tid; i < 8 * G; i += nt) s.bits[i] = 0;
    __syncthreads();
    for (int i = tid; i < m; i += nt) {
        const int j = J[i];
        atomicOr(&s.bits[j >> 5], 1u << (j & 31));
    }
    __syncthreads();
    auto count = [&](int g) {
        int c = 0;
        for (int w = 0; w < 8; ++w) c += __popc(s.bits[g * 8 + w]);
        return c;
    };
    const int per = (G + nt - 1) / nt, g0 = min(G, tid * per), g1 = min(G, g0 + per);
    int mine = 0;
    for (int g = g0; g < g1; ++g) mine += count(g);
    int x = mine;  // inclusive scan over the wave, then over the waves
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int at = x - mine;
    for (int w = 0; w < wave; ++w) at += wsum[w];
    for (int g = g0; g < g1; ++g) {
        s.pre[g] = at;
        at += count(g);
    }
    if (tid == nt - 1) s.pre[G] = at;
    __syncthreads();
    return s;
}

// f(position, member) for every member, ascending positions
template <typename F>
__device__ __forceinline__ void tb_members(const TbSet &s, F &&f) {
    for (int w = threadIdx.x; w < 8 * s.groups; w += blockDim.x) {
        u32 v = s.bits[w];
        int p = v ? tb_below(s, (i64)w * 32) : 0;
        for (; v; v &= v - 1) f(p++, w * 32 + __builtin_ctz(v));
    }
}

// per block of rb rows: the ascending union of their sources.  FILL = false: its size into cnt[g];
// FILL = true: the union into Jr[o..], the rb-wide coefficient columns and the range offsets, with
// o = off[g], or g * stride without a count
template <bool FILL, typename T>
__global__ __launch_bounds__(1024) void k_rb_union(const int32_t *__restrict__ J, const double *__restrict__ c64,
                                                   i64 N, int L, int rb, int32_t *__restrict__ cnt,
                                                   const i64 *__restrict__ off, i64 stride, int32_t *__restrict__ Jr,
                                                   T *__restrict__ cr, int32_t *__restrict__ Pr) {
    extern __shared__ u32 lds[];
    const int tid = threadIdx.x, nt = blockDim.x;
    const i64 g = blockIdx.x, r0 = g * rb, r1 = r0 + rb < N ? r0 + rb : N;
    const int m = (int)((r1 - r0) * L);
    const TbSet s = tb_union(lds, J + r0 * L, m, N);
    const int U = s.pre[s.groups];
    if (!FILL) {
        if (tid == 0) cnt[g] = U;
        return;
    }
    const i64 o = stride ? g * stride : off[g];
    tb_members(s, [&](int p, int j) { Jr[o + p] = j; });
    for (int i = tid; i < U * rb; i += nt) cr[o * rb + i] = T(0);
    __syncthreads();
    for (int i = tid; i < m; i += nt) {
        const i64 src = r0 * L + i;
        cr[(o + tb_below(s, J[src])) * rb + i / L] = (T)c64[src];
    }
    if (tid <= SS_RANGES)
        Pr[g * (SS_RANGES + 1) + tid] = (int32_t)(o + (tid == SS_RANGES ? U : tb_below(s, (i64)tid * N / SS_RANGES)));
}

// single-excitation table of one spin: sx[slot][I], slot = io (n - k) + iv, r = io-th occupied and
// t = iv-th empty orbital of string I, packed with the colex rank of I - r + t and the parity of
// the occupied orbitals strictly between r and t
__global__ __launch_bounds__(256) void k_sx(const u64 *__restrict__ strs, i64 N, int n, int k,
                                            u32 *__restrict__ sx) {
    __shared__ u32 bn[TB_BW * TB_BW];
    for (int t = threadIdx.x; t < TB_BW * TB_BW; t += blockDim.x) bn[t] = tb_binom(t / TB_BW, t % TB_BW);
    __syncthreads();
    const int nv = n - k;
    const i64 tot = N * (i64)(k * nv);
    for (i64 x = (i64)blockIdx.x * blockDim.x + threadIdx.x; x < tot; x += (i64)gridDim.x * blockDim.x) {
        const i64 slot = x / N, I = x - slot * N;
        const int io = (int)(slot / nv), iv = (int)(slot - (i64)io * nv);
        const u64 s = strs[I];
        u64 m = s, e = ~s & ((n < 64) ? ((1ull << n) - 1) : ~0ull);
        for (int i = 0; i < io; ++i) m &= m - 1;
        for (int i = 0; i < iv; ++i) e &= e - 1;
        const int r = __builtin_ctzll(m), t = __builtin_ctzll(e);
        const u64 j = s ^ (1ull << r) ^ (1ull << t);
        u32 rank = 0;
        int q = 0;
        for (u64 y = j; y; y &= y - 1, ++q) rank += bn[__builtin_ctzll(y) * TB_BW + q + 1];
        const int lo = r < t ? r : t, hi = r < t ? t : r;
        const bool neg = __popcll(s & ((1ull << hi) - 1) & ~((1ull << (lo + 1)) - 1)) & 1;
        sx[x] = sx_pack(rank, r, t, neg);
    }
}

void build_sx_dev(DevSpin &D) {
    const i64 tot = D.N * (i64)D.nsx;
    HIPOTF_REQUIRE(D.N < (1 << 20), "too many strings per spin for the packed tables (2^20)");
    HIPOTF_REQUIRE(D.n <= 32, "internal: excitation table build for n > 32");
    D.sx.alloc((size_t)tot * sizeof(u32));
    if (tot == 0) return;
    const i64 nb = std::min<i64>((tot + 255) / 256, 65536);
    hipLaunchKernelGGL(k_sx, dim3((unsigned)nb), dim3(256), 0, 0, D.strs.as<u64>(), D.N, D.n, D.k, D.sx.as<u32>());
    HIPOTF_CHECK(hipGetLastError());
    HIPOTF_CHECK(hipDeviceSynchronize());
}

__global__ __launch_bounds__(256) void k_jab(const u64 *__restrict__ strs, i64 N, int n,
                                             const double *__restrict__ eri, double *__restrict__ jab) {
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N * n) return;
    const i64 a = i / n;
    const int r = (int)(i - a * n);
    const u64 s = strs[a];
    const i64 n2 = (i64)n * n;
    double v = 0.0;
    for (int p = 0; p < n; ++p)
        if ((s >> p) & 1) v += eri[((i64)p * n + p) * n2 + (i64)r * n + r];
    jab[i] = v;
}

bool build_same_spin_dev(SameSpinTable &T, const DevSpin &S, const DevBuf &hdev, const DevBuf &eri64, int n) {
    const int L = 1 + S.nsx + S.ndx;
    if (L > TB_LP || n > 32 || S.N < 1 || S.N >= (1ll << 31) || (i64)S.N * L >= (1ll << 31)) return false;
    T.L = L;
    T.N = S.N;
    T.J.alloc((size_t)S.N * L * sizeof(int32_t));
    T.c64.alloc((size_t)S.N * L * sizeof(double));
    T.c32.alloc((size_t)S.N * L * sizeof(float));
    T.P.alloc((size_t)S.N * (SS_RANGES + 1) * sizeof(int32_t));
    T.gdiag.alloc((size_t)S.N * sizeof(double));
    hipLaunchKernelGGL(k_ss_rows, dim3((unsigned)S.N), dim3(256), 0, 0, S.strs.as<u64>(), S.N, n, S.k, L,
                       hdev.as<double>(), eri64.as<double>(), T.J.as<int32_t>(), T.c64.as<double>(),
                       T.c32.as<float>(), T.P.as<int32_t>(), T.gdiag.as<double>());
    HIPOTF_CHECK(hipGetLastError());
    HIPOTF_CHECK(hipDeviceSynchronize());
    T.dev_built = true;
    return true;
}

// Launch of a table kernel, one workgroup per row block.  (1024 threads where a block has many
// entries to place; LDS: the bits of the N strings, 144 KB at the limit of 2^20)
template <typename K, typename... Args>
static void launch_blocks(K kern, i64 nblk, i64 N, i64 entries, Args... args) {
    const size_t smem = tb_set_bytes(N);
    if (smem > 48 * 1024)
        HIPOTF_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(entries > 4096 ? 1024 : 256), smem, 0, args...);
    HIPOTF_CHECK(hipGetLastError());
}

// Sizes of the blocks' parts of a table, as first places and the total: counted on the device, or,
// where all blocks at their largest take no more than 16 MB, that many each without a count (a
// count, its two copies and their waits are most of the time of a small table)
struct TbPlaces {
    i64 stride = 0, total = 0;
    std::vector<i64> first;
};
template <typename K>
static TbPlaces tb_places(i64 nblk, i64 most, size_t bytes_each, K &&count) {
    TbPlaces p;
    if ((size_t)nblk * most * bytes_each <= 16u << 20) {
        p.stride = most;
        p.total = nblk * most;
        return p;
    }
    DevBuf cnt((size_t)nblk * sizeof(int32_t));
    count(cnt.as<int32_t>());
    std::vector<int32_t> h(nblk);
    HIPOTF_CHECK(hipMemcpy(h.data(), cnt.p, (size_t)nblk * sizeof(int32_t), hipMemcpyDeviceToHost));
    p.first.resize(nblk);
    for (i64 g = 0; g < nblk; ++g) {
        p.first[g] = p.total;
        p.total += h[g];
    }
    return p;
}

template <typename T>
static void row_blocks_t(SameSpinTable &S, RowBlockTable &R, int rb) {
    const i64 N = S.N, nblk = (N + rb - 1) / rb, most = std::min<i64>(N, (i64)rb * S.L);
    const int32_t *J = S.J.as<int32_t>();
    const double *c = S.c64.as<double>();
    const TbPlaces p = tb_places(nblk, most, 4 + rb * sizeof(T), [&](int32_t *cnt) {
        launch_blocks(k_rb_union<false, T>, nblk, N, (i64)rb * S.L, J, c, N, S.L, rb, cnt, (const i64 *)nullptr, (i64)0,
                      (int32_t *)nullptr, (T *)nullptr, (int32_t *)nullptr);
    });
    HIPOTF_REQUIRE(p.total < (1ll << 31), "row-block table too large for 32-bit offsets");
    DevBuf off;
    if (!p.stride) off.upload(p.first);
    R.rb = rb;
    R.nblk = nblk;
    R.J.alloc((size_t)p.total * sizeof(int32_t));
    R.c.alloc((size_t)p.total * rb * sizeof(T));
    R.P.alloc((size_t)nblk * (SS_RANGES + 1) * sizeof(int32_t));
    launch_blocks(k_rb_union<true, T>, nblk, N, (i64)rb * S.L, J, c, N, S.L, rb, (int32_t *)nullptr,
                  off.as<const i64>(), p.stride, R.J.as<int32_t>(), R.c.as<T>(), R.P.as<int32_t>());
    if (!p.stride) HIPOTF_CHECK(hipDeviceSynchronize());  // (off is freed here)
}
void row_blocks_dev(SameSpinTable &S, RowBlockTable &R, int rb, int prec) {
    if (prec == 0) row_blocks_t<double>(S, R, rb);
    else row_blocks_t<float>(S, R, rb);
}

// ---------------------------------------------------------------------------------------
// matrix-core row-SpMM table (MfmaBlockTable), one workgroup per block of rb rows: the union of its
// sources cut into nr ranges, each padded to whole groups of MB_GRP batches of 4 with its last
// source and coefficients 0; after the last range 2 more groups of source 0, which the kernel reads
// ahead but does not use.  FILL = false: the block's batches into cnt[g]; first place: first[g], or
// g * stride.  (From the same-spin rows themselves: by way of a row-block table of 16, filled in
// both precisions, converted and dropped again, preparing 18 orbitals / 2 + 7 took 19.4 ms, now
// 5.2; 14 / 7 + 7 1.60 -> 0.73, 8 / 4 + 4 0.35 -> 0.19)
// ---------------------------------------------------------------------------------------
template <bool FILL>
__global__ __launch_bounds__(1024) void k_mb_union(const int32_t *__restrict__ J, const double *__restrict__ c64,
                                                   i64 N, int L, int rb, int nr, int32_t *__restrict__ cnt,
                                                   const i64 *__restrict__ first, i64 stride,
                                                   int32_t *__restrict__ Pm, int32_t *__restrict__ Jm,
                                                   double *__restrict__ cm) {
    extern __shared__ u32 lds[];
    __shared__ int start[SS_RANGES + 1], base[SS_RANGES + 1];  // of each range: union position, batch
    const int tid = threadIdx.x, nt = blockDim.x;
    const i64 g = blockIdx.x, r0 = g * rb, r1 = r0 + rb < N ? r0 + rb : N;
    const int m = (int)((r1 - r0) * L);
    const TbSet s = tb_union(lds, J + r0 * L, m, N);
    if (tid <= nr) start[tid] = tid == nr ? s.pre[s.groups] : tb_below(s, (i64)(tid * (SS_RANGES / nr)) * N / SS_RANGES);
    __syncthreads();
    if (tid == 0) {
        base[0] = 0;
        for (int r = 0; r < nr; ++r)
            base[r + 1] = base[r] + (start[r + 1] - start[r] + 4 * MB_GRP - 1) / (4 * MB_GRP) * MB_GRP;
        if (!FILL) cnt[g] = base[nr] + 2 * MB_GRP;
    }
    if (!FILL) return;
    __syncthreads();
    const i64 o = stride ? g * stride : first[g];
    if (tid <= nr) Pm[g * (nr + 1) + tid] = (int32_t)(o + base[tid]);
    auto place = [&](int p) {  // entry of union position p
        int r = 0;
        while (r + 1 < nr && start[r + 1] <= p) ++r;
        return base[r] * 4 + p - start[r];
    };
    tb_members(s, [&](int p, int j) {
        const int d = place(p);
        Jm[o * 4 + d] = j;
        int r = 0;  // the last of its range: the padding too
        while (r + 1 < nr && start[r + 1] <= p) ++r;
        if (p + 1 == start[r + 1])
            for (int q = d + 1; q < base[r + 1] * 4; ++q) Jm[o * 4 + q] = j;
    });
    if (tid < 8 * MB_GRP) Jm[(o + base[nr]) * 4 + tid] = 0;
    for (int i = tid; i < (base[nr] + 2 * MB_GRP) * 4 * rb; i += nt) cm[o * 4 * rb + i] = 0.0;
    __syncthreads();
    for (int i = tid; i < m; i += nt) {
        const i64 src = r0 * L + i;
        const int q = i / L;
        cm[(o * 4 + place(tb_below(s, J[src]))) * rb + (rb == 16 ? q : (q % 4) * 2 + q / 4)] = c64[src];
    }
}

const MfmaBlockTable *mfma_blocks(SameSpinTable &T) {
    if (T.mfma) return T.mfma.get();
    if (!T.dev_built || T.N < 1) return nullptr;
    auto M = std::make_unique<MfmaBlockTable>();
    // blocks of 16 strings from 2,048 strings: 30% fewer gathered bytes than blocks of 8 for 1.4 times
    // the products.  FP64 sigma, blocks of 8 / 16: 16 orbitals / 8 + 8 electrons 110.9 / 104.5 ms, 18 / 5
    // + 5 52.7 / 50.2 ms, 14 / 7 + 7 (3,432 strings) 4.02 / 3.87 ms; but 13 / 5 + 7 (1,287 and 1,716)
    // 0.66 / 0.71 ms, 10 / 5 + 5 36 / 40 us: there half the waves, and the slices come from L2 anyway
    const int rb = M->rb = T.N >= MB_RB16_FROM ? 16 : 8;
    // as many source ranges as keep the gathered slice of 128 columns about within an XCD's 4 MB L2
    // (FP64 sigma, 16 orbitals / 8 + 8 electrons, slice 13.2 MB: 106.4 / 104.5 / 109.3 ms with 2 / 4 /
    // 8 ranges; 18 orbitals / 5 + 5, 8.8 MB: 54.4 / 50.2 / 50.7 ms with 1 / 2 / 4)
    while (M->nr < SS_RANGES && (double)T.N * 128 * 8 > 4.5e6 * M->nr) M->nr *= 2;
    const i64 N = T.N, nblk = M->nblk = (N + rb - 1) / rb;
    const i64 most = (std::min<i64>(N, (i64)rb * T.L) + 3) / 4 + (i64)M->nr * MB_GRP + 2 * MB_GRP;
    const int32_t *J = T.J.as<int32_t>();
    const double *c = T.c64.as<double>();
    const TbPlaces p = tb_places(nblk, most, 16 + 32 * rb, [&](int32_t *cnt) {
        launch_blocks(k_mb_union<false>, nblk, N, (i64)rb * T.L, J, c, N, T.L, rb, M->nr, cnt, (const i64 *)nullptr,
                      (i64)0, (int32_t *)nullptr, (int32_t *)nullptr, (double *)nullptr);
    });
    HIPOTF_REQUIRE(p.total < (1ll << 31) - 64, "matrix-core row-block table too large for 32-bit offsets");
    DevBuf first;
    if (!p.stride) first.upload(p.first);
    M->P.alloc((size_t)nblk * (M->nr + 1) * 4);
    M->J.alloc((size_t)p.total * 16);
    M->c64.alloc((size_t)p.total * 4 * rb * sizeof(double));
    launch_blocks(k_mb_union<true>, nblk, N, (i64)rb * T.L, J, c, N, T.L, rb, M->nr, (int32_t *)nullptr,
                  first.as<const i64>(), p.stride, M->P.as<int32_t>(), M->J.as<int32_t>(), M->c64.as<double>());
    if (!p.stride) HIPOTF_CHECK(hipDeviceSynchronize());  // (first is freed here)
    T.mfma = std::move(M);
    return T.mfma.get();
}

void build_jab_dev(DevBuf &jab, const DevSpin &A, int n, const DevBuf &eri64) {
    const i64 tot = A.N * n;
    jab.alloc((size_t)tot * sizeof(double));
    if (tot == 0) return;
    hipLaunchKernelGGL(k_jab, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, 0, A.strs.as<u64>(), A.N, n,
                       eri64.as<double>(), jab.as<double>());
    HIPOTF_CHECK(hipGetLastError());
    HIPOTF_CHECK(hipDeviceSynchronize());
}

}  // namespace hipotf
