// Alpha-beta part of the sigma build on the matrix cores (included by sigma.hip), n <= 18.
//
// For a destination alpha row Ia, with c running over its alpha connections -- the nsxA single
// excitations Ja_c = Ia - p_c + q_c with sign s_c, then Ia itself with the diagonal integral
// row sum_{p in Ia} (pp|..) -- the alpha-beta part of the sigma row is
//
//   sigma~[Ia, Ib] += sum_{r <= t} sum_{Jb : Ib = E_(r,t) Jb} sgn(r, t, Jb) Y[(r,t), Jb]
//   Y[(r,t), Jb]    = sum_c W[(r,t), c] x~[Ja_c, Jb],      W[(r,t), c] = s_c (p_c q_c | r t)
//
// E_(r,t) (r < t) moves the one beta electron of Jb that sits on r or t to the other orbital,
// with sgn the parity of the occupied orbitals of Jb strictly between r and t; it does not
// apply when both or neither are occupied.  The rows r = t apply when r is occupied and leave
// Jb as it is (sgn = +1).  Y is a dense product of the n(n+1)/2 x nca matrix W with the
// nca x NB matrix of source rows, so it runs as 16x16x4 MFMA tiles (FP64 or FP32 units) with
// no gathers: the rows that do not apply to a Jb are computed and dropped (47% of them at 16
// orbitals / 8 electrons).  Each element of Y is then added into an FP64 LDS copy of the
// destination row (ds_add_f64).  Same sums as the source-lane kernel (ab_src.hpp), in another
// order.
//
// Scatter.  Where an element of Y goes depends on (row, Jb) only, not on Ia, so targets come
// from a table built once per basis (k_ab_targets): one 16-bit word per element, bit 15 the
// sign, bits 0..14 the place among the destination elements, an element that does not apply
// pointing at a spare place of its lane.  The words are in MFMA-result order: a lane reads the
// four of a row tile as one 8-byte load (3.7 MB in all at 16 orbitals, served by the L2).  On
// gfx950 FP64 MFMAs and VALU operations of a SIMD do not overlap, so the VALU work per element
// is what the kernel pays on top of its products: 4 operations here, 22 when the validity, the
// colex rank and the sign were computed in place.  Measured, FP64, 16 orbitals / 8 + 8
// electrons: 33.1 -> 28.4 ms per launch (two launches; 20.7 ms of MFMA issue each); FP32, 14 orbitals, per
// vector: 2.85 -> 1.57 ms with the row tiles and k-steps of 14 orbitals (7 x 13) instead of 16 (9 x 17).
//
// Workgroup = destination alpha row (XCD-interleaved like the other alpha-beta kernels),
// NWV waves; beta strings in tiles of 16 (the MFMA's N), tiles dealt to the waves round robin.
// W sits in LDS in MFMA-operand order: the A operand of tile (k-step s, row tile m) for lane l
// is entry (s * MT + m) * 64 + l, a conflict-free 8- or 4-byte read.
//
// Two forms.  Whole row (MC = 0): the LDS holds all NB destination elements and W, one launch.
// Class split (MC > 0), where they do not fit together (FP64 from 16 orbitals / 7 electrons):
// the destinations are split by the top orbital tb = n - 1 into class N (tb empty: ranks [0, NN)
// in colex order) and class T (the rest), one launch per class with only that class in LDS.  A
// target stays in the class of its source unless the pair moves an electron onto or off tb, so
// the launch for class K computes the MO row tiles of the pairs without tb (and all r = t) on the
// class-K sources, and the MC tiles of pairs (r, tb) on the sources of the other class: every
// element of Y is computed once over both launches.
//
// Operand layout of v_mfma_{f64,f32}_16x16x4 on gfx950 (measured): lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16]; result element v of lane l is D[4 (l / 16) + v][l % 16] for f32 and
// D[4 v + l / 16][l % 16] for f64.
#pragma once

template <typename T>
struct AbMmaOps;
template <>
struct AbMmaOps<double> {
    typedef double V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mma(double a, double b, V4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static constexpr __device__ int row(int g, int v) { return 4 * v + g; }  // of result element v
};
template <>
struct AbMmaOps<float> {
    typedef float V4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ V4 mma(float a, float b, V4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static constexpr __device__ int row(int g, int v) { return 4 * g + v; }
};

// Orbital pair (r <= t) of W row i, or r = t = -1 for a padding row.  Rows r = t sit at result
// element v of lane group 0, four to a tile (the four groups of an instruction then never add to
// one place), the pairs r < t fill the other places in order.  Class split (mc > 0): rows below
// 16 mo as described for orbitals below tb = n - 1 (and r = t = tb), then the pairs (r, tb).
template <typename T>
__host__ __device__ inline void ab_mma_pair(int i, int n, int mo, int mc, int &r, int &t) {
    r = t = -1;
    if (i >= 16 * mo) {
        if (i - 16 * mo < n - 1) {
            r = i - 16 * mo;
            t = n - 1;
        }
        return;
    }
    const int tile = i >> 4, q = i & 15, left = n - 4 * tile;  // r = t rows of this tile: min(4, left)
    const bool f64 = sizeof(T) == 8;
    const int v = f64 ? q >> 2 : q;                              // place among group 0's elements
    if ((f64 ? (q & 3) == 0 : q < 4) && v < left) {
        r = t = 4 * tile + v;
        return;
    }
    int before = f64 ? (q + 3) >> 2 : (q < 4 ? q : 4);  // r = t places before q
    if (before > left) before = left > 0 ? left : 0;
    int e = i - ((4 * tile < n ? 4 * tile : n) + before);
    const int w = mc ? n - 1 : n;
    for (int a = 0; a < w - 1; ++a) {
        if (e < w - 1 - a) {
            r = a;
            t = a + 1 + e;
            return;
        }
        e -= w - 1 - a;
    }
}

__device__ __forceinline__ u32 ab_colex_rank(u64 s) {
    u32 rank = 0, j = 0;
    for (; s; s &= s - 1) {
        const u32 p = (u32)__builtin_ctzll(s);
        ++j;
        u32 c = j <= p ? 1u : 0u;  // C(p, j)
        for (u32 i = 0; i < j && c; ++i) c = c * (p - i) / (i + 1);
        rank += c;
    }
    return rank;
}

// target words of row tile m of column tile ct, one uint2 (result elements 0..3) per lane; column
// tiles of class N, then of class T (NN = NB and one class without a split)
template <typename T>
__global__ __launch_bounds__(64) void k_ab_targets(const u64 *__restrict__ strsB, int n, int NB, int NN, int mo,
                                                   int mc, uint2 *__restrict__ tab) {
    const int ct = blockIdx.x, m = blockIdx.y, lane = threadIdx.x, g = lane >> 4, col = lane & 15;
    const int nctN = (NN + 15) >> 4, cls = ct >= nctN;
    const int b0 = cls ? NN : 0, nb = cls ? NB - NN : NN, Jl = (ct - (cls ? nctN : 0)) * 16 + col;
    const int tc = m < mo ? cls : 1 - cls;                            // class of the targets
    const int t0 = tc ? NN : 0, nt = mc ? (tc ? NB - NN : NN) : NB;   // its first rank and size
    u32 w[4];
    for (int v = 0; v < 4; ++v) {
        int r, t;
        ab_mma_pair<T>(m * 16 + AbMmaOps<T>::row(g, v), n, mo, mc, r, t);
        w[v] = (u32)(nt + lane);
        if (r >= 0 && Jl < nb) {
            const u64 s = strsB[b0 + Jl], ob = (1ull << r) | (1ull << t);
            if (r == t) {
                if (s & ob) w[v] = (u32)(b0 + Jl - t0);
            } else if (__popcll(s & ob) == 1) {
                const u64 between = ((1ull << t) - 1) & ~((2ull << r) - 1);
                w[v] = (ab_colex_rank(s ^ ob) - (u32)t0) | ((u32)(__popcll(s & between) & 1) << 15);
            }
        }
    }
    tab[((i64)ct * (mo + mc) + m) * 64 + lane] = make_uint2(w[0] | w[1] << 16, w[2] | w[3] << 16);
}

// LDS bytes of k_ab_mma with NS destination elements in LDS
template <typename T, int MT, int KS>
constexpr size_t ab_mma_lds(i64 NS) {
    return (size_t)(NS + 64) * sizeof(double) + (size_t)KS * MT * 64 * sizeof(T) + (AB_SRC_CONN + 4 * 20) * 4 + MT * 16 * 4;
}

// KS: k-steps of 4 connections (4 KS >= nsxA + 1); dw rows are nwd entries wide.  MC > 0:
// destination class cls (0: ranks [0, NN), 1: [NN, NB)); otherwise the whole row (NN = NB).
template <typename T, int MO, int MC, int KS, int NWV, int WPE>
__global__ __launch_bounds__(NWV * 64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void k_ab_mma(const T *__restrict__ xt, T *__restrict__ s1, int nvst, int v0, const u32 *__restrict__ sxA,
              const uint2 *__restrict__ tab, const T *__restrict__ eri, const T *__restrict__ dw, int nwd, int n,
              i64 NA, int NB, int nsxA, int cls, int NN) {
    using Ops = AbMmaOps<T>;
    using V4 = typename Ops::V4;
    constexpr int BD = NWV * 64, MT = MO + MC, KR = 20;
    static_assert(KS <= KR, "source row table");
    // own columns and destinations [o0, o0 + NK); other columns [c0, c0 + NC) (MC > 0 only)
    const int o0 = MC && cls ? NN : 0, NK = MC ? (cls ? NB - NN : NN) : NB;
    const int c0 = MC && !cls ? NN : 0, NC = MC ? NB - NK : 0;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double *S = reinterpret_cast<double *>(smem_raw);                              // NK destinations, 64 spare
    T *Wl = reinterpret_cast<T *>(smem_raw + (size_t)(NK + 64) * sizeof(double));  // KS x MT x 64
    u32 *jrow = reinterpret_cast<u32 *>(Wl + KS * MT * 64);                        // source rows [g][KR]
    u32 *conn = jrow + 4 * KR;
    u32 *rowrt = conn + AB_SRC_CONN;                                               // r * n + t of a W row
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, col = lane & 15;
    const i64 per = (NA + 7) / 8;
    const i64 Ia = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (Ia >= NA) return;
    const int n2 = n * n;

    for (int t = tid; t < nsxA; t += BD) conn[t] = sxA[(i64)t * NA + Ia];
    for (int i = tid; i < MT * 16; i += BD) {
        int r, t;
        ab_mma_pair<T>(i, n, MO, MC, r, t);
        rowrt[i] = r >= 0 ? (u32)(r * n + t) : ~0u;
    }
    for (int t = tid; t < NK; t += BD) S[t] = 0.0;
    __syncthreads();
    // source rows of connection 4 s + g (past the last connection row Ia, against zero W)
    for (int e = tid; e < 4 * KS; e += BD) jrow[(e & 3) * KR + (e >> 2)] = (e < nsxA ? sx_J(conn[e]) : (u32)Ia) * (u32)NB;
    // W in operand order (zero past the last connection and in padding rows)
    for (int e = tid; e < KS * MT * 64; e += BD) {
        const int l = e & 63, m = (e >> 6) % MT, s = (e >> 6) / MT;
        const int c = 4 * s + (l >> 4);
        const u32 rt = rowrt[m * 16 + (l & 15)];
        T v = T(0);
        if (rt != ~0u && c <= nsxA) {
            if (c < nsxA) {
                const u32 d = conn[c];
                v = eri[(i64)(sx_r(d) * n + sx_s(d)) * n2 + rt];
                if (sx_neg(d)) v = -v;
            } else {
                v = dw[Ia * nwd + rt];
            }
        }
        Wl[e] = v;
    }
    __syncthreads();

    // the column tiles of [b0, b0 + nb), the first one at column tile ct0 of the target table, on the
    // row tiles [M0, M0 + NM)
    auto run = [&](auto m0_c, auto nm_c, int ct0, int b0, int nb) {
        constexpr int M0 = decltype(m0_c)::value, NM = decltype(nm_c)::value;
        const int ntiles = (nb + 15) >> 4;
        for (int nt = wave; nt < ntiles; nt += NWV) {
            const int Jl = nt * 16 + col;
            const u32 Jb = (u32)(b0 + (Jl < nb ? Jl : nb - 1));
            // B operands, all in flight at once; the other waves of the SIMD cover the latency
            T b[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) b[s] = xt[(size_t)((jrow[g * KR + s] + Jb) * (u32)nvst + (u32)v0)];
            uint2 tg[NM];
            const uint2 *tp = tab + ((i64)(ct0 + nt) * MT + M0) * 64 + lane;
            V4 acc[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m) acc[m] = V4{T(0), T(0), T(0), T(0)};
            // A operands PD products ahead (an LDS read takes about two FP64 MFMAs)
            constexpr int PD = 6;
            T a[PD];
            auto A = [&](int i) { return Wl[((i / NM) * MT + M0 + i % NM) * 64 + lane]; };
#pragma unroll
            for (int i = 0; i < PD; ++i) a[i] = A(i < KS * NM ? i : 0);
#pragma unroll
            for (int i = 0; i < KS * NM; ++i) {
                if (i == (KS > 6 ? KS - 6 : 0) * NM) {
                    // target words, into the registers the first operands have left
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int m = 0; m < NM; ++m) tg[m] = tp[m * 64];
                }
                acc[i % NM] = Ops::mma(a[i % PD], b[i / NM], acc[i % NM]);
                if (i + PD < KS * NM) a[i % PD] = A(i + PD);
            }
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const u32 w = v < 2 ? tg[m].x : tg[m].y;
                    const u32 at = v & 1 ? (w >> 16) & 0x7fffu : w & 0x7fffu;
                    const u32 sg = (v & 1 ? w : w << 16) & 0x80000000u;
                    atomicAdd(&S[at], flip_sign((double)acc[m][v], sg));
                }
        }
    };
    const int nctN = (NN + 15) >> 4;
    run(std::integral_constant<int, 0>{}, std::integral_constant<int, MO>{}, MC && cls ? nctN : 0, o0, NK);
    if constexpr (MC > 0)
        run(std::integral_constant<int, MO>{}, std::integral_constant<int, MC>{}, cls ? 0 : nctN, c0, NC);
    __syncthreads();
    for (int t = tid; t < NK; t += BD) {
        T &o = s1[(size_t)((Ia * NB + o0 + t) * nvst + v0)];
        o = (T)((double)o + S[t]);
    }
}
