// Rotation runs on excitation levels (included by rot.hip).
//
// In a pool whose generators only move electrons of a spin from the orbitals A to the disjoint
// orbitals C (a particle-hole pool, such as UCC from a reference determinant), a generator that
// excites k electrons of that spin takes a string with c = |s & C| to one with c + k and leaves
// the orbitals outside A and C alone.  A run of consecutive generators of one rank k therefore
// never couples elements of different blocks:
//   pair run (one alpha pattern u -> w, beta rank k):  { row u, level c } + { row w, level c + k }
//   row run (one spin moves, the other is the row):    { levels c, c + k, c + 2k, .. }
// for fixed occupation outside A and C.  One workgroup owns a few whole blocks (a bin) of one
// row (pair): their elements are loaded into LDS once, every generator of the run is applied
// there, and they are stored once.  At 16 orbitals / 8 electrons the largest pair block has
// 8,036 elements (129 KB of (l, r) values, 64 KB of l alone) where the row pair itself has
// 25,740 and had to stay in global memory; the row runs of doubles split into halves of 6,470.
//
// Bounds.  LDS bandwidth: 32 bytes per coupled pair forward, 64 in the adjoint sweep, against
// 128 bytes per cycle and CU; then the latency of a generator's phase (LDS read, a dependent
// chain of four FP64 operations, LDS write, barrier).  The pair lists are compact (one word per
// pair: two 14-bit slots and a sign, 0.9 MB for the 64 beta singles at 16 orbitals, L2 resident),
// and the words and angles of later generators are loaded while the current one runs.
// Measured at 16 orbitals (energy + gradient): pair runs 504 -> 143 ms adjoint and 212 -> 66 ms
// forward against row pairs in global memory, rows of doubles 151 -> 60 and 99 -> 21 ms; the LDS
// is busy half of an adjoint pair run.  Not kept: list words ordered so that no two of 16 (32)
// threads share a bank (an edge colouring: -1.5%, 0.1 s more in the first pass), l and r in
// separate arrays (same).
//
// Signs.  The elements are held in the alpha-major gauge x~ = (-1)^popc(b & M(a)) x, where a
// generator's sign splits into one factor per spin: the moved strings' factor is a bit of the
// list word, the alpha factor of a pair run is one bit per workgroup, and the rest is a constant
// bit of the generator.
#pragma once

constexpr int LV_SLOT_BITS = 14;
constexpr int LV_PAD = 4096; // words after the last list that idle threads may read
constexpr i64 LV_PART = 32ll << 20;  // gradient partials that one launch may write (256 MB)
constexpr int LV_RED = 64;  // generators between two flushes of the gradient sums

struct LvGen {              // one generator as one bin sees it
    double c, s;
    u32 off;                // its words in the list: first byte, count
    int32_t len;
    u32 kap, pad;           // its constant sign (bit 31)
};
static_assert(sizeof(LvGen) == 32, "two 16-byte loads");

// sign of the ladder operators ann (ascending), then cre (ascending), on string s of one spin
__host__ __device__ __forceinline__ int lv_canon(u64 s, u64 cre, u64 ann) {
    int par = 0;
    auto pop = [](u64 v) {
#ifdef __HIP_DEVICE_COMPILE__
        return (int)__popcll(v);
#else
        return __builtin_popcountll(v);
#endif
    };
    for (u64 m = ann; m; m &= m - 1) {
        const u64 b = m & (~m + 1);
        par += pop(s & (b - 1));
        s ^= b;
    }
    for (u64 m = cre; m; m &= m - 1) {
        const u64 b = m & (~m + 1);
        par += pop(s & (b - 1));
        s ^= b;
    }
    return par & 1;
}

struct LvArgs {
    double *l, *r;
    const int32_t *alist;   // pair run: (u, w) rows; NULL: row run
    i64 nunit, nel;         // row pairs or rows; elements per row
    int nbins, ng;
    const uint2 *slots;     // per slot: element | row (0: u, 1: w) << 31, gauge word of the element
    const int *soff;        // first slot of each bin, nbins + 1
    const u64 *rword;       // gauge word of each row
    const u64 *strsA;       // pair run: strings of the rows, and their pattern
    u64 acre, aann;
    const LvGen *gens;      // [nbins][gstride]
    i64 gstride;
    const u32 *list;
    double *partial;        // [nunit * nbins][ng]
};

// Wave sums of four values at once: lanes 12..15 end with the sums of a[0..3].  The values of two,
// then four lanes are dealt to the lanes of a quad while they are added, so the four sums share
// the later steps (8 VALU operations per value; one at a time takes 18).
__device__ __forceinline__ double wave_sum4(const double (&a)[4]) {
    const int lane = threadIdx.x & 63;
    auto dpp = [](double v, auto ctrl) {
        constexpr int CT = decltype(ctrl)::value;
        const long long b = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CT, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CT, 0xf, 0xf, false);
        return __longlong_as_double(((long long)hi << 32) | (u32)lo);
    };
    using X1 = std::integral_constant<int, 0xb1>;   // quad_perm 1,0,3,2
    using X2 = std::integral_constant<int, 0x4e>;   // quad_perm 2,3,0,1
    using S4 = std::integral_constant<int, 0x114>;  // row_shr 4
    using S8 = std::integral_constant<int, 0x118>;  // row_shr 8
    const bool o1 = lane & 1, o2 = lane & 2;
    const double u = (o1 ? a[1] : a[0]) + dpp(o1 ? a[0] : a[1], X1{});
    const double v = (o1 ? a[3] : a[2]) + dpp(o1 ? a[2] : a[3], X1{});
    double w = (o2 ? v : u) + dpp(o2 ? u : v, X2{});
    w += dpp(w, S4{});
    w += dpp(w, S8{});  // lanes 12..15 of each row of 16: the row's sums
    w += __shfl_xor(w, 16, 64);
    w += __shfl_xor(w, 32, 64);
    return w;
}

// MODE 0: forward rotations of l; 1: adjoint step on (l, r) with gradient sums, generators in
// reverse; 2: gradient sums only (nothing is written, so the generators need no barrier).  NP * bd
// threads' words cover the longest list.
template <int MODE, int NP>
__global__ __launch_bounds__(1024) void k_lv(LvArgs a) {
    using E = typename std::conditional<MODE == 0, double, double2>::type;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const i64 total = a.nunit * a.nbins, per = (total + 7) / 8;
    const i64 wk = (i64)(blockIdx.x & 7) * per + (blockIdx.x >> 3);  // contiguous range per XCD
    if ((i64)(blockIdx.x >> 3) >= per || wk >= total) return;
    const i64 unit = wk / a.nbins;
    const int bin = (int)(wk - unit * a.nbins);
    const int tid = threadIdx.x, bd = blockDim.x, lane = tid & 63, nw = bd >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int s0 = a.soff[bin], ns = a.soff[bin + 1] - s0;
    E *x = reinterpret_cast<E *>(smem_raw);
    // x: the bin's elements, then a zero per lane that idle threads rotate (it stays zero), then the
    // gradient sums [LV_RED][nw]
    double *red = reinterpret_cast<double *>(x + ns + 64);
    if (tid < 64) x[ns + tid] = E{};
    i64 ru = unit, rw = unit;
    int neg = 0;
    if (a.alist) {
        ru = a.alist[2 * unit];
        rw = a.alist[2 * unit + 1];
        neg = lv_canon(a.strsA[ru], a.acre, a.aann);
    }
    const u32 wu = (u32)a.rword[ru], ww = (u32)a.rword[rw];
    const i64 bu = ru * a.nel, bw = rw * a.nel;
    auto at = [&](uint2 sl) { return ((sl.x >> 31) ? bw : bu) + (i64)(sl.x & 0x7fffffffu); };
    auto flip = [&](uint2 sl) { return (u32)(__popc(sl.y & ((sl.x >> 31) ? ww : wu)) & 1) << 31; };
    auto sgn = [](double v, u32 f) { return __longlong_as_double(__double_as_longlong(v) ^ ((long long)f << 32)); };
    constexpr int LU = 4;  // elements in flight per thread
    for (int i = tid; i < ns; i += LU * bd) {
        uint2 sl[LU];
        double lv[LU], rv[LU];
#pragma unroll
        for (int q = 0; q < LU; ++q) sl[q] = a.slots[s0 + min(i + q * bd, ns - 1)];
#pragma unroll
        for (int q = 0; q < LU; ++q) {
            lv[q] = a.l[at(sl[q])];
            if (MODE) rv[q] = a.r[at(sl[q])];
        }
#pragma unroll
        for (int q = 0; q < LU; ++q)
            if (i + q * bd < ns) {
                const u32 f = flip(sl[q]);
                if constexpr (MODE == 0) x[i + q * bd] = sgn(lv[q], f);
                else x[i + q * bd] = make_double2(sgn(lv[q], f), sgn(rv[q], f));
            }
    }
    // Descriptors and list words by vector loads (their wait counter is not the LDS's), four and two
    // generators ahead in register rings of four: the loads are waited for in the order they were
    // issued, so a descriptor has to be older than the words in flight, and the generator loop is
    // unrolled by four because moving a register waits for its load.
    u32 vz;
    asm("v_mov_b32 %0, 0" : "=v"(vz));
    const LvGen *G = a.gens + (i64)bin * a.gstride;
    auto gen_at = [&](int kk) { return MODE == 1 ? a.ng - 1 - min(kk, a.ng - 1) : min(kk, a.ng - 1); };
    struct D { double c, s; u32 off; int len; u32 kap; };
    auto ld = [&](D &d, int kk) {
        const char *g = reinterpret_cast<const char *>(G) + ((u32)gen_at(kk) * (u32)sizeof(LvGen) + vz);
        const double2 cs = *reinterpret_cast<const double2 *>(g);
        const int4 ol = *reinterpret_cast<const int4 *>(g + 16);
        d.c = cs.x, d.s = cs.y, d.off = (u32)ol.x, d.len = ol.y, d.kap = (u32)ol.z;
    };
    // (threads past the end of a list read words of later ones, or the padding: slots of this plan
    // all the same, which they do not use)
    const u32 tid4 = (u32)tid * 4, bd4 = (u32)bd * 4;
    auto word = [&](u32 at) { return *reinterpret_cast<const u32 *>(reinterpret_cast<const char *>(a.list) + at); };
    auto words = [&](const D &d, u32 (&e)[NP]) {
#pragma unroll
        for (int q = 0; q < NP; ++q) e[q] = word(d.off + tid4 + q * bd4);
    };
    const u32 sflip = (u32)neg << 31;
    D d[4];
    u32 e[4][NP];
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 4; ++q) ld(d[q], q);
    words(d[0], e[0]);
    words(d[1], e[1]);
    __syncthreads();
    constexpr u32 SM = (1u << LV_SLOT_BITS) - 1;
    const u32 idle = (u32)(ns + lane);  // (a wave's idle threads rotate its own zeros)
    auto flush = [&](int k1, int cnt) {  // gradient sums of the cnt generators before order position k1
        __syncthreads();
        if (tid < cnt) {
            double t = 0.0;
            for (int w = 0; w < nw; ++w) t += red[tid * nw + w];
            a.partial[wk * a.ng + gen_at(k1 - cnt + tid)] = t;
        }
        __syncthreads();
    };
    auto reduce4 = [&](int k0) {  // the sums of generators k0 .. k0 + 3
        const double t = wave_sum4(acc);
        if ((lane & 60) == 12) red[(k0 % LV_RED + (lane & 3)) * nw + wave] = t;
    };
    auto step = [&](auto qc, int kk) {
        constexpr int Q = decltype(qc)::value;
        words(d[(Q + 2) & 3], e[(Q + 2) & 3]);
        const double c = d[Q].c, s = d[Q].s;
        const u32 gf = sflip ^ d[Q].kap;
        const int len = kk < a.ng ? d[Q].len : 0;
        if constexpr (MODE != 0 && Q == 0) {
            if (kk) {  // the previous four generators' sums
                reduce4(kk - 4);
                if (kk % LV_RED == 0) flush(kk, LV_RED);
            }
        }
        // the wave's first N words per thread (waves past the end of the list skip them)
        double sa = 0.0, sb = 0.0;
        auto apply = [&](auto nc) {
            constexpr int N = decltype(nc)::value;
            E xu[N], xw[N];
            u32 pu[N], pw[N];
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const bool act = tid + q * bd < len;
                pu[q] = act ? e[Q][q] & SM : idle;
                pw[q] = act ? (e[Q][q] >> LV_SLOT_BITS) & SM : idle;
                xu[q] = x[pu[q]];
                xw[q] = x[pw[q]];
            }
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const u32 sf = (e[Q][q] & 0x80000000u) ^ gf;
                const double ts = sgn(s, sf);
                if constexpr (MODE == 0) {
                    x[pu[q]] = c * xu[q] - ts * xw[q];
                    x[pw[q]] = ts * xu[q] + c * xw[q];
                } else if constexpr (MODE == 1) {
                    const double nlu = c * xu[q].x + ts * xw[q].x, nru = c * xu[q].y + ts * xw[q].y;
                    const double nlw = c * xw[q].x - ts * xu[q].x, nrw = c * xw[q].y - ts * xu[q].y;
                    // d/dtheta of the rotated r is t (r_w, -r_u) of the new values
                    sa += sgn(nlu * nrw - nlw * nru, sf);
                    x[pu[q]] = make_double2(nlu, nru);
                    x[pw[q]] = make_double2(nlw, nrw);
                } else {
                    sa += xu[q].x * xu[q].y + xw[q].x * xw[q].y;
                    sb += sgn(xu[q].x * xw[q].y - xw[q].x * xu[q].y, sf);
                }
            }
        };
        const int left = __builtin_amdgcn_readfirstlane(len - wave * 64);
        if (left > (NP > 1 ? bd : 0)) apply(std::integral_constant<int, NP>{});
        else if (left > 0) apply(std::integral_constant<int, 1>{});
        acc[Q] = MODE == 2 ? c * sb - s * sa : sa;
        ld(d[Q], kk + 4);
        if constexpr (MODE != 2) __syncthreads();
    };
    for (int kk = 0; kk < a.ng; kk += 4) {  // (steps past the last generator have no pairs)
        step(std::integral_constant<int, 0>{}, kk);
        step(std::integral_constant<int, 1>{}, kk + 1);
        step(std::integral_constant<int, 2>{}, kk + 2);
        step(std::integral_constant<int, 3>{}, kk + 3);
    }
    if constexpr (MODE != 0) {
        const int k0 = (a.ng - 1) & ~3;
        reduce4(k0);
        flush(a.ng, a.ng - k0 / LV_RED * LV_RED);
    }
    if constexpr (MODE != 2) {
        for (int i = tid; i < ns; i += bd) {
            const uint2 sl = a.slots[s0 + i];
            const u32 f = flip(sl);
            const E v = x[i];
            if constexpr (MODE == 0) {
                a.l[at(sl)] = sgn(v, f);
            } else {
                a.l[at(sl)] = sgn(v.x, f);
                a.r[at(sl)] = sgn(v.y, f);
            }
        }
    }
}

// A generator that moves no beta electron of a pair run (an alpha single): rows u and w of each
// pair rotated element by element, LV0_EL elements per workgroup.  HBM bound (32 bytes per
// element forward, 64 in the adjoint sweep).
constexpr int LV0_EL = 2048;
template <int MODE>
__global__ __launch_bounds__(256) void k_lv0(double *__restrict__ l, double *__restrict__ r,
                                             const int32_t *__restrict__ alist, i64 npairs, i64 nel, int nch,
                                             const u64 *__restrict__ rword, const u64 *__restrict__ strsA,
                                             const u64 *__restrict__ strsB, u64 acre, u64 aann,
                                             const LvGen *__restrict__ gen, double *__restrict__ partial) {
    const i64 wk = blockIdx.x, p = wk / nch;
    const i64 e0 = (wk - p * nch) * LV0_EL, e1 = min(nel, e0 + LV0_EL);
    const i64 ua = alist[2 * p], wa = alist[2 * p + 1];
    const u64 M = rword[ua] ^ rword[wa];
    const int neg = lv_canon(strsA[ua], acre, aann) ^ (int)(gen->kap >> 31);
    const double c = gen->c, s = gen->s;
    double acc = 0.0;
    constexpr int U = 4;
    for (i64 e = e0 + threadIdx.x; e < e1; e += U * 256) {
        u64 b[U];
        double lu[U], lw[U], ru[U], rw[U];
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const i64 i = min(e + q * 256, e1 - 1);
            b[q] = strsB[i];
            lu[q] = l[ua * nel + i];
            lw[q] = l[wa * nel + i];
            if (MODE) ru[q] = r[ua * nel + i], rw[q] = r[wa * nel + i];
        }
#pragma unroll
        for (int q = 0; q < U; ++q) {
            const i64 i = e + q * 256;
            if (i >= e1) continue;
            const bool sg = ((__popcll(b[q] & M) & 1) ^ neg) != 0;
            const double ts = sg ? -s : s, tc = sg ? -c : c;
            if (MODE == 0) {
                l[ua * nel + i] = c * lu[q] - ts * lw[q];
                l[wa * nel + i] = ts * lu[q] + c * lw[q];
            } else if (MODE == 1) {
                const double nlu = c * lu[q] + ts * lw[q], nlw = -ts * lu[q] + c * lw[q];
                acc += nlu * (-s * ru[q] + tc * rw[q]) + nlw * (-s * rw[q] - tc * ru[q]);
                l[ua * nel + i] = nlu;
                l[wa * nel + i] = nlw;
                r[ua * nel + i] = c * ru[q] + ts * rw[q];
                r[wa * nel + i] = -ts * ru[q] + c * rw[q];
            } else {
                acc += lu[q] * (-s * ru[q] + tc * rw[q]) + lw[q] * (-s * rw[q] - tc * ru[q]);
            }
        }
    }
    if (MODE) {
        const double t = block_sum(acc);
        if (threadIdx.x == 0) partial[wk] = t;
    }
}

// Column sums of pending [nrow][ng] partial blocks: out[k] = sum over rows, in fixed order.
// Stage 1: LV_SLICES row slices per 64 columns; stage 2 adds the slices.
constexpr int LV_PEND = 48, LV_SLICES = 16;
struct LvPend {
    i64 at[LV_PEND];        // first value in the partial buffer
    i64 nrow[LV_PEND];
    int ng[LV_PEND];
    int first[LV_PEND];     // result position
    int tile0[LV_PEND + 1]; // first 64-column tile
    int n;
};
__device__ __forceinline__ int lv_pend_of(const LvPend &p, int tile) {
    int d = 0;
    while (d + 1 < p.n && p.tile0[d + 1] <= tile) ++d;
    return d;
}
__global__ __launch_bounds__(256) void k_lv_sum1(LvPend p, const double *__restrict__ partial,
                                                 double *__restrict__ sums) {
    __shared__ double sm[256];
    const int tile = blockIdx.x, sl = blockIdx.y, d = lv_pend_of(p, tile);
    const int ng = p.ng[d], k0 = (tile - p.tile0[d]) * 64, nc = min(64, ng - k0);
    int w = 1;  // columns handled side by side: nc rounded up to a power of two
    while (w < nc) w *= 2;
    const int col = threadIdx.x & (w - 1), rl = threadIdx.x / w, nr = 256 / w;
    const i64 r0 = p.nrow[d] * sl / LV_SLICES, r1 = p.nrow[d] * (sl + 1) / LV_SLICES;
    double t = 0.0;
    if (col < nc)
        for (i64 i = r0 + rl; i < r1; i += nr) t += partial[p.at[d] + i * ng + k0 + col];
    sm[threadIdx.x] = t;
    __syncthreads();
    if (rl == 0 && col < nc) {
        for (int q = 1; q < nr; ++q) t += sm[q * w + col];
        sums[((i64)tile * LV_SLICES + sl) * 64 + col] = t;
    }
}
__global__ __launch_bounds__(64) void k_lv_sum2(LvPend p, const double *__restrict__ sums,
                                                double *__restrict__ dres) {
    const int tile = blockIdx.x, d = lv_pend_of(p, tile), k = (tile - p.tile0[d]) * 64 + (int)threadIdx.x;
    if (k >= p.ng[d]) return;
    double t = 0.0;
    for (int s = 0; s < LV_SLICES; ++s) t += sums[((i64)tile * LV_SLICES + s) * 64 + threadIdx.x];
    dres[p.first[d] + k] = t;
}

// c, s of the level descriptors from the device angles (gradient-only pass): entry i of bin b is
// position i
__global__ __launch_bounds__(256) void k_lv_cs(LvGen *__restrict__ g, const double *__restrict__ th, i64 n,
                                               i64 nent) {
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nent) return;
    const double t = th[i % n];
    g[i].c = cos(t);
    g[i].s = sin(t);
}

// ---- plans --------------------------------------------------------------------------------
static size_t seg_lds_budget();
// largest bin: (l, r) values with the gradient sums of 16 waves beside them, or l alone
static i64 lv_cap(bool back) {
    const i64 b = (i64)seg_lds_budget() - (back ? LV_RED * 16 * 8 : 0);
    return std::min<i64>(b / (back ? 16 : 8), 1 << LV_SLOT_BITS) - 64;
}
static size_t lv_lds(const LevelPlan &L, bool back, int bd) {
    return ((size_t)L.maxslot + 64) * (back ? 16 : 8) + (back ? (size_t)LV_RED * (bd / 64) * 8 : 0);
}

// The blocks, bins and pair lists of (spin, pair or row run, rank kb); NULL if the pool is not
// particle-hole in that spin or a block does not fit the LDS even for one vector
static LevelPlan *level_plan(DevPool *P, int spin, bool pair, int kb) {
    if (kb < 1 || kb > 4 || (P->cm[spin] & P->am[spin]) != 0) return nullptr;
    auto &slot = P->lv[spin][pair ? 1 : 0][kb];
    if (slot) return slot->ok ? slot.get() : nullptr;
    slot = std::make_unique<LevelPlan>();
    LevelPlan &L = *slot;
    const HostBasis &hb = P->basis->host;
    if (hb.norb > 32) return nullptr;
    const SpinSpace &S = spin == 0 ? hb.A : hb.B;
    const u64 C = P->cm[spin], out = ~(C | P->am[spin]);
    // blocks: occupation outside A and C, and the level (pair) or the level modulo kb (row)
    std::map<std::pair<u64, int>, std::vector<u32>> blocks;  // slots: element | row << 31
    for (i64 i = 0; i < S.N; ++i) {
        const u64 s = S.strs[i];
        const int c = __builtin_popcountll(s & C);
        if (pair) {
            blocks[{s & out, c}].push_back((u32)i);
            if (c >= kb) blocks[{s & out, c - kb}].push_back((u32)i | 0x80000000u);
        } else {
            blocks[{s & out, c % kb}].push_back((u32)i);
        }
    }
    std::vector<std::vector<u32>> bl;
    for (auto &kv : blocks) {
        auto &v = kv.second;
        bool two = false;  // both sides of a pair, or more than one level
        const int c0 = __builtin_popcountll(S.strs[v[0] & 0x7fffffffu] & C);
        for (u32 e : v) two |= pair ? (e >> 31) != (v[0] >> 31) : __builtin_popcountll(S.strs[e] & C) != c0;
        if (two) {
            if (pair) std::stable_sort(v.begin(), v.end(), [](u32 a, u32 b) { return (a >> 31) < (b >> 31); });
            bl.push_back(std::move(v));
        }
    }
    std::stable_sort(bl.begin(), bl.end(), [](const auto &a, const auto &b) { return a.size() > b.size(); });
    if (bl.empty() || (i64)bl[0].size() > lv_cap(false)) return nullptr;
    // bins: largest blocks first, smaller ones added while a bin stays within 5/4 of the largest
    // block (a bin of a few elements takes as long per generator as a full one) and the LDS.  The
    // blocks of a pool on a window of the orbitals hold a few elements each: where that makes more
    // workgroups than the chip holds at a time, bins of 512 elements (14 orbitals / 7 + 7, excitations
    // among orbitals 4 to 9, forward: 6.04 ms; 0.85 / 0.75 / 0.76 / 0.78 ms with 256 / 512 / 1024 / 2048.
    // Not in small spaces: 10 orbitals / 4 + 6, energy and gradient 0.91 -> 0.98 ms)
    const i64 big = (i64)bl[0].size(), capb = lv_cap(big <= lv_cap(true));
    i64 cap = big + big / 4, held = 0;
    for (const auto &v : bl) held += (i64)v.size();
    if ((spin == 0 ? hb.B : hb.A).N * (held / cap) > 2048) cap = std::max<i64>(cap, 512);
    cap = std::min(cap, capb);
    std::vector<std::vector<u32>> bins;
    std::vector<int> blocks_of;
    for (auto &v : bl) {
        size_t b = 0;
        while (b < bins.size() && (i64)(bins[b].size() + v.size()) > cap) ++b;
        if (b == bins.size()) bins.emplace_back(), blocks_of.push_back(0);
        bins[b].insert(bins[b].end(), v.begin(), v.end());
        ++blocks_of[b];
    }
    // (many small blocks: in the order of the rows and elements, for coalesced loads)
    for (size_t b = 0; b < bins.size(); ++b)
        if (blocks_of[b] > 8) std::sort(bins[b].begin(), bins[b].end());
    L.nbins = (int)bins.size();
    // slot of an element: [row side][element]
    std::vector<int> bin_of[2], loc[2];
    for (int q = 0; q < 2; ++q) bin_of[q].assign(S.N, -1), loc[q].assign(S.N, 0);
    std::vector<uint2> slots;
    std::vector<int> soff{0};
    for (int b = 0; b < L.nbins; ++b) {
        for (size_t i = 0; i < bins[b].size(); ++i) {
            const u32 e = bins[b][i], el = e & 0x7fffffffu;
            for (int q = 0; q < 2; ++q)
                if (!pair || q == (int)(e >> 31)) bin_of[q][el] = b, loc[q][el] = (int)i;
            u64 word = S.strs[el];
            if (spin == 0) {
                word = 0;
                for (u64 m = S.strs[el]; m; m &= m - 1) word ^= (m & (~m + 1)) - 1;
            }
            slots.push_back(make_uint2(e, (u32)word));
        }
        soff.push_back((int)slots.size());
        L.maxslot = std::max(L.maxslot, (int)bins[b].size());
    }
    // pair lists of every pattern of this rank, by bin
    std::vector<u32> list;
    L.pat.assign(P->lists.size(), -1);
    for (size_t q = 2; q < P->lists.size(); ++q) {
        const PairList &pl = P->lists[q];
        if (pl.spin != spin || __builtin_popcountll(pl.cre) != kb) continue;
        L.pat[q] = (int)(L.ol.size() / L.nbins);
        std::vector<std::vector<u32>> w(L.nbins);
        for (i64 j = 0; j < pl.len; ++j) {
            const int u = pl.h[2 * j], v = pl.h[2 * j + 1];
            const int b = bin_of[0][u];
            HIPOTF_REQUIRE(b >= 0 && b == bin_of[1][v], "internal: a pair leaves its level block");
            w[b].push_back((u32)loc[0][u] | ((u32)loc[1][v] << LV_SLOT_BITS) |
                           ((u32)lv_canon(S.strs[u], pl.cre, pl.ann) << 31));
        }
        for (int b = 0; b < L.nbins; ++b) {
            L.ol.push_back(make_int2((int)list.size() * 4, (int)w[b].size()));
            L.maxlen = std::max(L.maxlen, (int)w[b].size());
            list.insert(list.end(), w[b].begin(), w[b].end());
        }
    }
    if (L.maxlen > 4 * 1024) return nullptr;
    list.resize(list.size() + LV_PAD, 0u);
    HIPOTF_REQUIRE(list.size() < (1u << 29), "internal: level lists too long");
    // (one allocation and copy: of a small pool's first pass they are most of the cost)
    L.list_at = slots.size() * sizeof(uint2);
    L.soff_at = L.list_at + list.size() * sizeof(u32);
    std::vector<unsigned char> all(L.soff_at + soff.size() * sizeof(int));
    std::memcpy(all.data(), slots.data(), L.list_at);
    std::memcpy(all.data() + L.list_at, list.data(), list.size() * sizeof(u32));
    std::memcpy(all.data() + L.soff_at, soff.data(), soff.size() * sizeof(int));
    L.data.upload(all);
    L.ok = true;
    return &L;
}

// Threads of a run's workgroups, and list words per thread (1, 2 or 4) to cover the longest list.
// Two words per thread share the descriptor work, but where few waves are in flight on a CU (a
// bin that fills the LDS, or a small grid) a generator's phase is latency and one word on twice the
// waves is faster (12 orbitals: adjoint runs 31 -> 24 us, forward 24 -> 18; 14 orbitals, nine bins
// per CU: forward 12.2 ms per sweep with two words, 13.5 with one).  The gradient-only pass has no
// barrier between generators, its waves run ahead on their own, and two words are never slower
// (whole pool at 14 orbitals 7.5 -> 6.7 ms).  More than four waves come in whole rounds of the
// CU's four SIMDs.
static int lv_threads(const LevelPlan &L, int np) {
    const int t = (L.maxlen + np - 1) / np, m = t > 256 ? 256 : 64;
    return std::max(64, (t + m - 1) / m * m);
}
static int lv_words(const LevelPlan &L, bool back, bool grad, i64 nblk) {
    if (L.maxlen > 2048) return 4;
    if (grad) return L.maxlen > 64 ? 2 : 1;
    if (L.maxlen > 1024) return 2;
    const int bd = lv_threads(L, 2);
    const i64 perCU = std::min<i64>((i64)(seg_lds_budget() / lv_lds(L, back, bd)), (nblk + 255) / 256);
    return perCU * (bd / 64) >= 16 ? 2 : 1;
}
