// Grid layout of the step kernel: meshes numbered line by line, stepped in
// patches with the neighbours' fields in LDS and the matrices as stencil classes
// (see GridArgs).  Same arithmetic per row as step_tile (sfg_kernels.hip), which a change
// here has to follow (the persistent schedule steps the same runs by either): every
// sum runs in column order, and the FP64 form is bit-identical to the reference.
#include <hip/hip_cooperative_groups.h>

#include <algorithm>
#include <type_traits>

#include "sfg_device.h"

namespace sfg {

template <class T> struct vec16;
template <> struct vec16<float> { using type = float4; };
template <> struct vec16<double> { using type = double2; };

// The 32 distinct products of one row over the union pattern (the reference's
// 44 csr_matvec calls, time_evolution/elastic_wave.c:533-580, 599-646).
template <class T>
struct Products {
    T s1u = 0, s1w = 0, s2u = 0, s2w = 0, s3u = 0, s3w = 0;
    T s4u = 0, s4w = 0, s5u = 0, s5w = 0, s6u = 0, s6w = 0;
    T mu1t = 0, mu1 = 0, mlx1 = 0, mlx2 = 0, mu2t = 0, mu2 = 0, mu3t = 0, mu3 = 0, mlx3 = 0, mlx4 = 0;
    T mw1t = 0, mw1 = 0, mly1 = 0, mly2 = 0, mw2t = 0, mw2 = 0, mw3t = 0, mw3 = 0, mly3 = 0, mly4 = 0;
};

// Per-row coefficients of the right-hand side.
template <class T>
struct RowCoef {
    T c11, c13, c33, c44, dx, dy, dxx, dyy, dxxp, dyyp;
};

// Right-hand sides of the 14 split equations, operand order of
// elastic_wave.c:585-591 (u) and :651-657 (w): u1, u2, u3, Lx1..4, then w1, w2,
// w3, Ly1..4.
template <class T>
__device__ __forceinline__ void split_rhs(const Products<T> &p, const RowCoef<T> &c, T dt, T fu, T fw, T r[14])
{
    r[0] = -c.c11 * p.s1u - T(2.0) * c.dx * p.mu1t - c.dx * c.dx * p.mu1 + p.mlx1 + p.mlx2 + fu;
    r[1] = -c.c13 * p.s3w - c.c44 * p.s4w - c.dx * p.mu2t - c.dy * p.mu2t - c.dx * c.dy * p.mu2;
    r[2] = -c.c44 * p.s2u - T(2.0) * c.dy * p.mu3t - c.dy * c.dy * p.mu3 + p.mlx3 + p.mlx4;
    r[3] = -dt * c.c11 * c.dxx * p.s5u - dt * c.dx * p.mlx1 + p.mlx1;
    r[4] = -dt * c.c44 * c.dyyp * p.s5w - dt * c.dy * p.mlx2 + p.mlx2;
    r[5] = -dt * c.c13 * c.dxxp * p.s6w - dt * c.dx * p.mlx3 + p.mlx3;
    r[6] = -dt * c.c44 * c.dyy * p.s6u - dt * c.dy * p.mlx4 + p.mlx4;
    r[7] = -c.c44 * p.s1w - T(2.0) * c.dx * p.mw1t - c.dx * c.dx * p.mw1 + p.mly1 + p.mly2 + fw;
    r[8] = -c.c44 * p.s3u - c.c13 * p.s4u - c.dx * p.mw2t - c.dy * p.mw2t - c.dx * c.dy * p.mw2;
    r[9] = -c.c33 * p.s2w - T(2.0) * c.dy * p.mw3t - c.dy * c.dy * p.mw3 + p.mly3 + p.mly4;
    r[10] = -dt * c.c44 * c.dxx * p.s5w - dt * c.dx * p.mly1 + p.mly1;
    r[11] = -dt * c.c13 * c.dyyp * p.s5u - dt * c.dy * p.mly2 + p.mly2;
    r[12] = -dt * c.c44 * c.dxxp * p.s6u - dt * c.dx * p.mly3 + p.mly3;
    r[13] = -dt * c.c33 * c.dyy * p.s6w - dt * c.dy * p.mly4 + p.mly4;
}

__device__ __forceinline__ float lane_value(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_value(double v, int l)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}

// base[i] with the byte offset i * sizeof held in 32 bits: a uniform base and a
// 32-bit lane offset are one load or store, without 64-bit address arithmetic per
// lane (runs of 2^28 nodes or more do not take this layout).
template <class T>
__device__ __forceinline__ const T &at32(const T *base, uint32_t bytes)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes);
}
template <class T>
__device__ __forceinline__ T &at32(T *base, uint32_t bytes)
{
    return *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + bytes);
}

// One table entry: M, S1..S6 and the halo position of the column relative to the
// row's own (a small integer, exact in T).
template <class T>
struct alignas(8 * sizeof(T)) Entry {
    T v[7], off;
};

// Values of T per halo position in LDS: part A holds U, W, Lx1..4, Ly1..4, part B
// the split displacements and velocities.  Strides of an odd number of 16-byte
// words keep the 16-byte reads of neighbouring positions on different banks (FP32:
// 12 = 3 words; FP64: 10 and 14 = 5 and 7 words; part B in FP32 is 3 words as is).
template <class T> constexpr int LDS_A = sizeof(T) == 4 ? 12 : 10;
template <class T> constexpr int LDS_B = sizeof(T) == 4 ? 12 : 14;

// N consecutive values between LDS and registers in 16-byte pieces (8-byte for the rest)
template <int N, class T>
__device__ __forceinline__ void lds_get(const T *p, T *v)
{
    using V16 = typename vec16<T>::type;
    constexpr int E = 16 / sizeof(T);
#pragma unroll
    for (int k = 0; k < N / E; ++k) {
        const V16 w = reinterpret_cast<const V16 *>(p)[k];
        if constexpr (E == 4) v[4 * k] = w.x, v[4 * k + 1] = w.y, v[4 * k + 2] = w.z, v[4 * k + 3] = w.w;
        else v[2 * k] = w.x, v[2 * k + 1] = w.y;
    }
    if constexpr (N % E == 2) {
        const float2 w = *reinterpret_cast<const float2 *>(p + N - 2);
        v[N - 2] = w.x;
        v[N - 1] = w.y;
    }
}
template <int N, class T>
__device__ __forceinline__ void lds_put(T *p, const T *v)
{
    using V16 = typename vec16<T>::type;
    constexpr int E = 16 / sizeof(T);
#pragma unroll
    for (int k = 0; k < N / E; ++k) {
        V16 w;
        if constexpr (E == 4) w = make_float4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]);
        else w = make_double2(v[2 * k], v[2 * k + 1]);
        reinterpret_cast<V16 *>(p)[k] = w;
    }
    if constexpr (N % E == 2) *reinterpret_cast<float2 *>(p + N - 2) = make_float2(v[N - 2], v[N - 1]);
}

// The stencil of one class spread over a wave: lane k holds nonzero k (at most
// (2 GRID_REACH + 1)^2 = 25 of them).
template <class T>
struct Stencil {
    int off;
    T v[7];
    __device__ __forceinline__ void load(const Entry<T> *tab, int len, int lane)
    {
        const Entry<T> e = tab[min(lane, max(len - 1, 0))];
        off = (int)e.off;
#pragma unroll
        for (int m = 0; m < 7; ++m) v[m] = e.v[m];
    }
    __device__ __forceinline__ int offset(int k) const { return __builtin_amdgcn_readlane(off, k); }
    __device__ __forceinline__ T value(int m, int k) const { return lane_value(v[m], k); }
};

// One patch of one shot, step t (buffers by slot = t & 1, so that the loads of
// the state do not wait for the step counter).
//
// U, W and the 8 memory fields of the patch and its halo go to LDS (part A); every
// row forms the products that rows outside the damping layers need (and S5, S6
// where the patch has M-PML rows).  Only patches with M-PML rows also stage the 12
// split displacements and velocities (part B): with TOG beside part A, all products
// in one walk; else over it after a barrier, in a second walk of the M-PML rows.  A row
// outside the layers multiplies those products by exact zeros, in FP64 too: while the
// fields are finite, leaving them at zero changes no bit of U and W (a sum plus a signed
// zero is unchanged, and the displacements, which start at +0, never become -0).  Once a
// split field has overflowed the reference's form has a NaN there (zero times infinity)
// and this one has not; the energy guard ends such a run either way.  The patch's class
// table precedes them in LDS.
template <class T, int PREC, bool CPS, int MODE, bool TOG>
__device__ __forceinline__ void grid_tile(const StepArgs<T> &a, const GridArgs<T> &g, int t, int slot, int patch, int s,
                                          bool lead)
{
    constexpr bool EXACT = PREC == 0, KAHAN = PREC >= 2, C16 = PREC == 3;
    constexpr int NC = C16 ? 3 : 6;
    extern __shared__ __align__(64) unsigned char sfg_lds_raw[];
    const GridShape &gs = g.g;
    const int R = gs.most, tid = threadIdx.x, lane = tid & 63;
    const int wid = patch * (R >> 6) + __builtin_amdgcn_readfirstlane(tid >> 6);
    const int at = patch * R + tid;              // place of the thread's row
    const int W = gs.W, halo = gs.halo;
    Entry<T> *tab = reinterpret_cast<Entry<T> *>(sfg_lds_raw);
    constexpr int SA = LDS_A<T>, SB = LDS_B<T>;
    T *lds_a = reinterpret_cast<T *>(sfg_lds_raw + sizeof(Entry<T>) * gs.table);
    T *lds_b = TOG ? lds_a + (size_t)halo * SA : lds_a;
    const int py = patch / gs.px, px = patch - py * gs.px;
    const int x0 = px * gs.pw - gs.hx, y0 = py * gs.ph - gs.hy;
    const size_t F = (size_t)g.np;               // field stride
    const T *in = a.state + ((size_t)slot * a.S + s) * NFIELD * F;
    T *out = a.state + ((size_t)(slot ^ 1) * a.S + s) * NFIELD * F;
    const T *uwin = a.uw + ((size_t)slot * a.S + s) * 2 * F;
    T *uwout = a.uw + ((size_t)(slot ^ 1) * a.S + s) * 2 * F;

    // halo positions of this thread: q and q + R (clamped into the mesh: a position
    // outside it is staged but never read)
    uint32_t hn[2];                              // their byte offsets
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int q = min(tid + b * R, halo - 1);
        const int qy = (q * g.magic) >> 16, qx = q - qy * W;
        hn[b] = (uint32_t)(min(max(y0 + qy, 0), gs.lines - 1) * gs.pitch + min(max(x0 + qx, 0), gs.line - 1)) * sizeof(T);
    }
    const int row = g.rows[at];
    const int key = g.cls[at];
    const int info = g.info[at];
    const int wave_info = ro(g.slice)[wid];
    const int bkind = ro(g.bkind)[patch];
    const int toff = MODE == GRID_ROWS ? 0 : ro(g.toff)[patch], tlen = MODE == GRID_ROWS ? 0 : ro(g.tlen)[patch];
    const bool second = halo > R;
    auto fetch_a = [&](int b, T *v) __attribute__((always_inline)) {
        v[0] = at32(uwin, hn[b]);
        v[1] = at32(uwin + F, hn[b]);
#pragma unroll
        for (int f = 0; f < 8; ++f) v[2 + f] = at32(in + (LX1 + f) * F, hn[b]);
    };
    auto fetch_b = [&](int b, T *v) __attribute__((always_inline)) {
#pragma unroll
        for (int f = 0; f < 12; ++f) v[f] = at32(in + (U1 + f) * F, hn[b]);
    };
    T sa[2][10], sb[2][12];
    fetch_a(0, sa[0]);
    if (second) fetch_a(1, sa[1]);
    if (TOG && bkind == 2) {
        fetch_b(0, sb[0]);
        if (second) fetch_b(1, sb[1]);
    }
    // the patch's class table: 8 words of T per entry, copied in 16-byte pieces
    if constexpr (MODE != GRID_ROWS) {
        using V16 = typename vec16<T>::type;
        const V16 *src = reinterpret_cast<const V16 *>(g.tab + (size_t)toff * 8);
        V16 *dst = reinterpret_cast<V16 *>(tab);
        for (int q = tid; q < (int)sizeof(T) / 2 * tlen; q += R) dst[q] = src[q];
    }
    const int wlen = wave_info & 0xff;           // longest row of the wave
    const bool uniform = (wave_info & 0x100) != 0;
    // the row's stencil: first table entry, nonzeros; its own halo position
    // (a lane without a row stands at the wave's first one: it walks along, see walk)
    const bool valid = row >= 0;
    const int own0 = __builtin_amdgcn_readfirstlane(key >> 12 & 0xfff);
    const int e0 = key & 0xfff, own = valid ? key >> 12 & 0xfff : own0, rlen = key >> 24;
    const int r = valid ? row : 0;
    // byte offsets of the row in the state (lines `pitch` nodes apart) and among the coefficients
    const int oy = (own * g.magic) >> 16, sr = valid ? (y0 + oy) * gs.pitch + x0 + own - oy * W : 0;
    const uint32_t rb = (uint32_t)sr * sizeof(T), rw = (uint32_t)sr * 4, rc = (uint32_t)r * sizeof(T);
    const int pk = info & GI_KIND;
    // a row no M-PML row gathers from steps the sums of its split fields (FP32
    // forms, StepArgs::agg)
    const bool agg = !EXACT && pk == 0;
    const bool pml = bkind == 2 && pk == 2;

    // ---- own-row state and coefficients, requested ahead of the products ----
    const size_t C6 = (size_t)NC * F;
    const T *cin = KAHAN ? a.comp + ((size_t)slot * a.S + s) * C6 : nullptr;
    T *cout = KAHAN ? a.comp + ((size_t)(slot ^ 1) * a.S + s) * C6 : nullptr;
    const uint32_t *win = reinterpret_cast<const uint32_t *>(cin);
    uint32_t *wout = reinterpret_cast<uint32_t *>(cout);
    T disp[6], vel[6], acc[6], kt[6];            // acc holds p in the FP32 forms
#pragma unroll
    for (int q = 0; q < 6; ++q) disp[q] = vel[q] = acc[q] = kt[q] = T(0);
    if (agg) {
        acc[0] = at32(in + U1TT * F, rb);
        acc[3] = at32(in + W1TT * F, rb);
        if constexpr (C16) {
            const uint32_t w = at32(win, rw);
            kt[0] = bf16_lo(w);
            kt[3] = bf16_hi(w);
        } else if constexpr (KAHAN) {
            kt[0] = at32(cin, rb);
            kt[3] = at32(cin + F, rb);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            disp[q] = at32(in + (U1 + q) * F, rb);
            if constexpr (EXACT) vel[q] = at32(in + (U1T + q) * F, rb);
            acc[q] = at32(in + (U1TT + q) * F, rb);
        }
        if constexpr (C16) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const uint32_t w = at32(win + k * F, rw);
                kt[2 * k] = bf16_lo(w);
                kt[2 * k + 1] = bf16_hi(w);
            }
        } else if constexpr (KAHAN) {
#pragma unroll
            for (int q = 0; q < 6; ++q) kt[q] = at32(cin + q * F, rb);
        }
    }
    // shared media: [coef][node]; one per shot: [shot][coef][node]
    const size_t cs = (size_t)a.n;
    const T *cf = a.coef + (CPS ? (size_t)s * NCOEF * cs : 0);
    RowCoef<T> c{};
    c.c11 = at32(cf + C11 * cs, rc);
    c.c13 = at32(cf + C13 * cs, rc);
    c.c33 = at32(cf + C33 * cs, rc);
    c.c44 = at32(cf + C44 * cs, rc);
    const T mass = at32(cf + MASS * cs, rc);
    T mrow = T(1);
    if constexpr (CPS) mrow = at32(cf + MROW * cs, rc);

    // hand t + 1 to the next launch (here, where t has arrived, not at the start)
    if (lead) __hip_atomic_store(&a.ctrl->step[slot ^ 1], t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // a finished shot leaves here, the whole block at once
    if (t >= (a.S == 1 ? g.steps0 : a.nsteps_max)) return;

    auto stash_a = [&](int b) __attribute__((always_inline)) {
        if (tid + b * R < halo) lds_put<10>(lds_a + (tid + b * R) * SA, sa[b]);
    };
    auto stash_b = [&](int b) __attribute__((always_inline)) {
        if (tid + b * R < halo) lds_put<12>(lds_b + (tid + b * R) * SB, sb[b]);
    };
    stash_a(0);
    if (second) stash_a(1);
    if (TOG && bkind == 2) {
        stash_b(0);
        if (second) stash_b(1);
    }
    __syncthreads();

    using PA = std::integral_constant<int, 10>;  // fields a walk reads: part A,
    using PB = std::integral_constant<int, 12>;  // part B,
    using PAB = std::integral_constant<int, 22>; // or both
    auto fields = [&](auto nf, int j, T *x) __attribute__((always_inline)) {
        constexpr int NF = decltype(nf)::value;
        if constexpr (NF != 12) lds_get<10>(lds_a + j * SA, x);
        if constexpr (NF != 10) lds_get<12>(lds_b + j * SB, x + NF - 12);
    };
    Stencil<T> st;
    if (MODE != GRID_ROWS && uniform) st.load(tab + __builtin_amdgcn_readfirstlane(e0), wlen, lane);
    // Calls nz(the staged fields of the column, M, S1..S6 values) over the row's
    // nonzeros in column order.  A wave of one class broadcasts the stencil from its
    // lanes with v_readlane (through the scalar cache, which every launch finds cold, a
    // nonzero took 500-1000 cycles, and a scalar load in flight turns every LDS wait
    // into a full drain); the lanes of other waves read their own entries of the table.
    // v_readlane must not read a lane that is switched off, so a wave of one class walks with
    // all its lanes, also those that are not `on`, whose products are not used.
    auto walk = [&](bool on, auto np, auto &&nz) __attribute__((always_inline)) {
        constexpr int NP = decltype(np)::value;
        if (wlen == 0 || __builtin_amdgcn_ballot_w64(on) == 0) return;
        if constexpr (MODE == GRID_ROWS) {
            if (!on) return;
            constexpr int AHEAD = EXACT ? 2 : 4;
            const size_t m0 = (size_t)ro(g.moff)[wid];
            for (int k0 = 0; k0 < wlen; k0 += AHEAD) {
                T v[AHEAD][7];
                int o[AHEAD];
                // (positions past the row's end repeat its last nonzero, unused)
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    const int k = max(min(k0 + u, rlen - 1), 0);
                    const T *q = g.mval + (m0 + k) * (7 * 64) + lane;
                    o[u] = g.sdel[(m0 + k) * 64 + lane];
#pragma unroll
                    for (int m = 0; m < 7; ++m) v[u][m] = q[m * 64];
                }
                // (keeps the loads together: the compiler would sink each behind its test)
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) {
                    asm volatile("" : "+v"(o[u]));
#pragma unroll
                    for (int m = 0; m < 7; ++m) asm volatile("" : "+v"(v[u][m]));
                }
#pragma unroll
                for (int u = 0; u < AHEAD; ++u)
                    if (k0 + u < rlen) {
                        T x[NP];
                        fields(np, own + o[u], x);
                        nz(x, v[u][0], v[u][1], v[u][2], v[u][3], v[u][4], v[u][5], v[u][6]);
                    }
            }
        } else {
            // M per row: the next MA values are on their way while MA are used
            constexpr int MA = MODE == GRID_CLASS_S ? 4 : 1;
            const T *mv = nullptr;
            T m[MA], mn[MA];
            if constexpr (MODE == GRID_CLASS_S) {
                mv = g.mval + (size_t)ro(g.moff)[wid] * 64 + lane;
#pragma unroll
                for (int u = 0; u < MA; ++u) m[u] = mv[min(u, wlen - 1) * 64];
            }
            using B0 = std::integral_constant<int, 0>;
            using B1 = std::integral_constant<int, 1>;
            auto all = [&](int len, auto &&one) __attribute__((always_inline)) {
                if constexpr (MODE == GRID_CLASS_S) {
                    for (int k0 = 0; k0 < len; k0 += MA) {
#pragma unroll
                        for (int u = 0; u < MA; ++u) mn[u] = mv[min(k0 + MA + u, wlen - 1) * 64];
#pragma unroll
                        for (int u = 0; u < MA; u += 2) {
                            if (k0 + u < len) one(k0 + u, B0{}, m[u]);
                            if (k0 + u + 1 < len) one(k0 + u + 1, B1{}, m[u + 1]);
                        }
#pragma unroll
                        for (int u = 0; u < MA; ++u) m[u] = mn[u];
                    }
                } else {
                    for (int k = 0; k < len; k += 2) {
                        one(k, B0{}, T(0));
                        if (k + 1 < len) one(k + 1, B1{}, T(0));
                    }
                }
            };
            // part A alone: the next column's fields are read while these are used
            // (two buffers in turn); both parts: there are enough of them in flight
            constexpr bool TWO = NP == 10;
            T x[TWO ? 2 : 1][NP];
            if (uniform) {
                if constexpr (TWO) fields(np, own + st.offset(0), x[0]);
                all(wlen, [&](int k, auto B, T mk) __attribute__((always_inline)) {
                    constexpr int b = TWO ? decltype(B)::value : 0;
                    if constexpr (TWO) {
                        fields(np, own + st.offset(min(k + 1, wlen - 1)), x[1 - b]);
                        __builtin_amdgcn_sched_barrier(0);
                    } else {
                        fields(np, own + st.offset(k), x[0]);
                    }
                    nz(x[b], MODE == GRID_CLASS_S ? mk : st.value(0, k), st.value(1, k), st.value(2, k), st.value(3, k),
                       st.value(4, k), st.value(5, k), st.value(6, k));
                });
            } else if (on) {
                const Entry<T> *e = tab + e0;
                Entry<T> c = e[0], next;
                all(rlen, [&](int k, auto, T mk) __attribute__((always_inline)) {
                    fields(np, own + (int)c.off, x[0]);
                    next = e[min(k + 1, rlen - 1)];
                    nz(x[0], MODE == GRID_CLASS_S ? mk : c.v[0], c.v[1], c.v[2], c.v[3], c.v[4], c.v[5], c.v[6]);
                    c = next;
                });
            }
        }
    };
    Products<T> p;
    // products of U, W (S1..S4, and with `layers` S5, S6) and of the memory fields
    auto products_a = [&](auto layers, const T *x, T am, T a1, T a2, T a3, T a4, T a5, T a6)
        __attribute__((always_inline)) {
        const T U = x[0], V = x[1];
        p.s1u = mac<EXACT>(p.s1u, a1, U); p.s1w = mac<EXACT>(p.s1w, a1, V);
        p.s2u = mac<EXACT>(p.s2u, a2, U); p.s2w = mac<EXACT>(p.s2w, a2, V);
        p.s3u = mac<EXACT>(p.s3u, a3, U); p.s3w = mac<EXACT>(p.s3w, a3, V);
        p.s4u = mac<EXACT>(p.s4u, a4, U); p.s4w = mac<EXACT>(p.s4w, a4, V);
        if constexpr (decltype(layers)::value) {
            p.s5u = mac<EXACT>(p.s5u, a5, U); p.s5w = mac<EXACT>(p.s5w, a5, V);
            p.s6u = mac<EXACT>(p.s6u, a6, U); p.s6w = mac<EXACT>(p.s6w, a6, V);
        }
        p.mlx1 = mac<EXACT>(p.mlx1, am, x[2]); p.mlx2 = mac<EXACT>(p.mlx2, am, x[3]);
        p.mlx3 = mac<EXACT>(p.mlx3, am, x[4]); p.mlx4 = mac<EXACT>(p.mlx4, am, x[5]);
        p.mly1 = mac<EXACT>(p.mly1, am, x[6]); p.mly2 = mac<EXACT>(p.mly2, am, x[7]);
        p.mly3 = mac<EXACT>(p.mly3, am, x[8]); p.mly4 = mac<EXACT>(p.mly4, am, x[9]);
    };
    // products of U1..W3 and U1t..W3t with M
    auto products_b = [&](const T *x, T am) __attribute__((always_inline)) {
        p.mu1 = mac<EXACT>(p.mu1, am, x[0]); p.mu2 = mac<EXACT>(p.mu2, am, x[1]); p.mu3 = mac<EXACT>(p.mu3, am, x[2]);
        p.mw1 = mac<EXACT>(p.mw1, am, x[3]); p.mw2 = mac<EXACT>(p.mw2, am, x[4]); p.mw3 = mac<EXACT>(p.mw3, am, x[5]);
        p.mu1t = mac<EXACT>(p.mu1t, am, x[6]); p.mu2t = mac<EXACT>(p.mu2t, am, x[7]);
        p.mu3t = mac<EXACT>(p.mu3t, am, x[8]); p.mw1t = mac<EXACT>(p.mw1t, am, x[9]);
        p.mw2t = mac<EXACT>(p.mw2t, am, x[10]); p.mw3t = mac<EXACT>(p.mw3t, am, x[11]);
    };
    if (TOG && bkind == 2) {
        walk(valid, PAB{}, [&](const T *x, T am, T a1, T a2, T a3, T a4, T a5, T a6) __attribute__((always_inline)) {
            products_a(std::true_type{}, x, am, a1, a2, a3, a4, a5, a6);
            products_b(x + 10, am);
        });
    } else if (bkind == 2) {
        walk(valid, PA{}, [&](const T *x, T am, T a1, T a2, T a3, T a4, T a5, T a6) __attribute__((always_inline)) {
            products_a(std::true_type{}, x, am, a1, a2, a3, a4, a5, a6);
        });
    } else {
        walk(valid, PA{}, [&](const T *x, T am, T a1, T a2, T a3, T a4, T a5, T a6) __attribute__((always_inline)) {
            products_a(std::false_type{}, x, am, a1, a2, a3, a4, a5, a6);
        });
    }
    // the row's own U, W and memory fields
    T self[10];
    fields(PA{}, own, self);
    const T own_u = self[0], own_w = self[1], *mem = self + 2;
    if (bkind == 2) {
        if constexpr (!TOG) {
            __syncthreads();
            fetch_b(0, sb[0]);
            if (second) fetch_b(1, sb[1]);
            stash_b(0);
            if (second) stash_b(1);
            __syncthreads();
            walk(pml, PB{}, [&](const T *x, T am, T, T, T, T, T, T) __attribute__((always_inline)) {
                products_b(x, am);
            });
        }
        if (pml) {
            c.dx = at32(cf + DX * cs, rc);
            c.dy = at32(cf + DY * cs, rc);
            c.dxx = at32(cf + DXX * cs, rc);
            c.dyy = at32(cf + DYY * cs, rc);
            c.dxxp = at32(cf + DXXP * cs, rc);
            c.dyyp = at32(cf + DYYP * cs, rc);
        }
    }
    if (!valid) return;
    // rows outside the layers: these products meet zero profiles only
    if (!pml) {
        p.s5u = p.s5w = p.s6u = p.s6w = T(0);
        p.mu1t = p.mu1 = p.mu2t = p.mu2 = p.mu3t = p.mu3 = T(0);
        p.mw1t = p.mw1 = p.mw2t = p.mw2 = p.mw3t = p.mw3 = T(0);
    }
    if constexpr (CPS) {
        // per-shot density: scale this row of the operator's M
        p.mu1t *= mrow; p.mu1 *= mrow; p.mlx1 *= mrow; p.mlx2 *= mrow; p.mu2t *= mrow; p.mu2 *= mrow;
        p.mu3t *= mrow; p.mu3 *= mrow; p.mlx3 *= mrow; p.mlx4 *= mrow;
        p.mw1t *= mrow; p.mw1 *= mrow; p.mly1 *= mrow; p.mly2 *= mrow; p.mw2t *= mrow; p.mw2 *= mrow;
        p.mw3t *= mrow; p.mw3 *= mrow; p.mly3 *= mrow; p.mly4 *= mrow;
    }
    // source term: see step_tile
    const double ps = ro(a.wavelet)[t];
    double su = 0.0 * ps * a.src_u, sw = 0.0 * ps * a.src_w;
    if (info & GI_SRC)
        for (int q = a.src_ptr[r]; q < a.src_ptr[r + 1]; ++q)
            if (a.src_shot[q] == s) {
                su = 1.0 * ps * a.src_wt[2 * q];
                sw = 1.0 * ps * a.src_wt[2 * q + 1];
            }
    const T dt = a.dt;
    T rhs[14];
    split_rhs(p, c, dt, (T)su, (T)sw, rhs);

    // ---- lumped-mass solve with Dirichlet clamp (:681-729) ------------
    T an[6], ln[8];
    if constexpr (EXACT) {
        const bool clamp = CPS ? at32(a.flag + (size_t)s * a.n, (uint32_t)r * 4) == 1 : (info & GI_CLAMP) != 0;
        if (mass != T(0)) {
            if (clamp) {
#pragma unroll
                for (int q = 0; q < 6; ++q) an[q] = T(0);
#pragma unroll
                for (int q = 0; q < 8; ++q) ln[q] = T(0);
            } else {
                const T m1 = T(1.0) * mass;
#pragma unroll
                for (int q = 0; q < 3; ++q) an[q] = rhs[q] / m1, an[3 + q] = rhs[7 + q] / m1;
#pragma unroll
                for (int q = 0; q < 4; ++q) ln[q] = rhs[3 + q] / m1, ln[4 + q] = rhs[10 + q] / m1;
            }
        } else {
            // zero lumped mass: the reference leaves the outputs untouched
#pragma unroll
            for (int q = 0; q < 6; ++q) an[q] = acc[q];
#pragma unroll
            for (int q = 0; q < 8; ++q) ln[q] = mem[q];
            atomicOr(&a.ctrl->err, 1);
        }
    } else {
        // mass holds 1/mass_lump with the Dirichlet flag folded in as 0
#pragma unroll
        for (int q = 0; q < 3; ++q) an[q] = rhs[q] * mass, an[3 + q] = rhs[7 + q] * mass;
#pragma unroll
        for (int q = 0; q < 4; ++q) ln[q] = rhs[3 + q] * mass, ln[4 + q] = rhs[10 + q] * mass;
    }

    // ---- Newmark update (:757-776) ---------------------------------------
    const T ca = a.ca, al = a.alpha, cd = a.cd, de = a.delta;
    T cn[6];
    T sum_u, sum_w;
    if (agg) {
        // the three split updates of a summed row, added (see step_tile)
        const T an_s[2] = {an[0] + an[1] + an[2], an[3] + an[4] + an[5]};
        T res[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const T d = h ? own_w : own_u;
            const T pv = acc[3 * h];
            if constexpr (KAHAN) {
                const T inc = pv * dt + al * an_s[h] * dt * dt;
                const T y = inc - kt[3 * h];
                const T sm = d + y;
                cn[3 * h] = (sm - d) - y;
                if constexpr (!C16) at32(cout + h * F, rb) = cn[3 * h];
                res[h] = sm;
            } else {
                res[h] = d + pv * dt + al * an_s[h] * dt * dt;
            }
            at32(out + (U1TT + 3 * h) * F, rb) = pv + (de + ca) * an_s[h] * dt;
        }
        sum_u = res[0];
        sum_w = res[1];
        if constexpr (C16) at32(wout, rw) = bf16_bits(cn[0]) | (bf16_bits(cn[3]) << 16);
    } else {
        T dn[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const T d = disp[q];
            if constexpr (EXACT) {
                dn[q] = d + vel[q] * dt + (ca * acc[q] + al * an[q]) * dt * dt;
                at32(out + (U1T + q) * F, rb) = vel[q] + (cd * acc[q] + de * an[q]) * dt;
                at32(out + (U1TT + q) * F, rb) = an[q];
            } else {
                // p-form: the acceleration slot holds p = v + ca dt a
                const T pv = acc[q];
                if constexpr (KAHAN) {
                    const T inc = pv * dt + al * an[q] * dt * dt;
                    const T y = inc - kt[q];
                    const T sm = d + y;
                    cn[q] = (sm - d) - y;
                    if constexpr (!C16) at32(cout + q * F, rb) = cn[q];
                    dn[q] = sm;
                } else {
                    dn[q] = d + pv * dt + al * an[q] * dt * dt;
                }
                at32(out + (U1T + q) * F, rb) = pv + de * an[q] * dt;
                at32(out + (U1TT + q) * F, rb) = pv + (de + ca) * an[q] * dt;
            }
            at32(out + (U1 + q) * F, rb) = dn[q];
        }
        if constexpr (C16) {
#pragma unroll
            for (int k = 0; k < 3; ++k) at32(wout + k * F, rw) = bf16_bits(cn[2 * k]) | (bf16_bits(cn[2 * k + 1]) << 16);
        }
        sum_u = dn[0] + dn[1] + dn[2];
        sum_w = dn[3] + dn[4] + dn[5];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) at32(out + (LX1 + q) * F, rb) = ln[q];
    at32(uwout, rb) = sum_u;
    at32(uwout + F, rb) = sum_w;

    // ---- receivers sitting on this node --------------------------------
    if (info & GI_REC) {
        for (int q = a.rec_ptr[r]; q < a.rec_ptr[r + 1]; ++q) {
            const size_t w = ((size_t)s * a.nsteps_max + t) * a.rec_num + a.rec_idx[q];
            a.seis_u[w] = (double)sum_u;
            a.seis_w[w] = (double)sum_w;
        }
    }
}

template <class T, int PREC, bool CPS, int MODE, bool TOG>
__global__ __launch_bounds__(GRID_BLOCK) void grid_step_kernel(const StepArgs<T> a, const GridArgs<T> g, int slot)
{
    const int t = __hip_atomic_load(&a.ctrl->step[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned int bid = blockIdx.x, nact = 1;
    unsigned int nb = (unsigned int)g.g.npatch;
    bool lead = bid == 0 && threadIdx.x == 0;
    if (a.S > 1) {
        // shots are sorted by decreasing step count: the active ones come first,
        // and the launch hands out only their tiles
        if (lead) __hip_atomic_store(&a.ctrl->step[slot ^ 1], t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lead = false;
        nact = t < a.nsteps_max ? (unsigned int)ro(a.active)[t] : 0u;
        nb *= nact;
        if (bid >= nb) return;
    }
    if (a.xcd_stripe > 0) bid = xcd_striped(bid, nb, (unsigned int)a.xcd_stripe);
    else if (a.xcd_remap) bid = xcd_contiguous(bid, nb);
    // shot after shot: neighbouring patches of a shot follow each other, so their common
    // halo is still in L2 (patch after patch, the shots of each together: 128 shots Q4
    // 400 x 400 FP32 1214 us per step against 844, 64 shots Q4 300 x 300 FP64 850 / 645)
    grid_tile<T, PREC, CPS, MODE, TOG>(a, g, t, slot, (int)(bid % (unsigned int)g.g.npatch),
                                       (int)(bid / (unsigned int)g.g.npatch), lead);
}

template <class T, int PREC, bool CPS>
static hipError_t launch_grid_mode(const StepArgs<T> &a, const GridArgs<T> &g, int nshots, int slot, size_t lds,
                                   hipStream_t st)
{
    const dim3 grid((unsigned int)g.g.npatch * (unsigned int)nshots), block(g.g.most);
#define SFG_GM(M, TG) hipLaunchKernelGGL((grid_step_kernel<T, PREC, CPS, M, TG>), grid, block, lds, st, a, g, slot)
    switch (g.mode) {
    case GRID_CLASS: if (g.together) SFG_GM(GRID_CLASS, true); else SFG_GM(GRID_CLASS, false); break;
    case GRID_CLASS_S: if (g.together) SFG_GM(GRID_CLASS_S, true); else SFG_GM(GRID_CLASS_S, false); break;
    case GRID_ROWS: if (g.together) SFG_GM(GRID_ROWS, true); else SFG_GM(GRID_ROWS, false); break;
    default: return hipErrorInvalidValue;
    }
#undef SFG_GM
    return hipGetLastError();
}

hipError_t launch_grid_step(int precision, bool cps, const void *sa, const void *ga, int nshots, int slot, size_t lds,
                            hipStream_t st)
{
#define SFG_GS(T, P)                                                                                                 \
    (cps ? launch_grid_mode<T, P, true>(*(const StepArgs<T> *)sa, *(const GridArgs<T> *)ga, nshots, slot, lds, st)  \
         : launch_grid_mode<T, P, false>(*(const StepArgs<T> *)sa, *(const GridArgs<T> *)ga, nshots, slot, lds, st))
    switch (precision) {
    case 0: return SFG_GS(double, 0);
    case 1: return SFG_GS(float, 1);
    case 2: return SFG_GS(float, 2);
    case 3: return SFG_GS(float, 3);
    default: return hipErrorInvalidValue;
    }
#undef SFG_GS
}

// One tile of a multi-run's grid launch: a run's tiles are its (patch, shot) pairs,
// patches fastest.
template <class T, int PREC, bool TOG>
__device__ __forceinline__ void multi_grid_tile(const GridRun<T> *__restrict__ runs, const int *__restrict__ tile_start,
                                                int nruns, int t, int slot, int tile)
{
    int r = 0;
    while (r + 1 < nruns && tile >= tile_start[r + 1]) ++r;
    const StepArgs<T> &a = runs[r].a;
    const GridArgs<T> &g = runs[r].g;
    const int local = tile - tile_start[r], s = local / g.g.npatch, patch = local - s * g.g.npatch;
    if (a.S > 1 && s >= (t < a.nsteps_max ? ro(a.active)[t] : 0)) return;
#define SFG_GT(C, M) grid_tile<T, PREC, C, M, TOG>(a, g, t, slot, patch, s, false)
    if (a.cps) {
        if (g.mode == GRID_CLASS) SFG_GT(true, GRID_CLASS);
        else if (g.mode == GRID_CLASS_S) SFG_GT(true, GRID_CLASS_S);
        else SFG_GT(true, GRID_ROWS);
    } else {
        if (g.mode == GRID_CLASS) SFG_GT(false, GRID_CLASS);
        else if (g.mode == GRID_CLASS_S) SFG_GT(false, GRID_CLASS_S);
        else SFG_GT(false, GRID_ROWS);
    }
#undef SFG_GT
}

// Several grid-layout runs in one launch per step (see multi_step_kernel).
template <class T, int PREC, bool TOG>
__global__ __launch_bounds__(GRID_BLOCK) void multi_grid_kernel(const GridRun<T> *__restrict__ runs,
                                                                const int *__restrict__ tile_start, int nruns,
                                                                int xcd_remap, int slot)
{
    const int t = begin_step(runs[0].a.ctrl, slot);
    const unsigned int nb = gridDim.x;
    unsigned int bid = blockIdx.x;
    if (xcd_remap > 1) bid = xcd_striped(bid, nb, (unsigned int)(xcd_remap - 1));
    else if (xcd_remap) bid = xcd_contiguous(bid, nb);
    multi_grid_tile<T, PREC, TOG>(runs, tile_start, nruns, t, slot, (int)bid);
}

// Persistent form for small batches (see multi_persistent_kernel): a cooperative grid
// steps nsteps steps, each block taking every gridDim.x-th tile (these runs have few and
// equal tiles), with a grid-wide barrier between steps.  Fields are staged in two parts,
// the form of less LDS, so that at least two blocks fit a CU.  The launch after which the
// guard interval is over for every run (finish) hands the step count on.
template <class T, int PREC>
__global__ __launch_bounds__(GRID_BLOCK, 2) void multi_grid_persistent_kernel(const GridRun<T> *__restrict__ runs,
                                                                              const int *__restrict__ tile_start,
                                                                              int nruns, int ntiles, int slot,
                                                                              int nsteps, int finish)
{
    cooperative_groups::grid_group grid = cooperative_groups::this_grid();
    Ctrl *ctrl = runs[0].a.ctrl;
    const int t0 = __hip_atomic_load(&ctrl->step[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int k = 0; k < nsteps; ++k) {
        for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
            multi_grid_tile<T, PREC, false>(runs, tile_start, nruns, t0 + k, (slot + k) & 1, tile);
            __syncthreads(); // (the next tile overwrites the LDS)
        }
        grid.sync();
    }
    if (finish && blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(&ctrl->step[slot ^ (nsteps & 1)], t0 + nsteps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

static const void *grid_persistent_fn(int precision)
{
    switch (precision) {
    case 0: return (const void *)multi_grid_persistent_kernel<double, 0>;
    case 1: return (const void *)multi_grid_persistent_kernel<float, 1>;
    case 2: return (const void *)multi_grid_persistent_kernel<float, 2>;
    case 3: return (const void *)multi_grid_persistent_kernel<float, 3>;
    default: return nullptr;
    }
}

hipError_t grid_persistent_blocks_per_cu(int precision, int most, size_t lds, int *per_cu)
{
    const void *f = grid_persistent_fn(precision);
    if (!f) return hipErrorInvalidValue;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, f, most, lds);
}

hipError_t launch_grid_persistent(int precision, const void *runs_dev, const int *tile_start_dev, int nruns, int ntiles,
                                  int most, int blocks, int slot, int nsteps, size_t lds, bool finish, hipStream_t st)
{
    const void *f = grid_persistent_fn(precision);
    if (!f) return hipErrorInvalidValue;
    int fin = finish ? 1 : 0;
    void *kargs[] = {(void *)&runs_dev, (void *)&tile_start_dev, (void *)&nruns, (void *)&ntiles,
                     (void *)&slot, (void *)&nsteps, (void *)&fin};
    return hipLaunchCooperativeKernel(f, dim3(blocks), dim3(most), kargs, (unsigned int)lds, st);
}

hipError_t launch_multi_grid(int precision, const void *runs_dev, const int *tile_start_dev, int nruns, int ntiles,
                             int most, int xcd_remap, int slot, size_t lds, bool together, hipStream_t st)
{
#define SFG_MG(T, P, TG)                                                                                   \
    hipLaunchKernelGGL((multi_grid_kernel<T, P, TG>), dim3(ntiles), dim3(most), lds, st,                  \
                       (const GridRun<T> *)runs_dev, tile_start_dev, nruns, xcd_remap, slot)
    switch (precision) {
    case 0: if (together) SFG_MG(double, 0, true); else SFG_MG(double, 0, false); break;
    case 1: if (together) SFG_MG(float, 1, true); else SFG_MG(float, 1, false); break;
    case 2: if (together) SFG_MG(float, 2, true); else SFG_MG(float, 2, false); break;
    case 3: if (together) SFG_MG(float, 3, true); else SFG_MG(float, 3, false); break;
    default: return hipErrorInvalidValue;
    }
#undef SFG_MG
    return hipGetLastError();
}

// FP64 patches may take more than the default 64 KB of dynamic LDS
// (GRID_HALO_MAX x 24 values x 8 bytes + GRID_TABLE entries of 64 bytes = 122 KB)
hipError_t allow_grid_lds()
{
    const int bytes = (int)((GRID_HALO_MAX * 24 + GRID_TABLE * 8) * sizeof(double));
#define SFG_GF(C, M, TG) (const void *)grid_step_kernel<double, 0, C, M, TG>
    const void *f[] = {SFG_GF(false, GRID_CLASS, true), SFG_GF(false, GRID_CLASS_S, true), SFG_GF(false, GRID_ROWS, true),
                       SFG_GF(true, GRID_CLASS, true), SFG_GF(true, GRID_CLASS_S, true), SFG_GF(true, GRID_ROWS, true),
                       SFG_GF(false, GRID_CLASS, false), SFG_GF(false, GRID_CLASS_S, false),
                       SFG_GF(false, GRID_ROWS, false), SFG_GF(true, GRID_CLASS, false),
                       SFG_GF(true, GRID_CLASS_S, false), SFG_GF(true, GRID_ROWS, false),
                       (const void *)multi_grid_kernel<double, 0, true>, (const void *)multi_grid_kernel<double, 0, false>,
                       grid_persistent_fn(0)};
#undef SFG_GF
    hipError_t e = hipSuccess;
    for (const void *k : f)
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    return e;
}

// ---- plan building ---------------------------------------------------------------

__global__ void grid_reach_kernel(int n, const int *rp, const int *ci, int line, int *reach, int *bad)
{
    int mx = 0, my = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int iy = i / line, ix = i - iy * line;
        for (int k = rp[i]; k < rp[i + 1]; ++k) {
            const int j = ci[k], jy = j / line, jx = j - jy * line;
            mx = max(mx, abs(jx - ix));
            my = max(my, abs(jy - iy));
        }
    }
    if (mx > GRID_REACH || my > GRID_REACH) atomicOr(bad, 1);
    atomicMax(&reach[0], min(mx, GRID_REACH));
    atomicMax(&reach[1], min(my, GRID_REACH));
}

hipError_t launch_grid_reach(int n, const int *rp, const int *ci, int line, int *reach, int *bad, hipStream_t st)
{
    hipLaunchKernelGGL(grid_reach_kernel, dim3(std::min((n + 255) / 256, 2048)), dim3(256), 0, st, n, rp, ci, line, reach,
                       bad);
    return hipGetLastError();
}

__device__ __forceinline__ unsigned long long mix(unsigned long long h, unsigned long long v)
{
    h ^= v + 0x9E3779B97F4A7C15ull + (h << 6) + (h >> 2);
    h *= 0xD6E8FEB86659FD93ull;
    return h ^ (h >> 32);
}

// position of column j relative to row i in units of a halo of width W
__device__ __forceinline__ int halo_offset(int i, int j, int line, int W)
{
    const int iy = i / line, jy = j / line;
    return (jy - iy) * W + (j - jy * line) - (i - iy * line);
}

// (columns within GRID_REACH of the row: equal j - i means equal dx and dy)
__global__ void grid_hash_kernel(int n, const int *rp, const int *ci, const double *v, size_t nnz,
                                 unsigned long long *h)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        unsigned long long hs = 1469598103934665603ull, hm = 88172645463325252ull;
        for (int k = rp[i]; k < rp[i + 1]; ++k) {
            unsigned long long x[7];
            for (int m = 0; m < 7; ++m) x[m] = (unsigned long long)__double_as_longlong(v[m * nnz + k]);
            hs = mix(hs, (unsigned long long)(ci[k] - i));
            for (int m = 1; m < 7; ++m) hs = mix(hs, x[m]);
            hm = mix(hm, x[0]);
        }
        h[i] = hs;
        h[(size_t)n + i] = mix(hs, hm);
    }
}

hipError_t launch_grid_hash(int n, const int *rp, const int *ci, const double *v64, size_t nnz,
                            unsigned long long *h, hipStream_t st)
{
    hipLaunchKernelGGL(grid_hash_kernel, dim3(std::min((n + 63) / 64, 8192)), dim3(64), 0, st, n, rp, ci, v64, nnz, h);
    return hipGetLastError();
}

__global__ void grid_check_kernel(int n, const int *rp, const int *ci, const double *v, size_t nnz, int m0,
                                  const int *cls, const int *rep, int *bad)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const int r = rep[cls[i]], len = rp[i + 1] - rp[i];
        bool same = len == rp[r + 1] - rp[r];
        for (int q = 0; same && q < len; ++q) {
            const int k = rp[i] + q, kr = rp[r] + q;
            same = ci[k] - i == ci[kr] - r;
            for (int m = m0; m < 7; ++m)
                same = same && __double_as_longlong(v[m * nnz + k]) == __double_as_longlong(v[m * nnz + kr]);
        }
        if (!same) atomicOr(bad, 1);
    }
}

hipError_t launch_grid_check(int n, const int *rp, const int *ci, const double *v64, size_t nnz, int m0, const int *cls,
                             const int *rep, int *bad, hipStream_t st)
{
    hipLaunchKernelGGL(grid_check_kernel, dim3(std::min((n + 63) / 64, 8192)), dim3(64), 0, st, n, rp, ci, v64, nnz, m0,
                       cls, rep, bad);
    return hipGetLastError();
}

// One block per patch: a row's place is the number of rows with a smaller key
// (ties by position), counted over the patch's keys in LDS.
__global__ __launch_bounds__(GRID_BLOCK) void grid_sort_kernel(const GridShape g, int mode, const int *rp,
                                                               const int *key, const int *cptr, int *rows, int *cls,
                                                               int *slice, int *smax)
{
    __shared__ int keys[GRID_BLOCK], srow[GRID_BLOCK], scls[GRID_BLOCK];
    const int tid = threadIdx.x, patch = blockIdx.x, R = g.most;
    const int py = patch / g.px, px = patch - py * g.px;
    const int x = px * g.pw + tid % g.pw, y = py * g.ph + tid / g.pw;
    const bool in = tid < g.pw * g.ph && x < g.line && y < g.lines;
    const int row = in ? y * g.line + x : -1;
    const int len = in ? rp[row + 1] - rp[row] : 0;
    const int c = !in ? 0 : (mode == GRID_ROWS ? 0 : cptr[key[row]]) | len << 24;
    keys[tid] = !in ? 0x7fffffff : mode == GRID_ROWS ? -len : c & 0xffffff;
    __syncthreads();
    int rank = 0;
    for (int q = 0; q < R; ++q) rank += keys[q] < keys[tid] || (keys[q] == keys[tid] && q < tid);
    srow[rank] = row;
    scls[rank] = c;
    __syncthreads();
    const size_t o = (size_t)patch * R + tid;
    rows[o] = srow[tid];
    cls[o] = scls[tid];
    if ((tid & 63) == 0) {
        int m = 0, same = 1;
        for (int l = 0; l < 64; ++l) {
            const int r = srow[tid + l];
            if (r < 0) continue;
            m = max(m, rp[r + 1] - rp[r]);
            same = same && scls[tid + l] == scls[tid];
        }
        const int w = patch * (R / 64) + tid / 64;
        smax[w] = m;
        slice[w] = m | (mode != GRID_ROWS && same ? 0x100 : 0);
    }
}

hipError_t launch_grid_sort(const GridShape &g, int mode, const int *rp, const int *key, const int *cptr, int *rows,
                            int *cls, int *slice, int *smax, hipStream_t st)
{
    if (g.most > GRID_BLOCK || g.most % 64 || g.pw * g.ph > g.most) return hipErrorInvalidValue;
    hipLaunchKernelGGL(grid_sort_kernel, dim3(g.npatch), dim3(g.most), 0, st, g, mode, rp, key, cptr, rows, cls, slice,
                       smax);
    return hipGetLastError();
}

// keys of the places: entry | nonzeros << 24 -> entry | halo position << 12 | nonzeros << 24
__global__ __launch_bounds__(GRID_BLOCK) void grid_place_kernel(const GridShape g, const int *rows, int *cls)
{
    const int patch = blockIdx.x, py = patch / g.px, px = patch - py * g.px;
    const size_t at = (size_t)patch * g.most + threadIdx.x;
    const int row = rows[at];
    if (row < 0) {
        cls[at] = 0;
        return;
    }
    const int y = row / g.line, x = row - y * g.line;
    const int own = (y - py * g.ph + g.hy) * g.W + x - px * g.pw + g.hx;
    cls[at] = (cls[at] & ~0xfff000) | own << 12;
}

hipError_t launch_grid_place(const GridShape &g, const int *rows, int *cls, hipStream_t st)
{
    hipLaunchKernelGGL(grid_place_kernel, dim3(g.npatch), dim3(g.most), 0, st, g, rows, cls);
    return hipGetLastError();
}

template <class E>
__global__ void grid_table_kernel(int nitems, const int *rep, const int *dst, const int *rp, const int *ci, int line,
                                  int W, const E *v, size_t nnz, E *tab)
{
    const int c = blockIdx.x;
    if (c >= nitems) return;
    const int r = rep[c], k0 = rp[r], len = rp[r + 1] - k0;
    for (int q = threadIdx.x; q < len; q += blockDim.x) {
        E *o = tab + ((size_t)dst[c] + q) * 8;
        for (int m = 0; m < 7; ++m) o[m] = v[m * nnz + k0 + q];
        o[7] = (E)halo_offset(r, ci[k0 + q], line, W);
    }
}

hipError_t launch_grid_table(int nitems, const int *rep, const int *dst, const int *rp, const int *ci, int line, int W,
                             const void *vals, size_t nnz, int elem, void *tab, hipStream_t st)
{
    if (elem == 8)
        hipLaunchKernelGGL(grid_table_kernel<double>, dim3(nitems), dim3(64), 0, st, nitems, rep, dst, rp, ci, line, W,
                           (const double *)vals, nnz, (double *)tab);
    else
        hipLaunchKernelGGL(grid_table_kernel<float>, dim3(nitems), dim3(64), 0, st, nitems, rep, dst, rp, ci, line, W,
                           (const float *)vals, nnz, (float *)tab);
    return hipGetLastError();
}

template <class E>
__global__ __launch_bounds__(64) void grid_values_kernel(int mode, const int *rows, const int *moff, const int *smax,
                                                         const int *rp, const int *ci, int line, int W, const E *v,
                                                         size_t nnz, E *mval, int *sdel)
{
    const int w = blockIdx.x, lane = threadIdx.x;
    const int row = rows[(size_t)w * 64 + lane], m0 = moff[w];
    const int k0 = row >= 0 ? rp[row] : 0, len = row >= 0 ? rp[row + 1] - k0 : 0;
    for (int q = 0; q < smax[w]; ++q) {
        const size_t slot = (size_t)m0 + q;
        if (mode == GRID_CLASS_S) {
            mval[slot * 64 + lane] = q < len ? v[k0 + q] : E(0);
        } else {
            for (int m = 0; m < 7; ++m) mval[(slot * 7 + m) * 64 + lane] = q < len ? v[m * nnz + k0 + q] : E(0);
            sdel[slot * 64 + lane] = q < len ? halo_offset(row, ci[k0 + q], line, W) : 0;
        }
    }
}

hipError_t launch_grid_values(int nwaves, int mode, const int *rows, const int *moff, const int *smax, const int *rp,
                              const int *ci, int line, int W, const void *vals, size_t nnz, int elem, void *mval,
                              int *sdel, hipStream_t st)
{
    if (elem == 8)
        hipLaunchKernelGGL(grid_values_kernel<double>, dim3(nwaves), dim3(64), 0, st, mode, rows, moff, smax, rp, ci,
                           line, W, (const double *)vals, nnz, (double *)mval, sdel);
    else
        hipLaunchKernelGGL(grid_values_kernel<float>, dim3(nwaves), dim3(64), 0, st, mode, rows, moff, smax, rp, ci, line,
                           W, (const float *)vals, nnz, (float *)mval, sdel);
    return hipGetLastError();
}

__global__ __launch_bounds__(GRID_BLOCK) void grid_info_kernel(const int *rows, const int *pml, const int *src_ptr,
                                                               const int *rec_ptr, const int *flag,
                                                               unsigned char *info, int *bkind)
{
    __shared__ int most;
    if (threadIdx.x == 0) most = 0;
    __syncthreads();
    const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int r = rows[at];
    int v = 0;
    if (r >= 0) {
        v = pml[r];
        atomicMax(&most, v);
        if (src_ptr[r + 1] > src_ptr[r]) v |= GI_SRC;
        if (rec_ptr[r + 1] > rec_ptr[r]) v |= GI_REC;
        if (flag && flag[r] == 1) v |= GI_CLAMP;
    }
    info[at] = (unsigned char)v;
    __syncthreads();
    if (threadIdx.x == 0) bkind[blockIdx.x] = most;
}

hipError_t launch_grid_info(const GridShape &g, const int *rows, const int *pml, const int *src_ptr,
                            const int *rec_ptr, const int *flag, unsigned char *info, int *bkind, hipStream_t st)
{
    hipLaunchKernelGGL(grid_info_kernel, dim3(g.npatch), dim3(g.most), 0, st, rows, pml, src_ptr, rec_ptr, flag, info,
                       bkind);
    return hipGetLastError();
}

} // namespace sfg
