// SQMR on the chip: many steps in one kernel, for problems whose state fits
// the register files and LDS.
//
// Small problems are bound by launches, not by work: step by step each of a
// step's four kernels pays its launch, a cold instruction cache (16–25 KB of
// straight code for the stencil) and the round trips of its first loads; a
// stencil launch of six blocks takes 16 µs.  Here every block keeps a box of
// cells for up to 512 steps: r, q and the stencil factors of its cells in
// registers, d and z in LDS or registers, and the scaled search direction
// X = q·T⁻¹ ∘ q of the box and its halo in LDS.  Per step the blocks exchange
// two things through memory: the partial sums of the two reductions, which
// also order the step, and the new r of their cells, from which each block
// forms its neighbours' q = r + β q itself.  What bounds a step are those two
// exchanges (about 2.5 µs each, a store and a load that meet at the device's
// coherence point) and 1.3–2.5 µs of LDS reads and FP64 arithmetic per box.
//
// Measured (FP64 SQMR, µs per step, step by step → resident): 16³ 35 → 7.3,
// 24³ 34 → 7.8, 36³ 37 → 10, 48³ 45 → 13; μ ≠ 1 on 48³ 49 → 15, full ε 70 → 15;
// FP32 vectors on 64³ 52 → 16 (19 with d and z in registers and 45 of those spilled).  A step takes 1.3–2 µs longer with two cells per
// thread than with one, and less with 256 threads of two cells than with 512
// of one (14.4 → 11.6 µs on 41×36×45: half the waves at each barrier, and the
// registers hold everything).  1,024 cells per block hold FP32 vectors with
// diagonal ε only, and those with d and z in LDS: no form uses scratch memory.
// With FP64 vectors, 1/μ or corner ε they spill 90–500 registers, and a trial
// of 16×8×8 boxes with FP64 vectors (428 spilled registers, 660 bytes of scratch
// a lane) ended in an illegal memory access.  Its index code, which is that of
// every form, stays inside all arrays (resident_index.hpp, host_checks.cpp);
// what else differed was the scratch and a step's end in the step itself, and
// no cause was shown, so it is not built: beyond 256 boxes of 512 cells those
// problems run step by step.
//
// A block only ever waits for blocks of its own launch, which is cooperative
// (every block has a place on the chip at once), and gives up after a limit.
#include "resident.hpp"
#include "resident_index.hpp"
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>

namespace mfd {

template <typename R>
struct ResArgs {
    DGrid<double> g;               // the grid, or its reflection along the axes of g.rmask
    const c64 *qs, *epsd, *epso, *muinv;
    c64 om2;
    cx<R> *r, *q, *d, *z;
    int64_t vs;                    // unknowns per right-hand side
    int nbx, nby, nb, rhs0;        // boxes per axis and per right-hand side; first right-hand side
    int steps, chunk;
    double near;
    unsigned long long *slots;     // [right-hand side of the launch][2][nb][8]
    cx<R> *xch;                    // [right-hand side of the launch][nb][cells of a box][3]: the boxes' new r
    Scal *scal;
};

// a value of another block's r: written by stores and read by loads that go to
// the device's coherence point (relaxed agent-scope atomics, 8 bytes each)
__device__ inline c64 sub(const c64 *p) {
    return mk<double>(__hip_atomic_load(&p->re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                      __hip_atomic_load(&p->im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline c32 sub(const c32 *p) {
    const unsigned long long w = __hip_atomic_load((const unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    c32 v;
    __builtin_memcpy(&v, &w, 8);
    return v;
}

constexpr unsigned long long RES_TICKS = 3000000000ull;   // 30 s of the 100 MHz counter

// Sum of v over the 64 lanes of a wave, in every lane, by register moves
// between lanes (a shuffle through the LDS path takes several times as long)
template <int CTRL>
__device__ inline double lane_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double wave_sum(double v) {
    v = lane_add<0xb1>(v);    // quad_perm 1,0,3,2
    v = lane_add<0x4e>(v);    // quad_perm 2,3,0,1
    v = lane_add<0x141>(v);   // row_half_mirror
    v = lane_add<0x140>(v);   // row_mirror: the sum of each row of 16 lanes
    double r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const long long b = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_readlane((int)b, 16 * k), hi = __builtin_amdgcn_readlane((int)(b >> 32), 16 * k);
        r[k] = __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
    }
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// A sum over all threads of all nb blocks of a right-hand side, in a fixed
// order, which is also the step's barrier: once it is complete every block has
// arrived, and what its threads published before (and waited for) can be
// read.  Each block stores its partial sums as words of 32 data bits and the
// 32-bit tag of this arrival, so a word is valid by itself and no fence or
// counter is needed.
template <int NV, int NT>
__device__ inline void arrive(unsigned long long *slots, int box, unsigned tag, double (&v)[NV], double (*sh)[3]) {
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x;
#pragma unroll
    for (int a = 0; a < NV; ++a) v[a] = wave_sum(v[a]);
    if ((tid & 63) == 0)
#pragma unroll
        for (int a = 0; a < NV; ++a) sh[tid >> 6][a] = v[a];
    // the stores this wave published have reached the coherence point before
    // it passes the barrier, so before its block's arrival can be seen
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid < 2 * NV) {
        double s = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += sh[w][tid >> 1];
        const unsigned long long bits = (unsigned long long)__double_as_longlong(s);
        const unsigned long long word = ((tid & 1) ? (bits & 0xffffffff00000000ull) : (bits << 32)) | tag;
        __hip_atomic_store(&slots[8 * box + tid], word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
// Thread b waits for block b's words (after the time limit *fail is set, for
// the whole block); the sums are then in v of every thread.
template <int NV, int NT>
__device__ inline void collect(const unsigned long long *slots, int nb, unsigned tag, double (&v)[NV], double (*sh)[3],
                               int *fail) {
    constexpr int NW = NT / 64;
    const int tid = threadIdx.x;
    double t[NV];
#pragma unroll
    for (int a = 0; a < NV; ++a) t[a] = 0;
    for (int b = tid; b < nb; b += NT) {
        unsigned long long w[2 * NV];
        unsigned spins = 0;
        unsigned long long t0 = 0;
        while (true) {
            bool ok = true;
#pragma unroll
            for (int a = 0; a < 2 * NV; ++a)
                w[a] = __hip_atomic_load(&slots[8 * b + a], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int a = 0; a < 2 * NV; ++a) ok = ok && (unsigned)w[a] == tag;
            if (ok) break;
            if ((++spins & 255u) == 0) {
                const unsigned long long now = wall_clock64();
                if (t0 == 0) t0 = now;
                else if (now - t0 > RES_TICKS) { *fail = 1; break; }
            }
        }
#pragma unroll
        for (int a = 0; a < NV; ++a)
            t[a] += __longlong_as_double((long long)((w[2 * a + 1] & 0xffffffff00000000ull) | (w[2 * a] >> 32)));
    }
    if ((tid & ~63) < nb)
#pragma unroll
        for (int a = 0; a < NV; ++a) t[a] = wave_sum(t[a]);
    if ((tid & 63) == 0)
#pragma unroll
        for (int a = 0; a < NV; ++a) sh[tid >> 6][a] = t[a];
    __syncthreads();
#pragma unroll
    for (int a = 0; a < NV; ++a) {
        double s = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) s += sh[w][a];
        v[a] = s;
    }
}

template <typename R, bool OFFD, bool MU, int TX, int TY, int TZ, int CPT>
__global__ __launch_bounds__(TX * TY * TZ / CPT, TX *TY *TZ / CPT <= 256 ? 1 : 2) void k_resident(ResArgs<R> A) {
    using C = BoxCfg<TX, TY, TZ, CPT>;
    constexpr int NT = C::NT, NHS = C::NHS, NW = NT / 64;
    // 1D factors of the box's columns, rows and planes: 1/∆l_D, 1/∆l_P, their
    // products with the plane's and the previous plane's 1/∆l_D (zero past a
    // non-Bloch end, and on a one-cell Bloch axis, where the second difference
    // is a multiple of the value itself and part of the diagonal), ∆l_D, ∆l_P;
    // then the previous 1/∆l_D (MU) and the corner-average weights (OFFD)
    enum { D_ = 0, P_, EP, EM, SD, SP, DM, W0 = DM + (MU ? 1 : 0), W1, NROW = W0 + (OFFD ? 2 : 0) };
    __shared__ c64 Xs[C::XS];
    __shared__ c64 tb[NROW][C::NTAB];
    constexpr bool DZL = box_dz_lds<C>(sizeof(cx<R>));   // d and z: in LDS, else in registers
    constexpr int MX = C::MX, MY = C::MY, MZ = C::MZ;
    constexpr bool ML = MU && CPT * NT <= 512;   // (MU) 1/μ of the box and one cell behind it in LDS
    __shared__ cx<R> Dz[DZL ? 6 * CPT * NT : 1];
    __shared__ c64 Ms[ML ? 3 * MX * MY * MZ : 1];
    __shared__ double sh[NW][3], sh2[NW][3];
    __shared__ Scal S;              // the same in every block
    __shared__ double s_tot[3], s_c2t2;   // of the step being finished: its sums, and the d, z coefficients
    __shared__ c64 s_c2a;
    __shared__ int s_stop, fail;
    __shared__ c64 wph[27];         // phase of a staged value by its wraps: none, low, high end of each axis (1, 3, 9)
    const DGrid<double> &g = A.g;
    const int tid = threadIdx.x;
    const int rl = (int)blockIdx.x / A.nb, box = (int)blockIdx.x - rl * A.nb, rhs = A.rhs0 + rl;
    const bool lead = box == 0 && tid == 0;
    {
        const Scal &G = A.scal[rhs];
        if (G.done || G.conv) {   // nothing to do (every block reads a flag set before the launch)
            if (lead) A.scal[rhs].done = 1;
            return;
        }
        if (tid == 0) {
            S = G;
            fail = 0;
            s_stop = 0;
        }
        if (tid < 27) {
            auto f = [&](int w, c64 lo, c64 hi) { return w == 0 ? mk<double>(1, 0) : (w == 1 ? lo : hi); };
            wph[tid] = f(tid % 3, g.phinv[0], g.ph[0]) * f(tid / 3 % 3, g.phinv[1], g.ph[1]) * f(tid / 9, g.phinv[2], g.ph[2]);
        }
    }
    unsigned long long *slA = A.slots + (size_t)rl * RES_SLOT_WORDS * A.nb, *slB = slA + 8 * A.nb;
    const int bx = box % A.nbx, by = (box / A.nbx) % A.nby, bz = box / (A.nbx * A.nby);
    const int i0 = bx * TX, j0 = by * TY, k0 = bz * TZ;
    const int N0 = g.N[0], N1 = g.N[1], N2 = g.N[2];
    const int64_t off = (int64_t)rhs * A.vs;
    cx<R> *rg = A.r + off, *qg = A.q + off, *dg = A.d + off, *zg = A.z + off;
    const BoxIndex<C> ix{N0, N1, N2, g.bloch[0], g.bloch[1], g.bloch[2], g.rmask, A.nbx, A.nby, g.cmpfirst, g.c0, g.nc, (int)g.M};
    auto inw = [&](int c) { return ix.inw(c); };
    auto phase = [&](c64 v, unsigned code) -> c64 {
        if (ix.slot_code(code)) v = v * wph[ix.slot_code(code)];
        return v;
    };
    // vector entries by 32-bit byte offset from the (uniform) base
    constexpr unsigned VB = sizeof(cx<R>);
    auto vent = [](auto *base, unsigned o) { return (decltype(base))((char *)base + o); };
    auto vcent = [](const c64 *base, unsigned o) { return *(const c64 *)((const char *)base + o); };
    cx<R> *xch = A.xch + (size_t)rl * A.nb * (3 * CPT * NT);   // the boxes' r
    auto xidx = [&](int i, int j, int k, int c) -> unsigned { return VB * ix.xidx(i, j, k, c); };
    auto vidx = [&](int p, int c) -> unsigned { return VB * (unsigned)ix.vidx(p, c); };

    // ---- this thread's cells, CPT neighbours along z (along y on a one-cell z
    // axis); one past a Bloch end (img) stands for its image
    int ii, jq, kq;
    ix.first_cell(tid, ii, jq, kq);
    constexpr int UJ = C::UJ, UK = C::UK, SX = C::SX, SY = C::SY, SZ = C::SZ, SU = C::SU;
    const int at0 = ix.staged(ii, jq, kq);
    bool own[CPT], img[CPT];
    unsigned mycode[CPT];
    int p[CPT];
    cx<R> r[CPT][3], q[CPT][3], qp[CPT][3];
    c64 qs[CPT][3];
    cx<R> d[DZL ? 1 : CPT][3], z[DZL ? 1 : CPT][3];
#pragma unroll
    for (int u = 0; u < CPT; ++u) {
        const int jj = jq + u * UJ, kk = kq + u * UK;
        own[u] = i0 + ii < N0 && j0 + jj < N1 && k0 + kk < N2;
        p[u] = ix.locate(i0 + ii, j0 + jj, k0 + kk, mycode[u]);
        img[u] = !own[u] && p[u] >= 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bool on = p[u] >= 0 && inw(c);
            r[u][c] = on ? *vent(rg, vidx(p[u], c)) : mk<R>((R)0, (R)0);
            q[u][c] = on ? *vent(qg, vidx(p[u], c)) : mk<R>((R)0, (R)0);
            qs[u][c] = on ? A.qs[3 * p[u] + c] : mk<double>(0, 0);
            const bool mine = own[u] && inw(c);
            const cx<R> dv = mine ? *vent(dg, vidx(p[u], c)) : mk<R>((R)0, (R)0);
            const cx<R> zv = mine ? *vent(zg, vidx(p[u], c)) : mk<R>((R)0, (R)0);
            if (DZL) {   // (each thread reads its own values only)
                Dz[(6 * u + c) * NT + tid] = dv;
                Dz[(6 * u + 3 + c) * NT + tid] = zv;
            } else {
                d[DZL ? 0 : u][c] = dv;
                z[DZL ? 0 : u][c] = zv;
            }
        }
    }
    // ---- its share of the halo: offset of its q·T⁻¹, offset of its r among the
    // boxes', and the place in LDS with the component and wraps (bit 31: there
    // is a value; bit 30: the slot is in use)
    unsigned hoff[NHS], hx[NHS], hpos[NHS];
    cx<R> hq[NHS];
#pragma unroll
    for (int s = 0; s < NHS; ++s) {
        const int h = tid + s * NT;
        int hi, hj, hk, c;
        hoff[s] = hx[s] = 0;
        hpos[s] = 0;
        hq[s] = mk<R>((R)0, (R)0);
        if (h >= C::NHALO) continue;
        ix.halo(h, hi, hj, hk, c);
        unsigned code;
        const int ph = ix.locate(i0 + hi, j0 + hj, k0 + hk, code);
        const int lp = ix.staged(hi, hj, hk) + c;
        hpos[s] = ix.pack(lp, c, code);
        if (ph >= 0 && inw(c)) {
            hoff[s] = 16u * (unsigned)(3 * ph + c);
            hx[s] = xidx(i0 + hi, j0 + hj, k0 + hk, c);
            hpos[s] |= 1u << 31;
            hq[s] = *vent(qg, vidx(ph, c));
        }
        Xs[lp] = mk<double>(0, 0);
    }
    auto fill = [&](int t, int ia, int Na, bool bloch, const c64 *sdD, const c64 *sdP, const c64 *inD, const c64 *inP) {
        ia = min(ia, Na - 1);
        const int im = ia > 0 ? ia - 1 : Na - 1;
        const c64 dd = inD[ia], pp = inP[ia], sD = sdD[ia];
        const c64 dm = ia > 0 || bloch ? inD[im] : mk<double>(0, 0);
        const bool one = Na == 1 && bloch;
        tb[D_][t] = dd;
        tb[P_][t] = pp;
        tb[EP][t] = one ? mk<double>(0, 0) : pp * dd;
        tb[EM][t] = one ? mk<double>(0, 0) : pp * dm;
        tb[SD][t] = sD;
        tb[SP][t] = sdP[ia];
        if (MU) tb[DM][t] = dm;
        if (OFFD) {
            tb[W0][t] = (0.5 * sD) * pp;
            tb[W1][t] = (0.5 * sdD[im]) * pp;
        }
    };
#define MFD_FILL(t, ia, a) fill(t, ia, g.N[a], g.bloch[a] != 0, g.sdl[DUAL][a], g.sdl[PRIM][a], g.sdlinv[DUAL][a], g.sdlinv[PRIM][a])
    if (tid < TX) MFD_FILL(tid, i0 + tid, 0);
    else if (tid < TX + TY) MFD_FILL(tid, j0 + tid - TX, 1);
    else if (tid < C::NTAB) MFD_FILL(tid, k0 + tid - TX - TY, 2);
#undef MFD_FILL
    auto neg = [&](int c, c64 v) { return (g.rmask >> c) & 1 ? -v : v; };   // E_c along a reflected axis
    auto stage_own = [&]() {
#pragma unroll
        for (int u = 0; u < CPT; ++u)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                Xs[at0 + u * SU + c] = phase(neg(c, cvt<double>(q[u][c]) * qs[u][c]), img[u] ? mycode[u] : 0u);
    };
    auto stage_halo = [&](int s, c64 hqs) {
        const int c = ix.slot_comp(hpos[s]);
        Xs[ix.slot_place(hpos[s])] = phase(neg(c, cvt<double>(hq[s]) * hqs), hpos[s]);
    };
    auto halo_qs = [&](int s) { return vcent(A.qs, hoff[s]); };
    auto mu_at = [&](int x, int y, int w, int c) -> c64 { return A.muinv[3 * ix.mu_cell(x, y, w) + c]; };   // 1/μ at a cell of g
    if (ML)
        for (int e = tid; e < 3 * MX * MY * MZ; e += NT) {
            const int cell = e / 3, mi = cell % MX, mj = (cell / MX) % MY, mk_ = cell / (MX * MY);
            Ms[e] = mu_at(i0 + mi - 1, j0 + mj - 1, C::SLAB ? 0 : k0 + mk_ - 1, e - 3 * cell);
        }
    __syncthreads();
    stage_own();
#pragma unroll
    for (int s = 0; s < NHS; ++s)
        if (hpos[s] >> 31) stage_halo(s, halo_qs(s));
    c64 rho = mk<double>(S.rho_re, S.rho_im);

    const c64 zp = !C::SLAB ? mk<double>(1, 0) : (g.bloch[2] ? g.ph[2] : mk<double>(0, 0));
    const c64 zm = !C::SLAB ? mk<double>(1, 0) : (g.bloch[2] ? g.phinv[2] : mk<double>(0, 0));
    // the end of a step, done while the next one's first sum is under way: one
    // thread of a wave with little else to do advances the scalars ...
    auto finish = [&](int done) {
        if (tid == NT - 64) {
            sqmr_advance(S, s_tot);
            s_c2t2 = S.c2t2;
            s_c2a = mk<double>(S.c2a_re, S.c2a_im);
            s_stop = S.conv || (done % A.chunk == 0 && S.tau <= A.near * S.cn);
        }
    };
    // ... and d = c²θ² d + c²α q, z += d follow with the step's q
    auto dz_update = [&]() {
        const c64 c2a = s_c2a;
        const double c2t2 = s_c2t2;
#pragma unroll
        for (int u = 0; u < CPT; ++u)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                cx<R> &dv = DZL ? Dz[(6 * u + c) * NT + tid] : d[DZL ? 0 : u][c];
                cx<R> &zv = DZL ? Dz[(6 * u + 3 + c) * NT + tid] : z[DZL ? 0 : u][c];
                const c64 de = c2t2 * cvt<double>(dv) + c2a * cvt<double>(qp[u][c]);
                dv = cvt<R>(de);
                zv = cvt<R>(cvt<double>(zv) + de);
            }
    };
    bool pend = false;   // a step whose end is still to be done
#pragma clang loop unroll(disable)
    for (int it = 0; it < A.steps; ++it) {
        __syncthreads();
        // (opaque, so that addresses are not kept in registers across the loop)
#pragma unroll
        for (int u = 0; u < CPT; ++u) asm volatile("" : "+v"(p[u]));
#pragma unroll
        for (int s = 0; s < NHS; ++s) asm volatile("" : "+v"(hoff[s]), "+v"(hx[s]), "+v"(hpos[s]));
        c64 t[CPT][3];
        double sg[2] = {0, 0};
        {
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                // ---- t = P q of the own cell.  P's diagonal is 1 exactly, so
                // the second differences are formed without their own diagonal
                const int jj = jq + u * UJ, kk = kq + u * UK;
                const int at = at0 + u * SU, tX = ii, tY = TX + jj, tZ = TX + TY + kk;
                // staged value of component c at (+di, +dj, +dk)
                auto ld = [&](int c, int di, int dj, int dk) -> c64 {
                    const c64 v = Xs[at + c + di * SX + dj * SY + dk * SZ];
                    if (C::SLAB && dk > 0) return zp * v;
                    if (C::SLAB && dk < 0) return zm * v;
                    return v;
                };
                c64 o[3];
                // 1/∆l_D and 1/∆l_P, and their products for the second
                // differences
                auto D = [&](int t) { return tb[D_][t]; };
                auto P = [&](int t) { return tb[P_][t]; };
                if (!MU) {
                    o[0] = D(tX) * (P(tY) * (ld(1, 1, 0, 0) - ld(1, 0, 0, 0) - ld(1, 1, -1, 0) + ld(1, 0, -1, 0)) +
                                    P(tZ) * (ld(2, 1, 0, 0) - ld(2, 0, 0, 0) - ld(2, 1, 0, -1) + ld(2, 0, 0, -1)));
                    o[0] = o[0] - tb[EP][tY] * ld(0, 0, 1, 0) - tb[EM][tY] * ld(0, 0, -1, 0);
                    o[0] = o[0] - tb[EP][tZ] * ld(0, 0, 0, 1) - tb[EM][tZ] * ld(0, 0, 0, -1);
                    o[1] = D(tY) * (P(tZ) * (ld(2, 0, 1, 0) - ld(2, 0, 0, 0) - ld(2, 0, 1, -1) + ld(2, 0, 0, -1)) +
                                    P(tX) * (ld(0, 0, 1, 0) - ld(0, 0, 0, 0) - ld(0, -1, 1, 0) + ld(0, -1, 0, 0)));
                    o[1] = o[1] - tb[EP][tZ] * ld(1, 0, 0, 1) - tb[EM][tZ] * ld(1, 0, 0, -1);
                    o[1] = o[1] - tb[EP][tX] * ld(1, 1, 0, 0) - tb[EM][tX] * ld(1, -1, 0, 0);
                    o[2] = D(tZ) * (P(tX) * (ld(0, 0, 0, 1) - ld(0, 0, 0, 0) - ld(0, -1, 0, 1) + ld(0, -1, 0, 0)) +
                                    P(tY) * (ld(1, 0, 0, 1) - ld(1, 0, 0, 0) - ld(1, 0, -1, 1) + ld(1, 0, -1, 0)));
                    o[2] = o[2] - tb[EP][tX] * ld(2, 1, 0, 0) - tb[EM][tX] * ld(2, -1, 0, 0);
                    o[2] = o[2] - tb[EP][tY] * ld(2, 0, 1, 0) - tb[EM][tY] * ld(2, 0, -1, 0);
                } else {
                    // H = μ⁻¹ Cₑ X at the cell and one behind it along each axis
                    // (behind a non-Bloch end it is zero: the ghost values and
                    // the weight of the own value are)
                    auto DMt = [&](int t) { return tb[MU ? DM : 0][t]; };
                    auto mu = [&](int c, int a) -> c64 {   // 1/μ_c at the cell (a < 0) or one behind along a
                        const int x = tX - (a == 0), y = tY - TX - (a == 1), w = tZ - TX - TY - (a == 2);
                        if (!ML) return mu_at(i0 + x, j0 + y, k0 + w, c);
                        return Ms[ix.mu_staged(x, y, w) + c];
                    };
                    const c64 hx = mu(0, -1) * (D(tY) * (ld(2, 0, 1, 0) - ld(2, 0, 0, 0)) - D(tZ) * (ld(1, 0, 0, 1) - ld(1, 0, 0, 0)));
                    const c64 hxy = mu(0, 1) * (DMt(tY) * (ld(2, 0, 0, 0) - ld(2, 0, -1, 0)) - D(tZ) * (ld(1, 0, -1, 1) - ld(1, 0, -1, 0)));
                    const c64 hxz = mu(0, 2) * (D(tY) * (ld(2, 0, 1, -1) - ld(2, 0, 0, -1)) - DMt(tZ) * (ld(1, 0, 0, 0) - ld(1, 0, 0, -1)));
                    o[1] = P(tZ) * (hx - hxz);
                    o[2] = -(P(tY) * (hx - hxy));
                    const c64 hy = mu(1, -1) * (D(tZ) * (ld(0, 0, 0, 1) - ld(0, 0, 0, 0)) - D(tX) * (ld(2, 1, 0, 0) - ld(2, 0, 0, 0)));
                    const c64 hyx = mu(1, 0) * (D(tZ) * (ld(0, -1, 0, 1) - ld(0, -1, 0, 0)) - DMt(tX) * (ld(2, 0, 0, 0) - ld(2, -1, 0, 0)));
                    const c64 hyz = mu(1, 2) * (DMt(tZ) * (ld(0, 0, 0, 0) - ld(0, 0, 0, -1)) - D(tX) * (ld(2, 1, 0, -1) - ld(2, 0, 0, -1)));
                    o[0] = -(P(tZ) * (hy - hyz));
                    o[2] = o[2] + P(tX) * (hy - hyx);
                    const c64 hz = mu(2, -1) * (D(tX) * (ld(1, 1, 0, 0) - ld(1, 0, 0, 0)) - D(tY) * (ld(0, 0, 1, 0) - ld(0, 0, 0, 0)));
                    const c64 hzx = mu(2, 0) * (DMt(tX) * (ld(1, 0, 0, 0) - ld(1, -1, 0, 0)) - D(tY) * (ld(0, -1, 1, 0) - ld(0, -1, 0, 0)));
                    const c64 hzy = mu(2, 1) * (D(tX) * (ld(1, 1, -1, 0) - ld(1, 0, -1, 0)) - DMt(tY) * (ld(0, 0, 0, 0) - ld(0, 0, -1, 0)));
                    o[0] = o[0] + P(tY) * (hz - hzy);
                    o[1] = o[1] - P(tX) * (hz - hzx);
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        if (own[u]) o[c] = o[c] - A.om2 * (A.epsd[3 * p[u] + c] * ld(c, 0, 0, 0));
                }
                if (OFFD && own[u]) {
                    // −ω² Σ_w ½ Σ_corners ε_uw · (∆l-weighted mean of X_w along w)
                    const c64 *eo = A.epso;
                    const int i = i0 + tX, j = j0 + tY - TX, k = k0 + tZ - TX - TY, pc = p[u];
                    const int cpx = ix.next_x(pc, i), cpy = ix.next_y(pc, j), cpz = ix.next_z(pc, k);
                    const c64 hom = 0.5 * A.om2;
                    const c64 e0 = eo[3 * pc], e1 = eo[3 * pc + 1], e2 = eo[3 * pc + 2];
                    const c64 ax = tb[W0][tX] * ld(0, 0, 0, 0) + tb[W1][tX] * ld(0, -1, 0, 0);
                    const c64 ay = tb[W0][tY] * ld(1, 0, 0, 0) + tb[W1][tY] * ld(1, 0, -1, 0);
                    const c64 az = tb[W0][tZ] * ld(2, 0, 0, 0) + tb[W1][tZ] * ld(2, 0, 0, -1);
                    if (inw(0)) {
                        c64 sv = e0 * ay + e1 * az;
                        if (cpx >= 0)
                            sv = sv + eo[3 * cpx] * (tb[W0][tY] * ld(1, 1, 0, 0) + tb[W1][tY] * ld(1, 1, -1, 0)) +
                                 eo[3 * cpx + 1] * (tb[W0][tZ] * ld(2, 1, 0, 0) + tb[W1][tZ] * ld(2, 1, 0, -1));
                        o[0] = o[0] - hom * sv;
                    }
                    if (inw(1)) {
                        c64 sv = e0 * ax + e2 * az;
                        if (cpy >= 0)
                            sv = sv + eo[3 * cpy] * (tb[W0][tX] * ld(0, 0, 1, 0) + tb[W1][tX] * ld(0, -1, 1, 0)) +
                                 eo[3 * cpy + 2] * (tb[W0][tZ] * ld(2, 0, 1, 0) + tb[W1][tZ] * ld(2, 0, 1, -1));
                        o[1] = o[1] - hom * sv;
                    }
                    if (inw(2)) {
                        c64 sv = e1 * ax + e2 * ay;
                        if (cpz >= 0)
                            sv = sv + eo[3 * cpz + 1] * (tb[W0][tX] * ld(0, 0, 0, 1) + tb[W1][tX] * ld(0, -1, 0, 1)) +
                                 eo[3 * cpz + 2] * (tb[W0][tY] * ld(1, 0, 0, 1) + tb[W1][tY] * ld(1, 0, -1, 1));
                        o[2] = o[2] - hom * sv;
                    }
                }
                // the output scaling q T = qs T² (T² the product of the stretched ∆l)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const c64 T2 = tb[c == 0 ? SD : SP][tX] * tb[c == 1 ? SD : SP][tY] * tb[c == 2 ? SD : SP][tZ];
                    c64 tv = neg(c, (qs[u][c] * T2) * o[c]);
                    const c64 qc = cvt<double>(q[u][c]);
                    if (!MU) tv = tv + qc;
                    tv = cvt<double>(cvt<R>(tv));   // as stored by the step-by-step form
                    if (own[u]) {   // (zero outside the window)
                        sg[0] += qc.re * tv.re - qc.im * tv.im;
                        sg[1] += qc.re * tv.im + qc.im * tv.re;
                    }
                    t[u][c] = tv;
                }
            }
            arrive<2, NT>(slA, box, 2u * it + 1u, sg, sh);
        }
        if (pend) finish(it);
        collect<2, NT>(slA, A.nb, 2u * it + 1u, sg, sh2, &fail);
        if (fail) break;
        if (pend) {
            dz_update();
            pend = false;
            if (s_stop) break;
        }
        if (sg[0] == 0.0 && sg[1] == 0.0) {   // breakdown: no step
            if (tid == 0) {
                S.breakdown = 1;
                S.conv = 1;
                S.alpha_re = S.alpha_im = S.apend_re = S.apend_im = 0;
                S.c2t2 = S.c2a_re = S.c2a_im = 0;
            }
            __syncthreads();
            break;
        }
        const c64 al = cdiv(rho, mk<double>(sg[0], sg[1]));
        double acc[3] = {0, 0, 0};
#pragma unroll
        for (int u = 0; u < CPT; ++u)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                if (own[u]) {
                    const c64 v = cvt<double>(r[u][c]) - al * t[u][c];
                    r[u][c] = cvt<R>(v);
                    acc[0] += v.re * v.re + v.im * v.im;
                    acc[1] += v.re * v.re - v.im * v.im;
                    acc[2] += 2.0 * v.re * v.im;
                }
        // the box's new r to the exchange, in runs of consecutive words (through
        // the staging buffer, free between the curl-curl and the next staging):
        // written cell by cell each store would touch six times the lines
        {
            cx<R> *xr = (cx<R> *)Xs;
#pragma unroll
            for (int u = 0; u < CPT; ++u)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    xr[3 * ix.in_box(ii, jq + u * UJ, kq + u * UK) + c] = r[u][c];
            __syncthreads();
            constexpr int W = VB / 8;
            const unsigned long long *xw = (const unsigned long long *)Xs;
            unsigned long long *gw = (unsigned long long *)(xch + (size_t)box * (3 * CPT * NT));
#pragma unroll
            for (int s = 0; s < 3 * CPT * W; ++s)
                __hip_atomic_store(gw + s * NT + tid, xw[s * NT + tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        arrive<3, NT>(slB, box, 2u * it + 2u, acc, sh);
        c64 hqs[NHS];
#pragma unroll
        for (int s = 0; s < NHS; ++s)
            if (hpos[s] >> 31) hqs[s] = halo_qs(s);
        collect<3, NT>(slB, A.nb, 2u * it + 2u, acc, sh2, &fail);
        if (fail) break;
        asm volatile("" ::: "memory");
        cx<R> hr[NHS];
#pragma unroll
        for (int s = 0; s < NHS; ++s)
            if (hpos[s] >> 31) hr[s] = sub(vent(xch, hx[s]));
#pragma unroll
        for (int u = 0; u < CPT; ++u)
            if (img[u])
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (inw(c)) r[u][c] = sub(vent(xch, xidx(i0 + ii, j0 + jq + u * UJ, k0 + kq + u * UK, c)));
        const c64 rho1 = mk<double>(acc[1], acc[2]);
        const c64 be = iszero(rho) ? mk<double>(0, 0) : cdiv(rho1, rho);
        if (tid == NT - 64) {   // for the finish of this step
            s_tot[0] = acc[0];
            s_tot[1] = acc[1];
            s_tot[2] = acc[2];
            S.sig_re = sg[0];
            S.sig_im = sg[1];
            S.alpha_re = S.apend_re = al.re;
            S.alpha_im = S.apend_im = al.im;
        }
        rho = rho1;
        pend = true;
#pragma unroll
        for (int u = 0; u < CPT; ++u)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                qp[u][c] = q[u][c];
                q[u][c] = cvt<R>(cvt<double>(r[u][c]) + be * cvt<double>(qp[u][c]));
            }
        stage_own();
#pragma unroll
        for (int s = 0; s < NHS; ++s)
            if (hpos[s] >> 31) {
                hq[s] = cvt<R>(cvt<double>(hr[s]) + be * cvt<double>(hq[s]));
                stage_halo(s, hqs[s]);
            } else if (hpos[s] >> 30) Xs[ix.slot_place(hpos[s])] = mk<double>(0, 0);   // (r went through here)
    }
    __syncthreads();
    if (pend) {   // the last step's end
        finish(A.steps);
        __syncthreads();
        dz_update();
    }
    if (fail) {   // uniform over the block; the solve then ends with an error, whatever the others store
        if (tid == 0) atomicMin(&A.scal[rhs].stag, RESIDENT_TIMEOUT);
        return;
    }
#pragma unroll
    for (int u = 0; u < CPT; ++u)
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (own[u] && inw(c)) {
                *vent(rg, vidx(p[u], c)) = r[u][c];
                *vent(qg, vidx(p[u], c)) = q[u][c];
                *vent(dg, vidx(p[u], c)) = DZL ? Dz[(6 * u + c) * NT + tid] : d[DZL ? 0 : u][c];
                *vent(zg, vidx(p[u], c)) = DZL ? Dz[(6 * u + 3 + c) * NT + tid] : z[DZL ? 0 : u][c];
            }
    if (lead) scal_store(A.scal[rhs], S);
}

__global__ void k_res_clear(unsigned long long *slots, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) slots[i] = 0;
}

constexpr int RES_DEVICES = 64;   // whose capacity is kept

// blocks that can be resident on the current device at once (0: none, or the
// query failed, which is not kept)
static int res_capacity(std::atomic<int> *known, int dev, const void *kernel, int threads) {
    if (dev >= 0 && dev < RES_DEVICES)
        if (const int c = known[dev].load(std::memory_order_relaxed)) return c;
    int per = 0, cus = 0, coop = 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev) != hipSuccess || !coop ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, 0) != hipSuccess) {
        hipGetLastError();
        return 0;
    }
    if (dev >= 0 && dev < RES_DEVICES) known[dev].store(per * cus, std::memory_order_relaxed);
    return per * cus;
}

struct ResPlan {
    const void *kernel = nullptr;
    int nbx = 0, nby = 0, nb = 0, cap = 0;
    int threads = 0, cells = 0;   // per box
    int box[3] = {0, 0, 0};
};

// the kernel and boxes for an operator: the smallest boxes that have a place on
// the chip each
template <typename R, bool OFFD, bool MU>
static ResPlan res_plan2(const DGrid<double> &g, int dev) {
    ResPlan P;
    auto shape = [&](int tx, int ty, int tz) {
        P.nbx = (g.N[0] + tx - 1) / tx;
        P.nby = (g.N[1] + ty - 1) / ty;
        P.nb = P.nbx * P.nby * ((g.N[2] + tz - 1) / tz);
        P.cells = tx * ty * tz;
        P.box[0] = tx;
        P.box[1] = ty;
        P.box[2] = tz;
    };
#define MFD_RES(X, Y, Z, CPT)                                                  \
    do {                                                                       \
        P.kernel = (const void *)k_resident<R, OFFD, MU, X, Y, Z, CPT>;        \
        P.threads = X * Y * Z / CPT;                                           \
        static std::atomic<int> known[RES_DEVICES];                            \
        P.cap = std::min(res_capacity(known, dev, P.kernel, P.threads), RES_BOXES); \
        shape(X, Y, Z);                                                        \
        if (P.nb <= P.cap) return P;                                           \
    } while (0)
    // (four cells per thread of FP64 vectors, of 1/μ or of corner ε would need
    // scratch memory: see above)
    constexpr bool FOUR = sizeof(R) == 4 && !MU && !OFFD;
    if (g.N[2] == 1) {
        MFD_RES(16, 8, 1, 1);
        MFD_RES(32, 16, 1, 2);
        if constexpr (FOUR) MFD_RES(32, 32, 1, 4);
    } else {
        MFD_RES(8, 4, 4, 1);
        MFD_RES(8, 8, 4, 1);
        MFD_RES(16, 8, 4, 2);
        if constexpr (FOUR) MFD_RES(16, 8, 8, 4);
    }
#undef MFD_RES
    return P;
}

template <typename R>
static ResPlan res_plan(const mfd_op *op) {
    const DGrid<double> &g = op->G.d64;
    const int dev = op->ctx->device;
    if (op->full) return res_plan2<R, true, false>(g, dev);
    if (op->has_mu) return res_plan2<R, false, true>(g, dev);
    return res_plan2<R, false, false>(g, dev);
}

template <typename R>
static int res_xch(const ResPlan &P, int64_t n) {
    return res_room(P.nb, P.cells, sizeof(cx<R>), sizeof(double) * NPART * 4, n);
}
static_assert(RES_BOXES * RES_SLOT_WORDS * sizeof(unsigned long long) <= sizeof(double) * NPART * 4, "a right-hand side's slots");

// A refused launch costs 38 ms (the runtime tries to make the cooperative queue),
// so a context asks again after 10 s only
constexpr int64_t RES_RETRY_NS = 10000000000ll;
static int64_t now_ns() { return std::chrono::steady_clock::now().time_since_epoch() / std::chrono::nanoseconds(1); }

template <typename R>
bool resident_ok(const mfd_op *op, int64_t nrhs, int chunk) {
    if (now_ns() < op->ctx->res_retry.load(std::memory_order_relaxed)) return false;
    if (op->tile_set[0] == 1 || op->tile_set[1] == 1 || op->csr || op->gd || !(op->ee_all || op->rev) || (op->has_mu && op->full)) return false;
    if (op->G.d64.M > RES_MAX_CELLS) return false;
    const ResPlan P = res_plan<R>(op);
    if (P.nb > P.cap || res_xch<R>(P, op->n) == 0) return false;
    const DGrid<double> &g = op->G.d64;
    const ResForm f = {sizeof(R) == 8, op->has_mu != 0, op->full != 0, g.N[2] == 1, g.nc};
    return res_pays(f, P.nb, P.cells, P.cap, g.M, nrhs, nrhs == 1 ? std::max(chunk, 512) : chunk);
}

template <typename R>
void resident_trace(const mfd_op *op) {
    const ResPlan P = res_plan<R>(op);
    fprintf(stderr, "[mfd resident] %s boxes %dx%dx%d, %d threads, %d boxes\n", sizeof(R) == 8 ? "fp64" : "fp32", P.box[0],
            P.box[1], P.box[2], P.threads, P.nb);
}

template <typename R>
int resident_steps(mfd_op *op, int64_t nrhs, int steps, int chunk, double near) {
    Workspace &w = op->ws;
    hipStream_t s = op->stream;
    const ResPlan P = res_plan<R>(op);
    ResArgs<R> A;
    A.g = op->rev ? op->G.r64 : op->G.d64;
    A.qs = op->d64.qs;
    A.epsd = op->d64.epsd;
    A.epso = op->d64.epso;
    A.muinv = op->d64.muinv;
    A.om2 = op->d64.om2;
    A.r = (cx<R> *)w.r;
    A.q = (cx<R> *)w.q;
    A.d = (cx<R> *)w.d;
    A.z = (cx<R> *)w.z;
    A.vs = op->n;
    A.nbx = P.nbx;
    A.nby = P.nby;
    A.nb = P.nb;
    A.steps = steps;
    A.chunk = chunk;
    A.near = near;
    A.slots = (unsigned long long *)w.part;
    A.scal = w.scal;
    A.xch = res_xch<R>(P, op->n) == 1 ? (cx<R> *)(w.part + (size_t)nrhs * NPART * 4) : (cx<R> *)w.r64;
    const int64_t group = std::max(1, P.cap / A.nb);   // right-hand sides per launch
    for (int64_t r0 = 0; r0 < nrhs; r0 += group) {
        const int nr = (int)std::min<int64_t>(group, nrhs - r0);
        A.rhs0 = (int)r0;
        const int words = nr * RES_SLOT_WORDS * A.nb;
        k_res_clear<<<(words + 255) / 256, 256, 0, s>>>(A.slots, words);
        void *args[] = {&A};
        const hipError_t e = hipLaunchCooperativeKernel(P.kernel, dim3((unsigned)(nr * A.nb)), dim3((unsigned)P.threads), args, 0, s);
        // whatever the reason: too few places, or another process has the device's
        // one cooperative queue (hipErrorIllegalState).  An error of earlier work
        // comes up again in the step-by-step launches.
        if (e != hipSuccess) {
            hipGetLastError();
            op->ctx->res_retry.store(now_ns() + RES_RETRY_NS, std::memory_order_relaxed);
            return RESIDENT_REFUSED;
        }
    }
    return MFD_OK;
}

template bool resident_ok<double>(const mfd_op *, int64_t, int);
template bool resident_ok<float>(const mfd_op *, int64_t, int);
template void resident_trace<double>(const mfd_op *);
template void resident_trace<float>(const mfd_op *);
template int resident_steps<double>(mfd_op *, int64_t, int, int, double);
template int resident_steps<float>(mfd_op *, int64_t, int, int, double);

}  // namespace mfd
