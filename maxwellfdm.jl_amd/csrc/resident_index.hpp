// Which cells, halo values and memory places a thread of the resident solver
// works on, as plain integer code that host_checks.cpp runs on the CPU for
// every box shape: each access against the array it goes to, each staged place
// written once, each exchanged value read where its owner writes it.
#pragma once
#include <cstddef>
#include <cstdint>

#ifndef MFD_HD
#ifdef __HIPCC__
#define MFD_HD __host__ __device__
#else
#define MFD_HD
#endif
#endif

namespace mfd {

template <int TX_, int TY_, int TZ_, int CPT_>
struct BoxCfg {
    static constexpr int TX = TX_, TY = TY_, TZ = TZ_, CPT = CPT_;   // cells of the box, cells per thread
    static constexpr bool SLAB = TZ == 1;            // one-cell z axis: no z halo is staged
    static constexpr int CELLS = TX * TY * TZ, NT = CELLS / CPT;     // NT: threads
    static constexpr int XH = TX + 2, YH = TY + 2, ZH = SLAB ? 1 : TZ + 2;
    static constexpr int XS = XH * YH * ZH * 3;      // staged values
    static constexpr int HZ = SLAB ? 0 : 2 * XH * YH, HY = 2 * TZ * XH, HX = 2 * TZ * TY;
    static constexpr int NHALO = 3 * (HZ + HY + HX); // staged values outside the box
    static constexpr int NHS = (NHALO + NT - 1) / NT;
    static constexpr int NTAB = TX + TY + TZ;
    static constexpr int MX = TX + 1, MY = TY + 1, MZ = SLAB ? 1 : TZ + 1;   // (μ) the box and one cell behind it
    // strides of the staged values; from one of a thread's cells to its next
    static constexpr int SX = 3, SY = 3 * XH, SZ = SLAB ? 0 : 3 * XH * YH, SU = SLAB ? SY : SZ;
    static constexpr int UJ = SLAB ? 1 : 0, UK = SLAB ? 0 : 1;
};

// the boxes of a grid (N cells an axis, nbx, nby boxes along x, y; the
// reflection along the axes of rmask of the caller's cells) and its vectors
template <class C>
struct BoxIndex {
    int N0, N1, N2, bl0, bl1, bl2, rmask, nbx, nby;
    int cmpfirst, c0, nc, M;   // order and component window of the vectors

    MFD_HD inline bool inw(int c) const { return (unsigned)(c - c0) < (unsigned)nc; }

    // the caller's cell of (i, j, k) with its wraps (base 3: none, low, high end
    // of x, y, z), or −1 for a non-Bloch ghost and beyond
    MFD_HD inline int locate(int i, int j, int k, unsigned &code) const {
        code = 0;
        bool ok = true;
        auto wrap = [&](int &v, int N, int bloch, unsigned w) {
            if (v < 0) { ok = ok && bloch; v += N; code += w; }
            else if (v >= N) { ok = ok && bloch && v == N; v = 0; code += 2 * w; }
        };
        wrap(i, N0, bl0, 1u);
        wrap(j, N1, bl1, 3u);
        wrap(k, N2, bl2, 9u);
        if (rmask & 1) i = N0 - 1 - i;
        if (rmask & 2) j = N1 - 1 - j;
        if (rmask & 4) k = N2 - 1 - k;
        return ok ? i + N0 * (j + N1 * k) : -1;
    }
    // place of component c of the (wrapped) cell i, j, k among the boxes' r
    MFD_HD inline unsigned xidx(int i, int j, int k, int c) const {
        i = i < 0 ? i + N0 : (i >= N0 ? i - N0 : i);
        j = j < 0 ? j + N1 : (j >= N1 ? j - N1 : j);
        k = k < 0 ? k + N2 : (k >= N2 ? k - N2 : k);
        const int bi = i / C::TX, bj = j / C::TY, bk = k / C::TZ;
        return (unsigned)((bi + nbx * (bj + nby * bk)) * (3 * C::CELLS) +
                          3 * in_box(i - bi * C::TX, j - bj * C::TY, k - bk * C::TZ) + c);
    }
    // number of a cell within its box
    MFD_HD static inline int in_box(int i, int j, int k) { return i + C::TX * (j + C::TY * k); }
    // component c of the caller's cell p in the vectors
    MFD_HD inline int vidx(int p, int c) const { return cmpfirst ? 3 * p + c : p + M * (c - c0); }
    // a thread's first cell in its box: the others follow along z (along y on a
    // one-cell z axis)
    MFD_HD static inline void first_cell(int tid, int &i, int &j, int &k) {
        i = tid % C::TX;
        j = C::SLAB ? C::CPT * (tid / C::TX) : (tid / C::TX) % C::TY;
        k = C::SLAB ? 0 : C::CPT * (tid / (C::TX * C::TY));
    }
    // place of component 0 of a cell of the box or its halo among the staged values
    MFD_HD static inline int staged(int i, int j, int k) {
        return ((C::SLAB ? 0 : (k + 1) * C::YH * C::XH) + (j + 1) * C::XH + i + 1) * 3;
    }
    // halo value h (0 ≤ h < NHALO) of a box: its cell and component
    MFD_HD static inline void halo(int h, int &i, int &j, int &k, int &c) {
        if (h < 3 * C::HZ) {
            const int pz = h / (3 * C::XH * C::YH), f = h - pz * (3 * C::XH * C::YH), row = f / (3 * C::XH);
            k = pz ? C::TZ : -1;
            j = row - 1;
            i = f - row * (3 * C::XH);
            c = i % 3;
            i = i / 3 - 1;
        } else if (h < 3 * (C::HZ + C::HY)) {
            h -= 3 * C::HZ;
            const int row = h / (3 * C::XH);
            k = row >> 1;
            j = (row & 1) ? C::TY : -1;
            i = h - row * (3 * C::XH);
            c = i % 3;
            i = i / 3 - 1;
        } else {
            h -= 3 * (C::HZ + C::HY);
            const int cell = h / 3;
            c = h - 3 * cell;
            i = (cell & 1) ? C::TX : -1;
            k = (cell >> 1) / C::TY;
            j = (cell >> 1) - k * C::TY;
        }
    }
    // a halo slot's staged place, component and wraps in one word (bit 30: in use;
    // bit 31, set by the caller: there is a value)
    MFD_HD static inline unsigned pack(int lp, int c, unsigned code) { return 1u << 30 | (unsigned)lp << 8 | (unsigned)c << 6 | code; }
    MFD_HD static inline int slot_place(unsigned w) { return (int)((w >> 8) & 0xffffu); }
    MFD_HD static inline int slot_comp(unsigned w) { return (int)(w >> 6) & 3; }
    MFD_HD static inline unsigned slot_code(unsigned w) { return w & 63u; }

    // the caller's cell whose 1/μ the cell (x, y, w) takes (clamped, so that
    // reads past the box's end stay inside)
    MFD_HD inline int mu_cell(int x, int y, int w) const {
        x = x < N0 - 1 ? x : N0 - 1;
        y = y < N1 - 1 ? y : N1 - 1;
        w = w < N2 - 1 ? w : N2 - 1;
        if (x < 0) x += N0;
        if (y < 0) y += N1;
        if (w < 0) w += N2;
        if (rmask & 1) x = N0 - 1 - x;
        if (rmask & 2) y = N1 - 1 - y;
        if (rmask & 4) w = N2 - 1 - w;
        return x + N0 * (y + N1 * w);
    }
    // place of component 0 of cell (x, y, w) of the box or one behind it in the staged 1/μ
    MFD_HD static inline int mu_staged(int x, int y, int w) {
        return 3 * (x + 1 + C::MX * (y + 1 + C::MY * (C::SLAB ? 0 : w + 1)));
    }
    // the cell one on along x, y, z from cell p = (i, j, k) (wrapped), or −1
    MFD_HD inline int next_x(int p, int i) const { return i + 1 < N0 ? p + 1 : (bl0 ? p - (N0 - 1) : -1); }
    MFD_HD inline int next_y(int p, int j) const { return j + 1 < N1 ? p + N0 : (bl1 ? p - (N1 - 1) * N0 : -1); }
    MFD_HD inline int next_z(int p, int k) const { return k + 1 < N2 ? p + N0 * N1 : (bl2 ? p - (N2 - 1) * N0 * N1 : -1); }
};

// Whether d and z of a box lie in LDS (vb bytes a value): while they fit beside
// the staged box, which takes most of the 160 KB
template <class C>
MFD_HD constexpr bool box_dz_lds(size_t vb) { return C::CELLS * vb <= 8192; }

constexpr int RES_BOXES = 256;      // boxes of a launch at most
constexpr int RES_SLOT_WORDS = 16;  // 8-byte words of a box's partial sums: two arrivals of 8

// Where the boxes exchange r (values per right-hand side: 3 per cell of every
// box): 1, the second and third slots of the partial sums (part_bytes each),
// which the steps of the resident kernel leave free; 2, the residual and probe
// vectors r64, et, et2 (16 bytes a value, n values), free inside a cycle and
// consecutive; 0: neither has the room.
MFD_HD inline int res_room(int boxes, int cells, size_t vb, size_t part_bytes, int64_t n) {
    const size_t need = vb * 3 * (size_t)boxes * (size_t)cells;
    if (need <= 2 * part_bytes) return 1;
    return need <= 3 * 16 * (size_t)n ? 2 : 0;
}

// Whether nrhs right-hand sides run resident rather than step by step.  Boxes of
// several right-hand sides that do not share the chip run as one launch after
// the other, so the resident time of a step grows with the launches; step by
// step the launches serve all right-hand sides and only the traffic grows.
// Both sides as measured (µs per step, resident / step by step): 24³ 2 RHS 9.4 /
// 21.6, 8 36.1 / 31.5, 16 70 / 39; 31×31×32 2 20.4 / 25.1, 4 39.6 / 30.6, 16 157 /
// 60; 48³ 4 55 / 58, 8 110 / 97; FP32 64³ 2 41 / 48, 4 82 / 71 (1,024 cells a box
// at 20 µs, 17 since), 40³ with 2 RHS and launches of one step (check_every = 1)
// 104 / 62; 180×170 (Ex, Ey) 2 9.9 / 19, 16 57 / 49.  The constants
// below are fits to 76 systems on 15 grids, 1 to 16 right-hand sides: the choice is the
// faster one but near the crossing (1.26 times the faster at worst).
// steps: of a launch (a launch takes about 26 µs beside its steps, and several
// right-hand sides are looked at after every chunk, one only every 512 steps).
struct ResForm {
    bool fp64, mu, full;   // vectors; 1/μ, corner ε
    bool plane;            // one-cell z axis
    int nc;                // components of the window
};
inline bool res_pays(const ResForm &f, int boxes, int box_cells, int cap, int64_t cells, int64_t nrhs, int steps) {
    const bool tensor = f.mu || f.full;
    const double launch = (f.plane ? (box_cells <= 128 ? 6.8 : (box_cells <= 512 ? 9.4 : 13.0))
                                   : (box_cells <= 128 ? 8.4 : (box_cells <= 256 ? 9.8 : (box_cells <= 512 ? 12.4 : 16.2)))) *
                              (tensor ? 1.1 : 1.0) + 26.0 / steps;
    const int64_t per = cap / boxes < 1 ? 1 : cap / boxes, launches = (nrhs + per - 1) / per;
    // ns per unknown and step of the four kernels: the marching stencil serves a
    // plane of three components less well, a window's has a kernel of its own
    const double ns = (f.fp64 ? (tensor ? 0.037 : 0.032) : (tensor ? 0.027 : 0.020)) * (f.plane && f.nc == 3 ? 1.35 : 1.0);
    const double fixed = f.plane ? 15.5 : (f.full ? 26.0 : 20.0);
    return (double)launches * launch <= fixed + 1e-3 * ns * (double)(f.nc * cells * nrhs);
}

// 32-bit byte offsets into the vectors (16 bytes a value) hold up to here
constexpr int64_t RES_MAX_CELLS = 1 << 22;

}  // namespace mfd
