// Shape of a stencil launch's tiles, as plain integer code (host_checks.cpp runs
// it on the CPU, against measured shapes).
#pragma once
#include <cstdint>

namespace mfd {

constexpr int GRID_YZ = 65535;   // blocks along y and z of a launch

// Makes tiles of ty rows and kz planes larger (rows up to ty_max) until a launch
// over nrhs right-hand sides keeps to the grid's limits and, where it reduces,
// to part_max partial sums per right-hand side.  False: no such tile is large
// enough (a plane of more than 512·part_max cells, or of too many rows).
inline bool tile_fit(const int *N, int64_t nrhs, bool narrow, int ty_max, bool reduces, int part_max, int &ty, int &kz) {
    while (true) {
        const int rows = narrow ? 2 * ty : ty;
        const int64_t nx = (N[0] + (narrow ? 31 : 63)) / (narrow ? 32 : 64), ny = (N[1] + rows - 1) / rows;
        const int64_t nch = (N[2] + kz - 1) / kz;
        const bool many = reduces && nx * ny * nch > part_max;
        if (ny <= GRID_YZ && nch * nrhs <= GRID_YZ && !many) return true;
        if (nch > 1 && (many || nch * nrhs > GRID_YZ)) kz = kz < N[2] / 2 ? 2 * kz : N[2];
        else if (ty < ty_max) ty *= 2;
        else return false;
    }
}

// the kernel a launch runs
struct TileKernel {
    bool fp64;              // vectors
    bool apply;             // A itself rather than the solver's P
    bool mu, full, gd;      // 1/μ, corner ε, grad-div (P only)
    bool rev;               // a reflected grid (boundft HH on some axis)
    bool win;               // a component window
    bool narrow;            // 32-wide tiles of twice the rows
    bool cocg;              // COCG's fused P (64-wide only)
};

// A launch takes as many rounds of blocks as the fullest CU has, so its time is
// that CU's.  How many 4-row blocks (256 threads) share a CU follows from the
// kernel's registers: three where it keeps to 168 (A on FP32 vectors with
// diagonal ε, μ = 1), two up to 256, one beyond (P with μ ≠ 1; the grad-div
// form by its LDS); 8-row blocks are alone.  A block costs its planes and two
// more (the first plane's halo and the prologue).  In units of two 4-row blocks
// side by side, one alone takes 0.8 of the time (P 0.7), three 1.2, and an 8-row
// block, which reads fewer halo rows but fills the CU with one barrier's waves,
// 0.97 or 1.03: A with diagonal or full ε is up to 9% faster in 4 rows, P, FP32
// with μ ≠ 1, and FP64 with μ ≠ 1 or HEE on one tile along x up to 6% in 8.  With 64×4 tiles of 16 planes
// 144×120×100 is 630 tiles, three on some CUs, where 20 planes make it 450, two
// on each.
//
// Fitted to sweeps of shapes: P on 14 grids of 52 to 203 cells an axis (whole
// steps, FP64 and FP32, one and three right-hand sides), within 2.5% of the
// fastest; A on 27 grids of 16 to 203 cells with diagonal and full ε, μ ≠ 1 and
// boundft HEE, FP64 and FP32, one and three right-hand sides: 0.2% slower than
// the fastest on average, 3.8% at worst.  The constants of P, which served A as
// well, lost up to 48% there (µs per apply, 4 × 16 → those → these: μ ≠ 1
// 190×33×120 47.1 → 57.1 → 44.1, FP32 96×90×100 65.9 → 69.4 → 46.8, FP32 HEE
// 150×60×170 61.3 → 62.3 → 52.7).
// COCG's fused P, which moves four more vectors, on 10 grids of 24 to 170 cells:
// 2.5% (FP64) and 0.4% slower than the fastest; with P's constants and the width
// of tiles that it does not have it lost up to 33% (µs per step, 4 × 16 → those →
// these: 150×60×170 229.4 → 303.2 → 228.7, FP32 146.7 → 220.0 → 146.2; 70×66×72
// with three right-hand sides 159.1 → 175.5 → 139.9; 190×33×120 99.1 → 108.2 →
// 106.4, where 8 planes would take 99.7).
// P against 4 × 16 with planes halved while a launch had fewer than 256 tiles (µs
// per step): full ε 144×120×100 330.6 → 274.7, μ ≠ 1 80×76×70 96.2 → 80.0, boundft
// HEE 100×90×96 127.1 → 107.5, 110×112×90 138.6 → 121.0, 56×58×52 41.7 → 37.8.
// More than 20 planes lose again (203×180×151: 24 planes 618 µs, 20 planes 593).
inline void tile_rule(const int *N, int64_t nrhs, const TileKernel &K, int &ty_out, int &kz_out) {
    const int per4 = !K.apply && (K.mu || K.gd) ? 1 : (K.apply && !K.fp64 && !K.mu && !K.full && !K.win ? 3 : 2);
    const double alone = K.apply || (K.cocg && !K.fp64) ? 0.8 : (K.cocg ? 0.65 : (per4 == 1 ? 0.5 : 0.7));
    const int nx = (N[0] + (K.narrow ? 31 : 63)) / (K.narrow ? 32 : 64);
    const bool eight_pays = !(K.apply || K.cocg) || per4 == 3 || (K.mu && !K.fp64) || ((K.mu || K.rev) && nx == 1);
    const double eight = eight_pays ? 0.97 : 1.03;
    double least = 1e300;
    for (int ty = 8; ty >= 4; ty /= 2) {
        if (ty == 8 && K.gd && !K.apply) continue;
        const int rows = K.narrow ? 2 * ty : ty;
        const int64_t cols = (int64_t)nx * ((N[1] + rows - 1) / rows);
        for (int kz = 1; kz <= (N[2] < 20 ? N[2] : 20); ++kz) {
            const int64_t most = (cols * ((N[2] + kz - 1) / kz) * nrhs + 255) / 256;
            double rounds;
            if (ty == 8) rounds = (double)most * eight;
            else if (per4 == 1) rounds = (double)most * alone;
            else rounds = (double)(most / per4) * (per4 == 3 ? 1.2 : 1.0) + (most % per4 == 1 ? alone : (most % per4 ? 1.0 : 0.0));
            const double cost = rounds * (kz + 2);
            if (cost < least) {
                least = cost;
                ty_out = ty;
                kz_out = kz;
            }
        }
    }
}

}  // namespace mfd
