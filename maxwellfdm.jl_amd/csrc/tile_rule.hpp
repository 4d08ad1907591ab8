// Shape of a stencil launch's tiles, as plain integer code (host_checks.cpp runs
// it on the CPU).
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

}  // namespace mfd
