// CPU checks of host- and device-shared integer code (needs no GPU and no HIP):
//   host_checks resident    the resident solver's index code, every box shape
//   host_checks scal        the store of a right-hand side's scalars
//   host_checks pays TX TY TZ N0 N1 N2 nc fp64 mu full nrhs steps
//                           whether that many right-hand sides run resident
//   host_checks tile N0 N1 N2 nrhs fp64 apply mu full gd rev win narrow cocg
//                           rows and planes of a tile
//   host_checks fit N0 N1 N2 nrhs narrow ty_max reduces ty kz
//                           the tile made large enough ("no": none is)
// Prints what it covered; a failed check prints itself and ends with status 1.
#include "resident_index.hpp"
#include "scal.hpp"
#include "tile_rule.hpp"
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

using namespace mfd;

#define REQUIRE(c)                                                                        \
    do {                                                                                  \
        if (!(c)) { printf("%s:%d: failed: %s\n", __FILE__, __LINE__, #c); exit(1); }     \
    } while (0)

static long n_grids = 0, n_accesses = 0;

// One grid: every block and thread, as k_resident goes through them.  vb: bytes
// of a vector value.
template <class C>
static void check_grid(const int N[3], int bloch, int rmask, int cmpfirst, int c0, int nc, size_t vb) {
    constexpr int TX = C::TX, TY = C::TY, TZ = C::TZ, CPT = C::CPT, NT = C::NT;
    const int nbx = (N[0] + TX - 1) / TX, nby = (N[1] + TY - 1) / TY, nbz = (N[2] + TZ - 1) / TZ, nb = nbx * nby * nbz;
    const long M = (long)N[0] * N[1] * N[2];
    const int64_t n = (int64_t)nc * M;
    REQUIRE(M <= RES_MAX_CELLS);
    const BoxIndex<C> ix{N[0], N[1], N[2], bloch & 1, bloch >> 1 & 1, bloch >> 2 & 1, rmask, nbx, nby, cmpfirst, c0, nc, (int)M};
    const size_t part_bytes = 16384 * 4 * sizeof(double);
    const int room = res_room(nb, C::CELLS, vb, part_bytes, n);
    const size_t xch_values = (size_t)nb * 3 * C::CELLS;
    if (room == 1) REQUIRE(xch_values * vb <= 2 * part_bytes);
    if (room == 2) REQUIRE(xch_values * vb <= 3 * 16 * (size_t)n);
    REQUIRE(3 * 16 * (uint64_t)M < (1ull << 32) && xch_values * vb < (1ull << 32));
    ++n_grids;
    auto wrapped = [&](int v, int a) { return v < 0 ? v + N[a] : (v >= N[a] ? v - N[a] : v); };
    // the place in the exchange that the owner of (wrapped) cell i, j, k writes
    auto owner_place = [&](int i, int j, int k, int c) {
        i = wrapped(i, 0); j = wrapped(j, 1); k = wrapped(k, 2);
        const int b = i / TX + nbx * (j / TY + nby * (k / TZ));
        return (long)b * 3 * C::CELLS + 3 * (i % TX + TX * (j % TY + TY * (k % TZ))) + c;
    };
    auto caller_cell = [&](int i, int j, int k) {   // of a cell of the grid, by the definition of rmask
        if (rmask & 1) i = N[0] - 1 - i;
        if (rmask & 2) j = N[1] - 1 - j;
        if (rmask & 4) k = N[2] - 1 - k;
        return i + (long)N[0] * (j + (long)N[1] * k);
    };
    // a located cell: the right one, inside every array it indexes
    auto cell = [&](int i, int j, int k, int p, unsigned code) {
        REQUIRE(code < 27);
        const int id[3] = {i, j, k};
        bool in = true;
        for (int a = 0; a < 3; ++a) in = in && (bloch >> a & 1 ? id[a] >= -1 && id[a] <= N[a] : id[a] >= 0 && id[a] < N[a]);
        REQUIRE((p >= 0) == in);
        if (!in) return;
        REQUIRE(p == caller_cell(wrapped(i, 0), wrapped(j, 1), wrapped(k, 2)));
        unsigned want = 0, w = 1;
        for (int a = 0; a < 3; ++a, w *= 3) want += w * (id[a] < 0 ? 1 : (id[a] >= N[a] ? 2 : 0));
        REQUIRE(code == want);
        for (int c = 0; c < 3; ++c) {
            if (!ix.inw(c)) continue;
            REQUIRE(ix.vidx(p, c) >= 0 && ix.vidx(p, c) < n);
            REQUIRE(3L * p + c < 3 * M);
            REQUIRE((long)ix.xidx(i, j, k, c) == owner_place(i, j, k, c) && ix.xidx(i, j, k, c) < xch_values);
            n_accesses += 3;
        }
    };
    std::vector<unsigned char> stagedby(C::XS), cells(C::CELLS), inbox(C::CELLS);
    for (int box = 0; box < nb; ++box) {
        const int i0 = box % nbx * TX, j0 = box / nbx % nby * TY, k0 = box / (nbx * nby) * TZ;
        memset(stagedby.data(), 0, stagedby.size());
        memset(cells.data(), 0, cells.size());
        for (int tid = 0; tid < NT; ++tid) {
            int ii, jq, kq;
            ix.first_cell(tid, ii, jq, kq);
            const int at0 = ix.staged(ii, jq, kq);
            for (int u = 0; u < CPT; ++u) {
                const int jj = jq + u * C::UJ, kk = kq + u * C::UK;
                REQUIRE(ii >= 0 && ii < TX && jj >= 0 && jj < TY && kk >= 0 && kk < TZ);
                const int q = ix.in_box(ii, jj, kk);
                REQUIRE(q >= 0 && q < C::CELLS && !cells[q]);
                cells[q] = 1;
                unsigned code;
                const int i = i0 + ii, j = j0 + jj, k = k0 + kk, p = ix.locate(i, j, k, code);
                cell(i, j, k, p, code);
                const bool own = i < N[0] && j < N[1] && k < N[2];
                REQUIRE(!own || (p >= 0 && code == 0));
                const int at = at0 + u * C::SU;
                REQUIRE(at == ix.staged(ii, jj, kk));
                for (int c = 0; c < 3; ++c) {
                    REQUIRE(at + c >= 0 && at + c < C::XS);
                    ++stagedby[at + c];
                }
                // the staged values that its stencil reads: at most two axes off
                for (int di = -1; di <= 1; ++di)
                    for (int dj = -1; dj <= 1; ++dj)
                        for (int dk = -1; dk <= 1; ++dk) {
                            if (di && dj && dk) continue;
                            const int v = at + di * C::SX + dj * C::SY + dk * C::SZ;
                            REQUIRE(v >= 0 && v + 2 < C::XS);
                            REQUIRE(v == ix.staged(ii + di, jj + dj, C::SLAB ? 0 : kk + dk));
                            ++n_accesses;
                        }
                for (int a = -1; a < 3; ++a) {   // 1/μ at the cell and behind it
                    const int x = ii - (a == 0), y = jj - (a == 1), w = kk - (a == 2);
                    const int m = ix.mu_cell(i0 + x, j0 + y, k0 + w), s = ix.mu_staged(x, y, w);
                    REQUIRE(m >= 0 && m < M && s >= 0 && s + 2 < 3 * C::MX * C::MY * C::MZ);
                    n_accesses += 2;
                }
                if (own) {   // corner ε one cell on (never on a reflected grid)
                    const int f = i + N[0] * (j + N[1] * k);
                    const int px = ix.next_x(f, i), py = ix.next_y(f, j), pz = ix.next_z(f, k);
                    const int to[3] = {px, py, pz}, id[3] = {i, j, k}, st[3] = {1, N[0], N[0] * N[1]};
                    for (int a = 0; a < 3; ++a) {
                        const bool end = id[a] + 1 == N[a], on = !end || (bloch >> a & 1);
                        REQUIRE((to[a] >= 0) == on && to[a] < M);
                        if (on) REQUIRE(to[a] == f + (end ? -(N[a] - 1) : 1) * st[a]);
                    }
                }
            }
            for (int s = 0; s < C::NHS; ++s) {
                const int h = tid + s * NT;
                if (h >= C::NHALO) continue;
                int hi, hj, hk, c;
                ix.halo(h, hi, hj, hk, c);
                REQUIRE(c >= 0 && c < 3 && hi >= -1 && hi <= TX && hj >= -1 && hj <= TY && (C::SLAB ? hk == 0 : hk >= -1 && hk <= TZ));
                const int lp = ix.staged(hi, hj, hk) + c;
                REQUIRE(lp >= 0 && lp < C::XS);
                ++stagedby[lp];
                unsigned code;
                const int ph = ix.locate(i0 + hi, j0 + hj, k0 + hk, code);
                cell(i0 + hi, j0 + hj, k0 + hk, ph, code);
                const unsigned word = ix.pack(lp, c, code);
                REQUIRE(ix.slot_place(word) == lp && ix.slot_comp(word) == c && ix.slot_code(word) == code && word >> 30 == 1);
                REQUIRE(ix.slot_place(word | 1u << 31) == lp);
                n_accesses += 3;
            }
        }
        for (unsigned char v : cells) REQUIRE(v == 1);
        for (unsigned char v : stagedby) REQUIRE(v == 1);   // the box and its halo, each value by one thread
        // staged 1/μ: the place of its fill is the place of its reads
        for (int e = 0; e < 3 * C::MX * C::MY * C::MZ; ++e) {
            const int q = e / 3, mi = q % C::MX, mj = q / C::MX % C::MY, mk = q / (C::MX * C::MY);
            REQUIRE(ix.mu_staged(mi - 1, mj - 1, mk - 1) + e % 3 == e);
            const int m = ix.mu_cell(i0 + mi - 1, j0 + mj - 1, C::SLAB ? 0 : k0 + mk - 1);
            REQUIRE(m >= 0 && m < M);
        }
        // the box's r through the staging buffer, in runs of 8-byte words
        const size_t words = 3 * C::CELLS * vb / 8, runs = 3 * CPT * (vb / 8);
        REQUIRE(words == runs * NT && words * 8 <= C::XS * 16 && (size_t)(box + 1) * words * 8 <= xch_values * vb);
    }
    REQUIRE((size_t)nb * RES_SLOT_WORDS * 8 <= part_bytes || nb > RES_BOXES);
}

template <class C>
static void check_shape(const char *name, size_t vb) {
    const int T[3] = {C::TX, C::TY, C::TZ};
    const long before = n_grids;
    // sizes at and around the box's edges on each axis, then grids of as many
    // boxes as a launch holds
    std::vector<std::vector<int>> sizes(3);
    for (int a = 0; a < 3; ++a) {
        const int t = T[a], cand[] = {1, t - 1, t, t + 1, 2 * t + 1};
        for (int v : cand)
            if (v >= 1 && (!C::SLAB || a < 2 || v == 1)) {
                bool seen = false;
                for (int w : sizes[a]) seen = seen || w == v;
                if (!seen) sizes[a].push_back(v);
            }
    }
    // each with the grid itself, a reflection and a component window; every
    // combination of ends on the small ones
    int turn = 0;
    auto every = [&](const int N[3], bool all) {
        const int boxes = ((N[0] + T[0] - 1) / T[0]) * ((N[1] + T[1] - 1) / T[1]) * ((N[2] + T[2] - 1) / T[2]);
        if (boxes > RES_BOXES) return;
        const int win[5][2] = {{0, 1}, {1, 1}, {2, 1}, {0, 2}, {1, 2}};
        for (int bloch = 0; bloch < 8; bloch += all ? 1 : 7) {
            ++turn;
            check_grid<C>(N, bloch, 0, turn & 1, 0, 3, vb);
            check_grid<C>(N, bloch, 1 + turn % 7, turn >> 1 & 1, 0, 3, vb);
            check_grid<C>(N, bloch, 0, 0, win[turn % 5][0], win[turn % 5][1], vb);
        }
    };
    for (int x : sizes[0])
        for (int y : sizes[1])
            for (int z : sizes[2]) {
                const int N[3] = {x, y, z};
                if ((x > T[0] + 1) + (y > T[1] + 1) + (z > T[2] + 1) <= 1) every(N, true);   // (three boxes on one axis)
            }
    // near the limit of 256 boxes: cubes (squares), slabs and rods
    const int lim[][3] = {{6, 6, 7}, {4, 8, 8}, {8, 4, 8}, {16, 16, 1}, {1, 16, 16}, {256, 1, 1}, {1, 256, 1}, {1, 1, 256}, {15, 17, 1}, {3, 5, 17}};
    for (auto &l : lim) {
        if (C::SLAB && l[2] > 1) continue;
        int N[3];
        for (int a = 0; a < 3; ++a) N[a] = l[a] * T[a] > 1 ? l[a] * T[a] - 1 : 1;
        every(N, false);
    }
    printf("%s: %ld grids\n", name, n_grids - before);
}

static void resident() {
#define SHAPE(X, Y, Z, P, VB) check_shape<BoxCfg<X, Y, Z, P>>(#X "x" #Y "x" #Z ", " #P " a thread, " #VB " bytes", VB)
    // the dispatched shapes (with FP32 vectors only the exchange shrinks), and
    // those of FP32 vectors only
    SHAPE(8, 4, 4, 1, 16);
    SHAPE(8, 8, 4, 1, 16);
    SHAPE(16, 8, 4, 2, 16);
    SHAPE(16, 8, 1, 1, 16);
    SHAPE(32, 16, 1, 2, 16);
    SHAPE(16, 8, 8, 4, 8);
    SHAPE(32, 32, 1, 4, 8);
    // not dispatched: 1,024 cells a box with FP64 vectors
    SHAPE(16, 8, 8, 4, 16);
    SHAPE(32, 32, 1, 4, 16);
#undef SHAPE
    printf("resident ok: %ld grids, %ld accesses\n", n_grids, n_accesses);
}

// a mark set after the scalars were read survives their store; all else is stored
static void scal() {
    Scal s, to;
    memset((void *)&s, 0x5a, sizeof s);
    memset((void *)&to, 0, sizeof to);
    to.stag = -1;
    scal_store(to, s);
    REQUIRE(to.stag == -1);
    to.stag = s.stag;
    REQUIRE(!memcmp((const void *)&to, (const void *)&s, sizeof s));
    printf("scal ok\n");
}

int main(int argc, char **argv) {
    if (argc == 2 && !strcmp(argv[1], "resident")) { resident(); return 0; }
    if (argc == 2 && !strcmp(argv[1], "scal")) { scal(); return 0; }
    if (argc == 14 && !strcmp(argv[1], "pays")) {
        int v[12];
        for (int k = 0; k < 12; ++k) v[k] = atoi(argv[2 + k]);
        int boxes = 1;
        for (int a = 0; a < 3; ++a) boxes *= (v[3 + a] + v[a] - 1) / v[a];
        const ResForm f = {v[7] != 0, v[8] != 0, v[9] != 0, v[5] == 1, v[6]};
        printf("%d\n", (int)res_pays(f, boxes, v[0] * v[1] * v[2], RES_BOXES, (int64_t)v[3] * v[4] * v[5], v[10], v[11]));
        return 0;
    }
    if (argc == 15 && !strcmp(argv[1], "tile")) {
        int v[13], ty = 0, kz = 0;
        for (int k = 0; k < 13; ++k) v[k] = atoi(argv[2 + k]);
        const TileKernel K = {v[4] != 0, v[5] != 0, v[6] != 0, v[7] != 0, v[8] != 0, v[9] != 0, v[10] != 0, v[11] != 0, v[12] != 0};
        tile_rule(v, v[3], K, ty, kz);
        printf("%d %d\n", ty, kz);
        return 0;
    }
    if (argc == 11 && !strcmp(argv[1], "fit")) {
        int v[9];
        for (int k = 0; k < 9; ++k) v[k] = atoi(argv[2 + k]);
        if (tile_fit(v, v[3], v[4] != 0, v[5], v[6] != 0, 16384, v[7], v[8])) printf("%d %d\n", v[7], v[8]);
        else printf("no\n");
        return 0;
    }
    printf("usage: host_checks resident | scal | pays ... | tile ... | fit ...\n");
    return 2;
}
