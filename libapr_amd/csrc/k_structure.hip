/*
 * k_structure.hip -- pulling scheme, linear particle structure and particle
 * sampling on gfx950.
 *
 *  - level pyramid + particle-cell seeds: 2x2x2 max downsample of the level
 *    map fused with PullingScheme::fill (LocalParticleCellSet.hpp:58-91,
 *    PullingScheme.hpp:140-168).
 *  - pulling scheme: one in-place pass per level, top to bottom, fusing
 *    set_ascendant_neighbours, set_filler and fill_neighbours/fill_parent
 *    (PullingScheme.hpp:111-393).  The per-cell predicates only test states
 *    that the pass cannot create or destroy (ASCENDANT; SEED-or-PROPOGATE),
 *    so concurrent in-place updates give the sequential result.
 *  - linear structure (LinearAccess.hpp:210-524): equivalence optimisation
 *    level by level, then per-row particle counts (a wave per row, 16 cells
 *    per lane), one exclusive scan over all rows in particle order (which is
 *    xz_end_vec), and a wave-per-row fill of y_vec with ballot prefix counts.
 *  - sampling (ParticleData.hpp:221-261): mean pyramid of the image, then a
 *    row-parallel gather.
 */
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "aprh_internal.hpp"
#include "tiles.hpp"

namespace aprh {

namespace {

constexpr int MAXL = 24;
enum : uint8_t { EMPTY = 0, SEED = 1, BOUNDARY = 2, FILLER = 3, UPSEED = 4, ASC = 8, PROP = 15, ASCN = 16 };

struct Dims {
    int64_t y, x, z;
};

/* ---- four cells in a 32-bit word, one byte each ---- */
__device__ __forceinline__ uint32_t rep4(uint32_t b) { return b * 0x01010101u; }
/* 0x80 in every byte of w that is 0 */
__device__ __forceinline__ uint32_t zero4(uint32_t w) { return ~(((w & 0x7f7f7f7fu) + 0x7f7f7f7fu) | w | 0x7f7f7f7fu); }
/* bit k of the result <- bit 7 of byte k */
__device__ __forceinline__ uint32_t bits4(uint32_t flags) { return (((flags >> 7) & 0x01010101u) * 0x10204080u) >> 28; }
/* per byte, values below 128: the larger of two */
__device__ __forceinline__ uint32_t max4(uint32_t a, uint32_t b) {
    const uint32_t ge = (((a | 0x80808080u) - b) >> 7) & 0x01010101u;
    const uint32_t m = ge * 0xFFu;
    return (a & m) | (b & ~m);
}
/* SEED or EMPTY per byte from four levels (below 32): >= level (mode 0), <= level (1), == level (2) */
__device__ __forceinline__ uint32_t seed4(uint32_t w, int level, int mode) {
    const uint32_t ge = w + rep4(128u - (uint32_t)level), le = rep4(128u + (uint32_t)level) - w;
    const uint32_t t = mode == 0 ? ge : mode == 1 ? le : ge & le;
    return (t >> 7) & 0x01010101u;
}
__device__ __forceinline__ uint8_t seed_of(uint8_t m, int level, int mode) {
    const bool seed = (mode == 0) ? (m >= level) : (mode == 1) ? (m <= level) : (m == level);
    return seed ? SEED : EMPTY;
}

/* level map of level l from level l + 1 (max of the clamped 2x2x2 block) and the seeds of level l; with
   fpct, also the seeds of level l + 1 itself (the top level: every fine cell is in exactly one block).
   A lane takes eight coarse cells along y: four 16-byte row loads at any alignment.  At the top of
   1024 x 1024 x 256 maps, seeds and first level took 0.28 ms a byte at a time in two launches. */
struct DownArgs {
    const uint8_t* fine;
    Dims fd;
    uint8_t* coarse;
    Dims cd;
    uint8_t* pct;
    int level, mode;
    uint8_t* fpct;     /* seeds of the fine level (mode 0), or nullptr */
    int64_t G;
    FastDiv fg, fx;    /* division by the groups of a row, by cd.x */
    int i32;
};
__device__ __forceinline__ void level_down_body(const DownArgs& a, int64_t G, int64_t t) {
    const Dims fd = a.fd, cd = a.cd;
    const int64_t ng = (cd.y + 7) >> 3, total = ng * cd.x * cd.z;
    for (int64_t i = t * blockDim.x + threadIdx.x; i < total; i += G * blockDim.x) {
        int64_t g, x, z;
        if (a.i32) {
            const uint32_t r = a.fg.div((uint32_t)i), zz = a.fx.div(r);
            g = (uint32_t)i - r * (uint32_t)ng;
            x = r - zz * (uint32_t)cd.x;
            z = zz;
        } else {
            const int64_t r = i / ng;
            g = i - r * ng;
            z = r / cd.x;
            x = r - z * cd.x;
        }
        const int64_t y0 = 16 * g, c0 = 8 * g;
        const int64_t x1 = min(2 * x + 1, fd.x - 1), z1 = min(2 * z + 1, fd.z - 1);
        const int64_t rows[4] = {(2 * z * fd.x + 2 * x) * fd.y, (2 * z * fd.x + x1) * fd.y, (z1 * fd.x + 2 * x) * fd.y, (z1 * fd.x + x1) * fd.y};
        const int64_t o = (z * cd.x + x) * cd.y + c0;
        if (y0 + 16 <= fd.y) {
            uint32_t w[4][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) __builtin_memcpy(w[q], a.fine + rows[q] + y0, 16);
            if (a.fpct) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint32_t f[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) f[k] = seed4(w[q][k], a.level + 1, 0);
                    __builtin_memcpy(a.fpct + rows[q] + y0, f, 16);   /* rows that coincide get the same bytes twice */
                }
            }
            uint32_t m[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                uint32_t h[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int q = 2 * k + u;
                    const uint32_t v = max4(max4(w[0][q], w[1][q]), max4(w[2][q], w[3][q]));
                    const uint32_t p = max4(v, v >> 8);
                    h[u] = (p & 0xFFu) | ((p >> 8) & 0xFF00u);
                }
                m[k] = h[0] | (h[1] << 16);
            }
            const uint32_t sd[2] = {seed4(m[0], a.level, a.mode), seed4(m[1], a.level, a.mode)};
            __builtin_memcpy(a.coarse + o, m, 8);
            __builtin_memcpy(a.pct + o, sd, 8);
        } else {
            for (int j = 0; j < 8 && c0 + j < cd.y; ++j) {
                const int64_t ya = y0 + 2 * j, yb = min(ya + 1, fd.y - 1);
                uint8_t m = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint8_t va = a.fine[rows[q] + ya], vb = a.fine[rows[q] + yb];
                    m = max(m, max(va, vb));
                    if (a.fpct) {
                        a.fpct[rows[q] + ya] = seed_of(va, a.level + 1, 0);
                        a.fpct[rows[q] + yb] = seed_of(vb, a.level + 1, 0);
                    }
                }
                a.coarse[o + j] = m;
                a.pct[o + j] = seed_of(m, a.level, a.mode);
            }
        }
    }
}

/* one pulling-scheme level (PullingScheme.hpp:111-132 loop body): set_ascendant_neighbours
   and fill_neighbours on this level, set_filler on the finer one, fill_parent on the coarser
   one.  One lane per 8 consecutive y cells: the 3x3x3 neighbourhood predicates are formed as bit masks
   over the 9 neighbouring rows (10 bits: y0-1 .. y0+8), dilated along y by shifts.
   A lane marches over a run of zc planes, keeping the ASCENDANT / SEED-or-PROPOGATE masks of the planes
   z-1, z, z+1 (each the OR over rows x-1, x, x+1): every plane's three rows are loaded once instead of
   three times.  A cell's state is written only by its owner lane, so the cached words of the own row are
   current, and the 16 x 2 x 2 children of a lane's cells belong to it alone, so set_filler rewrites them
   as whole words: four row loads at once, where one load and store after the other for every child made a
   chain of up to 64 (28 us for a level of a few thousand cells, 10 us now).
   atomics: fill_parent ORs whole parent words; else it stores the bytes it turns to ASCENDANT (inside one
   block, where other waves read them after a barrier, and for parent rows that straddle words). */
struct PullArgs {
    uint8_t* P;
    Dims d;
    uint8_t* Pc;
    Dims dc;
    uint8_t* Pp;
    Dims dp;
    int is_top, has_parent;
    int zc, atomics;
    int64_t G;
};
__device__ __forceinline__ void pull_level8_body(const PullArgs& a, int64_t G, int64_t t) {
    uint8_t* const P = a.P;
    const Dims dc = a.dc, dp = a.dp;
    const bool is_top = a.is_top, has_parent = a.has_parent;
    const int yn = (int)a.d.y, xn = (int)a.d.x, zn = (int)a.d.z, ZC = a.zc;
    const int nwr = (yn + 7) >> 3;
    const int nzc = (zn + ZC - 1) / ZC;
    const int64_t total = (int64_t)nwr * xn * nzc;
    /* parent rows whose words never straddle two rows */
    const bool par_words = a.atomics && (dp.y & 3) == 0 && ((uintptr_t)a.Pp & 3) == 0;
    for (int64_t i = t * blockDim.x + threadIdx.x; i < total; i += G * blockDim.x) {
        const int w = (int)(i % nwr);
        const int64_t r = i / nwr;
        const int x = (int)(r % xn), zc = (int)(r / xn);
        const int y0 = w * 8;
        const int z_begin = zc * ZC, z_end = min(zn, z_begin + ZC);
        /* the rows x - 1, x, x + 1 of plane zz at y0 - 4 .. y0 + 11, one 16-byte load each at any alignment
           (x and zz clamped: the loads carry no branches, and masks() leaves out what lies outside); near
           the row's ends only the ten cells y0 - 1 .. y0 + 8, zeros past them */
        auto load3 = [&](int zz, uint32_t (&v)[3][4]) {
            const int zc2 = min(max(zz, 0), zn - 1);
            const uint8_t* rows[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) rows[k] = P + ((int64_t)zc2 * xn + min(max(x + k - 1, 0), xn - 1)) * yn;
            if (y0 >= 4 && y0 + 12 <= yn) {
#pragma unroll
                for (int k = 0; k < 3; ++k) __builtin_memcpy(v[k], rows[k] + y0 - 4, 16);
            } else if (y0 + 8 <= yn) {
                uint8_t l[3], r[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    __builtin_memcpy(&v[k][1], rows[k] + y0, 8);
                    l[k] = rows[k][max(y0 - 1, 0)];
                    r[k] = rows[k][min(y0 + 8, yn - 1)];
                }
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    v[k][0] = y0 > 0 ? (uint32_t)l[k] << 24 : 0u;
                    v[k][3] = y0 + 8 < yn ? r[k] : 0u;
                }
            } else {
                uint8_t c[3][9];
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int j = 0; j < 9; ++j) c[k][j] = rows[k][min(max(y0 - 1 + j, 0), yn - 1)];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    v[k][0] = y0 > 0 ? (uint32_t)c[k][0] << 24 : 0u;
                    v[k][1] = v[k][2] = v[k][3] = 0u;
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (y0 + j < yn) v[k][1 + (j >> 2)] |= (uint32_t)c[k][1 + j] << (8 * (j & 3));
                }
            }
        };
        /* masks of plane zz (0 outside the volume; bit k <-> y0 - 1 + k); own row's words in own[] */
        auto masks = [&](int zz, const uint32_t (&v)[3][4], uint32_t& am, uint32_t& sm, uint32_t own[2]) {
            am = 0;
            sm = 0;
            own[0] = v[1][1];
            own[1] = v[1][2];
            if (zz < 0 || zz >= zn) return;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if ((k == 0 && x == 0) || (k == 2 && x == xn - 1)) continue;
                const uint32_t lf = v[k][0] >> 24, c0 = v[k][1], c1 = v[k][2], rt = v[k][3] & 0xFFu;
                am |= (bits4(zero4(c0 ^ rep4(ASC))) << 1) | (bits4(zero4(c1 ^ rep4(ASC))) << 5) | (lf == ASC ? 1u : 0u) | (rt == ASC ? 0x200u : 0u);
                sm |= (bits4(zero4(c0 ^ rep4(SEED)) | zero4(c0 ^ rep4(PROP))) << 1) | (bits4(zero4(c1 ^ rep4(SEED)) | zero4(c1 ^ rep4(PROP))) << 5) |
                      (lf == SEED || lf == PROP ? 1u : 0u) | (rt == SEED || rt == PROP ? 0x200u : 0u);
            }
        };
        uint32_t pa0, ps0, pa1, ps1, pa2, ps2;
        uint32_t cur[2] = {0, 0}, nxt[2] = {0, 0};
        uint32_t v0[3][4], v1[3][4], v2[3][4];
        load3(z_begin - 1, v0);
        load3(z_begin, v1);
        load3(z_begin + 1, v2);
        masks(z_begin - 1, v0, pa0, ps0, nxt);
        masks(z_begin, v1, pa1, ps1, cur);
        for (int z = z_begin; z < z_end; ++z) {
            masks(z + 1, v2, pa2, ps2, nxt);
            if (z + 1 < z_end) load3(z + 2, v2);
            const uint32_t am = pa0 | pa1 | pa2, sm = ps0 | ps1 | ps2;
            const uint32_t ad = am | (am << 1) | (am >> 1), sd = sm | (sm << 1) | (sm >> 1);
            uint8_t* row = P + ((int64_t)z * xn + x) * yn;
            uint32_t nb[2] = {0, 0};
            uint32_t fill = 0, up = 0;   /* cells whose children are filled; cells that raise their parent */
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t old = (cur[j >> 2] >> (8 * (j & 3))) & 0xFFu;
                const bool any_asc = (ad >> (j + 1)) & 1u, any_sp = (sd >> (j + 1)) & 1u;
                uint32_t nw = old;
                if (!is_top) {
                    if (old == EMPTY) nw = any_asc ? ASCN : (any_sp ? BOUNDARY : EMPTY);
                    else if (old == SEED) nw = any_asc ? PROP : SEED;
                } else if (old == EMPTY && any_sp) {
                    nw = BOUNDARY;
                }
                nb[j >> 2] |= nw << (8 * (j & 3));
                if (y0 + j < yn) {
                    fill |= (uint32_t)(!is_top && (nw == ASCN || nw == PROP)) << j;
                    up |= (uint32_t)(nw == SEED || nw == PROP || nw == ASC) << j;
                }
            }
            if (y0 + 8 <= yn) {
                if (nb[0] != cur[0] || nb[1] != cur[1]) __builtin_memcpy(row + y0, nb, 8);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint8_t v = (uint8_t)(nb[j >> 2] >> (8 * (j & 3)));
                    if (y0 + j < yn && v != (uint8_t)(cur[j >> 2] >> (8 * (j & 3)))) row[y0 + j] = v;
                }
            }
            /* fill_parent.  The parent level holds only EMPTY, SEED and ASCENDANT now (its seeds, and
               ASCENDANT from this pass), so every non-SEED byte wanted becomes ASCENDANT, in any order
               between lanes that share a parent cell or word */
            if (has_parent && up) {
                uint8_t* pp = a.Pp + ((int64_t)(z / 2) * dp.x + (x / 2)) * dp.y + (y0 / 2);
                const uint32_t want = (up & 3u ? 0xFFu : 0u) | (up & 0xCu ? 0xFF00u : 0u) | (up & 0x30u ? 0xFF0000u : 0u) | (up & 0xC0u ? 0xFF000000u : 0u);
                uint32_t cur4 = 0;
                if (y0 / 2 + 4 <= dp.y) {
                    __builtin_memcpy(&cur4, pp, 4);
                } else {
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        if (y0 / 2 + q < dp.y) cur4 |= (uint32_t)pp[q] << (8 * q);
                }
                const uint32_t isseed = (zero4(cur4 ^ rep4(SEED)) >> 7) * 0xFFu, isasc = (zero4(cur4 ^ rep4(ASC)) >> 7) * 0xFFu;
                const uint32_t turn = want & ~isseed & ~isasc;
                if (turn) {
                    if (par_words) {
                        atomicOr((uint32_t*)pp, turn & rep4(ASC));
                    } else {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if ((turn >> (8 * q)) & 0xFFu) pp[q] = ASC;
                    }
                }
            }
            /* set_filler: empty children of ASCENDANTNEIGHBOUR / PROPOGATE become FILLER */
            if (fill) {
                const int cz = (z == zn - 1 && (dc.z & 1)) ? 1 : 2, cx = (x == xn - 1 && (dc.x & 1)) ? 1 : 2;
                uint8_t* c00 = a.Pc + ((int64_t)(2 * z) * dc.x + 2 * x) * dc.y + 2 * y0;
                uint8_t* crow[4] = {c00, c00 + (cx == 2 ? dc.y : 0), c00 + (cz == 2 ? dc.x * dc.y : 0),
                                    c00 + (cx == 2 ? dc.y : 0) + (cz == 2 ? dc.x * dc.y : 0)};
                if (2 * y0 + 16 <= dc.y) {
                    uint32_t m[4];   /* FILLER in the two children of every such cell */
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        m[q] = (((fill >> (2 * q)) & 1u) ? 0x0000FFFFu : 0u) | (((fill >> (2 * q + 1)) & 1u) ? 0xFFFF0000u : 0u);
                    uint32_t v[4][4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) __builtin_memcpy(v[q], crow[q], 16);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint32_t any = 0;
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const uint32_t f = (zero4(v[q][k]) >> 7) * (uint32_t)FILLER & m[k];
                            v[q][k] |= f;
                            any |= f;
                        }
                        if (any) __builtin_memcpy(crow[q], v[q], 16);   /* rows that coincide get the same bytes twice */
                    }
                } else {
                    for (int j = 0; j < 8; ++j) {
                        if (!((fill >> j) & 1u)) continue;
                        const int cy = (y0 + j == yn - 1 && (dc.y & 1)) ? 1 : 2;
                        for (int q = 0; q < 4; ++q)
                            for (int c = 0; c < cy; ++c)
                                if (crow[q][2 * j + c] == EMPTY) crow[q][2 * j + c] = FILLER;
                    }
                }
            }
            pa0 = pa1;
            ps0 = ps1;
            pa1 = pa2;
            ps1 = ps2;
            cur[0] = nxt[0];
            cur[1] = nxt[1];
        }
    }
}

/* equivalence optimisation step for one level (LinearAccess.hpp:265-294): a lane takes eight cells along
   y, i.e. four parent cells, and writes only under parents of type 1 .. min_type.  (A cell per lane with
   its own division: 0.37 ms over the levels of a 2048 x 2048 x 512 volume.) */
struct UpseedArgs {
    uint8_t* P;
    Dims d;
    const uint8_t* Pp;
    Dims dp;
    int min_type;
    int64_t G;
    FastDiv fg, fx;   /* division by the groups of a row, by d.x */
    int i32;
};
__device__ __forceinline__ void upseed_body(const UpseedArgs& a, int64_t G, int64_t t) {
    const Dims d = a.d, dp = a.dp;
    const int64_t ng = (d.y + 7) >> 3, total = ng * d.x * d.z;
    for (int64_t i = t * blockDim.x + threadIdx.x; i < total; i += G * blockDim.x) {
        int64_t g, x, z;
        if (a.i32) {
            const uint32_t r = a.fg.div((uint32_t)i), zz = a.fx.div(r);
            g = (uint32_t)i - r * (uint32_t)ng;
            x = r - zz * (uint32_t)d.x;
            z = zz;
        } else {
            const int64_t r = i / ng;
            g = i - r * ng;
            z = r / d.x;
            x = r - z * d.x;
        }
        const uint8_t* pp = a.Pp + ((z / 2) * dp.x + (x / 2)) * dp.y + 4 * g;
        uint32_t s = 0;
        if (4 * g + 4 <= dp.y) {
            __builtin_memcpy(&s, pp, 4);
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (4 * g + q < dp.y) s |= (uint32_t)pp[q] << (8 * q);
        }
        uint32_t on = 0;   /* parents of type 1 .. min_type */
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t v = (s >> (8 * q)) & 0xFFu;
            on |= (uint32_t)(v > 0 && v <= (uint32_t)a.min_type) << q;
        }
        if (!on) continue;
        const int64_t y0 = 8 * g;
        uint8_t* p = a.P + (z * d.x + x) * d.y + y0;
        if (on == 0xFu && y0 + 8 <= d.y) {
            const uint32_t u[2] = {rep4(UPSEED), rep4(UPSEED)};
            __builtin_memcpy(p, u, 8);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if ((on >> q) & 1u) {
                    p[2 * q] = UPSEED;
                    if (y0 + 2 * q + 1 < d.y) p[2 * q + 1] = UPSEED;
                }
        }
    }
}

/* row table of the APR levels l_min..l_max and the particle-cell maps that define them */
struct RowTable {
    int n_levels;                 /* APR levels l_min..l_max           */
    int l_min, l_max;
    int64_t row_begin[MAXL];      /* xz_end index of row 0 of level    */
    int64_t rows_x[MAXL];         /* x_num of the APR level            */
    int64_t map_off[MAXL];        /* byte offset of the pct map used   */
    int64_t map_y[MAXL], map_x[MAXL]; /* dims of that pct map           */
    int64_t y_max;                /* y_num at l_max                    */
    int64_t row_prefix[MAXL + 1]; /* first global row of each APR level */
    int min_type;
    /* the l_max rows (z, x) read pct row (z/2, x/2) of l_max - 1, so up to four of them hold
       identical particles: work items are the rows below l_max, then one per such pct row */
    int64_t top_z;                /* z_num at l_max                    */
    int64_t top_pz;               /* z_num at l_max - 1                */
    int64_t n_work;               /* row_prefix[top] + map_x * top_pz  */
};

/* weight of one pct cell for APR level li (0 or 1; 0..2 at l_max) */
__device__ __forceinline__ int cell_weight(const RowTable& t, int li, uint8_t st, int64_t yy) {
    if (li == t.n_levels - 1) {
        if (st > 0 && st <= t.min_type) return 1 + ((2 * yy < t.y_max - 1) ? 1 : 0);
        return 0;
    }
    return (st > t.min_type && st <= UPSEED) ? 1 : 0;
}

__device__ __forceinline__ int row_level_of(const RowTable& t, int64_t r) {
    int li = 0;
    while (li + 1 < t.n_levels && r >= t.row_prefix[li + 1]) ++li;
    return li;
}

constexpr int CPL = 16;   /* cells per lane per chunk: a wave covers 1024 cells of a row */

/* weights of the CPL cells [c0, c0 + CPL) of a row (0 beyond its end) */
__device__ __forceinline__ void chunk_weights(const RowTable& t, int li, const uint8_t* p, int ylen, int c0, int w[CPL]) {
    if (c0 + CPL <= ylen) {   /* one 16-byte load at any alignment */
        uint4 v;
        __builtin_memcpy(&v, p + c0, 16);
        const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < CPL; ++j) w[j] = cell_weight(t, li, (uint8_t)(words[j >> 2] >> (8 * (j & 3))), c0 + j);
    } else {
#pragma unroll
        for (int j = 0; j < CPL; ++j) w[j] = (c0 + j < ylen) ? cell_weight(t, li, p[c0 + j], c0 + j) : 0;
    }
}

/* the APR rows of work item w (1, or up to 4 sharing a pct row at l_max) and its cells */
struct WorkRows {
    int li;
    const uint8_t* p;     /* pct row          */
    int ylen;
    int n;                /* destination rows */
    int64_t r[4];
};
__device__ __forceinline__ WorkRows work_rows(const RowTable& t, const uint8_t* maps, int64_t w) {
    WorkRows o;
    const int top = t.n_levels - 1;
    if (w < t.row_prefix[top]) {
        o.li = row_level_of(t, w);
        o.p = maps + t.map_off[o.li] + (w - t.row_prefix[o.li]) * t.map_y[o.li];
        o.n = 1;
        o.r[0] = w;
    } else {
        const int64_t prow = w - t.row_prefix[top];
        const int64_t zm = prow / t.map_x[top], xm = prow - zm * t.map_x[top];
        o.li = top;
        o.p = maps + t.map_off[top] + prow * t.map_y[top];
        /* rows (2zm, 2xm), (2zm, 2xm+1), (2zm+1, 2xm), (2zm+1, 2xm+1) that exist, in that order */
        const bool hx = 2 * xm + 1 < t.rows_x[top], hz = 2 * zm + 1 < t.top_z;
        const int64_t r00 = t.row_prefix[top] + 2 * zm * t.rows_x[top] + 2 * xm;
        o.r[0] = r00;
        o.r[1] = hx ? r00 + 1 : r00 + t.rows_x[top];
        o.r[2] = hx ? r00 + t.rows_x[top] : r00;
        o.r[3] = r00 + t.rows_x[top] + 1;
        o.n = 1 + (hx ? 1 : 0) + (hz ? 1 : 0) + ((hx && hz) ? 1 : 0);
    }
    o.ylen = (int)t.map_y[o.li];
    return o;
}

/* particles of each APR row: 16 lanes per work item, 256 cells per step (short rows of small
   volumes and coarse levels keep the lanes busy; long rows loop) */
constexpr int COUNT_LANES = 16;
__device__ __forceinline__ void row_count_body(const uint8_t* __restrict__ maps, const RowTable& t, int64_t nrows, uint32_t* cnt,
                                               int64_t G, int64_t blk) {
    const int lane = threadIdx.x & (COUNT_LANES - 1);
    const int64_t wid = (blk * blockDim.x + threadIdx.x) / COUNT_LANES;
    const int64_t nw = (G * blockDim.x) / COUNT_LANES;
    (void)nrows;
    for (int64_t w = wid; w < t.n_work; w += nw) {
        const WorkRows wr = work_rows(t, maps, w);
        uint32_t c = 0;
        for (int base = 0; base < wr.ylen; base += COUNT_LANES * CPL) {
            int wt[CPL];
            chunk_weights(t, wr.li, wr.p, wr.ylen, base + lane * CPL, wt);
#pragma unroll
            for (int j = 0; j < CPL; ++j) c += (uint32_t)wt[j];
        }
        /* the 16 lanes of a group share w, so they are active together */
        for (int o = COUNT_LANES / 2; o > 0; o >>= 1) c += __shfl_xor(c, o, COUNT_LANES);
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k < wr.n) cnt[wr.r[k]] = c;
        }
    }
}

/* y values of each APR row from its scanned offset.  A group of FILL_LANES lanes (a whole wave
   for long rows, 16 lanes for short ones) takes one work item; a lane takes CPL consecutive
   cells of a FILL_LANES * CPL-cell chunk; a prefix sum over the group places each lane's values
   in the group's LDS stage, which the group then copies to y_vec with consecutive lanes on
   consecutive entries (once per destination row). */
constexpr int FILL_WAVES = 4;
/* level images for a row fill that also samples: APR level index li -> image of that level
   (the converted image at l_max, the mean pyramid below), rows in (z, x) order like the APR rows */
struct RowImages {
    const uint16_t* img[MAXL];
    int64_t y[MAXL];
    uint16_t* parts;   /* nullptr: no sampling */
};

template <int FILL_LANES>
__device__ __forceinline__ void row_fill_body(const uint8_t* __restrict__ maps, const RowTable& t, int64_t nrows,
                                              const uint64_t* __restrict__ row_off, uint16_t* y_vec, const RowImages& ri, int64_t G,
                                              int64_t blk) {
    constexpr int FILL_GROUPS = FILL_WAVES * 64 / FILL_LANES;
    __shared__ uint16_t stage[FILL_GROUPS][2 * FILL_LANES * CPL];
    const int lane = threadIdx.x & (FILL_LANES - 1);
    uint16_t* st = stage[threadIdx.x / FILL_LANES];
    const int64_t wid = (blk * blockDim.x + threadIdx.x) / FILL_LANES;
    const int64_t nw = (G * blockDim.x) / FILL_LANES;
    (void)nrows;
    /* the 16 lanes of a group share w (and every loop bound below), so they are active together */
    for (int64_t w = wid; w < t.n_work; w += nw) {
        const WorkRows wr = work_rows(t, maps, w);
        const bool top = (wr.li == t.n_levels - 1);
        uint64_t pos[4] = {0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (k < wr.n) pos[k] = row_off[wr.r[k]];
        for (int base = 0; base < wr.ylen; base += FILL_LANES * CPL) {
            int wt[CPL];
            const int c0 = base + lane * CPL;
            chunk_weights(t, wr.li, wr.p, wr.ylen, c0, wt);
            int c = 0;
#pragma unroll
            for (int j = 0; j < CPL; ++j) c += wt[j];
            /* inclusive prefix over the group */
            int incl = c;
            for (int o = 1; o < FILL_LANES; o <<= 1) {
                const int v = __shfl_up(incl, o, FILL_LANES);
                if (lane >= o) incl += v;
            }
            const int total = __shfl(incl, FILL_LANES - 1, FILL_LANES);
            int q = incl - c;
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int yy = c0 + j;
                if (wt[j] >= 1) st[q++] = (uint16_t)(top ? 2 * yy : yy);
                if (wt[j] == 2) st[q++] = (uint16_t)(2 * yy + 1);
            }
            __threadfence_block();
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (k >= wr.n) break;
                uint16_t* dst = y_vec + pos[k];
                if (ri.parts) {
                    /* sample_image's gather (ParticleData.hpp:221-261) for this row's particles */
                    const uint16_t* irow = ri.img[wr.li] + (wr.r[k] - t.row_prefix[wr.li]) * ri.y[wr.li];
                    uint16_t* pdst = ri.parts + pos[k];
                    int i = lane;
                    /* four particles per lane in flight */
                    for (; i + 3 * FILL_LANES < total; i += 4 * FILL_LANES) {
                        const uint16_t y0 = st[i], y1 = st[i + FILL_LANES], y2 = st[i + 2 * FILL_LANES], y3 = st[i + 3 * FILL_LANES];
                        const uint16_t v0 = irow[y0], v1 = irow[y1], v2 = irow[y2], v3 = irow[y3];
                        dst[i] = y0;
                        dst[i + FILL_LANES] = y1;
                        dst[i + 2 * FILL_LANES] = y2;
                        dst[i + 3 * FILL_LANES] = y3;
                        pdst[i] = v0;
                        pdst[i + FILL_LANES] = v1;
                        pdst[i + 2 * FILL_LANES] = v2;
                        pdst[i + 3 * FILL_LANES] = v3;
                    }
                    for (; i < total; i += FILL_LANES) {
                        const uint16_t yv = st[i];
                        dst[i] = yv;
                        pdst[i] = irow[yv];
                    }
                } else {
                    for (int i = lane; i < total; i += FILL_LANES) dst[i] = st[i];
                }
                pos[k] += (uint64_t)total;
            }
            __threadfence_block();   /* the stage is rewritten by the next chunk */
        }
    }
}

/* xz_end_vec of each row: its offset + its count */
__device__ __forceinline__ void rows_xz_body(const uint64_t* __restrict__ row_off, const uint32_t* __restrict__ cnt, const RowTable& t,
                                             uint64_t* xz_end, int64_t nrows, int64_t blk) {
    const int64_t r = blk * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    const int li = row_level_of(t, r);
    xz_end[t.row_begin[li] + (r - t.row_prefix[li])] = row_off[r] + cnt[r];
}

/* exclusive scan, three phases over blocks of 1024 */
__device__ __forceinline__ void scan_blocks_body(const uint32_t* __restrict__ in, uint64_t* out, uint64_t* block_sums, int64_t n,
                                                 int64_t blk) {
    __shared__ uint64_t sh[1024];
    const int64_t i = blk * 1024 + threadIdx.x;
    uint64_t v = i < n ? in[i] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        uint64_t a = threadIdx.x >= (unsigned)o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += a;
        __syncthreads();
    }
    if (i < n) out[i] = sh[threadIdx.x] - v;
    if (threadIdx.x == 1023) block_sums[blk] = sh[1023];
    __syncthreads();   /* sh is reused by the next tile of a persistent block */
}

__device__ __forceinline__ void scan_sums_body(uint64_t* block_sums, int64_t nb, uint64_t* total) {
    /* single block: exclusive scan of the block sums (serial chunks per thread) */
    __shared__ uint64_t sh[1024];
    const int64_t per = (nb + 1023) / 1024;
    const int64_t b = (int64_t)threadIdx.x * per;
    uint64_t s = 0;
    for (int64_t k = b; k < min(b + per, nb); ++k) s += block_sums[k];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        uint64_t a = threadIdx.x >= (unsigned)o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += a;
        __syncthreads();
    }
    uint64_t run = sh[threadIdx.x] - s;
    for (int64_t k = b; k < min(b + per, nb); ++k) {
        uint64_t v = block_sums[k];
        block_sums[k] = run;
        run += v;
    }
    if (threadIdx.x == 1023) *total = sh[1023];
}

__device__ __forceinline__ void scan_add_body(uint64_t* out, const uint64_t* __restrict__ block_sums, int64_t n, int64_t blk) {
    const int64_t i = blk * blockDim.x + threadIdx.x;
    if (i < n) out[i] += block_sums[i / 1024];
}

/* tile bodies of the pulling scheme and the structure */
struct LevelDown {
    using Args = DownArgs;
    static constexpr int THREADS = 256;
    static const char* name() { return "pulling_level_down"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { level_down_body(a, a.G, t); }
};
struct PullLevel {
    using Args = PullArgs;
    static constexpr int THREADS = 256;
    static const char* name() { return "pulling_level"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { pull_level8_body(a, a.G, t); }
};
struct Upseed {
    using Args = UpseedArgs;
    static constexpr int THREADS = 256;
    static const char* name() { return "upseed"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { upseed_body(a, a.G, t); }
};

/* The coarsest levels (at most SMALL_CELLS cells each) in one block: a launch of their own costs each
   of them more than its work.  The same bodies over one block, a barrier between levels (all waves of a
   block run on one CU and share its vector L1, so a barrier makes their writes visible to each other). */
constexpr int64_t SMALL_CELLS = 16384;
constexpr int SMALL_THREADS = 1024;
struct SmallLevels {
    uint8_t* P;                /* particle-cell tree                                   */
    uint8_t* LV;               /* level maps below the top (LevelDown)                 */
    const uint8_t* level_top;  /* map of the top level                                 */
    int lmin, s, top;          /* levels s .. lmin here; s <= top - 1                  */
    int min_type;
    int64_t off[MAXL + 1];
    Dims d[MAXL + 1];
};
struct SmallDown {
    using Args = SmallLevels;
    static constexpr int THREADS = SMALL_THREADS;
    static const char* name() { return "pulling_small_down"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t) {
        for (int l = a.s; l >= a.lmin; --l) {
            const uint8_t* fine = l + 1 == a.top ? a.level_top : a.LV + a.off[l + 1];
            DownArgs d;
            d.fine = fine;
            d.fd = a.d[l + 1];
            d.coarse = a.LV + a.off[l];
            d.cd = a.d[l];
            d.pct = a.P + a.off[l];
            d.level = l;
            d.mode = l == a.lmin ? 1 : 2;
            d.fpct = l + 1 == a.top ? a.P + a.off[a.top] : nullptr;
            d.i32 = 0;
            level_down_body(d, 1, 0);
            __syncthreads();
        }
    }
};
struct SmallPull {
    using Args = SmallLevels;
    static constexpr int THREADS = SMALL_THREADS;
    static const char* name() { return "pulling_small"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t) {
        for (int l = a.s; l >= a.lmin; --l) {
            PullArgs p;
            p.P = a.P + a.off[l];
            p.d = a.d[l];
            p.Pc = a.P + a.off[l + 1];
            p.dc = a.d[l + 1];
            p.has_parent = l > a.lmin;
            p.Pp = p.has_parent ? a.P + a.off[l - 1] : nullptr;
            p.dp = p.has_parent ? a.d[l - 1] : Dims{1, 1, 1};
            p.is_top = 0;
            p.zc = 1;
            p.atomics = 0;
            pull_level8_body(p, 1, 0);
            __syncthreads();
        }
        for (int l = a.lmin + 1; l <= a.s; ++l) {
            UpseedArgs u;
            u.P = a.P + a.off[l];
            u.d = a.d[l];
            u.Pp = a.P + a.off[l - 1];
            u.dp = a.d[l - 1];
            u.min_type = a.min_type;
            u.i32 = 0;
            upseed_body(u, 1, 0);
            __syncthreads();
        }
    }
};
struct RowCount {
    struct Args {
        const uint8_t* maps;
        RowTable t;
        int64_t nrows;
        uint32_t* cnt;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "row_count"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { row_count_body(a.maps, a.t, a.nrows, a.cnt, a.G, t); }
};
template <int LANES>
struct RowFill {
    struct Args {
        const uint8_t* maps;
        RowTable t;
        int64_t nrows;
        const uint64_t* row_off;
        uint16_t* y_vec;
        int64_t G;
        RowImages ri;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return LANES == 64 ? "row_fill" : "row_fill_short"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        row_fill_body<LANES>(a.maps, a.t, a.nrows, a.row_off, a.y_vec, a.ri, a.G, t);
    }
};
struct RowsXz {
    struct Args {
        const uint64_t* row_off;
        const uint32_t* cnt;
        RowTable t;
        uint64_t* xz_end;
        int64_t nrows;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "rows_xz"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { rows_xz_body(a.row_off, a.cnt, a.t, a.xz_end, a.nrows, t); }
};
struct ScanBlocks {
    struct Args {
        const uint32_t* in;
        uint64_t* out;
        uint64_t* block_sums;
        int64_t n;
    };
    static constexpr int THREADS = 1024;
    static const char* name() { return "scan_blocks"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { scan_blocks_body(a.in, a.out, a.block_sums, a.n, t); }
};
struct ScanSums {
    struct Args {
        uint64_t* block_sums;
        int64_t nb;
        uint64_t* total;
    };
    static constexpr int THREADS = 1024;
    static const char* name() { return "scan_sums"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t) { scan_sums_body(a.block_sums, a.nb, a.total); }
};
struct ScanAdd {
    struct Args {
        uint64_t* out;
        const uint64_t* block_sums;
        int64_t n;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "scan_add"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) { scan_add_body(a.out, a.block_sums, a.n, t); }
};

/* mean of the 2x2x2 block in the reference's summation order (PixelData.hpp:952-962), stored
   as the pyramid's element type (u16: truncation like a float -> uint16 assignment) */
template <typename T> __device__ __forceinline__ T pyr_store(float m);
template <> __device__ __forceinline__ uint16_t pyr_store<uint16_t>(float m) { return (uint16_t)(int32_t)m; }
template <> __device__ __forceinline__ float pyr_store<float>(float m) { return m; }

/* a lane takes the coarse cells of 8 bytes of a fine row (2 u16 cells, a float cell) from four fine
   rows (16 bytes of floats: 1024 x 1024 x 20 23 us for the first level, 15 with 8; u16 is alike with both), loaded at any alignment; the sums of a u16 cell are exact in any order, those of a float cell
   run in the order above.  fg, fx: division by the groups of a row and by cd.x (32-bit indices), or
   fits == 0 */
constexpr int PYR_BYTES = 8;
struct PyrDiv {
    FastDiv fg, fx;
    int fits;
};
template <typename T>
__global__ __launch_bounds__(256) void k_pyr_down(const T* __restrict__ fine, Dims fd, T* coarse, Dims cd, PyrDiv dv) {
    constexpr int NF = PYR_BYTES / sizeof(T), NC = NF / 2;
    const int64_t ng = (cd.y + NC - 1) / NC;
    const int64_t total = ng * cd.x * cd.z;
    for (int64_t i = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        int64_t g, x, z;
        if (dv.fits) {
            const uint32_t r = dv.fg.div((uint32_t)i), zz = dv.fx.div(r);
            g = (uint32_t)i - r * (uint32_t)ng;
            x = r - zz * (uint32_t)cd.x;
            z = zz;
        } else {
            const int64_t r = i / ng;
            g = i - r * ng;
            z = r / cd.x;
            x = r - z * cd.x;
        }
        const int64_t x0 = 2 * x, x1 = min(2 * x + 1, fd.x - 1), z0 = 2 * z, z1 = min(2 * z + 1, fd.z - 1), y0 = NF * g;
        const T* rows[4] = {fine + (z0 * fd.x + x0) * fd.y, fine + (z0 * fd.x + x1) * fd.y, fine + (z1 * fd.x + x0) * fd.y,
                            fine + (z1 * fd.x + x1) * fd.y};
        uint32_t w[4][PYR_BYTES / 4];
        if (y0 + NF <= fd.y) {
#pragma unroll
            for (int q = 0; q < 4; ++q) __builtin_memcpy(w[q], rows[q] + y0, PYR_BYTES);
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                T e[NF];
#pragma unroll
                for (int j = 0; j < NF; ++j) e[j] = rows[q][min(y0 + j, fd.y - 1)];
                __builtin_memcpy(w[q], e, PYR_BYTES);
            }
        }
        T o[NC];
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            if constexpr (std::is_same<T, uint16_t>::value) {
                uint32_t s = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) s += (w[q][j] & 0xFFFFu) + (w[q][j] >> 16);
                o[j] = pyr_store<T>((float)s / 8.0f);
            } else {
                float s = __uint_as_float(w[0][2 * j]);
                s = s + __uint_as_float(w[0][2 * j + 1]);
#pragma unroll
                for (int q = 1; q < 4; ++q) {
                    s = s + __uint_as_float(w[q][2 * j]);
                    s = s + __uint_as_float(w[q][2 * j + 1]);
                }
                o[j] = pyr_store<T>(s / 8.0f);
            }
        }
        T* dst = coarse + (z * cd.x + x) * cd.y + NC * g;
        if (NC * g + NC <= cd.y) {
            __builtin_memcpy(dst, o, NC * sizeof(T));
        } else {
#pragma unroll
            for (int j = 0; j < NC - 1; ++j)
                if (NC * g + j < cd.y) dst[j] = o[j];
        }
    }
}

template <typename T>
struct LevelPtrs {
    const T* img[MAXL];
    int64_t y[MAXL], x[MAXL];
    int64_t row_begin[MAXL];
    int64_t nrows[MAXL];
    int64_t rows_prefix[MAXL + 1];
    int n_levels;
};

/* one wave per row; lanes stride the row's particles */
template <typename T>
__global__ __launch_bounds__(256) void k_gather(LevelPtrs<T> L, const uint64_t* __restrict__ xz_end, const uint16_t* __restrict__ y_vec,
                                                T* parts, int64_t total_rows) {
    const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    const int64_t nw = ((int64_t)gridDim.x * blockDim.x) / 64;
    for (int64_t r = wid; r < total_rows; r += nw) {
        int li = 0;
        while (li + 1 < L.n_levels && r >= L.rows_prefix[li + 1]) ++li;
        const int64_t row = r - L.rows_prefix[li];
        const int64_t xzi = L.row_begin[li] + row;
        const uint64_t b = xz_end[xzi - 1], e = xz_end[xzi];
        const int64_t z = row / L.x[li], x = row % L.x[li];
        const T* plane = L.img[li] + (z * L.x[li] + x) * L.y[li];
        /* four independent particles per lane in flight */
        uint64_t i = b + lane;
        for (; i + 192 < e; i += 256) {
            const uint16_t y0 = y_vec[i], y1 = y_vec[i + 64], y2 = y_vec[i + 128], y3 = y_vec[i + 192];
            const T v0 = plane[y0], v1 = plane[y1], v2 = plane[y2], v3 = plane[y3];
            parts[i] = v0;
            parts[i + 64] = v1;
            parts[i + 128] = v2;
            parts[i + 192] = v3;
        }
        for (; i < e; i += 64) parts[i] = plane[y_vec[i]];
    }
}

}  // namespace

void exclusive_scan_u32_async(aprh_context* ctx, const uint32_t* in, uint64_t* out, int64_t n, uint64_t* d_total) {
    if (n <= 0) {
        launch_zero(ctx, d_total, 8);
        return;
    }
    const int64_t nb = cdiv(n, 1024);
    Buf bsum(ctx->pool, (size_t)(nb + 1) * 8);
    launch_tiles<ScanBlocks>(ctx, {in, out, bsum.as<uint64_t>(), n}, nb);
    launch_tiles<ScanSums>(ctx, {bsum.as<uint64_t>(), nb, d_total}, 1);
    launch_tiles<ScanAdd>(ctx, {out, bsum.as<uint64_t>(), n}, cdiv(n, 256));
}

uint64_t exclusive_scan_u32(aprh_context* ctx, const uint32_t* in, uint64_t* out, int64_t n) {
    if (n <= 0) return 0;
    hipStream_t st = ctx->stream;
    uint64_t* d_total = (uint64_t*)ctx->d_flags + 8;
    exclusive_scan_u32_async(ctx, in, out, n, d_total);
    uint64_t total = 0;
    HIP_CHECK(hipMemcpyAsync(&total, d_total, 8, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    return total;
}

template <typename T>
std::vector<int64_t> build_pyramid(aprh_context* ctx, const aprh_apr& a, const T* img, Buf& pyr);
template <typename T>
void pyramid_levels(aprh_context* ctx, const aprh_apr& a, const T* img, T* Pyr, const std::vector<int64_t>& off, int first);

/* layout of the particle-cell tree levels lmin .. lmax-1 in one u8 buffer (8-byte aligned
   levels, so whole-word passes apply): element offsets, off[top + 1] = total */
std::vector<int64_t> pct_layout(const aprh_apr& a) {
    const int top = a.l_max - 1;
    std::vector<int64_t> off(std::max(top + 2, 1), 0);
    for (int l = a.l_min; l <= top; ++l) off[l + 1] = off[l] + (a.y_num[l] * a.x_num[l] * a.z_num[l] + 7) / 8 * 8;
    return off;
}

namespace {
/* the largest level below the top that goes with the small ones (lmin - 1: none) */
int small_level(const aprh_apr& a, const std::vector<int64_t>& zn) {
    int s = a.l_min - 1;
    while (s + 1 <= a.l_max - 2 && a.y_num[s + 1] * a.x_num[s + 1] * zn[s + 1] <= SMALL_CELLS) ++s;
    return s;
}
SmallLevels small_levels(const aprh_apr& a, int s, const std::vector<int64_t>& zn, const std::vector<int64_t>& off, uint8_t* P) {
    SmallLevels v;
    std::memset(&v, 0, sizeof(v));
    v.P = P;
    v.lmin = a.l_min;
    v.s = s;
    v.top = a.l_max - 1;
    if (v.top > MAXL) throw Error(APRH_ERR_UNSUPPORTED, "too many levels");
    for (int l = a.l_min; l <= v.top; ++l) {
        v.off[l] = off[l];
        v.d[l] = Dims{a.y_num[l], a.x_num[l], zn[l]};
    }
    return v;
}
}  // namespace

/* PullingScheme::fill of every level (LocalParticleCellSet.hpp:58-91): the 2x2x2 max pyramid of the level
   map with the seeds of each level, the top level's straight from the map.  zn: z extent per level (the
   APR's, or a patch's).  Levels below the top exist: l_max > 2 */
void seed_levels(aprh_context* ctx, const aprh_apr& a, const uint8_t* level_top, const std::vector<int64_t>& zn, uint8_t* P,
                 const std::vector<int64_t>& off) {
    const int top = a.l_max - 1, lmin = a.l_min;
    auto D = [&](int l) { return Dims{a.y_num[l], a.x_num[l], zn[l]}; };
    Buf lev(ctx->pool, (size_t)std::max<int64_t>(off[top + 1], 8));
    uint8_t* LV = lev.as<uint8_t>();
    const int s = small_level(a, zn);
    const uint8_t* fine = level_top;
    for (int l = top - 1; l > s; --l) {
        const int64_t ng = cdiv(a.y_num[l], 8), n = ng * a.x_num[l] * zn[l];
        DownArgs d{fine, D(l + 1), LV + off[l], D(l), P + off[l], l, l == lmin ? 1 : 2, l + 1 == top ? P + off[top] : nullptr,
                   stride_tiles(n, 256), FastDiv(), FastDiv(), fits32(n) ? 1 : 0};
        if (d.i32) {
            d.fg = FastDiv((uint64_t)ng);
            d.fx = FastDiv((uint64_t)a.x_num[l]);
        }
        launch_tiles<LevelDown>(ctx, d, d.G);
        fine = LV + off[l];
    }
    if (s >= lmin) {
        SmallLevels v = small_levels(a, s, zn, off, P);
        v.LV = LV;
        v.level_top = level_top;
        launch_tiles<SmallDown>(ctx, v, 1);
    }
}

namespace {
/* seeds of one patch's plane range into the global particle-cell tree level:
   global(z + oz) |= SEED where local(z) == SEED, z in [z_lo, z_hi), z + oz < global z extent */
struct SeedMerge {
    struct Args {
        const uint8_t* local;
        uint8_t* global;
        int64_t plane;        /* y * x of the level */
        int64_t z_lo, z_hi, oz, gz;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "seed_merge"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        const int64_t zh = min(a.z_hi, a.gz - a.oz);
        if (zh <= a.z_lo) return;
        const int64_t n = (zh - a.z_lo) * a.plane;
        const uint8_t* src = a.local + a.z_lo * a.plane;
        uint8_t* dst = a.global + (a.z_lo + a.oz) * a.plane;
        for (int64_t i = t * blockDim.x + threadIdx.x; i < n; i += a.G * blockDim.x)
            if (src[i] == SEED) dst[i] = SEED;
    }
};

/* blocked sampling of one level: rows (z + oz, x) for patch planes z in [z_lo, z_hi) take the
   patch pyramid's values at (y, x, z) (ParticleData.hpp:329-362); one wave per row */
template <typename T>
struct GatherPatch {
    struct Args {
        const T* img;                 /* patch pyramid level, (z, x, y) with y fastest */
        int64_t Y, X;
        const uint64_t* xz_end;
        const uint16_t* y_vec;
        int64_t row_begin;            /* xz_end index of the level's row (0, 0) */
        int64_t z_lo, z_hi, oz;
        T* parts;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "gather_patch"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        const int lane = threadIdx.x & 63;
        const int64_t nrows = (a.z_hi - a.z_lo) * a.X;
        const int64_t wpb = blockDim.x / 64;
        for (int64_t r = t * wpb + (threadIdx.x >> 6); r < nrows; r += a.G * wpb) {
            const int64_t z = a.z_lo + r / a.X, x = r % a.X;
            const int64_t rid = a.row_begin + (z + a.oz) * a.X + x;
            const uint64_t b = a.xz_end[rid - 1], e = a.xz_end[rid];
            const T* row = a.img + (z * a.X + x) * a.Y;
            for (uint64_t i = b + lane; i < e; i += 64) {
                const int64_t y = a.y_vec[i];
                if (y < a.Y) a.parts[i] = row[y];
            }
        }
    }
};
}  // namespace

/* z extents per level of a patch of zp planes (the pyramid / particle-cell tree geometry of the
   patch: ceil(zp / 2^(l_max - l))) */
std::vector<int64_t> patch_z_extents(const aprh_apr& a, int64_t zp) {
    std::vector<int64_t> zn(a.l_max + 1, 0);
    for (int l = 0; l <= a.l_max; ++l) zn[l] = cdiv(zp, (int64_t)1 << (a.l_max - l));
    return zn;
}

/* PullingScheme::fill_patch for every level (APRConverterBatch.hpp:287-322,
   PullingScheme.hpp:175-244): the patch's own seeds (its level map and the max pyramid of it),
   merged into the global tree P over the patch's non-ghost planes of each level */
void seed_patch(aprh_context* ctx, const aprh_apr& a, uint8_t* P, const std::vector<int64_t>& off, const uint8_t* level_top_patch,
                int64_t zp, int64_t z0, int64_t gl, int64_t gr) {
    const int top = a.l_max - 1;
    const std::vector<int64_t> zn = patch_z_extents(a, zp);
    std::vector<int64_t> loff(top + 2, 0);
    for (int l = a.l_min; l <= top; ++l) loff[l + 1] = loff[l] + (a.y_num[l] * a.x_num[l] * zn[l] + 7) / 8 * 8;
    Buf local(ctx->pool, (size_t)std::max<int64_t>(loff[top + 1], 8));
    seed_levels(ctx, a, level_top_patch, zn, local.as<uint8_t>(), loff);
    for (int l = a.l_min; l <= top; ++l) {
        const int64_t f = (int64_t)1 << (a.l_max - l);
        const int64_t zl = gl / f, zr = gr / f, oz = z0 / f - zl;
        const int64_t plane = a.y_num[l] * a.x_num[l];
        const int64_t G = stride_tiles(std::max<int64_t>((zn[l] - zl - zr) * plane, 1), 256 * 4);
        launch_tiles<SeedMerge>(ctx, {local.as<uint8_t>() + loff[l], P + off[l], plane, zl, zn[l] - zr, oz, a.z_num[l], G}, G);
    }
}

/* ParticleData::sample_parts_from_img_blocked (ParticleData.hpp:292-362) on a device image:
   per z block the mean pyramid of the patch (ghosts included) and the rows of its non-ghost
   planes of each level; rows past a level's z extent are skipped; particles no block reaches
   stay 0 */
void sample_blocked_u16(aprh_context* ctx, const aprh_apr& a, const uint16_t* img, int64_t z_block_size, int64_t ghost_z,
                        uint16_t* parts) {
    launch_zero(ctx, parts, std::max<uint64_t>(a.total, 1) * 2);
    const int64_t Z = a.org[2], plane = a.org[0] * a.org[1];
    const int64_t nb = std::max<int64_t>(Z / z_block_size, 1);
    for (int64_t bk = 0; bk < nb; ++bk) {
        const int64_t z0 = bk * z_block_size, zf = (bk == nb - 1) ? Z : (bk + 1) * z_block_size;
        const int64_t gl = std::min(z0, ghost_z), gr = std::min(Z - zf, ghost_z);
        const int64_t zp = zf + gr - (z0 - gl);
        const uint16_t* pimg = img + (z0 - gl) * plane;
        aprh_apr pa;
        pa.l_min = a.l_min;
        pa.l_max = a.l_max;
        pa.y_num = a.y_num;
        pa.x_num = a.x_num;
        pa.z_num = patch_z_extents(a, zp);
        int64_t tot = 0;
        const std::vector<int64_t> poff = pyramid_layout(pa, &tot);
        Buf pyr(ctx->pool, (size_t)std::max<int64_t>(tot, 1) * 2);
        if (a.l_max > a.l_min) pyramid_levels<uint16_t>(ctx, pa, pimg, pyr.as<uint16_t>(), poff, a.l_max - 1);
        for (int l = a.l_min; l <= a.l_max; ++l) {
            const int64_t f = (int64_t)1 << (a.l_max - l);
            const int64_t zl = gl / f, zr = gr / f, oz = z0 / f - zl;
            const int64_t zh = std::min(pa.z_num[l] - zr, a.z_num[l] - oz);
            if (zh <= zl) continue;
            const uint16_t* lvimg = (l == a.l_max) ? pimg : pyr.as<uint16_t>() + poff[l];
            const int64_t G = stride_tiles((zh - zl) * a.x_num[l], 4, 16384);
            launch_tiles<GatherPatch<uint16_t>>(ctx, {lvimg, a.y_num[l], a.x_num[l], a.xz_end.as<uint64_t>(), a.y_vec.as<uint16_t>(),
                                                      (int64_t)a.level_xz_vec[l], zl, zh, oz, parts, G},
                                                G);
        }
        HIP_CHECK(hipStreamSynchronize(ctx->stream));
    }
}

void build_structure(aprh_context* ctx, aprh_apr& a, const uint8_t* level_top, const aprh_params& par) {
    build_structure_seeded(ctx, a, level_top, nullptr, par);
}

void build_structure_seeded(aprh_context* ctx, aprh_apr& a, const uint8_t* level_top, uint8_t* seeded, const aprh_params& par) {
    hipStream_t st = ctx->stream;
    const int lmax = a.l_max, lmin = a.l_min;
    if (lmax <= 2) {
        if (ctx->async_mode) throw Error(APRH_ERR_UNSUPPORTED, "batched conversion of volumes with l_max <= 2");
        /* LinearAccess.hpp:229-260: every pixel is a particle at l_max */
        const int64_t yL = a.y_num[lmax], xL = a.x_num[lmax], zL = a.z_num[lmax];
        std::vector<uint64_t> xz(a.n_xz, 0);
        uint64_t c = 0;
        for (int64_t z = 0; z < zL; ++z)
            for (int64_t x = 0; x < xL; ++x) {
                c += (uint64_t)yL;
                xz[a.level_xz_vec[lmax] + z * xL + x] = c;
            }
        /* the reference leaves the lower rows at 0 and skips the partial sum */
        std::vector<uint16_t> yv(c);
        uint64_t k = 0;
        for (int64_t z = 0; z < zL; ++z)
            for (int64_t x = 0; x < xL; ++x)
                for (int64_t y = 0; y < yL; ++y) yv[k++] = (uint16_t)y;
        a.total = c;
        a.xz_end.reset(ctx->pool, a.n_xz * 8);
        a.y_vec.reset(ctx->pool, std::max<uint64_t>(c, 1) * 2);
        HIP_CHECK(hipMemcpyAsync(a.xz_end.ptr(), xz.data(), a.n_xz * 8, hipMemcpyHostToDevice, st));
        HIP_CHECK(hipMemcpyAsync(a.y_vec.ptr(), yv.data(), c * 2, hipMemcpyHostToDevice, st));
        HIP_CHECK(hipStreamSynchronize(st));
        return;
    }
    mark(ctx, ST_PULLING);
    /* particle-cell tree levels lmin .. top (= lmax - 1), one contiguous u8 buffer */
    const int top = lmax - 1;
    const std::vector<int64_t> off = pct_layout(a);
    Buf pct;
    uint8_t* P = seeded;
    auto D = [&](int l) { return Dims{a.y_num[l], a.x_num[l], a.z_num[l]}; };
    if (!P) {
        pct.reset(ctx->pool, (size_t)off[top + 1]);
        P = pct.as<uint8_t>();
        seed_levels(ctx, a, level_top, a.z_num, P, off);
    }
    const int min_type = par.neighborhood_optimization ? 1 : 2;
    const int small = small_level(a, a.z_num);
    /* pulling scheme, top to bottom; the coarsest levels' equivalence optimisation with their own */
    for (int l = top; l > std::max(small, lmin - 1); --l) {
        const bool has_parent = (l - 1) >= lmin;
        const bool is_top = (l == top);
        uint8_t* Pc = is_top ? nullptr : P + off[l + 1];
        uint8_t* Pp = has_parent ? P + off[l - 1] : nullptr;
        auto pargs = [&](int zc) {
            const int64_t G = stride_tiles(cdiv(a.y_num[l], 8) * a.x_num[l] * cdiv(a.z_num[l], zc), 256);
            return PullArgs{P + off[l], D(l), Pc, is_top ? Dims{1, 1, 1} : D(l + 1), Pp, has_parent ? D(l - 1) : Dims{1, 1, 1},
                            is_top ? 1 : 0, has_parent ? 1 : 0, zc, 1, G};
        };
        /* runs of 4 planes load each row half as often as single planes; levels of fewer than about 256
           thousand lanes that way take shorter runs, since a lane walks its planes one after another */
        const int64_t lanes1 = cdiv(a.y_num[l], 8) * a.x_num[l] * a.z_num[l];
        const int zc = lanes1 >= 4 * 262144 ? 4 : lanes1 >= 2 * 262144 ? 2 : 1;
        const PullArgs p = pargs(zc);
        if (ctx->recorder) {
            const PullArgs p4 = pargs(4);
            launch_tiles_alts(ctx, {tile_alt<PullLevel>(p, p.G, "planes per lane by size"), tile_alt<PullLevel>(p4, p4.G, "4 planes per lane")},
                              0);
        } else {
            launch_tiles<PullLevel>(ctx, p, p.G);
        }
    }
    if (small >= lmin) {
        SmallLevels v = small_levels(a, small, a.z_num, off, P);
        v.min_type = min_type;
        launch_tiles<SmallPull>(ctx, v, 1);
    }
    mark(ctx, ST_STRUCTURE);
    /* equivalence optimisation, levels upward in order */
    for (int l = std::max(small, lmin) + 1; l <= top; ++l) {
        const int64_t ng = cdiv(a.y_num[l], 8), n = ng * a.x_num[l] * a.z_num[l];
        UpseedArgs u{P + off[l], D(l), P + off[l - 1], D(l - 1), min_type, stride_tiles(n, 256), FastDiv(), FastDiv(), fits32(n) ? 1 : 0};
        if (u.i32) {
            u.fg = FastDiv((uint64_t)ng);
            u.fx = FastDiv((uint64_t)a.x_num[l]);
        }
        launch_tiles<Upseed>(ctx, u, u.G);
    }
    /* segment table over APR levels lmin..lmax */
    RowTable t;
    std::memset(&t, 0, sizeof(t));
    t.l_min = lmin;
    t.l_max = lmax;
    t.n_levels = lmax - lmin + 1;
    if (t.n_levels > MAXL) throw Error(APRH_ERR_UNSUPPORTED, "too many levels");
    t.min_type = min_type;
    t.y_max = a.y_num[lmax];
    int64_t rp = 0;
    for (int l = lmin; l <= lmax; ++l) {
        const int li = l - lmin;
        const int ml = (l == lmax) ? top : l;   /* pct map providing the cells */
        t.row_begin[li] = (int64_t)a.level_xz_vec[l];
        t.rows_x[li] = a.x_num[l];
        t.map_off[li] = off[ml];
        t.map_y[li] = a.y_num[ml];
        t.map_x[li] = a.x_num[ml];
        t.row_prefix[li] = rp;
        rp += a.x_num[l] * a.z_num[l];
    }
    t.row_prefix[t.n_levels] = rp;
    t.top_z = a.z_num[lmax];
    t.top_pz = a.z_num[top];
    t.n_work = t.row_prefix[t.n_levels - 1] + a.x_num[top] * a.z_num[top];
    /* per-row counts, exclusive scan over rows in particle order, xz_end_vec, y_vec */
    Buf cnt(ctx->pool, (size_t)rp * 4);
    Buf rowoff(ctx->pool, (size_t)rp * 8);
    const int64_t RG = stride_tiles(t.n_work, 16, 16384);   /* 16 lanes per work item, 16 items per block */
    launch_tiles<RowCount>(ctx, {P, t, rp, cnt.as<uint32_t>(), RG}, RG);
    if (ctx->async_mode) {
        /* y_vec and xz_end_vec are preallocated (y_vec for the upper bound P <= N); the count
           stays on the device */
        exclusive_scan_u32_async(ctx, cnt.as<uint32_t>(), rowoff.as<uint64_t>(), rp, ctx->slot_total);
    } else {
        a.total = exclusive_scan_u32(ctx, cnt.as<uint32_t>(), rowoff.as<uint64_t>(), rp);
        a.xz_end.reset(ctx->pool, a.n_xz * 8);
        a.y_vec.reset(ctx->pool, std::max<uint64_t>(a.total, 1) * 2);
    }
    launch_zero(ctx, a.xz_end.ptr(), a.n_xz * 8);
    launch_tiles<RowsXz>(ctx, {rowoff.as<uint64_t>(), cnt.as<uint32_t>(), t, a.xz_end.as<uint64_t>(), rp}, cdiv(rp, 256));
    RowImages ri;
    std::memset(&ri, 0, sizeof(ri));
    SampleReq* sr = ctx->sample_req;
    if (sr && sr->img && !ctx->async_mode && !ctx->recorder && a.total <= sr->capacity) {
        if (sr->top_built) {
            /* level lmax-1 came with the y pass */
            pyramid_levels<uint16_t>(ctx, a, sr->img, sr->pyr.as<uint16_t>(), sr->pyr_off, lmax - 2);
        } else {
            sr->pyr_off = build_pyramid<uint16_t>(ctx, a, sr->img, sr->pyr);
        }
        for (int l = lmin; l <= lmax; ++l) {
            ri.img[l - lmin] = (l == lmax) ? sr->img : sr->pyr.as<uint16_t>() + sr->pyr_off[l];
            ri.y[l - lmin] = a.y_num[l];
        }
        ri.parts = sr->parts;
        sr->done = true;
    }
    /* a wave per work item for long rows, 16 lanes (256 cells at once) for short ones.  Measured with rows of 100 to
       1500 cells in 40 M voxels, 16 / 64 lanes: 320 cells 46 / 49 us, 384 44 / 43, 512 42 / 37; with the sampling, whose
       gathers want more lanes, 200 cells 110 / 127, 256 155 / 136, 384 164 / 109 */
    {
        const int64_t FG16 = stride_tiles(t.n_work, FILL_WAVES * 4, 16384), FG64 = stride_tiles(t.n_work, FILL_WAVES, 16384);
        const typename RowFill<16>::Args f16{P, t, rp, rowoff.as<uint64_t>(), a.y_vec.as<uint16_t>(), FG16, ri};
        const typename RowFill<64>::Args f64{P, t, rp, rowoff.as<uint64_t>(), a.y_vec.as<uint16_t>(), FG64, ri};
        const int prefer = t.map_y[t.n_levels - 1] > (ri.parts ? 14 : 24) * CPL ? 1 : 0;
        if (ctx->recorder)
            launch_tiles_alts(ctx, {tile_alt<RowFill<16>>(f16, FG16, "16 lanes per item"), tile_alt<RowFill<64>>(f64, FG64, "64 lanes per item")},
                              prefer);
        else if (prefer)
            launch_tiles<RowFill<64>>(ctx, f64, FG64);
        else
            launch_tiles<RowFill<16>>(ctx, f16, FG16);
    }
    if (ctx->keep_intermediates) {
        a.pct.clear();
        a.pct_dims.assign(3 * (top + 1), 0);
        a.pct.resize(top + 1);
        for (int l = lmin; l <= top; ++l) {
            const size_t nb2 = (size_t)(a.y_num[l] * a.x_num[l] * a.z_num[l]);
            a.pct[l].reset(ctx->pool, nb2);
            HIP_CHECK(hipMemcpyAsync(a.pct[l].ptr(), P + off[l], nb2, hipMemcpyDeviceToDevice, st));
            a.pct_dims[3 * l] = a.y_num[l];
            a.pct_dims[3 * l + 1] = a.x_num[l];
            a.pct_dims[3 * l + 2] = a.z_num[l];
        }
    }
    if (!ctx->async_mode) HIP_CHECK(hipStreamSynchronize(st));
}

/* layout of the mean pyramid of an image over levels lmin .. lmax-1 (PixelData.hpp:1036-1058):
   one buffer, 16-byte aligned levels; per-level element offsets and the total */
std::vector<int64_t> pyramid_layout(const aprh_apr& a, int64_t* total) {
    std::vector<int64_t> off(a.l_max + 1, 0);
    int64_t tot = 0;
    for (int l = a.l_min; l < a.l_max; ++l) {
        off[l] = tot;
        tot += (a.y_num[l] * a.x_num[l] * a.z_num[l] + 7) / 8 * 8;
    }
    *total = tot;
    return off;
}

/* levels `first` .. lmin of the pyramid, each from the level above (the image above lmax-1) */
template <typename T>
void pyramid_levels(aprh_context* ctx, const aprh_apr& a, const T* img, T* Pyr, const std::vector<int64_t>& off, int first) {
    hipStream_t st = ctx->stream;
    const int lmax = a.l_max, lmin = a.l_min;
    for (int l = first; l >= lmin; --l) {
        const T* fine = (l == lmax - 1) ? img : Pyr + off[l + 1];
        const Dims fd{a.y_num[l + 1], a.x_num[l + 1], a.z_num[l + 1]}, cd{a.y_num[l], a.x_num[l], a.z_num[l]};
        T* coarse = Pyr + off[l];
        const int64_t ng = cdiv(cd.y, PYR_BYTES / 2 / (int64_t)sizeof(T)), work = ng * cd.x * cd.z;
        PyrDiv dv;
        dv.fits = fits32(work) ? 1 : 0;
        if (dv.fits) {
            dv.fg = FastDiv((uint64_t)ng);
            dv.fx = FastDiv((uint64_t)cd.x);
        }
        hipLaunchKernelGGL(k_pyr_down<T>, dim3((unsigned)std::min<int64_t>(cdiv(work, 256), 16384)), dim3(256), 0, st, fine, fd, coarse, cd, dv);
        HIP_LAUNCH_CHECK();
    }
}

template <typename T>
std::vector<int64_t> build_pyramid(aprh_context* ctx, const aprh_apr& a, const T* img, Buf& pyr) {
    int64_t tot = 0;
    std::vector<int64_t> off = pyramid_layout(a, &tot);
    pyr.reset(ctx->pool, (size_t)std::max<int64_t>(tot, 1) * sizeof(T));
    pyramid_levels<T>(ctx, a, img, pyr.as<T>(), off, a.l_max - 1);
    return off;
}

/* pyr_ext: caller-provided pyramid memory of at least sample_pyramid_bytes() (nothing is
   allocated then); nullptr: the pyramid comes from the context's pool */
template <typename T>
void launch_sample(aprh_context* ctx, const aprh_apr& a, const T* img, T* parts, T* pyr_ext) {
    hipStream_t st = ctx->stream;
    const int lmax = a.l_max, lmin = a.l_min;
    Buf pyr;
    std::vector<int64_t> off;
    T* Pyr = pyr_ext;
    if (pyr_ext) {
        int64_t tot = 0;
        off = pyramid_layout(a, &tot);
        pyramid_levels<T>(ctx, a, img, pyr_ext, off, a.l_max - 1);
    } else {
        off = build_pyramid<T>(ctx, a, img, pyr);
        Pyr = pyr.as<T>();
    }
    LevelPtrs<T> L;
    std::memset(&L, 0, sizeof(L));
    L.n_levels = lmax - lmin + 1;
    int64_t rp = 0;
    for (int l = lmin; l <= lmax; ++l) {
        const int li = l - lmin;
        L.img[li] = (l == lmax) ? img : Pyr + off[l];
        L.y[li] = a.y_num[l];
        L.x[li] = a.x_num[l];
        L.row_begin[li] = (int64_t)a.level_xz_vec[l];
        L.nrows[li] = a.x_num[l] * a.z_num[l];
        L.rows_prefix[li] = rp;
        rp += L.nrows[li];
    }
    L.rows_prefix[L.n_levels] = rp;
    if (a.total > 0) {
        hipLaunchKernelGGL(k_gather<T>, dim3(8192), dim3(256), 0, st, L, a.xz_end.as<uint64_t>(), a.y_vec.as<uint16_t>(), parts, rp);
        HIP_LAUNCH_CHECK();
    }
    HIP_CHECK(hipStreamSynchronize(st));
}

void launch_sample_u16(aprh_context* ctx, const aprh_apr& a, const uint16_t* img, uint16_t* parts, uint16_t* pyr_ext) {
    launch_sample<uint16_t>(ctx, a, img, parts, pyr_ext);
}
void launch_sample_f32(aprh_context* ctx, const aprh_apr& a, const float* img, float* parts) { launch_sample<float>(ctx, a, img, parts, nullptr); }

size_t sample_pyramid_bytes(const aprh_apr& a, size_t elem) {
    int64_t tot = 0;
    pyramid_layout(a, &tot);
    return (size_t)tot * elem;
}

}  // namespace aprh
