/*
 * k_particles.hip -- operations on the particles of a device-resident APR:
 * tree (interior cells), fill_tree_mean, piecewise-constant reconstruction,
 * APR convolution and Richardson-Lucy.
 *
 *  - tree (APR::initialize_tree_dense, APR.hpp:633-689): per-level dense u8
 *    maps; one wave per particle row marks the parents of its particles, the
 *    maps are OR-ed upward through the (0,0,0) child, and the linear tree
 *    access is built by row counts + scan + fill.
 *  - fill_tree_mean (APRTreeNumerics.hpp:63-202): tree levels from the top
 *    down; a wave holds the children of one tree row in LDS and each node
 *    accumulates scale*value/8 over its particle children first and its tree
 *    children second, both in (z, x, y) order -- the order in which the
 *    reference's two passes reach every node -- so the sums are bit-equal.
 *  - piecewise-constant images (APRReconstruction::reconstruct_constant,
 *    APRReconstruction.hpp:80-120, :297-394): at level l_max + level_delta,
 *    one wave per image row over the particles of every level above it and,
 *    where finer particles live, the tree means of that level.
 *  - convolution: every particle sums stencil x level image over its reflected
 *    or zero-padded window in the reference's (z, x, y) tap order.
 *  - Richardson-Lucy (APRNumerics.hpp:549-593) with an optional relative-update
 *    stopping rule; the update norms are reduced in a fixed order.
 */
#include <algorithm>
#include <cmath>

#include "aprh_internal.hpp"
#include "tiles.hpp"

namespace aprh {

namespace {

constexpr int MAXL = 24;

/* rows of a linear access (APR or tree) over levels lo..hi */
struct Rows {
    int n_levels, l_lo;
    int64_t prefix[MAXL + 1];     /* first global row id of each level */
    int64_t row_begin[MAXL];      /* index in xz_end of row 0          */
    int64_t x_num[MAXL], y_num[MAXL], z_num[MAXL];
};

Rows make_rows(const std::vector<int64_t>& yn, const std::vector<int64_t>& xn, const std::vector<int64_t>& zn,
               const std::vector<uint64_t>& level_xz, int lo, int hi) {
    Rows r;
    std::memset(&r, 0, sizeof(r));
    r.n_levels = std::max(hi - lo + 1, 0);
    r.l_lo = lo;
    if (r.n_levels > MAXL) throw Error(APRH_ERR_UNSUPPORTED, "too many levels");
    int64_t p = 0;
    for (int l = lo; l <= hi; ++l) {
        const int i = l - lo;
        r.prefix[i] = p;
        r.row_begin[i] = (int64_t)level_xz[l];
        r.x_num[i] = xn[l];
        r.y_num[i] = yn[l];
        r.z_num[i] = zn[l];
        p += xn[l] * zn[l];
    }
    r.prefix[r.n_levels] = p;
    return r;
}

__device__ __forceinline__ int row_level(const Rows& R, int64_t r) {
    int li = 0;
    while (li + 1 < R.n_levels && r >= R.prefix[li + 1]) ++li;
    return li;
}

__device__ __forceinline__ uint16_t f2u16(float v) {
    /* g++/x86-64 float->uint16 conversion: truncation through int32 */
    if (!(v > -2147483648.0f && v < 2147483648.0f)) return 0;
    return (uint16_t)(int32_t)v;
}

template <typename D> struct Cvt;
template <> struct Cvt<float> {
    static __device__ __forceinline__ float from(float v) { return v; }
    static __device__ __forceinline__ float from(uint16_t v) { return (float)v; }
};
template <> struct Cvt<uint16_t> {
    static __device__ __forceinline__ uint16_t from(float v) { return f2u16(v); }
    static __device__ __forceinline__ uint16_t from(uint16_t v) { return v; }
};

/* ---------------- tree build ---------------- */
/* APR particle (level l) marks tree cell (l-1, y/2, x/2, z/2) */
__global__ __launch_bounds__(256) void k_mark_parents(Rows R, const uint64_t* __restrict__ xz_end, const uint16_t* __restrict__ y_vec,
                                                      uint8_t* const* maps, int64_t total_rows) {
    const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    const int64_t nw = ((int64_t)gridDim.x * blockDim.x) / 64;
    for (int64_t r = wid; r < total_rows; r += nw) {
        const int li = row_level(R, r);
        const int level = R.l_lo + li;
        const int64_t row = r - R.prefix[li];
        const int64_t z = row / R.x_num[li], x = row % R.x_num[li];
        const uint64_t b = xz_end[R.row_begin[li] + row - 1], e = xz_end[R.row_begin[li] + row];
        uint8_t* m = maps[level - 1];
        const int64_t pyn = (R.y_num[li] + 1) / 2, pxn = (R.x_num[li] + 1) / 2;
        uint8_t* prow = m + ((z / 2) * pxn + (x / 2)) * pyn;
        for (uint64_t i = b + lane; i < e; i += 64) prow[y_vec[i] / 2] = 1;
    }
}

/* tree[l](y,x,z) |= tree[l+1](2y,2x,2z) */
__global__ void k_or_up(uint8_t* m, int64_t yn, int64_t xn, int64_t zn, const uint8_t* __restrict__ c, int64_t cyn, int64_t cxn) {
    const size_t n = (size_t)(yn * xn * zn);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const int64_t y = (int64_t)(i % (size_t)yn);
        const int64_t r = (int64_t)(i / (size_t)yn);
        const int64_t x = r % xn, z = r / xn;
        m[i] = m[i] | c[((2 * z) * cxn + 2 * x) * cyn + 2 * y];
    }
}

/* per-row count of a 0/1 map row (LinearAccess::initialize_tree_access_dense, LinearAccess.hpp:75-90):
   one wave per row */
__global__ __launch_bounds__(256) void k_map_row_count(Rows R, const uint8_t* const* maps, uint32_t* cnt, int64_t total_rows) {
    const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    const int64_t nw = ((int64_t)gridDim.x * blockDim.x) / 64;
    for (int64_t r = wid; r < total_rows; r += nw) {
        const int li = row_level(R, r);
        const int64_t row = r - R.prefix[li];
        const int64_t yn = R.y_num[li];
        const uint8_t* p = maps[R.l_lo + li] + row * yn;
        uint32_t c = 0;
        for (int64_t y = lane; y < yn; y += 64) c += p[y];
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
        if (lane == 0) cnt[r] = c;
    }
}

__global__ __launch_bounds__(256) void k_map_row_fill(Rows R, const uint8_t* const* maps, const uint64_t* __restrict__ xz_end,
                                                      uint16_t* y_vec, int64_t total_rows) {
    const int64_t wid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    const int64_t nw = ((int64_t)gridDim.x * blockDim.x) / 64;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int64_t r = wid; r < total_rows; r += nw) {
        const int li = row_level(R, r);
        const int64_t row = r - R.prefix[li];
        const int64_t yn = R.y_num[li];
        const uint8_t* p = maps[R.l_lo + li] + row * yn;
        uint64_t o = xz_end[R.row_begin[li] + row - 1];
        for (int64_t y0 = 0; y0 < yn; y0 += 64) {
            const int64_t y = y0 + lane;
            const bool on = y < yn && p[y];
            const uint64_t b = __ballot(on);
            if (on) y_vec[o + __popcll(b & lt)] = (uint16_t)y;
            o += __popcll(b);
        }
    }
}

/* xz_end[row_begin + row] = inclusive scan value of global row r */
__global__ void k_rows_to_xz(Rows R, const uint64_t* __restrict__ excl, const uint32_t* __restrict__ cnt, uint64_t* xz_end,
                             int64_t total_rows) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= total_rows) return;
    const int li = row_level(R, r);
    xz_end[R.row_begin[li] + (r - R.prefix[li])] = excl[r] + cnt[r];
}

/* first index in [b, e) with y_vec >= y */
__device__ __forceinline__ uint64_t row_lower(const uint16_t* __restrict__ yv, uint64_t b, uint64_t e, int64_t y) {
    while (b < e) {
        const uint64_t mid = (b + e) >> 1;
        if ((int64_t)yv[mid] < y) b = mid + 1;
        else e = mid;
    }
    return b;
}

/* ---------------- tree means ---------------- */
/* The tree nodes of one row (zp, xp) of tree level t under child cells [c0, c0 + P): a wave puts the four
   child rows' particles and tree nodes (level t + 1) into LDS by their y, then takes one node per lane.
   The children's order is the reference's: its two passes, particles then tree nodes, each in (z, x, y)
   order.  Bound by the latency of row ends, children, then nodes, and on the largest level by its bytes;
   eight 64-entry loads are in flight.  (Before, a level's children went through a dense scratch image of the
   whole level, a clear, two scatters and a gather: the levels below the finest of a 1024 x 1024 x 256 APR
   took 0.39 ms, now 0.17; of 256 x 256 x 128 87 us, now 58.) */
template <typename T, int P>
struct TreeStage {
    float v[4][P];
    uint8_t t[4][P];
};
struct TreeArgs {
    Rows AR, TR;
    int l_min, t_l_max;
    const uint64_t* xz;
    const uint16_t* yv;
    const void* parts;
    const uint64_t* txz;
    const uint16_t* tyv;
    float* tree;
};
template <typename T, int P>
__device__ __forceinline__ void tree_mean_piece(const TreeArgs& a, int t, int64_t row, int64_t c0, TreeStage<T, P>& st, int lane) {
    const Rows& TR = a.TR;
    const int c = t + 1;   /* child level; APR and tree levels share the level geometry */
    const bool tree_child = c <= a.t_l_max;
    /* the child level's dims: the APR's where it has the level, else the tree's */
    const int ai = c - a.l_min;
    const int64_t cyn = ai >= 0 ? a.AR.y_num[ai] : TR.y_num[c], cxn = ai >= 0 ? a.AR.x_num[ai] : TR.x_num[c],
                  czn = ai >= 0 ? a.AR.z_num[ai] : TR.z_num[c];
    const int64_t pxn = TR.x_num[t], pzn = TR.z_num[t], pyn = TR.y_num[t];
    const int64_t zp = row / pxn, xp = row % pxn;
    const int nz = (int)min((int64_t)2, czn - 2 * zp), nx = (int)min((int64_t)2, cxn - 2 * xp);
    /* lanes 0..3: particle rows (a, b) of the children, 4..7: their tree rows, 8: this row's nodes */
    uint64_t b = 0, e = 0;
    if (lane < 9) {
        const int r = lane & 3, za = r >> 1, xb = r & 1;
        const bool part = lane < 4, node = lane == 8;
        if (node || (za < nz && xb < nx && (part ? ai >= 0 : tree_child))) {
            const int64_t cr = (2 * zp + za) * cxn + (2 * xp + xb);
            const int64_t id = node ? TR.row_begin[t] + row : part ? a.AR.row_begin[ai] + cr : TR.row_begin[c] + cr;
            const uint64_t* xz = part ? a.xz : a.txz;
            b = xz[id - 1];
            e = xz[id];
            if (cyn > P && e > b) {
                const uint16_t* yv = part ? a.yv : a.tyv;
                b = row_lower(yv, b, e, node ? c0 / 2 : c0);
                e = row_lower(yv, b, e, node ? (c0 + P) / 2 : c0 + P);
            }
        }
    }
    const uint64_t nb = ((uint64_t)__builtin_amdgcn_readlane((int)(b >> 32), 8) << 32) | (uint32_t)__builtin_amdgcn_readlane((int)b, 8);
    const int np = __builtin_amdgcn_readlane((int)(e - b), 8);
    if (np == 0) return;
#pragma unroll
    for (int k = 0; k < P / 64; ++k) ((uint32_t*)st.t)[k * 64 + lane] = 0;
    /* batches of 64 children of one list, eight in flight */
    constexpr int U = 8;
    uint64_t todo = __ballot(lane < 8 && e > b), sb = 0;
    int k = 0, items = 0, list = 0;
    for (;;) {
        uint64_t qb[U];
        int qn[U], ql[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k >= items) {
                k = items = 0;
                if (todo) {
                    list = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    sb = ((uint64_t)__builtin_amdgcn_readlane((int)(b >> 32), list) << 32) | (uint32_t)__builtin_amdgcn_readlane((int)b, list);
                    items = __builtin_amdgcn_readlane((int)(e - b), list);
                }
            }
            qb[u] = sb + (uint64_t)k;
            qn[u] = items - k;
            ql[u] = list;
            k += 64;
        }
        if (qn[0] <= 0) break;
        int yy[U];
        float vv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            yy[u] = 0;
            vv[u] = 0.0f;
            if (lane < qn[u]) {
                const uint64_t i = qb[u] + (uint64_t)lane;
                yy[u] = (ql[u] < 4 ? a.yv : a.tyv)[i];
                vv[u] = ql[u] < 4 ? Cvt<float>::from(((const T*)a.parts)[i]) : a.tree[i];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (lane < qn[u]) {
                const int p = yy[u] - (int)c0;
                if (p >= 0 && p < P) {
                    st.v[ql[u] & 3][p] = vv[u];
                    st.t[ql[u] & 3][p] = ql[u] < 4 ? 1 : 2;
                }
            }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   /* the lanes read each other's writes below */
    /* boundary scale factors (APRTreeNumerics.hpp:99-113) */
    float sxz = (float)((((2 * pxn != cxn) && (xp == pxn - 1)) + ((2 * pzn != czn) && (zp == pzn - 1))) * 2);
    if (sxz == 0) sxz = 1;
    const float syxz = (2 * pyn != cyn) ? sxz * 2 : sxz;
    for (int n = lane; n < np; n += 64) {
        const int64_t yp = a.tyv[nb + (uint64_t)n];
        const float s = (yp == pyn - 1) ? syxz : sxz;
        const int ny = (int)min((int64_t)2, cyn - 2 * yp), p = (int)(2 * yp - c0);
        float acc = 0.0f;
        for (int pass = 1; pass <= 2; ++pass)
            for (int za = 0; za < nz; ++za)
                for (int xb = 0; xb < nx; ++xb)
                    for (int cc = 0; cc < ny; ++cc)
                        if (st.t[za * 2 + xb][p + cc] == pass) acc = s * st.v[za * 2 + xb][p + cc] / 8.0f + acc;
        a.tree[nb + (uint64_t)n] = acc;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   /* the next piece rewrites the stage */
}

constexpr int TREE_P = 512, TREE_P_SMALL = 128;   /* child cells per piece */
template <typename T>
__global__ __launch_bounds__(256) void k_tree_mean(TreeArgs a, int t) {
    __shared__ TreeStage<T, TREE_P> st[4];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t rows = a.TR.x_num[t] * a.TR.z_num[t];
    for (int64_t r = xcd_block(blockIdx.x, gridDim.x) * 4 + wv; r < rows; r += (int64_t)gridDim.x * 4)
        tree_mean_piece<T, TREE_P>(a, t, r, (int64_t)blockIdx.y * TREE_P, st[wv], lane);
}
/* the small tree levels t_hi .. 0 in one block, a barrier between levels (its waves share a CU's vector L1,
   so a level's values are visible to the next): separate launches would cost more than their work */
constexpr int TREE_SMALL_THREADS = 1024;
template <typename T>
__global__ __launch_bounds__(TREE_SMALL_THREADS) void k_tree_small(TreeArgs a, int t_hi) {
    __shared__ TreeStage<T, TREE_P_SMALL> st[TREE_SMALL_THREADS / 64];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int t = t_hi; t >= 0; --t) {
        const int64_t rows = a.TR.x_num[t] * a.TR.z_num[t], pieces = (2 * a.TR.y_num[t] + TREE_P_SMALL - 1) / TREE_P_SMALL;
        for (int64_t i = wv; i < rows * pieces; i += TREE_SMALL_THREADS / 64)
            tree_mean_piece<T, TREE_P_SMALL>(a, t, i / pieces, (i % pieces) * TREE_P_SMALL, st[wv], lane);
        __syncthreads();
    }
}

/* ---------------- piecewise-constant images ---------------- */
/* Where the pixels of an image at APR level li (counted from l_min) come from: the particles of levels
   0 .. li, then the tree nodes of li (where finer particles live).  A cell of level s covers 2^(li - s)
   pixels a side. */
struct ReconArgs {
    int l_lo;                  /* l_min                                          */
    int64_t rb[MAXL];          /* index in xz_end of the level's row (0, 0)      */
    int64_t trb[MAXL];         /* index in t_xz_end of the same tree row, or -1: no tree nodes wanted there */
    int64_t xn[MAXL];
    const uint64_t* xz;
    const uint16_t* yv;
    const void* parts;
    const uint64_t* txz;
    const uint16_t* tyv;
    const float* tv;
};
/* the image of one level */
struct ReconImage {
    int li;
    uint32_t X, rows;          /* x_num, rows (z, x)                            */
    int64_t Y;
    void* out;
    uint8_t* lev;              /* level of the covering particle, or nullptr    */
};
/* the images of levels l_min .. in one buffer */
struct LevelImages {
    int n;
    int64_t block0[MAXL], blocks;   /* first block of each level, the finest level first; their number */
    uint32_t X[MAXL], rows[MAXL];
    int G[MAXL];               /* lanes per row                                 */
    int64_t Y[MAXL];
    float* out[MAXL];
};

constexpr int RC_BYTES = 4096;   /* of a row's values in LDS, per wave */

/* n elements staged in LDS to dst in 16-byte words at any alignment, the last ones singly */
template <typename E, int G>
__device__ __forceinline__ void store_staged(E* dst, const E* lds, int n, int lane) {
    constexpr int V = 16 / sizeof(E);
    for (int i = lane * V; i < n; i += G * V) {
        if (i + V <= n) {
            const uint4 w = *(const uint4*)(lds + i);
            __builtin_memcpy(dst + i, &w, 16);
        } else {
            for (int j = i; j < n; ++j) dst[j] = lds[j];
        }
    }
}

/* Pixels [c0, c0 + cn) of row (z, x) of level li's image: the wave finds the row of every level above it
   and writes the levels' values into LDS coarse to fine, so a finer level stands where two overlap; then the
   piece leaves in 16-byte words.  A lane takes four pixels at a time from one load of y and one of values:
   four entries of level li, two of the next, else a quarter, half or all of one (a lane per pixel issued
   four times the instructions, which bound it: the images of 1024 x 1024 x 256 0.77 ms, now 0.50).  search: the row is longer than the piece.
   VALS: values from parts / tree, else the levels themselves; LEV: the levels to ls as bytes.
   HOLES: the structure's particles need not cover the image: a pixel without any is 0 (as is its level), or
   takes the coarser tree nodes that are wanted and reach it.
   G < 64: each G lanes take a row of their own, with its (z, x) and stage; whole rows only (c0 = 0, no search) */
template <typename T, typename D, bool VALS, bool LEV, bool HOLES, int G>
__device__ __forceinline__ void recon_stage(const ReconArgs& a, int li, uint32_t z, uint32_t x, int64_t c0, int cn, bool search, D* st,
                                            uint8_t* ls, int lane) {
    constexpr int LOG = sizeof(D) == 2 ? 11 : 10;
    static_assert(!HOLES || G == 64, "incomplete structures take one row per wave");
    const int sl = G == 64 ? lane : lane & (G - 1);
    if constexpr (HOLES) {
        for (int i = lane; i < RC_BYTES / (int)sizeof(D); i += 64) {
            st[i] = (D)0;
            if (LEV) ls[i] = 0;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    const int tree = a.trb[li] >= 0 ? li + 1 : -1;
    /* lane s: the entries of source s under this row (under the piece), and of the tree nodes of li after them;
       HOLES: lane 2 s those of level s, lane 2 s + 1 those of its tree nodes */
    uint64_t b = 0, e = 0;
    const bool tr = HOLES ? lane & 1 : sl == tree;
    const int s = HOLES ? lane >> 1 : tr ? li : sl, d = li - s;
    if (cn > 0 && s <= li && (!HOLES || !tr || a.trb[s] >= 0)) {
        const int64_t r = (tr ? a.trb[s] : a.rb[s]) + (int64_t)(z >> d) * a.xn[s] + (x >> d);
        const uint64_t* xz = tr ? a.txz : a.xz;
        b = xz[r - 1];
        e = xz[r];
        if (search && e > b) {
            const uint16_t* yv = tr ? a.tyv : a.yv;
            b = row_lower(yv, b, e, c0 >> d);
            e = row_lower(yv, b, e, ((c0 + cn - 1) >> d) + 1);
        }
    }
    const int base = (int)c0;
    uint64_t todo = __ballot(e > b);
    if constexpr (G < 64) {   /* sources that any of the wave's rows has */
#pragma unroll
        for (int o = 32; o >= G; o >>= 1) todo |= todo >> o;
        todo &= ((uint64_t)1 << G) - 1;
    }
    while (todo) {
        const int q = __builtin_ctzll(todo);
        todo &= todo - 1;
        uint64_t sb;
        int cnt;
        if constexpr (G == 64) {
            sb = ((uint64_t)__builtin_amdgcn_readlane((int)(b >> 32), q) << 32) | (uint32_t)__builtin_amdgcn_readlane((int)b, q);
            cnt = __builtin_amdgcn_readlane((int)(e - b), q);
        } else {
            const int from = (lane & ~(G - 1)) | q;
            sb = ((uint64_t)(uint32_t)__shfl((int)(b >> 32), from, 64) << 32) | (uint32_t)__shfl((int)b, from, 64);
            cnt = __shfl((int)(e - b), from, 64);
        }
        const bool tr = HOLES ? q & 1 : q == tree;
        const int s = HOLES ? q >> 1 : tr ? li : q, d = li - s;
        const int lv = a.l_lo + s;
        const uint16_t* yv = (tr ? a.tyv : a.yv) + sb;
        /* entries i .. i + E - 1 */
        auto load = [&](auto& y, auto& v, int i) {
            constexpr int E = sizeof(y) / 2;
            __builtin_memcpy(y, yv + i, 2 * E);
            if (!VALS) {
#pragma unroll
                for (int j = 0; j < E; ++j) v[j] = Cvt<D>::from((uint16_t)lv);
            } else if (tr) {
                float f[E];
                __builtin_memcpy(f, a.tv + sb + i, 4 * E);
#pragma unroll
                for (int j = 0; j < E; ++j) v[j] = Cvt<D>::from(f[j]);
            } else {
                T t[E];
                __builtin_memcpy(t, (const T*)a.parts + sb + i, E * sizeof(T));
#pragma unroll
                for (int j = 0; j < E; ++j) v[j] = Cvt<D>::from(t[j]);
            }
        };
        /* W pixels from p on, a multiple of W */
        auto put = [&](auto w, int p, D v) {
            constexpr int W = decltype(w)::value;
            if (p >= cn) return;
            D q[W];
            uint8_t l[W];
#pragma unroll
            for (int j = 0; j < W; ++j) {
                q[j] = v;
                l[j] = (uint8_t)lv;
            }
            __builtin_memcpy(__builtin_assume_aligned(st + p, W * sizeof(D)), q, sizeof(q));
            if (LEV) __builtin_memcpy(__builtin_assume_aligned(ls + p, W), l, W);
        };
        /* E entries per lane; the last lane's end with the row's last one, so it may repeat some */
        auto entries = [&](auto n, auto w) {
            constexpr int E = decltype(n)::value;
            for (int k = sl * E; k < cnt; k += G * E) {
                uint16_t y[E];
                D v[E];
                load(y, v, min(k, cnt - E));
#pragma unroll
                for (int j = 0; j < E; ++j) put(w, ((int)y[j] << d) - base, v[j]);
            }
        };
        using std::integral_constant;
        if (d == 0) {
            if (cnt >= 4) entries(integral_constant<int, 4>(), integral_constant<int, 1>());
            else entries(integral_constant<int, 1>(), integral_constant<int, 1>());
        } else if (d == 1) {
            if (cnt >= 2) entries(integral_constant<int, 2>(), integral_constant<int, 2>());
            else entries(integral_constant<int, 1>(), integral_constant<int, 2>());
        } else {
            /* four pixels per lane; a cell that starts before the piece (wider than it) fills it from 0 */
            const int m = min(d, LOG) - 2;
            for (int k = sl; k < cnt << m; k += G) {
                uint16_t y[1];
                D v[1];
                load(y, v, k >> m);
                put(integral_constant<int, 4>(), max(((int)y[0] << d) - base, 0) + ((k & ((1 << m) - 1)) << 2), v[0]);
            }
        }
    }
    /* the wave's own LDS writes are in order; the compiler must not move the reads up */
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
/* the same, and the piece to dst (its levels to ldst) */
template <typename T, typename D, bool VALS, bool LEV, bool HOLES, int G>
__device__ __forceinline__ void recon_piece(const ReconArgs& a, int li, uint32_t z, uint32_t x, int64_t c0, int cn, bool search, D* st,
                                            uint8_t* ls, D* dst, uint8_t* ldst, int lane) {
    recon_stage<T, D, VALS, LEV, HOLES, G>(a, li, z, x, c0, cn, search, st, ls, lane);
    store_staged<D, G>(dst, st, cn, lane & (G - 1));
    if (LEV) store_staged<uint8_t, G>(ldst, ls, cn, lane & (G - 1));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   /* the next piece rewrites the stage */
}

/* The image of one level in one pass: a wave per row (blockIdx.y: 4096 bytes of it).  Bound by memory:
   particles and y are read once at the finest level and from L2 by the 4^d rows below a coarser one, and
   the image is written once.  (Before, a level's image was the coarser one upsampled, then its particles
   scattered over it: three passes over the finest level, 1.12 ms for 1000 x 1023 x 255 u16 against
   0.29 ms, 4.6 TB/s.) */
template <typename T, typename D, bool VALS, bool LEV, bool HOLES, int G>
__global__ __launch_bounds__(256) void k_recon(ReconArgs a, ReconImage im) {
    constexpr int CHUNK = RC_BYTES / (int)sizeof(D), R = 64 / G;
    __shared__ __align__(16) D stage[4][CHUNK];
    __shared__ __align__(16) uint8_t lstage[4][LEV ? CHUNK : 16];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c0 = (int64_t)blockIdx.y * CHUNK;
    const int cn = (int)min((int64_t)CHUNK, im.Y - c0);
    for (int64_t row0 = (xcd_block(blockIdx.x, gridDim.x) * 4 + wv) * R; row0 < (int64_t)im.rows; row0 += (int64_t)gridDim.x * 4 * R) {
        const int sub = G == 64 ? 0 : lane / G;
        const bool on = row0 + sub < (int64_t)im.rows;
        const uint32_t row = (uint32_t)row0 + (on ? sub : 0), z = row / im.X, x = row - z * im.X;
        const int64_t o = (int64_t)row * im.Y + c0;
        recon_piece<T, D, VALS, LEV, HOLES, G>(a, im.li, z, x, c0, on ? cn : 0, G == 64 && gridDim.y > 1, stage[wv] + sub * (CHUNK / R),
                                               lstage[wv] + (LEV ? sub * (CHUNK / R) : 0), (D*)im.out + o, LEV ? im.lev + o : nullptr, lane);
    }
}

/* *holes when a pixel of the image has no particle */
__global__ __launch_bounds__(256) void k_holes(ReconArgs a, ReconImage im, int* holes) {
    constexpr int CHUNK = RC_BYTES / 2;
    __shared__ __align__(16) uint16_t stage[4][CHUNK];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c0 = (int64_t)blockIdx.y * CHUNK;
    const int cn = (int)min((int64_t)CHUNK, im.Y - c0);
    bool found = false;
    for (int64_t rowl = xcd_block(blockIdx.x, gridDim.x) * 4 + wv; rowl < (int64_t)im.rows; rowl += (int64_t)gridDim.x * 4) {
        const uint32_t row = (uint32_t)rowl, z = row / im.X, x = row - z * im.X;
        recon_stage<uint16_t, uint16_t, false, false, true, 64>(a, im.li, z, x, c0, cn, gridDim.y > 1, stage[wv], nullptr, lane);
        for (int i = lane; i < cn; i += 64) found = found || stage[wv][i] == 0;   /* levels start at 1 */
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (found) atomicOr(holes, 1);
}

/* the float images of several levels in one launch: none of them needs another, and together they fill the
   chip where the coarse ones alone would each cost a launch */
template <typename T, bool HOLES, bool SHORT>
__global__ __launch_bounds__(256) void k_level_images(ReconArgs a, LevelImages m) {
    constexpr int CHUNK = RC_BYTES / 4;
    __shared__ __align__(16) float stage[4][CHUNK];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c0 = (int64_t)blockIdx.y * CHUNK;
    for (int64_t v = blockIdx.x; v < m.blocks; v += gridDim.x) {
        int li = m.n - 1;
        while (li > 0 && v >= m.block0[li - 1]) --li;
        /* each level is dealt out over the XCDs by itself: the rows of a coarse one cost little */
        const int G = SHORT ? m.G[li] : 64, per = 256 / G;
        const int64_t row0 = xcd_block(v - m.block0[li], ((int64_t)m.rows[li] + per - 1) / per) * per + wv * (64 / G);
        if (c0 >= m.Y[li] || row0 >= m.rows[li]) continue;
        const int cn = (int)min((int64_t)CHUNK, m.Y[li] - c0);
        auto rows = [&](auto g) {
            constexpr int GG = decltype(g)::value, R = 64 / GG;
            const int sub = GG == 64 ? 0 : lane / GG;
            const bool on = row0 + sub < (int64_t)m.rows[li];
            const uint32_t row = (uint32_t)row0 + (on ? sub : 0), X = m.X[li], z = row / X, x = row - z * X;
            recon_piece<T, float, true, false, HOLES, GG>(a, li, z, x, c0, on ? cn : 0, GG == 64 && m.Y[li] > CHUNK, stage[wv] + sub * (CHUNK / R),
                                                          nullptr, m.out[li] + (int64_t)row * m.Y[li] + c0, nullptr, lane);
        };
        if constexpr (!SHORT) {
            rows(std::integral_constant<int, 64>());
        } else {
            if (G == 64) rows(std::integral_constant<int, 64>());
            else if (G == 32) rows(std::integral_constant<int, 32>());
            else rows(std::integral_constant<int, 16>());
        }
    }
}

__global__ void k_fill_f32(float* p, size_t n, float v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

/* a stored structure is well formed: rows non-decreasing within [0, total], y strictly
   increasing inside a row and below the level's y_num */
__global__ void k_validate_rows(Rows R, const uint64_t* __restrict__ xz_end, const uint16_t* __restrict__ y_vec, int64_t total_rows,
                                uint64_t total, int* err) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= total_rows) return;
    const int li = row_level(R, r);
    const int64_t row = r - R.prefix[li];
    const uint64_t b = xz_end[R.row_begin[li] + row - 1], e = xz_end[R.row_begin[li] + row];
    if (e < b || e > total) {
        atomicAdd(err, 1);
        return;
    }
    int bad = 0;
    for (uint64_t i = b; i < e; ++i) {
        if ((int64_t)y_vec[i] >= R.y_num[li]) bad = 1;
        if (i > b && y_vec[i] <= y_vec[i - 1]) bad = 1;
    }
    if (bad) atomicAdd(err, 1);
}

const dim3 kGrid(4096), kBlock(256);

}  // namespace

/* ======================================================================== */

namespace {
/* sources of the images of levels l_min .. hi; tree nodes of level `tree` only, or of all levels below l_max */
ReconArgs recon_sources(const aprh_apr& a, int hi, int tree = -1) {
    ReconArgs r;
    std::memset(&r, 0, sizeof(r));
    r.l_lo = a.l_min;
    if (hi - a.l_min >= MAXL) throw Error(APRH_ERR_UNSUPPORTED, "too many levels");
    for (int l = a.l_min; l <= hi; ++l) {
        const int i = l - a.l_min;
        r.rb[i] = (int64_t)a.level_xz_vec[l];
        r.xn[i] = a.x_num[l];
        r.trb[i] = l < a.l_max && l <= a.t_l_max && a.t_total > 0 && (tree < 0 || l == tree) ? (int64_t)a.t_level_xz[l] : -1;
    }
    r.xz = a.xz_end.as<uint64_t>();
    r.yv = a.y_vec.as<uint16_t>();
    r.txz = a.t_xz_end.as<uint64_t>();
    r.tyv = a.t_y_vec.as<uint16_t>();
    return r;
}
ReconImage recon_image(const aprh_apr& a, int level, void* out, uint8_t* lev) {
    /* dims are at most 65535, so a level has fewer than 2^32 rows */
    return {level - a.l_min, (uint32_t)a.x_num[level], (uint32_t)(a.x_num[level] * a.z_num[level]), a.y_num[level], out, lev};
}
}  // namespace

void validate_structure(aprh_context* ctx, aprh_apr& a) {
    hipStream_t st = ctx->stream;
    Rows R = make_rows(a.y_num, a.x_num, a.z_num, a.level_xz_vec, a.l_min, a.l_max);
    const int64_t nrows = R.prefix[R.n_levels];
    Buf err(ctx->pool, 4);
    HIP_CHECK(hipMemsetAsync(err.ptr(), 0, 4, st));
    if (nrows > 0) {
        hipLaunchKernelGGL(k_validate_rows, dim3((unsigned)cdiv(nrows, 256)), kBlock, 0, st, R, a.xz_end.as<uint64_t>(),
                           a.y_vec.as<uint16_t>(), nrows, a.total, err.as<int>());
        HIP_LAUNCH_CHECK();
    }
    int h_err = 0;
    uint64_t first = 0, last = 0;
    HIP_CHECK(hipMemcpyAsync(&h_err, err.ptr(), 4, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipMemcpyAsync(&first, a.xz_end.ptr(), 8, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipMemcpyAsync(&last, a.xz_end.as<uint64_t>() + a.n_xz - 1, 8, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    if (h_err || first != 0 || last != a.total)
        throw Error(APRH_ERR_INVALID_ARGUMENT, "malformed APR structure (xz_end_vec / y_vec do not describe the given dimensions)");
    /* the particles of a stored structure need not cover the image */
    const ReconImage im = recon_image(a, a.l_max, nullptr, nullptr);
    HIP_CHECK(hipMemsetAsync(err.ptr(), 0, 4, st));
    hipLaunchKernelGGL(k_holes, dim3((unsigned)std::min<int64_t>(cdiv(im.rows, 4), 1 << 20), (unsigned)cdiv(im.Y, RC_BYTES / 2)), kBlock, 0, st,
                       recon_sources(a, a.l_max), im, err.as<int>());
    HIP_LAUNCH_CHECK();
    HIP_CHECK(hipMemcpyAsync(&h_err, err.ptr(), 4, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    a.complete = h_err == 0;
}

void ensure_tree(aprh_context* ctx, aprh_apr& a) {
    if (a.tree_built) return;
    hipStream_t st = ctx->stream;
    /* tree geometry (GenInfo::init_tree, GenInfo.hpp:68-99) */
    const int64_t y = a.org[0], x = a.org[1], z = a.org[2];
    const int64_t md = std::max(std::max(y, x), z);
    const int lm = (int)std::ceil(std::log2((double)md));
    a.t_l_max = std::max(lm - 1, 0);
    if (a.t_l_max + 1 > a.l_max) throw Error(APRH_ERR_UNSUPPORTED, "tree of a degenerate APR");
    a.t_y.assign(a.t_l_max + 1, 0);
    a.t_x.assign(a.t_l_max + 1, 0);
    a.t_z.assign(a.t_l_max + 1, 0);
    for (int l = 0; l <= a.t_l_max; ++l) {
        const double cs = std::round(std::pow(2.0, (double)(a.t_l_max - l + 1)));
        a.t_y[l] = (int64_t)std::ceil((double)y / cs);
        a.t_x[l] = (int64_t)std::ceil((double)x / cs);
        a.t_z[l] = (int64_t)std::ceil((double)z / cs);
    }
    a.t_level_xz.assign(a.t_l_max + 2, 0);
    uint64_t ct = 1;
    a.t_level_xz[0] = 1;
    for (int i = 0; i <= a.t_l_max; ++i) {
        ct += (uint64_t)(a.t_x[i] * a.t_z[i]);
        a.t_level_xz[i + 1] = ct;
    }
    a.t_n_xz = ct;
    /* dense maps, one byte per tree cell */
    std::vector<int64_t> off(a.t_l_max + 2, 0);
    for (int l = 0; l <= a.t_l_max; ++l) off[l + 1] = off[l] + a.t_y[l] * a.t_x[l] * a.t_z[l];
    Buf maps(ctx->pool, (size_t)std::max<int64_t>(off[a.t_l_max + 1], 1));
    HIP_CHECK(hipMemsetAsync(maps.ptr(), 0, (size_t)off[a.t_l_max + 1], st));
    std::vector<uint8_t*> mp(MAXL, nullptr);
    for (int l = 0; l <= a.t_l_max; ++l) mp[l] = maps.as<uint8_t>() + off[l];
    Buf d_mp(ctx->pool, MAXL * sizeof(uint8_t*));
    HIP_CHECK(hipMemcpyAsync(d_mp.ptr(), mp.data(), MAXL * sizeof(uint8_t*), hipMemcpyHostToDevice, st));
    if (a.total > 0) {
        Rows R = make_rows(a.y_num, a.x_num, a.z_num, a.level_xz_vec, a.l_min, a.l_max);
        hipLaunchKernelGGL(k_mark_parents, dim3(8192), kBlock, 0, st, R, a.xz_end.as<uint64_t>(), a.y_vec.as<uint16_t>(),
                           (uint8_t* const*)d_mp.ptr(), R.prefix[R.n_levels]);
        HIP_LAUNCH_CHECK();
    }
    for (int l = a.t_l_max - 1; l >= 0; --l) {
        hipLaunchKernelGGL(k_or_up, kGrid, kBlock, 0, st, mp[l], a.t_y[l], a.t_x[l], a.t_z[l], mp[l + 1], a.t_y[l + 1], a.t_x[l + 1]);
        HIP_LAUNCH_CHECK();
    }
    /* linear access of the tree */
    Rows TR = make_rows(a.t_y, a.t_x, a.t_z, a.t_level_xz, 0, a.t_l_max);
    const int64_t nrows = TR.prefix[TR.n_levels];
    Buf cnt(ctx->pool, (size_t)std::max<int64_t>(nrows, 1) * 4);
    Buf excl(ctx->pool, (size_t)std::max<int64_t>(nrows, 1) * 8);
    a.t_xz_end.reset(ctx->pool, a.t_n_xz * 8);
    HIP_CHECK(hipMemsetAsync(a.t_xz_end.ptr(), 0, a.t_n_xz * 8, st));
    uint64_t total = 0;
    if (nrows > 0) {
        hipLaunchKernelGGL(k_map_row_count, dim3((unsigned)std::min<int64_t>(cdiv(nrows, 4), 16384)), kBlock, 0, st, TR,
                           (const uint8_t* const*)d_mp.ptr(), cnt.as<uint32_t>(), nrows);
        HIP_LAUNCH_CHECK();
        total = exclusive_scan_u32(ctx, cnt.as<uint32_t>(), excl.as<uint64_t>(), nrows);
        hipLaunchKernelGGL(k_rows_to_xz, dim3((unsigned)cdiv(nrows, 256)), kBlock, 0, st, TR, excl.as<uint64_t>(), cnt.as<uint32_t>(),
                           a.t_xz_end.as<uint64_t>(), nrows);
        HIP_LAUNCH_CHECK();
    }
    a.t_total = total;
    a.t_y_vec.reset(ctx->pool, std::max<uint64_t>(total, 1) * 2);
    if (nrows > 0 && total > 0) {
        hipLaunchKernelGGL(k_map_row_fill, dim3((unsigned)std::min<int64_t>(cdiv(nrows, 4), 16384)), kBlock, 0, st, TR,
                           (const uint8_t* const*)d_mp.ptr(), a.t_xz_end.as<uint64_t>(), a.t_y_vec.as<uint16_t>(), nrows);
        HIP_LAUNCH_CHECK();
    }
    HIP_CHECK(hipStreamSynchronize(st));
    a.tree_built = true;
}

template <typename T>
void tree_mean(aprh_context* ctx, aprh_apr& a, const T* parts, float* tree) {
    ensure_tree(ctx, a);
    hipStream_t st = ctx->stream;
    if (a.t_total == 0) return;
    Rows AR = make_rows(a.y_num, a.x_num, a.z_num, a.level_xz_vec, a.l_min, a.l_max);
    Rows TR = make_rows(a.t_y, a.t_x, a.t_z, a.t_level_xz, 0, a.t_l_max);
    /* the top tree level straight from the particle rows of l_max when they have the regular
       shape; the levels below from the rows of their children */
    const bool top = tree_mean_top<T>(ctx, a, parts, tree);
    const int t_first = top ? a.t_l_max - 1 : a.t_l_max;
    if (t_first < 0) return;
    TreeArgs ta;
    ta.AR = AR;
    ta.TR = TR;
    ta.l_min = a.l_min;
    ta.t_l_max = a.t_l_max;
    ta.xz = a.xz_end.as<uint64_t>();
    ta.yv = a.y_vec.as<uint16_t>();
    ta.parts = parts;
    ta.txz = a.t_xz_end.as<uint64_t>();
    ta.tyv = a.t_y_vec.as<uint16_t>();
    ta.tree = tree;
    /* tree levels of at most 16 rows, a row per wave of one block, go to one launch */
    int t_small = t_first;
    while (t_small >= 0 && a.t_x[t_small] * a.t_z[t_small] > TREE_SMALL_THREADS / 64) --t_small;
    for (int t = t_first; t > t_small; --t) {
        const int64_t rows = a.t_x[t] * a.t_z[t];
        hipLaunchKernelGGL(k_tree_mean<T>, dim3((unsigned)std::min<int64_t>(cdiv(rows, 4), 1 << 20), (unsigned)cdiv(2 * a.t_y[t], TREE_P)), kBlock, 0,
                           st, ta, t);
        HIP_LAUNCH_CHECK();
    }
    if (t_small >= 0) {
        hipLaunchKernelGGL(k_tree_small<T>, dim3(1), dim3(TREE_SMALL_THREADS), 0, st, ta, t_small);
        HIP_LAUNCH_CHECK();
    }
}

std::vector<HostStencil> downsampled_stencils(const HostStencil& in, int nlevels, bool normalize) {
    /* APRStencil::downsample_stencil (APRStencil.hpp:12-78): per output tap the area-overlap
       weighted sum over input taps, visited in (z, x, y) input order */
    std::vector<HostStencil> out((size_t)std::max(nlevels, 1));
    out[0] = in;
    if (normalize) {
        /* PixelData::normalize (PixelData.hpp:771-781) */
        float sum = 0;
        for (float v : out[0].w) sum += v;
        for (auto& v : out[0].w) v /= sum;
    }
    const int nd = (in.sz > 1) + (in.sx > 1) + (in.sy > 1);
    for (int d = 1; d < nlevels; ++d) {
        const int step = (int)std::pow(2.0f, (float)d);
        const int factor = (int)std::pow((float)step, (float)nd);
        auto ds = [&](int n) { return n > 1 ? std::max(2 * (((n - 1) / 2 + step - 1) / step) + 1, 3) : 1; };
        HostStencil& o = out[(size_t)d];
        o.sy = ds(in.sy);
        o.sx = ds(in.sx);
        o.sz = ds(in.sz);
        o.w.assign((size_t)o.sy * o.sx * o.sz, 0.0f);
        const int oz = (o.sz / 2) * step - in.sz / 2, ox = (o.sx / 2) * step - in.sx / 2, oy = (o.sy / 2) * step - in.sy / 2;
        auto overlap = [&](int dcell, int off_i) {
            return (float)std::max(std::min(dcell * step + step, off_i + step) - std::max(dcell * step, off_i), 0);
        };
        for (int dz = 0; dz < o.sz; ++dz)
            for (int dx = 0; dx < o.sx; ++dx)
                for (int dy = 0; dy < o.sy; ++dy) {
                    float acc = 0.0f;
                    for (int iz = 0; iz < in.sz; ++iz) {
                        const float wz = overlap(dz, oz + iz);
                        for (int ix = 0; ix < in.sx; ++ix) {
                            const float wx = overlap(dx, ox + ix);
                            for (int iy = 0; iy < in.sy; ++iy) {
                                const float wy = overlap(dy, oy + iy);
                                acc += (wx * wy * wz) * in.w[((size_t)iz * in.sx + ix) * in.sy + iy];
                            }
                        }
                    }
                    o.w[((size_t)dz * o.sx + dx) * o.sy + dy] = acc;
                }
        float sum = 0;
        for (auto& v : o.w) {
            v /= (float)factor;
            sum += v;
        }
        if (normalize) {
            const float nf = 1.0f / sum;
            for (auto& v : o.w) v *= nf;
        }
    }
    return out;
}

/* 1-D factors (fy, fx, fz) with fz (x) fx (x) fy == w to within 1e-6 of max|w|, if they exist */
bool rank1_factors(const HostStencil& s, std::vector<float>& fy, std::vector<float>& fx, std::vector<float>& fz) {
    size_t c = 0;
    double mx = 0;
    for (size_t i = 0; i < s.w.size(); ++i)
        if (std::fabs((double)s.w[i]) > mx) {
            mx = std::fabs((double)s.w[i]);
            c = i;
        }
    if (mx == 0) return false;
    const int cy = (int)(c % s.sy), cx = (int)((c / s.sy) % s.sx), cz = (int)(c / ((size_t)s.sy * s.sx));
    auto W = [&](int z, int x, int y) { return (double)s.w[((size_t)z * s.sx + x) * s.sy + y]; };
    const double wc = W(cz, cx, cy);
    std::vector<double> dy(s.sy), dx(s.sx), dz(s.sz);
    for (int y = 0; y < s.sy; ++y) dy[y] = W(cz, cx, y) / wc;
    for (int x = 0; x < s.sx; ++x) dx[x] = W(cz, x, cy) / wc;
    for (int z = 0; z < s.sz; ++z) dz[z] = W(z, cx, cy);
    for (int z = 0; z < s.sz; ++z)
        for (int x = 0; x < s.sx; ++x)
            for (int y = 0; y < s.sy; ++y)
                if (std::fabs(dz[z] * dx[x] * dy[y] - W(z, x, y)) > 1e-6 * mx) return false;
    fy.assign(dy.begin(), dy.end());
    fx.assign(dx.begin(), dx.end());
    fz.assign(dz.begin(), dz.end());
    return true;
}

template <typename T>
void convolve(aprh_context* ctx, aprh_apr& a, const std::vector<HostStencil>& stencils, const T* in, float* out, bool reflect,
              const float* tree_in) {
    if (stencils.empty()) throw Error(APRH_ERR_INVALID_ARGUMENT, "no stencils");
    if (a.total == 0) return;
    ensure_tree(ctx, a);
    Buf tree_buf;
    const float* tree_vals = tree_in;
    if (!tree_vals) {
        /* APRFilter.hpp:1088: tree means of the input */
        tree_buf.reset(ctx->pool, std::max<uint64_t>(a.t_total, 1) * 4);
        tree_mean(ctx, a, in, tree_buf.as<float>());
        tree_vals = tree_buf.as<float>();
    }
    conv_levels<T>(ctx, a, stencils, ctx->conv_mode == APRH_CONV_SEPARABLE, in, tree_vals, out, reflect, 0, nullptr, false, nullptr,
                   nullptr);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

namespace {
/* lanes per row of an image at `level`: what a short row's entries fill, four a lane, if they hold its sources
   (a wave's time is its chain of loads, however few lanes have one: 30 x 1000 x 1000 u16 0.43 ms with a wave per
   row, 0.12 with 16 lanes; 128 x 600 x 600 0.18, 0.09 with 32; rows of 160 take one pass of a wave either way) */
int recon_lanes(const aprh_apr& a, int level, int64_t y) {
    const int sources = level - a.l_min + 2;
    if (!a.complete) return 64;
    if (y <= 64 && sources <= 16) return 16;
    return y <= 128 && sources <= 32 ? 32 : 64;
}

template <typename T, typename D, bool VALS, bool LEV>
void launch_recon(aprh_context* ctx, const aprh_apr& a, const ReconArgs& r, const ReconImage& im) {
    if (im.rows == 0 || im.Y == 0) return;
    const int G = recon_lanes(a, im.li + a.l_min, im.Y);
    const dim3 grid((unsigned)std::min<int64_t>(cdiv(im.rows, 256 / G), 1 << 20), (unsigned)cdiv(im.Y, RC_BYTES / (int64_t)sizeof(D)));
    if (!a.complete) hipLaunchKernelGGL((k_recon<T, D, VALS, LEV, true, 64>), grid, kBlock, 0, ctx->stream, r, im);
    else if (G == 64) hipLaunchKernelGGL((k_recon<T, D, VALS, LEV, false, 64>), grid, kBlock, 0, ctx->stream, r, im);
    else if (G == 32) hipLaunchKernelGGL((k_recon<T, D, VALS, LEV, false, 32>), grid, kBlock, 0, ctx->stream, r, im);
    else hipLaunchKernelGGL((k_recon<T, D, VALS, LEV, false, 16>), grid, kBlock, 0, ctx->stream, r, im);
    HIP_LAUNCH_CHECK();
}

/* lev (optional): also the level of the particle covering each pixel, as bytes */
template <typename T, typename U>
void reconstruct(aprh_context* ctx, aprh_apr& a, const T* parts, int level, U* img, uint8_t* lev) {
    if (level < a.l_min || level > a.l_max) throw Error(APRH_ERR_INVALID_ARGUMENT, "reconstruction level out of range");
    Buf tree;
    if (level < a.l_max) {
        ensure_tree(ctx, a);
        tree.reset(ctx->pool, std::max<uint64_t>(a.t_total, 1) * 4);
        tree_mean(ctx, a, parts, tree.as<float>());
    }
    ReconArgs r = recon_sources(a, level, level);
    r.parts = parts;
    r.tv = tree.as<float>();
    const ReconImage im = recon_image(a, level, img, lev);
    if (lev) launch_recon<T, U, true, true>(ctx, a, r, im);
    else launch_recon<T, U, true, false>(ctx, a, r, im);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}
}  // namespace

template <typename T>
void level_images(aprh_context* ctx, const aprh_apr& a, const T* parts, const float* tree, const std::vector<float*>& out) {
    ReconArgs r = recon_sources(a, a.l_max);
    r.parts = parts;
    r.tv = tree;
    LevelImages m;
    std::memset(&m, 0, sizeof(m));
    int64_t ymax = 1;
    for (int l = a.l_min; l <= a.l_max; ++l) {
        const int i = m.n++;
        m.X[i] = (uint32_t)a.x_num[l];
        m.Y[i] = a.y_num[l];
        m.out[i] = out[(size_t)l];
        m.rows[i] = (uint32_t)(a.x_num[l] * a.z_num[l]);   /* dims are at most 65535 */
        ymax = std::max(ymax, a.y_num[l]);
    }
    /* with the short rows' forms in it the kernel runs 5 % slower over long ones (1024 x 1024 x 256: 0.56, 0.59 ms) */
    const bool shrt = recon_lanes(a, a.l_max, a.y_num[a.l_max]) < 64;
    for (int i = m.n - 1; i >= 0; --i) {
        m.G[i] = shrt ? recon_lanes(a, i + a.l_min, a.y_num[i + a.l_min]) : 64;
        m.block0[i] = m.blocks;
        m.blocks += cdiv(m.rows[i], 256 / m.G[i]);
    }
    const dim3 grid((unsigned)std::min<int64_t>(m.blocks, 1 << 20), (unsigned)cdiv(ymax, RC_BYTES / 4));
    if (!a.complete) hipLaunchKernelGGL((k_level_images<T, true, false>), grid, kBlock, 0, ctx->stream, r, m);
    else if (shrt) hipLaunchKernelGGL((k_level_images<T, false, true>), grid, kBlock, 0, ctx->stream, r, m);
    else hipLaunchKernelGGL((k_level_images<T, false, false>), grid, kBlock, 0, ctx->stream, r, m);
    HIP_LAUNCH_CHECK();
}
template void level_images<uint16_t>(aprh_context*, const aprh_apr&, const uint16_t*, const float*, const std::vector<float*>&);
template void level_images<float>(aprh_context*, const aprh_apr&, const float*, const float*, const std::vector<float*>&);

/* APRReconstruction::reconstruct_level (APRReconstruction.hpp:131-171): every pixel takes the
   level of the particle covering it.  At a coarser level L (the patch form, :397-490) a pixel
   covered by finer particles takes L from the tree. */
void reconstruct_level(aprh_context* ctx, aprh_apr& a, int level, void* img, int idt) {
    if (level < a.l_min || level > a.l_max) throw Error(APRH_ERR_INVALID_ARGUMENT, "reconstruction level out of range");
    if (level < a.l_max) ensure_tree(ctx, a);
    const ReconArgs r = recon_sources(a, level, level);
    const ReconImage im = recon_image(a, level, img, nullptr);
    if (idt == APRH_DTYPE_U16) launch_recon<uint16_t, uint16_t, false, false>(ctx, a, r, im);
    else launch_recon<uint16_t, float, false, false>(ctx, a, r, im);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

namespace {
/* the patch out of a level image: out[z, x, y] = full[(z + zb) >> s, (x + xb) >> s, (y + yb) >> s]
   (s > 0: nearest-neighbour upsampling by 2^s), y fastest in both */
template <typename U>
struct CropPatch {
    struct Args {
        const U* full;
        U* out;
        int64_t fy, fx;
        int64_t py, px, n;
        int64_t yb, xb, zb;
        int s;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "crop_patch"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        for (int64_t i = t * blockDim.x + threadIdx.x; i < a.n; i += a.G * blockDim.x) {
            const int64_t y = i % a.py, r = i / a.py;
            const int64_t x = r % a.px, z = r / a.px;
            a.out[i] = a.full[(((z + a.zb) >> a.s) * a.fx + ((x + a.xb) >> a.s)) * a.fy + ((y + a.yb) >> a.s)];
        }
    }
};
}  // namespace

namespace {
/* |grad| from the per-axis gradients, in APRNumerics::gradient_magnitude_*'s order
   (APRNumerics.hpp:216-283): g_y^2, + g_x^2, + g_z^2 (absent axes skipped), sqrtf */
struct GradMag {
    struct Args {
        float* g;          /* in: g_y, out: magnitude */
        const float* gx;   /* nullptr: no x axis */
        const float* gz;   /* nullptr: no z axis */
        uint64_t n;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "grad_mag"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        for (uint64_t i = (uint64_t)t * blockDim.x + threadIdx.x; i < a.n; i += (uint64_t)a.G * blockDim.x) {
            float m = a.g[i] * a.g[i];
            if (a.gx) m = m + a.gx[i] * a.gx[i];
            if (a.gz) m = m + a.gz[i] * a.gz[i];
            a.g[i] = sqrtf(m);
        }
    }
};
}  // namespace

namespace {
/* APRNumerics::face_neighbour_filter (APRNumerics.hpp:305-355) along one dimension: one lane
   per particle (a wave per row).  The neighbours of each face come from the random iterator's
   search (APRIterator.hpp:283-394, RandomAccess.hpp:92-170): the same-level cell, else (above
   l_min) the parent-level cell containing the face neighbour, else (below l_max) the four
   children on the face, counted where they are particles provided the first one is.  Cells
   are found by binary search in their row; coordinates follow the reference's unsigned 16-bit
   arithmetic, and the four l_max rows under the first parent row read row (0, 0), as the
   reference's random access resolves them. */
struct FaceFilter {
    struct Args {
        Rows R;
        const uint64_t* xz_end;
        const uint16_t* y_vec;
        const void* in;
        int in_u16;
        float* out;
        float f0, f1, f2;
        int dim;
        int64_t total_rows;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "face_neighbour_filter"; }

    static __device__ __forceinline__ float val(const Args& a, int64_t i) {
        return a.in_u16 ? (float)((const uint16_t*)a.in)[i] : ((const float*)a.in)[i];
    }
    /* particle index at (level, z, x, y) or -1 */
    static __device__ __forceinline__ int64_t find(const Args& a, int level, int64_t z, int64_t x, int64_t y) {
        const Rows& R = a.R;
        const int li = level - R.l_lo;
        if (li < 0 || li >= R.n_levels) return -1;
        if (z < 0 || x < 0 || y < 0 || z >= R.z_num[li] || x >= R.x_num[li] || y >= R.y_num[li]) return -1;
        if (li == R.n_levels - 1 && z < 2 && x < 2) {
            z = 0;
            x = 0;
        }
        const int64_t rid = R.row_begin[li] + z * R.x_num[li] + x;
        uint64_t lo = a.xz_end[rid - 1], hi = a.xz_end[rid];
        const uint64_t e = hi;
        while (lo < hi) {
            const uint64_t mid = (lo + hi) >> 1;
            if ((int64_t)a.y_vec[mid] < y) lo = mid + 1;
            else hi = mid;
        }
        return (lo < e && (int64_t)a.y_vec[lo] == y) ? (int64_t)lo : -1;
    }
    static __device__ __forceinline__ int64_t u16c(int64_t v) { return (int64_t)(uint16_t)v; }

    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        const int lane = threadIdx.x & 63;
        const int64_t wpb = blockDim.x / 64;
        const Rows& R = a.R;
        const int l_min = R.l_lo, l_max = R.l_lo + R.n_levels - 1;
        for (int64_t r = t * wpb + (threadIdx.x >> 6); r < a.total_rows; r += a.G * wpb) {
            const int li = row_level(R, r);
            const int level = R.l_lo + li;
            const int64_t row = r - R.prefix[li];
            const int64_t z = row / R.x_num[li], x = row % R.x_num[li];
            const uint64_t b = a.xz_end[R.row_begin[li] + row - 1], e = a.xz_end[R.row_begin[li] + row];
            for (uint64_t i = b + lane; i < e; i += 64) {
                const int64_t y = a.y_vec[i];
                const float cur = val(a, (int64_t)i);
                float o = cur * a.f1;
                for (int k = 0; k < 2; ++k) {
                    const int sgn = k == 0 ? 1 : -1;
                    const int dy = a.dim == 0 ? sgn : 0, dx = a.dim == 1 ? sgn : 0, dz = a.dim == 2 ? sgn : 0;
                    const float ft = k == 0 ? a.f2 : a.f0;
                    float sum = 0.0f, cnt = 0.0f;
                    const int64_t ny = u16c(y + dy), nx = u16c(x + dx), nz = u16c(z + dz);
                    int64_t n = find(a, level, nz, nx, ny);
                    if (n < 0 && level > l_min) n = find(a, level - 1, nz / 2, nx / 2, ny / 2);
                    if (n >= 0) {
                        sum += val(a, n);
                        cnt += 1.0f;
                    } else if (level < l_max) {
                        const int64_t cy = u16c(ny * 2 + (dy < 0)), cx = u16c(nx * 2 + (dx < 0)), cz = u16c(nz * 2 + (dz < 0));
                        for (int c = 0; c < 4; ++c) {
                            const int o0 = c & 1, o1 = c >> 1;
                            int64_t yy = cy, xx = cx, zz = cz;
                            if (a.dim == 0) { xx += o0; zz += o1; }
                            else if (a.dim == 1) { yy += o0; zz += o1; }
                            else { yy += o0; xx += o1; }
                            const int64_t m = find(a, level + 1, u16c(zz), u16c(xx), u16c(yy));
                            if (m < 0) {
                                if (c == 0) break;
                                continue;
                            }
                            sum += val(a, m);
                            cnt += 1.0f;
                        }
                    }
                    if (cnt > 0.0f) o += ft * sum / cnt;
                    else o += ft * cur;
                }
                a.out[i] = o;
            }
        }
    }
};
}  // namespace

void face_neighbour_filter(aprh_context* ctx, const aprh_apr& a, const void* in, int in_dtype, float* out, const float* filter3, int dim) {
    if (a.total == 0) return;
    Rows R = make_rows(a.y_num, a.x_num, a.z_num, a.level_xz_vec, a.l_min, a.l_max);
    const int64_t rows = R.prefix[R.n_levels];
    const int64_t G = stride_tiles(rows, 4, 16384);
    launch_tiles<FaceFilter>(ctx, {R, a.xz_end.as<uint64_t>(), a.y_vec.as<uint16_t>(), in, in_dtype == APRH_DTYPE_U16 ? 1 : 0, out,
                                   filter3[0], filter3[1], filter3[2], dim, rows, G},
                             G);
}

void gradient_magnitude_combine(aprh_context* ctx, float* g, const float* gx, const float* gz, uint64_t n) {
    if (n == 0) return;
    const int64_t G = stride_tiles((int64_t)n, 256 * 4);
    launch_tiles<GradMag>(ctx, {g, gx, gz, n, G}, G);
}

namespace {
struct LocalStdStep {
    struct Args {
        int mode;
        float* p;
        const void* q;
        uint64_t n;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "local_std_step"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        for (uint64_t i = (uint64_t)t * blockDim.x + threadIdx.x; i < a.n; i += (uint64_t)a.G * blockDim.x) {
            if (a.mode == 0) {
                a.p[i] = (float)((const uint16_t*)a.q)[i];
            } else if (a.mode == 1) {
                a.p[i] = a.p[i] * a.p[i];
            } else {
                const float m = ((const float*)a.q)[i];
                const float d = a.p[i] - m * m;
                a.p[i] = sqrtf(d < 0.0f ? 0.0f : d);
            }
        }
    }
};
}  // namespace

namespace {
/* elementwise steps of APRNumerics::richardson_lucy_tv (APRNumerics.hpp:431-525), in the
   reference's operation order:
   mode 0, div_norm_grad's normalisation: m = sqrtf(g_z^2 + g_x^2 + g_y^2) (absent axes are
           zero), each component divided by m where m > 1e-6 (compared in double);
   mode 1, the divergence sum: a = b + a;
   mode 2, the update: a = a * b / (1 - reg * c) */
struct TvStep {
    struct Args {
        int mode;
        float* a;
        float* b;   /* mode 0: g_x or nullptr; 1, 2: read only */
        float* c;   /* mode 0: g_z or nullptr; 2: read only     */
        float reg;
        uint64_t n;
        int64_t G;
    };
    static constexpr int THREADS = 256;
    static const char* name() { return "rl_tv_step"; }
    static __device__ __forceinline__ void run(const Args& a, int64_t t) {
        for (uint64_t i = (uint64_t)t * blockDim.x + threadIdx.x; i < a.n; i += (uint64_t)a.G * blockDim.x) {
            if (a.mode == 0) {
                const float y = a.a[i], x = a.b ? a.b[i] : 0.0f, z = a.c ? a.c[i] : 0.0f;
                const float m = sqrtf(z * z + x * x + y * y);
                if ((double)m > 1e-6) {
                    if (a.c) a.c[i] = z / m;
                    if (a.b) a.b[i] = x / m;
                    a.a[i] = y / m;
                }
            } else if (a.mode == 1) {
                a.a[i] = a.b[i] + a.a[i];
            } else {
                a.a[i] = a.a[i] * a.b[i] / (1.0f - a.reg * a.c[i]);
            }
        }
    }
};
}  // namespace

void rl_tv_step(aprh_context* ctx, int mode, float* p, float* q, float* r, float reg, uint64_t n) {
    if (n == 0) return;
    const int64_t G = stride_tiles((int64_t)n, 256 * 4);
    launch_tiles<TvStep>(ctx, {mode, p, q, r, reg, n, G}, G);
}

void fill_f32(aprh_context* ctx, float* p, size_t n, float v) {
    if (n == 0) return;
    hipLaunchKernelGGL(k_fill_f32, kGrid, kBlock, 0, ctx->stream, p, n, v);
    HIP_LAUNCH_CHECK();
}

void local_std_step(aprh_context* ctx, int mode, float* p, const void* q, uint64_t n) {
    if (n == 0) return;
    const int64_t G = stride_tiles((int64_t)n, 256 * 4);
    launch_tiles<LocalStdStep>(ctx, {mode, p, q, n, G}, G);
}

bool patch_limits(const aprh_apr& a, aprh_patch& p) {
    /* ReconPatch::check_limits (APRReconstruction.hpp:38-64): extents ceil(dim * 2^level_delta),
       which must fit an int32 */
    if (p.level_delta > 30 || p.level_delta < -30) return false;
    int64_t m[3];
    for (int d = 0; d < 3; ++d) {
        const int64_t dim = a.org[d];
        m[d] = p.level_delta >= 0 ? (dim << p.level_delta) : ((dim + ((int64_t)1 << -p.level_delta) - 1) >> -p.level_delta);
        if (m[d] > INT32_MAX) return false;
    }
    int32_t* b[3] = {&p.y_begin, &p.x_begin, &p.z_begin};
    int32_t* e[3] = {&p.y_end, &p.x_end, &p.z_end};
    for (int d = 0; d < 3; ++d) {
        *b[d] = std::max(0, *b[d]);
        *e[d] = *e[d] < 0 ? (int32_t)m[d] : (int32_t)std::min<int64_t>(m[d], *e[d]);
    }
    return p.y_begin < p.y_end && p.x_begin < p.x_end && p.z_begin < p.z_end;
}

/* APRReconstruction::reconstruct_constant / reconstruct_level over a patch (:296-394, :397-490):
   the level image of level min(l_max, l_max + level_delta), cut to the patch (and upsampled by
   2^level_delta when level_delta > 0).  parts == nullptr: the level image. */
void reconstruct_patch(aprh_context* ctx, aprh_apr& a, const void* parts, int pdt, const aprh_patch& p, void* img, int idt) {
    const int level = a.l_max + std::min(p.level_delta, 0);
    const int s = std::max(p.level_delta, 0);
    const int64_t fy = a.y_num[level], fx = a.x_num[level], fz = a.z_num[level];
    const int64_t py = p.y_end - p.y_begin, px = p.x_end - p.x_begin, pz = p.z_end - p.z_begin;
    const size_t es = idt == APRH_DTYPE_U16 ? 2 : 4;
    auto full_image = [&](void* dst) {
        if (parts) reconstruct_any(ctx, a, parts, pdt, level, dst, idt);
        else reconstruct_level(ctx, a, level, dst, idt);
    };
    if (s == 0 && py == fy && px == fx && pz == fz) {
        full_image(img);
        return;
    }
    Buf full(ctx->pool, (size_t)(fy * fx * fz) * es);
    full_image(full.ptr());
    const int64_t n = py * px * pz;
    const int64_t G = stride_tiles(n, 256 * 4);
    if (idt == APRH_DTYPE_U16)
        launch_tiles<CropPatch<uint16_t>>(ctx, {full.as<uint16_t>(), (uint16_t*)img, fy, fx, py, px, n, p.y_begin, p.x_begin, p.z_begin, s, G}, G);
    else
        launch_tiles<CropPatch<float>>(ctx, {full.as<float>(), (float*)img, fy, fx, py, px, n, p.y_begin, p.x_begin, p.z_begin, s, G}, G);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

void reconstruct_any(aprh_context* ctx, aprh_apr& a, const void* parts, int pdt, int level, void* img, int idt, uint8_t* lev) {
    if (pdt == 0 && idt == 0) reconstruct<uint16_t, uint16_t>(ctx, a, (const uint16_t*)parts, level, (uint16_t*)img, lev);
    else if (pdt == 0 && idt == 1) reconstruct<uint16_t, float>(ctx, a, (const uint16_t*)parts, level, (float*)img, lev);
    else if (pdt == 1 && idt == 0) reconstruct<float, uint16_t>(ctx, a, (const float*)parts, level, (uint16_t*)img, lev);
    else reconstruct<float, float>(ctx, a, (const float*)parts, level, (float*)img, lev);
}

template void tree_mean<uint16_t>(aprh_context*, aprh_apr&, const uint16_t*, float*);
template void tree_mean<float>(aprh_context*, aprh_apr&, const float*, float*);
template void convolve<uint16_t>(aprh_context*, aprh_apr&, const std::vector<HostStencil>&, const uint16_t*, float*, bool, const float*);
template void convolve<float>(aprh_context*, aprh_apr&, const std::vector<HostStencil>&, const float*, float*, bool, const float*);

/* APRNumerics::richardson_lucy (APRNumerics.hpp:549-593): per iteration the tree means of u,
   blur = u (*) flip(psf) with relative_blur = in / blur in the convolution's epilogue, the tree
   means of relative_blur, and u *= relative_blur (*) psf in the second convolution's epilogue
   with the partial sums of the relative-update norm (stopping rule, when tol > 0) */
template <typename T>
int richardson_lucy(aprh_context* ctx, aprh_apr& a, const T* in, float* u, const std::vector<HostStencil>& psf,
                    const std::vector<HostStencil>& psf_flipped, int max_iter, bool resume, double tol, double* last_rel) {
    hipStream_t st = ctx->stream;
    const size_t P = a.total;
    if (!resume && P > 0) {
        hipLaunchKernelGGL(k_fill_f32, kGrid, kBlock, 0, st, u, P, 1.0f);
        HIP_LAUNCH_CHECK();
    }
    if (P > 0) ensure_tree(ctx, a);
    const bool sep = ctx->conv_mode == APRH_CONV_SEPARABLE;
    const bool in_u16 = std::is_same<T, uint16_t>::value;
    Buf blur(ctx->pool, std::max<size_t>(P, 1) * 4), tree(ctx->pool, std::max<uint64_t>(a.t_total, 1) * 4);
    Buf part, sums(ctx->pool, 2 * sizeof(double));
    int it = 0;
    double rel = 0;
    for (it = 0; it < max_iter && P > 0; ++it) {
        tree_mean<float>(ctx, a, u, tree.as<float>());
        conv_levels<float>(ctx, a, psf_flipped, sep, u, tree.as<float>(), blur.as<float>(), true, 1, in, in_u16, nullptr, nullptr);
        tree_mean<float>(ctx, a, blur.as<float>(), tree.as<float>());
        int64_t np = 0;
        conv_levels<float>(ctx, a, psf, sep, blur.as<float>(), tree.as<float>(), u, true, 2, nullptr, false, &part, &np);
        reduce_norm_parts(ctx, part.as<double>(), np, sums.as<double>());
        double h[2];
        HIP_CHECK(hipMemcpyAsync(h, sums.ptr(), 16, hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        rel = h[1] > 0 ? std::sqrt(h[0] / h[1]) : 0.0;
        if (tol > 0 && rel < tol) {
            ++it;
            break;
        }
    }
    if (last_rel) *last_rel = rel;
    return it;
}

template int richardson_lucy<uint16_t>(aprh_context*, aprh_apr&, const uint16_t*, float*, const std::vector<HostStencil>&,
                                       const std::vector<HostStencil>&, int, bool, double, double*);
template int richardson_lucy<float>(aprh_context*, aprh_apr&, const float*, float*, const std::vector<HostStencil>&,
                                    const std::vector<HostStencil>&, int, bool, double, double*);

}  // namespace aprh
