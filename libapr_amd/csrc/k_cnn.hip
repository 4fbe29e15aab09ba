/*
 * k_cnn.hip -- the learned Richardson-Lucy warm start: a 3-D convolutional
 * network (no counterpart in the reference) trained and run on the GPU with
 * hand-written MFMA kernels.
 *
 * Network: four "valid" 3x3x3 convolutions, 1 -> 16 -> 16 -> 16 -> 1
 * channels, ReLU after the first three, residual output y = x + conv4.  A
 * tile of side S + 8 gives an output tile of side S (64 in training; over
 * a whole volume as its size suggests).
 * Parameters (f32 master copy, 14737 values): W1[27][16] b1[16]
 * W2[27][16][16] b2[16] W3[27][16][16] b3[16] W4[27][16] b4, tap =
 * (dz * 3 + dx) * 3 + dy.
 *
 * Precision: layers 1-3 run on v_mfma_f32_16x16x32_bf16 (bf16 weights and
 * activations, f32 accumulation); layer 4 (one output channel) runs on the
 * same MFMA with its f32 weights split into two bf16 parts, and its input
 * gradient on the VALU in f32.  Activations are stored channels-last
 * (16 bf16 = 32 B per voxel) for the convolutions and, in training, also
 * channel-planar for the weight-gradient GEMMs, whose reduction dimension is
 * the voxels.
 *
 * MFMA operand layout (16x16x32 bf16, verified on the device): lane l holds
 * A[l % 16][(l / 16) * 8 + j] and B[(l / 16) * 8 + j][l % 16] for j < 8, and
 * the result D[(l / 16) * 4 + i][l % 16] for i < 4.
 *  - convolution (forward and input gradient): M = 16 output channels, N = 16
 *    output voxels, K = pairs of taps x 16 input channels (14 MFMAs);
 *  - weight gradient: M = 16 input channels (or taps), N = 16 output
 *    channels (or taps), K = 32 voxels along y.
 */
#include <algorithm>
#include <cmath>
#include <random>

#include "aprh_internal.hpp"
#include "tiles.hpp"

namespace aprh {

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int CH = 16, NT = 27, NPAIR = 14;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + NT * CH, OFF_W2 = OFF_B1 + CH, OFF_B2 = OFF_W2 + NT * CH * CH, OFF_W3 = OFF_B2 + CH,
              OFF_B3 = OFF_W3 + NT * CH * CH, OFF_W4 = OFF_B3 + CH, OFF_B4 = OFF_W4 + NT * CH, N_PARAMS = OFF_B4 + 1;

/* float -> bf16, round to nearest even */
__host__ __device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u;
    __builtin_memcpy(&u, &f, 4);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
/* the same rounding (to nearest even) in one instruction, for finite values */
__device__ __forceinline__ uint16_t f2bf_hw(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf2f(uint16_t h) {
    const uint32_t u = (uint32_t)h << 16;
    float f;
    __builtin_memcpy(&f, &u, 4);
    return f;
}
__device__ __forceinline__ uint32_t pack2(uint16_t lo, uint16_t hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
/* two floats -> two bf16 (round to nearest even, finite values) in one word */
__device__ __forceinline__ uint32_t pack2_bf16(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}
#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ void tap_offsets(int tap, int& dz, int& dx, int& dy) {
    dz = tap / 9;
    dx = (tap / 3) % 3;
    dy = tap % 3;
}

__device__ __forceinline__ void decompose(int v, int s, int& z, int& x, int& y) {
    z = v / (s * s);
    const int r = v - z * s * s;
    x = r / s;
    y = r - x * s;
}

/* four channels of a channel-last activation */
__device__ __forceinline__ void store_channels(uint16_t* p, const uint16_t (&h)[4]) {
    *(uint2*)p = make_uint2(pack2(h[0], h[1]), pack2(h[2], h[3]));
}

/* ---------------- forward ---------------- */

/* The forward layers run over bricks of 16 (y) x 8 (x) x 4 (z) output voxels.  A block stages the
   brick's input, (brick + 2)^3 voxels, in LDS once, and its four waves take the brick's 32 y rows of 16
   voxels: a row is the N of its MFMAs.  Every brick has the full layout, so a voxel's place is a shift
   and a mask; rows past the output's x or z edge and lanes past its y edge are never stored (an MFMA
   column depends on its own operand column only). */
constexpr int BY = 16, BX = 8, BZ = 4, IY = BY + 2, IX = BX + 2, IZ = BZ + 2, ROWS = BX * BZ;

/* brick br of a launch over T tiles of nby x nbx x nbz bricks, y fastest.  The kernels number
   their blocks XCD by XCD (xcd_block), so neighbouring bricks, which share their halo voxels,
   meet in one L2 */
__device__ __forceinline__ void brick_origin(uint32_t br, uint32_t nby, uint32_t nbx, uint32_t nbz, int& t, int& z0, int& x0, int& y0) {
    const uint32_t by = br % nby;
    br /= nby;
    const uint32_t bx = br % nbx;
    br /= nbx;
    const uint32_t bz = br % nbz;
    t = (int)(br / nbz);
    y0 = (int)by * BY;
    x0 = (int)bx * BX;
    z0 = (int)bz * BZ;
}

/* LDS offset (in voxels of the staged brick) of tap t */
__host__ __device__ constexpr int tap_vox(int t) { return ((t / 9) * IX + (t / 3) % 3) * IY + t % 3; }
__device__ __forceinline__ int tap_lds(int tap) { return tap_vox(min(tap, NT - 1)); }
/* The 27 taps of a 16 -> 16 layer in 14 pairs, one MFMA each (K = 2 taps x 16 channels), such that one A
   operand serves many outputs: pairs 0-8 are dy = 0, 1 of row (dz, dx); 9-11 are dy = 2 of (dz, 0) and
   (dz, 1); 12 is dy = 2 of (0, 2) and (1, 2); 13 is tap 26 alone (its odd half has zero weights and reads
   tap 26 again).  Tap of half h of pair p, NT for none: */
__host__ __device__ constexpr int pair_tap(int p, int h) {
    return p < 9 ? 3 * p + h : p < 12 ? 9 * (p - 9) + 3 * h + 2 : p == 12 ? 9 * h + 8 : h ? NT : 26;
}

/* Outputs of a wave: WZ x WX rows of 16 voxels from (kz0, kx0) of the brick.  A row (z, x) of the input is
   read once for each kind of pair and meets every output it belongs to: 56 LDS reads for 112 MFMAs (one
   read per MFMA asks for twice the LDS rate that the matrix cores then leave).  The weights are the A
   operand, so lane (g, m), which reads channels (g & 1) * 8 .. + 7 of half g >> 1 of the pair, voxel m,
   gets channels 4 g .. 4 g + 3 of voxel m: 8 bytes of a channel-last store or mask, where voxels 4 g .. of
   channel m made four 2-byte accesses of each.  16 tiles of 64^3, forward layers with planar copies
   245 -> 162 us, input gradients 339 -> 222, first layer 169 -> 85. */
constexpr int WZ = 2, WX = 4;
static_assert(4 * WZ * WX == ROWS && BX == 2 * WX && BZ == 2 * WZ, "the four waves' rows make up the brick");
__device__ __forceinline__ void rows_mfma(const uint16_t* tile, int kz0, int kx0, int lane, const u32x4 (&w)[NPAIR], f32x4 (&acc)[WZ][WX]) {
    const int g = lane >> 4, lo = ((kz0 * IX + kx0) * IY + (lane & 15)) * CH + (g & 1) * 8, th = g >> 1;
    const uint16_t* ba = tile + lo + th * CH;                        /* dy 0, 1               */
    const uint16_t* bb = tile + lo + 2 * CH + th * IY * CH;          /* dy 2 of x, x + 1      */
    const uint16_t* bc = tile + lo + 2 * CH + th * IX * IY * CH;     /* dy 2 of z, z + 1      */
    const uint16_t* bd = tile + lo + 2 * CH;                         /* dy 2 alone            */
    auto add = [&](f32x4& c, u32x4 a, int p) { c = mfma(w[p], a, c); };
    auto at = [&](const uint16_t* b, int z, int x) { return *(const u32x4*)(b + (z * IX + x) * IY * CH); };
#pragma unroll
    for (int z = 0; z < WZ; ++z)
#pragma unroll
        for (int x = 0; x < WX; ++x) acc[z][x] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int z = 0; z < WZ + 2; ++z)
#pragma unroll
        for (int x = 0; x < WX + 2; ++x) {
            const u32x4 a = at(ba, z, x);
#pragma unroll
            for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx)
                    if (z - dz >= 0 && z - dz < WZ && x - dx >= 0 && x - dx < WX) add(acc[z - dz][x - dx], a, 3 * dz + dx);
            if (x < WX) {
                const u32x4 b = at(bb, z, x);
#pragma unroll
                for (int dz = 0; dz < 3; ++dz)
                    if (z - dz >= 0 && z - dz < WZ) add(acc[z - dz][x], b, 9 + dz);
            }
            if (x >= 2 && z < WZ) add(acc[z][x - 2], at(bc, z, x), 12);
            if (x >= 2 && z >= 2) add(acc[z - 2][x - 2], at(bd, z, x), 13);
        }
}

/* The bricks of a layer over the tiles of an image, of which the last ones end within a tile: tile t has the
   y x z bricks tab[t].y x tab[t].z x tab[t].w from number tab[t].x on, and what lies outside them nothing wanted
   depends on (tab nullptr: all tiles alike).  The wanted bricks are numbered without gaps: launched over whole
   tiles, the XCDs whose share was the image's ends had nothing to do (128^3 in eight tiles of 74^3: 0.30 ms,
   0.26 this way; 150^3 0.70, 0.44). */
struct BrickMap {
    const int4* tab;
    int T;
};
__device__ __forceinline__ void wanted_brick(const BrickMap& m, uint32_t br, uint32_t nby, uint32_t nbx, uint32_t nbz, int& t, int& z0, int& x0,
                                             int& y0) {
    if (!m.tab) return brick_origin(br, nby, nbx, nbz, t, z0, x0, y0);
    const int lane = threadIdx.x & 63;
    int4 e = make_int4(0x7FFFFFFF, 1, 1, 1);
    if (lane < m.T) e = m.tab[lane];
    const int own = __popcll(__ballot((uint32_t)e.x <= br)) - 1;
    int none;
    brick_origin(br - (uint32_t)__builtin_amdgcn_readlane(e.x, own), (uint32_t)__builtin_amdgcn_readlane(e.y, own),
                 (uint32_t)__builtin_amdgcn_readlane(e.z, own), (uint32_t)__builtin_amdgcn_readlane(e.w, own), none, z0, x0, y0);
    t = own;
}
/* an image whose tiles the network reads and writes in place of tile buffers */
struct Volume {
    const void* img;
    int64_t yn, xn, zn;
    const int* org;
    float inv_scale, scale, floor_v;
    float* out;
};

__device__ __forceinline__ int64_t refl_any(int64_t q, int64_t n) {
    /* reflection about the edge samples, repeated for windows wider than the volume */
    if (q >= 0 && q < n) return q;
    if (n == 1) return 0;
    const int64_t per = 2 * (n - 1);
    q %= per;
    if (q < 0) q += per;
    return q < n ? q : per - q;
}

/* stages the brick's input, IZ x IX x IY voxels of 16 channels from (z0, x0, y0) + off of a tile
   of side sin, as tile[(lz * IX + lx) * IY + ly][16], 16-byte chunk c at tile[8 c].
   DIRECT (the forward layers, off = 0): every chunk goes straight from global memory to LDS
   (global_load_lds_dwordx4: lane l of a wave writes the wave's base + 16 l, which is the chunk
   order), so all of a brick's loads are in flight at once and hold no registers.  Positions past
   the input's far edges load a clamped position instead of zero: in a valid convolution they feed
   only outputs past the output's edge, which are never stored.
   Otherwise (the input gradients, off = -2, zero outside the input) through registers. */
constexpr int NCH = IZ * IX * IY * 2, NCH_PT = (NCH + 255) / 256;
template <bool DIRECT>
__device__ __forceinline__ void stage_brick(uint16_t* tile, const uint16_t* __restrict__ it, int sin, int off, int z0, int x0, int y0) {
    __syncthreads();   /* the previous brick's waves are done with the tile */
    if constexpr (DIRECT) {
        const int wbase = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 64;
#pragma unroll
        for (int j = 0; j < NCH_PT; ++j) {
            const int c = threadIdx.x + 256 * j;
            if (c < NCH) {
                const int q = c >> 1, h = c & 1;
                const int ly = q % IY, r = q / IY, lx = r % IX, lz = r / IX;
                const int zi = min(z0 + lz, sin - 1), xi = min(x0 + lx, sin - 1), yi = min(y0 + ly, sin - 1);
                __builtin_amdgcn_global_load_lds((const void*)(it + (int64_t)((zi * sin + xi) * sin + yi) * CH + h * 8),
                                                 LDS_PTR(tile + (wbase + 256 * j) * 8), 16, 0, 0);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    } else {
        for (int c = threadIdx.x; c < NCH; c += 256) {
            const int q = c >> 1, h = c & 1;
            const int ly = q % IY, r = q / IY, lx = r % IX, lz = r / IX;
            const int zi = z0 + off + lz, xi = x0 + off + lx, yi = y0 + off + ly;
            u32x4 v = {0u, 0u, 0u, 0u};
            if ((unsigned)zi < (unsigned)sin && (unsigned)xi < (unsigned)sin && (unsigned)yi < (unsigned)sin)
                v = *(const u32x4*)(it + (int64_t)((zi * sin + xi) * sin + yi) * CH + h * 8);
            *(u32x4*)&tile[c * 8] = v;
        }
    }
    __syncthreads();
}

/* layer 1: x (f32, side s0) -> a (bf16, side s1 = s0 - 2), ReLU(conv + b1).  The brick's input goes
   straight to LDS as f32 (global_load_lds_dword, clamped at the far edges as in stage_brick) and
   is rounded to bf16 when the operand is built; lane (g, m) holds taps g * 8 .. g * 8 + 7 of
   voxel m.  IMG: the input is read from an image of T, reflected past its ends and scaled (before, a pass
   of its own made the tiles: 74 us per 32 of 72^3) */
constexpr int NIN1 = IZ * IX * IY, NIN1_PT = (NIN1 + 255) / 256;
template <typename T, bool IMG>
__global__ __launch_bounds__(256) void k_l1_lds(const float* __restrict__ x, int s0, int s1, const u32x4* __restrict__ W1p,
                                                const float* __restrict__ b1, uint16_t* a_cl, uint16_t* a_pl, uint32_t nbricks, uint32_t nby,
                                                uint32_t nbx, uint32_t nbz, BrickMap map, Volume vol) {
    __shared__ __attribute__((aligned(16))) float tile[NIN1_PT * 256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const u32x4 wb = W1p[lane];
    const f32x4 bias = *(const f32x4*)(b1 + g * 4);
    int toff[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) toff[j] = tap_lds(g * 8 + j);
    const int nv = s1 * s1 * s1, nin = s0 * s0 * s0;
    for (uint32_t br = (uint32_t)xcd_block(blockIdx.x, gridDim.x); br < nbricks; br += gridDim.x) {
        int t, z0, x0, y0;
        wanted_brick(map, br, nby, nbx, nbz, t, z0, x0, y0);
        const float* xt = x + (int64_t)t * nin;
        __syncthreads();   /* the previous brick's waves are done with the tile */
        float in[NIN1_PT];
#pragma unroll
        for (int j = 0; j < NIN1_PT; ++j) {
            const int c = threadIdx.x + 256 * j;
            in[j] = 0.0f;
            if (c < NIN1) {
                const int ly = c % IY, r = c / IY, lx = r % IX, lz = r / IX;
                const int zi = min(z0 + lz, s0 - 1), xi = min(x0 + lx, s0 - 1), yi = min(y0 + ly, s0 - 1);
                if constexpr (IMG) {
                    const int64_t gy = refl_any(vol.org[3 * t] - 4 + yi, vol.yn), gx = refl_any(vol.org[3 * t + 1] - 4 + xi, vol.xn),
                                  gz = refl_any(vol.org[3 * t + 2] - 4 + zi, vol.zn);
                    in[j] = (float)((const T*)vol.img)[(gz * vol.xn + gx) * vol.yn + gy] * vol.inv_scale;
                } else {
                    __builtin_amdgcn_global_load_lds((const void*)(xt + (zi * s0 + xi) * s0 + yi), LDS_PTR(tile + wave * 64 + 256 * j), 4, 0, 0);
                }
            }
        }
        if constexpr (IMG) {
#pragma unroll
            for (int j = 0; j < NIN1_PT; ++j) tile[threadIdx.x + 256 * j] = in[j];
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        __syncthreads();
        for (int row = wave; row < ROWS; row += 4) {
            const int kx = row % BX, kz = row / BX;
            if (x0 + kx >= s1 || z0 + kz >= s1) continue;
            const float* base = &tile[(kz * IX + kx) * IY + m];
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) f[j] = base[toff[j]];
            const u32x4 av = {pack2_bf16(f[0], f[1]), pack2_bf16(f[2], f[3]), pack2_bf16(f[4], f[5]), pack2_bf16(f[6], f[7])};
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = mfma(wb, av, acc);
            if (y0 + m >= s1) continue;
            /* channels 4 g .. of voxel m */
            const int v = ((z0 + kz) * s1 + x0 + kx) * s1 + y0 + m;
            uint16_t hv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) hv[i] = f2bf_hw(fmaxf(acc[i] + bias[i], 0.0f));
            store_channels(a_cl + ((int64_t)t * nv + v) * CH + g * 4, hv);
            if (a_pl) {
#pragma unroll
                for (int i = 0; i < 4; ++i) a_pl[((int64_t)t * CH + g * 4 + i) * nv + v] = hv[i];
            }
        }
    }
}

/* 16 -> 16 convolution: out(v) = sum_tap W[tap] in(v + tap + off) (zero outside the input), then
   + bias, ReLU, and / or the mask (ReLU derivative of a stored activation).  K of an MFMA is a pair
   of taps x 16 input channels (rows_mfma) */
template <bool DIRECT>
__global__ __launch_bounds__(256, 3) void k_conv16_lds(const uint16_t* __restrict__ in_cl, int sin, int sout, int off,
                                                    const u32x4* __restrict__ Wp, const float* __restrict__ bias,
                                                    const uint16_t* __restrict__ mask_cl, uint16_t* out_cl, uint16_t* out_pl, int relu,
                                                    uint32_t nbricks, uint32_t nby, uint32_t nbx, uint32_t nbz, BrickMap map) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[IZ * IX * IY * CH];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const int kz0 = (wave >> 1) * WZ, kx0 = (wave & 1) * WX;
    u32x4 w[NPAIR];
#pragma unroll
    for (int p = 0; p < NPAIR; ++p) w[p] = Wp[p * 64 + lane];
    f32x4 bv = {0.f, 0.f, 0.f, 0.f};
    if (bias) bv = *(const f32x4*)(bias + g * 4);
    const int nv = sout * sout * sout;
    for (uint32_t br = (uint32_t)xcd_block(blockIdx.x, gridDim.x); br < nbricks; br += gridDim.x) {
        int t, z0, x0, y0;
        wanted_brick(map, br, nby, nbx, nbz, t, z0, x0, y0);
        stage_brick<DIRECT>(tile, in_cl + (int64_t)t * sin * sin * sin * CH, sin, off, z0, x0, y0);
        if (x0 + kx0 >= sout || z0 + kz0 >= sout) continue;
        f32x4 acc[WZ][WX];
        rows_mfma(tile, kz0, kx0, lane, w, acc);
#pragma unroll
        for (int kz = 0; kz < WZ; ++kz)
#pragma unroll
            for (int kx = 0; kx < WX; ++kx) {
                const int zo = z0 + kz0 + kz, xo = x0 + kx0 + kx;
                if (xo >= sout || zo >= sout) continue;
                const int vrow = (zo * sout + xo) * sout + y0;
                uint16_t hv[4];
                /* channels 4 g .. of voxel m */
                if (y0 + m >= sout) continue;
                const int64_t vc = ((int64_t)t * nv + vrow + m) * CH + g * 4;
                uint16_t mk[4];
                if (mask_cl) __builtin_memcpy(mk, __builtin_assume_aligned(mask_cl + vc, 8), 8);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float val = acc[kz][kx][i] + bv[i];
                    if (relu) val = fmaxf(val, 0.0f);
                    if (mask_cl && !(bf2f(mk[i]) > 0.0f)) val = 0.0f;
                    hv[i] = f2bf_hw(val);
                }
                if (out_cl) store_channels(out_cl + vc, hv);
                if (out_pl) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) out_pl[((int64_t)t * CH + g * 4 + i) * nv + vrow + m] = hv[i];
                }
            }
    }
}

/* layer 4 + residual (+ loss gradient): y = x(centre) + b4 + sum W4 a3, on the MFMA.  The weights
   keep f32 accuracy as two bf16 parts: W4p holds bf16(W4) in output channels 0-7 and
   bf16(W4 - bf16(W4)) in channels 8-15, so channel 0 + channel 8 is the layer's output.  Lane
   m < 16 takes voxel m of each row.
   With a target, also the loss gradient g4 = 2 (y - tgt) gscale and per-block partial sums of
   (y - tgt)^2 and g4.  IMG: the residual comes from an image of T and the output goes to one, scaled and
   floored (before, a pass of its own wrote the tiles back: 27 us per 32 of 64^3) */
template <typename T, bool IMG>
__global__ __launch_bounds__(256, 3) void k_l4_lds(const uint16_t* __restrict__ a3_cl, int S, const float* __restrict__ x,
                                                const u32x4* __restrict__ W4p, const float* __restrict__ b4, const float* __restrict__ tgt,
                                                float* y, float* g4, float gscale, double* part, uint32_t nbricks, uint32_t nby, uint32_t nbx,
                                                uint32_t nbz, BrickMap map, Volume vol) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[IZ * IX * IY * CH];
    __shared__ double red[2][IMG ? 1 : 256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kz0 = (wave >> 1) * WZ, kx0 = (wave & 1) * WX;
    u32x4 w[NPAIR];
#pragma unroll
    for (int p = 0; p < NPAIR; ++p) w[p] = W4p[p * 64 + lane];
    const float bv = b4[0];
    const int s3 = S + 2, s0 = S + 8;
    const int nv = S * S * S, n3 = s3 * s3 * s3, n0 = s0 * s0 * s0;
    double dsum = 0, gsum = 0;
    for (uint32_t br = (uint32_t)xcd_block(blockIdx.x, gridDim.x); br < nbricks; br += gridDim.x) {
        int t, z0, x0, y0;
        wanted_brick(map, br, nby, nbx, nbz, t, z0, x0, y0);
        stage_brick<true>(tile, a3_cl + (int64_t)t * n3 * CH, s3, 0, z0, x0, y0);
        if (x0 + kx0 >= S || z0 + kz0 >= S) continue;
        /* the residual (and target) loads go out before the MFMA chains */
        const int yo = y0 + lane;
        float xv[WZ][WX], tv[WZ][WX];
        int64_t at[WZ][WX];
#pragma unroll
        for (int kz = 0; kz < WZ; ++kz)
#pragma unroll
            for (int kx = 0; kx < WX; ++kx) {
                const int zo = z0 + kz0 + kz, xo = x0 + kx0 + kx;
                bool mine = lane < 16 && yo < S && xo < S && zo < S;
                xv[kz][kx] = tv[kz][kx] = 0.0f;
                if constexpr (IMG) {
                    const int64_t gy = vol.org[3 * t] + yo, gx = vol.org[3 * t + 1] + xo, gz = vol.org[3 * t + 2] + zo;
                    mine = mine && gy < vol.yn && gx < vol.xn && gz < vol.zn;
                    at[kz][kx] = mine ? (gz * vol.xn + gx) * vol.yn + gy : -1;
                    if (mine) xv[kz][kx] = (float)((const T*)vol.img)[at[kz][kx]] * vol.inv_scale;
                } else {
                    at[kz][kx] = mine ? (int64_t)t * nv + (zo * S + xo) * S + yo : -1;
                    if (mine) {
                        xv[kz][kx] = x[(int64_t)t * n0 + ((zo + 4) * s0 + xo + 4) * s0 + yo + 4];
                        if (tgt) tv[kz][kx] = tgt[at[kz][kx]];
                    }
                }
            }
        f32x4 acc[WZ][WX];
        rows_mfma(tile, kz0, kx0, lane, w, acc);
#pragma unroll
        for (int kz = 0; kz < WZ; ++kz)
#pragma unroll
            for (int kx = 0; kx < WX; ++kx) {
                const float a = acc[kz][kx][0] + __shfl_down(acc[kz][kx][0], 32, 64);
                const int64_t i = at[kz][kx];
                if (i < 0) continue;
                const float out = xv[kz][kx] + bv + a;
                if constexpr (IMG) {
                    vol.out[i] = fmaxf(out * vol.scale, vol.floor_v);
                } else {
                    y[i] = out;
                    if (tgt) {
                        const float d = out - tv[kz][kx];
                        const float gv = 2.0f * d * gscale;
                        g4[i] = gv;
                        dsum += (double)d * (double)d;
                        gsum += (double)gv;
                    }
                }
            }
    }
    if constexpr (IMG) return;
    if (!part) return;
    red[0][threadIdx.x] = dsum;
    red[1][threadIdx.x] = gsum;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            red[0][threadIdx.x] += red[0][threadIdx.x + o];
            red[1][threadIdx.x] += red[1][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = red[0][0];
        part[2 * blockIdx.x + 1] = red[1][0];
    }
}

/* ---------------- backward ---------------- */

/* g3(u)[c] = mask(a3(u)[c]) * sum_tap W4[tap][c] g4(u - tap); one thread per voxel of side S + 2 */
__global__ __launch_bounds__(256) void k_l4_bwd(const float* __restrict__ g4, int S, const float* __restrict__ W4,
                                                const uint16_t* __restrict__ a3_cl, uint16_t* g3_cl, uint16_t* g3_pl, int T) {
    __shared__ float w[NT * CH];
    for (int i = threadIdx.x; i < NT * CH; i += blockDim.x) w[i] = W4[i];
    __syncthreads();
    const int s3 = S + 2;
    const int nv = S * S * S, n3 = s3 * s3 * s3;
    const int64_t total = (int64_t)T * n3;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int t = (int)(i / n3), u = (int)(i % n3);
        int zu, xu, yu;
        decompose(u, s3, zu, xu, yu);
        float acc[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[c] = 0.0f;
        const float* gt = g4 + (int64_t)t * nv;
        for (int tap = 0; tap < NT; ++tap) {
            int dz, dx, dy;
            tap_offsets(tap, dz, dx, dy);
            const int z = zu - dz, x = xu - dx, y = yu - dy;
            if (z < 0 || z >= S || x < 0 || x >= S || y < 0 || y >= S) continue;
            const float gv = gt[(z * S + x) * S + y];
#pragma unroll
            for (int c = 0; c < CH; ++c) acc[c] += w[tap * CH + c] * gv;
        }
        /* the voxel's 16 channels as two 16-byte words each way (32-byte aligned) */
        const u32x4* ap = (const u32x4*)(a3_cl + i * CH);
        u32x4* gp = (u32x4*)(g3_cl + i * CH);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const u32x4 av = ap[h];
            u32x4 o;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = h * 8 + 2 * q;
                const uint16_t lo = f2bf(bf2f((uint16_t)(av[q] & 0xffffu)) > 0.0f ? acc[c] : 0.0f);
                const uint16_t hi = f2bf(bf2f((uint16_t)(av[q] >> 16)) > 0.0f ? acc[c + 1] : 0.0f);
                o[q] = pack2(lo, hi);
                g3_pl[((int64_t)t * CH + c) * n3 + u] = lo;
                g3_pl[((int64_t)t * CH + c + 1) * n3 + u] = hi;
            }
            gp[h] = o;
        }
    }
}

/* Planar buffers end with this many readable bytes: the weight-gradient kernels load whole words
   past the end of a row (and mask what they loaded), so the last row's loads leave the data */
constexpr size_t PL_PAD = 32;

/* 8 consecutive planar bf16 values starting at y0 of a row (zero from y >= ylim): one 16-byte load at
   any alignment where all eight are inside */
__device__ __forceinline__ u32x4 load8(const uint16_t* row, int y0, int ylim) {
    u32x4 r = {0u, 0u, 0u, 0u};
    if (y0 + 8 <= ylim) {
        __builtin_memcpy(&r, row + y0, 16);
    } else if (y0 < ylim) {
        uint16_t h[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = (y0 + j < ylim) ? row[y0 + j] : (uint16_t)0;
        r = (u32x4){pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
    }
    return r;
}

/* the values j < n of a word of two (element 2k and 2k + 1) */
__device__ __forceinline__ uint32_t pair_mask(int k, int n) { return n >= 2 * k + 2 ? ~0u : n == 2 * k + 1 ? 0xffffu : 0u; }

/* Weight gradients of a layer with 16 input channels:
     dW[tap][cin][cout] = sum_v a(v + tap)[cin] g(v)[cout], db[cout] = sum_v g(v)[cout].
   M = cin, N = cout, K = 32 voxels along y; lane (g, m) holds 8 consecutive voxels of channel m.  An item
   is a run of xs rows along x of one (tile, z, 32 voxels of y): per row the wave loads the three new
   windows of `a` (z, z + 1, z + 2 at x + 2; 10 voxels each: a 16-byte and a 4-byte load at any alignment),
   keeps the windows of the two rows before in registers, and makes the taps' dy = 1, 2 operands by
   shifting the 10 voxels by one and two.  27 MFMAs run per 3 window loads, and the next row's loads are
   issued before them.  (Before: eight 2-byte loads per operand, 27 operands per row, 3.03 ms for 16
   tiles of 64^3 against 0.33 ms.)  The block's four waves add up in LDS, in wave order, and leave one
   partial: part[block][tap * 256 + cin * 16 + cout], then db.
   ONE: the last layer, whose g is one f32 channel (column 0 of N; no db): part[block][tap * 16 + cin]. */
template <bool ONE>
__global__ __launch_bounds__(256, 2) void k_dw(const uint16_t* __restrict__ a_pl, const void* __restrict__ g_pl, int sg, int xs, int nseg,
                                               int64_t items, float* part) {
    constexpr int W = ONE ? NT * CH : NT * 256 + CH;
    __shared__ float sum[W];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const int64_t wid = (int64_t)blockIdx.x * 4 + wave;
    const int64_t nw = (int64_t)gridDim.x * 4;
    const int sa = sg + 2;
    const int64_t ng = (int64_t)sg * sg * sg, na = (int64_t)sa * sa * sa;
    const int nch = (sg + 31) / 32;
    f32x4 acc[NT];
#pragma unroll
    for (int k = 0; k < NT; ++k) acc[k] = (f32x4){0.f, 0.f, 0.f, 0.f};
    float dbs = 0.0f;
    for (int64_t it = wid; it < items; it += nw) {
        const int ch = (int)(it % nch);
        int64_t r = it / nch;
        const int seg = (int)(r % nseg);
        r /= nseg;
        const int z = (int)(r % sg), t = (int)(r / sg);
        const int y0 = ch * 32 + g * 8, x0 = seg * xs, x1 = min(x0 + xs, sg);
        const bool on = y0 < sg;
        uint32_t am[5], bm[4];
#pragma unroll
        for (int k = 0; k < 5; ++k) am[k] = pair_mask(k, sa - y0);
#pragma unroll
        for (int k = 0; k < 4; ++k) bm[k] = pair_mask(k, sg - y0);
        const uint16_t* ap = a_pl + ((int64_t)t * CH + m) * na + (int64_t)z * sa * sa + y0;
        /* the 10 voxels y0 .. y0 + 9 of row (z + dz, x) */
        auto window = [&](int dz, int x, uint32_t (&w)[5]) {
#pragma unroll
            for (int k = 0; k < 5; ++k) w[k] = 0u;
            if (on) {
                const uint16_t* p = ap + (dz * sa + x) * sa;
                __builtin_memcpy(w, p, 16);
                __builtin_memcpy(w + 4, p + 8, 4);
#pragma unroll
                for (int k = 0; k < 5; ++k) w[k] &= am[k];
            }
        };
        auto row_g = [&](int x) {
            u32x4 v = {0u, 0u, 0u, 0u};
            if constexpr (ONE) {
                if (m == 0 && on) {
                    const float* p = (const float*)g_pl + (int64_t)t * ng + ((int64_t)z * sg + x) * sg + y0;
                    float f[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) f[j] = y0 + j < sg ? p[j] : 0.0f;
                    v = (u32x4){pack2_bf16(f[0], f[1]), pack2_bf16(f[2], f[3]), pack2_bf16(f[4], f[5]), pack2_bf16(f[6], f[7])};
                }
            } else if (on) {
                __builtin_memcpy(&v, (const uint16_t*)g_pl + ((int64_t)t * CH + m) * ng + ((int64_t)z * sg + x) * sg + y0, 16);
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] &= bm[k];
            }
            return v;
        };
        uint32_t win[3][3][5];   /* [x slot][dz] */
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int dz = 0; dz < 3; ++dz) window(dz, x0 + dx, win[dx][dz]);
        u32x4 bv = row_g(x0);
        for (int x = x0; x < x1; ++x) {
            uint32_t nxt[3][5];
            u32x4 bn = {0u, 0u, 0u, 0u};
            const bool more = x + 1 < x1;
            if (more) {
#pragma unroll
                for (int dz = 0; dz < 3; ++dz) window(dz, x + 3, nxt[dz]);
                bn = row_g(x + 1);
            }
            if constexpr (!ONE) {
#pragma unroll
                for (int q = 0; q < 4; ++q) dbs += bf2f((uint16_t)(bv[q] & 0xffffu)) + bf2f((uint16_t)(bv[q] >> 16));
            }
#pragma unroll
            for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const uint32_t* w = win[dx][dz];
                    const u32x4 a0 = {w[0], w[1], w[2], w[3]};
                    const u32x4 a1 = {__builtin_amdgcn_alignbit(w[1], w[0], 16), __builtin_amdgcn_alignbit(w[2], w[1], 16),
                                      __builtin_amdgcn_alignbit(w[3], w[2], 16), __builtin_amdgcn_alignbit(w[4], w[3], 16)};
                    const u32x4 a2 = {w[1], w[2], w[3], w[4]};
                    const int k = dz * 9 + dx * 3;
                    acc[k] = mfma(a0, bv, acc[k]);
                    acc[k + 1] = mfma(a1, bv, acc[k + 1]);
                    acc[k + 2] = mfma(a2, bv, acc[k + 2]);
                }
            if (more) {
#pragma unroll
                for (int dz = 0; dz < 3; ++dz)
#pragma unroll
                    for (int k = 0; k < 5; ++k) {
                        win[0][dz][k] = win[1][dz][k];
                        win[1][dz][k] = win[2][dz][k];
                        win[2][dz][k] = nxt[dz][k];
                    }
                bv = bn;
            }
        }
    }
    dbs += __shfl_xor(dbs, 16);
    dbs += __shfl_xor(dbs, 32);
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int k = 0; k < NT; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int o = ONE ? k * CH + g * 4 + i : k * 256 + (g * 4 + i) * CH + m;
                    if (!ONE || m == 0) sum[o] = w == 0 ? acc[k][i] : sum[o] + acc[k][i];
                }
            if (!ONE && lane < 16) sum[NT * 256 + m] = w == 0 ? dbs : sum[NT * 256 + m] + dbs;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < W; i += 256) part[(int64_t)blockIdx.x * W + i] = sum[i];
}

/* dW1[tap][cout] = sum_v x(v + tap) g1(v)[cout], db1: M = tap (two blocks of 16), N = cout, K = voxels v.
   One partial per block: part[block][tap * 16 + cout], then db1 */
__global__ __launch_bounds__(256) void k_dw_l1(const float* __restrict__ x, const uint16_t* __restrict__ g1_pl, int S, float* part, int T) {
    __shared__ float sum[NT * CH + CH];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 15, g = lane >> 4;
    const int64_t wid = (int64_t)blockIdx.x * 4 + wave;
    const int64_t nw = (int64_t)gridDim.x * 4;
    const int s1 = S + 6, s0 = S + 8;
    const int n1 = s1 * s1 * s1, n0 = s0 * s0 * s0;
    const int nch = (s1 + 31) / 32;
    const int64_t items = (int64_t)T * s1 * s1 * nch;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    float dbs = 0.0f;
    for (int64_t it = wid; it < items; it += nw) {
        const int ch = (int)(it % nch);
        const int64_t row = it / nch;
        const int t = (int)(row / (s1 * s1)), zx = (int)(row % (s1 * s1));
        const int z = zx / s1, x0 = zx % s1;
        const int y0 = ch * 32 + g * 8;
        const u32x4 bv = load8(g1_pl + ((int64_t)t * CH + m) * n1 + (z * s1 + x0) * s1, y0, s1);
#pragma unroll
        for (int q = 0; q < 4; ++q) dbs += bf2f((uint16_t)(bv[q] & 0xffffu)) + bf2f((uint16_t)(bv[q] >> 16));
        const float* xt = x + (int64_t)t * n0;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
            const int tap = mb * 16 + m;
            float f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (tap < NT) {
                const int dz = tap / 9, dx = (tap / 3) % 3, dy = tap % 3;
                const float* xr = xt + ((z + dz) * s0 + x0 + dx) * s0 + dy + y0;
                if (y0 + 8 <= s1) {
                    __builtin_memcpy(f, xr, 16);
                    __builtin_memcpy(f + 4, xr + 4, 16);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (y0 + j < s1) f[j] = xr[j];
                }
            }
            const u32x4 av = {pack2(f2bf(f[0]), f2bf(f[1])), pack2(f2bf(f[2]), f2bf(f[3])), pack2(f2bf(f[4]), f2bf(f[5])),
                              pack2(f2bf(f[6]), f2bf(f[7]))};
            acc[mb] = mfma(av, bv, acc[mb]);
        }
    }
    dbs += __shfl_xor(dbs, 16);
    dbs += __shfl_xor(dbs, 32);
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int tap = mb * 16 + g * 4 + i, o = tap * CH + m;
                    if (tap < NT) sum[o] = w == 0 ? acc[mb][i] : sum[o] + acc[mb][i];
                }
            if (lane < 16) sum[NT * CH + m] = w == 0 ? dbs : sum[NT * CH + m] + dbs;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < NT * CH + CH; i += 256) part[(int64_t)blockIdx.x * (NT * CH + CH) + i] = sum[i];
}

/* grad[off + i] = sum_p part[p * count + i] for i < count: 16 columns x 16 rows of partials a block, each
   row's thread summing every 16th partial, the rows then added in order.  (One thread per column took
   0.45 ms a layer for 2048 partials; 0.006 ms now.) */
__global__ __launch_bounds__(256) void k_reduce_parts(const float* __restrict__ part, int64_t nparts, int count, float* grad, int off) {
    __shared__ float sum[16][16];
    const int c = threadIdx.x & 15, r = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + c;
    float s = 0.0f;
    if (i < count) {
#pragma unroll 8
        for (int64_t p = r; p < nparts; p += 16) s += part[p * count + i];
    }
    sum[r][c] = s;
    __syncthreads();
    if (r == 0 && i < count) {
        for (int k = 1; k < 16; ++k) s += sum[k][c];
        grad[off + i] = s;
    }
}

/* the loss and the last layer's bias gradient from the blocks' pairs of partial sums */
__global__ __launch_bounds__(256) void k_loss(float* loss, float* db4, const double* __restrict__ part, int nblocks, double scale) {
    __shared__ double red[2][256];
    double s = 0, b = 0;
    for (int i = threadIdx.x; i < nblocks; i += 256) {
        s += part[2 * i];
        b += part[2 * i + 1];
    }
    red[0][threadIdx.x] = s;
    red[1][threadIdx.x] = b;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            red[0][threadIdx.x] += red[0][threadIdx.x + o];
            red[1][threadIdx.x] += red[1][threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        loss[0] = (float)(red[0][0] * scale);
        db4[0] = (float)red[1][0];
    }
}

__global__ void k_adam(float* p, const float* __restrict__ g, float* m, float* v, int n, float lr, float b1, float b2, float eps, float bc1,
                       float bc2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / bc1) / (sqrtf(vi / bc2) + eps);
}

/* lane-packed bf16 weights for the MFMA kernels */
__global__ void k_pack(const float* __restrict__ P, u32x4* W1p, u32x4* W2p, u32x4* W3p, u32x4* W2t, u32x4* W3t, u32x4* W4p) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;   /* 0 .. 64 + 5 * 14 * 64 */
    if (idx >= 64 + 5 * NPAIR * 64) return;
    uint16_t h[8];
    u32x4* dst;
    if (idx < 64) {
        const int l = idx, n = l & 15, g = l >> 4;
        for (int j = 0; j < 8; ++j) {
            const int k = g * 8 + j;
            h[j] = k < NT ? f2bf(P[OFF_W1 + k * CH + n]) : (uint16_t)0;
        }
        dst = W1p + l;
    } else if (idx >= 64 + 4 * NPAIR * 64) {
        /* layer 4: bf16(W4[tap][cin]) in output columns 0-7, the bf16 remainder in columns 8-15 */
        const int q = idx - 64 - 4 * NPAIR * 64;
        const int p = q / 64, l = q % 64, n = l & 15, g = l >> 4;
        const int tap = pair_tap(p, g >> 1), c0 = (g & 1) * 8;
        for (int j = 0; j < 8; ++j) {
            const float wv = tap < NT ? P[OFF_W4 + tap * CH + c0 + j] : 0.0f;
            const uint16_t hi = f2bf(wv);
            h[j] = n < 8 ? hi : f2bf(wv - bf2f(hi));
        }
        dst = W4p + q;
    } else {
        const int r = idx - 64;
        const int which = r / (NPAIR * 64), q = r % (NPAIR * 64);
        const int p = q / 64, l = q % 64, n = l & 15, g = l >> 4;
        const int tap = pair_tap(p, g >> 1), c0 = (g & 1) * 8;
        const int offw = (which == 0 || which == 2) ? OFF_W2 : OFF_W3;
        const bool transposed = which >= 2;
        for (int j = 0; j < 8; ++j) {
            const int cin = c0 + j;
            float wv = 0.0f;
            if (tap < NT) {
                /* forward: W[tap][cin][n]; input gradient: W[26 - tap][n][cin] */
                wv = transposed ? P[offw + ((NT - 1 - tap) * CH + n) * CH + cin] : P[offw + (tap * CH + cin) * CH + n];
            }
            h[j] = f2bf(wv);
        }
        dst = (which == 0 ? W2p : which == 1 ? W3p : which == 2 ? W2t : W3t) + p * 64 + l;
    }
    *dst = (u32x4){pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7])};
}

/* tiles of side s = size + 2 * halo starting at (origin - halo), reflect-padded, divided by scale; tiles along
   the grid's y */
template <typename T>
__global__ void k_extract(const T* __restrict__ img, int64_t yn, int64_t xn, int64_t zn, const int* __restrict__ org, int ntiles, int s, int halo,
                          float inv_scale, float* out) {
    const int64_t nv = (int64_t)s * s * s;
    for (int t = blockIdx.y; t < ntiles; t += gridDim.y) {
        for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += (int64_t)gridDim.x * blockDim.x) {
            const uint32_t v = (uint32_t)i, row = v / (uint32_t)s, y = v - row * (uint32_t)s, z = row / (uint32_t)s, x = row - z * (uint32_t)s;
            const int64_t gy = refl_any((int64_t)org[3 * t] - halo + y, yn);
            const int64_t gx = refl_any((int64_t)org[3 * t + 1] - halo + x, xn);
            const int64_t gz = refl_any((int64_t)org[3 * t + 2] - halo + z, zn);
            out[t * nv + i] = (float)img[(gz * xn + gx) * yn + gy] * inv_scale;
        }
    }
}

template <typename T>
__global__ __launch_bounds__(256) void k_sum(const T* __restrict__ v, size_t n, double* part) {
    __shared__ double red[256];
    double s = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) s += (double)v[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

const dim3 kBlk(256);

}  // namespace

}  // namespace aprh

/* ======================================================================== */

struct aprh_cnn {
    aprh_context* ctx = nullptr;
    aprh::Buf P, M, V, G;                        /* params, Adam moments, gradient (f32) */
    aprh::Buf W1p, W2p, W3p, W2t, W3t, W4p;      /* packed bf16 weights                  */
    int step = 0;
    float last_loss = 0;
    /* Gaussian applied to the warm-start particles (sizes 1: none) */
    float post_sigma[3] = {0.0f, 0.0f, 0.0f};
    int32_t post_size[3] = {1, 1, 1};
};

namespace aprh {

namespace {

/* blocks of the weight-gradient kernels, one partial each: two waves on each SIMD (k_dw holds 27
   accumulators), or as many as fit for the light first layer */
constexpr int DW_BLOCKS = 512, DW1_BLOCKS = 2048;
/* rows along x of one k_dw item: the two rows loaded ahead of it stay a small share, and 16 tiles of
   64^3 give each wave about 8 items */
constexpr int DW_ROWS = 16;

/* the bricks of T tiles of output side s, and a grid of at most cap blocks over them */
struct Bricks {
    uint32_t n, ny, nx, nz;
    unsigned grid;
};
/* one layer of a pass over an image's tiles: their wanted bricks */
struct LayerBricks {
    BrickMap map;
    int64_t n;
};
Bricks bricks(int T, int s, int64_t cap, const LayerBricks* wanted = nullptr) {
    Bricks b;
    b.ny = (uint32_t)cdiv(s, BY);
    b.nx = (uint32_t)cdiv(s, BX);
    b.nz = (uint32_t)cdiv(s, BZ);
    const int64_t n = wanted ? wanted->n : (int64_t)T * b.ny * b.nx * b.nz;
    if (n > 0x7FFFFFFF) throw Error(APRH_ERR_INVALID_ARGUMENT, "too many tiles in one network pass");
    b.n = (uint32_t)n;
    b.grid = (unsigned)std::min<int64_t>(n, cap);
    return b;
}

/* 16 -> 16 convolution of T tiles (input side sin, output side sout, input offset off) */
void conv16(hipStream_t st, const uint16_t* in_cl, int sin, int sout, int off, const u32x4* Wp, const float* bias,
            const uint16_t* mask_cl, uint16_t* out_cl, uint16_t* out_pl, int relu, int T, const LayerBricks* wanted = nullptr) {
    const Bricks b = bricks(T, sout, 65536, wanted);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(b.grid), kBlk, 0, st, in_cl, sin, sout, off, Wp, bias, mask_cl, out_cl, out_pl, relu, b.n, b.ny, b.nx, b.nz,
                           wanted ? wanted->map : BrickMap());
    };
    if (off == 0) launch(k_conv16_lds<true>);
    else launch(k_conv16_lds<false>);
    HIP_LAUNCH_CHECK();
}

void pack(aprh_cnn* n) {
    hipLaunchKernelGGL(k_pack, dim3((64 + 5 * NPAIR * 64 + 255) / 256), kBlk, 0, n->ctx->stream, n->P.as<float>(), n->W1p.as<u32x4>(),
                       n->W2p.as<u32x4>(), n->W3p.as<u32x4>(), n->W2t.as<u32x4>(), n->W3t.as<u32x4>(), n->W4p.as<u32x4>());
    HIP_LAUNCH_CHECK();
}

struct Acts {
    Buf a1c, a1p, a2c, a2p, a3c, a3p;
};

/* blocks of the layer-4 kernel (one loss partial each) */
int l4_blocks(int T, int S) { return (int)bricks(T, S, 4096).grid; }

/* forward of T tiles (input side S + 8); planar copies when training; part holds l4_blocks(T, S)
   pairs of loss partials.  With an image (dt its type) the tiles at vol->org are read from it and written
   to its output instead of x and y, at the layers' wanted bricks */
void forward(aprh_cnn* n, const float* x, int T, int S, float* y, Acts& A, bool train, const float* tgt, float* g4, double* part,
             const Volume* vol = nullptr, int dt = APRH_DTYPE_F32, const LayerBricks* wanted = nullptr) {
    hipStream_t st = n->ctx->stream;
    const int s0 = S + 8, s1 = S + 6, s2 = S + 4, s3 = S + 2;
    auto vox = [&](int s) { return (size_t)T * s * s * s; };
    A.a1c.reset(n->ctx->pool, vox(s1) * CH * 2);
    A.a2c.reset(n->ctx->pool, vox(s2) * CH * 2);
    A.a3c.reset(n->ctx->pool, vox(s3) * CH * 2);
    if (train) {
        A.a1p.reset(n->ctx->pool, vox(s1) * CH * 2 + PL_PAD);
        A.a2p.reset(n->ctx->pool, vox(s2) * CH * 2 + PL_PAD);
        A.a3p.reset(n->ctx->pool, vox(s3) * CH * 2 + PL_PAD);
    }
    const Volume v = vol ? *vol : Volume();
    auto layer = [&](int k) { return wanted ? wanted + k : nullptr; };
    auto map = [&](int k) { return wanted ? wanted[k].map : BrickMap(); };
    const float* P = n->P.as<float>();
    {
        const Bricks b = bricks(T, s1, 65536, layer(0));
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(b.grid), kBlk, 0, st, x, s0, s1, (const u32x4*)n->W1p.as<u32x4>(), P + OFF_B1, A.a1c.as<uint16_t>(),
                               train ? A.a1p.as<uint16_t>() : (uint16_t*)nullptr, b.n, b.ny, b.nx, b.nz, map(0), v);
        };
        if (!vol) launch(k_l1_lds<float, false>);
        else if (dt == APRH_DTYPE_U16) launch(k_l1_lds<uint16_t, true>);
        else launch(k_l1_lds<float, true>);
        HIP_LAUNCH_CHECK();
    }
    conv16(st, A.a1c.as<uint16_t>(), s1, s2, 0, n->W2p.as<u32x4>(), P + OFF_B2, nullptr, A.a2c.as<uint16_t>(),
           train ? A.a2p.as<uint16_t>() : nullptr, 1, T, layer(1));
    conv16(st, A.a2c.as<uint16_t>(), s2, s3, 0, n->W3p.as<u32x4>(), P + OFF_B3, nullptr, A.a3c.as<uint16_t>(),
           train ? A.a3p.as<uint16_t>() : nullptr, 1, T, layer(2));
    const Bricks b4 = bricks(T, S, vol ? 65536 : 4096, layer(3));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(b4.grid), kBlk, 0, st, (const uint16_t*)A.a3c.as<uint16_t>(), S, x, (const u32x4*)n->W4p.as<u32x4>(),
                           P + OFF_B4, tgt, y, g4, 1.0f / (float)vox(S), part, b4.n, b4.ny, b4.nx, b4.nz, map(3), v);
    };
    if (!vol) launch(k_l4_lds<float, false>);
    else if (dt == APRH_DTYPE_U16) launch(k_l4_lds<uint16_t, true>);
    else launch(k_l4_lds<float, true>);
    HIP_LAUNCH_CHECK();
}

void train_step(aprh_cnn* n, const float* x, const float* tgt, int T, int S, float lr, float* loss_out, float* grads_out) {
    hipStream_t st = n->ctx->stream;
    Pool* pool = n->ctx->pool;
    const int s1 = S + 6, s2 = S + 4, s3 = S + 2;
    auto vox = [&](int s) { return (size_t)T * s * s * s; };
    const int nblk_l4 = l4_blocks(T, S);
    Buf y(pool, vox(S) * 4), g4(pool, vox(S) * 4), part(pool, (size_t)nblk_l4 * 2 * 8);
    Acts A;
    forward(n, x, T, S, y.as<float>(), A, true, tgt, g4.as<float>(), part.as<double>());
    float* G = n->G.as<float>();
    const float* P = n->P.as<float>();
    /* loss and db4 */
    Buf dloss(pool, 4);
    hipLaunchKernelGGL(k_loss, dim3(1), kBlk, 0, st, dloss.as<float>(), G + OFF_B4, (const double*)part.as<double>(), nblk_l4,
                       1.0 / (double)vox(S));
    HIP_LAUNCH_CHECK();
    /* layer 4 */
    Buf g3c(pool, vox(s3) * CH * 2), g3p(pool, vox(s3) * CH * 2 + PL_PAD);
    hipLaunchKernelGGL(k_l4_bwd, dim3((unsigned)std::min<size_t>((vox(s3) + 255) / 256, 8192)), kBlk, 0, st, (const float*)g4.as<float>(), S,
                       P + OFF_W4, (const uint16_t*)A.a3c.as<uint16_t>(), g3c.as<uint16_t>(), g3p.as<uint16_t>(), T);
    HIP_LAUNCH_CHECK();
    Buf pbuf(pool, (size_t)std::max<int64_t>((int64_t)DW_BLOCKS * (NT * 256 + CH), (int64_t)DW1_BLOCKS * (NT * CH + CH)) * 4);
    auto reduce = [&](int64_t nparts, int count, int off) {
        hipLaunchKernelGGL(k_reduce_parts, dim3((unsigned)cdiv(count, 16)), kBlk, 0, st, (const float*)pbuf.as<float>(), nparts, count, G, off);
        HIP_LAUNCH_CHECK();
    };
    /* weight gradients of a layer over gradients of side sg, into G + off */
    auto dw = [&](const Buf& act, const Buf& grad, int sg, bool one, int off) {
        const int nseg = (int)cdiv(sg, DW_ROWS);
        const int64_t items = (int64_t)T * sg * nseg * cdiv(sg, 32);
        const unsigned grid = (unsigned)std::min<int64_t>(DW_BLOCKS, cdiv(items, 4));
        if (one)
            hipLaunchKernelGGL(k_dw<true>, dim3(grid), kBlk, 0, st, (const uint16_t*)act.as<uint16_t>(), (const void*)grad.ptr(), sg, DW_ROWS,
                               nseg, items, pbuf.as<float>());
        else
            hipLaunchKernelGGL(k_dw<false>, dim3(grid), kBlk, 0, st, (const uint16_t*)act.as<uint16_t>(), (const void*)grad.ptr(), sg, DW_ROWS,
                               nseg, items, pbuf.as<float>());
        HIP_LAUNCH_CHECK();
        reduce(grid, one ? NT * CH : NT * 256 + CH, off);
    };
    dw(A.a3p, g4, S, true, OFF_W4);
    /* layer 3 weights, then the gradient of a2 */
    dw(A.a2p, g3p, s3, false, OFF_W3);
    Buf g2c(pool, vox(s2) * CH * 2), g2p(pool, vox(s2) * CH * 2 + PL_PAD);
    conv16(st, g3c.as<uint16_t>(), s3, s2, -2, n->W3t.as<u32x4>(), nullptr, A.a2c.as<uint16_t>(), g2c.as<uint16_t>(), g2p.as<uint16_t>(),
           0, T);
    /* layer 2 weights, then the gradient of a1 */
    dw(A.a1p, g2p, s2, false, OFF_W2);
    Buf g1p(pool, vox(s1) * CH * 2 + PL_PAD);
    conv16(st, g2c.as<uint16_t>(), s2, s1, -2, n->W2t.as<u32x4>(), nullptr, A.a1c.as<uint16_t>(), nullptr, g1p.as<uint16_t>(), 0, T);
    /* layer 1: its bias gradient follows its weights' in the partials as in the parameters */
    static_assert(OFF_B1 == OFF_W1 + NT * CH && OFF_B2 == OFF_W2 + NT * 256 && OFF_B3 == OFF_W3 + NT * 256, "bias after weights");
    const unsigned grid1 = (unsigned)std::min<int64_t>(DW1_BLOCKS, cdiv((int64_t)T * s1 * s1 * cdiv(s1, 32), 4));
    hipLaunchKernelGGL(k_dw_l1, dim3(grid1), kBlk, 0, st, x, (const uint16_t*)g1p.as<uint16_t>(), S, pbuf.as<float>(), T);
    HIP_LAUNCH_CHECK();
    reduce(grid1, NT * CH + CH, OFF_W1);
    if (grads_out) HIP_CHECK(hipMemcpyAsync(grads_out, G, N_PARAMS * 4, hipMemcpyDeviceToHost, st));
    if (lr > 0) {
        n->step += 1;
        const float b1 = 0.9f, b2 = 0.999f;
        const float bc1 = 1.0f - std::pow(b1, (float)n->step), bc2 = 1.0f - std::pow(b2, (float)n->step);
        hipLaunchKernelGGL(k_adam, dim3((N_PARAMS + 255) / 256), kBlk, 0, st, n->P.as<float>(), (const float*)G, n->M.as<float>(),
                           n->V.as<float>(), N_PARAMS, lr, b1, b2, 1e-8f, bc1, bc2);
        HIP_LAUNCH_CHECK();
        pack(n);
    }
    float loss = 0;
    HIP_CHECK(hipMemcpyAsync(&loss, dloss.ptr(), 4, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    n->last_loss = loss;
    if (loss_out) *loss_out = loss;
}

double device_mean(aprh_context* ctx, const void* v, int dt, size_t n) {
    const int nb = 1024;
    Buf part(ctx->pool, nb * 8);
    if (dt == APRH_DTYPE_U16)
        hipLaunchKernelGGL(k_sum<uint16_t>, dim3(nb), kBlk, 0, ctx->stream, (const uint16_t*)v, n, part.as<double>());
    else
        hipLaunchKernelGGL(k_sum<float>, dim3(nb), kBlk, 0, ctx->stream, (const float*)v, n, part.as<double>());
    HIP_LAUNCH_CHECK();
    std::vector<double> h(nb);
    HIP_CHECK(hipMemcpyAsync(h.data(), part.ptr(), nb * 8, hipMemcpyDeviceToHost, ctx->stream));
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    double s = 0;
    for (double d : h) s += d;
    return n ? s / (double)n : 0.0;
}

/* the wanted bricks of layer l along an axis of n voxels in tiles of side S, of which the output is wanted
   e = 6 - 2 l voxels past the axis' end */
int64_t bricks_along(int64_t n, int S, int l, int b) {
    const int e = 6 - 2 * l;
    const int64_t tiles = cdiv(n, S);
    return (tiles - 1) * cdiv(S + e, b) + cdiv(n - (tiles - 1) * S + e, b);
}

/* tiles per batch: their activations (32 bytes a voxel and layer) are to stay in the 256 MB cache from one layer
   to the next (512 x 500 x 130 in 74^3 tiles, 6 / 16 / 32 a batch: 3.99 / 3.62 / 3.68 ms) */
int tiles_per_batch(int S) { return (int)std::max<int64_t>(1, std::min<int64_t>(64, (int64_t)16 * 74 * 74 * 74 / ((int64_t)S * S * S))); }

/* The side of the tiles.  Every output depends on its own neighbourhood alone, so it is free; what counts is the
   bricks of 16 x 8 x 4 that the layers need, which overhang the tiles' and the image's ends.  Their cost, per
   brick as measured in ns, and 20 us of each batch's launches and last waves decide: 128^3 takes one tile
   (0.23 ms; 74^3 tiles 0.26, 64^3 tiles 0.25), 512 x 500 x 130 takes 136^3 (3.23 ms; 74^3 3.39), 333 x 250 x 77
   138^3 (0.70 ms; 74^3 0.76). */
int tile_side(int64_t yn, int64_t xn, int64_t zn) {
    constexpr double ns[4] = {6.5, 10.7, 10.7, 13.0};
    int best = 0;
    double least = 0;
    for (int S = 32; S <= 138; S += 2) {
        double cost = 20000.0 * (double)cdiv(cdiv(yn, S) * cdiv(xn, S) * cdiv(zn, S), tiles_per_batch(S));
        for (int l = 0; l < 4; ++l)
            cost += ns[l] * (double)bricks_along(yn, S, l, BY) * (double)bricks_along(xn, S, l, BX) * (double)bricks_along(zn, S, l, BZ);
        if (best == 0 || cost < least) {
            best = S;
            least = cost;
        }
    }
    return best;
}

/* the network over a whole volume in tiles; out = y * scale (floored) */
void apply_volume(aprh_cnn* n, const void* img, int dt, int64_t yn, int64_t xn, int64_t zn, float scale, float floor_v, float* out) {
    hipStream_t st = n->ctx->stream;
    Pool* pool = n->ctx->pool;
    const int S = tile_side(yn, xn, zn);
    const int ty = (int)cdiv(yn, S), tx = (int)cdiv(xn, S), tz = (int)cdiv(zn, S);
    const int ntiles = ty * tx * tz;
    const bool whole = yn % S == 0 && xn % S == 0 && zn % S == 0;   /* all tiles alike */
    const int B = tiles_per_batch(S);   /* at most 64: wanted_brick looks a tile up in one wave */
    /* per layer and tile the wanted bricks (layer l's output is wanted 6 - 2 l voxels past the image's end), then
       the tiles' origins */
    std::vector<int4> tab((size_t)ntiles * 4);
    std::vector<int> org((size_t)ntiles * 3);
    std::vector<int64_t> count((size_t)cdiv(ntiles, B) * 4, 0);
    for (int k = 0, z = 0; z < tz; ++z)
        for (int x = 0; x < tx; ++x)
            for (int y = 0; y < ty; ++y, ++k) {
                org[3 * k] = y * S;
                org[3 * k + 1] = x * S;
                org[3 * k + 2] = z * S;
                for (int l = 0; l < 4; ++l) {
                    const int e = 6 - 2 * l;
                    auto along = [&](int64_t n, int o, int b) { return (int)cdiv(std::min<int64_t>(S, n - o) + e, b); };
                    int64_t& c = count[(size_t)(k / B) * 4 + l];
                    const int4 q = make_int4((int)c, along(yn, y * S, BY), along(xn, x * S, BX), along(zn, z * S, BZ));
                    tab[(size_t)l * ntiles + k] = q;
                    c += (int64_t)q.y * q.z * q.w;
                }
            }
    std::vector<uint8_t> host(tab.size() * 16 + org.size() * 4);
    std::memcpy(host.data(), tab.data(), tab.size() * 16);
    std::memcpy(host.data() + tab.size() * 16, org.data(), org.size() * 4);
    Buf dev(pool, host.size());
    HIP_CHECK(hipMemcpyAsync(dev.ptr(), host.data(), host.size(), hipMemcpyHostToDevice, st));
    const int4* dtab = dev.as<int4>();
    const int* dorg = (const int*)(dtab + tab.size());
    for (int t0 = 0; t0 < ntiles; t0 += B) {
        const int T = std::min(B, ntiles - t0);
        const Volume vol{img, yn, xn, zn, dorg + 3 * t0, 1.0f / scale, scale, floor_v, out};
        LayerBricks wanted[4];
        for (int l = 0; l < 4 && !whole; ++l)
            wanted[l] = {{dtab + (size_t)l * ntiles + t0, T}, count[(size_t)(t0 / B) * 4 + l]};
        Acts A;
        forward(n, nullptr, T, S, nullptr, A, false, nullptr, nullptr, nullptr, &vol, dt, whole ? nullptr : wanted);
    }
    HIP_CHECK(hipStreamSynchronize(st));
}

}  // namespace

}  // namespace aprh

using namespace aprh;

namespace {
void check_cnn(aprh_context* ctx, aprh_cnn* n) {
    check_ctx(ctx);
    if (!n) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL network");
    if (n->ctx != ctx) throw Error(APRH_ERR_INVALID_ARGUMENT, "network belongs to another context");
}
void check_tile_size(int S) {
    if (S < 1 || S > 128) throw Error(APRH_ERR_INVALID_ARGUMENT, "tile side must be in 1..128");
}
}  // namespace

extern "C" {

int aprh_cnn_param_count(void) { return N_PARAMS; }

int aprh_cnn_create(aprh_context* ctx, uint64_t seed, aprh_cnn** out) {
    APRH_TRY
    check_ctx(ctx);
    if (!out) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL out");
    aprh_cnn* n = new aprh_cnn();
    n->ctx = ctx;
    try {
        n->P.reset(ctx->pool, N_PARAMS * 4);
        n->M.reset(ctx->pool, N_PARAMS * 4);
        n->V.reset(ctx->pool, N_PARAMS * 4);
        n->G.reset(ctx->pool, N_PARAMS * 4);
        n->W1p.reset(ctx->pool, 64 * 16);
        n->W2p.reset(ctx->pool, NPAIR * 64 * 16);
        n->W3p.reset(ctx->pool, NPAIR * 64 * 16);
        n->W2t.reset(ctx->pool, NPAIR * 64 * 16);
        n->W3t.reset(ctx->pool, NPAIR * 64 * 16);
        n->W4p.reset(ctx->pool, NPAIR * 64 * 16);
        /* He initialisation for layers 1-3, small last layer (the network starts near the identity) */
        std::mt19937_64 rng(seed);
        std::vector<float> p(N_PARAMS, 0.0f);
        std::normal_distribution<float> n1(0.0f, std::sqrt(2.0f / 27.0f)), n2(0.0f, std::sqrt(2.0f / 432.0f)), n4(0.0f, 1e-3f);
        for (int i = OFF_W1; i < OFF_B1; ++i) p[i] = n1(rng);
        for (int i = OFF_W2; i < OFF_B2; ++i) p[i] = n2(rng);
        for (int i = OFF_W3; i < OFF_B3; ++i) p[i] = n2(rng);
        for (int i = OFF_W4; i < OFF_B4; ++i) p[i] = n4(rng);
        HIP_CHECK(hipMemcpyAsync(n->P.ptr(), p.data(), N_PARAMS * 4, hipMemcpyHostToDevice, ctx->stream));
        HIP_CHECK(hipMemsetAsync(n->M.ptr(), 0, N_PARAMS * 4, ctx->stream));
        HIP_CHECK(hipMemsetAsync(n->V.ptr(), 0, N_PARAMS * 4, ctx->stream));
        HIP_CHECK(hipMemsetAsync(n->G.ptr(), 0, N_PARAMS * 4, ctx->stream));
        pack(n);
        HIP_CHECK(hipStreamSynchronize(ctx->stream));
    } catch (...) {
        delete n;
        throw;
    }
    *out = n;
    APRH_CATCH
}

int aprh_cnn_destroy(aprh_cnn* n) {
    APRH_TRY
    if (!n) return APRH_OK;
    (void)hipSetDevice(n->ctx->device);
    (void)hipStreamSynchronize(n->ctx->stream);
    delete n;
    APRH_CATCH
}

int aprh_cnn_get_params(aprh_context* ctx, aprh_cnn* n, float* out) {
    APRH_TRY
    check_cnn(ctx, n);
    if (!out) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL out");
    copy_any(ctx, out, n->P.ptr(), N_PARAMS * 4);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    APRH_CATCH
}

int aprh_cnn_set_params(aprh_context* ctx, aprh_cnn* n, const float* in) {
    APRH_TRY
    check_cnn(ctx, n);
    if (!in) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL params");
    copy_any(ctx, n->P.ptr(), in, N_PARAMS * 4);
    HIP_CHECK(hipMemsetAsync(n->M.ptr(), 0, N_PARAMS * 4, ctx->stream));
    HIP_CHECK(hipMemsetAsync(n->V.ptr(), 0, N_PARAMS * 4, ctx->stream));
    n->step = 0;
    pack(n);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    APRH_CATCH
}

int aprh_cnn_forward_tiles(aprh_context* ctx, aprh_cnn* n, const float* in, int32_t T, int32_t S, float* out) {
    APRH_TRY
    check_cnn(ctx, n);
    check_tile_size(S);
    if (!in || !out || T < 1) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad tiles");
    const size_t ni = (size_t)T * (S + 8) * (S + 8) * (S + 8), no = (size_t)T * S * S * S;
    DevIn x(ctx, in, ni * 4);
    DevOut y(ctx, out, no * 4);
    Acts A;
    forward(n, (const float*)x.ptr, T, S, (float*)y.ptr, A, false, nullptr, nullptr, nullptr);
    y.finish(ctx);
    APRH_CATCH
}

int aprh_cnn_train_step(aprh_context* ctx, aprh_cnn* n, const float* in, const float* target, int32_t T, int32_t S, float lr, float* loss,
                        float* grads_out) {
    APRH_TRY
    check_cnn(ctx, n);
    check_tile_size(S);
    if (!in || !target || T < 1 || lr < 0) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad training batch");
    const size_t ni = (size_t)T * (S + 8) * (S + 8) * (S + 8), no = (size_t)T * S * S * S;
    DevIn x(ctx, in, ni * 4), t(ctx, target, no * 4);
    float* gh = nullptr;
    std::vector<float> gbuf;
    if (grads_out) {
        gbuf.resize(N_PARAMS);
        gh = gbuf.data();
    }
    train_step(n, (const float*)x.ptr, (const float*)t.ptr, T, S, lr, loss, gh);
    if (grads_out) copy_any(ctx, grads_out, gbuf.data(), N_PARAMS * 4);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
    APRH_CATCH
}

int aprh_cnn_extract_tiles(aprh_context* ctx, const void* image, int dtype, int64_t y, int64_t x, int64_t z, const int32_t* origins,
                           int32_t T, int32_t size, int32_t halo, float scale, float* out) {
    APRH_TRY
    check_ctx(ctx);
    if (!image || !origins || !out || T < 1 || size < 1 || halo < 0 || !(scale > 0) || y < 1 || x < 1 || z < 1)
        throw Error(APRH_ERR_INVALID_ARGUMENT, "bad tile extraction");
    if (dtype != APRH_DTYPE_U16 && dtype != APRH_DTYPE_F32) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad dtype");
    const int s = size + 2 * halo;
    const size_t n = (size_t)(y * x * z);
    DevIn im(ctx, image, n * (dtype == APRH_DTYPE_U16 ? 2 : 4));
    DevIn org(ctx, origins, (size_t)T * 3 * 4);
    DevOut o(ctx, out, (size_t)T * s * s * s * 4);
    const dim3 grid((unsigned)std::min<int64_t>(cdiv((int64_t)s * s * s, 256), 8192), (unsigned)std::min(T, 65535));
    if (dtype == APRH_DTYPE_U16)
        hipLaunchKernelGGL(k_extract<uint16_t>, grid, kBlk, 0, ctx->stream, (const uint16_t*)im.ptr, y, x, z, (const int*)org.ptr, T, s, halo,
                           1.0f / scale, (float*)o.ptr);
    else
        hipLaunchKernelGGL(k_extract<float>, grid, kBlk, 0, ctx->stream, (const float*)im.ptr, y, x, z, (const int*)org.ptr, T, s, halo,
                           1.0f / scale, (float*)o.ptr);
    HIP_LAUNCH_CHECK();
    o.finish(ctx);
    APRH_CATCH
}

int aprh_mean(aprh_context* ctx, const void* data, int dtype, uint64_t n, double* mean) {
    APRH_TRY
    check_ctx(ctx);
    if (!data || !mean || (dtype != APRH_DTYPE_U16 && dtype != APRH_DTYPE_F32)) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad arguments");
    DevIn d(ctx, data, std::max<uint64_t>(n, 1) * (dtype == APRH_DTYPE_U16 ? 2 : 4));
    *mean = device_mean(ctx, d.ptr, dtype, n);
    APRH_CATCH
}

int aprh_cnn_apply(aprh_context* ctx, aprh_cnn* n, const void* image, int dtype, int64_t y, int64_t x, int64_t z, float scale, float* out) {
    APRH_TRY
    check_cnn(ctx, n);
    if (!image || !out || y < 1 || x < 1 || z < 1) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad arguments");
    if (dtype != APRH_DTYPE_U16 && dtype != APRH_DTYPE_F32) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad dtype");
    const size_t nv = (size_t)(y * x * z);
    DevIn im(ctx, image, nv * (dtype == APRH_DTYPE_U16 ? 2 : 4));
    DevOut o(ctx, out, nv * 4);
    if (!(scale > 0)) scale = (float)device_mean(ctx, im.ptr, dtype, nv);
    if (!(scale > 0)) scale = 1.0f;
    /* tiles read their neighbours' voxels while finished ones are written: in place needs a copy of the image */
    const size_t bytes = nv * (dtype == APRH_DTYPE_U16 ? 2 : 4);
    const void* src = im.ptr;
    Buf copy;
    if ((const char*)src < (const char*)o.ptr + nv * 4 && (const char*)o.ptr < (const char*)src + bytes) {
        copy.reset(ctx->pool, bytes);
        HIP_CHECK(hipMemcpyAsync(copy.ptr(), src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
        src = copy.ptr();
    }
    apply_volume(n, src, dtype, y, x, z, scale, -INFINITY, (float*)o.ptr);
    o.finish(ctx);
    APRH_CATCH
}

int aprh_cnn_warm_start(aprh_context* ctx, aprh_cnn* n, aprh_apr* a, const void* parts, int dtype, float* u0) {
    APRH_TRY
    check_cnn(ctx, n);
    if (!a || !parts || !u0) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL argument");
    if (dtype != APRH_DTYPE_U16 && dtype != APRH_DTYPE_F32) throw Error(APRH_ERR_INVALID_ARGUMENT, "bad dtype");
    const int64_t yn = a->org[0], xn = a->org[1], zn = a->org[2];
    const size_t nv = (size_t)(yn * xn * zn);
    DevIn p(ctx, parts, std::max<uint64_t>(a->total, 1) * (dtype == APRH_DTYPE_U16 ? 2 : 4));
    DevOut u(ctx, u0, std::max<uint64_t>(a->total, 1) * 4);
    Buf rec(ctx->pool, nv * 4), pred(ctx->pool, nv * 4);
    /* piecewise-constant image of the particles (APRReconstruction::reconstruct_constant) */
    reconstruct_any(ctx, *a, p.ptr, dtype, a->l_max, rec.ptr(), APRH_DTYPE_F32);
    float scale = (float)device_mean(ctx, rec.ptr(), APRH_DTYPE_F32, nv);
    if (!(scale > 0)) scale = 1.0f;
    /* the estimate must stay positive for the multiplicative updates */
    apply_volume(n, rec.ptr(), APRH_DTYPE_F32, yn, xn, zn, scale, 1e-3f * scale, pred.as<float>());
    launch_sample_f32(ctx, *a, pred.as<float>(), (float*)u.ptr);
    if (n->post_size[0] * n->post_size[1] * n->post_size[2] > 1 && a->total > 0) {
        /* the post filter: APRFilter::convolve_pencil of the estimate with a normalised Gaussian
           (downsampled per level, reflected boundary) */
        HostStencil hs;
        hs.sy = n->post_size[0];
        hs.sx = n->post_size[1];
        hs.sz = n->post_size[2];
        hs.w.assign((size_t)(hs.sy * hs.sx * hs.sz), 0.0f);
        if (aprh_gaussian_stencil(n->post_sigma, n->post_size, 1, hs.w.data()) != APRH_OK)
            throw Error(APRH_ERR_INVALID_ARGUMENT, "post filter stencil");
        const std::vector<HostStencil> v = downsampled_stencils(hs, a->l_max - a->l_min, true);
        Buf tmp(ctx->pool, a->total * 4);
        convolve<float>(ctx, *a, v, (const float*)u.ptr, tmp.as<float>(), true);
        launch_copy(ctx, u.ptr, tmp.ptr(), a->total * 4);
    }
    u.finish(ctx);
    APRH_CATCH
}

int aprh_cnn_set_post_filter(aprh_cnn* n, const float* sigma3, const int32_t* size3) {
    APRH_TRY
    if (!n) throw Error(APRH_ERR_INVALID_ARGUMENT, "NULL network");
    if (!sigma3 || !size3) {
        for (int d = 0; d < 3; ++d) n->post_sigma[d] = 0.0f, n->post_size[d] = 1;
    } else {
        for (int d = 0; d < 3; ++d) {
            if (size3[d] < 1 || size3[d] > 15 || size3[d] % 2 == 0) throw Error(APRH_ERR_INVALID_ARGUMENT, "post filter sizes: odd, 1..15");
            if (size3[d] > 1 && !(sigma3[d] > 0.0f)) throw Error(APRH_ERR_INVALID_ARGUMENT, "post filter sigma must be positive");
        }
        for (int d = 0; d < 3; ++d) n->post_sigma[d] = sigma3[d], n->post_size[d] = size3[d];
    }
    APRH_CATCH
}

}  // extern "C"
