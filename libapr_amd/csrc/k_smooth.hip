/*
 * k_smooth.hip -- APRReconstruction::reconstruct_smooth (APRReconstruction.hpp:270-295).
 *
 * The piecewise-constant image is smoothed along y, x and z by running-sum means whose
 * half-width at a pixel is off = min(T(floor(2^(l_max - level) / scale)), T(offset_max))
 * (level = the level of the particle covering the pixel, offset_max = min(20, n/2 - 1))
 * -- calc_sat_adaptive_y / _x / _z (:528-876).
 *
 * The cumulative sums of a line are a sequential float recursion in the
 * reference's own order.  The reference keeps a ring of 2 offset_max + 2
 * cumulative rows for x and z; its entries are the prefix sums of the pass's
 * input (a ring slot is read only before it is reused).  The output of a pixel
 * then depends only on those sums, its own offset and its position: the
 * kernels apply the reference's sequence of stores for that pixel, converting
 * to the image type T at every store as the reference's assignments do
 * (float / double -> uint16 through int32 truncation, the x86-64 conversion).
 *
 * Each pass is one kernel that reads and writes the image once and keeps the
 * sums in LDS: whole lines along y, a ring of 2 offset_max + 2 sums per lane
 * along x and z.  A 512 x 480 x 200 f32 image, its reconstruction included:
 * 2.02 ms with the sums in a scratch image and a second kernel per pass, 0.64 ms
 * now.
 */
#include <type_traits>

#include "aprh_internal.hpp"

namespace aprh {

namespace {

__device__ __forceinline__ uint16_t sm_f2u16(float v) {
    if (!(v > -2147483648.0f && v < 2147483648.0f)) return 0;
    return (uint16_t)(int32_t)v;
}
__device__ __forceinline__ uint16_t sm_d2u16(double v) {
    if (!(v > -2147483648.0 && v < 2147483648.0)) return 0;
    return (uint16_t)(int32_t)v;
}

template <typename T> struct SmT;
template <> struct SmT<float> {
    static __device__ __forceinline__ float f(float v) { return v; }
    static __device__ __forceinline__ float d(double v) { return (float)v; }
};
template <> struct SmT<uint16_t> {
    static __device__ __forceinline__ uint16_t f(float v) { return sm_f2u16(v); }
    static __device__ __forceinline__ uint16_t d(double v) { return sm_d2u16(v); }
};

/* std::min((T)floor(pow(2, d_max - level) / scale), (T)offset_max) */
template <typename T>
__device__ __forceinline__ int sm_offset(int level, float scale, int om, int d_max) {
    const T a = SmT<T>::d(floor(ldexp(1.0, d_max - level) / (double)scale));
    const T b = (T)om;
    return max((int)(a < b ? a : b), 0);   /* never below 0, whatever the scale: the sums' indices stay inside */
}

/* half-widths by level, in LDS: the division is done once per level and block.  Levels are at most 16 (dims
   are at most 65535), and 0 where no particle covers the pixel */
constexpr int SM_LEVELS = 32;
template <typename T>
__device__ __forceinline__ void sm_offsets(int* tab, float scale, int om, int d_max) {
    if (threadIdx.x < SM_LEVELS) tab[threadIdx.x] = sm_offset<T>((int)threadIdx.x, scale, om, d_max);
    __syncthreads();
}

/* calc_sat_adaptive_y (APRReconstruction.hpp:528-646): the stores of pixel k in the reference's
   order; sum(i): the line's prefix sum at i, last: the one at yn - 1 */
template <typename T, typename Sum>
__device__ __forceinline__ T sm_pixel_y(const Sum& sum, float last, int k, int yn, int offi, int om) {
    const float off = (float)offi;
    const float div = 2 * off + 1;
    const float kf = (float)k;
    T s = (T)0;
    if (k >= 1 && k <= om + 1 && kf <= off + 1) s = SmT<T>::f(-sum(0) / div);
    if (kf >= off + 1) s = SmT<T>::f(-sum(k - offi - 1) / div);
    if (kf < (float)yn - off) s = SmT<T>::f((float)s + sum(k + offi) / div);
    if (k >= yn - om && kf >= (float)yn - off) {
        const float counter = kf - ((float)yn - off) + 1;
        s = SmT<T>::f((float)s * div);
        s = SmT<T>::f((float)s + last);
        s = SmT<T>::d((double)s * (1.0 / (double)(div - counter)));
    }
    if (k >= 1 && k < om + 1 && kf < off + 1) s = SmT<T>::d((double)s * ((double)div / (1.0 * k + (double)off)));
    if (k == 0) s = SmT<T>::f((float)s * (div / (off + 1)));
    return s;
}

/* y pass: a block takes nl whole lines into LDS, one lane per line runs the prefix sums in place, then
   all lanes form the outputs along y.  Bound by the sequential sums and the loads in front of them, so
   a block takes few lines (SM_Y_LDS bytes) and several blocks share a CU. */
constexpr int SM_Y_LDS = 24 * 1024, SM_Y_LDS_MAX = 144 * 1024;
template <typename T>
__global__ __launch_bounds__(256) void k_sm_y(T* __restrict__ m, const uint8_t* __restrict__ lev, int yn, int64_t nlines, int nl, int pitch,
                                              float scale, int om, int d_max) {
    extern __shared__ __align__(16) float lines[];
    __shared__ int offs[SM_LEVELS];
    sm_offsets<T>(offs, scale, om, d_max);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t line0 = (int64_t)blockIdx.x * nl;
    const int n = (int)min((int64_t)nl, nlines - line0);
    for (int l = wv; l < n; l += 4) {
        const T* src = m + (line0 + l) * yn;
#pragma unroll 4
        for (int k = lane; k < yn; k += 64) lines[l * pitch + k] = (float)src[k];
    }
    __syncthreads();
    if ((int)threadIdx.x < n) {
        float* t = lines + threadIdx.x * pitch;
        float s = 0.0f;
        int k = 0;
        for (; k + 16 <= yn; k += 16) {
            float v[16];
#pragma unroll
            for (int j = 0; j < 16; ++j) v[j] = t[k + j];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                s += v[j];
                t[k + j] = s;
            }
        }
        for (; k < yn; ++k) {
            s += t[k];
            t[k] = s;
        }
    }
    __syncthreads();
    for (int l = wv; l < n; l += 4) {
        const int64_t p = (line0 + l) * yn;
        const float* t = lines + l * pitch;
#pragma unroll 2
        for (int k = lane; k < yn; k += 64)
            m[p + k] = sm_pixel_y<T>([&](int i) { return t[i]; }, t[yn - 1], k, yn, offs[lev[p + k]], om);
    }
}

/* x pass (axis 1) and z pass (axis 2): lane = (outer line, y), marching along the axis with the last
   2 om + 2 prefix sums in an LDS ring (slot = index mod the ring's size, a column per lane, so lanes
   never share a slot and need no barrier); the output trails the sums by om.
   calc_sat_adaptive_x / _z (APRReconstruction.hpp:649-876): low end, middle and high end stores of
   pixel i, the later ones overriding; the z pass tests the x index at its low end, as the
   reference does (:821).  Eight samples ahead are loaded at a time.  YAX: the same march for the y
   pass (axis 0), for lines longer than the LDS holds (SM_Y_LDS_MAX). */
constexpr int SM_D = 8;
template <typename T, bool YAX>
__global__ __launch_bounds__(256) void k_sm_outer(T* m, const uint8_t* __restrict__ lev, int64_t yn, int64_t xn, int64_t zn, int axis,
                                                  float scale, int om, int d_max) {
    extern __shared__ __align__(16) float ring[];
    __shared__ int offs[SM_LEVELS];
    sm_offsets<T>(offs, scale, om, d_max);
    const int64_t lane = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t outer = YAX ? xn * zn : axis == 1 ? zn : xn, inner = YAX ? 1 : yn;
    if (lane >= outer * inner) return;
    const int64_t y = lane % inner, o = lane / inner;
    const int n = (int)(YAX ? yn : axis == 1 ? xn : zn);
    const int64_t stride = YAX ? 1 : axis == 1 ? yn : xn * yn;
    const int64_t base = (!YAX && axis == 1 ? o * xn * yn : o * yn) + y;
    const int R = 2 * om + 2;
    float* my = ring + threadIdx.x;
    float t = 0.0f;
    int w = 0;   /* ring slot of index j */
    auto load = [&](int j0, T (&v)[SM_D], uint8_t (&lv)[SM_D]) {
#pragma unroll
        for (int d = 0; d < SM_D; ++d) {
            const int j = j0 + d, i = j - om;
            v[d] = j < n ? m[base + j * stride] : (T)0;
            lv[d] = i >= 0 && i < n ? lev[base + i * stride] : (uint8_t)0;
        }
    };
    auto at = [&](int back) -> float {   /* the sum of index j - back, 0 <= back < R */
        int q = w - back;
        q = q < 0 ? q + R : q;
        return my[q * 256];
    };
    T cur[SM_D], nxt[SM_D];
    uint8_t lc[SM_D], ln[SM_D];
    load(0, cur, lc);
    for (int j0 = 0; j0 < n + om; j0 += SM_D) {
        load(j0 + SM_D, nxt, ln);
#pragma unroll
        for (int d = 0; d < SM_D; ++d) {
            const int j = j0 + d;
            if (j >= n + om) break;
            if (j < n) {
                t = (j == 0) ? (float)cur[d] : (float)cur[d] + t;
                my[w * 256] = t;
            }
            const int i = j - om;
            if (i >= 0) {
                const int off = offs[lc[d]];
                const int64_t lo_index = axis == 1 ? (int64_t)i : o;
                const int64_t p = base + i * stride;
                const bool low = i <= om && lo_index < off + 1, mid = i >= 1 && i >= off + 1 && i < n - off,
                           high = i >= n - om && i >= n - off;
                if constexpr (YAX) {
                    m[p] = sm_pixel_y<T>([&](int q) { return at(j - q); }, t, i, n, off, om);
                } else if (low || mid || high) {
                    /* one quotient: the last of the stores that apply */
                    float num, den;
                    if (high) {
                        num = t - at(om + off + 1);
                        den = (float)(n - i + off);
                    } else if (mid) {
                        num = at(om - off) - at(om + off + 1);
                        den = (float)(2 * off + 1);
                    } else {
                        num = at(om - off);
                        den = (float)(i + off + 1);
                    }
                    m[p] = SmT<T>::f(num / den);
                }
            }
            w = w + 1 == R ? 0 : w + 1;
        }
#pragma unroll
        for (int d = 0; d < SM_D; ++d) {
            cur[d] = nxt[d];
            lc[d] = ln[d];
        }
    }
}

template <typename T>
void smooth_passes(aprh_context* ctx, T* img, const uint8_t* lev, int64_t yn, int64_t xn, int64_t zn, const float* scale3, int offset_max,
                   int d_max) {
    hipStream_t st = ctx->stream;
    auto march = [&](auto yax, int axis, int64_t n, int64_t lanes) {
        constexpr bool YAX = decltype(yax)::value;
        const int om = std::min<int>(offset_max, (int)(n / 2 - 1));
        hipLaunchKernelGGL((k_sm_outer<T, YAX>), dim3((unsigned)cdiv(lanes, 256)), dim3(256), (size_t)(2 * om + 2) * 256 * 4, st, img, lev, yn, xn,
                           zn, axis, scale3[axis], om, d_max);
        HIP_LAUNCH_CHECK();
    };
    if (((yn | 1) * 4) > SM_Y_LDS_MAX) {
        march(std::true_type{}, 0, yn, xn * zn);
    } else if (yn > 1) {
        const int om = std::min<int>(offset_max, (int)(yn / 2 - 1));
        const int64_t lines = xn * zn;
        const int pitch = (int)yn | 1;   /* odd: the lanes' lines start on different banks */
        const int nl = (int)std::min<int64_t>(64, std::max<int64_t>(1, SM_Y_LDS / (4 * pitch)));
        const size_t lds = (size_t)nl * pitch * 4;
        if (lds > 65536)
            HIP_CHECK(hipFuncSetAttribute((const void*)k_sm_y<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k_sm_y<T>, dim3((unsigned)cdiv(lines, nl)), dim3(256), lds, st, img, lev, (int)yn, lines, nl, pitch, scale3[0], om,
                           d_max);
        HIP_LAUNCH_CHECK();
    }
    if (xn > 1) march(std::false_type{}, 1, xn, zn * yn);
    if (zn > 1) march(std::false_type{}, 2, zn, xn * yn);
}

}  // namespace

/* APRReconstruction::reconstruct_smooth: reconstruct_constant with the pixels' levels, then the
   adaptive means along y, x and z (offset_max 20, d_max = l_max) */
void reconstruct_smooth(aprh_context* ctx, aprh_apr& a, const void* parts, int pdt, const float* scale3, void* img, int idt) {
    const int L = a.l_max;
    const int64_t yn = a.y_num[L], xn = a.x_num[L], zn = a.z_num[L];
    const int64_t N = yn * xn * zn;
    if (N == 0) return;
    if (cdiv(xn * zn, 64) >= (int64_t(1) << 31) || xn * yn >= (int64_t(1) << 40))
        throw Error(APRH_ERR_UNSUPPORTED, "image too large for reconstruct_smooth");
    Buf lev(ctx->pool, (size_t)N);
    reconstruct_any(ctx, a, parts, pdt, L, img, idt, lev.as<uint8_t>());
    if (idt == APRH_DTYPE_U16) smooth_passes<uint16_t>(ctx, (uint16_t*)img, lev.as<uint8_t>(), yn, xn, zn, scale3, 20, L);
    else smooth_passes<float>(ctx, (float*)img, lev.as<uint8_t>(), yn, xn, zn, scale3, 20, L);
    HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

}  // namespace aprh
