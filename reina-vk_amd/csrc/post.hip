// post.hip — bloom and ACES-fitted tone mapping to RGBA8, in Reina's dispatch
// order (src/Reina.cpp:472-577):
//   blurX(rtImage -> ping, threshold)   shaders/postprocessing/bloom/blurX.comp.glsl:8
//   blurY(ping -> pong)                 shaders/postprocessing/bloom/blurY.comp.glsl:8
//   combine(rtImage, pong -> ping)      shaders/postprocessing/bloom/combine.comp.glsl:15-27
//   tonemap(ping -> out RGBA8)          shaders/postprocessing/tonemap/tonemapping.comp.glsl:41-84
// Kept from the reference: the Gaussian's sigma is the radius percentage
// itself while the half-width is 3 * size * radius / 100 pixels, and taps that
// are out of bounds or under the threshold still add to the weight sum; no
// sRGB encode. UNORM8 conversion: floor(c * 255 + 0.5).
//
// The blur's sums run over the taps in order with separate multiplies and
// adds (the result's bits depend on it), so its cost is 6 VALU operations per
// tap and pixel. Two kernels:
//   k_blur_row     blurX: one block per row, the thresholded row staged in LDS
//   k_blur_column  blurY, combine and tonemap: one lane per column, rows read
//                  straight from memory (64 columns = 1 KB per load)
// Both give a lane several neighbouring outputs, so a sample is loaded once
// for all of them, and take the weights from the kernel arguments (scalar
// registers). They leave out the taps whose weight is exactly zero: sigma is
// the percentage, so of the 577 taps of a 1920-pixel row at the default
// radius only the middle 145 have a weight that FP32 can hold. A zero weight
// adds nothing to a finite sum; a row or column window holding a non-finite
// value (zero times which is NaN) sums every tap (add_every_tap). 1920x1080,
// radius 5: blurX 1091 -> 58 us, blurY with combine and tonemap 620 -> 65 us
// (3.6 G operations of the weighted taps: 46 us each at one per lane and
// clock); 341x213: 38 -> 16 us. With a NaN in one row, or in every row, all of
// it: 1920x1080 1642 -> 167 and 281 us, 1080x1350 974 -> 138 and 203 us,
// 341x213 41 -> 28 and 31 us.
// k_blur and k_combine_tonemap, with the taps' weights in LDS, take the sizes
// those two do not (see launch_postprocess).
#include <hip/hip_runtime.h>

#include <cmath>

#include "rt_math.h"
#include "wavefront.h"

namespace rt {

constexpr int kTile = 256;        // output pixels per block along the blur axis
constexpr int kMaxHalf = 1024;    // LDS-staged half-width; larger kernels read HBM directly

RT_HD float gauss(float x, float sigma) { return expf_(((-x) * x) / ((2.0f * sigma) * sigma)); }

// axis 1 = X (along rows), 0 = Y (along columns)
template <int AXIS, bool THRESH>
__global__ __launch_bounds__(256) void k_blur(const float4* __restrict__ in, float4* __restrict__ out, uint32_t W,
                                              uint32_t H, BloomPushConsts b) {
    __shared__ float s_w[2 * kMaxHalf + 1];
    __shared__ float4 s_px[kTile + 2 * kMaxHalf];
    const uint32_t len = AXIS ? W : H;        // extent along the blur axis
    const uint32_t lines = AXIS ? H : W;
    const uint32_t line = blockIdx.y;
    const int32_t start = (int32_t)(blockIdx.x * kTile);
    if (line >= lines) return;
    float radiusPx = ((float)(int32_t)len * b.radius) / 100.0f;
    int32_t k = f2i_(radiusPx * 3.0f + 0.5f);
    bool staged = k <= kMaxHalf;
    if (staged) {
        for (int32_t t = threadIdx.x; t <= 2 * k; t += blockDim.x) s_w[t] = gauss((float)(t - k), b.radius);
        for (int32_t t = threadIdx.x; t < kTile + 2 * k; t += blockDim.x) {
            int32_t c = start - k + t;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (c >= 0 && c < (int32_t)len) {
                uint64_t idx = AXIS ? ((uint64_t)line * W + (uint32_t)c) : ((uint64_t)(uint32_t)c * W + line);
                v = in[idx];
            }
            s_px[t] = v;
        }
        __syncthreads();
    }
    int32_t pos = start + (int32_t)threadIdx.x;
    if (pos >= (int32_t)len) return;
    V3 c = v3(0.0f, 0.0f, 0.0f);
    float ws = 0.0f;
    for (int32_t i = -k; i <= k; ++i) {
        float w = staged ? s_w[i + k] : gauss((float)i, b.radius);
        ws = ws + w;
        int32_t cc = pos + i;
        if (cc < 0 || cc >= (int32_t)len) continue;
        float4 p;
        if (staged) {
            p = s_px[(int32_t)threadIdx.x + i + k];
        } else {
            uint64_t idx = AXIS ? ((uint64_t)line * W + (uint32_t)cc) : ((uint64_t)(uint32_t)cc * W + line);
            p = in[idx];
        }
        V3 rgb = v3(p.x, p.y, p.z);
        if (THRESH) {
            float lum = dot(rgb, v3(0.299f, 0.587f, 0.114f));
            if (lum < b.threshold) continue;
        }
        c = add(c, scale(rgb, w));
    }
    if (ws < 0.0001f) c = v3(0.0f, 0.0f, 0.0f);
    else c = divs(c, ws);
    uint64_t o = AXIS ? ((uint64_t)line * W + (uint32_t)pos) : ((uint64_t)(uint32_t)pos * W + line);
    out[o] = make_float4(c.x, c.y, c.z, 1.0f);
}

__device__ __forceinline__ float rrt1(float v) {
    float a = v * (v + 0.0245786f) - 0.000090537f;
    float bb = v * (0.983729f * v + 0.4329510f) + 0.238081f;
    return a / bb;
}

__device__ __forceinline__ uint32_t unorm8(float c) { return (uint32_t)f2i_(floorf(c * 255.0f + 0.5f)) & 0xFFu; }

// combine and tonemap of one pixel; scale = 2^exposure
__device__ __forceinline__ uchar4 combine_tonemap(float4 o, V3 bl, float intensity, float exposure_scale, float4& combined) {
    V3 c = v3(o.x + bl.x * intensity, o.y + bl.y * intensity, o.z + bl.z * intensity);
    combined = make_float4(c.x, c.y, c.z, 1.0f);
    const float e = exposure_scale;
    c = v3(c.x * e, c.y * e, c.z * e);
    c = v3(dot(c, v3(0.59719f, 0.35458f, 0.04823f)), dot(c, v3(0.07600f, 0.90834f, 0.01566f)),
           dot(c, v3(0.02840f, 0.13383f, 0.83777f)));
    c = v3(rrt1(c.x), rrt1(c.y), rrt1(c.z));
    c = v3(dot(c, v3(1.60475f, -0.53108f, -0.07367f)), dot(c, v3(-0.10208f, 1.10813f, -0.00605f)),
           dot(c, v3(-0.00327f, -0.07276f, 1.07602f)));
    c = v3(clampf_(c.x, 0.0f, 1.0f), clampf_(c.y, 0.0f, 1.0f), clampf_(c.z, 0.0f, 1.0f));
    return make_uchar4((unsigned char)unorm8(c.x), (unsigned char)unorm8(c.y), (unsigned char)unorm8(c.z), 255);
}

// combine + tonemap fused: the combined image is also written (it is the
// reference's ping image at that point).
__global__ __launch_bounds__(256) void k_combine_tonemap(const float4* __restrict__ orig, const float4* __restrict__ bloom,
                                                         float4* __restrict__ combined, uchar4* __restrict__ out,
                                                         uint32_t n, float intensity, float exposure_scale) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 bl = bloom[i];
    float4 c;
    const uchar4 t = combine_tonemap(orig[i], v3(bl.x, bl.y, bl.z), intensity, exposure_scale, c);
    combined[i] = c;
    out[i] = t;
}

// ---- blur over the taps with a weight ----------------------------------------
constexpr int kTapPad = 16;      // zero weights before the first and after the last tap
constexpr int kMaxTapHalf = 448; // 3.7 KB of the 4 KB of kernel arguments
// No sum of samples up to this overflows (the weights add up to 2.51 sigma + 1 at most).
constexpr float kFinite = 1.0e34f;

// w[kTapPad + i + half] is the weight of tap i, zero outside [-k, k].
struct Taps {
    int32_t k;      // the stencil's half-width
    int32_t half;   // a multiple of 4; every tap beyond it has weight zero
    float wsum;     // sum over all taps, in tap order
    float w[2 * kMaxTapHalf + 1 + 2 * kTapPad];
};

// Adds the taps of samples m0..m0+U-1 to R neighbouring outputs: sample m is
// tap m - half of output 0, m - 1 - half of output 1, ...
template <int R, int U>
__device__ __forceinline__ void add_taps(const Taps& t, int m0, const float (&x)[3][U], float (&c)[R][3]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const float w = t.w[kTapPad + m0 + u - j];
#pragma unroll
            for (int a = 0; a < 3; ++a) c[j][a] = c[j][a] + x[a][u] * w;
        }
    }
}

// Adds every tap of R neighbouring outputs, those without a weight too: a
// sample that is not finite makes them NaN (zero times which is NaN).
// load(m, x): samples m..m+U-1 as add_taps numbers them, zero outside the image.
// Samples that all R outputs take without a weight are one multiply-add per
// channel, into z: all it can add is zero or NaN.
template <int R, int U, typename Load>
__device__ __forceinline__ void add_every_tap(const Taps& t, Load load, float (&c)[R][3]) {
    const int first = t.half - t.k, last = t.half + t.k;   // the stencil of output 0; output j's is j further
    float z[3] = {0.0f, 0.0f, 0.0f};
    for (int m = first & ~(U - 1); m <= last + R - 1; m += U) {
        float x[3][U];
        load(m, x);
        if (m >= first + R - 1 && m + U - 1 <= last) {     // in all R stencils
            if (m >= 0 && m <= 2 * t.half + R - 1) {
                add_taps<R, U>(t, m, x, c);
            } else {
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) z[a] = z[a] + x[a][u] * 0.0f;
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int j = 0; j < R; ++j) {
                    const int i = m + u - j;               // tap i - half
                    if (i < first || i > last) continue;
                    const float w = i < 0 || i > 2 * t.half ? 0.0f : t.w[kTapPad + i];
#pragma unroll
                    for (int a = 0; a < 3; ++a) c[j][a] = c[j][a] + x[a][u] * w;
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
#pragma unroll
        for (int a = 0; a < 3; ++a) c[j][a] = c[j][a] + z[a];
    }
}

__device__ __forceinline__ V3 blur_mean(const float (&c)[3], float wsum) {
    return wsum < 0.0001f ? v3(0.0f, 0.0f, 0.0f) : v3(c[0] / wsum, c[1] / wsum, c[2] / wsum);
}

// blurX of row blockIdx.x. The row's three channels lie in LDS, `half` zeros on
// either side; a lane's R outputs are neighbours, so R = 4 reads four samples of
// a channel with one 16-byte load for 16 multiply-adds. out.w is 1, or 2 in a
// row whose samples are not all finite (or near overflow).
template <int R, int U>
__global__ __launch_bounds__(1024) void k_blur_row(const float4* __restrict__ in, float4* __restrict__ out, uint32_t W,
                                                   uint32_t pitch, float threshold, const Taps t) {
    extern __shared__ __align__(16) float s_row[];   // [3][pitch]
    const float4* src = in + (uint64_t)blockIdx.x * W;
    float4* dst = out + (uint64_t)blockIdx.x * W;
    bool bad = false;
    for (uint32_t p = threadIdx.x; p < pitch; p += blockDim.x) {
        const int32_t x = (int32_t)p - t.half;
        float r = 0.0f, g = 0.0f, b = 0.0f;
        if (x >= 0 && x < (int32_t)W) {
            const float4 v = src[x];
            if (!(dot(v3(v.x, v.y, v.z), v3(0.299f, 0.587f, 0.114f)) < threshold)) { r = v.x; g = v.y; b = v.z; }
            bad = bad || !(fabsf(r) <= kFinite && fabsf(g) <= kFinite && fabsf(b) <= kFinite);
        }
        s_row[p] = r;
        s_row[pitch + p] = g;
        s_row[2 * pitch + p] = b;
    }
    const bool every = __syncthreads_or(bad ? 1 : 0) != 0;   // every tap counts
    for (uint32_t x0 = threadIdx.x * R; x0 < W; x0 += blockDim.x * R) {
        float c[R][3];
#pragma unroll
        for (int j = 0; j < R; ++j) c[j][0] = c[j][1] = c[j][2] = 0.0f;
        if (!every) {
            const float* p0 = s_row + x0;
            for (int m = 0; m < 2 * t.half + R; m += U) {
                float x[3][U];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if constexpr (R == 4) {   // x0, m and pitch are multiples of 4
#pragma unroll
                        for (int u = 0; u < U; u += 4) {
                            const float4 v = *reinterpret_cast<const float4*>(p0 + a * pitch + m + u);
                            x[a][u] = v.x; x[a][u + 1] = v.y; x[a][u + 2] = v.z; x[a][u + 3] = v.w;
                        }
                    } else {
#pragma unroll
                        for (int u = 0; u < U; ++u) x[a][u] = p0[a * pitch + m + u];
                    }
                }
                add_taps<R, U>(t, m, x, c);
            }
        } else {
            add_every_tap<R, 4>(t, [&](int m, float (&x)[3][4]) {
                const int32_t p = (int32_t)x0 + m;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    if constexpr (R == 4) {   // p and pitch are multiples of 4
                        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                        if ((uint32_t)p < pitch) v = *reinterpret_cast<const float4*>(s_row + a * pitch + p);
                        x[a][0] = v.x; x[a][1] = v.y; x[a][2] = v.z; x[a][3] = v.w;
                    } else {
#pragma unroll
                        for (int u = 0; u < 4; ++u) x[a][u] = (uint32_t)(p + u) < pitch ? s_row[a * pitch + p + u] : 0.0f;
                    }
                }
            }, c);
        }
#pragma unroll
        for (int j = 0; j < R; ++j) {
            if (x0 + j >= W) break;
            const V3 v = blur_mean(c[j], t.wsum);
            dst[x0 + j] = make_float4(v.x, v.y, v.z, every ? 2.0f : 1.0f);
        }
    }
}

// blurY, combine and tonemap of 64 columns x 4 R rows; wave w takes R rows and
// loads U samples at a time (enough in flight to cover the load's latency).
template <int R, int U>
__global__ __launch_bounds__(256) void k_blur_column(const float4* __restrict__ blurx, const float4* __restrict__ orig,
                                                     float4* __restrict__ combined, uchar4* __restrict__ out, uint32_t W,
                                                     uint32_t H, float intensity, float exposure_scale, const Taps t) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t xb = blockIdx.x * 64u, x = xb + lane;
    const int32_t yb = (int32_t)(blockIdx.y * 4u * R);
    // rows that k_blur_row marked, among all that the sums below read: k either
    // side, and the zero-weight taps up to the next multiple of U
    const int32_t reach = t.k > t.half + U ? t.k : t.half + U;
    bool bad = false;
    for (int32_t y = yb - reach + (int32_t)threadIdx.x; y < yb + 4 * R + reach; y += 256)
        if (y >= 0 && y < (int32_t)H) bad = bad || blurx[(uint64_t)y * W + xb].w != 1.0f;
    const bool every = __syncthreads_or(bad ? 1 : 0) != 0;
    const int32_t y0 = __builtin_amdgcn_readfirstlane(yb + (int32_t)(wave * R));
    if (x >= W || y0 >= (int32_t)H) return;
    float c[R][3];
#pragma unroll
    for (int j = 0; j < R; ++j) c[j][0] = c[j][1] = c[j][2] = 0.0f;
    const float4* col = blurx + x;
    const auto load = [&](int m, auto& s) {
#pragma unroll
        for (int u = 0; u < (int)(sizeof(s[0]) / sizeof(float)); ++u) {
            const int32_t y = y0 - t.half + m + u;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (y >= 0 && y < (int32_t)H) v = col[(uint64_t)(uint32_t)y * W];
            s[0][u] = v.x; s[1][u] = v.y; s[2][u] = v.z;
        }
    };
    if (!every) {
        for (int m = 0; m < 2 * t.half + R; m += U) {
            float s[3][U];
            load(m, s);
            add_taps<R, U>(t, m, s, c);
        }
    } else {
        add_every_tap<R, 4>(t, load, c);
    }
#pragma unroll
    for (int j = 0; j < R; ++j) {
        if (y0 + j >= (int32_t)H) break;
        const uint64_t o = (uint64_t)(uint32_t)(y0 + j) * W + x;
        float4 cm;
        const uchar4 ldr = combine_tonemap(orig[o], blur_mean(c[j], t.wsum), intensity, exposure_scale, cm);
        combined[o] = cm;
        out[o] = ldr;
    }
}

// The taps of a blur over `len` pixels; false where k_blur has to do it: a
// radius that is not positive and finite, or more taps than the kernel
// arguments hold (radius above 31 on images over 480 pixels).
static bool make_taps(uint32_t len, float radius, Taps& t) {
    const float k = ((float)(int32_t)len * radius) / 100.0f * 3.0f + 0.5f;
    if (!(radius > 0.0f && k >= 0.0f && k < 1.0e6f)) return false;
    t.k = (int32_t)k;
    // expf_ returns 0 below -103.97: beyond sqrt(2 * 103.98) sigma nothing is left
    const float reach = 14.43f * radius + 2.0f;
    int32_t h = reach < (float)t.k ? (int32_t)reach : t.k;
    if (h > kMaxTapHalf) return false;
    float w[kMaxTapHalf + 1];
    for (int32_t i = 0; i <= h; ++i) w[i] = gauss((float)i, radius);   // even in i
    while (h > 0 && w[h] == 0.0f) --h;
    t.half = (h + 3) & ~3;
    for (int32_t i = 0; i < 2 * t.half + 1 + 2 * kTapPad; ++i) {
        const int32_t tap = i - kTapPad - t.half, a = tap < 0 ? -tap : tap;
        t.w[i] = a <= h ? w[a] : 0.0f;
    }
    t.wsum = 0.0f;
    for (int32_t i = -h; i <= h; ++i) t.wsum = t.wsum + w[i < 0 ? -i : i];
    return true;
}

template <int R, int U>
static void launch_blur_row(const float4* in, float4* out, uint32_t W, uint32_t H, uint32_t pitch, float threshold,
                            const Taps& t, hipStream_t st) {
    uint32_t threads = ((W + R - 1) / R + 63u) & ~63u;
    if (threads > 1024u) threads = 1024u;
    hipLaunchKernelGGL((k_blur_row<R, U>), dim3(H), dim3(threads), 3u * pitch * sizeof(float), st, in, out, W, pitch, threshold, t);
}

template <int R, int U>
static void launch_blur_column(const float4* blurx, const float4* orig, float4* combined, uchar4* out, uint32_t W,
                               uint32_t H, float intensity, float exposure_scale, const Taps& t, hipStream_t st) {
    hipLaunchKernelGGL((k_blur_column<R, U>), dim3((W + 63) / 64, (H + 4 * R - 1) / (4 * R)), dim3(256), 0, st, blurx, orig,
                       combined, out, W, H, intensity, exposure_scale, t);
}

// k_blur_row holds a row in 64 KB of LDS: rows of up to about 5,200 pixels.
constexpr uint32_t kRowLds = 65536;

hipError_t launch_postprocess(const float4* in, float4* ping, float4* pong, uchar4* out, uint32_t W, uint32_t H,
                              const BloomPushConsts& b, const TonemappingPushConsts& t, hipStream_t st) {
    const float e = exp2f_(t.exposure);
    hipError_t err;
    Taps tx, ty;
    if (make_taps(W, b.radius, tx) && make_taps(H, b.radius, ty)) {
        // staged width: the last lane's last group of samples ends at W + 2 half + 16
        const uint32_t pitch = (W + 2u * (uint32_t)tx.half + 16u + 3u) & ~3u;
        if (3ull * pitch * sizeof(float) <= kRowLds && (H + 3u) / 4u <= 65535u) {
            // outputs per lane: as many as leave a few waves for each of the 1,024 SIMDs.
            // us with few | many outputs: 341x213 15 | 30, 512x512 35 | 45, 724x724 71 | 57,
            // 1024x1024 114 | 61, 1920x1080 231 | 110
            if ((uint64_t)W * H >= (1u << 19)) launch_blur_row<4, 4>(in, pong, W, H, pitch, b.threshold, tx, st);
            else launch_blur_row<1, 16>(in, pong, W, H, pitch, b.threshold, tx, st);
            err = hipGetLastError();
            if (err != hipSuccess) return err;
            if ((uint64_t)W * H >= (1u << 19)) launch_blur_column<8, 8>(pong, in, ping, out, W, H, b.intensity, e, ty, st);
            else launch_blur_column<1, 16>(pong, in, ping, out, W, H, b.intensity, e, ty, st);
            return hipGetLastError();
        }
    }
    dim3 gx((W + kTile - 1) / kTile, H);
    hipLaunchKernelGGL((k_blur<1, true>), gx, dim3(kTile), 0, st, in, ping, W, H, b);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    dim3 gy((H + kTile - 1) / kTile, W);
    hipLaunchKernelGGL((k_blur<0, false>), gy, dim3(kTile), 0, st, ping, pong, W, H, b);
    err = hipGetLastError();
    if (err != hipSuccess) return err;
    uint32_t n = W * H;
    hipLaunchKernelGGL(k_combine_tonemap, dim3((n + 255) / 256), dim3(256), 0, st, in, pong, ping, out, n,
                       b.intensity, e);
    return hipGetLastError();
}

}  // namespace rt
