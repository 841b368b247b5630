// nt_infer.hip — full-image inference at texel centres (train.cu:917-961) for reference
// textures of the image's size: latent sample, MLP, fp32 outputs and the squared error
// against the Catmull-Rom targets.
//
// What bounds it: the outputs written and the textures read once (486 MB at 2048^2 with the
// reference network, 75 us at the 6.5 TB/s that large streams reach here), and instruction
// issue, about 105 us of it. A wave walks a strip of 32 pixels down `rows` image rows, one
// 32-sample MFMA tile a row, so that what depends on the column only (the footprint columns
// and fractions, the Catmull-Rom column weights) is computed once, and a texture row is read
// once per strip, not once per row that taps it: its four column taps are summed when it
// enters a five-row window of sums in registers, and a pixel's target is four of those sums
// weighted by the row weights. Lane group g samples grids g, g + 2 and textures g, g + 2
// only. Outputs go through LDS, so that a wave stores its 32 pixels as whole cache lines.
// 2048^2: reference network 1,111 -> 178 us, two grids of 16 channels 771 -> 211 us, four
// 944 -> 403 us (one sample per lane with per-feature footprints, integer modulos and 16 taps
// of every texture before). Three waves per SIMD (168 registers) spill and take 275 us.
#include <type_traits>

#include "nt_internal.hpp"

namespace ntk {

namespace {

// Wrap for coordinates within one period of the grid or image: texel centres lie inside it,
// so bilinear corners reach one texel past either edge and Catmull-Rom taps two.
__device__ __forceinline__ int wrap_once(int c, int size)
{
    return c < 0 ? c + size : (c >= size ? c - size : c);
}

// The column half of a bilinear footprint (mip 0): wrapped columns and the fraction.
struct Column {
    int x0, x1;
    float fx;
};
__device__ __forceinline__ Column column_of(float u, int w)
{
    const float t = fmaf(u, (float)w, -0.5f), b = floorf(t);
    return Column{wrap_once((int)b, w), wrap_once((int)b + 1, w), t - b};
}

typedef float f3 __attribute__((ext_vector_type(3), aligned(4))); // a 12-byte load

constexpr int kPixelStride = 20; // floats per pixel of a wave's LDS rows (16 outputs; 16-byte rows, spread banks)

template <class S>
struct InferLayout {
    static constexpr int frag_bytes = S::fwd_total() * kWave * 16;
    static constexpr int bias_bytes = ((S::bias_total() * 4 + 15) / 16) * 16;
    static constexpr int bytes = frag_bytes + bias_bytes + kFwdWaves * 32 * kPixelStride * 4;
};

} // namespace

// NT: textures per lane (textures g and g + 2): 1 for up to two textures, else 2.
template <class S, int C, int NT>
__global__ __launch_bounds__(kFwdThreads, 2) void inference_kernel(InferDesc d)
{
    constexpr int L = S::L, NH = S::NH, KQ0 = S::K0 / 16, HQ = S::H / 16, HA = S::t32(S::H);
    // Grids per lane: 16 and 3 channels, grids g and g + 2; 8 channels, four channels of both.
    constexpr int NG = C == 16 ? KQ0 / 2 : 2;
    using LY = InferLayout<S>;
    extern __shared__ __align__(16) unsigned char smem[];
    h8 *frags = (h8 *)smem;
    float *bias = (float *)(smem + LY::frag_bytes);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 31, g = lane >> 5;
    float *pix = (float *)(smem + LY::frag_bytes + LY::bias_bytes) + wave * 32 * kPixelStride;
    stage_forward<S, C, kFwdThreads>(d.mlp, frags, bias, tid);
    __syncthreads();

    // The lane's grids and textures, selected once.
    const float *vals[NG];
    int gw[NG], gh[NG];
    bool on[NG];
#pragma unroll
    for (int j = 0; j < NG; ++j) {
        const InferGrid &a = d.grid[C == 8 ? j : 2 * j], &b = d.grid[C == 8 ? j : 2 * j + 1];
        vals[j] = g ? sreg(b.values) + (C == 8 ? 4 : 0) : sreg(a.values);
        gw[j] = g ? sreg(b.w) : sreg(a.w);
        gh[j] = g ? sreg(b.h) : sreg(a.h);
        on[j] = (C == 8 ? j : 2 * j + g) < d.G;
    }
    const float4 *tex[NT];
    int nch[NT], out0[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        tex[j] = (const float4 *)(g ? sreg(d.tex[2 * j + 1]) : sreg(d.tex[2 * j]));
        nch[j] = g ? sreg(d.tex_nch[2 * j + 1]) : sreg(d.tex_nch[2 * j]);
        out0[j] = g ? sreg(d.tex_out0[2 * j + 1]) : sreg(d.tex_out0[2 * j]);
    }
    const int W = d.image_w, H = d.image_h, stride = d.out_stride;

    float sse = 0.f;
    const int nstrips = d.strips_x * d.strips_y;
    for (int st = blockIdx.x * kFwdWaves + wave; st < nstrips; st += gridDim.x * kFwdWaves) {
        const int sy = st / d.strips_x, px0 = 32 * (st - sy * d.strips_x), px = min(px0 + c, W - 1);
        const int y0 = sy * d.rows, y1 = min(y0 + d.rows, H), np = min(W - px0, 32);
        const float u = div_pow2((float)px + 0.5f, (float)W, d.inv_w); // train.cu:926-933
        Column col[NG];
#pragma unroll
        for (int j = 0; j < NG; ++j)
            col[j] = column_of(u, gw[j]);
        // Catmull-Rom columns: taps gx .. gx + 3, gx the pixel's column less one or two.
        float wx[4];
        const int gx = cr_axis(u, W, wx);
        int xo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            xo[i] = wrap_once(gx + i, W);
        // One texture row's four column taps, and their sums weighted by the column weights.
        auto row_taps = [&](int y, float4 (&p)[NT][4]) {
            const uint32_t base = (uint32_t)wrap_once(y, H) * (uint32_t)W;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    p[j][i] = load_global(tex[j] + (base + (uint32_t)xo[i]));
        };
        auto row_sums = [&](const float4 (&p)[NT][4], float4 (&h)[NT]) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                h[j] = make_float4(p[j][0].x * wx[0], p[j][0].y * wx[0], p[j][0].z * wx[0], p[j][0].w * wx[0]);
#pragma unroll
                for (int i = 1; i < 4; ++i) {
                    h[j].x = fmaf(p[j][i].x, wx[i], h[j].x);
                    h[j].y = fmaf(p[j][i].y, wx[i], h[j].y);
                    h[j].z = fmaf(p[j][i].z, wx[i], h[j].z);
                    h[j].w = fmaf(p[j][i].w, wx[i], h[j].w);
                }
            }
        };
        // Column sums of rows y - 2 .. y + 2: row y - 2 + k in entry (y - y0 + k) % 5, the row
        // loop unrolled by five so that the entries stay in registers without moves.
        float4 win[5][NT];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            float4 p[NT][4];
            row_taps(y0 - 2 + k, p);
            row_sums(p, win[k]);
        }
        // Outputs without a texture channel have target 0.
#pragma unroll
        for (int k = 0; k < 2; ++k)
            *(float4 *)(pix + c * kPixelStride + 8 * k + 4 * g) = make_float4(0.f, 0.f, 0.f, 0.f);

        auto one_row = [&](auto phase, int y) {
            constexpr int PH = decltype(phase)::value;
            const float v = div_pow2((float)y + 0.5f, (float)H, d.inv_h);

            // ---- latents (train.cu:284-310, mip 0): corner contributions rounded to fp16 and
            // summed in fp16, corner by corner
            h8 x0[KQ0];
#pragma unroll
            for (int q = 0; q < KQ0; ++q)
                x0[q] = (h8)(_Float16)0.f;
            constexpr int F4 = C == 16 ? 4 : 1;
            using Texel = typename std::conditional<C == 3, f3, float4>::type;
            Texel tx[NG][4][F4];
            float wgt[NG][4];
#pragma unroll
            for (int j = 0; j < NG; ++j) {
                const float t = fmaf(v, (float)gh[j], -0.5f), b = floorf(t), fy = t - b;
                const int r0 = wrap_once((int)b, gh[j]) * gw[j], r1 = wrap_once((int)b + 1, gh[j]) * gw[j];
                const float ax = 1.f - col[j].fx, ay = 1.f - fy;
                wgt[j][0] = ax * ay;
                wgt[j][1] = col[j].fx * ay;
                wgt[j][2] = ax * fy;
                wgt[j][3] = col[j].fx * fy;
                const uint32_t at[4] = {(uint32_t)(r0 + col[j].x0), (uint32_t)(r0 + col[j].x1),
                                        (uint32_t)(r1 + col[j].x0), (uint32_t)(r1 + col[j].x1)};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if constexpr (C == 3) {
                        tx[j][k][0] = *(const __attribute__((address_space(1))) f3 *)(vals[j] + at[k] * 3u);
                    } else {
#pragma unroll
                        for (int i = 0; i < F4; ++i)
                            tx[j][k][i] = load_global((const float4 *)vals[j] + (at[k] * (uint32_t)(C / 4) + (uint32_t)i));
                    }
                }
            }
            // The row's taps: issued after the latents, needed after the MLP.
            float4 taps[NT][4];
            row_taps(y + 2, taps);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (C == 3) {
                // Two values per fp16 add: channels 0 and 1 of each grid, then channel 2 of both.
                h2 a01[2] = {{(_Float16)0.f, (_Float16)0.f}, {(_Float16)0.f, (_Float16)0.f}};
                h2 a2 = {(_Float16)0.f, (_Float16)0.f};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const f2 p = {rn32(wgt[j][k] * tx[j][k][0][0]), rn32(wgt[j][k] * tx[j][k][0][1])};
                        a01[j] = a01[j] + __builtin_convertvector(p, h2);
                    }
                    const f2 p = {rn32(wgt[0][k] * tx[0][k][0][2]), rn32(wgt[1][k] * tx[1][k][0][2])};
                    a2 = a2 + __builtin_convertvector(p, h2);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    x0[0][3 * j] = on[j] ? a01[j][0] : (_Float16)0.f;
                    x0[0][3 * j + 1] = on[j] ? a01[j][1] : (_Float16)0.f;
                    x0[0][3 * j + 2] = on[j] ? a2[j] : (_Float16)0.f;
                }
            } else if constexpr (C == 8) {
#pragma unroll
                for (int j = 0; j < NG; ++j) {
                    h4 a = {(_Float16)0.f, (_Float16)0.f, (_Float16)0.f, (_Float16)0.f};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float4 &t = tx[j][k][0];
                        const float w = wgt[j][k];
                        const f2 p0 = {rn32(w * t.x), rn32(w * t.y)}, p1 = {rn32(w * t.z), rn32(w * t.w)};
                        a = a + __builtin_shufflevector(__builtin_convertvector(p0, h2), __builtin_convertvector(p1, h2), 0, 1,
                                                        2, 3);
                    }
#pragma unroll
                    for (int ch = 0; ch < 4; ++ch)
                        x0[0][4 * j + ch] = on[j] ? a[ch] : (_Float16)0.f;
                }
            } else {
#pragma unroll
                for (int j = 0; j < NG; ++j)
#pragma unroll
                    for (int i = 0; i < F4; i += 2) {
                        h8 a = (h8)(_Float16)0.f;
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            a = accumulate_products(a, wgt[j][k], tx[j][k][i], tx[j][k][i + 1]);
                        x0[2 * j + i / 2] = on[j] ? a : (h8)(_Float16)0.f;
                    }
            }

            // ---- MLP forward (mlp.h:65-99)
            h8 xh[HQ];
            {
                f16v acc[HA];
                layer_forward<KQ0, HA>(frags + S::fwd_off(0) * kWave, bias + S::bias_off(0), x0, acc, lane);
                to_fragments<HQ, HA, true>(acc, xh);
#pragma unroll
                for (int l = 1; l < NH; ++l) {
                    layer_forward<HQ, HA>(frags + S::fwd_off(l) * kWave, bias + S::bias_off(l), xh, acc, lane);
                    to_fragments<HQ, HA, true>(acc, xh);
                }
            }
            f16v out[1];
            layer_forward<HQ, 1>(frags + S::fwd_off(L - 1) * kWave, bias + S::bias_off(L - 1), xh, out, lane);

            // ---- targets (train.cu:935-960): rows gy .. gy + 3, gy = y - 1 or y - 2 (the
            // image size's rounding); each texture's channels to their outputs' places
            row_sums(taps, win[(PH + 4) % 5]);
            float wy[4];
            const int gy = __builtin_amdgcn_readfirstlane(cr_axis(v, H, wy));
            const bool late = gy == y - 1;
            // A lane's targets may fall among the zeros that the pixel's other lane stored.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                float t4[4];
#pragma unroll
                for (int ch = 0; ch < 4; ++ch) {
                    auto at = [&](int k) {
                        const float4 &h = win[(PH + k) % 5][j];
                        return ch == 0 ? h.x : ch == 1 ? h.y : ch == 2 ? h.z : h.w;
                    };
                    t4[ch] = late ? fmaf(at(4), wy[3], fmaf(at(3), wy[2], fmaf(at(2), wy[1], at(1) * wy[0])))
                                  : fmaf(at(3), wy[3], fmaf(at(2), wy[2], fmaf(at(1), wy[1], at(0) * wy[0])));
                }
#pragma unroll
                for (int ch = 0; ch < 4; ++ch)
                    if (ch < nch[j])
                        pix[c * kPixelStride + out0[j] + ch] = t4[ch];
            }
            // The rows are the wave's own: no workgroup barrier.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            float4 yo[2];
            const bool valid = c < np;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int o = 8 * k + 4 * g;
                const float4 t = *(const float4 *)(pix + c * kPixelStride + o);
                const float tt[4] = {t.x, t.y, t.z, t.w};
                float yy[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    yy[r] = (float)(_Float16)out[0][4 * k + r];
                    const float err = yy[r] - tt[r];
                    sse = valid && o + r < stride ? fmaf(err, err, sse) : sse;
                }
                yo[k] = make_float4(yy[0], yy[1], yy[2], yy[3]);
            }
            // ---- outputs: the row's pixels are consecutive in memory, `stride` floats each
            const int64_t s0 = (int64_t)y * W + px0;
            float *dst = d.out32 + s0 * stride;
            if (stride == 16 && ((uintptr_t)dst & 15u) == 0) {
                // One pixel is 64 bytes: swap halves through LDS so that a store instruction
                // covers 16 whole pixels.
                __builtin_amdgcn_wave_barrier();
                float4 *row = (float4 *)(pix + c * kPixelStride);
                row[g] = yo[0];
                row[2 + g] = yo[1];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const int p = 16 * k + (lane >> 2);
                    const float4 o = *(const float4 *)(pix + p * kPixelStride + 4 * (lane & 3));
                    if (p < np)
                        store_stream(dst + 16 * p + 4 * (lane & 3), o);
                }
            } else {
                __builtin_amdgcn_wave_barrier();
                float *row = pix + c * kPixelStride;
                *(float4 *)(row + 4 * g) = yo[0];
                *(float4 *)(row + 8 + 4 * g) = yo[1];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                for (int i = lane; i < np * stride; i += 64) {
                    const int p = (int)(((float)i + 0.5f) * d.inv_stride);
                    dst[i] = pix[p * kPixelStride + i - p * stride];
                }
            }
            // The places without a texture channel hold target 0 again for the next row.
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int k = 0; k < 2; ++k)
                *(float4 *)(pix + c * kPixelStride + 8 * k + 4 * g) = make_float4(0.f, 0.f, 0.f, 0.f);
        };
        for (int y = y0; y < y1; y += 5) {
            one_row(std::integral_constant<int, 0>{}, y);
            if (y + 1 < y1)
                one_row(std::integral_constant<int, 1>{}, y + 1);
            if (y + 2 < y1)
                one_row(std::integral_constant<int, 2>{}, y + 2);
            if (y + 3 < y1)
                one_row(std::integral_constant<int, 3>{}, y + 3);
            if (y + 4 < y1)
                one_row(std::integral_constant<int, 4>{}, y + 4);
        }
    }
    // The workgroup's squared error: its waves' sums in wave order.
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
        sse += __shfl_xor(sse, off);
    __syncthreads();
    float *part = (float *)smem;
    if (lane == 0)
        part[wave] = sse;
    __syncthreads();
    if (tid == 0) {
        float s = part[0];
        for (int k = 1; k < kFwdWaves; ++k)
            s += part[k];
        if (d.sse_partial)
            d.sse_partial[blockIdx.x] = s;
        else if (s != 0.f)
            global_add(d.sse, s);
    }
}

// The fixed-order SSE reduction: thread t sums partial[t], partial[t + 1024], ... in index
// order, then a pairwise tree over the sums; the result is the same bits on every run.
__global__ __launch_bounds__(1024) void sse_reduce_kernel(const float *partial, int n, float *sse)
{
    __shared__ float part[1024];
    const int t = threadIdx.x;
    float v[8]; // kFwdMaxBlocks * kFwdWaves partials at most
#pragma unroll
    for (int k = 0; k < 8; ++k)
        v[k] = t + 1024 * k < n ? partial[t + 1024 * k] : 0.f;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        s += v[k];
    part[t] = s;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if (t < w)
            part[t] += part[t + w];
        __syncthreads();
    }
    if (t == 0)
        sse[0] = sse[0] + part[0];
}
static_assert(kFwdMaxBlocks * kFwdWaves <= 8 * 1024, "sse_reduce_kernel reads eight partials a thread");

hipError_t launch_sse_reduce(const float *partial, int n, float *sse, hipStream_t s)
{
    hipLaunchKernelGGL(sse_reduce_kernel, dim3(1), dim3(1024), 0, s, partial, n, sse);
    return hipGetLastError();
}

template <class S, int C>
static hipError_t launch_infer(const InferDesc &d, hipStream_t s)
{
    const auto k = d.ntex > 2 ? inference_kernel<S, C, 2> : inference_kernel<S, C, 1>;
    hipLaunchKernelGGL(k, dim3(d.blocks), dim3(kFwdThreads), InferLayout<S>::bytes, s, d);
    return hipGetLastError();
}

hipError_t launch_inference(int shape, const InferDesc &d, hipStream_t s)
{
    switch (shape) {
    case kShapeRef:
        return launch_infer<Shape<16, 32, 2>, 3>(d, s);
    case kShapeC1:
        return launch_infer<Shape<16, 64, 2>, 8>(d, s);
    case kShapeC2:
        return launch_infer<Shape<32, 64, 2>, 16>(d, s);
    case kShapeC4:
        return launch_infer<Shape<64, 64, 3>, 16>(d, s);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace ntk
