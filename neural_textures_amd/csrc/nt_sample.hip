// nt_sample.hip — latent sample + MLP at caller-given coordinates (nt_forward): trilinear over
// a grid's mips (train.cu:263-314) or 16-tap Catmull-Rom on mip 0.
//
// What bounds it: for few samples latency (weights, coordinates, one round of texel loads, the
// layers in sequence), for many the scattered texel loads and instruction issue. Each lane
// computes the footprints of the grids it samples only (16 and 3 channels: grids g and g + 2;
// 8 channels: four channels of both grids, so that config 1's one grid uses every lane), wraps
// a coordinate with one conditional add or subtract (an integer modulo only for coordinates
// more than a grid away), and issues all texels of a footprint before their first product. The
// first tile is sampled before the barrier that publishes the weights. Catmull-Rom, 65,536
// samples: a 256^2 grid with the 8-64-64-3 network 28.0 -> 8.9 us, a 512^2 one 39.6 -> 10.6, the reference network
// 27.4 -> 15.5, four grids of 16 channels 236 -> 41 (a footprint per feature, tap by tap,
// before); 5,000 samples of two grids 30.2 -> 12.6 us. Trilinear, 500,000 samples over four
// mips: the reference network 164 -> 52 us, two grids 93 -> 86, four 158 -> 146 (bound by their
// 64-byte texel reads, 1 GB through the L1s with four grids).
#include <type_traits>

#include "nt_internal.hpp"

namespace ntk {

namespace {

template <class S>
struct SampleLayout {
    static constexpr int frag_bytes = S::fwd_total() * kWave * 16;
    static constexpr int bias_bytes = ((S::bias_total() * 4 + 15) / 16) * 16;
    static constexpr int bytes = frag_bytes + bias_bytes;
};

typedef float f3 __attribute__((ext_vector_type(3), aligned(4))); // a 12-byte load

// A coordinate wrapped into [0, size) like the reference's texel addressing, for any int.
__device__ __forceinline__ int wrap_any(int c, int size)
{
    int r = c < 0 ? (int)((uint32_t)c + (uint32_t)size) : (c >= size ? c - size : c);
    if ((unsigned)r >= (unsigned)size)
        r = wrap_coord(c, size);
    return r;
}

// The channels of one texel that a lane reads: all 3, all 16, or four of 8.
template <int C>
struct Texel {
    static constexpr int N = C == 16 ? 4 : 1; // loads
    using T = typename std::conditional<C == 3, f3, float4>::type;
    T v[N];
    template <class Index>
    __device__ __forceinline__ void load(const float *base, Index texel, int g)
    {
        if constexpr (C == 3) {
            v[0] = *(const __attribute__((address_space(1))) f3 *)(base + (size_t)texel * 3u);
        } else {
            const float4 *p = (const float4 *)(base + (size_t)texel * (uint32_t)C) + (C == 8 ? g : 0);
#pragma unroll
            for (int i = 0; i < N; ++i)
                v[i] = load_global(p + i);
        }
    }
    // Channel ch of the lane's (compile-time after unrolling).
    __device__ __forceinline__ float at(int ch) const
    {
        if constexpr (C == 3) {
            return v[0][ch];
        } else {
            const float4 &q = v[ch >> 2];
            return (ch & 3) == 0 ? q.x : (ch & 3) == 1 ? q.y : (ch & 3) == 2 ? q.z : q.w;
        }
    }
};

// Channels per lane and grid, and where channel ch of the lane's j-th grid goes in its layer-0
// fragments (input_feature).
template <int C>
constexpr int lane_channels() { return C == 8 ? 4 : C; }
template <int C>
constexpr int frag_of(int j, int ch) { return C == 16 ? 2 * j + (ch >> 3) : 0; }
template <int C>
constexpr int elem_of(int j, int ch) { return C == 16 ? (ch & 7) : C == 8 ? 4 * j + ch : 3 * j + ch; }

} // namespace

// WIDE: texel indices in 64 bits, for grids of 2^32 texels and more (51.5 GB with 3 channels).
// Below, 32 bits hold them: 64-bit rows cost the reference network's 500,000 trilinear samples
// 51.1 -> 53.8 us.
template <class S, int C, bool CR, bool WIDE>
__global__ __launch_bounds__(kFwdThreads) void sample_kernel(SampleDesc d)
{
    using Index = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
    constexpr int L = S::L, NH = S::NH, KQ0 = S::K0 / 16, HQ = S::H / 16, HA = S::t32(S::H);
    constexpr int NG = C == 16 ? KQ0 / 2 : 2, NC = lane_channels<C>(); // grids per lane, channels of each
    using LY = SampleLayout<S>;
    extern __shared__ __align__(16) unsigned char smem[];
    h8 *frags = (h8 *)smem;
    float *bias = (float *)(smem + LY::frag_bytes);
    // First float (as two words), width and height of every (grid, mip): the mip differs per lane.
    __shared__ int4 level[NT_MAX_GRIDS * NT_MAX_MIPS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 31, g = lane >> 5;
    if (!CR && tid < NT_MAX_GRIDS * NT_MAX_MIPS) {
        const int gi = tid / NT_MAX_MIPS, m = tid % NT_MAX_MIPS;
        const GridDesc &q = d.grid[gi];
        const uintptr_t p = (uintptr_t)(q.values + q.mip_off[m] * C);
        level[tid] = make_int4((int)(uint32_t)p, (int)(uint32_t)(p >> 32), mip_dim(q.w, m), mip_dim(q.h, m));
    }
    stage_forward<S, C, kFwdThreads>(d.mlp, frags, bias, tid);
    if (!CR)
        __syncthreads(); // the levels

    h8 x0[KQ0];
    auto sample = [&](int tile) {
        const int s = tile * 32 + c, sc = s < d.count ? s : 0;
        const float *p = d.uvz + 3 * (int64_t)sc;
        const float u = load_global(p), v = load_global(p + 1), z = CR ? 0.f : load_global(p + 2);
#pragma unroll
        for (int q = 0; q < KQ0; ++q)
            x0[q] = (h8)(_Float16)0.f;
#pragma unroll
        for (int j = 0; j < NG; ++j) {
            // 16 and 3 channels: grid 2j + g; 8 channels: grid j. Entries past G repeat grid 0.
            const GridDesc &ga = d.grid[C == 8 ? j : 2 * j], &gb = d.grid[C == 8 ? j : 2 * j + 1];
            const bool on = (C == 8 ? j : 2 * j + g) < d.G;
            if (C == 8 && j >= d.G)
                continue; // uniform
            if constexpr (CR) {
                const int w = g ? sreg(gb.w) : sreg(ga.w), h = g ? sreg(gb.h) : sreg(ga.h);
                const float *vals = g ? sreg(gb.values + gb.mip_off[0] * C) : sreg(ga.values + ga.mip_off[0] * C);
                float wx[4], wy[4];
                const int gx = cr_axis(u, w, wx), gy = cr_axis(v, h, wy);
                int xs[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    xs[i] = wrap_any((int)((uint32_t)gx + (uint32_t)i), w);
                float acc[NC];
#pragma unroll
                for (int ch = 0; ch < NC; ++ch)
                    acc[ch] = 0.f;
                // Rows of taps loaded together: all four, or with 16 channels one.
                constexpr int RB = C == 16 ? 1 : 4;
#pragma unroll
                for (int r0 = 0; r0 < 4; r0 += RB) {
                    Texel<C> t[RB][4];
#pragma unroll
                    for (int r = 0; r < RB; ++r) {
                        const Index row = (Index)wrap_any((int)((uint32_t)gy + (uint32_t)(r0 + r)), h) * (uint32_t)w;
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            t[r][i].load(vals, row + (uint32_t)xs[i], g);
                    }
#pragma unroll
                    for (int r = 0; r < RB; ++r)
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const float wxy = wx[i] * wy[r0 + r];
#pragma unroll
                            for (int ch = 0; ch < NC; ++ch)
                                acc[ch] = fmaf(t[r][i].at(ch), wxy, acc[ch]);
                        }
                    // (holds the compiler to one block of rows' registers)
                    if constexpr (C == 16)
                        __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int ch = 0; ch < NC; ++ch)
                    x0[frag_of<C>(j, ch)][elem_of<C>(j, ch)] = on ? (_Float16)acc[ch] : (_Float16)0.f;
            } else {
                // Mip pair (train.cu:266-281) and the corner sums: contributions rounded to fp16,
                // added in fp16, corner by corner and mip by mip (train.cu:293-310).
                const int gi = C == 8 ? j : 2 * j + g;
                const int top = max((g ? sreg(gb.num_mips) : sreg(ga.num_mips)) - 1, 0);
                const float fz = floorf(z), frac = z - fz;
                const int base = (int)fz;
                const float mw[2] = {1.f - frac, frac};
                _Float16 a[NC];
#pragma unroll
                for (int ch = 0; ch < NC; ++ch)
                    a[ch] = (_Float16)0.f;
#pragma unroll
                for (int mi = 0; mi < 2; ++mi) {
                    if (mi == 1 && !(frac > 0.f))
                        continue;
                    const int m = max(min((int)((uint32_t)base + (uint32_t)mi), top), 0);
                    const int4 lv = level[gi * NT_MAX_MIPS + m];
                    const float *vals = (const float *)(((uintptr_t)(uint32_t)lv.y << 32) | (uint32_t)lv.x);
                    const int w = lv.z, h = lv.w;
                    const Footprint f = bilinear_footprint(u, v, (float)w, (float)h, mw[mi]);
                    const int x[2] = {wrap_any(f.x0, w), wrap_any((int)((uint32_t)f.x0 + 1u), w)};
                    const Index y[2] = {(Index)wrap_any(f.y0, h) * (uint32_t)w,
                                        (Index)wrap_any((int)((uint32_t)f.y0 + 1u), h) * (uint32_t)w};
                    Texel<C> t[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        t[k].load(vals, y[k >> 1] + (uint32_t)x[k & 1], g);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        // Two channels per conversion and add.
#pragma unroll
                        for (int ch = 0; ch + 1 < NC; ch += 2) {
                            const f2 p2 = {rn32(f.w[k] * t[k].at(ch)), rn32(f.w[k] * t[k].at(ch + 1))};
                            const h2 s2 = h2{a[ch], a[ch + 1]} + __builtin_convertvector(p2, h2);
                            a[ch] = s2[0];
                            a[ch + 1] = s2[1];
                        }
                        if constexpr (NC & 1)
                            a[NC - 1] = a[NC - 1] + half_of_product(f.w[k], t[k].at(NC - 1));
                    }
                }
#pragma unroll
                for (int ch = 0; ch < NC; ++ch)
                    x0[frag_of<C>(j, ch)][elem_of<C>(j, ch)] = on ? a[ch] : (_Float16)0.f;
            }
        }
    };

    const int ntiles = (d.count + 31) / 32, step = gridDim.x * kFwdWaves;
    int tile = blockIdx.x * kFwdWaves + wave;
    if (tile < ntiles)
        sample(tile);
    __syncthreads(); // the weights
    while (tile < ntiles) {
        const int s = tile * 32 + c;
        const bool valid = s < d.count;
        if (d.features != nullptr && valid) {
            const int nf = d.G * C;
#pragma unroll
            for (int q = 0; q < KQ0; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int feat = input_feature<C>(q, g, e);
                    if (feat < nf)
                        d.features[(int64_t)s * nf + feat] = h_bits(x0[q][e]);
                }
        }

        // MLP forward (mlp.h:65-99)
        h8 xh[HQ];
        {
            f16v acc[HA];
            layer_forward<KQ0, HA, true>(frags + S::fwd_off(0) * kWave, bias + S::bias_off(0), x0, acc, lane);
            to_fragments<HQ, HA, true>(acc, xh);
#pragma unroll
            for (int l = 1; l < NH; ++l) {
                layer_forward<HQ, HA, true>(frags + S::fwd_off(l) * kWave, bias + S::bias_off(l), xh, acc, lane);
                to_fragments<HQ, HA, true>(acc, xh);
            }
        }
        f16v out[1];
        layer_forward<HQ, 1, true>(frags + S::fwd_off(L - 1) * kWave, bias + S::bias_off(L - 1), xh, out, lane);
        if (valid) {
            // Lane group g holds output rows 4g .. 4g+3 and 8+4g .. 8+4g+3: with a row stride
            // that is a multiple of 4 each run of four is one 8-byte store.
            uint16_t *orow = d.out16 + (int64_t)s * d.out_stride;
            const bool quads = (d.out_stride & 3) == 0;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int o = 8 * j + 4 * g;
                const f2 v0 = {out[0][4 * j], out[0][4 * j + 1]}, v1 = {out[0][4 * j + 2], out[0][4 * j + 3]};
                const h2 h0 = __builtin_convertvector(v0, h2), h1 = __builtin_convertvector(v1, h2);
                if (quads) {
                    if (o < d.out_stride)
                        *(uint2 *)(orow + o) = make_uint2(__builtin_bit_cast(uint32_t, h0), __builtin_bit_cast(uint32_t, h1));
                } else {
                    const _Float16 hv[4] = {h0[0], h0[1], h1[0], h1[1]};
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (o + r < d.out_stride)
                            orow[o + r] = h_bits(hv[r]);
                }
            }
        }
        tile += step;
        if (tile < ntiles)
            sample(tile);
    }
}

template <class S, int C>
static hipError_t launch_sample_shape(const SampleDesc &d, bool catmull_rom, hipStream_t s)
{
    bool wide = false;
    for (int gi = 0; gi < d.G; ++gi)
        wide |= (int64_t)d.grid[gi].w * d.grid[gi].h >= (1ll << 32);
    const auto k = wide ? (catmull_rom ? sample_kernel<S, C, true, true> : sample_kernel<S, C, false, true>)
                        : (catmull_rom ? sample_kernel<S, C, true, false> : sample_kernel<S, C, false, false>);
    hipLaunchKernelGGL(k, dim3(forward_blocks(d.count)), dim3(kFwdThreads), SampleLayout<S>::bytes, s, d);
    return hipGetLastError();
}

hipError_t launch_sample(int shape, bool catmull_rom, const SampleDesc &d, hipStream_t s)
{
    switch (shape) {
    case kShapeRef:
        return launch_sample_shape<Shape<16, 32, 2>, 3>(d, catmull_rom, s);
    case kShapeC1:
        return launch_sample_shape<Shape<16, 64, 2>, 8>(d, catmull_rom, s);
    case kShapeC2:
        return launch_sample_shape<Shape<32, 64, 2>, 16>(d, catmull_rom, s);
    case kShapeC4:
        return launch_sample_shape<Shape<64, 64, 3>, 16>(d, catmull_rom, s);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace ntk
