// nt_codec.hip — BC6H-style latent block codec (the reference has no encoder; its BC6
// decode emulation is train.cu:159-202). Per 4x4 block and channel: two fp16 endpoints
// (stored as order keys) and sixteen 4-bit indices into the BC6H interpolation weights.
//
// Encode: one thread per (block, channel). Endpoints are the min and max order key of the
// block's fp16-rounded values; each index minimises |v - decode(i)| in fp32 (lowest index
// wins ties), found among three candidate levels, or by binary searches over the 16 decoded
// levels where levels can coincide. Integer key arithmetic plus IEEE fp32 compares make the
// result bit-exact against the CPU restatement (a linear scan). Decode: one thread per (texel, 4 channels), float4 stores.
#include <algorithm>

#include "nt_internal.hpp"

namespace ntk {

// Indices of the levels nearest to the N values v[p]: for each, the first i minimising
// |v - L[i]| in fp32, exactly what a linear scan with a strict "<" finds. The 16 decoded
// levels are non-decreasing (the interpolated keys are, and the key order is the value
// order). With j the number of levels below v, the errors are non-increasing on [0, j) and
// non-decreasing on [j, 16) (fp32 rounding is monotone), so the minimum is at j - 1 or j;
// at j - 1 it is the first index of that error only if level j - 2 is farther, else (a
// plateau of equal levels or of equal rounded errors, rare) a binary search over [0, j)
// finds the first. N searches run step by step together, so each step's N LDS reads are
// issued at once.
//
// R is the thread's padded level column: R[0] = R[1] = L[0], R[2 + i] = L[i], R[18] = L[15]
// (entries kLevelStride floats apart), so levels j - 2, j - 1 and j (clamped to the ends) are
// R[j], R[j + 1], R[j + 2] for every j in [0, 16] without index clamps; at j = 0 and j = 16
// levels j - 1 and j read equal, so the comparison between them picks j - 1 (clamped to 0) as
// it must. A thread's entries are one workgroup (256 floats) apart, so they all lie in the
// thread's own LDS bank: reads at any level are free of conflicts (with a row per thread, the
// levels side by side, the lanes' reads fell in random banks).
constexpr int kLevelRows = 19;
constexpr int kLevelStride = 256;

typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef short s2 __attribute__((ext_vector_type(2)));

template <int N>
__device__ __forceinline__ void codec_nearest_n(const float *R, const float *v, int *idx)
{
    const float *q[N];
#pragma unroll
    for (int p = 0; p < N; ++p)
        q[p] = R + 2 * kLevelStride;
#pragma unroll
    for (int step = 8; step > 0; step >>= 1) {
        float l[N];
#pragma unroll
        for (int p = 0; p < N; ++p)
            l[p] = q[p][(step - 1) * kLevelStride];
#pragma unroll
        for (int p = 0; p < N; ++p)
            q[p] += l[p] < v[p] ? step * kLevelStride : 0;
    }
    float lm[N], lc[N], l2[N];
#pragma unroll
    for (int p = 0; p < N; ++p) {
        l2[p] = q[p][-2 * kLevelStride];
        lm[p] = q[p][-kLevelStride];
        lc[p] = q[p][0];
    }
    float a[N];
    int j[N];
    bool need[N], any = false;
#pragma unroll
    for (int p = 0; p < N; ++p) {
        j[p] = (int)(q[p] - (R + 2 * kLevelStride)) / kLevelStride;
        a[p] = fabsf(v[p] - lm[p]);
        const bool upper = fabsf(v[p] - lc[p]) < a[p];
        idx[p] = upper ? j[p] : max(j[p] - 1, 0);
        need[p] = j[p] >= 2 && !upper && fabsf(v[p] - l2[p]) <= a[p];
        any |= need[p];
    }
    if (!any)
        return;
#pragma unroll
    for (int p = 0; p < N; ++p) {
        if (!need[p])
            continue;
        int lo = 0, hi = j[p] - 1; // the first index in [lo, hi] whose error is <= a
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int mid = (lo + hi) >> 1;
            const bool le = fabsf(v[p] - R[(2 + mid) * kLevelStride]) <= a[p];
            hi = lo < hi && le ? mid : hi;
            lo = lo < hi && !le ? mid + 1 : lo;
        }
        idx[p] = lo;
    }
}

// The same indices where the order keys k0 .. k1 of a block's values span at least
// kCandidateSpan: three candidate levels per value instead of a search. Level m's key is
// k0 + round(kd w_m / 64), kd = k1 - k0, w_m = round(64 m / 15), so in steps of kd / 15 it
// lies within D = 7/64 + 7.5/kd of m (0.344 at kd = 32). For a value whose fp16 key lies
// p steps above k0, levels m < p - D are below it and levels m > p + D are not, so with
// i = floor(p - D') (D' = 0.36: D and the fp32 arithmetic's error, below 0.004) the levels
// j - 1 and j around it (j levels below the value) are among i, i + 1, i + 2: i <= j - 1, and
// i + 2 >= j as D + D' < 1. Neighbouring levels are at least one key apart, and at most 2^10
// times as far apart in value as the next pair, so no two errors on one side of the value
// are equal after fp32 rounding, and counting the strict improvements along the three gives
// the first index of the least error. A value past the last level reads the row's padding
// (level 15 again), which never improves.
// What bounds the search: VALU issue (11 instructions a value against 26 for the binary
// search) and the LDS reads (12 bytes a value against 28). 4096^2 x 16 channels of N(0, 0.5):
// 310 -> 215 us, 5.9 TB/s of the 1.28 GB moved (VALU issue 80 % of the time, 398 instructions
// a wave against 673); blocks of a smooth image, whose values span fewer keys and take the
// binary search, 495 -> 490 us.
constexpr uint32_t kCandidateSpan = 32;

__device__ __forceinline__ int codec_nearest_candidate(const float *R, float v, float key, float scale, float bias)
{
    // scale = 15 / kd, bias = -(scale k0 + D'): below zero converts to 0.
    // (a plain v_cvt_u32_f32, which clamps, without a float maximum before it).
    uint32_t i;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(i) : "v"(fmaf(key, scale, bias)));
    const float *q = R + (2 + i) * kLevelStride;
    const float e0 = fabsf(v - q[0]), e1 = fabsf(v - q[kLevelStride]), e2 = fabsf(v - q[2 * kLevelStride]);
    return (int)i + (e1 < e0) + (e2 < e1);
}

// Encode: a workgroup takes 256/C horizontally adjacent blocks of one block row, thread
// (block, channel). The 16 decoded levels of a thread's (block, channel) are computed once
// into its LDS column; each pixel's index is then found among them (above). The nibbles are
// assembled in LDS and stored as whole 32-bit words.
template <int C>
__global__ __launch_bounds__(256) void codec_encode_kernel(const float *values, int W, int H,
                                                           uint8_t *blocks)
{
    constexpr int BPW = 256 / C; // blocks per workgroup
    __shared__ float lev[kLevelRows * kLevelStride];
    __shared__ __align__(16) uint8_t nib[BPW][16 * C + 16]; // 16 bytes past a multiple of 256: other banks for each block
    const int tid = threadIdx.x, lb = tid / C, c = tid % C;
    const int bw = (W + 3) >> 2, bh = (H + 3) >> 2;
    const int bx = blockIdx.x * BPW + lb;
    float *R = lev + tid;
    const bool active = lb < BPW && bx < bw; // C = 12 leaves 256 % 12 threads idle
    // A block's sixteen loads, from clamped (always valid) addresses, so that none sits under a
    // branch waiting for its own round trip; pixels past the image edge are masked afterwards.
    // Each row's base (the workgroup's first column) is uniform and the thread's byte offset
    // in it is below 2^15: no address arithmetic per load.
    const int x0 = 4 * BPW * (int)blockIdx.x;
    uint32_t off[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
        off[q] = (uint32_t)(min(4 * lb + q, W - 1 - x0) * C + c) * 4u;
    for (int by = blockIdx.y; by < bh; by += gridDim.y) {
        uint8_t *rec = blocks + ((int64_t)by * bw + bx) * (12 * C);
        if (active) {
            float raw[16];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const char *row = (const char *)(values + ((int64_t)min(4 * by + r, H - 1) * W + x0) * C);
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    raw[4 * r + q] = load_global((const float *)(row + off[q]));
            }
            const bool whole = 4 * bx + 3 < W && 4 * by + 3 < H;
            float v[16];
            us2 key[8]; // order keys, two pixels each
            uint32_t kmin = 0xFFFFu, kmax = 0u;
            if (whole) {
                // A block wholly inside the image (all but the last block row and column):
                // the order keys two pixels per instruction (codec_key on each 16-bit half:
                // h ^ 0xFFFF for a set sign bit, h ^ 0x8000 else), with packed min and max.
                us2 kmn = {0xFFFF, 0xFFFF}, kmx = {0, 0};
#pragma unroll
                for (int p = 0; p < 16; p += 2) {
                    // (A NaN gives the lower bound, as fmin(fmax()) does: the median of three of
                    // which one is NaN is the least of the three, taken from the first on, where
                    // a signalling NaN turns quiet and the bound that follows last remains.)
                    v[p] = __builtin_amdgcn_fmed3f(raw[p], 65504.f, -65504.f);
                    v[p + 1] = __builtin_amdgcn_fmed3f(raw[p + 1], 65504.f, -65504.f);
                    const f2 pv = {v[p], v[p + 1]};
                    const us2 hb = __builtin_bit_cast(us2, __builtin_convertvector(pv, h2));
                    const us2 sg = __builtin_bit_cast(us2, __builtin_bit_cast(s2, hb) >> (short)15);
                    key[p / 2] = hb ^ ((sg & (unsigned short)0x7FFF) | (unsigned short)0x8000);
                    kmn = __builtin_elementwise_min(kmn, key[p / 2]);
                    kmx = __builtin_elementwise_max(kmx, key[p / 2]);
                }
                kmin = kmn.x < kmn.y ? kmn.x : kmn.y;
                kmax = kmx.x > kmx.y ? kmx.x : kmx.y;
            } else {
#pragma unroll
                for (int p = 0; p < 16; ++p) {
                    const bool in = 4 * bx + (p & 3) < W && 4 * by + (p >> 2) < H;
                    v[p] = in ? fminf(fmaxf(raw[p], -65504.f), 65504.f) : 0.f;
                    const uint32_t k = codec_key(h_bits((_Float16)v[p]));
                    kmin = in && k < kmin ? k : kmin;
                    kmax = in && k > kmax ? k : kmax;
                    key[p >> 1][p & 1] = (unsigned short)k;
                }
                // Pixels past the edge: a key in range (their indices are written as 0).
#pragma unroll
                for (int p = 0; p < 16; ++p)
                    if (!(4 * bx + (p & 3) < W && 4 * by + (p >> 2) < H))
                        key[p >> 1][p & 1] = (unsigned short)kmin;
            }
            *(uint32_t *)(rec + 4 * c) = kmin | (kmax << 16);
            // The sixteen levels, two per instruction after the interpolation: key
            // (64 k0 + (k1 - k0) w + 32) >> 6 (= codec_interp), formed in the high half of
            // (k0 << 16) + ((k1 - k0) w + 32) << 10, then codec_unkey on each half
            // (k ^ 0x8000 for a set top bit, k ^ 0xFFFF else) and the fp16 -> fp32 widening.
            float lv[16];
            const uint32_t kbase = (kmin << 16) + (32u << 10), kd = kmax - kmin;
#pragma unroll
            for (int i = 0; i < 16; i += 2) {
                // 24-bit factors: kd < 2^16, w << 10 <= 2^16.
                const uint32_t k0 = kbase + __umul24(kd, (uint32_t)codec_weight(i) << 10);
                const uint32_t k1 = kbase + __umul24(kd, (uint32_t)codec_weight(i + 1) << 10);
                const uint32_t kk = __builtin_amdgcn_perm(k1, k0, 0x07060302u); // the high halves
                // 0xFFFF in each half whose top bit is set (op_sel_hi: the shift count of the
                // high half is the inline constant's low half too).
                uint32_t top;
                asm("v_pk_ashrrev_i16 %0, 15, %1 op_sel_hi:[0,1]" : "=v"(top) : "v"(kk));
                const uint32_t hv = kk ^ (~top | 0x80008000u);
                const f2 fv = __builtin_convertvector(__builtin_bit_cast(h2, hv), f2);
                lv[i] = fv[0];
                lv[i + 1] = fv[1];
            }
            R[0] = lv[0];
            R[kLevelStride] = lv[0];
#pragma unroll
            for (int i = 0; i < 16; ++i)
                R[(2 + i) * kLevelStride] = lv[i];
            R[18 * kLevelStride] = lv[15];
            int idx[16];
            // One of the two for the whole wave, so that a wave never runs both.
            if (__ballot(kd < kCandidateSpan) == 0) {
                const float scale = 15.f / (float)kd, bias = fmaf(-scale, (float)kmin, -0.36f);
#pragma unroll
                for (int p = 0; p < 16; ++p)
                    idx[p] = codec_nearest_candidate(R, v[p], (float)key[p >> 1][p & 1], scale, bias);
            } else {
                // Four searches at a time: 94 registers and five waves per SIMD (eight at a time:
                // 110 and four, which costs both paths 8 %).
#pragma unroll
                for (int p = 0; p < 16; p += 4)
                    codec_nearest_n<4>(R, v + p, idx + p);
            }
            if (!whole) {
#pragma unroll
                for (int p = 0; p < 16; ++p)
                    if (!(4 * bx + (p & 3) < W && 4 * by + (p >> 2) < H))
                        idx[p] = 0;
            }
#pragma unroll
            for (int p = 0; p < 16; ++p)
                nib[lb][p * C + c] = (uint8_t)idx[p];
        }
        __syncthreads();
        if (active) {
            // Index area: nibble p*C + c; word w packs nibbles 8w .. 8w+7, low nibble first.
            // x | x >> 4 puts each odd byte's nibble above the even byte's before it.
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const int w = c + k * C;
                const uint2 n = *(const uint2 *)&nib[lb][8 * w];
                const uint32_t word = __builtin_amdgcn_perm(n.y | n.y >> 4, n.x | n.x >> 4, 0x06040200u);
                *(uint32_t *)(rec + 4 * C + 4 * w) = word;
            }
        }
        __syncthreads();
    }
}

// Decode: thread = (texel column x, 4 channels) of one block row, grid y over block rows.
// The thread loads its block's four endpoint pairs once and the index nibbles of the four
// pixel rows (all loads first), then stores one float4 per row: consecutive lanes write
// consecutive 16 bytes of a texel row (streaming stores).
template <int C>
__global__ __launch_bounds__(256) void codec_decode_kernel(const uint8_t *blocks, int W, int H,
                                                           float *values)
{
    constexpr int G4 = C / 4;
    const int bw = (W + 3) >> 2, bh = (H + 3) >> 2;
    const int row_items = W * G4;
    for (int by = blockIdx.y; by < bh; by += gridDim.y) {
        for (int i = blockIdx.x * 256 + threadIdx.x; i < row_items; i += gridDim.x * 256) {
            const int x = i / G4, cg = i - x * G4;
            const uint8_t *rec = blocks + ((int64_t)by * bw + (x >> 2)) * (12 * C);
            const uint4 e = load_global((const uint4 *)(rec + 16 * cg));
            uint32_t idx[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                idx[r] = load_global((const uint16_t *)(rec + 4 * C + (4 * r + (x & 3)) * (C / 2) + 2 * cg));
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int y = 4 * by + r;
                if (y >= H)
                    break;
                float4 out;
                out.x = codec_value(e.x & 0xFFFFu, e.x >> 16, idx[r] & 15);
                out.y = codec_value(e.y & 0xFFFFu, e.y >> 16, (idx[r] >> 4) & 15);
                out.z = codec_value(e.z & 0xFFFFu, e.z >> 16, (idx[r] >> 8) & 15);
                out.w = codec_value(e.w & 0xFFFFu, e.w >> 16, (idx[r] >> 12) & 15);
                store_stream(values + ((int64_t)y * W + x) * C + 4 * cg, out);
            }
        }
    }
}

// Expand every mip of every codec grid into fp16 texels (the first pass of the two-pass
// decode): one thread per (texel, 8 channels), one 16-byte store. Work items are numbered
// over the concatenated (grid, mip) levels; level k starts at item d.start[k].
__global__ __launch_bounds__(256) void codec_expand_kernel(CodecExpandDesc d)
{
    constexpr int C = 16, G8 = C / 8;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= d.start[d.levels])
        return;
    int k = 0;
    for (int j = 1; j < d.levels; ++j)
        k = i >= d.start[j] ? j : k;
    const int64_t local = i - d.start[k];
    const int W = d.w[k];
    const int64_t texel = local / G8;
    const int cg = (int)(local % G8);
    const int x = (int)(texel % W), y = (int)(texel / W);
    const uint8_t *rec = d.blocks[k] + ((int64_t)(y >> 2) * ((W + 3) >> 2) + (x >> 2)) * (12 * C);
    const int pix = ((y & 3) << 2) + (x & 3);
    const uint4 e0 = *(const uint4 *)(rec + 32 * cg);
    const uint4 e1 = *(const uint4 *)(rec + 32 * cg + 16);
    const uint32_t idx = *(const uint32_t *)(rec + 4 * C + pix * (C / 2) + 4 * cg);
    const uint32_t ends[8] = {e0.x, e0.y, e0.z, e0.w, e1.x, e1.y, e1.z, e1.w};
    uint32_t packed[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const uint32_t lo = codec_unkey(codec_interp(ends[e] & 0xFFFFu, ends[e] >> 16, (idx >> (4 * e)) & 15));
        const uint32_t hi =
            codec_unkey(codec_interp(ends[e + 1] & 0xFFFFu, ends[e + 1] >> 16, (idx >> (4 * e + 4)) & 15));
        packed[e / 2] = lo | (hi << 16);
    }
    *(uint4 *)(d.out[k] + texel * C + 8 * cg) = make_uint4(packed[0], packed[1], packed[2], packed[3]);
}

hipError_t launch_codec_expand(const CodecExpandDesc &d, hipStream_t s)
{
    const int64_t total = d.start[d.levels];
    if (total <= 0)
        return hipSuccess;
    hipLaunchKernelGGL(codec_expand_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, d);
    return hipGetLastError();
}

template <int C>
static hipError_t encode_c(const float *values, int w, int h, uint8_t *blocks, hipStream_t s)
{
    const int bw = (w + 3) / 4, bh = (h + 3) / 4;
    const int gx = (bw + 256 / C - 1) / (256 / C), gy = bh < 65535 ? bh : 65535;
    hipLaunchKernelGGL(codec_encode_kernel<C>, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, values, w, h,
                       blocks);
    return hipGetLastError();
}

template <int C>
static hipError_t decode_c(const uint8_t *blocks, int w, int h, float *values, hipStream_t s)
{
    const int64_t row_items = (int64_t)w * (C / 4);
    const int bh = (h + 3) / 4;
    // At most 256 block rows of workgroups, each looping over the rest (measured: a little
    // faster than one workgroup row per block row).
    const int gx = (int)std::min<int64_t>((row_items + 255) / 256, 65535), gy = bh < 256 ? bh : 256;
    hipLaunchKernelGGL(codec_decode_kernel<C>, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, blocks, w, h,
                       values);
    return hipGetLastError();
}

hipError_t launch_codec_encode(const float *values, int w, int h, int C, uint8_t *blocks, hipStream_t s)
{
    switch (C) {
    case 4:
        return encode_c<4>(values, w, h, blocks, s);
    case 8:
        return encode_c<8>(values, w, h, blocks, s);
    case 12:
        return encode_c<12>(values, w, h, blocks, s);
    case 16:
        return encode_c<16>(values, w, h, blocks, s);
    default:
        return hipErrorInvalidValue;
    }
}

hipError_t launch_codec_decode(const uint8_t *blocks, int w, int h, int C, float *values, hipStream_t s)
{
    switch (C) {
    case 4:
        return decode_c<4>(blocks, w, h, values, s);
    case 8:
        return decode_c<8>(blocks, w, h, values, s);
    case 12:
        return decode_c<12>(blocks, w, h, values, s);
    case 16:
        return decode_c<16>(blocks, w, h, values, s);
    default:
        return hipErrorInvalidValue;
    }
}

} // namespace ntk
