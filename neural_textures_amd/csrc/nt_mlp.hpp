// nt_mlp.hpp — the tiny fp16 MLP on gfx950 MFMA (v_mfma_f32_32x32x16_f16).
//
// Replaces the tcnn warp-MMA MLP of the reference (mlp.h:18-362). Formulation: the wave
// computes Y^T = W^T X^T, so weights are the A operand (32 output rows per tile, staged in
// LDS as ready-to-load fragments) and activations the B operand (one sample per lane
// column, 32 samples per wave tile). The D accumulator layout of one layer is reused, in
// registers, as the B operand of the next layer by permuting the K index of the next
// layer's weight fragments — activations never leave VGPRs between layers.
//
// Feature index carried by element e (0..7) of k-step fragment q in lane group g = lane/32:
//   "natural" layout (network input as gathered): f = 16q + 8g + e
//   "chained" layout (any layer output / dX):     f = 16q + 8(e>>2) + 4g + (e&3)
// Chained fragment q is elements [8(q&1), 8(q&1)+8) of D tile q>>1.
#pragma once

#include "nt_device.hpp"

namespace ntk {

constexpr int kWave = 64;

// Padded widths: K0 network input, H hidden, NH hidden layers, output padded to 16.
template <int K0_, int H_, int NH_>
struct Shape {
    static constexpr int K0 = K0_, H = H_, NH = NH_, L = NH_ + 1, OUT = 16;
    static_assert(K0 % 16 == 0 && K0 <= 64 && H % 16 == 0 && H <= 64 && NH >= 1 && NH <= 5,
                  "unsupported MLP shape");
    __host__ __device__ static constexpr int kin(int l) { return l == 0 ? K0 : H; }
    __host__ __device__ static constexpr int kout(int l) { return l == L - 1 ? OUT : H; }
    __host__ __device__ static constexpr int t32(int w) { return (w + 31) / 32; }
    __host__ __device__ static constexpr int fwd_frags(int l) { return t32(kout(l)) * (kin(l) / 16); }
    __host__ __device__ static constexpr int bwd_frags(int l) { return t32(kin(l)) * (kout(l) / 16); }
    __host__ __device__ static constexpr int fwd_off(int l)
    {
        int o = 0;
        for (int j = 0; j < l; ++j)
            o += fwd_frags(j);
        return o;
    }
    __host__ __device__ static constexpr int fwd_total() { return fwd_off(L); }
    __host__ __device__ static constexpr int bwd_off(int l)
    {
        int o = fwd_total();
        for (int j = 0; j < l; ++j)
            o += bwd_frags(j);
        return o;
    }
    __host__ __device__ static constexpr int all_frags() { return bwd_off(L); }
    // fp32 bias rows per layer, padded to whole 32-row tiles.
    __host__ __device__ static constexpr int bias_off(int l)
    {
        int o = 0;
        for (int j = 0; j < l; ++j)
            o += 32 * t32(kout(j));
        return o;
    }
    __host__ __device__ static constexpr int bias_total() { return bias_off(L); }
    // Gradient partial layout: per layer kout*kin weights then kout biases.
    __host__ __device__ static constexpr int grad_off(int l)
    {
        int o = 0;
        for (int j = 0; j < l; ++j)
            o += kout(j) * kin(j) + kout(j);
        return o;
    }
    __host__ __device__ static constexpr int grad_total() { return grad_off(L); }
    // dW tiles (32x32), enumerated from the last layer down.
    __host__ __device__ static constexpr int dw_tiles(int l) { return t32(kout(l)) * t32(kin(l)); }
    __host__ __device__ static constexpr int dw_start(int l)
    {
        int o = 0;
        for (int j = L - 1; j > l; --j)
            o += dw_tiles(j);
        return o;
    }
    __host__ __device__ static constexpr int dw_total() { return dw_start(-1); }
};

__device__ __forceinline__ int chained_feature(int q, int g, int e)
{
    return 16 * q + 8 * (e >> 2) + 4 * g + (e & 3);
}
__device__ __forceinline__ int natural_feature(int q, int g, int e) { return 16 * q + 8 * g + e; }
// Layer-0 input feature of element e of k-step fragment q in lane group g: lane group g
// holds grids g and g + 2, channels 8(q & 1) .. 8(q & 1) + 7.
__host__ __device__ constexpr int grid_feature(int q, int g, int e)
{
    return 16 * (g + 2 * (q >> 1)) + 8 * (q & 1) + e;
}


// Network pointers and unpadded sizes, as kernels see them.
struct MlpDesc {
    const uint16_t *W[6];
    const uint16_t *B[6];
    int sizes[7];
    int num_layers;
};

// Element idx = fragment * 64 + lane of the forward/backward weight fragments, in the
// order layer_forward / layer_backward_dx read them.
template <class S, bool GRID_ORDER = false>
__device__ h8 weight_fragment(const MlpDesc &m, int idx)
{
    const int f = idx / kWave, lane = idx % kWave, c = lane & 31, g = lane >> 5;
    h8 v;
    int l = 0;
    const bool fwd = f < S::fwd_total();
    if (fwd) {
        while (l + 1 < S::L && f >= S::fwd_off(l + 1))
            ++l;
    } else {
        while (l + 1 < S::L && f >= S::bwd_off(l + 1))
            ++l;
    }
    const int kin = S::kin(l), kout = S::kout(l);
    const uint16_t *W = m.W[l];
    if (fwd) {
        // Forward fragment (a, q) of layer l, lane (c, g), element e: W_l[k][n] with
        // n = 32a + c and k the layer's input feature for (q, g, e).
        const int local = f - S::fwd_off(l), qn = kin / 16;
        const int a = local / qn, q = local % qn;
        const int n = 32 * a + c;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = l > 0 ? chained_feature(q, g, e) : GRID_ORDER ? grid_feature(q, g, e) : natural_feature(q, g, e);
            v[e] = (n < kout && k < kin) ? bits_h(W[n * kin + k]) : (_Float16)0.f;
        }
    } else {
        // Backward (dX) fragment (m, q) of layer l: A[k][kk] = W_l[k][n], k = 32m + c,
        // n = chained output feature of (q, g, e).
        const int local = f - S::bwd_off(l), qn = kout / 16;
        const int mt = local / qn, q = local % qn;
        const int k = 32 * mt + c;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int n = chained_feature(q, g, e);
            v[e] = (n < kout && k < kin) ? bits_h(W[n * kin + k]) : (_Float16)0.f;
        }
    }
    return v;
}

// Layer-0 input feature of element e of k-step fragment q in lane group g for networks on
// C-channel grids. 16 channels: grid_feature (grids g and g + 2, eight consecutive channels
// per fragment). 3 channels (up to four grids, one k-step): lane group g holds grid g's
// channels (e = 0..2), grid g + 2's (e = 3..5) and two of the padding features 12..15
// (e = 6, 7), so that each lane samples two grids and the two groups together cover all
// sixteen inputs. 8 channels (up to two grids): channels 4g .. 4g + 3 of grid 0 (e = 0..3) and
// of grid 1 (e = 4..7), the chained order, so that one grid occupies both lane groups.
template <int C>
__host__ __device__ constexpr int input_feature(int q, int g, int e)
{
    if constexpr (C == 16)
        return grid_feature(q, g, e);
    else if constexpr (C == 3)
        return e < 3 ? 3 * g + e : e < 6 ? 3 * (g + 2) + (e - 3) : 12 + 2 * g + (e - 6);
    else
        return 16 * q + 8 * (e >> 2) + 4 * g + (e & 3);
}

// Layer l's forward fragments, items tid, tid + NT, ... (an item is a fragment's lane): a
// lane's eight inputs of one output row are 16 consecutive bytes of the weight row (layer 0
// with 16 channels; with 3 eight scattered halves) or two runs of 8 bytes (chained order), so the
// fragments are read with those loads, all of them issued before the first LDS store.
template <class S, int C, int l, int NT>
__device__ __forceinline__ void stage_forward_layer(const MlpDesc &m, h8 *frags, int tid)
{
    constexpr int kin = S::kin(l), kout = S::kout(l), qn = kin / 16;
    constexpr int items = S::fwd_frags(l) * kWave, N = (items + NT - 1) / NT;
    const uint16_t *W = m.W[l];
    h8 v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int idx = min(tid + j * NT, items - 1), f = idx / kWave, lane = idx % kWave;
        const int c = lane & 31, g = lane >> 5, a = f / qn, q = f % qn;
        const int n = 32 * a + c;
        const uint16_t *row = W + min(n, kout - 1) * kin;
        if constexpr (l > 0 || C == 8) {
            const uint2 lo = load_global((const uint2 *)(row + chained_feature(q, g, 0)));
            const uint2 hi = load_global((const uint2 *)(row + chained_feature(q, g, 4)));
            v[j] = __builtin_bit_cast(h8, make_uint4(lo.x, lo.y, hi.x, hi.y));
        } else if constexpr (C == 3) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[j][e] = bits_h(load_global(row + input_feature<C>(q, g, e)));
        } else {
            v[j] = __builtin_bit_cast(h8, load_global((const uint4 *)(row + input_feature<C>(q, g, 0))));
        }
        if (n >= kout)
            v[j] = (h8)(_Float16)0.f;
    }
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (tid + j * NT < items)
            frags[S::fwd_off(l) * kWave + tid + j * NT] = v[j];
}

// Stage the forward weight fragments and fp32 biases of a network on C-channel grids
// (input_feature order) in LDS, NT threads; the caller synchronises afterwards. Weights that
// are not 16-byte aligned are read element by element.
template <class S, int C, int NT>
__device__ __forceinline__ void stage_forward(const MlpDesc &m, h8 *frags, float *bias, int tid)
{
    uintptr_t mis = 0;
#pragma unroll
    for (int l = 0; l < S::L; ++l)
        mis |= (uintptr_t)m.W[l] & 15u;
    if (mis == 0) {
        stage_forward_layer<S, C, 0, NT>(m, frags, tid);
        stage_forward_layer<S, C, 1, NT>(m, frags, tid);
        if constexpr (S::L > 2)
            stage_forward_layer<S, C, 2, NT>(m, frags, tid);
        if constexpr (S::L > 3)
            stage_forward_layer<S, C, 3, NT>(m, frags, tid);
        static_assert(S::L <= 4, "at most four layers");
    } else {
        for (int idx = tid; idx < S::fwd_total() * kWave; idx += NT) {
            const int f = idx / kWave, lane = idx % kWave, c = lane & 31, g = lane >> 5;
            int l = 0;
            while (l + 1 < S::L && f >= S::fwd_off(l + 1))
                ++l;
            const int kin = S::kin(l), qn = kin / 16, local = f - S::fwd_off(l);
            const int n = 32 * (local / qn) + c, q = local % qn;
            h8 v;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = l > 0 ? chained_feature(q, g, e) : input_feature<C>(q, g, e);
                v[e] = n < S::kout(l) ? bits_h(m.W[l][n * kin + k]) : (_Float16)0.f;
            }
            frags[idx] = v;
        }
    }
#pragma unroll
    for (int l = 0; l < S::L; ++l)
        for (int n = tid; n < 32 * S::t32(S::kout(l)); n += NT)
            bias[S::bias_off(l) + n] = n < m.sizes[l + 1] ? h2f(m.B[l][n]) : 0.f;
}

// fp32 bias row idx (layers back to back, each padded to 32-row tiles).
template <class S>
__device__ float bias_value(const MlpDesc &m, int idx)
{
    int l = 0;
    while (l + 1 < S::L && idx >= S::bias_off(l + 1))
        ++l;
    const int n = idx - S::bias_off(l);
    return n < m.sizes[l + 1] ? h2f(m.B[l][n]) : 0.f;
}

// Stage forward (and, unless FWD_ONLY, backward) weight fragments and fp32 biases in LDS,
// layer 0 in natural or grid_feature input order. All threads of the block take part; the
// caller synchronises afterwards.
template <class S, bool FWD_ONLY = false, bool GRID_ORDER = false>
__device__ void stage_weights(const MlpDesc &m, h8 *frags, float *bias, int tid, int nthreads)
{
    constexpr int nfrags = FWD_ONLY ? S::fwd_total() : S::all_frags();
    for (int idx = tid; idx < nfrags * kWave; idx += nthreads)
        frags[idx] = weight_fragment<S, GRID_ORDER>(m, idx);
    for (int idx = tid; idx < S::bias_total(); idx += nthreads)
        bias[idx] = bias_value<S>(m, idx);
}

// One forward layer for one 32-sample tile: acc[a] = bias + W^T x. With PREFETCH all of the
// layer's weight fragments are read from LDS before the first MFMA and the row tiles'
// accumulation chains are interleaved (more registers, no LDS round trip per MFMA).
template <int KQ, int NA, bool PREFETCH = false>
__device__ __forceinline__ void layer_forward(const h8 *frags, const float *bias, const h8 (&x)[KQ],
                                              f16v (&acc)[NA], int lane)
{
    const int g = lane >> 5;
    // Rows 32a + 8j + 4g .. +3 of the bias are one 16-byte LDS read (bias is 16-byte aligned).
    const float4 *b4 = (const float4 *)(bias + 4 * g);
    if constexpr (PREFETCH) {
        h8 w[NA][KQ];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int q = 0; q < KQ; ++q)
                w[a][q] = frags[(a * KQ + q) * kWave + lane];
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float4 v = b4[8 * a + 2 * j];
                acc[a][4 * j] = v.x;
                acc[a][4 * j + 1] = v.y;
                acc[a][4 * j + 2] = v.z;
                acc[a][4 * j + 3] = v.w;
            }
#pragma unroll
        for (int q = 0; q < KQ; ++q)
#pragma unroll
            for (int a = 0; a < NA; ++a)
                acc[a] = mfma32(w[a][q], x[q], acc[a]);
        return;
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 v = b4[8 * a + 2 * j];
            acc[a][4 * j] = v.x;
            acc[a][4 * j + 1] = v.y;
            acc[a][4 * j + 2] = v.z;
            acc[a][4 * j + 3] = v.w;
        }
#pragma unroll
        for (int q = 0; q < KQ; ++q)
            acc[a] = mfma32(frags[(a * KQ + q) * kWave + lane], x[q], acc[a]);
    }
}

// One forward layer for two 32-sample tiles: each weight fragment read from LDS feeds the
// MFMAs of both tiles, which also gives two independent accumulation chains.
template <int KQ, int NA>
__device__ __forceinline__ void layer_forward2(const h8 *frags, const float *bias, const h8 (&x0)[KQ],
                                               const h8 (&x1)[KQ], f16v (&acc0)[NA], f16v (&acc1)[NA], int lane)
{
    const int g = lane >> 5;
    const float4 *b4 = (const float4 *)(bias + 4 * g);
#pragma unroll
    for (int a = 0; a < NA; ++a) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 v = b4[8 * a + 2 * j];
            acc0[a][4 * j] = acc1[a][4 * j] = v.x;
            acc0[a][4 * j + 1] = acc1[a][4 * j + 1] = v.y;
            acc0[a][4 * j + 2] = acc1[a][4 * j + 2] = v.z;
            acc0[a][4 * j + 3] = acc1[a][4 * j + 3] = v.w;
        }
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            const h8 w = frags[(a * KQ + q) * kWave + lane];
            acc0[a] = mfma32(w, x0[q], acc0[a]);
            acc1[a] = mfma32(w, x1[q], acc1[a]);
        }
    }
}

// D tiles -> chained fp16 fragments, with optional ReLU (mlp.h:35-38). The ReLU is taken
// after the conversion, as a signed 16-bit max with 0 on the pair (v_pk_max_i16): negative
// halves and -0 have the sign bit set, so they become +0. fp16 rounding is monotone, so
// this equals rounding max(x, 0), in one instruction per pair instead of a float max (and
// its NaN canonicalisation) per element.
template <int NQ, int NA, bool RELU>
__device__ __forceinline__ void to_fragments(const f16v (&acc)[NA], h8 (&y)[NQ])
{
    typedef short s2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const f2 v = {acc[q >> 1][8 * (q & 1) + e], acc[q >> 1][8 * (q & 1) + e + 1]};
            h2 h = __builtin_convertvector(v, h2); // v_cvt_pk_f16_f32
            if (RELU)
                h = __builtin_bit_cast(h2, __builtin_elementwise_max(__builtin_bit_cast(s2, h), (s2)0));
            y[q][e] = h[0];
            y[q][e + 1] = h[1];
        }
    }
}

// ReLU backward (mlp.h:240-252): dY_prev = fp16(acc) where the layer input x > 0, else 0.
// x is a ReLU output (to_fragments: never negative, no -0), so x > 0 exactly when its bits
// are nonzero: the mask min(bits, 1) multiplies the converted pair as 16-bit integers
// (v_pk_min_u16, v_pk_mul_lo_u16 after one v_cvt_pk_f16_f32 per pair).
template <int NQ, int NA>
__device__ __forceinline__ void relu_backward(const f16v (&acc)[NA], const h8 (&x)[NQ], h8 (&dy)[NQ])
{
    // Written as instructions: the compiler turns the equivalent vector code into per-lane
    // compares and lane masks.
    const uint32_t ones = 0x00010001u;
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const f2 v = {acc[q >> 1][8 * (q & 1) + e], acc[q >> 1][8 * (q & 1) + e + 1]};
            const uint32_t hv = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, h2));
            const h2 xv = {x[q][e], x[q][e + 1]};
            uint32_t m, r;
            asm("v_pk_min_u16 %0, %1, %2" : "=v"(m) : "v"(__builtin_bit_cast(uint32_t, xv)), "v"(ones));
            asm("v_pk_mul_lo_u16 %0, %1, %2" : "=v"(r) : "v"(hv), "v"(m));
            const h2 rh = __builtin_bit_cast(h2, r);
            dy[q][e] = rh[0];
            dy[q][e + 1] = rh[1];
        }
}

// dX for one layer: acc[m] = W dY over the layer's output features (chained dY frags).
// PREFETCH as in layer_forward.
template <int NQ, int MA, bool PREFETCH = false>
__device__ __forceinline__ void layer_backward_dx(const h8 *frags, const h8 (&dy)[NQ],
                                                  f16v (&acc)[MA], int lane)
{
    if constexpr (PREFETCH) {
        h8 w[MA][NQ];
#pragma unroll
        for (int m = 0; m < MA; ++m)
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                w[m][q] = frags[(m * NQ + q) * kWave + lane];
#pragma unroll
        for (int m = 0; m < MA; ++m)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                acc[m][e] = 0.f;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int m = 0; m < MA; ++m)
                acc[m] = mfma32(w[m][q], dy[q], acc[m]);
        return;
    }
#pragma unroll
    for (int m = 0; m < MA; ++m) {
#pragma unroll
        for (int e = 0; e < 16; ++e)
            acc[m][e] = 0.f;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            acc[m] = mfma32(frags[(m * NQ + q) * kWave + lane], dy[q], acc[m]);
    }
}

} // namespace ntk
