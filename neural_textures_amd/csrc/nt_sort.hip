// nt_sort.hip — the sample order of NT_SAMPLES_RANDOM steps. Each sample's texel (the
// placement the train kernel uses: random_texel of its seed) falls in a 64 x 64-texel bin;
// the sample indices are sorted by bin, stably, so that consecutive slots — one chunk of the
// train kernel — lie close together in the image and their target taps, latent corners and
// gradient atomics share cache lines in the L2. The kernel reads the sample of each slot from
// the order and places it exactly as before: the samples and their results are unchanged,
// only the order of the fp32 sums moves. A stable sort by key has one result, so the order is
// the same on every run.
//
// The sort is a counting sort by digits, all integer work. sort_count_kernel: each workgroup
// takes a tile of consecutive samples (4,096, or more so that there are at most 256 tiles),
// computes their bin keys (stored for the later passes) and counts them per first digit in
// LDS (the whole key when it has at most ten bits, config 2's 1,024 bins; else its top eight
// bits). sort_first_pass_kernel: each workgroup derives where its tile's samples of each
// digit start from all tiles' counts (the digits' totals, scanned, plus the digit's counts
// in earlier tiles). Each of its eight waves then places a contiguous part of the tile in
// order, 64 a round: it has its own row of running places (the tile's, plus the counts of the
// waves before it), so a sample's place is its digit's entry + the lanes before it with the
// same digit (ballots on the digit bits), and rounds need no barrier. Keys of more than ten
// bits then go through sort_segment_kernel: one workgroup per first digit sorts that digit's
// segment by the remaining key bits the same way, writing the final order.
//
// What bounds it: the latency of the rounds. With one row of places a workgroup of 256 and
// two barriers in each round of 256 items, the first pass took 19.3 us for 262,144 samples in
// 1,024 bins (64 workgroups), now 12.1; for a million samples in 4,096 bins 20.3 -> 18.1 us (the
// scattered stores of two arrays) and the segments 13.3 -> 9.7 us. A step of two grids 188.7 ->
// 180.5 us, of four 823 -> 814 us. More threads in the count kernel (1,024) gain nothing.
#include <hip/hip_runtime.h>

#include "nt_internal.hpp"

namespace ntk {

namespace {

constexpr int kSortThreads = 256; // the counts and the path
constexpr int kPassThreads = 512, kPassWaves = kPassThreads / 64;
constexpr int kPassRegs = 8; // items per lane loaded at once: a wave's part of a tile of 4,096
constexpr int kSortMaxDigits = 1024; // digits of a one-pass sort (keys of at most ten bits)

__device__ __forceinline__ uint32_t bin_key(const RandomOrderDesc &d, uint32_t i)
{
    uint32_t tx, ty;
    random_texel(mix_seed(i, d.step), d.image_w, d.image_h, tx, ty);
    return (ty >> d.bin_shift) * (uint32_t)d.bins_x + (tx >> d.bin_shift);
}

// The lanes of the wave that are active and hold the same digit (`bits` bits) as this lane.
__device__ __forceinline__ uint64_t match_digit(uint32_t digit, int bits, uint64_t active)
{
    uint64_t m = active;
    for (int b = 0; b < bits; ++b) {
        const bool set = (digit >> b) & 1u;
        const uint64_t bal = __ballot(set);
        m &= set ? bal : ~bal;
    }
    return m;
}

// Writes to a wave's own LDS row are read by other lanes of the same wave: no barrier.
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One round of a wave's stable counting-sort pass over 64 items, one a lane. row[x]: where the
// wave's next item of digit x goes. Returns the item's place (valid items only).
__device__ __forceinline__ uint32_t round_place(uint32_t digit, int bits, bool valid, uint32_t *row)
{
    const uint64_t m = match_digit(digit, bits, __ballot(valid));
    const uint64_t before = m & ((1ull << (threadIdx.x & 63)) - 1ull);
    const uint32_t place = valid ? row[digit] : 0u;
    wave_order();
    if (valid && before == 0) // the lowest lane of each digit
        row[digit] = place + (uint32_t)__popcll(m);
    wave_order();
    return place + (uint32_t)__popcll(before);
}

// The sum of s over the threads before this one (part: a word per wave).
__device__ __forceinline__ uint32_t exclusive_scan(uint32_t s, uint32_t *part)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint32_t inc = s;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t x = __shfl_up(inc, off);
        inc += lane >= off ? x : 0u;
    }
    if (lane == 63)
        part[w] = inc;
    __syncthreads();
    uint32_t run = inc - s;
#pragma unroll
    for (int v = 0; v < kPassWaves - 1; ++v)
        run += v < w ? part[v] : 0u;
    return run;
}

// A digit's counts of every wave, turned into the waves' first places from `run` on.
template <int ND>
__device__ __forceinline__ void wave_places(uint32_t (*rows)[ND], int digit, uint32_t run)
{
    uint32_t c[kPassWaves];
#pragma unroll
    for (int v = 0; v < kPassWaves; ++v)
        c[v] = rows[v][digit];
#pragma unroll
    for (int v = 0; v < kPassWaves; ++v) {
        rows[v][digit] = run;
        run += c[v];
    }
}

// Counts per tile and first digit: tile-major rows of max(4, digits) counts.
__global__ __launch_bounds__(kSortThreads) void sort_count_kernel(RandomOrderDesc d)
{
    __shared__ uint32_t hist[kSortMaxDigits];
    const int t = threadIdx.x;
    const int ndig = 1 << d.high_bits, low = d.key_bits - d.high_bits;
    for (int x = t; x < kSortMaxDigits; x += kSortThreads)
        hist[x] = 0;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * d.tile, lim = min(first + d.tile, (int64_t)d.n);
    for (int64_t r = first; r < lim; r += kSortThreads) {
        const int64_t j = r + t;
        if (j < lim) {
            const uint32_t key = bin_key(d, (uint32_t)j);
            d.keys[j] = (uint16_t)key;
            atomicAdd(&hist[key >> low], 1u);
        }
    }
    __syncthreads();
    const int stride = ndig < 4 ? 4 : ndig;
    for (int x = t; x < stride; x += kSortThreads)
        d.counts[(int64_t)blockIdx.x * stride + x] = x < ndig ? hist[x] : 0u;
}

// base[x] (x < max(4, digits)): where this workgroup's first sample of first digit x goes.
// Thread t sums digits 4g .. 4g + 3 (g = t mod G, G = max(4, digits) / 4 groups) over the
// tiles of range t / G (512 / G ranges), 16-byte loads issued 16 at a time; the ranges are
// added in LDS, then the groups' totals scanned.
__device__ __forceinline__ void tile_bases(const RandomOrderDesc &d, uint32_t *base, uint32_t (*red)[kPassThreads][4],
                                           uint32_t *part)
{
    const int t = threadIdx.x, tile = blockIdx.x;
    const int ndig = 1 << d.high_bits, stride = ndig < 4 ? 4 : ndig;
    const int groups = stride / 4, ranges = kPassThreads / groups;
    const int g = t % groups, r = t / groups;
    const int per = (d.tiles + ranges - 1) / ranges, b_lo = min(r * per, d.tiles), b_hi = min(b_lo + per, d.tiles);
    uint32_t tot[4] = {0u, 0u, 0u, 0u}, pre[4] = {0u, 0u, 0u, 0u};
    for (int b0 = b_lo; b0 < b_hi; b0 += 16) {
        uint4 x[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            x[q] = make_uint4(0u, 0u, 0u, 0u);
            if (b0 + q < b_hi)
                x[q] = *(const uint4 *)(d.counts + (int64_t)(b0 + q) * stride + 4 * g);
        }
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const uint32_t e[4] = {x[q].x, x[q].y, x[q].z, x[q].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                tot[c] += e[c];
                pre[c] += b0 + q < tile ? e[c] : 0u;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        red[0][t][c] = tot[c];
        red[1][t][c] = pre[c];
    }
    __syncthreads();
    uint32_t s = 0;
    if (t < groups) {
        for (int q = 1; q < ranges; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                tot[c] += red[0][q * groups + t][c];
                pre[c] += red[1][q * groups + t][c];
            }
        s = tot[0] + tot[1] + tot[2] + tot[3];
    }
    uint32_t run = exclusive_scan(s, part);
    if (t < groups) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            base[4 * t + c] = run + pre[c];
            run += tot[c];
        }
    }
    __syncthreads();
}

// The first pass (see the top of the file): the final order for keys of at most ten bits;
// else keys and sample indices into the alternate buffers, grouped by their top eight bits,
// and (workgroup 0) each group's start.
__global__ __launch_bounds__(kPassThreads) void sort_first_pass_kernel(RandomOrderDesc d)
{
    __shared__ uint32_t base[kSortMaxDigits];
    __shared__ uint32_t rows[kPassWaves][kSortMaxDigits];
    __shared__ uint32_t red[2][kPassThreads][4];
    __shared__ uint32_t part[kPassWaves];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ndig = 1 << d.high_bits, low = d.key_bits - d.high_bits;
    for (int x = t; x < kPassWaves * kSortMaxDigits; x += kPassThreads)
        rows[0][x] = 0;
    __syncthreads();
    // The wave's part of the tile.
    const int64_t end = min((int64_t)(blockIdx.x + 1) * d.tile, (int64_t)d.n);
    const int per = (d.tile + kPassThreads - 1) / kPassThreads * 64;
    const int64_t first = (int64_t)blockIdx.x * d.tile + (int64_t)w * per, lim = min(first + per, end);
    uint32_t *row = rows[w];
    auto load = [&](int64_t c0, uint32_t (&key)[kPassRegs]) {
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k) {
            const int64_t j = c0 + k * 64 + lane;
            key[k] = j < lim ? d.keys[j] : 0u;
        }
    };
    for (int64_t c0 = first; c0 < lim; c0 += kPassRegs * 64) {
        uint32_t key[kPassRegs];
        load(c0, key);
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k)
            if (c0 + k * 64 + lane < lim)
                atomicAdd(&row[key[k] >> low], 1u);
    }
    tile_bases(d, base, red, part);
    if (low && blockIdx.x == 0) {
        for (int x = t; x < ndig; x += kPassThreads)
            d.seg[x] = base[x];
        if (t == 0)
            d.seg[ndig] = (uint32_t)d.n;
    }
    for (int x = t; x < ndig; x += kPassThreads)
        wave_places(rows, x, base[x]);
    __syncthreads();
    uint32_t *out = low ? d.vals_alt : d.vals;
    for (int64_t c0 = first; c0 < lim; c0 += kPassRegs * 64) {
        uint32_t key[kPassRegs];
        load(c0, key);
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k) {
            if (c0 + k * 64 >= lim)
                break; // uniform over the wave
            const int64_t j = c0 + k * 64 + lane;
            const bool valid = j < lim;
            const uint32_t pos = round_place(key[k] >> low, d.high_bits, valid, row);
            if (valid && pos < (uint32_t)d.n) {
                out[pos] = (uint32_t)j;
                if (low)
                    d.keys_alt[pos] = (uint16_t)key[k];
            }
        }
    }
}

__global__ __launch_bounds__(kPassThreads) void sort_segment_kernel(RandomOrderDesc d)
{
    __shared__ uint32_t rows[kPassWaves][256];
    __shared__ uint32_t part[kPassWaves];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6), h = blockIdx.x;
    const int low = d.key_bits - d.high_bits, nlow = 1 << low;
    const uint32_t lmask = (uint32_t)nlow - 1u;
    const uint32_t start = d.seg[h], end = d.seg[h + 1];
    for (int x = t; x < kPassWaves * 256; x += kPassThreads)
        rows[0][x] = 0;
    __syncthreads();
    // The wave's part of the segment.
    const int64_t per = ((int64_t)end - start + kPassThreads - 1) / kPassThreads * 64;
    const int64_t first = (int64_t)start + w * per, lim = min(first + per, (int64_t)end);
    uint32_t *row = rows[w];
    for (int64_t c0 = first; c0 < lim; c0 += kPassRegs * 64) {
        uint32_t key[kPassRegs];
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k) {
            const int64_t i = c0 + k * 64 + lane;
            key[k] = i < lim ? d.keys_alt[i] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k)
            if (c0 + k * 64 + lane < lim)
                atomicAdd(&row[key[k] & lmask], 1u);
    }
    __syncthreads();
    uint32_t total = 0;
    if (t < nlow)
#pragma unroll
        for (int v = 0; v < kPassWaves; ++v)
            total += rows[v][t];
    const uint32_t before = exclusive_scan(total, part);
    if (t < nlow)
        wave_places(rows, t, start + before);
    __syncthreads();
    for (int64_t c0 = first; c0 < lim; c0 += kPassRegs * 64) {
        uint32_t key[kPassRegs], val[kPassRegs];
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k) {
            const int64_t i = c0 + k * 64 + lane;
            key[k] = i < lim ? d.keys_alt[i] : 0u;
            val[k] = i < lim ? d.vals_alt[i] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kPassRegs; ++k) {
            if (c0 + k * 64 >= lim)
                break; // uniform over the wave
            const bool valid = c0 + k * 64 + lane < lim;
            const uint32_t pos = round_place(key[k] & lmask, low, valid, row);
            if (valid && pos < end)
                d.vals[pos] = val[k];
        }
    }
}

// The train kernel's tiles of 1,024 slots, each reordered in place along a path through its
// bins (stable within a path step, so the order stays the same on every run): a bin's four
// 16-texel-wide strips left to right, down the first, up the next, in steps of four rows, so
// that the path leaves a bin at the corner where the next one of its row begins and 32
// consecutive samples (a wave of the train kernel) lie close together (16 x 32 texels where
// a 16th of the texels is drawn). Keys {bin, path step, slot} are distinct, so a bitonic sort
// gives one result: four keys a thread, strides of 256 and 512 in the thread, up to 32 by
// lane exchanges, 64 and 128 through LDS. 8 us for 262,144 samples, 14 us for a million
// (latency of the 55 exchange steps), which buys the train kernel's scatter 56 and 418 us.
__global__ __launch_bounds__(kSortThreads) void sort_path_kernel(RandomOrderDesc d)
{
    constexpr int kN = kRandomPathTile, kK = kN / kSortThreads;
    static_assert(kN == 1024 && kK == 4, "ten slot bits in the key; four keys a thread");
    __shared__ uint32_t xch[kN], val[kN];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kN;
    const int m = (int)min((int64_t)kN, (int64_t)d.n - base);
    uint32_t key[kK];
#pragma unroll
    for (int k = 0; k < kK; ++k) {
        const int i = k * kSortThreads + t;
        key[k] = 0xFFFFFFFFu;
        if (i < m) {
            const uint32_t idx = d.vals[base + i];
            val[i] = idx;
            uint32_t tx, ty;
            random_texel(mix_seed(idx, d.step), d.image_w, d.image_h, tx, ty);
            const uint32_t bin = (ty >> 6) * (uint32_t)d.bins_x + (tx >> 6);
            const uint32_t strip = (tx >> 4) & 3u, row = (ty >> 2) & 15u;
            key[k] = (bin << 16) | (strip << 14) | ((strip & 1u ? 15u - row : row) << 10) | (uint32_t)i;
        }
    }
#pragma unroll
    for (int size = 2; size <= kN; size <<= 1) {
#pragma unroll
        for (int j = size >> 1; j > 0; j >>= 1) {
            if (j >= kSortThreads) {
                const int dk = j / kSortThreads;
#pragma unroll
                for (int k = 0; k < kK; ++k)
                    if (!(k & dk)) {
                        const bool up = ((k * kSortThreads) & size) == 0; // size > 256: the thread's bits do not matter
                        const uint32_t a = key[k], b = key[k | dk];
                        key[k] = up ? min(a, b) : max(a, b);
                        key[k | dk] = up ? max(a, b) : min(a, b);
                    }
                continue;
            }
            if (j >= 64) {
                __syncthreads(); // the last exchange's reads are done
#pragma unroll
                for (int k = 0; k < kK; ++k)
                    xch[k * kSortThreads + t] = key[k];
                __syncthreads();
            }
#pragma unroll
            for (int k = 0; k < kK; ++k) {
                const int i = k * kSortThreads + t;
                const uint32_t other = j >= 64 ? xch[i ^ j] : (uint32_t)__shfl_xor((int)key[k], j);
                const bool low = ((i & j) == 0) == ((i & size) == 0);
                key[k] = low ? min(key[k], other) : max(key[k], other);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kK; ++k) {
        const int i = k * kSortThreads + t;
        if (i < m)
            d.vals[base + i] = val[key[k] & (kN - 1)];
    }
}

} // namespace

void random_order_tiles(int n, int *tile, int *tiles)
{
    // Tiles of 4,096 samples, at most 256 of them (a whole multiple of 256 samples each).
    int64_t t = kRandomSortTile;
    if (((int64_t)n + t - 1) / t > kRandomSortMaxTiles)
        t = (((int64_t)n + kRandomSortMaxTiles - 1) / kRandomSortMaxTiles + 255) / 256 * 256;
    *tile = (int)t;
    *tiles = (int)(((int64_t)n + t - 1) / t);
}

int random_order_high_bits(int key_bits, int tiles)
{
    // One pass when each workgroup's read of all tiles' counts stays within 64 Ki counts.
    const int64_t stride = key_bits < 2 ? 4 : (int64_t)1 << key_bits;
    if (key_bits <= 10 && stride * tiles <= 65536)
        return key_bits;
    return key_bits < 8 ? key_bits : 8;
}

static size_t random_order_seg_offset(int tiles, int high_bits)
{
    const size_t ndig = (size_t)1 << high_bits;
    return ((ndig < 4 ? 4 : ndig) * (size_t)tiles + 63) / 64 * 64;
}

size_t random_order_count_bytes(int n, int key_bits)
{
    int tile, tiles;
    random_order_tiles(n, &tile, &tiles);
    const int high = random_order_high_bits(key_bits, tiles);
    const size_t ndig = (size_t)1 << high;
    // The counts, then the first digits' segment starts (two-pass keys).
    return random_order_seg_offset(tiles, high) * sizeof(uint32_t) + (ndig + 1) * sizeof(uint32_t);
}

size_t random_order_count_bytes_bound()
{
    // One pass: at most 64 Ki counts; two: 256 digits of at most 256 tiles.
    static_assert(256 * kRandomSortMaxTiles <= 65536, "two-pass counts");
    return 65536 * sizeof(uint32_t) + (kSortMaxDigits + 1) * sizeof(uint32_t);
}

hipError_t launch_random_order(const RandomOrderDesc &d, hipStream_t s, const uint32_t **order)
{
    int tile, tiles;
    random_order_tiles(d.n, &tile, &tiles);
    if (d.n <= 0 || d.key_bits < 1 || d.key_bits > 16 || d.tile != tile || d.tiles != tiles ||
        d.high_bits != random_order_high_bits(d.key_bits, d.tiles))
        return hipErrorInvalidValue;
    RandomOrderDesc e = d;
    e.seg = d.counts + random_order_seg_offset(d.tiles, d.high_bits);
    hipLaunchKernelGGL(sort_count_kernel, dim3((unsigned)e.tiles), dim3(kSortThreads), 0, s, e);
    hipLaunchKernelGGL(sort_first_pass_kernel, dim3((unsigned)e.tiles), dim3(kPassThreads), 0, s, e);
    if (e.key_bits > e.high_bits)
        hipLaunchKernelGGL(sort_segment_kernel, dim3(1u << e.high_bits), dim3(kPassThreads), 0, s, e);
    *order = e.vals;
    return hipGetLastError();
}

hipError_t launch_random_path(const RandomOrderDesc &d, hipStream_t s)
{
    // Bins of 64 x 64 texels, at most 65,536 of them (random_order's 16-bit keys).
    if (d.n <= 0 || d.bin_shift != 6)
        return hipErrorInvalidValue;
    const int tiles = (int)(((int64_t)d.n + kRandomPathTile - 1) / kRandomPathTile);
    hipLaunchKernelGGL(sort_path_kernel, dim3((unsigned)tiles), dim3(kSortThreads), 0, s, d);
    return hipGetLastError();
}

} // namespace ntk
