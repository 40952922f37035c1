// Stable LSD radix sort of (u32 key, u32 value) pairs, digits of 8 or 10 bits,
// for wave64.  Each pass: per-block digit counts -> device scan (digit-major) ->
// scatter with stable block-local ranks computed by per-wave ballot matching.
// Stability is what makes equal tile keys keep the emission order that the
// per-pixel f32 sums depend on.
#pragma once

#include "scan.hpp"

namespace ochre {

// Threads per block: 512 for large inputs with 10-bit digits, where a block's 1,024
// counts are stored and read a line apart (plain call of 10,000 glyphs: k_rs_count
// 31.7 -> 25.1 us a pass, the call 832 -> 806).
inline constexpr int rs_threads(int bits, int items) { return bits == 10 && items == 16 ? 512 : 256; }
// Keys per thread: 16, or 4 for small inputs, whose blocks would otherwise be too
// few to reach every CU (a plain call of 61 glyphs, 15,000 keys: 270 us with 4,
// 278 with 16; 150,000 keys 308 / 326, 300,000 348 / 348, 600,000 450 / 416).
constexpr int RS_ITEMS_LARGE = 16, RS_ITEMS_SMALL = 4;
constexpr int64_t RS_SMALL = (int64_t)1 << 18;  // keys up to which a block takes 4 per thread
inline int rs_items(int64_t n) { return n <= RS_SMALL ? RS_ITEMS_SMALL : RS_ITEMS_LARGE; }
// Digit width: 10 bits where that saves a pass over 8 (a plain call of 2,500 glyphs,
// 18-bit keys: 438 -> 417 us, 10,000 glyphs, 20 bits: 838 -> 827; k_rs_scatter 50 us
// a pass either way on 2.4 million keys).
inline int rs_digit_bits(int key_bits) { return (key_bits + 9) / 10 < (key_bits + 7) / 8 ? 10 : 8; }

__device__ inline uint64_t lanemask_lt() {
    const int lane = lane_id();
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// counts[digit * nblocks + block]
template <int BITS, int ITEMS>
__global__ __launch_bounds__(rs_threads(BITS, ITEMS)) void k_rs_count(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                    uint32_t* __restrict__ counts, uint32_t nblocks) {
    constexpr int DIGITS = 1 << BITS, RS_NT = rs_threads(BITS, ITEMS), RS_WAVES = RS_NT / WAVE;
    __shared__ uint32_t hist[RS_WAVES][DIGITS];
    const int tid = threadIdx.x;
    const int wid = tid / WAVE;
    for (int i = tid; i < RS_WAVES * DIGITS; i += RS_NT) (&hist[0][0])[i] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (RS_NT * ITEMS);
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        int64_t i = base + (int64_t)j * RS_NT + tid;
        if (i < n) {
            uint32_t d = (keys[i] >> shift) & (DIGITS - 1u);
            atomicAdd(&hist[wid][d], 1u);
        }
    }
    __syncthreads();
    for (int d = tid; d < DIGITS; d += RS_NT) {
        uint32_t s = 0;
#pragma unroll
        for (int w = 0; w < RS_WAVES; w++) s += hist[w][d];
        counts[(int64_t)d * nblocks + blockIdx.x] = s;
    }
}

// Scatter.  offsets[digit * nblocks + block] = exclusive global start.
// The block's pairs are first placed in LDS in digit order (block-local stable
// positions: digit start + the wave's offset in the digit + the rank within
// the wave), then written out in that order, so that consecutive threads
// store consecutive addresses of one digit's run.
template <int BITS, int ITEMS>
struct RsScatterLds {
    static constexpr int DIGITS = 1 << BITS, RS_NT = rs_threads(BITS, ITEMS), RS_WAVES = RS_NT / WAVE,
                         TILE_KEYS = RS_NT * ITEMS;
    uint16_t cnt[RS_WAVES][DIGITS];  // per wave and digit: count, then the wave's start within the digit
    uint16_t dstart[DIGITS];         // the digit's first position in the block
    uint32_t goff[DIGITS];           // the digit's global start for this block
    uint32_t wtot[RS_WAVES];
    uint32_t buf[TILE_KEYS];  // keys, then values, in digit order
    uint16_t dig[TILE_KEYS];  // the digit at each position
};

template <int BITS, int ITEMS>
__global__ __launch_bounds__(rs_threads(BITS, ITEMS), 4) void k_rs_scatter(const uint32_t* __restrict__ keys_in,
                                                      const uint32_t* __restrict__ vals_in, int64_t n, int shift,
                                                      const uint32_t* __restrict__ offsets, uint32_t nblocks,
                                                      uint32_t* __restrict__ keys_out,
                                                      uint32_t* __restrict__ vals_out) {
    using Lds = RsScatterLds<BITS, ITEMS>;
    constexpr int DIGITS = Lds::DIGITS, RS_NT = Lds::RS_NT, RS_WAVES = Lds::RS_WAVES, PER = DIGITS / RS_NT;  // consecutive digits per thread
    __shared__ Lds s;
    const int tid = threadIdx.x;
    const int wid = tid / WAVE;
    const int lane = lane_id();
    for (int i = tid; i < RS_WAVES * DIGITS; i += RS_NT) (&s.cnt[0][0])[i] = 0;
    for (int d = tid; d < DIGITS; d += RS_NT) s.goff[d] = offsets[(int64_t)d * nblocks + blockIdx.x];
    __syncthreads();
    const uint64_t lt = lanemask_lt();
    // Items of wave w: base + w*64*ITEMS + j*64 + lane, so (j, lane) order is index order.
    const int64_t bbase = (int64_t)blockIdx.x * Lds::TILE_KEYS;
    const int64_t wbase = bbase + (int64_t)wid * (WAVE * ITEMS);
    const int nb = (int)(n - bbase < (int64_t)Lds::TILE_KEYS ? n - bbase : (int64_t)Lds::TILE_KEYS);  // items in this block
    uint32_t key[ITEMS], val[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        int64_t i = wbase + (int64_t)j * WAVE + lane;
        key[j] = i < n ? keys_in[i] : 0u;
        val[j] = i < n ? vals_in[i] : 0u;
    }
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        bool valid = wbase + (int64_t)j * WAVE + lane < n;
        uint32_t d = (key[j] >> shift) & (DIGITS - 1u);
        uint64_t match = __ballot(valid);
#pragma unroll
        for (int b = 0; b < BITS; b++) {
            uint64_t m = __ballot((d >> b) & 1u);
            match &= ((d >> b) & 1u) ? m : ~m;
        }
        uint32_t prior = valid ? s.cnt[wid][d] : 0u;
        rank[j] = prior + (uint32_t)__popcll(match & lt);
        // The lowest lane of each match group advances the wave-private counter.
        if (valid && (match & lt) == 0) s.cnt[wid][d] = (uint16_t)(prior + (uint32_t)__popcll(match));
    }
    __syncthreads();
    // per digit: the waves' starts within the digit, and the digit's total; the
    // digits' starts in the block by a scan of the totals
    {
        uint32_t tot[PER], sum = 0;
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int d = tid * PER + k;
            tot[k] = 0;
#pragma unroll
            for (int w = 0; w < RS_WAVES; w++) {
                const uint32_t c = s.cnt[w][d];
                s.cnt[w][d] = (uint16_t)tot[k];
                tot[k] += c;
            }
            sum += tot[k];
        }
        const uint32_t incl = wave_incl_scan(sum, OpAdd());
        if (lane == WAVE - 1) s.wtot[wid] = incl;
        __syncthreads();
        uint32_t at = incl - sum;
#pragma unroll
        for (int w = 0; w < RS_WAVES; w++)
            if (w < wid) at += s.wtot[w];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            s.dstart[tid * PER + k] = (uint16_t)at;
            at += tot[k];
        }
    }
    __syncthreads();
    // rank[j] becomes the item's position in the block
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        if (wbase + (int64_t)j * WAVE + lane < n) {
            const uint32_t d = (key[j] >> shift) & (DIGITS - 1u);
            rank[j] += (uint32_t)s.dstart[d] + s.cnt[wid][d];
            s.buf[rank[j]] = key[j];
            s.dig[rank[j]] = (uint16_t)d;
        }
    }
    __syncthreads();
    for (int i = tid; i < nb; i += RS_NT) {
        const uint32_t d = s.dig[i];
        keys_out[s.goff[d] + (uint32_t)i - s.dstart[d]] = s.buf[i];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < ITEMS; j++)
        if (wbase + (int64_t)j * WAVE + lane < n) s.buf[rank[j]] = val[j];
    __syncthreads();
    for (int i = tid; i < nb; i += RS_NT) {
        const uint32_t d = s.dig[i];
        vals_out[s.goff[d] + (uint32_t)i - s.dstart[d]] = s.buf[i];
    }
}

}  // namespace ochre
