// mpm_sort.hip -- stable LSD radix sort of u32 keys with their input index.
//
// Same contract as molla's RadixSortKernel (molla-compute-primitives/src/
// radix_sort.rs:1-30): stable, so ties keep their input order; the values are
// the input indices 0..n-1, which is what every caller sorts.  Only the key
// bits that can be non-zero are sorted, in equal digits of at most
// radix_plan's width.  Each pass is three launches:
//   k_radix_hist     per-block digit histogram (blocks of 4096 keys, LDS atomics)
//   k_radix_rows     per digit: exclusive scan of the blocks' counts, total
//   k_radix_scatter  the digits' bases from the totals, then a stable scatter:
//                    each wave ranks its 512 (wide digits: 1024) consecutive
//                    keys in rounds of 64 with ballots (the lanes that share a digit) and digit
//                    counters of its own, with no barrier between the rounds,
//                    and the block's keys leave through LDS in digit order.
// What bounds a pass at 2 M keys is the scatter: a block's latency (its loads,
// the ballots, whose rounds overlap bit by bit, the stage) with two blocks per
// CU.  Wide digits trade passes for counters: 18 key bits (a 256^3 grid) are
// two passes of 9 bits.  A key query of 2 M random particles takes 66 us
// (scatter 15, histogram 5, rows 4 us per pass); three passes of 8 bits with
// barriers in every round, unstaged stores and a three-launch scan took 154.
#include <algorithm>

#include "mpm_internal.hpp"
#include "mpm_blockscan.hpp"
#include "mpm_radix_plan.hpp"

namespace mpm {

// Threads of a block, by its digits: eight waves rank 512 keys each in half
// the rounds of four, but hold twice the counters, whose clear and sums come
// to outweigh the rounds at 4096 digits.  A key query, four waves / eight: of
// 20,000 keys in one pass of 12 bits 41.8 / 46.2 us, of 60,000 in two of 7
// 49.8 / 43.3, of 400,000 in two of 8 54.8 / 48.2, of 2 M in two of 9 71.6 /
// 66.8 us.  Sixteen waves gain another 1 us at 60,000 and nothing at 2 M.
constexpr int MANY_DIGIT = 10;  // eight waves up to this width
template <int THREADS>
struct SortShape {
    static constexpr int WAVES = THREADS / 64, ITEMS = SORT_TILE / THREADS;
    static constexpr int PER = (1 << (THREADS == 512 ? MANY_DIGIT : MAX_DIGIT)) / THREADS;  // digits per thread
};

uint32_t* radix_input(uint32_t* keys, uint32_t n, int bits, uint32_t* scratch) {
    return radix_plan(n, bits).passes % 2 ? scratch : keys;
}

template <int SORT_THREADS>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_hist(const uint32_t* __restrict__ keys, uint32_t n, int shift,
                                                             int width, uint32_t* __restrict__ hist) {
    constexpr int SORT_ITEMS = SortShape<SORT_THREADS>::ITEMS;
    extern __shared__ uint32_t lds[];
    const uint32_t R = 1u << width;
    for (uint32_t d = threadIdx.x; d < R; d += SORT_THREADS) lds[d] = 0u;
    __syncthreads();
    const uint32_t base = blockIdx.x * SORT_TILE;
    uint32_t k[SORT_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        const uint32_t i = base + r * SORT_THREADS + threadIdx.x;
        k[r] = i < n ? keys[i] : 0u;
    }
    // keys in nearly sorted order put a wave on one digit, whose 64 adds to
    // one word would run one after the other: such a wave adds once
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        const uint32_t d = (k[r] >> shift) & (R - 1u);
        const bool valid = base + r * SORT_THREADS + threadIdx.x < n;
        const uint64_t all = __ballot(valid);
        if (__ballot(valid && d == (uint32_t)__builtin_amdgcn_readfirstlane(int(d))) == all) {
            if (valid && (threadIdx.x & 63u) == 0u) atomicAdd(&lds[d], (uint32_t)__popcll(all));
        } else if (valid) {
            atomicAdd(&lds[d], 1u);
        }
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < R; d += SORT_THREADS) hist[(size_t)blockIdx.x * R + d] = lds[d];
}

// hist is block-major ([block][digit], so that the kernels around this one
// move whole rows): each digit's exclusive sum over the blocks in place, and
// its total.  A block takes ROW_DIGITS digits; its threads split the blocks
// into ROW_SEGS segments, whose sums one wave per digit scans.  Bound by its
// two rounds of loads, one of which goes where a segment's counts fit in
// registers (up to 512 blocks, 2 M keys): a key query of 2 M 67.6 -> 66.0 us.
constexpr int ROW_DIGITS = 16;
constexpr int ROW_SEGS = 64;
constexpr int ROW_HELD = 8;
__global__ __launch_bounds__(ROW_DIGITS * ROW_SEGS) void k_radix_rows(uint32_t* __restrict__ hist, uint32_t nblocks,
                                                                      uint32_t R, uint32_t* __restrict__ total) {
    __shared__ uint32_t part[ROW_SEGS][ROW_DIGITS + 1];
    const uint32_t c = threadIdx.x % ROW_DIGITS, seg = threadIdx.x / ROW_DIGITS;
    const uint32_t d = blockIdx.x * ROW_DIGITS + c;
    const uint32_t len = (nblocks + ROW_SEGS - 1u) / ROW_SEGS;
    const uint32_t b0 = min(seg * len, nblocks), b1 = min(b0 + len, nblocks);
    // up to ROW_HELD rows stay in registers, so that their counts are read once
    const bool held = len <= uint32_t(ROW_HELD);
    uint32_t v[ROW_HELD];
    uint32_t sum = 0u;
    if (held) {
#pragma unroll
        for (int q = 0; q < ROW_HELD; ++q) {
            v[q] = d < R && b0 + q < b1 ? hist[(size_t)(b0 + q) * R + d] : 0u;
            sum += v[q];
        }
    } else if (d < R) {
#pragma unroll 8
        for (uint32_t b = b0; b < b1; ++b) sum += hist[(size_t)b * R + d];
    }
    part[seg][c] = sum;
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;  // wave w scans digit w
    {
        const uint32_t mine = part[lane][wave], incl = wave_incl_scan(mine);
        part[lane][wave] = incl - mine;
        if (lane == 63u && blockIdx.x * ROW_DIGITS + wave < R) total[blockIdx.x * ROW_DIGITS + wave] = incl;
    }
    __syncthreads();
    if (d >= R) return;
    uint32_t run = part[seg][c];
    if (held) {
#pragma unroll
        for (int q = 0; q < ROW_HELD; ++q) {
            if (b0 + q < b1) hist[(size_t)(b0 + q) * R + d] = run;
            run += v[q];
        }
        return;
    }
#pragma unroll 8
    for (uint32_t b = b0; b < b1; ++b) {
        const uint32_t h = hist[(size_t)b * R + d];
        hist[(size_t)b * R + d] = run;
        run += h;
    }
}
static_assert(ROW_SEGS == 64, "one lane per segment");

// vin null: the values are the indices.  lb (may be null; single-pass sorts
// only): receives the first position of every key in [0, n_lb].
template <int SORT_THREADS>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_scatter(const uint32_t* __restrict__ kin,
                                                                const uint32_t* __restrict__ vin,
                                                                uint32_t* __restrict__ kout,
                                                                uint32_t* __restrict__ vout, uint32_t n, int shift,
                                                                int width, const uint32_t* __restrict__ hist,
                                                                const uint32_t* __restrict__ total,
                                                                uint32_t* __restrict__ lb, uint32_t n_lb) {
    constexpr int SORT_WAVES = SortShape<SORT_THREADS>::WAVES, SORT_ITEMS = SortShape<SORT_THREADS>::ITEMS;
    constexpr uint32_t PER = SortShape<SORT_THREADS>::PER;
    extern __shared__ uint32_t lds[];
    __shared__ uint32_t s_wave[64];
    const uint32_t R = 1u << width;
    uint32_t* base = lds;  // R words: where the block's keys of a digit go, less their place in the stage
    uint16_t* cnt = reinterpret_cast<uint16_t*>(lds + R);  // [digit][wave]
    uint32_t *skey = lds + R, *sval = skey + SORT_TILE;                      // the stage, once cnt is done with
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t first = blockIdx.x * SORT_TILE + uint32_t(wave) * (SORT_ITEMS * 64);
    uint32_t key[SORT_ITEMS], val[SORT_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        const uint32_t i = first + r * 64 + lane;
        key[r] = i < n ? kin[i] : 0u;
        val[r] = vin && i < n ? vin[i] : i;
    }
    for (uint32_t i = tid; i < R * SORT_WAVES / 2; i += SORT_THREADS) lds[R + i] = 0u;
    // a thread holds R / threads digits in a row (one where R is less)
    const uint32_t per = R > uint32_t(SORT_THREADS) ? R / SORT_THREADS : 1u, d0 = uint32_t(tid) * per;
    uint32_t tot[PER], at[PER];
    uint32_t sum = 0u;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        const bool on = q < per && d0 + q < R;
        tot[q] = on ? total[d0 + q] : 0u;
        at[q] = on ? hist[(size_t)blockIdx.x * R + d0 + q] : 0u;
        sum += tot[q];
    }
    uint32_t run = block_excl_scan(sum, s_wave, (uint32_t*)nullptr);
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        if (q >= per || d0 + q >= R) continue;
        if (lb && blockIdx.x == 0 && d0 + q <= n_lb) lb[d0 + q] = run;
        at[q] += run;
        run += tot[q];
    }
    if (lb && blockIdx.x == 0 && tid == 0 && n_lb >= R) lb[R] = n;
    // the lanes of each round that share a digit: one bit of all rounds at a
    // time, so that the rounds' ballots overlap
    const uint64_t lt = (1ull << lane) - 1ull;
    uint64_t same[SORT_ITEMS];
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) same[r] = __ballot(first + r * 64 + lane < n);
    for (int bit = shift; bit < shift + width; ++bit)
#pragma unroll
        for (int r = 0; r < SORT_ITEMS; ++r) {
            const bool on = (key[r] >> bit) & 1u;
            const uint64_t m = __ballot(on);
            same[r] &= on ? m : ~m;
        }
    uint32_t rank[SORT_ITEMS];
    auto counter = [&](int r) { return ((key[r] >> shift) & (R - 1u)) * SORT_WAVES + uint32_t(wave); };
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        rank[r] = 0u;
        if (first + r * 64 + lane < n) rank[r] = counter_add(cnt, counter(r), same[r], lt);
    }
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r)
        rank[r] = counter_half(rank[r], counter(r)) - (uint32_t)__popcll(same[r] & ~lt);
    __syncthreads();
    // places in the stage: digits ascending, the waves' keys of a digit in order
    static_assert(SORT_WAVES % 4 == 0, "four counters of a digit are one word");
    constexpr int CW = SORT_WAVES / 4;
    uint64_t* cnt4 = reinterpret_cast<uint64_t*>(cnt);
    uint64_t c4[PER][CW];
    uint32_t mine = 0u;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q)
#pragma unroll
        for (int w = 0; w < CW; ++w) {
            const uint64_t c = q < per && d0 + q < R ? cnt4[(d0 + q) * CW + w] : 0ull;
            mine += uint32_t(c & 0xffffu) + uint32_t((c >> 16) & 0xffffu) + uint32_t((c >> 32) & 0xffffu) +
                    uint32_t(c >> 48);
            c4[q][w] = c;
        }
    uint32_t place = block_excl_scan(mine, s_wave, (uint32_t*)nullptr);
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
        if (q >= per || d0 + q >= R) continue;
        base[d0 + q] = at[q] - place;
#pragma unroll
        for (int w = 0; w < CW; ++w) {
            uint64_t out = 0ull;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                out |= uint64_t(place) << (16 * k);
                place += uint32_t(c4[q][w] >> (16 * k)) & 0xffffu;
            }
            cnt4[(d0 + q) * CW + w] = out;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r)
        rank[r] += cnt[((key[r] >> shift) & (R - 1u)) * SORT_WAVES + uint32_t(wave)];
    __syncthreads();  // the stage overwrites the counters
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        if (first + r * 64 + lane >= n) continue;
        skey[rank[r]] = key[r];
        sval[rank[r]] = val[r];
    }
    __syncthreads();
    // staged order: a digit's keys leave as one run
    const uint32_t held = min(n - blockIdx.x * SORT_TILE, uint32_t(SORT_TILE));
#pragma unroll
    for (int r = 0; r < SORT_ITEMS; ++r) {
        const uint32_t i = r * SORT_THREADS + tid;
        if (i >= held) continue;
        const uint32_t k = skey[i], pos = base[(k >> shift) & (R - 1u)] + i;
        kout[pos] = k;
        vout[pos] = sval[i];
    }
}

hipError_t radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t n, int bits, uint32_t* scratch, uint32_t* lb,
                            uint32_t n_lb, bool* lb_done, hipStream_t s) {
    if (lb_done) *lb_done = false;
    if (n == 0) return hipSuccess;
    const uint32_t nb = sort_blocks(n);
    const RadixPlan plan = radix_plan(n, bits);
    const uint32_t R = 1u << plan.width;
    uint32_t* k2 = scratch;
    uint32_t* v2 = scratch + n;
    uint32_t* hist = scratch + 2 * (size_t)n;
    uint32_t* total = hist + (size_t)R * nb;
    const uint32_t* kin = radix_input(keys, n, bits, scratch);
    const uint32_t* vin = nullptr;  // the first pass's values are the indices
    const bool with_lb = lb && plan.passes == 1;
    for (int p = 0; p < plan.passes; ++p) {
        const int shift = plan.width * p;
        uint32_t *kout = kin == keys ? k2 : keys, *vout = kin == keys ? v2 : vals;
        const bool many = plan.width <= MANY_DIGIT;
        const dim3 threads(many ? 512 : 256);
        auto* khist = many ? k_radix_hist<512> : k_radix_hist<256>;
        auto* kscatter = many ? k_radix_scatter<512> : k_radix_scatter<256>;
        hipLaunchKernelGGL(khist, dim3(nb), threads, R * 4, s, kin, n, shift, plan.width, hist);
        hipLaunchKernelGGL(k_radix_rows, dim3((R + ROW_DIGITS - 1) / ROW_DIGITS), dim3(ROW_DIGITS * ROW_SEGS), 0, s, hist,
                           nb, R, total);
        hipLaunchKernelGGL(kscatter, dim3(nb), threads,
                           R * 4 + std::max<uint32_t>(R * (threads.x / 64) * 2, 2 * SORT_TILE * 4), s, kin, vin, kout,
                           vout, n, shift, plan.width, hist, total, with_lb ? lb : nullptr, n_lb);
        kin = kout;
        vin = vout;
    }
    if (lb_done) *lb_done = with_lb;
    return hipGetLastError();
}

}  // namespace mpm
