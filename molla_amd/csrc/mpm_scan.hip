// mpm_scan.hip -- tables of the sorted particle layout: the tile lower-bound
// table, the static active list and the chunk list.
//
// Chunks (one block of the particle pass each, `chunk_cap` = 256 threads x
// particles per thread) are cut from the sorted particle array so that a
// chunk never leaves its tile row.  Two rules:
//   greedy rows (span 4 or 6 tiles; 6 is the default): a chunk starts at
//     each row's first particle and runs for chunk_cap particles or until
//     the next particle would make it span more than `span` tiles, so chunks
//     start anywhere inside a tile and only a row's last chunk (or one cut by
//     the span) is partly filled;
//   aligned segments (8): chunks of chunk_cap from the start of each aligned
//     group of four tiles, or of eight where those eight hold at least two
//     chunks' worth.
// Greedy rows of four tiles make ~10 % fewer chunks than the aligned rule on
// the 2 M scene and ~14 % fewer on the 512-scene batch; six tiles ~11 % and
// ~18 % (boxes up to 27 x 7 x 7 cells at the sort, inside the 1600-cell LDS
// box with room for the motion until the next sort).
//
// A tile's static mark and, at a row's first tile, the row's chunk count are
// functions of the lower-bound table, so one prefix sum over the tiles of the
// pair (mark, chunks) places both lists; nothing runs over the particles.
// What bounds this work on all but the largest scenes is the number of
// dependent launches, hence the shapes below:
//   k_layout_one    up to LAYOUT_ONE particles and LAYOUT_TILES tiles: keys,
//                   sort, table and both lists in one block;
//   k_layout_block  up to LAYOUT_TILES tiles: table and lists in one block;
//   the rest        one launch per step, the prefix sum in three.
// With the chunk spread and the reorder, a sort of 8,192 particles in a 32^3
// grid is 3 launches (36 us of kernels in a trace), of 200,003 in 61^3 7 (73
// us), of 2 M in 256^3 15 (290 us); lists built from per-particle flags took
// 27 to 32 launches and about 130, 190 and 480 us.  The lines: k_layout_one
// still beats the separate launches at its 16,384 particles (36 us against
// ~60), where the 14 bits of a slot and its 16 keys per thread end (98 of the
// CU's 160 KB of LDS are in use); one block walks 8,192 tiles in 15 us, as long
// as the four launches it saves.
#include <algorithm>

#include "mpm_internal.hpp"
#include "mpm_blockscan.hpp"

namespace mpm {

constexpr uint32_t LAYOUT_THREADS = 1024;
constexpr uint32_t LAYOUT_TILES = 8192;
constexpr uint32_t LAYOUT_ONE = 16384;

// The chunk rule of a sorted layout.
struct ChunkRule {
    uint32_t cap;   // particles per chunk
    uint32_t span;  // greedy: tiles per chunk; 0: aligned segments
};

// A tile's scene and coordinates.
struct TilePos {
    const SceneDev* sc;
    uint32_t scene, x, y, z;
};
__device__ __forceinline__ TilePos tile_pos(const SceneDev* scenes, const uint32_t* tile_scene, uint32_t t) {
    TilePos p;
    p.scene = tile_scene[t];
    p.sc = scenes + p.scene;
    const uint32_t W = p.sc->W, tl = t - p.sc->tile_base, r = tl / W;
    p.x = tl - r * W;
    p.z = r / W;
    p.y = r - p.z * W;
    return p;
}

// A tile is on the static list when any tile within one tile of it (each
// axis, same scene) holds a particle: P2G can reach it before the next sort.
// Occupancy of a 3-tile x-run is one difference of the lower-bound table.
template <class LB>
__device__ __forceinline__ bool tile_static(const TilePos& p, LB lb) {
    const int W = int(p.sc->W);
    const uint32_t xa = p.x > 0u ? p.x - 1u : 0u, xb = min(p.x + 1u, uint32_t(W - 1));
    bool on = false;
    for (int dz = -1; dz <= 1; ++dz)
        for (int dy = -1; dy <= 1; ++dy) {
            const int ny = int(p.y) + dy, nz = int(p.z) + dz;
            if (ny < 0 || nz < 0 || ny >= W || nz >= W) continue;
            const uint32_t row = p.sc->tile_base + uint32_t(W * (ny + W * nz));
            on = on || lb(row + xb + 1u) > lb(row + xa);
        }
    return on;
}

// Calls emit(start, count) for every chunk of the tile row starting at tile
// t0 (W tiles), ascending.
template <class LB, class F>
__device__ __forceinline__ void walk_row(LB lb, uint32_t t0, uint32_t W, const ChunkRule& rule, F emit) {
    if (rule.span) {
        const uint32_t end = lb(t0 + W);
        uint32_t s = lb(t0), tt = 0u;
        while (s < end) {
            while (lb(t0 + tt + 1u) <= s) ++tt;  // the tile holding slot s
            const uint32_t nxt = min(s + rule.cap, lb(t0 + min(tt + rule.span, W)));
            emit(s, nxt - s);
            s = nxt;
        }
        return;
    }
    for (uint32_t g8 = 0u; g8 < W; g8 += 8u) {
        const uint32_t e8 = min(g8 + 8u, W);
        const uint32_t step = lb(t0 + e8) - lb(t0 + g8) >= 2u * rule.cap ? 8u : 4u;
        for (uint32_t g = g8; g < e8; g += step) {
            const uint32_t end = lb(t0 + min(g + step, e8));
            for (uint32_t s = lb(t0 + g); s < end; s += rule.cap) emit(s, min(rule.cap, end - s));
        }
    }
}

template <class LB>
__device__ __forceinline__ uint32_t row_chunks(LB lb, uint32_t t0, uint32_t W, const ChunkRule& rule) {
    uint32_t n = 0u;
    walk_row(lb, t0, W, rule, [&](uint32_t, uint32_t) { ++n; });
    return n;
}

// Writes the row's chunks from chunks[at] on; returns the index past the last.
template <class LB>
__device__ __forceinline__ uint32_t emit_row(LB lb, uint32_t t0, const TilePos& p, const ChunkRule& rule, uint32_t at,
                                             Chunk* __restrict__ chunks) {
    walk_row(lb, t0, p.sc->W, rule, [&](uint32_t start, uint32_t count) {
        Chunk ch;
        ch.scene = p.scene;
        ch.start = start;
        ch.count = count;
        ch.pad = chunk_row_tag(p.y, p.z);  // read by stencil_escapes
        chunks[at++] = ch;
    });
    return at;
}

// The static marks and lists of all tiles by one block whose lower-bound
// table is in LDS.  Thread t takes tiles [t K, (t + 1) K).
template <class LB>
__device__ __forceinline__ void layout_lists(LB lb, const LayoutArgs& q, const ChunkRule& rule, uint64_t* s_wave) {
    constexpr uint32_t MOST = LAYOUT_TILES / LAYOUT_THREADS;
    const uint32_t K = (q.total_tiles + LAYOUT_THREADS - 1u) / LAYOUT_THREADS;
    const uint32_t t0 = threadIdx.x * K, cnt = t0 < q.total_tiles ? min(K, q.total_tiles - t0) : 0u;
    uint32_t marks = 0u, rows = 0u, flag[MOST];
    uint64_t sum = 0;  // (static tiles, chunks) of the thread's tiles
#pragma unroll
    for (uint32_t k = 0; k < MOST; ++k) flag[k] = k < cnt ? q.tile_flag[t0 + k] : 0u;
#pragma unroll
    for (uint32_t k = 0; k < MOST; ++k) {
        if (k >= cnt) continue;
        const TilePos p = tile_pos(q.scenes, q.tile_scene, t0 + k);
        if (tile_static(p, lb)) marks |= 1u << k;
        if (p.x == 0u) rows |= 1u << k;
    }
#pragma unroll
    for (uint32_t k = 0; k < MOST; ++k) {
        if (k >= cnt) continue;
        const bool on = (marks >> k) & 1u;
        q.tile_flag[t0 + k] = (flag[k] & ~FLAG_STATIC) | (on ? FLAG_STATIC : 0u);
        sum += on ? 1u : 0u;
    }
    for (uint32_t m = rows; m; m &= m - 1u) {
        const uint32_t t = t0 + uint32_t(__ffs(m) - 1);
        sum += uint64_t(row_chunks(lb, t, q.scenes[q.tile_scene[t]].W, rule)) << 32;
    }
    uint64_t total = 0;
    const uint64_t at = block_excl_scan(sum, s_wave, &total);
    uint32_t si = uint32_t(at), ci = uint32_t(at >> 32);
    for (uint32_t m = marks; m; m &= m - 1u) q.slist[si++] = t0 + uint32_t(__ffs(m) - 1);
    for (uint32_t m = rows; m; m &= m - 1u) {
        const uint32_t t = t0 + uint32_t(__ffs(m) - 1);
        ci = emit_row(lb, t, tile_pos(q.scenes, q.tile_scene, t), rule, ci, q.chunks);
    }
    if (threadIdx.x == 0) {
        *q.scount = uint32_t(total);
        if (q.host_scount) *q.host_scount = uint32_t(total);
        *q.n_chunks = uint32_t(total >> 32);
    }
}

__global__ __launch_bounds__(LAYOUT_THREADS) void k_layout_block(LayoutArgs q, ChunkRule rule) {
    __shared__ uint32_t s_lb[LAYOUT_TILES + 1];
    __shared__ uint64_t s_wave[64];
    for (uint32_t t = threadIdx.x; t <= q.total_tiles; t += LAYOUT_THREADS) s_lb[t] = q.tile_lb[t];
    __syncthreads();
    layout_lists([&](uint32_t t) { return s_lb[t]; }, q, rule, s_wave);
}

// Keys, sort and lists of a small layout.  A key (13 bits) and its slot (14
// bits) share a word, so a pass of the sort moves one word per particle; the
// passes rank as k_radix_scatter does, 16 waves of up to 1024 keys.
constexpr uint32_t ONE_WAVES = LAYOUT_THREADS / 64;
constexpr uint32_t ONE_ITEMS = LAYOUT_ONE / LAYOUT_THREADS;
constexpr uint32_t ONE_FLY = 8;    // rounds of counters in flight
constexpr uint32_t ONE_DIGIT = 9;  // 512 tiles (a 32^3 grid) in one pass

__global__ __launch_bounds__(LAYOUT_THREADS) void k_layout_one(StepArgs a, uint32_t n_scenes, LayoutArgs q,
                                                               ChunkRule rule, int bits,
                                                               const uint32_t* __restrict__ ids) {
    __shared__ uint32_t s_key[LAYOUT_ONE];
    __shared__ alignas(4) uint16_t s_cnt[ONE_WAVES << ONE_DIGIT];
    __shared__ uint32_t s_base[1 << ONE_DIGIT];
    __shared__ uint16_t s_lb[LAYOUT_TILES + 1];
    __shared__ uint64_t s_wave[64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, n = q.n;
    // four particles' loads in flight per thread: their latency, not their
    // number, is what counts in one block.  Slots are read in order, also where
    // the keys go in the order of the ids: a gather through the ids' slots
    // took 22 instead of 13 us for 16,384 particles
    for (uint32_t i0 = tid; i0 < n; i0 += 4u * LAYOUT_THREADS) {
        uint32_t at[4], key[4];
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t i = min(i0 + u * LAYOUT_THREADS, n - 1u);
            at[u] = ids ? min(ids[i], n - 1u) : i;
            if (n_scenes == 1u) {  // the scene in scalar registers
                key[u] = tile_key(a.scenes[0], a.ps, a.cap, i);
                continue;
            }
            uint32_t lo = 0u, hi = n_scenes;  // the last scene starting at or before the slot
            while (hi - lo > 1u) {
                const uint32_t mid = (lo + hi) / 2u;
                if (a.scenes[mid].pbase <= i) lo = mid;
                else hi = mid;
            }
            key[u] = tile_key(a.scenes[lo], a.ps, a.cap, i);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t i = i0 + u * LAYOUT_THREADS;
            if (i < n) s_key[at[u]] = key[u] << 14 | i;
        }
    }
    // rounds of 64 keys per wave: a wave's keys are consecutive
    const uint32_t rounds = (n + LAYOUT_THREADS - 1u) / LAYOUT_THREADS;
    const uint32_t first = wave * rounds * 64u + lane;
    const int passes = (bits + int(ONE_DIGIT) - 1) / int(ONE_DIGIT), width = (bits + passes - 1) / passes;
    const uint32_t R = 1u << width;
    const uint64_t lt = (1ull << lane) - 1ull;
#pragma unroll 1
    for (int pass = 0; pass < passes; ++pass) {
        const int shift = 14 + pass * width;
        for (uint32_t d = tid; d < ONE_WAVES << width; d += LAYOUT_THREADS) s_cnt[d] = 0u;
        __syncthreads();
        // the rounds' ballots overlap, one bit of all rounds at a time
        uint32_t key[ONE_ITEMS], pos[ONE_ITEMS];
        uint64_t same[ONE_ITEMS];
#pragma unroll
        for (uint32_t r = 0; r < ONE_ITEMS; ++r) {
            const uint32_t i = first + r * 64u;
            const bool valid = r < rounds && i < n;
            key[r] = valid ? s_key[i] : 0u;
            same[r] = __ballot(valid);
        }
        for (int bit = shift; bit < shift + width; ++bit)
#pragma unroll
            for (uint32_t r = 0; r < ONE_ITEMS; ++r) {
                const bool on = (key[r] >> bit) & 1u;
                const uint64_t m = __ballot(on);
                same[r] &= on ? m : ~m;
            }
        auto counter = [&](uint32_t r) { return (wave << width) + ((key[r] >> shift) & (R - 1u)); };
#pragma unroll
        for (uint32_t h = 0; h < ONE_ITEMS; h += ONE_FLY) {
#pragma unroll
            for (uint32_t r = h; r < h + ONE_FLY; ++r) {
                pos[r] = 0u;
                if (r < rounds && first + r * 64u < n) pos[r] = counter_add(s_cnt, counter(r), same[r], lt);
            }
#pragma unroll
            for (uint32_t r = h; r < h + ONE_FLY; ++r)
                pos[r] = counter_half(pos[r], counter(r)) - (uint32_t)__popcll(same[r] & ~lt);
            __builtin_amdgcn_sched_barrier(0);  // more in flight does not fit the registers
        }
        __syncthreads();
        uint32_t mine = 0u;  // keys of digit tid (R <= 512 <= threads)
        if (tid < R) {
            uint32_t c[ONE_WAVES];
#pragma unroll
            for (uint32_t w = 0; w < ONE_WAVES; ++w) c[w] = s_cnt[(w << width) + tid];
#pragma unroll
            for (uint32_t w = 0; w < ONE_WAVES; ++w) {
                s_cnt[(w << width) + tid] = uint16_t(mine);
                mine += c[w];
            }
        }
        const uint32_t base = uint32_t(block_excl_scan(uint64_t(mine), s_wave, (uint64_t*)nullptr));
        if (tid < R) s_base[tid] = base;
        __syncthreads();
        // in place: every key is in a register
#pragma unroll
        for (uint32_t r = 0; r < ONE_ITEMS; ++r) {
            const uint32_t d = (key[r] >> shift) & (R - 1u);
            pos[r] += s_base[d] + s_cnt[(wave << width) + d];
        }
#pragma unroll
        for (uint32_t r = 0; r < ONE_ITEMS; ++r)
            if (r < rounds && first + r * 64u < n) s_key[pos[r]] = key[r];
        __syncthreads();
    }
#pragma unroll 4
    for (uint32_t j = tid; j < n; j += LAYOUT_THREADS) {
        q.keys[j] = s_key[j] >> 14;
        q.src[j] = s_key[j] & (LAYOUT_ONE - 1u);
    }
    for (uint32_t t = tid; t <= q.total_tiles; t += LAYOUT_THREADS) {
        uint32_t lo = 0u, hi = n;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) / 2u;
            if ((s_key[mid] >> 14) < t) lo = mid + 1u;
            else hi = mid;
        }
        s_lb[t] = uint16_t(lo);  // n <= 16384
        q.tile_lb[t] = lo;
    }
    __syncthreads();
    layout_lists([&](uint32_t t) { return uint32_t(s_lb[t]); }, q, rule, s_wave);
}

// ---- layouts of any size ----

// tile_lb[k] = first sorted slot whose key is >= k, for k in [0, total].
__global__ void k_tile_lb(const uint32_t* __restrict__ keys, uint32_t n, uint32_t* __restrict__ lb, uint32_t total) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k <= total; k += gridDim.x * blockDim.x) {
        uint32_t first = 0, last = n;
        while (first < last) {
            const uint32_t mid = first + (last - first) / 2;
            if (keys[mid] < k) first = mid + 1;
            else last = mid;
        }
        lb[k] = first;
    }
}

// The (static mark, chunks of the row starting here) pair of each tile.
constexpr int TILE_THREADS = 256;
constexpr uint32_t TILE_SPAN = 1024;  // tiles of lower bounds staged beyond the block's own (rows of up to 1024 tiles)

// A block's tiles with their rows' lower bounds in LDS.
struct TileSpan {
    const uint32_t* s_lb;
    uint32_t t0;
    __device__ __forceinline__ uint32_t operator()(uint32_t t) const { return s_lb[t - t0]; }
};
__device__ __forceinline__ TileSpan stage_span(const LayoutArgs& q, uint32_t* s_lb) {
    const uint32_t t0 = blockIdx.x * TILE_THREADS;
    const uint32_t end = min(t0 + TILE_THREADS + q.max_W, q.total_tiles);  // entries t0 .. end
    for (uint32_t t = t0 + threadIdx.x; t <= end; t += TILE_THREADS) s_lb[t - t0] = q.tile_lb[t];
    __syncthreads();
    return {s_lb, t0};
}

__global__ __launch_bounds__(TILE_THREADS) void k_tile_marks(LayoutArgs q, ChunkRule rule,
                                                             uint64_t* __restrict__ pairs) {
    __shared__ uint32_t s_lb[TILE_THREADS + TILE_SPAN + 1];
    const TileSpan lb = stage_span(q, s_lb);
    const uint32_t t = blockIdx.x * TILE_THREADS + threadIdx.x;
    if (t >= q.total_tiles) return;
    const TilePos p = tile_pos(q.scenes, q.tile_scene, t);
    const bool on = tile_static(p, [&](uint32_t k) { return q.tile_lb[k]; });
    q.tile_flag[t] = (q.tile_flag[t] & ~FLAG_STATIC) | (on ? FLAG_STATIC : 0u);
    pairs[t] = (on ? 1ull : 0ull) | (p.x == 0u ? uint64_t(row_chunks(lb, t, p.sc->W, rule)) << 32 : 0ull);
}

// `pos`: the exclusive prefix sums of the pairs.
__global__ __launch_bounds__(TILE_THREADS) void k_tile_emit(LayoutArgs q, ChunkRule rule,
                                                            const uint64_t* __restrict__ pos) {
    __shared__ uint32_t s_lb[TILE_THREADS + TILE_SPAN + 1];
    const TileSpan lb = stage_span(q, s_lb);
    const uint32_t t = blockIdx.x * TILE_THREADS + threadIdx.x;
    if (t >= q.total_tiles) return;
    const TilePos p = tile_pos(q.scenes, q.tile_scene, t);
    const uint64_t at = pos[t];
    const bool on = (q.tile_flag[t] & FLAG_STATIC) != 0u;
    if (on) q.slist[uint32_t(at)] = t;
    // the last tile knows the static count, the last row's first tile the chunk count
    if (t + 1 == q.total_tiles) {
        const uint32_t tiles = uint32_t(at) + (on ? 1u : 0u);
        *q.scount = tiles;
        if (q.host_scount) *q.host_scount = tiles;
    }
    if (p.x == 0u) {
        const uint32_t end = emit_row(lb, t, p, rule, uint32_t(at >> 32), q.chunks);
        if (t + p.sc->W == q.total_tiles) *q.n_chunks = end;
    }
}

// Exclusive prefix sum of u64 values in place, SCAN_TILE per block.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const uint64_t* __restrict__ v, uint32_t n,
                                                              uint64_t* __restrict__ sums) {
    __shared__ uint64_t s_wave[64];
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t i = blockIdx.x * SCAN_TILE + k * SCAN_THREADS + threadIdx.x;
        if (i < n) s += v[i];
    }
    uint64_t tot = 0;
    block_excl_scan(s, s_wave, &tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ __launch_bounds__(1024) void k_scan_top(uint64_t* __restrict__ sums, uint32_t nb) {
    __shared__ uint64_t s_wave[64];
    uint64_t carry = 0;
    for (uint32_t off = 0; off < nb; off += 1024u) {
        const uint32_t i = off + threadIdx.x;
        uint64_t tot = 0;
        const uint64_t e = block_excl_scan(i < nb ? sums[i] : uint64_t(0), s_wave, &tot);
        if (i < nb) sums[i] = carry + e;
        carry += tot;
    }
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_down(uint64_t* __restrict__ v, uint32_t n,
                                                            const uint64_t* __restrict__ sums) {
    __shared__ uint64_t s_wave[64];
    uint64_t run = sums[blockIdx.x];
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        const uint32_t i = blockIdx.x * SCAN_TILE + k * SCAN_THREADS + threadIdx.x;
        uint64_t tot = 0;
        const uint64_t e = block_excl_scan(i < n ? v[i] : uint64_t(0), s_wave, &tot);
        if (i < n) v[i] = run + e;
        run += tot;
    }
}

size_t layout_scratch_words(uint32_t total_tiles) {
    return (size_t)total_tiles + (total_tiles + SCAN_TILE - 1) / SCAN_TILE;
}

bool layout_fits_one(uint32_t n, uint32_t total_tiles) { return n <= LAYOUT_ONE && total_tiles <= LAYOUT_TILES; }

static bool chunk_rule(uint32_t cap, uint32_t seg_tiles, ChunkRule& rule) {
    if (cap == 0 || cap > CHUNK_PARTICLES * MAX_PPT || (seg_tiles != 4 && seg_tiles != 6 && seg_tiles != 8))
        return false;
    rule = {cap, seg_tiles == 8 ? 0u : seg_tiles};
    return true;
}

hipError_t launch_layout_one(const StepArgs& a, uint32_t n_scenes, const LayoutArgs& q, uint32_t chunk_cap,
                             uint32_t seg_tiles, int bits, const uint32_t* ids, hipStream_t s) {
    ChunkRule rule;
    if (!chunk_rule(chunk_cap, seg_tiles, rule) || !layout_fits_one(q.n, q.total_tiles)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_layout_one, dim3(1), dim3(LAYOUT_THREADS), 0, s, a, n_scenes, q, rule, std::max(bits, 1),
                       ids);
    return hipGetLastError();
}

hipError_t launch_layout(const LayoutArgs& q, bool lb_done, uint32_t chunk_cap, uint32_t seg_tiles, uint64_t* scratch,
                         hipStream_t s) {
    ChunkRule rule;
    if (!chunk_rule(chunk_cap, seg_tiles, rule) || q.max_W > TILE_SPAN) return hipErrorInvalidValue;
    const uint32_t T = q.total_tiles;
    if (!lb_done)
        hipLaunchKernelGGL(k_tile_lb, dim3(std::min<unsigned>((T + 256) / 256, 16384u)), dim3(256), 0, s, q.keys, q.n,
                           q.tile_lb, T);
    if (T <= LAYOUT_TILES) {
        hipLaunchKernelGGL(k_layout_block, dim3(1), dim3(LAYOUT_THREADS), 0, s, q, rule);
        return hipGetLastError();
    }
    const unsigned tb = (T + TILE_THREADS - 1) / TILE_THREADS, nb = (T + SCAN_TILE - 1) / SCAN_TILE;
    uint64_t *pairs = scratch, *sums = scratch + T;
    hipLaunchKernelGGL(k_tile_marks, dim3(tb), dim3(TILE_THREADS), 0, s, q, rule, pairs);
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_THREADS), 0, s, pairs, T, sums);
    hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, sums, nb);
    hipLaunchKernelGGL(k_scan_down, dim3(nb), dim3(SCAN_THREADS), 0, s, pairs, T, sums);
    hipLaunchKernelGGL(k_tile_emit, dim3(tb), dim3(TILE_THREADS), 0, s, q, rule, pairs);
    return hipGetLastError();
}

__global__ void k_copy_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst) { *dst = *src; }

// One device word to another, on the stream (no host round trip).
hipError_t launch_copy_u32(const uint32_t* src, uint32_t* dst, hipStream_t s) {
    hipLaunchKernelGGL(k_copy_u32, dim3(1), dim3(1), 0, s, src, dst);
    return hipGetLastError();
}

}  // namespace mpm
