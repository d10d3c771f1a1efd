// radix_sort.hip - stable LSD key/value radix sort (reduce-then-scan).
//
// Replaces the CUB DeviceRadixSort::SortPairs call of RadixSort
// (NexusBVH/src/Cuda/Setup.cu:62-112). Semantics: stable sort of
// (key, value) pairs on key bits [begin_bit, end_bit); keys are carried whole.
//
// Design (gfx950, wave64):
//  * the digit counts of every pass are computed once (here, or fused into
//    the Morton kernel of the build pipeline) and give the global start of
//    each digit;
//  * each pass is three kernels with no waiting between blocks:
//      upsweep    per-tile digit counts into a digit-major table,
//      row scan   one block per digit: exclusive prefix over the tiles plus
//                 the digit's global start,
//      downsweep  loads a tile warp-striped (row k of wave w holds 64
//                 consecutive inputs), ranks it stably with per-row 64-lane
//                 ballot matching and per-wave LDS counters, scatters it into
//                 LDS in digit order and writes it out from LDS, so runs of
//                 one digit go to consecutive addresses;
//  * keys and values are read with the nontemporal hint (each pass streams
//    them once; measured 7% faster at 28.1M keys); stores stay normal, since
//    the scattered runs of a pass are combined in L2;
//  * small inputs are sorted in runs of 2,048 keys in LDS and the runs merged
//    by rank (k_sort_runs, k_sort_merge): one to three launches in all, where
//    the passes above take three each, 4 to 9 us a launch however few the keys;
//  * block b works on tile (b % 8) * per + b / 8: blocks are dispatched to
//    the 8 XCDs round-robin, so each XCD gets a contiguous range of tiles
//    and the table lines its blocks write and read stay in its own L2.
//    Correctness does not depend on the dispatch order.
#include "device_common.h"
#include "nxb_internal.h"

namespace nxb {

constexpr int kSortThreads = 256;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kMaxPasses = 11;        // 64 key bits in 6-bit digits
constexpr int kScanThreads = 1024;    // row-scan block

template <typename K>
__device__ __forceinline__ uint32_t digit_of(K key, uint32_t shift, uint32_t mask) {
    return (uint32_t)(key >> shift) & mask;
}

// Digit of one pass: `width` bits from bit `shift`, with 32-bit bit-field
// instructions. 64-bit keys get one kernel instantiation per key word (HI:
// shift >= 32); a digit that straddles the words comes from a funnel shift.
template <typename K, bool HI>
__device__ __forceinline__ uint32_t pass_digit(K key, uint32_t shift, uint32_t width) {
    if constexpr (sizeof(K) == 4) {
        return __builtin_amdgcn_ubfe((uint32_t)key, shift, width);
    } else if constexpr (HI) {
        return __builtin_amdgcn_ubfe((uint32_t)(key >> 32), shift - 32, width);
    } else {
        return __builtin_amdgcn_alignbit((uint32_t)(key >> 32), (uint32_t)key, shift) & ((1u << width) - 1u);
    }
}

// Lanes of the wave whose digit equals this lane's: the AND over the digit
// bits of ballot(bit) or its complement, one v_bitop3 per half and bit
// (truth table 0x90: a & ~(b ^ c)).
template <int BITS>
__device__ __forceinline__ uint64_t match_digit(uint32_t d) {
    uint32_t lo = ~0u, hi = ~0u;
#pragma unroll
    for (int b = 0; b < BITS; ++b) {
        uint32_t set = (uint32_t)((int32_t)(d << (31 - b)) >> 31);  // all ones when bit b is set
        uint64_t m = ballot(set != 0);
        lo = __builtin_amdgcn_bitop3_b32(lo, (uint32_t)m, set, 0x90);
        hi = __builtin_amdgcn_bitop3_b32(hi, (uint32_t)(m >> 32), set, 0x90);
    }
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint32_t xcd_tile(uint32_t block, uint32_t per) { return (block & 7u) * per + (block >> 3); }

// Exclusive scan of one value per thread over a block of NW waves.
template <int NW>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* tmp, uint32_t* total) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off);
        if (lane >= (uint32_t)off) x += y;
    }
    if (lane == 63) tmp[w] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int k = 0; k < NW; ++k) {
        uint32_t t = tmp[k];
        if ((uint32_t)k < w) before += t;
        all += t;
    }
    __syncthreads();
    if (total) *total = all;
    return before + x - v;
}

// Zeroes the used words of every histogram copy.
__global__ void k_sort_init(uint32_t* hist, uint32_t hist_words) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < kHistCopies * hist_words; i += gridDim.x * blockDim.x)
        hist[(i / hist_words) * kHistCopyWords + i % hist_words] = 0;
}

// Digit counts of every pass at once (block b adds into copy b % kHistCopies).
template <typename K, int BITS>
__global__ __launch_bounds__(kSortThreads) void k_sort_histogram(const K* __restrict__ keys, uint32_t n,
                                                                 uint32_t begin_bit, uint32_t end_bit,
                                                                 uint32_t passes, uint32_t* hist) {
    constexpr int RADIX = 1 << BITS;
    __shared__ uint32_t sh[kMaxPasses * RADIX];
    for (uint32_t i = threadIdx.x; i < passes * RADIX; i += kSortThreads) sh[i] = 0;
    __syncthreads();
    const uint32_t stride = gridDim.x * kSortThreads;
    for (uint32_t i = blockIdx.x * kSortThreads + threadIdx.x; i < n; i += stride) {
        K key = keys[i];
        for (uint32_t p = 0; p < passes; ++p) {
            uint32_t shift = begin_bit + p * BITS;
            uint32_t w = min((uint32_t)BITS, end_bit - shift);
            uint32_t d = digit_of(key, shift, (1u << w) - 1u);
            // one add for the wave when its lanes share the digit
            uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
            uint64_t active = ballot(true);
            if (ballot(d == d0) == active) {
                if (mask_rank(active) == 0) atomicAdd(&sh[p * RADIX + d0], (uint32_t)__popcll(active));
            } else {
                atomicAdd(&sh[p * RADIX + d], 1u);
            }
        }
    }
    __syncthreads();
    uint32_t* copy = hist + (blockIdx.x % kHistCopies) * kHistCopyWords;
    for (uint32_t i = threadIdx.x; i < passes * RADIX; i += kSortThreads) {
        uint32_t c = sh[i];
        if (c) atomic_add_agent(&copy[i], c);
    }
}

// Upsweep: counts[d * tiles + t] = number of keys of tile t with digit d.
// A block counts TPB consecutive tiles of TILE keys, all loads issued up
// front. Each wave has kUpRows counter rows (lane & 3 picks the row), so
// lanes sharing a digit meet on one LDS address at most 16 at a time; a row
// of 64 keys with one common digit is added once.
constexpr int kUpRows = 4;

template <typename K, int BITS, int TILE, int TPB, bool HI>
__global__ __launch_bounds__(kSortThreads) void k_sort_upsweep(const K* __restrict__ keys, uint32_t n,
                                                               uint32_t shift, uint32_t width, uint32_t tiles,
                                                               uint32_t per, uint32_t* __restrict__ counts) {
    constexpr int RADIX = 1 << BITS;
    constexpr int ITEMS = TILE / kSortThreads;
    static_assert(ITEMS * kSortThreads == TILE, "tile must be a multiple of the block");
    const uint32_t first = xcd_tile(blockIdx.x, per) * TPB;
    if (first >= tiles) return;
    __shared__ uint32_t wh[TPB][kSortWaves * kUpRows][RADIX];
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    for (uint32_t i = tid; i < (uint32_t)(TPB * kSortWaves * kUpRows * RADIX); i += kSortThreads)
        (&wh[0][0][0])[i] = 0;
    const uint32_t base = first * TILE;
    K key[TPB * ITEMS];
#pragma unroll
    for (int k = 0; k < TPB * ITEMS; ++k) {
        uint32_t idx = base + k * kSortThreads + tid;
        key[k] = idx < n ? __builtin_nontemporal_load(keys + idx) : (K)0;
    }
    __syncthreads();
    const uint32_t row = w * kUpRows + (lane & (kUpRows - 1));
#pragma unroll
    for (int k = 0; k < TPB * ITEMS; ++k) {
        const bool ok = base + k * kSortThreads + tid < n;
        const uint32_t d = pass_digit<K, HI>(key[k], shift, width);
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);  // lane 0: valid whenever any lane is
        const uint64_t act = ballot(ok);
        if (ballot(ok && d == d0) == act) {
            if (lane == 0 && act != 0) atomicAdd(&wh[k / ITEMS][w * kUpRows][d0], (uint32_t)__popcll(act));
        } else if (ok) {
            atomicAdd(&wh[k / ITEMS][row][d], 1u);
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TPB; ++t) {
        if (first + t < tiles) {
            for (uint32_t d = tid; d < (uint32_t)RADIX; d += kSortThreads) {
                uint32_t c = 0;
#pragma unroll
                for (int r = 0; r < kSortWaves * kUpRows; ++r) c += wh[t][r][d];
                counts[(size_t)d * tiles + first + t] = c;
            }
        }
    }
}

// Row scan: row d of the count table becomes the output position of the
// first key of digit d in each tile: the global start of digit d (counts of
// smaller digits, summed over the histogram copies) plus the counts of
// digit d in earlier tiles. The row is staged through LDS in chunks with
// coalesced loads and stores; each thread scans kRowPerThread entries.
constexpr uint32_t kRowPerThread = 8;
constexpr uint32_t kRowChunk = kScanThreads * kRowPerThread;

__global__ __launch_bounds__(kScanThreads) void k_sort_rowscan(uint32_t* counts, uint32_t tiles,
                                                               const uint32_t* __restrict__ hist) {
    constexpr int NW = kScanThreads / 64;
    __shared__ uint32_t tmp[NW];
    __shared__ uint32_t buf[kRowChunk];
    const uint32_t d = blockIdx.x, tid = threadIdx.x;
    uint32_t* row = counts + (size_t)d * tiles;
    // the first chunk of the row is loaded before the digit start is
    // summed, so that the two loads overlap
    uint32_t first[kRowPerThread];
#pragma unroll
    for (uint32_t k = 0; k < kRowPerThread; ++k) {
        uint32_t i = k * kScanThreads + tid;
        first[k] = i < min(kRowChunk, tiles) ? row[i] : 0u;
    }
    // thread t < d sums digit t over the histogram copies (all its loads
    // issued before the first add)
    static_assert(kScanThreads >= 512, "one thread per smaller digit");
    uint32_t s = 0;
    if (tid < d) {
        uint32_t h[kHistCopies];
#pragma unroll
        for (uint32_t c = 0; c < kHistCopies; ++c) h[c] = hist[c * kHistCopyWords + tid];
#pragma unroll
        for (uint32_t c = 0; c < kHistCopies; ++c) s += h[c];
    }
    uint32_t carry = 0;
    block_exclusive_scan<NW>(s, tmp, &carry);

    for (uint32_t c0 = 0; c0 < tiles; c0 += kRowChunk) {
        const uint32_t len = min(kRowChunk, tiles - c0);
#pragma unroll
        for (uint32_t k = 0; k < kRowPerThread; ++k) {
            uint32_t i = k * kScanThreads + tid;
            if (i < len) buf[i] = c0 == 0 ? first[k] : row[c0 + i];
        }
        __syncthreads();
        const uint32_t seg = tid * kRowPerThread;
        uint32_t v[kRowPerThread];
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t k = 0; k < kRowPerThread; ++k) {
            v[k] = seg + k < len ? buf[seg + k] : 0u;
            sum += v[k];
        }
        uint32_t total = 0;
        uint32_t run = carry + block_exclusive_scan<NW>(sum, tmp, &total);
#pragma unroll
        for (uint32_t k = 0; k < kRowPerThread; ++k) {
            if (seg + k < len) buf[seg + k] = run;
            run += v[k];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kRowPerThread; ++k) {
            uint32_t i = k * kScanThreads + tid;
            if (i < len) row[c0 + i] = buf[i];
        }
        carry += total;
        __syncthreads();
    }
}

// Loads rows k = 0..ITEMS-1 of a wave's part of a tile (row k: input
// first + 64k) with every load issued before the first one is used: indexes
// past n are clamped to n - 1, and fix_rows (called where the rows are first
// used) gives them the all-ones key. (A load inside a branch, or a value
// chosen between a load and the index, makes the compiler wait for each row
// before issuing the next.) Requires n >= 1.
template <typename K, int ITEMS>
__device__ __forceinline__ void load_rows(const K* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
                                          uint32_t n, uint32_t first, K* key, uint32_t* val) {
    if (vals_in) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t i = min(first + k * 64, n - 1);
            key[k] = __builtin_nontemporal_load(keys_in + i);
            val[k] = __builtin_nontemporal_load(vals_in + i);
        }
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            key[k] = __builtin_nontemporal_load(keys_in + min(first + k * 64, n - 1));
            val[k] = first + k * 64;
        }
    }
}

// Inputs past n get the all-ones key: its digit is the largest of the pass
// and they come last in input order, so they take the last LDS slots and are
// never written out.
template <typename K, int ITEMS>
__device__ __forceinline__ void fix_rows(uint32_t n, uint32_t first, K* key, uint32_t* val) {
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (first + k * 64 >= n) {
            key[k] = ~(K)0;
            val[k] = 0;
        }
    }
}

// Downsweep: stable scatter of one tile to the positions of the scanned table.
//
// A tile is THREADS * ITEMS keys. Per-wave digit counters are 16 bits, two
// waves to a 32-bit LDS word (counts and slots stay below 2^16). With
// TWO_PHASE the LDS staging buffer holds keys only: keys are scattered and
// written out first, then the values go through the same buffer, which
// halves the LDS of a tile for 8-byte keys. WPE is the occupancy the
// register allocation is held to (waves per SIMD).
template <typename K, int BITS, int ITEMS, bool HI, int THREADS, bool TWO_PHASE, int WPE>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(WPE))) void k_sort_downsweep(
    const K* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, K* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, uint32_t n, uint32_t shift, uint32_t width,
    const uint32_t* __restrict__ offsets, uint32_t tiles, uint32_t per) {
    constexpr int RADIX = 1 << BITS;
    constexpr int WAVES = THREADS / 64;
    constexpr int TILE = THREADS * ITEMS;
    constexpr int DPT = RADIX >= THREADS ? RADIX / THREADS : 1;  // digits per thread
    static_assert(WAVES % 2 == 0 && TILE < 65536, "packed 16-bit wave counters");
    const uint32_t tile = xcd_tile(blockIdx.x, per);
    if (tile >= tiles) return;
    __shared__ K skeys[TILE];
    __shared__ uint32_t svals[TWO_PHASE ? 1 : TILE];
    // rank counters, then the LDS slot of each wave's first key of a digit;
    // wave w uses bits 16*(w&1) of row w/2
    __shared__ uint32_t wave_off[WAVES / 2][RADIX];
    __shared__ uint32_t delta[RADIX];  // output position minus LDS slot, per digit
    __shared__ uint32_t scan_tmp[WAVES];

    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const uint32_t wrow = w >> 1, wsh = (w & 1) * 16;
    // thread t owns digits [t*DPT, t*DPT+DPT); their output positions first
    const bool owns = RADIX >= THREADS || tid < (uint32_t)RADIX;
    uint32_t gbase[DPT];
#pragma unroll
    for (int j = 0; j < DPT; ++j) gbase[j] = owns ? offsets[(size_t)(tid * DPT + j) * tiles + tile] : 0u;
    for (uint32_t i = tid; i < (uint32_t)(WAVES / 2 * RADIX); i += THREADS) (&wave_off[0][0])[i] = 0;

    // Row k of wave w holds the 64 consecutive inputs from
    // tile*TILE + (w*ITEMS + k)*64.
    const uint32_t base = tile * TILE;
    const uint32_t valid_count = min((uint32_t)TILE, n - base);
    K key[ITEMS];
    uint32_t val[ITEMS];
    load_rows<K, ITEMS>(keys_in, vals_in, n, base + w * ITEMS * 64 + lane, key, val);
    fix_rows<K, ITEMS>(n, base + w * ITEMS * 64 + lane, key, val);
    __syncthreads();

    // Stable rank within the wave (rows in order, lanes in order): lanes with
    // equal digits in a row are found by ballot matching; the lowest of them
    // adds the group's count to the wave's LDS counter (LDS atomics of one
    // wave are performed in issue order, so row k+1 sees row k) and its old
    // value is the group's base, fetched by the peers after the last row.
    uint32_t rl[ITEMS], lbase[ITEMS];  // rl = rank among peers | leader lane << 8
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        uint32_t d = pass_digit<K, HI>(key[k], shift, width);
        uint64_t peers = match_digit<BITS>(d);
        uint32_t rr = mask_rank(peers);
        rl[k] = rr | ((uint32_t)__builtin_ctzll(peers) << 8);
        // (a scalar first: a conditional store into the array itself makes the
        // compiler carry the whole array through the branch)
        uint32_t got = 0;
        if (rr == 0)
            got = __hip_atomic_fetch_add(&wave_off[wrow][d], (uint32_t)__popcll(peers) << wsh, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP) >> wsh;
        lbase[k] = got;
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) rl[k] = (rl[k] & 0xFFu) + (__shfl(lbase[k], (int)(rl[k] >> 8)) & 0xFFFFu);
    __syncthreads();

    // Per owned digit: the tile count (the waves' counts summed); after the
    // block scan, the LDS slot of each wave's first key (the counts are read
    // again from LDS rather than kept in registers across the scan, which
    // keeps the kernel within its 64 registers) and the output shift.
    uint32_t tsum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
#pragma unroll
        for (int ww = 0; ww < WAVES; ww += 2) {
            const uint32_t pair = owns ? wave_off[ww >> 1][tid * DPT + j] : 0u;
            tsum += (pair & 0xFFFFu) + (pair >> 16);
        }
    }
    uint32_t slot = block_exclusive_scan<WAVES>(tsum, scan_tmp, nullptr);
    if (owns) {
#pragma unroll
        for (int j = 0; j < DPT; ++j) {
            uint32_t d = tid * DPT + j;
            delta[d] = gbase[j] - slot;
#pragma unroll
            for (int ww = 0; ww < WAVES; ww += 2) {
                const uint32_t pair = wave_off[ww >> 1][d];
                uint32_t s0 = slot;
                slot += pair & 0xFFFFu;
                wave_off[ww >> 1][d] = s0 | (slot << 16);
                slot += pair >> 16;
            }
        }
    }
    __syncthreads();

    uint32_t pos[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        pos[k] = ((wave_off[wrow][pass_digit<K, HI>(key[k], shift, width)] >> wsh) & 0xFFFFu) + rl[k];
        skeys[pos[k]] = key[k];
        if constexpr (!TWO_PHASE) svals[pos[k]] = val[k];
    }
    __syncthreads();

    // Write out from LDS: runs of one digit go to consecutive addresses.
    if constexpr (!TWO_PHASE) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            uint32_t i = k * THREADS + tid;
            if (i < valid_count) {
                K kk = skeys[i];
                uint32_t o = delta[pass_digit<K, HI>(kk, shift, width)] + i;
                if (o < n) {  // always true when the table is consistent
                    keys_out[o] = kk;
                    vals_out[o] = svals[i];
                }
            }
        }
    } else {
        uint32_t out[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            uint32_t i = k * THREADS + tid;
            K kk = skeys[i];
            out[k] = i < valid_count ? delta[pass_digit<K, HI>(kk, shift, width)] + i : n;
            if (out[k] < n) keys_out[out[k]] = kk;  // out[k] < n always holds for i < valid_count
        }
        __syncthreads();
        uint32_t* sv = reinterpret_cast<uint32_t*>(skeys);
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) sv[pos[k]] = val[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            if (out[k] < n) vals_out[out[k]] = sv[k * THREADS + tid];
        }
    }
}

// ---- small inputs: runs sorted in LDS, then merged -------------------------
//
// Sorts every run of kRunKeys keys (block b: run b) on bits [begin_bit,
// end_bit): the keys stay in registers from pass to pass and go through LDS
// for the reordering. Ranking as in k_sort_downsweep (row k of wave w holds 64
// consecutive elements). Elements past n carry the all-ones key and stay last.
// Bound by the latency of a pass's five barriers (2.5 us a pass; 256 threads
// 26 us a run of 64-bit Morton keys, 512 and 1024 threads 21 us; runs of 4,096
// keys 31 us, of 8,192 keys 52 us).
constexpr int kRunThreads = 512;
constexpr uint32_t kRunKeys = 2048;
constexpr int kRunItems = kRunKeys / kRunThreads;

template <typename K>
__global__ __launch_bounds__(kRunThreads) void k_sort_runs(const K* __restrict__ keys_in,
                                                           const uint32_t* __restrict__ vals_in,
                                                           K* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
                                                           uint32_t n, uint32_t begin_bit, uint32_t end_bit) {
    constexpr int BITS = 8, RADIX = 1 << BITS, WAVES = kRunThreads / 64, ITEMS = kRunItems;
    __shared__ K skeys[kRunKeys];
    __shared__ uint32_t svals[kRunKeys];
    __shared__ uint32_t wave_off[WAVES / 2][RADIX];  // as in k_sort_downsweep
    __shared__ uint32_t scan_tmp[WAVES];
    const uint32_t tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const uint32_t wrow = w >> 1, wsh = (w & 1) * 16;
    const uint32_t local = w * ITEMS * 64 + lane, first = blockIdx.x * kRunKeys + local;
    K key[ITEMS];
    uint32_t val[ITEMS];
    load_rows<K, ITEMS>(keys_in, vals_in, n, first, key, val);
    fix_rows<K, ITEMS>(n, first, key, val);
    for (uint32_t shift = begin_bit; shift < end_bit; shift += BITS) {
        const uint32_t width = min((uint32_t)BITS, end_bit - shift);
        auto digit = [&](K k) {
            if constexpr (sizeof(K) == 8)
                return shift >= 32 ? pass_digit<K, true>(k, shift, width) : pass_digit<K, false>(k, shift, width);
            else
                return pass_digit<K, false>(k, shift, width);
        };
        for (uint32_t i = tid; i < (uint32_t)(WAVES / 2 * RADIX); i += kRunThreads) (&wave_off[0][0])[i] = 0;
        __syncthreads();
        uint32_t rl[ITEMS], lbase[ITEMS];  // rl = rank among peers | leader lane << 8
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t d = digit(key[k]);
            const uint64_t peers = match_digit<BITS>(d);
            const uint32_t rr = mask_rank(peers);
            rl[k] = rr | ((uint32_t)__builtin_ctzll(peers) << 8);
            uint32_t got = 0;
            if (rr == 0)
                got = __hip_atomic_fetch_add(&wave_off[wrow][d], (uint32_t)__popcll(peers) << wsh, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP) >> wsh;
            lbase[k] = got;
        }
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) rl[k] = (rl[k] & 0xFFu) + (__shfl(lbase[k], (int)(rl[k] >> 8)) & 0xFFFFu);
        __syncthreads();
        // thread d: the slot of each wave's first key of digit d
        uint32_t tsum = 0;
        if (tid < (uint32_t)RADIX) {
#pragma unroll
            for (int ww = 0; ww < WAVES / 2; ++ww) {
                const uint32_t pair = wave_off[ww][tid];
                tsum += (pair & 0xFFFFu) + (pair >> 16);
            }
        }
        uint32_t slot = block_exclusive_scan<WAVES>(tsum, scan_tmp, nullptr);
        if (tid < (uint32_t)RADIX) {
#pragma unroll
            for (int ww = 0; ww < WAVES / 2; ++ww) {
                const uint32_t pair = wave_off[ww][tid];
                const uint32_t s0 = slot;
                slot += pair & 0xFFFFu;
                wave_off[ww][tid] = s0 | (slot << 16);
                slot += pair >> 16;
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t pos = ((wave_off[wrow][digit(key[k])] >> wsh) & 0xFFFFu) + rl[k];
            skeys[pos] = key[k];
            svals[pos] = val[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            key[k] = skeys[local + k * 64];
            val[k] = svals[local + k * 64];
        }
    }
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (first + k * 64 < n) {
            keys_out[first + k * 64] = key[k];
            vals_out[first + k * 64] = val[k];
        }
    }
}

// Merges every group of up to kMergeRuns sorted runs of `run` keys (a multiple
// of kMergeThreads * kMergeSamples) into one, by rank: an element's place is
// its index in its own run plus, for every other run of the group, the number
// of elements before it there (equal ones count as before in earlier runs, as
// after in later ones, so the merge is stable). Each run is searched first
// among kMergeSamples samples in LDS, then among the run / kMergeSamples
// elements between two samples, kMergeUnroll runs at a time so that their
// loads overlap. mask: the key bits compared. Bound by latency up to ~100K keys
// (~6 us a level), then by the searches' instructions (15 runs of 12 to 16
// steps for every key: 35 us a level at 300K keys).
constexpr int kMergeThreads = 256;
constexpr uint32_t kMergeRuns = 16, kMergeSamples = 128, kMergeUnroll = 4;
static_assert(kMergeRuns % kMergeUnroll == 0 && kRunKeys % kMergeThreads == 0 && kRunKeys % kMergeSamples == 0, "runs");

template <typename K>
__global__ __launch_bounds__(kMergeThreads) void k_sort_merge(const K* __restrict__ keys,
                                                              const uint32_t* __restrict__ vals,
                                                              K* __restrict__ keys_out,
                                                              uint32_t* __restrict__ vals_out, uint32_t n,
                                                              uint32_t run, K mask) {
    __shared__ K sample[kMergeRuns][kMergeSamples];
    const uint32_t tid = threadIdx.x, i0 = blockIdx.x * kMergeThreads, i = i0 + tid;
    const uint32_t g0 = i0 - i0 % (run * kMergeRuns);        // the group's first element
    const uint32_t own = (i0 - g0) / run;                    // the block's run in the group
    const uint32_t runs = min(kMergeRuns, (n - g0 + run - 1) / run);
    const uint32_t gap = run / kMergeSamples;
    // sample k of a run: the last of its (k+1)-th `gap` elements; past n: larger than any masked key or equal to it
    for (uint32_t k = tid; k < runs * kMergeSamples; k += kMergeThreads) {
        const uint32_t at = g0 + (k + 1) * gap - 1;
        (&sample[0][0])[k] = at < n ? keys[at] & mask : ~(K)0;
    }
    const K key = keys[min(i, n - 1)];
    const uint32_t val = vals[min(i, n - 1)];
    const K x = key & mask;
    __syncthreads();
    uint32_t rank = g0 + (i - g0) % run;
    for (uint32_t r0 = 0; r0 < runs; r0 += kMergeUnroll) {
        uint32_t q[kMergeUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kMergeUnroll; ++u) q[u] = 0;
#pragma unroll
        for (uint32_t step = kMergeSamples / 2;; step >>= 1) {
            // the last round (step 0) tests the one sample left
#pragma unroll
            for (uint32_t u = 0; u < kMergeUnroll; ++u) {
                const K k = sample[min(r0 + u, runs - 1)][q[u] + (step ? step - 1 : 0)];
                const bool before = r0 + u < own ? !(x < k) : k < x;
                q[u] += before ? max(step, 1u) : 0u;
            }
            if (step == 0) break;
        }
        uint32_t base[kMergeUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kMergeUnroll; ++u) {
            base[u] = g0 + (r0 + u) * run;
            q[u] *= gap;
        }
        for (uint32_t step = gap / 2; step; step >>= 1) {
            K k[kMergeUnroll];
#pragma unroll
            for (uint32_t u = 0; u < kMergeUnroll; ++u) k[u] = keys[min(base[u] + q[u] + step - 1, n - 1)];
#pragma unroll
            for (uint32_t u = 0; u < kMergeUnroll; ++u) {
                const uint32_t at = q[u] + step - 1;
                const K m = k[u] & mask;
                const bool before = (r0 + u < own ? !(x < m) : m < x) && at < run && base[u] + at < n;
                q[u] += before ? step : 0u;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < kMergeUnroll; ++u)
            if (r0 + u < runs && r0 + u != own) rank += q[u];
    }
    if (i < n && rank < n) {  // rank < n always holds
        keys_out[rank] = key;
        vals_out[rank] = val;
    }
}

template <typename K>
__global__ void k_copy_pairs(const K* __restrict__ ki, const uint32_t* __restrict__ vi, K* __restrict__ ko,
                             uint32_t* __restrict__ vo, uint32_t n) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        ko[i] = ki[i];
        vo[i] = vi ? vi[i] : i;
    }
}

namespace {

// Tile shapes. Small: 256 threads, one LDS phase (keys and values staged
// together; 3-4 blocks per CU), for inputs that give fewer tiles than the
// chip holds of the wide shape. Wide: 1024 threads of 7 items, two LDS
// phases (74 KB of LDS), registers held to 64 so that two blocks share a
// CU; runs of one digit written out are longer than with the small 8-byte-key
// tile (7168 keys over 512 digits: 14 on average; 6 items per thread were
// 1% slower at 28.1M keys).
template <int KB, int BITS, bool WIDE>
struct TileShape {
    static constexpr int threads = WIDE ? 1024 : kSortThreads;
    static constexpr int items = WIDE ? 7 : (KB == 4 ? 16 : (BITS >= 9 ? 16 : 12));
    static constexpr bool two_phase = WIDE;
    static constexpr int wpe = WIDE ? 8 : 1;
    static constexpr int tile = threads * items;
    static constexpr int up_tiles = WIDE ? 1 : 2;  // tiles per upsweep block
};

constexpr uint32_t kWideMinKeys = 1u << 23;
// Keys up to which runs are sorted and merged, by the passes that the LSD sort
// would take (measured on Morton keys, us, merged / LSD):
//   8 passes (64-bit keys): 21 / 123 at 2,003, 33 / 141 at 16,411, 50 / 146 at
//     100K, 90 / 153 at 300K, 130 / 158 at 2^19, the most that two levels hold;
//   4 passes (32-bit keys): 11 / 64, 22 / 73, 36 / 75, 67 / 76, 104 / 77, equal
//     between 300K and 400K.
// Fewer passes: only up to one level, a launch or two against three per pass.
constexpr uint32_t merge_sort_max(uint32_t passes) {
    return passes >= 8 ? 1u << 19 : passes >= 4 ? 5u << 16 : kRunKeys * kMergeRuns;
}
static_assert(merge_sort_max(8) <= kRunKeys * kMergeRuns * kMergeRuns, "two levels of merging");

constexpr uint32_t tile_keys(uint32_t key_bytes, uint32_t bits, bool wide) {
    return wide ? (key_bytes == 8 ? TileShape<8, 8, true>::tile : TileShape<4, 8, true>::tile)
                : (key_bytes == 4 ? TileShape<4, 8, false>::tile
                                  : (bits >= 9 ? TileShape<8, 9, false>::tile : TileShape<8, 8, false>::tile));
}

template <typename K, int BITS, bool HI, bool WIDE>
void launch_pass(const K* src_k, const uint32_t* src_v, K* dk, uint32_t* dv, uint32_t n, uint32_t shift,
                 uint32_t width, const SortPlan& pl, SortScratch sc, uint32_t p, hipStream_t s) {
    using T = TileShape<(int)sizeof(K), BITS, WIDE>;
    constexpr int RADIX = 1 << BITS;
    const uint32_t per = (pl.tiles + 7) / 8;
    const uint32_t up_per = ((pl.tiles + T::up_tiles - 1) / T::up_tiles + 7) / 8;
    hipLaunchKernelGGL((k_sort_upsweep<K, BITS, T::tile, T::up_tiles, HI>), dim3(8 * up_per), dim3(kSortThreads), 0,
                       s, src_k, n, shift, width, pl.tiles, up_per, sc.counts);
    hipLaunchKernelGGL(k_sort_rowscan, dim3(RADIX), dim3(kScanThreads), 0, s, sc.counts, pl.tiles,
                       sc.hist + p * RADIX);
    hipLaunchKernelGGL((k_sort_downsweep<K, BITS, T::items, HI, T::threads, T::two_phase, T::wpe>), dim3(8 * per),
                       dim3(T::threads), 0, s, src_k, src_v, dk, dv, n, shift, width, sc.counts, pl.tiles, per);
}

template <typename K, int BITS, bool HI>
void launch_pass(const K* src_k, const uint32_t* src_v, K* dk, uint32_t* dv, uint32_t n, uint32_t shift,
                 uint32_t width, const SortPlan& pl, SortScratch sc, uint32_t p, hipStream_t s) {
    if (pl.wide) launch_pass<K, BITS, HI, true>(src_k, src_v, dk, dv, n, shift, width, pl, sc, p, s);
    else launch_pass<K, BITS, HI, false>(src_k, src_v, dk, dv, n, shift, width, pl, sc, p, s);
}

template <typename K, int BITS>
hipError_t run_passes(const K* keys_in, const uint32_t* values_in, K* keys_out, uint32_t* values_out, K* keys_tmp,
                      uint32_t* values_tmp, uint32_t n, const SortPlan& pl, SortScratch sc, hipStream_t s) {
    const K* src_k = keys_in;
    const uint32_t* src_v = values_in;
    for (uint32_t p = 0; p < pl.passes; ++p) {
        bool to_out = ((pl.passes - 1 - p) % 2) == 0;
        K* dk = to_out ? keys_out : keys_tmp;
        uint32_t* dv = to_out ? values_out : values_tmp;
        uint32_t shift = pl.begin + p * BITS;
        uint32_t width = min((uint32_t)BITS, pl.end - shift);
        if constexpr (sizeof(K) == 8) {
            if (shift >= 32) launch_pass<K, BITS, true>(src_k, src_v, dk, dv, n, shift, width, pl, sc, p, s);
            else launch_pass<K, BITS, false>(src_k, src_v, dk, dv, n, shift, width, pl, sc, p, s);
        } else {
            launch_pass<K, BITS, false>(src_k, src_v, dk, dv, n, shift, width, pl, sc, p, s);
        }
        src_k = dk;
        src_v = dv;
    }
    return hipGetLastError();
}

template <typename K, int BITS>
hipError_t run_histogram(const K* keys, uint32_t n, const SortPlan& pl, SortScratch sc, hipStream_t s) {
    uint32_t hgrid = min((n + kSortThreads * 16 - 1) / (kSortThreads * 16), 2048u);
    if (hgrid == 0) hgrid = 1;
    hipLaunchKernelGGL((k_sort_histogram<K, BITS>), dim3(hgrid), dim3(kSortThreads), 0, s, keys, n, pl.begin,
                       pl.end, pl.passes, sc.hist);
    return hipGetLastError();
}

// Levels of merging that n keys take: 0 (one run), 1 or 2.
template <typename K>
hipError_t run_merge_sort(const K* ki, const uint32_t* vi, K* ko, uint32_t* vo, K* kt, uint32_t* vt, uint32_t n,
                          const SortPlan& pl, hipStream_t s) {
    const uint32_t levels = n <= kRunKeys ? 0u : n <= kRunKeys * kMergeRuns ? 1u : 2u;
    const K mask = (K)(~(K)0 >> (8 * sizeof(K) - (pl.end - pl.begin))) << pl.begin;
    // the runs start where the last merge ends in the outputs
    K* dk = levels == 1 ? kt : ko;
    uint32_t* dv = levels == 1 ? vt : vo;
    hipLaunchKernelGGL(k_sort_runs<K>, dim3((n + kRunKeys - 1) / kRunKeys), dim3(kRunThreads), 0, s, ki, vi, dk, dv, n,
                       pl.begin, pl.end);
    uint32_t run = kRunKeys;
    for (uint32_t l = 0; l < levels; ++l, run *= kMergeRuns) {
        K* nk = dk == ko ? kt : ko;
        uint32_t* nv = dv == vo ? vt : vo;
        hipLaunchKernelGGL(k_sort_merge<K>, dim3((n + kMergeThreads - 1) / kMergeThreads), dim3(kMergeThreads), 0, s,
                           dk, dv, nk, nv, n, run, mask);
        dk = nk;
        dv = nv;
    }
    return hipGetLastError();
}

template <typename K>
hipError_t dispatch(bool hist_only, const void* ki, const uint32_t* vi, void* ko, uint32_t* vo, void* kt,
                    uint32_t* vt, uint32_t n, const SortPlan& pl, SortScratch sc, hipStream_t s) {
    const K* a = static_cast<const K*>(ki);
    K* o = static_cast<K*>(ko);
    K* t = static_cast<K*>(kt);
    switch (pl.bits) {
        case 6: return hist_only ? run_histogram<K, 6>(a, n, pl, sc, s) : run_passes<K, 6>(a, vi, o, vo, t, vt, n, pl, sc, s);
        case 7: return hist_only ? run_histogram<K, 7>(a, n, pl, sc, s) : run_passes<K, 7>(a, vi, o, vo, t, vt, n, pl, sc, s);
        case 8: return hist_only ? run_histogram<K, 8>(a, n, pl, sc, s) : run_passes<K, 8>(a, vi, o, vo, t, vt, n, pl, sc, s);
        case 9: return hist_only ? run_histogram<K, 9>(a, n, pl, sc, s) : run_passes<K, 9>(a, vi, o, vo, t, vt, n, pl, sc, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

SortPlan plan_sort(uint32_t n, uint32_t key_bits, uint32_t begin_bit, uint32_t end_bit, uint32_t digit_bits,
                   bool merge_ok) {
    SortPlan pl;
    pl.key_bits = key_bits;
    pl.begin = begin_bit;
    pl.end = end_bit;
    pl.bits = digit_bits;
    pl.passes = end_bit > begin_bit ? (end_bit - begin_bit + digit_bits - 1) / digit_bits : 0;
    pl.wide = n >= kWideMinKeys ? 1u : 0u;
    const uint32_t tile = tile_keys(key_bits / 8, digit_bits, pl.wide != 0);
    pl.tiles = (n + tile - 1) / tile;
    pl.merge = merge_ok && pl.passes && n <= merge_sort_max(pl.passes) ? 1u : 0u;
    return pl;
}

uint32_t default_digit_bits(uint32_t n, uint32_t key_bits) {
    if (key_bits == 32) return 7u;
    return n >= kWideMinKeys ? 9u : 8u;
}

size_t sort_scratch_bytes(uint32_t n, uint32_t key_bits, uint32_t digit_bits) {
    (void)key_bits;
    (void)digit_bits;
    // largest table: smallest tile with the widest radix (512)
    constexpr size_t min_tile = TileShape<8, 8, false>::tile;
    static_assert(min_tile <= TileShape<4, 8, false>::tile && min_tile <= TileShape<8, 9, false>::tile &&
                      min_tile <= TileShape<8, 8, true>::tile && min_tile <= TileShape<4, 8, true>::tile,
                  "count table sized by the smallest tile");
    size_t tiles = (n + min_tile - 1) / min_tile;
    if (tiles == 0) tiles = 1;
    return tiles * 512 * sizeof(uint32_t);
}

hipError_t launch_sort_prepare(const SortPlan& pl, SortScratch sc, hipStream_t s) {
    if (pl.passes > (uint32_t)kMaxPasses || (pl.passes << pl.bits) > kHistCopyWords) return hipErrorInvalidValue;
    if (pl.passes == 0 || pl.merge) return hipSuccess;
    hipLaunchKernelGGL(k_sort_init, dim3(kHistCopies), dim3(256), 0, s, sc.hist, pl.passes << pl.bits);
    return hipGetLastError();
}

hipError_t launch_sort_histogram(const void* keys, uint32_t n, const SortPlan& pl, SortScratch sc, hipStream_t s) {
    if (pl.passes == 0 || pl.merge || n <= 1) return hipSuccess;
    if (pl.key_bits == 32) return dispatch<uint32_t>(true, keys, nullptr, nullptr, nullptr, nullptr, nullptr, n, pl, sc, s);
    return dispatch<uint64_t>(true, keys, nullptr, nullptr, nullptr, nullptr, nullptr, n, pl, sc, s);
}

hipError_t launch_sort_passes(const void* keys_in, const uint32_t* values_in, void* keys_out, uint32_t* values_out,
                              void* keys_tmp, uint32_t* values_tmp, uint32_t n, const SortPlan& pl, SortScratch sc,
                              hipStream_t s) {
    if (pl.passes == 0 || n <= 1) {
        uint32_t blocks = (n + 255) / 256;
        uint32_t grid = blocks ? min(blocks, 4096u) : 1u;
        if (pl.key_bits == 32)
            hipLaunchKernelGGL(k_copy_pairs<uint32_t>, dim3(grid), dim3(256), 0, s,
                               static_cast<const uint32_t*>(keys_in), values_in, static_cast<uint32_t*>(keys_out),
                               values_out, n);
        else
            hipLaunchKernelGGL(k_copy_pairs<uint64_t>, dim3(grid), dim3(256), 0, s,
                               static_cast<const uint64_t*>(keys_in), values_in, static_cast<uint64_t*>(keys_out),
                               values_out, n);
        return hipGetLastError();
    }
    if (pl.merge) {
        if (pl.key_bits == 32)
            return run_merge_sort(static_cast<const uint32_t*>(keys_in), values_in, static_cast<uint32_t*>(keys_out),
                                  values_out, static_cast<uint32_t*>(keys_tmp), values_tmp, n, pl, s);
        return run_merge_sort(static_cast<const uint64_t*>(keys_in), values_in, static_cast<uint64_t*>(keys_out),
                              values_out, static_cast<uint64_t*>(keys_tmp), values_tmp, n, pl, s);
    }
    if (((size_t)pl.tiles << pl.bits) > sc.counts_words || pl.passes > (uint32_t)kMaxPasses ||
        (pl.passes << pl.bits) > kHistCopyWords)
        return hipErrorInvalidValue;
    if (pl.key_bits == 32)
        return dispatch<uint32_t>(false, keys_in, values_in, keys_out, values_out, keys_tmp, values_tmp, n, pl, sc, s);
    return dispatch<uint64_t>(false, keys_in, values_in, keys_out, values_out, keys_tmp, values_tmp, n, pl, sc, s);
}

hipError_t launch_radix_sort(const void* keys_in, const uint32_t* values_in, void* keys_out,
                             uint32_t* values_out, void* keys_tmp, uint32_t* values_tmp, uint32_t n,
                             uint32_t key_bits, uint32_t begin_bit, uint32_t end_bit, uint32_t digit_bits,
                             SortScratch sc, hipStream_t s) {
    if (end_bit < begin_bit || end_bit > key_bits || (key_bits != 32 && key_bits != 64)) return hipErrorInvalidValue;
    const bool any = digit_bits == 0;
    if (any) digit_bits = default_digit_bits(n, key_bits);
    if (digit_bits < 6 || digit_bits > 9) return hipErrorInvalidValue;
    SortPlan pl = plan_sort(n, key_bits, begin_bit, end_bit, digit_bits, any);
    hipError_t e = launch_sort_prepare(pl, sc, s);
    if (e != hipSuccess) return e;
    e = launch_sort_histogram(keys_in, n, pl, sc, s);
    if (e != hipSuccess) return e;
    return launch_sort_passes(keys_in, values_in, keys_out, values_out, keys_tmp, values_tmp, n, pl, sc, s);
}

}  // namespace nxb
