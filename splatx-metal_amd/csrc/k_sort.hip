// k_sort.hip — stable LSD radix sort of (key, i32 value) pairs for gfx950, keys u64 (the isect
// keys of sort_isect), u32 (depths) or u16 (tile ids).
//
// Contract: KernelBackend.h:130-148 / sort_isect (ascending unsigned key, stable, only bits
// [0, key_bits) significant). Design: digits of at most 8 bits (u64 keys 9), the key bits spread evenly over the
// fewest passes, so a 45-bit isect key needs 5 passes (the reference's 4-bit digits need 12) and a
// 13-bit tile id two (6 then 7 bits). A pass counts each tile's digits and places its keys with the counts of the
// tiles before it. Up to kRowKeys keys that is two launches (k_row_count, k_pass); above, and below 2^30 keys, the
// count matrix is scanned between them (k_rs_count, k_rs_reduce, k_rs_down, k_pass); no workgroup waits on
// another. The fallback at 2^30 keys and above is three launches per pass:
//   1. per-tile digit histogram (LDS counters)        -> hist[digit][tile], plus the digit totals
//   2. one workgroup per digit scans its row of hist   -> global start of (digit, tile)
//   3. stable scatter: each 64-lane wave ranks the keys of its quarter of the tile per digit with 8
//      ballots (lanes with an identical digit form one match mask) and per-wave LDS offsets, so
//      equal digits keep their relative order; the tile is reordered in LDS first so that the
//      global writes of each digit's run are contiguous.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "sx_kernels.h"
#include "sx_order.h"

namespace sxk {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kRounds = 16;
constexpr int kTile = kThreads * kRounds;  // 4096 keys per workgroup
constexpr int kBins = 256;
constexpr int kXcds = 8;  // XCDs of an MI355X (workgroups are dealt to them round-robin)

// Pass p of a sort on bits [0, key_bits) with digits of `dbits` bits covers bits [p dbits, p dbits +
// width), the last pass only what is left of key_bits (bits above key_bits never count).
__host__ __device__ inline uint32_t digit_mask(int p, int dbits, uint32_t key_bits) {
    const int width = min(dbits, static_cast<int>(key_bits) - p * dbits);
    return (1u << width) - 1u;
}

// Lanes of the wave whose 8-bit digit equals this lane's (among lanes where `valid`), from 8 ballots.
__device__ __forceinline__ uint64_t digit_match(uint32_t digit, bool valid) {
    uint64_t match = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const bool bit = (digit >> b) & 1u;
        const uint64_t bal = __ballot(bit);
        match &= bit ? bal : ~bal;
    }
    return match;
}

// Per-tile digit histogram -> hist[digit][tile]; the tile's counts are also added to the pass's
// digit totals (zeroed by k_zero_totals before the first pass). Equal digits of a wave are counted
// by one leader lane (match masks), so concentrated digits cost no LDS atomic contention.
template <class K>
__global__ void __launch_bounds__(kThreads) k_hist(const K* __restrict__ keys, int64_t n, int shift, uint32_t mask,
                                                   uint32_t* __restrict__ hist, int n_tiles,
                                                   uint32_t* __restrict__ totals) {
    __shared__ uint32_t h[kBins];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kTile;
    const int lane = threadIdx.x & 63;
    const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    K key[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const int64_t idx = base + r * kThreads + threadIdx.x;
        key[r] = idx < n ? keys[idx] : K(0);
    }
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const bool valid = base + r * kThreads + threadIdx.x < n;
        const uint32_t d = static_cast<uint32_t>(key[r] >> shift) & mask;
        const uint64_t match = digit_match(d, valid);
        if (valid && (match & lanes_below) == 0) atomicAdd(&h[d], static_cast<uint32_t>(__popcll(match)));
    }
    __syncthreads();
    const uint32_t c = h[threadIdx.x];
    hist[(size_t)threadIdx.x * n_tiles + blockIdx.x] = c;
    if (c) atomicAdd(&totals[threadIdx.x], c);
}

__global__ void __launch_bounds__(kThreads) k_zero_totals(uint32_t* __restrict__ totals, int n,
                                                          uint32_t* __restrict__ err) {
    for (int i = threadIdx.x; i < n; i += kThreads) totals[i] = 0;
    if (err && threadIdx.x == 0) *err = 0u;
}

template <int W = kWaves>
__device__ inline uint32_t block_excl_scan_u32(uint32_t v, uint32_t* s_wave, uint32_t* total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
        if (w < wave) pre += s_wave[w];
        tot += s_wave[w];
    }
    __syncthreads();
    if (total) *total = tot;
    return pre + x - v;
}

// One workgroup per digit d: hist[d][t] <- (keys of digits < d) + (keys of digit d in tiles < t),
// the global output start of tile t's run of digit d.
__global__ void __launch_bounds__(kThreads) k_scan_digit(uint32_t* __restrict__ hist, int n_tiles,
                                                         const uint32_t* __restrict__ totals) {
    __shared__ uint32_t s_wave[kWaves];
    const int d = blockIdx.x, tid = threadIdx.x;
    uint32_t all = 0;
    const uint32_t before = block_excl_scan_u32(totals[tid], s_wave, &all);
    __shared__ uint32_t s_base;
    if (tid == d) s_base = before;
    __syncthreads();
    uint32_t carry = s_base;
    uint32_t* row = hist + (size_t)d * n_tiles;
    constexpr int kItems = 4;
    for (int c0 = 0; c0 < n_tiles; c0 += kThreads * kItems) {
        const int i0 = c0 + tid * kItems;
        uint32_t v[kItems], sum = 0;
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            v[j] = i0 + j < n_tiles ? row[i0 + j] : 0u;
            sum += v[j];
        }
        uint32_t chunk = 0;
        uint32_t run = block_excl_scan_u32(sum, s_wave, &chunk) + carry;
#pragma unroll
        for (int j = 0; j < kItems; j++) {
            if (i0 + j < n_tiles) row[i0 + j] = run;
            run += v[j];
        }
        carry += chunk;
    }
}

// Stable scatter of one tile of 4096 keys. Wave w owns the contiguous quarter [1024 w, 1024 w + 1024)
// of the tile and walks it in 16 rounds of 64 keys; ranks among equal digits come from 64-lane
// match masks (8 ballots), so within the tile the order is (wave, round, lane) = input order. The
// tile is reordered by digit in LDS and then written out run by run: consecutive threads store
// consecutive addresses of one digit's output range.
template <class K>
__global__ void __launch_bounds__(kThreads) k_scatter(const K* __restrict__ kin, const int32_t* __restrict__ vin,
                                                      K* __restrict__ kout, int32_t* __restrict__ vout,
                                                      int64_t n, int shift, uint32_t mask, const uint32_t* __restrict__ hist,
                                                      int n_tiles) {
    constexpr int kPerWave = kTile / kWaves;  // 1024
    __shared__ K s_k[kTile];
    __shared__ int32_t s_v[kTile];
    __shared__ uint32_t s_gstart[kBins];  // global start of this tile's run of each digit
    __shared__ uint32_t s_lstart[kBins];  // local (in-tile) start of each digit's run
    __shared__ uint32_t s_woff[kWaves][kBins];  // per wave: next local slot of each digit
    __shared__ uint32_t s_wave[kWaves];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t base = (int64_t)blockIdx.x * kTile;
    const int tile_n = static_cast<int>(min<int64_t>(kTile, n - base));
    s_gstart[tid] = hist[(size_t)tid * n_tiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kWaves; w++) s_woff[w][tid] = 0;
    __syncthreads();
    K key[kRounds];
    int32_t val[kRounds];
    if (vin) {  // uniform; null values: the input index
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            const int i = wave * kPerWave + r * 64 + lane;
            key[r] = i < tile_n ? kin[base + i] : K(0);
            val[r] = i < tile_n ? vin[base + i] : 0;
        }
    } else {
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            const int i = wave * kPerWave + r * 64 + lane;
            key[r] = i < tile_n ? kin[base + i] : K(0);
            val[r] = i < tile_n ? static_cast<int32_t>(base + i) : 0;
        }
    }
    // per-wave digit histograms: one leader lane per distinct digit of a round; the ranks among
    // equal digits (and the leaders' counts) are kept for the placement below
    const uint64_t lanes_below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    uint8_t rank[kRounds];
    uint8_t cnt[kRounds];  // 0 unless this lane leads its digit group (then popcount - 1, fits 0..63)
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const bool valid = wave * kPerWave + r * 64 + lane < tile_n;
        const uint32_t d = static_cast<uint32_t>(key[r] >> shift) & mask;
        const uint64_t match = digit_match(d, valid);
        rank[r] = static_cast<uint8_t>(__popcll(match & lanes_below));
        cnt[r] = 0;
        if (valid && rank[r] == 0) {
            const uint32_t c = static_cast<uint32_t>(__popcll(match));
            cnt[r] = static_cast<uint8_t>(c - 1);
            s_woff[wave][d] += c;  // only this wave writes its row, one leader per digit
        }
    }
    __syncthreads();
    {
        // thread = digit: the digit's in-tile start, then each wave's start inside the digit's run
        uint32_t c[kWaves], tot = 0;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            c[w] = s_woff[w][tid];
            tot += c[w];
        }
        uint32_t all = 0;
        uint32_t run = block_excl_scan_u32(tot, s_wave, &all);
        s_lstart[tid] = run;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            s_woff[w][tid] = run;
            run += c[w];
        }
    }
    __syncthreads();
    uint32_t* woff = s_woff[wave];
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        if (wave * kPerWave + r * 64 >= tile_n) break;  // uniform within the wave
        const bool valid = wave * kPerWave + r * 64 + lane < tile_n;
        const uint32_t digit = static_cast<uint32_t>(key[r] >> shift) & mask;
        if (valid) {
            const uint32_t pos = woff[digit] + rank[r];
            s_k[pos] = key[r];
            s_v[pos] = val[r];
        }
        __builtin_amdgcn_wave_barrier();  // every lane has read woff[] before it is advanced
        if (valid && rank[r] == 0) woff[digit] += static_cast<uint32_t>(cnt[r]) + 1u;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    for (int p = tid; p < tile_n; p += kThreads) {
        const K k = s_k[p];
        const uint32_t d = static_cast<uint32_t>(k >> shift) & mask;
        const uint32_t g = s_gstart[d] + (static_cast<uint32_t>(p) - s_lstart[d]);
        kout[g] = k;
        vout[g] = s_v[p];
    }
}

// Lanes of the wave (among `valid_mask`) whose digit, the low NB bits of x, equals this lane's: one
// ballot per bit, each lane collecting the lanes that differ from it in that bit. Per bit: v_bfe_i32
// (the bit as 0 or ~0; written as asm, as the compiler otherwise makes a shift pair of it), the ballot's
// compare, and mis |= ballot ^ bit as one v_bitop3 per half (truth table 0xF6: src0 | (src1 ^ src2)).
template <int B, int NB>
__device__ __forceinline__ void digit_mismatch(uint32_t x, uint32_t& mis_lo, uint32_t& mis_hi) {
    if constexpr (B < NB) {
        uint32_t m;
        asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(x), "n"(B));
        const uint64_t bal = __ballot(m != 0u);
        mis_lo = __builtin_amdgcn_bitop3_b32(mis_lo, static_cast<uint32_t>(bal), m, 0xf6);
        mis_hi = __builtin_amdgcn_bitop3_b32(mis_hi, static_cast<uint32_t>(bal >> 32), m, 0xf6);
        digit_mismatch<B + 1, NB>(x, mis_lo, mis_hi);
    }
}
template <int NB>
__device__ __forceinline__ uint64_t digit_match_bits(uint32_t x, uint64_t valid_mask) {
    uint32_t mis_lo = 0u, mis_hi = 0u;
    digit_mismatch<0, NB>(x, mis_lo, mis_hi);
    return valid_mask & ~((static_cast<uint64_t>(mis_hi) << 32) | mis_lo);
}

// Set bits of `mask` in the lanes below this one.
__device__ __forceinline__ uint32_t lanes_below_count(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// ---- reduce-then-scan: the pass's prefixes without a chain between tiles ------------------------
// (One launch per pass whose tiles chain their prefixes by look-back is bound by that chain: config 5's sort
// took 1.69 ms so and 1.43 with a scan.) Each pass counts the digits of every tile (k_rs_count, digit-major: cnt[d][tile]), scans the
// whole count matrix once (the exclusive prefix of entry (d, tile) is where the tile's run of digit d
// starts in the output: all keys of smaller digits, then those of digit d in earlier tiles), and the
// pass kernel places its keys with these starts. Counts fit u32: a pass sorts fewer than 2^30 keys.
constexpr int kScanChunk = kThreads * 16;  // elements per workgroup of the count-matrix scan

// Digit counts of a tile -> cnt[d * n_tiles + tile] for d <= mask. Every workgroup of the grid
// writes its counts (zeros for a tile past the device count), so the scanned matrix is complete. A
// thread takes 16 consecutive keys (16-B loads) and adds each run of equal digits once: neighbouring
// keys often share the high digits (the tiles of one Gaussian along a row), and the lanes of a wave,
// 16 keys apart, rarely hit the same counter at once.
// err (optional): the sort's error word, zeroed by workgroup 0 (a sort that starts with this pass).
template <class K>
__global__ void __launch_bounds__(kThreads) k_rs_count(const K* __restrict__ keys, int64_t n, int shift, uint32_t mask,
                                                       uint32_t* __restrict__ cnt, int n_tiles,
                                                       const int64_t* __restrict__ n_dev, uint32_t* __restrict__ err) {
    static_assert(kRounds * sizeof(K) % 16 == 0, "a thread's keys are whole 16-B vectors");
    __shared__ uint32_t h[kBins];
    if (err && blockIdx.x == 0 && threadIdx.x == 0) *err = 0u;
    // tiles dealt XCD by XCD, as in k_pass (a grid of kXcds * ceil(n_tiles / kXcds)): a digit's counts
    // of consecutive tiles are neighbouring words of the matrix, and their partial lines then merge in
    // one L2
    const int per = (n_tiles + kXcds - 1) / kXcds;
    const int tile = static_cast<int>(blockIdx.x % kXcds) * per + static_cast<int>(blockIdx.x / kXcds);
    if (tile >= n_tiles) return;  // uniform
    if (n_dev) n = *n_dev;
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)tile * kTile + (int64_t)threadIdx.x * kRounds;
    K key[kRounds];
    if (i0 + kRounds <= n) {  // the library's own buffers: a tile (4096 keys) is 16-B aligned, and so is each thread's part
        constexpr int kVec = kRounds * sizeof(K) / 16;
        uint4 w[kVec];
#pragma unroll
        for (int q = 0; q < kVec; q++) w[q] = reinterpret_cast<const uint4*>(keys + i0)[q];
        __builtin_memcpy(key, w, sizeof(key));
    } else {
#pragma unroll
        for (int r = 0; r < kRounds; r++) key[r] = i0 + r < n ? keys[i0 + r] : K(0);
    }
    const int valid = static_cast<int>(min<int64_t>(kRounds, max<int64_t>(0, n - i0)));  // keys of the thread
    uint32_t run_d = static_cast<uint32_t>(key[0] >> shift) & mask, run_n = 0;
#pragma unroll
    for (int r = 0; r < kRounds; r++) {
        const uint32_t d = static_cast<uint32_t>(key[r] >> shift) & mask;
        if (r < valid) {
            if (d != run_d) {
                if (run_n) atomicAdd(&h[run_d], run_n);
                run_d = d;
                run_n = 0;
            }
            run_n++;
        }
    }
    if (run_n) atomicAdd(&h[run_d], run_n);
    __syncthreads();
    if (threadIdx.x <= mask) cnt[(size_t)threadIdx.x * n_tiles + tile] = h[threadIdx.x];
}

// Exclusive scan of v[0, len) in place, in two launches: chunk sums, then the scan of each chunk
// from its prefix, which each workgroup of the second adds up from the chunk sums before it (a few
// thousand words at most: cheaper than a launch that scans them first). v starts 64-B aligned (16-B
// loads).
__global__ void __launch_bounds__(kThreads) k_rs_reduce(const uint32_t* __restrict__ v, int64_t len,
                                                        uint32_t* __restrict__ sums) {
    __shared__ uint32_t s_wave[kWaves];
    const int64_t base = (int64_t)blockIdx.x * kScanChunk;
    uint32_t acc = 0;
    if (base + kScanChunk <= len) {  // four coalesced 16-B loads per thread
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 w = reinterpret_cast<const uint4*>(v + base)[q * kThreads + threadIdx.x];
            acc += w.x + w.y + w.z + w.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int64_t k = base + i * kThreads + threadIdx.x;
            acc += k < len ? v[k] : 0u;
        }
    }
    uint32_t all = 0;
    block_excl_scan_u32(acc, s_wave, &all);
    if (threadIdx.x == 0) sums[blockIdx.x] = all;
}

__global__ void __launch_bounds__(kThreads) k_rs_down(uint32_t* __restrict__ v, int64_t len,
                                                      const uint32_t* __restrict__ sums) {
    __shared__ uint32_t s_wave[kWaves];
    const int64_t i0 = (int64_t)blockIdx.x * kScanChunk + threadIdx.x * 16;  // 16 consecutive per thread
    uint32_t x[16], acc = 0;
    if (i0 + 16 <= len) {  // four 16-B loads
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 w = reinterpret_cast<const uint4*>(v + i0)[q];
            x[4 * q] = w.x;
            x[4 * q + 1] = w.y;
            x[4 * q + 2] = w.z;
            x[4 * q + 3] = w.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = i0 + i < len ? v[i0 + i] : 0u;
    }
#pragma unroll
    for (int i = 0; i < 16; i++) acc += x[i];
    uint32_t pre = 0;  // the chunks before this one
    for (int c = threadIdx.x; c < static_cast<int>(blockIdx.x); c += kThreads) pre += sums[c];
    uint32_t all = 0;
    (void)block_excl_scan_u32(pre, s_wave, &all);  // (its closing barrier frees s_wave)
    const uint32_t chunk_base = all;
    uint32_t run = block_excl_scan_u32(acc, s_wave, &all) + chunk_base;
    uint32_t y[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        y[i] = run;
        run += x[i];
    }
    if (i0 + 16 <= len) {
#pragma unroll
        for (int q = 0; q < 4; q++)
            reinterpret_cast<uint4*>(v + i0)[q] = make_uint4(y[4 * q], y[4 * q + 1], y[4 * q + 2], y[4 * q + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (i0 + i < len) v[i0 + i] = y[i];
    }
}

// ---- two launches per pass: the tiles' counts as rows, added up by the pass itself ---------------------
// Sorts of up to kRowKeys keys are bound by the latency of their launches (2 M u64 keys with a scan of the count
// matrix between count and pass: those two launches took 7 us of a pass's 28, 70 thousand keys 4.7 of 18.5).
// Here a tile's digit counts are one row (cnt[tile][T]), the rows of each kGroup tiles are also added up (gsum,
// integer atomics), and every workgroup of the pass reads the group rows and its own group's rows before it (at
// most 64 + 31 coalesced rows, in flight during the ranking): their sums are the digit's
// keys in earlier tiles, and a scan over the digits' totals is where each digit starts. Up to kDirectTiles tiles
// the tile rows alone. Workgroups of T threads sort digits of up to log2(T) bits: u64 keys take T = 512 (a 45-bit
// key in five passes instead of six), tile ids and depths 256.
constexpr int kGroup = 32;
constexpr int kDirectTiles = 64;

template <class K, int R, int T>
__global__ void __launch_bounds__(T) k_row_count(const K* __restrict__ keys, int64_t n, int shift, uint32_t mask,
                                                        uint32_t* __restrict__ cnt, uint32_t* __restrict__ gsum,
                                                        uint32_t* __restrict__ gsum_next, int n_groups, int n_tiles,
                                                        const int64_t* __restrict__ n_dev, uint32_t* __restrict__ err) {
    constexpr int kThreads = T, kBins = T;
    __shared__ uint32_t h[kBins];
    if (err && blockIdx.x == 0 && threadIdx.x == 0) *err = 0u;
    // the next pass's group sums (read by no workgroup of this launch) cleared, a slice per workgroup
    constexpr int kSlice = kBins / kGroup;
    if (gsum_next && threadIdx.x < kSlice)
        for (int k = static_cast<int>(blockIdx.x) * kSlice + threadIdx.x; k < n_groups * kBins; k += gridDim.x * kSlice)
            gsum_next[k] = 0u;
    // (tiles dealt XCD by XCD, as in the pass)
    const int per = (n_tiles + kXcds - 1) / kXcds;
    const int tile = static_cast<int>(blockIdx.x % kXcds) * per + static_cast<int>(blockIdx.x / kXcds);
    if (n_dev) n = *n_dev;
    if (tile >= n_tiles || (int64_t)tile * kThreads * R >= n) return;  // uniform; the pass reads no row past the keys
    h[threadIdx.x] = 0;
    __syncthreads();
    const int64_t i0 = (int64_t)tile * (kThreads * R) + (int64_t)threadIdx.x * R;
    K key[R];
    // whole vectors where the array starts at a multiple of a vector (a thread's keys then do too); a caller's own
    // device buffers (the allocation-free sort) need no more than a key's alignment
    using V = typename std::conditional<R * sizeof(K) % 16 == 0, uint4, uint2>::type;
    const bool aligned = (reinterpret_cast<uintptr_t>(keys) & (sizeof(V) - 1)) == 0;  // uniform
    if (aligned && i0 + R <= n) {
        constexpr int kVec = R * sizeof(K) / sizeof(V);
        static_assert(kVec * sizeof(V) == R * sizeof(K), "a thread's keys are whole vectors");
        V w[kVec];
#pragma unroll
        for (int q = 0; q < kVec; q++) w[q] = reinterpret_cast<const V*>(keys + i0)[q];
        __builtin_memcpy(key, w, sizeof(key));
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) key[r] = i0 + r < n ? keys[i0 + r] : K(0);
    }
    const int valid = static_cast<int>(min<int64_t>(R, max<int64_t>(0, n - i0)));
    uint32_t run_d = static_cast<uint32_t>(key[0] >> shift) & mask, run_n = 0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t d = static_cast<uint32_t>(key[r] >> shift) & mask;
        if (r < valid) {
            if (d != run_d) {
                if (run_n) atomicAdd(&h[run_d], run_n);
                run_d = d;
                run_n = 0;
            }
            run_n++;
        }
    }
    if (run_n) atomicAdd(&h[run_d], run_n);
    __syncthreads();
    if (threadIdx.x <= mask) {
        const uint32_t c = h[threadIdx.x];
        cnt[(size_t)tile * kBins + threadIdx.x] = c;
        if (gsum && c) atomicAdd(&gsum[(size_t)(tile / kGroup) * kBins + threadIdx.x], c);
    }
}

__global__ void __launch_bounds__(kThreads) k_zero_words(uint32_t* __restrict__ p, int n) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// The sums of rows [0, n) of digit tid (all) and of those below `below` (pre), eight rows in flight.
template <int T>
__device__ __forceinline__ void add_rows(const uint32_t* __restrict__ rows, int tid, int n, int below, uint32_t& pre,
                                         uint32_t& all) {
    for (int q = 0; q < n; q += 8) {  // uniform
        uint32_t v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = q + k < n ? rows[(size_t)(q + k) * T + tid] : 0u;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            all += v[k];
            pre += q + k < below ? v[k] : 0u;
        }
    }
}

// How a pass knows where a tile's run of each digit starts: kMatrix from the scanned count matrix of the
// reduce-then-scan path (starts[d * n_tiles + tile]), kRows from the tiles' rows of counts (starts = cnt, gsum).
enum { kMatrix = 0, kRows = 1 };
constexpr int kLeastBits = 4;  // narrower digits run with four ballots

// One pass: each tile's keys ranked by digit in LDS, reordered there and written out digit by digit.
// NB = the digit's width in bits (mask = 2^NB - 1; kRows: at most NB bits). R rounds of T keys per tile.
// X: each key also carries a u32 second value, read from xin at the key's input position and written to
// xout at its output position (null pointers when X is false). IDX: vin is null, and each key's value is
// its input position. kRows with digit_starts: the pass's first workgroup writes where each digit
// d < n_starts starts (for keys of one digit, the offset of each key value).
template <class K, int NB, int MODE, bool X, bool IDX, int R, int T>
__global__ void __launch_bounds__(T) k_pass(const K* __restrict__ kin, const int32_t* __restrict__ vin,
                                            K* __restrict__ kout, int32_t* __restrict__ vout, int64_t n, int shift,
                                            uint32_t mask, const int64_t* __restrict__ n_dev,
                                            const uint32_t* __restrict__ starts, int n_tiles,
                                            const uint32_t* __restrict__ xin, uint32_t* __restrict__ xout,
                                            const uint32_t* __restrict__ gsum, int32_t* __restrict__ digit_starts,
                                            int n_starts) {
    constexpr int kThreads = T, kBins = T, kWaves = T / 64, kRounds = R, kTile = T * R;  // this pass's tile
    constexpr int kPerWave = kTile / kWaves;
    __shared__ K s_k[kTile];
    // IDX (no input values: each key's value is its input position): no value registers, and the LDS
    // reorder moves the keys' 16-bit positions in the tile (83 VGPRs and 22 KB instead of 97 and 30 KB:
    // 5 waves per SIMD instead of 4)
    __shared__ typename std::conditional<IDX, uint16_t, int32_t>::type s_v[kTile];
    __shared__ uint32_t s_x[X ? kTile : 1];
    __shared__ uint32_t s_gstart[kBins];  // global start of this tile's run of each digit, minus its local start
    __shared__ uint32_t s_lstart[kBins];
    __shared__ uint32_t s_woff[kWaves][kBins];
    __shared__ uint32_t s_wave[kWaves];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    if (n_dev) n = *n_dev;  // (the grid is sized for a capacity)
    const int64_t n_work = (n + kTile - 1) / kTile;
    // XCD-aware tile order: the GPU deals workgroups to its kXcds XCDs round-robin (workgroup b to XCD
    // b % kXcds, each XCD taking its share in order), so tile (b % kXcds) * per + b / kXcds gives every XCD
    // a contiguous range of tiles. The runs of one digit that consecutive tiles write sit next to each
    // other in the output: written from the same L2, their partial lines merge before they leave it. The
    // grid has kXcds * ceil(tiles / kXcds) workgroups; the ones past the device count leave.
    // (Fewer workgroups per CU, or each looping over several tiles, measured slower.)
    const int64_t per = (n_work + kXcds - 1) / kXcds;
    {
        const int64_t k = blockIdx.x;
        const int64_t t = (k % kXcds) * per + k / kXcds;
        if (MODE == kRows && digit_starts && n_work == 0 && k == 0)
            for (int q = tid; q < n_starts; q += kThreads) digit_starts[q] = 0;
        if (k >= per * kXcds || t >= n_work) return;  // uniform
#pragma unroll
        for (int w = 0; w < kWaves; w++) s_woff[w][tid] = 0;
        __syncthreads();
        const uint32_t tile = static_cast<uint32_t>(t);
        // the tile's digit starts are requested now, so their latency overlaps the loads and the ranking
        uint32_t my_start = (MODE == kMatrix && tid <= mask) ? starts[(size_t)tid * n_tiles + tile] : 0u;
        const int64_t base = (int64_t)tile * kTile;
        const int tile_n = static_cast<int>(min<int64_t>(kTile, n - base));
        K key[kRounds];
        int32_t val[IDX ? 1 : kRounds];
        uint32_t xv[X ? kRounds : 1];
        if (X) {
#pragma unroll
            for (int r = 0; r < kRounds; r++) {
                const int i = wave * kPerWave + r * 64 + lane;
                xv[r] = i < tile_n ? xin[base + i] : 0u;
            }
        }
        // null values: the input index. The (uniform) choice is taken once around straight-line loads: a
        // choice per round compiles to a wait for every load before the next is issued.
        if (tile_n == kTile) {  // uniform
            if (vin) {
#pragma unroll
                for (int r = 0; r < kRounds; r++) {
                    const int i = wave * kPerWave + r * 64 + lane;
                    key[r] = kin[base + i];
                    val[r] = vin[base + i];
                }
            } else {
#pragma unroll
                for (int r = 0; r < kRounds; r++) {
                    const int i = wave * kPerWave + r * 64 + lane;
                    key[r] = kin[base + i];
                    if (!IDX) val[r] = static_cast<int32_t>(base + i);
                }
            }
        } else if (vin) {
#pragma unroll
            for (int r = 0; r < kRounds; r++) {
                const int i = wave * kPerWave + r * 64 + lane;
                key[r] = i < tile_n ? kin[base + i] : K(0);
                val[r] = i < tile_n ? vin[base + i] : 0;
            }
        } else {
#pragma unroll
            for (int r = 0; r < kRounds; r++) {
                const int i = wave * kPerWave + r * 64 + lane;
                key[r] = i < tile_n ? kin[base + i] : K(0);
                if (!IDX) val[r] = i < tile_n ? static_cast<int32_t>(base + i) : 0;
            }
        }
        uint32_t digit_total = 0u;  // kRows: the digit's keys in all tiles (my_start: in the tiles before this one)
        if (MODE == kRows && tid <= mask) {
            const int work = static_cast<int>(n_work), first = static_cast<int>(tile) / kGroup * kGroup;
            if (gsum) {
                add_rows<T>(gsum, tid, (work + kGroup - 1) / kGroup, first / kGroup, my_start, digit_total);
                uint32_t sub = 0u, all = 0u;
                add_rows<T>(starts + (size_t)first * kBins, tid, static_cast<int>(tile) - first, kGroup, sub, all);
                my_start += sub;
            } else {
                add_rows<T>(starts, tid, work, static_cast<int>(tile), my_start, digit_total);
            }
        }
        // per-wave digit counts, rounds in order; off[r] = the key's place among the wave's keys of its
        // digit (keys of earlier rounds, then lanes below it with the same digit). All lanes read the
        // digit's running count before one leader lane per digit group advances it.
        uint32_t off[kRounds];
        uint32_t* woff = s_woff[wave];
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            const bool valid = wave * kPerWave + r * 64 + lane < tile_n;
            uint32_t x = static_cast<uint32_t>(key[r] >> shift);
            if (MODE == kRows && NB == kLeastBits) x &= mask;  // (a digit of fewer bits than the ballots)
            const uint32_t d = x & mask;
            const uint64_t match = digit_match_bits<NB>(x, __ballot(valid));
            const uint32_t rank = lanes_below_count(match);
            const uint32_t prior = valid ? woff[d] : 0u;
            __builtin_amdgcn_wave_barrier();
            if (valid && rank == 0u) woff[d] = prior + static_cast<uint32_t>(__popcll(match));
            __builtin_amdgcn_wave_barrier();
            off[r] = prior + rank;
        }
        __syncthreads();
        {
            uint32_t c[kWaves], tot = 0;  // the tile's count of each digit
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                c[w] = s_woff[w][tid];
                tot += c[w];
            }
            uint32_t all = 0;
            if (MODE == kRows) {
                const uint32_t base_d = block_excl_scan_u32<kWaves>(digit_total, s_wave, &all);
                my_start += base_d;
                if (digit_starts && tile == 0u && tid < n_starts) digit_starts[tid] = static_cast<int32_t>(base_d);
            }
            uint32_t run = block_excl_scan_u32<kWaves>(tot, s_wave, &all);
            s_lstart[tid] = run;
#pragma unroll
            for (int w = 0; w < kWaves; w++) {
                s_woff[w][tid] = run;
                run += c[w];
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRounds; r++) {
            if (wave * kPerWave + r * 64 >= tile_n) break;  // uniform within the wave
            if (wave * kPerWave + r * 64 + lane < tile_n) {
                const uint32_t pos = woff[static_cast<uint32_t>(key[r] >> shift) & mask] + off[r];
                s_k[pos] = key[r];
                s_v[pos] = IDX ? static_cast<uint16_t>(wave * kPerWave + r * 64 + lane) : val[IDX ? 0 : r];
                if (X) s_x[pos] = xv[r];
            }
        }
        __syncthreads();
        if (tid <= static_cast<int>(mask)) s_gstart[tid] = my_start - s_lstart[tid];
        __syncthreads();
        const uint32_t n32 = static_cast<uint32_t>(n);  // (both modes sort fewer than 2^30 keys)
        for (int p = tid; p < tile_n; p += kThreads) {
            const K k = s_k[p];
            const uint32_t g = s_gstart[static_cast<uint32_t>(k >> shift) & mask] + static_cast<uint32_t>(p);
            if (g < n32) {  // always: no write lands out of range whatever the counts hold
                kout[g] = k;
                vout[g] = IDX ? static_cast<int32_t>(base + s_v[p]) : static_cast<int32_t>(s_v[p]);
                if (X) xout[g] = s_x[p];
            }
        }
    }
}

int tiles_for(int64_t n) { return static_cast<int>((n + kTile - 1) / kTile); }

// The tiles and groups of the two-launch passes over n keys (the capacity, with a device count), for n <= kRowKeys:
// tiles of 4 T keys up to kSmallKeys, which leave fewer compute units without one and rank four rounds one after
// another instead of eight, and of 8 T keys above. Measured: a step's tile sort with room for 0.9 M entries, 384 us a
// step in tiles of 4096, 376 of 1024; with room for 3 M, 47.5 us the sort in tiles of 4096, 44.6 of 2048 (52.6 with
// the scanned matrix); for 6 M, 85 us in rows of 4096-key tiles, 81 with the matrix, which the line at kRowKeys
// leaves it to. u64 keys: 1.5 M 115.7 us in tiles of 2048 keys, 2 M 149 and in tiles of 4096 121. groups 0: the tile
// rows alone.
constexpr int64_t kRowKeys = int64_t{1} << 22;
template <class K>
struct RowPlan {
    static constexpr int kT = sizeof(K) == 8 ? 512 : 256;
    static constexpr int kMaxBits = sizeof(K) == 8 ? 9 : 8;
    static constexpr int64_t kSmallKeys = sizeof(K) == 8 ? 3 << 19 : 1 << 20;
    int rounds, tiles, groups;
    bool fits;
    explicit RowPlan(int64_t n) {
        fits = n <= kRowKeys;
        rounds = n <= kSmallKeys ? 4 : 8;
        const int64_t t = (std::min(n, kRowKeys) + kT * rounds - 1) / (kT * rounds);
        tiles = static_cast<int>(std::max<int64_t>(t, 1));
        groups = tiles > kDirectTiles ? (tiles + kGroup - 1) / kGroup : 0;
    }
    size_t words() const { return static_cast<size_t>(tiles + 2 * groups) * kT; }
    static int passes(uint32_t key_bits) { return static_cast<int>((key_bits + kMaxBits - 1) / kMaxBits); }
};


// One pass over the digit of `mask`'s width at `shift`: the grid covers `tiles` tiles.
template <class K, int MODE, bool X, int R, int T>
void launch_pass(int tiles, hipStream_t s, const K* kin, const int32_t* vin, K* kout, int32_t* vout, int64_t n, int shift,
                 uint32_t mask, const int64_t* n_dev, const uint32_t* starts, const uint32_t* xin, uint32_t* xout,
                 const uint32_t* gsum = nullptr, int32_t* digit_starts = nullptr, int n_starts = 0) {
    const dim3 grid((tiles + kXcds - 1) / kXcds * kXcds);
    auto go = [&](auto nb) {
        constexpr int NB = decltype(nb)::value;
        if constexpr ((1 << NB) <= T && (MODE == kMatrix || NB >= kLeastBits)) {
            // (u64 keys come with their values; the first pass over positions has none)
            if (vin || sizeof(K) == 8)
                hipLaunchKernelGGL((k_pass<K, NB, MODE, X, false, R, T>), grid, dim3(T), 0, s, kin, vin, kout, vout, n, shift,
                                   mask, n_dev, starts, tiles, xin, xout, gsum, digit_starts, n_starts);
            else if constexpr (sizeof(K) < 8)
                hipLaunchKernelGGL((k_pass<K, NB, MODE, X, true, R, T>), grid, dim3(T), 0, s, kin, vin, kout, vout, n, shift,
                                   mask, n_dev, starts, tiles, xin, xout, gsum, digit_starts, n_starts);
        }
    };
    const int bits = __builtin_popcount(mask);
    switch (MODE == kRows ? std::max(kLeastBits, bits) : bits) {
        case 1: go(std::integral_constant<int, 1>{}); break;
        case 2: go(std::integral_constant<int, 2>{}); break;
        case 3: go(std::integral_constant<int, 3>{}); break;
        case 4: go(std::integral_constant<int, 4>{}); break;
        case 5: go(std::integral_constant<int, 5>{}); break;
        case 6: go(std::integral_constant<int, 6>{}); break;
        case 7: go(std::integral_constant<int, 7>{}); break;
        case 8: go(std::integral_constant<int, 8>{}); break;
        default: go(std::integral_constant<int, 9>{}); break;
    }
}

// x_dst[i] = x_src[pos[i]] (grid-stride)
__global__ void __launch_bounds__(kThreads) k_gather_x(const int32_t* __restrict__ pos, const uint32_t* __restrict__ x_src,
                                                       uint32_t* __restrict__ x_dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        x_dst[i] = x_src[pos[i]];
}
__global__ void __launch_bounds__(kThreads) k_copy_u32(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                       int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads)
        dst[i] = src[i];
}

constexpr int kMaxPasses = 8;
// scratch layout: a fixed header (digit totals of up to 8 passes, the error word) and then the tiles' counts: rows
// and their group sums, or a matrix of tiles x 256 words and its scan's chunk sums, or the three-launch path's
// histogram
constexpr int kErrWord = kMaxPasses * kBins;
constexpr int kHeaderWords = kMaxPasses * kBins + 64;
static_assert(kHeaderWords * sizeof(uint32_t) % 64 == 0, "the count matrix after the header is 64-B aligned");

// The number of passes of a sort of n keys on key_bits bits, of which the two-launch and the count-matrix path make
// digits of equal widths, give or take one.
template <class K>
int sort_passes(int64_t n, uint32_t key_bits) {
    return RowPlan<K>(n).fits ? RowPlan<K>::passes(key_bits) : static_cast<int>((key_bits + 7) / 8);
}

// The passes read `src` first and then alternate between the two sides: pass p writes side[p & 1],
// pass p > 0 reads side[(p - 1) & 1]. src may be side[1] (the sort then works in place over two
// buffers). n_dev: when set, the key count is read on the device from *n_dev (at most n, the capacity
// the grids are sized for), so the launches do not depend on it (a captured graph can replay them).
// Returns the number of passes, or -1 when nothing was launched because n_dev asks for the
// three-launch path. src_x (optional; then side_x too): a u32 second value per key that travels with it
// through the passes like the values (pass p writes side_x[p & 1]); the three-launch path, whose
// scatter does not carry it, gathers it once after the sort through the values, which must then be
// the input positions (src_v null).
template <class K>
int radix_sort_t(const K* src_k, const int32_t* src_v, K* const side_k[2], int32_t* const side_v[2], int64_t n,
                 uint32_t key_bits, void* scratch, bool clear_err, hipStream_t s, const int64_t* n_dev,
                 const uint32_t* src_x = nullptr, uint32_t* const* side_x = nullptr, SortExtra* ds = nullptr) {
    uint32_t* totals = static_cast<uint32_t*>(scratch);
    uint32_t* err = totals + kErrWord;
    key_bits = std::min<uint32_t>(key_bits, 8 * sizeof(K));
    // fewest passes, the bits spread evenly over them (longer runs per digit in each tile's writes than 8 + 5 for
    // a 13-bit tile id), narrower digits first: the first pass, over keys in the emit's order, has every digit in
    // each tile and so the shortest runs to write (config 5's 166 M tile ids: 1.026 -> 1.015 ms for the sort)
    const int passes = sort_passes<K>(n, key_bits);
    if (n <= 0 || passes == 0) {
        if (clear_err) hipLaunchKernelGGL(k_zero_totals, dim3(1), dim3(kThreads), 0, s, totals, 0, err);
        return 0;
    }
    if (n_dev && n >= (int64_t{1} << 30)) return -1;  // the three-launch path sizes its grids by the count
    const int narrow = static_cast<int>(key_bits) / passes, wide_from = passes - static_cast<int>(key_bits) % passes;
    auto shift_of = [&](int p) { return p * narrow + std::max(0, p - wide_from); };
    auto mask_of = [&](int p) { return (1u << (narrow + (p >= wide_from ? 1 : 0))) - 1u; };
    uint32_t* hist = totals + kHeaderWords;
    const K* kin = src_k;
    const int32_t* vin = src_v;
    auto x_in = [&](int p) { return !src_x ? nullptr : p == 0 ? src_x : const_cast<const uint32_t*>(side_x[(p - 1) & 1]); };
    if (const RowPlan<K> rows(n); rows.fits) {  // two launches per pass (see k_row_count)
        constexpr int T = RowPlan<K>::kT;
        uint32_t* const cnt = hist;
        // the passes' group sums in turn: a pass's count clears the next one's
        uint32_t* const gs[2] = {cnt + (size_t)rows.tiles * T, cnt + (size_t)(rows.tiles + rows.groups) * T};
        if (rows.groups && !(ds && ds->zeroed))
            hipLaunchKernelGGL(k_zero_words, dim3((rows.groups * T + kThreads - 1) / kThreads), dim3(kThreads), 0, s, gs[0],
                               rows.groups * T);
        if (ds) ds->written = passes == 1;
        auto pass = [&](auto r, auto x, int p) {
            constexpr int R = decltype(r)::value;
            constexpr bool X = decltype(x)::value;
            uint32_t* const g = rows.groups ? gs[p & 1] : nullptr;
            hipLaunchKernelGGL((k_row_count<K, R, T>), dim3((rows.tiles + kXcds - 1) / kXcds * kXcds), dim3(T), 0, s, kin, n,
                               shift_of(p), mask_of(p), cnt, g, g && p + 1 < passes ? gs[(p + 1) & 1] : nullptr,
                               rows.groups, rows.tiles, n_dev, (p == 0 && clear_err) ? err : nullptr);
            launch_pass<K, kRows, X, R, T>(rows.tiles, s, kin, vin, side_k[p & 1], side_v[p & 1], n, shift_of(p), mask_of(p),
                                           n_dev, cnt, x_in(p), X ? side_x[p & 1] : nullptr, g,
                                           ds && passes == 1 ? ds->starts : nullptr, ds ? ds->n : 0);
        };
        for (int p = 0; p < passes; p++) {
            auto with_rounds = [&](auto x) {
                if (rows.rounds == 4) pass(std::integral_constant<int, 4>{}, x, p);
                else pass(std::integral_constant<int, 8>{}, x, p);
            };
            if constexpr (sizeof(K) < 8) {
                if (src_x) with_rounds(std::true_type{});
                else with_rounds(std::false_type{});
            } else {
                with_rounds(std::false_type{});
            }
            kin = side_k[p & 1];
            vin = side_v[p & 1];
        }
        return passes;
    }
    const int tiles = tiles_for(n);
    if (n < (int64_t{1} << 30)) {  // reduce-then-scan (see k_rs_count)
        // (the digit totals are not used here; the first count kernel clears the error word)
        uint32_t* cnt = hist;                                  // (mask + 1) x tiles counts, then their starts
        uint32_t* sums = hist + (int64_t)tiles * kBins;        // the scan's chunk sums
        for (int p = 0; p < passes; p++) {
            const uint32_t mask = mask_of(p);
            const int64_t len = static_cast<int64_t>(mask + 1) * tiles;
            const int chunks = static_cast<int>((len + kScanChunk - 1) / kScanChunk);
            hipLaunchKernelGGL(k_rs_count<K>, dim3((tiles + kXcds - 1) / kXcds * kXcds), dim3(kThreads), 0, s, kin, n,
                               shift_of(p), mask, cnt, tiles, n_dev, (p == 0 && clear_err) ? err : nullptr);
            // (one workgroup scanning a small matrix in one launch measured slower than these)
            hipLaunchKernelGGL(k_rs_reduce, dim3(chunks), dim3(kThreads), 0, s, cnt, len, sums);
            hipLaunchKernelGGL(k_rs_down, dim3(chunks), dim3(kThreads), 0, s, cnt, len, sums);
            bool done = false;
            if constexpr (sizeof(K) < 8) {
                if (src_x) {
                    launch_pass<K, kMatrix, true, kRounds, kThreads>(tiles, s, kin, vin, side_k[p & 1], side_v[p & 1], n,
                                                                     shift_of(p), mask, n_dev, cnt, x_in(p), side_x[p & 1]);
                    done = true;
                }
            }
            if (!done)
                launch_pass<K, kMatrix, false, kRounds, kThreads>(tiles, s, kin, vin, side_k[p & 1], side_v[p & 1], n,
                                                                  shift_of(p), mask, n_dev, cnt, nullptr, nullptr);
            kin = side_k[p & 1];
            vin = side_v[p & 1];
        }
        return passes;
    }
    const int dbits = static_cast<int>((key_bits + passes - 1) / passes);
    hipLaunchKernelGGL(k_zero_totals, dim3(1), dim3(kThreads), 0, s, totals, passes * kBins,
                       clear_err ? err : nullptr);
    for (int p = 0; p < passes; p++) {
        const int shift = dbits * p;
        const uint32_t mask = digit_mask(p, dbits, key_bits);
        hipLaunchKernelGGL(k_hist<K>, dim3(tiles), dim3(kThreads), 0, s, kin, n, shift, mask, hist, tiles,
                           totals + p * kBins);
        hipLaunchKernelGGL(k_scan_digit, dim3(kBins), dim3(kThreads), 0, s, hist, tiles, totals + p * kBins);
        hipLaunchKernelGGL(k_scatter<K>, dim3(tiles), dim3(kThreads), 0, s, kin, vin, side_k[p & 1], side_v[p & 1],
                           n, shift, mask, hist, tiles);
        kin = side_k[p & 1];
        vin = side_v[p & 1];
    }
    if (src_x) {
        // the sorted values are the input positions: the second values follow them by a gather, into the
        // side the passes would have left them in (through side[0] when that is the input itself)
        const int blocks = static_cast<int>(std::min<int64_t>((n + kThreads - 1) / kThreads, int64_t{1} << 20));
        uint32_t* const dst = side_x[(passes - 1) & 1];
        if (dst != src_x) {
            hipLaunchKernelGGL(k_gather_x, dim3(blocks), dim3(kThreads), 0, s, vin, src_x, dst, n);
        } else {
            hipLaunchKernelGGL(k_gather_x, dim3(blocks), dim3(kThreads), 0, s, vin, src_x, side_x[0], n);
            hipLaunchKernelGGL(k_copy_u32, dim3(blocks), dim3(kThreads), 0, s, side_x[0], dst, n);
        }
    }
    return passes;
}

// In place over two buffers: a -> b -> a -> ...; the result is in a after an even pass count. With
// index_values the first pass takes each key's input position as its value (vals_a is not read).
template <class K>
int radix_sort_ab(K* keys_a, int32_t* vals_a, K* keys_b, int32_t* vals_b, int64_t n, uint32_t key_bits,
                  void* scratch, bool clear_err, hipStream_t s, const int64_t* n_dev, bool index_values = false,
                  uint32_t* x_a = nullptr, uint32_t* x_b = nullptr, SortExtra* ds = nullptr) {
    K* const sk[2] = {keys_b, keys_a};
    int32_t* const sv[2] = {vals_b, vals_a};
    uint32_t* const sx[2] = {x_b, x_a};
    const int passes = radix_sort_t<K>(keys_a, index_values ? nullptr : vals_a, sk, sv, n, key_bits, scratch,
                                       clear_err, s, n_dev, x_a, x_a ? sx : nullptr, ds);
    return passes < 0 ? -1 : (passes & 1);
}

// ---- the depth order within each tile (index-first intersections) --------------------------------
// When the Gaussians emit in index order, a stable sort on the tile ids leaves each tile's entries in
// index order; sorting them stably by the depth bits of their Gaussians (which the emit stored per
// entry) then gives the order of the reference's (tile | depth) keys: depth, ties by index. One
// workgroup per tile. A tile of at most 2048 entries is sorted in LDS by 8-bit LSD passes, wave w
// holding the w-th quarter of the list (in whole 64-key rounds) in registers and ranking with match
// masks as the sort's pass does; bytes on which every key of the tile agrees are skipped. A larger
// tile runs the same passes through global scratch, 2048 keys at a time in list order.
__device__ __forceinline__ uint32_t wave_and_u32(uint32_t x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x &= static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), o, 64));
    return x;
}
__device__ __forceinline__ uint32_t wave_or_u32(uint32_t x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(x), o, 64));
    return x;
}

// The bits in which the keys of the workgroup differ (AND and OR of each thread's `a` / `o`).
__device__ __forceinline__ uint32_t block_key_diff(uint32_t a, uint32_t o, uint32_t* s_and, uint32_t* s_or) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    a = wave_and_u32(a);
    o = wave_or_u32(o);
    if (lane == 0) {
        s_and[wave] = a;
        s_or[wave] = o;
    }
    __syncthreads();
    uint32_t A = ~0u, O = 0u;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        A &= s_and[w];
        O |= s_or[w];
    }
    return A ^ O;
}

// Ranks the wave's keys (rounds r < R, key index wave_base + 64 r + lane below `count`) by the byte at
// `shift`: off[r] = the key's place among the wave's keys of that digit (earlier rounds, then lower
// lanes); woff receives the wave's digit counts (zeroed by the caller).
template <int RMAX>
__device__ __forceinline__ void wave_rank_byte(const uint32_t* key, int R, int wave_base, int count, int shift,
                                               uint32_t* woff, uint32_t* off) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int r = 0; r < RMAX; r++) {
        if (r >= R) break;  // uniform
        const bool valid = wave_base + r * 64 + lane < count;
        const uint32_t x = key[r] >> shift;
        const uint32_t d = x & 255u;
        const uint64_t match = digit_match_bits<8>(x, __ballot(valid));
        const uint32_t rank = lanes_below_count(match);
        const uint32_t prior = valid ? woff[d] : 0u;
        __builtin_amdgcn_wave_barrier();
        if (valid && rank == 0u) woff[d] = prior + static_cast<uint32_t>(__popcll(match));
        __builtin_amdgcn_wave_barrier();
        off[r] = prior + rank;
    }
}

// thread = digit: the waves' counts of digit tid become their first output places, from `base` on;
// returns base + the digit's count
__device__ __forceinline__ uint32_t wave_starts(uint32_t (*s_woff)[kBins], uint32_t base) {
    const int tid = threadIdx.x;
    uint32_t run = base;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        const uint32_t c = s_woff[w][tid];
        s_woff[w][tid] = run;
        run += c;
    }
    return run;
}

// equal depths: runs up to this long are put in order in place, a tile with a longer one is sorted again
constexpr int kTieRun = 32;

// The run of keys equal to keys[i] that starts at i when one does (the key before differs, the next one
// equals it): its end, up to i + kTieRun + 1 (a longer run); i otherwise.
__device__ __forceinline__ int32_t tie_run_end(const uint32_t* keys, int32_t i, int32_t n) {
    const uint32_t k = keys[i];
    if ((i > 0 && keys[i - 1] == k) || i + 1 >= n || keys[i + 1] != k) return i;
    int32_t e = i + 2;
    while (e < n && e <= i + kTieRun && keys[e] == k) e++;
    return e;
}

// RMAX: rounds of 64 keys per wave that the kernel holds in registers. One launch takes every tile,
// heaviest first (tile_order): up to kCap = 256 RMAX entries in LDS, larger ones through global
// scratch. RMAX 8 (2048 entries, 12 KB of LDS) measured fastest: a separate launch for the tiles
// past 1024 entries with 16 rounds (twice the LDS) left its few long tiles running alone after
// the small ones, and 4 rounds send more tiles through global scratch. (One wave per small tile, with
// no workgroup barriers, measured slower: its ranking rounds wait on LDS one after another.)
// order_out (optional): workgroup 0 writes the rasterisers' tile order there instead (and the largest
// tile's count into *max_count), beside the sorting workgroups, which then take tile blockIdx.x - 1: the
// per-tile sorts gain nothing from running heaviest first, and the order costs no launch of its own.
// row_orig (optional, with id_of and splats): the lists are in an internal row order whose equal depths
// must go by original row (row_orig[id_of[value]]). After the depth sort, equal depths are runs of
// adjacent entries: a run of up to kTieRun entries is put in that order by the thread at its start (an
// insertion sort in LDS, or in global scratch for the large tiles); a tile with a longer run, or with
// one depth, is sorted again through global scratch, LSD by its original rows' varying bytes, then by
// its depth bytes (an entry's depth is word 3 of its Gaussian's splat record, splats[3 id_of[value]].w,
// the key the emit wrote). One compare per entry for tiles without equal depths. (The occupancy target
// of 7 waves per SIMD, which the LDS allows, keeps the register allocation of the tie work within it:
// without it 75 VGPRs, 6 waves.)
template <int RMAX>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(7)))
k_tile_depth_sort(const int32_t* __restrict__ offsets, int n_tiles, int32_t n_isects, const int64_t* __restrict__ n_dev,
                  const int32_t* __restrict__ tile_order, int32_t* __restrict__ vals,
                  const uint32_t* __restrict__ sdepth, uint32_t* __restrict__ sk0, uint32_t* __restrict__ sk1,
                  int32_t* __restrict__ sv, int32_t* __restrict__ order_out, uint32_t* __restrict__ max_count,
                  const int32_t* __restrict__ id_of, const int32_t* __restrict__ row_orig,
                  const float4* __restrict__ splats) {
    constexpr int kCap = kWaves * 64 * RMAX;
    __shared__ uint32_t s_key[kCap];
    __shared__ int32_t s_val[kCap];
    __shared__ uint32_t s_woff[kWaves][kBins];
    __shared__ uint32_t s_base[kBins];
    __shared__ uint32_t s_wave[kWaves];
    __shared__ uint32_t s_and[kWaves], s_or[kWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t n_all = n_dev ? static_cast<int32_t>(*n_dev) : n_isects;
    if (order_out && blockIdx.x == 0) {  // uniform
        static_assert(sizeof(OrderScratch) <= sizeof(s_woff), "the order's scratch fits in s_woff");
        tile_order_block<kThreads, 8>(offsets, n_tiles, n_all, order_out, max_count,
                                      reinterpret_cast<OrderScratch*>(&s_woff[0][0]));
        return;
    }
    const int bx = order_out ? static_cast<int>(blockIdx.x) - 1 : static_cast<int>(blockIdx.x);
    const int t = tile_order ? tile_order[bx] : bx;
    const int32_t start = offsets[t];
    const int32_t nt = (t + 1 < n_tiles ? offsets[t + 1] : n_all) - start;
    if (nt <= 1) return;  // uniform
    int32_t* const seg = vals + start;
    const bool by_orig = row_orig != nullptr;
    auto orig_of = [&](int32_t v) -> uint32_t { return static_cast<uint32_t>(row_orig[id_of[v]]); };
    auto depth_of = [&](int32_t v) -> uint32_t { return __float_as_uint(splats[3 * (size_t)id_of[v]].w); };
    // with row_orig, a tile with a run of equal depths longer than kTieRun (or with one depth) is sorted
    // again through global scratch (the large tiles' path): stage 1 by its original rows, stage 2 by its
    // depth bits
    int stage = 0;
    uint32_t key[RMAX];
    int32_t val[RMAX];
    uint32_t off[RMAX];
    if (nt <= kCap) {
        // wave w holds list entries [w Q, w Q + Q), Q a whole number of 64-entry rounds
        const int Q = ((nt + kWaves - 1) / kWaves + 63) & ~63;
        const int R = Q >> 6;
        const int wb = wave * Q;
#pragma unroll
        for (int r = 0; r < RMAX; r++) {
            const int i = wb + r * 64 + lane;
            val[r] = (r < R && i < nt) ? seg[i] : 0;
        }
        const uint32_t* const dk = sdepth + start;
        uint32_t a = ~0u, o = 0u;
#pragma unroll
        for (int r = 0; r < RMAX; r++) {
            const bool valid = r < R && wb + r * 64 + lane < nt;
            key[r] = valid ? dk[wb + r * 64 + lane] : 0u;
            if (valid) {
                a &= key[r];
                o |= key[r];
            }
        }
        const uint32_t diff = block_key_diff(a, o, s_and, s_or);
        if (diff == 0u && !by_orig) return;  // one depth: the index order stands
        if (diff == 0u) stage = 1;  // (one run: by original row alone)
        for (int p = 0; p < 4; p++) {
            const int shift = 8 * p;
            if (((diff >> shift) & 255u) == 0u) continue;  // uniform: every key has this byte
#pragma unroll
            for (int w = 0; w < kWaves; w++) s_woff[w][tid] = 0;
            __syncthreads();
            wave_rank_byte<RMAX>(key, R, wb, nt, shift, s_woff[wave], off);
            __syncthreads();
            {
                uint32_t tot = 0;
#pragma unroll
                for (int w = 0; w < kWaves; w++) tot += s_woff[w][tid];
                uint32_t all = 0;
                (void)wave_starts(s_woff, block_excl_scan_u32(tot, s_wave, &all));
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RMAX; r++) {
                if (r < R && wb + r * 64 + lane < nt) {
                    const uint32_t pos = s_woff[wave][(key[r] >> shift) & 255u] + off[r];
                    s_key[pos] = key[r];
                    s_val[pos] = val[r];
                }
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RMAX; r++) {
                const int i = wb + r * 64 + lane;
                if (r < R && i < nt) {
                    key[r] = s_key[i];
                    val[r] = s_val[i];
                }
            }
            __syncthreads();
        }
        if (by_orig && stage == 0) {
            // equal depths are adjacent now: each key against the one before it, from the lane below (DPP
            // wave shift) or, for lane 0, the wave's previous round
            int tie = 0;
            uint32_t carry = (wb > 0 && wb <= nt) ? s_key[wb - 1] : 0u;  // the key before the wave's first
#pragma unroll
            for (int r = 0; r < RMAX; r++) {
                if (r >= R) break;  // uniform
                const int i = wb + r * 64 + lane;
                const uint32_t prev = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
                    static_cast<int>(carry), static_cast<int>(key[r]), 0x138, 0xf, 0xf, false));  // wave_shr:1
                if (i < nt && i > 0) tie |= prev == key[r];
                carry = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key[r]), 63));
            }
            if (__syncthreads_or(tie)) {
                // the runs starting at this thread's entries (s_key holds the sorted keys): lengths, a byte
                // per round
                uint64_t runs = 0;
                int long_run = 0;
#pragma unroll
                for (int r = 0; r < RMAX; r++) {
                    const int i = wb + r * 64 + lane;
                    if (r < R && i < nt) {
                        const int32_t len = tie_run_end(s_key, i, nt) - i;
                        long_run |= len > kTieRun;
                        runs |= static_cast<uint64_t>(len > kTieRun ? 0 : len) << (8 * r);
                    }
                }
                if (__syncthreads_or(long_run)) {
                    stage = 1;  // (the whole tile again, from the values as loaded: any order will do)
                } else {
                    // the thread at a run's start replaces its keys (all equal) with the entries' original
                    // rows and sorts them with the values
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        const int i = wb + r * 64 + lane;
                        const int len = static_cast<int>((runs >> (8 * r)) & 255u);
                        if (len == 0) continue;
                        for (int m = i; m < i + len; m++) s_key[m] = orig_of(s_val[m]);
                        for (int m = i + 1; m < i + len; m++) {
                            const uint32_t km = s_key[m];
                            const int32_t vm = s_val[m];
                            int q = m;
                            for (; q > i && s_key[q - 1] > km; q--) {
                                s_key[q] = s_key[q - 1];
                                s_val[q] = s_val[q - 1];
                            }
                            s_key[q] = km;
                            s_val[q] = vm;
                        }
                    }
                    __syncthreads();
#pragma unroll
                    for (int r = 0; r < RMAX; r++) {
                        const int i = wb + r * 64 + lane;
                        if (r < R && i < nt) val[r] = s_val[i];
                    }
                }
            }
        }
        if (stage == 0) {
#pragma unroll
            for (int r = 0; r < RMAX; r++) {
                const int i = wb + r * 64 + lane;
                if (r < R && i < nt) seg[i] = val[r];
            }
            return;
        }
    }
    {
        // a tile of more than kCap entries (or one sorted again by original row): the keys go to sk0, then
        // each pass moves (key, value) between (sk0, vals) and (sk1, sv) over the tile's range, chunk by
        // chunk in list order
        uint32_t* src_k = sk0 + start;
        int32_t* src_v = seg;
        uint32_t* dst_k = sk1 + start;
        int32_t* dst_v = sv + start;
        uint32_t todo = 0u;
        if (stage == 0) {
            uint32_t a = ~0u, o = 0u;
            for (int32_t i = tid; i < nt; i += kThreads) {
                const uint32_t k = sdepth[start + i];
                sk0[start + i] = k;
                a &= k;
                o |= k;
            }
            todo = block_key_diff(a, o, s_and, s_or);  // (its barrier also orders the sk0 stores)
            if (todo == 0u && by_orig) stage = 1;
        }
        // (chunks of half the LDS path's rounds: this path's registers stay within the LDS path's)
        constexpr int kRG = RMAX / 2 > 0 ? RMAX / 2 : 1;
        constexpr int kChunk = kWaves * 64 * kRG;
        constexpr int kPerWave = kChunk / kWaves;
        for (;;) {
            if (stage > 0) {
                // the keys (scratch) replaced: 1 the entries' original rows, 2 their depth bits again
                uint32_t a = ~0u, o = 0u;
                for (int32_t i = tid; i < nt; i += kThreads) {
                    const uint32_t k = stage == 1 ? orig_of(src_v[i]) : depth_of(src_v[i]);
                    src_k[i] = k;
                    a &= k;
                    o |= k;
                }
                todo = block_key_diff(a, o, s_and, s_or);  // (orders the key stores)
            }
            for (int p = 0; p < 4; p++) {
                const int shift = 8 * p;
                if (((todo >> shift) & 255u) == 0u) continue;  // uniform
                s_base[tid] = 0;
                __syncthreads();
                for (int32_t i = tid; i < nt; i += kThreads) atomicAdd(&s_base[(src_k[i] >> shift) & 255u], 1u);
                __syncthreads();
                {
                    uint32_t all = 0;
                    const uint32_t b = block_excl_scan_u32(s_base[tid], s_wave, &all);
                    s_base[tid] = b;  // every thread has read its own digit's count above
                }
                __syncthreads();
                for (int32_t c0 = 0; c0 < nt; c0 += kChunk) {  // uniform
                    const int cn = static_cast<int>(min<int32_t>(kChunk, nt - c0));
                    const int wb = wave * kPerWave;
#pragma unroll
                    for (int r = 0; r < kRG; r++) {
                        const int i = wb + r * 64 + lane;
                        key[r] = i < cn ? src_k[c0 + i] : 0u;
                        val[r] = i < cn ? src_v[c0 + i] : 0;
                    }
#pragma unroll
                    for (int w = 0; w < kWaves; w++) s_woff[w][tid] = 0;
                    __syncthreads();
                    wave_rank_byte<kRG>(key, kRG, wb, cn, shift, s_woff[wave], off);
                    __syncthreads();
                    s_base[tid] = wave_starts(s_woff, s_base[tid]);
                    __syncthreads();
#pragma unroll
                    for (int r = 0; r < kRG; r++) {
                        if (wb + r * 64 + lane < cn) {
                            const uint32_t pos = s_woff[wave][(key[r] >> shift) & 255u] + off[r];
                            dst_k[pos] = key[r];
                            dst_v[pos] = val[r];
                        }
                    }
                    __syncthreads();  // s_woff is cleared for the next chunk; the next pass reads these stores
                }
                uint32_t* tk = src_k;
                src_k = dst_k;
                dst_k = tk;
                int32_t* tv = src_v;
                src_v = dst_v;
                dst_v = tv;
            }
            if (!by_orig || stage == 2) break;
            if (stage == 1) {
                stage = 2;
                continue;
            }
            // stage 0, as in LDS: runs of up to kTieRun fixed by the thread at their start (the original rows
            // in dst_k, the keys in src_k left for the other threads' run search), longer ones sorted again
            int tie = 0, long_run = 0;
            for (int32_t i = tid; i < nt; i += kThreads) {
                const int32_t len = tie_run_end(src_k, i, nt) - i;
                tie |= len > 0;
                long_run |= len > kTieRun;
            }
            if (__syncthreads_or(long_run)) {
                stage = 1;
                continue;
            }
            if (__syncthreads_or(tie)) {
                for (int32_t i = tid; i < nt; i += kThreads) {
                    const int32_t e = tie_run_end(src_k, i, nt);
                    for (int32_t m = i; m < e; m++) dst_k[m] = orig_of(src_v[m]);
                    for (int32_t m = i + 1; m < e; m++) {
                        const uint32_t km = dst_k[m];
                        const int32_t vm = src_v[m];
                        int32_t q = m;
                        for (; q > i && dst_k[q - 1] > km; q--) {
                            dst_k[q] = dst_k[q - 1];
                            src_v[q] = src_v[q - 1];
                        }
                        dst_k[q] = km;
                        src_v[q] = vm;
                    }
                }
                __syncthreads();  // the copy below reads other threads' runs
            }
            break;
        }
        if (src_v != seg)
            for (int32_t i = tid; i < nt; i += kThreads) seg[i] = src_v[i];
    }
}

} // namespace

SortZeroWords sort_zero_words_u16(void* scratch, int64_t n) {
    using Plan = RowPlan<uint16_t>;
    const Plan rows(n);
    if (!rows.fits || rows.groups == 0) return {nullptr, 0};
    return {static_cast<uint32_t*>(scratch) + kHeaderWords + (size_t)rows.tiles * Plan::kT, rows.groups * Plan::kT};
}

size_t sort_scratch_bytes(int64_t n) {
    const size_t tiles = static_cast<size_t>(std::max(1, tiles_for(n)));
    size_t words = 2 * tiles * kBins;
    // (for any key type; a smaller sort in the same scratch may take smaller tiles, so more rows)
    const int64_t m = std::min(n, kRowKeys);
    for (const int64_t k : {m, std::min(m, RowPlan<uint16_t>::kSmallKeys)}) words = std::max(words, RowPlan<uint16_t>(k).words());
    for (const int64_t k : {m, std::min(m, RowPlan<uint64_t>::kSmallKeys)}) words = std::max(words, RowPlan<uint64_t>(k).words());
    return sizeof(uint32_t) * (kHeaderWords + words);
}

uint32_t* sort_error_flag(void* scratch) { return static_cast<uint32_t*>(scratch) + kErrWord; }

int radix_sort(uint64_t* keys_a, int32_t* vals_a, uint64_t* keys_b, int32_t* vals_b, int64_t n, uint32_t key_bits,
               void* scratch, hipStream_t s, bool clear_err, const int64_t* n_dev) {
    return radix_sort_ab(keys_a, vals_a, keys_b, vals_b, n, key_bits, scratch, clear_err, s, n_dev);
}

int radix_sort(uint32_t* keys_a, int32_t* vals_a, uint32_t* keys_b, int32_t* vals_b, int64_t n, uint32_t key_bits,
               void* scratch, hipStream_t s, bool clear_err, const int64_t* n_dev) {
    return radix_sort_ab(keys_a, vals_a, keys_b, vals_b, n, key_bits, scratch, clear_err, s, n_dev);
}

int radix_sort(uint16_t* keys_a, int32_t* vals_a, uint16_t* keys_b, int32_t* vals_b, int64_t n, uint32_t key_bits,
               void* scratch, hipStream_t s, bool clear_err, const int64_t* n_dev) {
    return radix_sort_ab(keys_a, vals_a, keys_b, vals_b, n, key_bits, scratch, clear_err, s, n_dev);
}

int radix_sort_positions(uint16_t* keys_a, int32_t* vals_a, uint16_t* keys_b, int32_t* vals_b, int64_t n,
                         uint32_t key_bits, void* scratch, hipStream_t s, bool clear_err, const int64_t* n_dev,
                         uint32_t* x_a, uint32_t* x_b, SortExtra* ds) {
    return radix_sort_ab(keys_a, vals_a, keys_b, vals_b, n, key_bits, scratch, clear_err, s, n_dev, true, x_a, x_b, ds);
}

int radix_sort_positions(uint32_t* keys_a, int32_t* vals_a, uint32_t* keys_b, int32_t* vals_b, int64_t n,
                         uint32_t key_bits, void* scratch, hipStream_t s, bool clear_err, const int64_t* n_dev,
                         uint32_t* x_a, uint32_t* x_b, SortExtra* ds) {
    return radix_sort_ab(keys_a, vals_a, keys_b, vals_b, n, key_bits, scratch, clear_err, s, n_dev, true, x_a, x_b, ds);
}

constexpr int kDepthSortRounds = 8;

void tile_depth_sort(const int32_t* offsets, int n_tiles, int64_t n_isects, const int64_t* n_dev,
                     const int32_t* tile_order, int32_t* vals, const uint32_t* sdepth, uint32_t* scratch_k0,
                     uint32_t* scratch_k1, int32_t* scratch_v, hipStream_t s, int32_t* order_out,
                     uint32_t* max_count, const TieOrder* ties) {
    if (n_tiles <= 0 || (!order_out && !n_dev && n_isects <= 1)) return;
    if (ties && (!ties->id_of || !ties->row_orig || !ties->splats))
        throw std::invalid_argument("tile_depth_sort: incomplete tie order arguments");
    hipLaunchKernelGGL(k_tile_depth_sort<kDepthSortRounds>, dim3(n_tiles + (order_out ? 1 : 0)), dim3(kThreads), 0,
                       s, offsets, n_tiles, static_cast<int32_t>(n_isects), n_dev, tile_order, vals, sdepth,
                       scratch_k0, scratch_k1, scratch_v, order_out, max_count, ties ? ties->id_of : nullptr,
                       ties ? ties->row_orig : nullptr, ties ? ties->splats : nullptr);
}

void radix_sort_into(const uint64_t* keys, const int32_t* vals, uint64_t* keys_out, int32_t* vals_out,
                     uint64_t* keys_tmp, int32_t* vals_tmp, int64_t n, uint32_t key_bits, void* scratch,
                     hipStream_t s) {
    const int passes = sort_passes<uint64_t>(n, std::min<uint32_t>(key_bits, 64));
    // the last pass, passes - 1, writes side[(passes - 1) & 1]: make that side the output
    uint64_t* const sk[2] = {(passes & 1) ? keys_out : keys_tmp, (passes & 1) ? keys_tmp : keys_out};
    int32_t* const sv[2] = {(passes & 1) ? vals_out : vals_tmp, (passes & 1) ? vals_tmp : vals_out};
    (void)radix_sort_t<uint64_t>(keys, vals, sk, sv, n, key_bits, scratch, true, s, nullptr);
}

} // namespace sxk
