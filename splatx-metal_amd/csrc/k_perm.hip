// k_perm.hip — the arena's spatial row order (gfx950).
//
// The step reads and writes its parameter rows column by column (SoA), and the rows of one cache line
// are 32 consecutive rows. In the caller's order (the reference's) the rows a camera culls are spread
// over every line, so each step streams the whole arena. Kept in the order of a Morton curve over the
// means instead, the culled rows fill whole waves, which the update skips: the executor may hold the
// live rows [0, count) in that order, with the maps between its internal rows and the caller's
// (original) rows. Every result stays the caller's: depth first, the emit runs in original order (so
// the stable depth sort's ties go by original row); index first, it runs in internal order and the
// per-tile depth sort puts equal depths in original-row order; the MCMC noise is drawn by original row; a
// download puts each row in its original place as it packs it, and every other entry point that exchanges
// rows with the caller restores the original order first.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <stdexcept>
#include <type_traits>

#include "sx_step.h"

namespace sxk {
namespace {

constexpr int kBlock = 256;
inline int grid_for(int64_t n) { return static_cast<int>((n + kBlock - 1) / kBlock); }

// Per-block bounding boxes of the means of rows [0, count) (x, y, z columns at stride R): part[6 b ..
// 6 b + 6) = {min x, min y, min z, max x, max y, max z}; non-finite coordinates are left out.
__global__ void __launch_bounds__(kBlock) k_bbox_part(const float* __restrict__ m, size_t R, int count,
                                                      float* __restrict__ part) {
    __shared__ float s[6][kBlock / 64];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
    float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    if (i < count) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const float x = m[d * R + i];
            if (__builtin_isfinite(x)) {
                lo[d] = x;
                hi[d] = x;
            }
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fminf(lo[d], __shfl_xor(lo[d], o, 64));
            hi[d] = fmaxf(hi[d], __shfl_xor(hi[d], o, 64));
        }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            s[d][wave] = lo[d];
            s[3 + d][wave] = hi[d];
        }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = s[threadIdx.x][0];
#pragma unroll
        for (int w = 1; w < kBlock / 64; w++) v = threadIdx.x < 3 ? fminf(v, s[threadIdx.x][w]) : fmaxf(v, s[threadIdx.x][w]);
        part[6 * (size_t)blockIdx.x + threadIdx.x] = v;
    }
}

// One workgroup: the blocks' boxes into bbox[0..6).
__global__ void __launch_bounds__(kBlock) k_bbox_final(const float* __restrict__ part, int nb, float* __restrict__ bbox) {
    __shared__ float s[6][kBlock];
    float lo[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()};
    float hi[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
    for (int b = threadIdx.x; b < nb; b += kBlock)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            lo[d] = fminf(lo[d], part[6 * (size_t)b + d]);
            hi[d] = fmaxf(hi[d], part[6 * (size_t)b + 3 + d]);
        }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        s[d][threadIdx.x] = lo[d];
        s[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        float v = s[threadIdx.x][0];
        for (int t = 1; t < kBlock; t++) v = threadIdx.x < 3 ? fminf(v, s[threadIdx.x][t]) : fmaxf(v, s[threadIdx.x][t]);
        bbox[threadIdx.x] = v;
    }
}

// 10 bits of x spread to every third bit
__device__ __forceinline__ uint32_t spread3(uint32_t x) {
    x &= 0x3FFu;
    x = (x | (x << 16)) & 0x030000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// keys[i] = the 30-bit Morton code of row i's mean in the box (10 bits per axis; non-finite: 0), vals[i] = i
__global__ void __launch_bounds__(kBlock) k_morton(const float* __restrict__ m, size_t R, int count,
                                                   const float* __restrict__ bbox, uint32_t* __restrict__ keys,
                                                   int32_t* __restrict__ vals) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= count) return;
    uint32_t q[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float lo = bbox[d], ext = bbox[3 + d] - bbox[d];
        const float x = m[d * R + i];
        const float t = ext > 0.f ? (x - lo) / ext : 0.f;  // NaN (non-finite x) fails both compares below
        q[d] = t > 0.f ? static_cast<uint32_t>(fminf(t, 1.0f) * 1023.0f) : 0u;
    }
    keys[i] = spread3(q[0]) | (spread3(q[1]) << 1) | (spread3(q[2]) << 2);
    vals[i] = i;
}

// Rows between the arena's columns (SoA, stride R) and row-major arrays of DIM floats per row, a block of
// ROWS rows through LDS: the columns are read or written 64 rows at a time (256-B runs) and the row-major
// side element by element along each row, so both sides are coalesced also where the rows go to (dst) or
// come from (src) other places: a whole row is one run of 4 DIM bytes. Bound: HBM, 8 B per element. At 1 M rows and
// SH3 the 45-column group takes 0.104 ms to pack and 0.076 ms to unpack (3.5 and 4.7 TB/s), and the whole
// permutation of parameters and moments (18 arrays, through a row-major copy) about 0.95 ms. Before, a thread
// per row-major element touched the columns at a stride of DIM threads (an upload's and a download's kernels
// 0.97 and 0.73 ms), and a permutation gathered single floats from 177 columns (3.06 ms).

// aos[dst(k) * DIM + d] = soa[d * R + k] for rows k < n, dst(k) = dst_row[k] below n_perm, k at or past it
// (k where dst_row is null); rows whose place is at or past n_out are left out.
template <int DIM, int ROWS>
__global__ void __launch_bounds__(kBlock) k_rows_pack(const float* __restrict__ soa, size_t R, int n,
                                                      const int32_t* __restrict__ dst_row, int n_perm, int n_out,
                                                      float* __restrict__ aos) {
    constexpr int kPitch = DIM | 1;  // an odd pitch: no bank conflicts down a column
    __shared__ float s_v[ROWS * kPitch];
    __shared__ int32_t s_dst[ROWS];
    const int k0 = blockIdx.x * ROWS;
    const int m = min(ROWS, n - k0);
    for (int q = threadIdx.x; q < ROWS; q += kBlock) s_dst[q] = (dst_row && k0 + q < n_perm) ? dst_row[k0 + q] : k0 + q;
    const int r = threadIdx.x % ROWS;
#pragma unroll
    for (int d = threadIdx.x / ROWS; d < DIM; d += kBlock / ROWS)
        if (r < m) s_v[r * kPitch + d] = soa[(size_t)d * R + k0 + r];
    __syncthreads();
#pragma unroll 4
    for (int q = threadIdx.x; q < m * DIM; q += kBlock) {
        const int row = q / DIM, d = q - row * DIM;
        const int to = s_dst[row];
        if (to < n_out) aos[(size_t)to * DIM + d] = s_v[row * kPitch + d];
    }
}

// soa[d * R + k] = aos[src(k) * DIM + d] for rows k < n, src(k) = src_row[k] (k where src_row is null)
template <int DIM, int ROWS>
__global__ void __launch_bounds__(kBlock) k_rows_unpack(const float* __restrict__ aos, size_t R, int n,
                                                        const int32_t* __restrict__ src_row, float* __restrict__ soa) {
    constexpr int kPitch = DIM | 1;
    __shared__ float s_v[ROWS * kPitch];
    __shared__ int32_t s_src[ROWS];
    const int k0 = blockIdx.x * ROWS;
    const int m = min(ROWS, n - k0);
    for (int q = threadIdx.x; q < m; q += kBlock) s_src[q] = src_row ? src_row[k0 + q] : k0 + q;
    __syncthreads();
#pragma unroll 4
    for (int q = threadIdx.x; q < m * DIM; q += kBlock) {
        const int row = q / DIM, d = q - row * DIM;
        s_v[row * kPitch + d] = aos[(size_t)s_src[row] * DIM + d];
    }
    __syncthreads();
    const int r = threadIdx.x % ROWS;
#pragma unroll
    for (int d = threadIdx.x / ROWS; d < DIM; d += kBlock / ROWS)
        if (r < m) soa[(size_t)d * R + k0 + r] = s_v[r * kPitch + d];
}

// Calls f with the group's dimension as a compile-time constant (the six groups' dimensions at SH degrees 0-3)
// and the rows of a block: 256 for the narrow groups, 64 where a row is 96 B and more (12 KB of LDS at most).
template <class F>
void with_dim(int dim, F&& f) {
    switch (dim) {
        case 1: f(std::integral_constant<int, 1>{}, std::integral_constant<int, 256>{}); return;
        case 3: f(std::integral_constant<int, 3>{}, std::integral_constant<int, 256>{}); return;
        case 4: f(std::integral_constant<int, 4>{}, std::integral_constant<int, 256>{}); return;
        case 9: f(std::integral_constant<int, 9>{}, std::integral_constant<int, 256>{}); return;
        case 24: f(std::integral_constant<int, 24>{}, std::integral_constant<int, 64>{}); return;
        case 45: f(std::integral_constant<int, 45>{}, std::integral_constant<int, 64>{}); return;
        default: throw std::invalid_argument("arena rows: no such group dimension");
    }
}

// the maps of a permutation from the original order: internal row k holds original row src[k]
__global__ void __launch_bounds__(kBlock) k_perm_maps(const int32_t* __restrict__ src, int count,
                                                      int32_t* __restrict__ row_orig, int32_t* __restrict__ row_int) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= count) return;
    const int32_t o = src[k];
    row_orig[k] = o;
    row_int[o] = k;
}

}  // namespace

void arena_morton_keys(const Arena& A, int count, float* scratch, uint32_t* keys, int32_t* vals, hipStream_t s) {
    if (count <= 0) return;
    const int nb = grid_for(count);
    float* part = scratch + 8;  // scratch[0..6): the box
    hipLaunchKernelGGL(k_bbox_part, dim3(nb), dim3(kBlock), 0, s, A.p[0], static_cast<size_t>(A.rows), count, part);
    hipLaunchKernelGGL(k_bbox_final, dim3(1), dim3(kBlock), 0, s, part, nb, scratch);
    hipLaunchKernelGGL(k_morton, dim3(nb), dim3(kBlock), 0, s, A.p[0], static_cast<size_t>(A.rows), count, scratch,
                       keys, vals);
}

size_t arena_morton_scratch_floats(int count) { return 8 + 6 * static_cast<size_t>(grid_for(count)); }

void soa_to_rows(const float* soa, float* aos, int n, int dim, int stride, hipStream_t s, const int32_t* dst_row,
                 int n_perm, int n_out) {
    if (n <= 0) return;
    with_dim(dim, [&](auto D, auto B) {
        hipLaunchKernelGGL((k_rows_pack<D(), B()>), dim3((n + B() - 1) / B()), dim3(kBlock), 0, s, soa,
                           static_cast<size_t>(stride), n, dst_row, n_perm, n_out < 0 ? n : n_out, aos);
    });
}

void rows_to_soa(const float* aos, float* soa, int n, int dim, int stride, hipStream_t s, const int32_t* src_row) {
    if (n <= 0) return;
    with_dim(dim, [&](auto D, auto B) {
        hipLaunchKernelGGL((k_rows_unpack<D(), B()>), dim3((n + B() - 1) / B()), dim3(kBlock), 0, s, aos,
                           static_cast<size_t>(stride), n, src_row, soa);
    });
}

void arena_permute_rows(const Arena& A, const int dims[6], int count, const int32_t* src, float* tmp, hipStream_t s) {
    if (count <= 0) return;
    for (int g = 0; g < 6; g++) {
        if (dims[g] == 0) continue;
        for (float* col : {A.p[g], A.m[g], A.v[g]}) {
            if (!col) continue;
            soa_to_rows(col, tmp, count, dims[g], A.rows, s);
            rows_to_soa(tmp, col, count, dims[g], A.rows, s, src);
        }
    }
}

void perm_maps(const int32_t* src, int count, int32_t* row_orig, int32_t* row_int, hipStream_t s) {
    if (count <= 0) return;
    hipLaunchKernelGGL(k_perm_maps, dim3(grid_for(count)), dim3(kBlock), 0, s, src, count, row_orig, row_int);
}

}  // namespace sxk
