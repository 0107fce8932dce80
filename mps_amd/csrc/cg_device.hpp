// cg_device.hpp — what the conjugate-gradient kernels share: the segment
// layout, the per-segment scalars, the fixed-order reductions and the SELL row
// product.  Include it where floating-point contraction is off: the row
// product rounds each multiply and add by itself.
#pragma once

#include "mps_internal.hpp"

namespace mps {

constexpr int kMaxBlocks = 1024;  // per segment
// Threads per block of the per-iteration kernels (apply, step): 1024 blocks
// of 512 fill every SIMD with 8 waves, twice the loads in flight of 256.
constexpr int kCgBlock = 512;

struct CgScalars {
    double gam[2];     // r.r by iteration parity
    double alp[2];     // alpha by iteration parity
    double thr;        // stop when rho2 <= thr
    double rho2;       // latest residual^2 (unscaled sum a_ii r_i^2, or r.r for inner solves)
    double red[3];     // results of k_reduce_parts
    int iter;          // apply launches run (read by every block of k_cg_step)
    int max_iter;
    int done;
    int converged;
    int frozen;        // timing mode: kernels leave every scalar as it is
    int fin;           // completed updates, written once when the segment stops
    int bail;          // resident CG: a workgroup gave up; the host runs the solve again by launches
    unsigned tag0;     // resident CG: exchange tags of this launch start after it
};

struct Seg {
    int nseg;
    const int* blk_off;  // nseg + 1: first block of each segment
    const int* row_off;  // nseg + 1: first row of each segment
};

__device__ __forceinline__ int seg_of_block(const Seg& sg, int b) {
    int lo = 0, hi = sg.nseg - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sg.blk_off[mid] <= b)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

struct BlockRows {
    int seg, v, nb, b0;  // segment, block within it, its block count, its first block
    int lb;              // the block's place among the segment's contiguous row ranges
    int r0, r1;          // rows of this block
};

// Row range of this block: contiguous within the segment, whole multiples of
// 64 rows from the segment start, XCD-grouped.
__device__ __forceinline__ BlockRows block_rows(const Seg& sg) {
    BlockRows br;
    br.seg = seg_of_block(sg, blockIdx.x);
    br.b0 = sg.blk_off[br.seg];
    br.v = blockIdx.x - br.b0;
    br.nb = sg.blk_off[br.seg + 1] - br.b0;
    const int base = sg.row_off[br.seg];
    const int rows = sg.row_off[br.seg + 1] - base;
    const int per = ((rows + br.nb - 1) / br.nb + 63) & ~63;
    const int lb = xcd_block(br.v, br.nb);
    br.lb = lb;
    br.r0 = base + lb * per;
    const int end = base + rows;
    br.r1 = br.r0 + per < end ? br.r0 + per : end;
    if (br.r0 > end) br.r0 = end;
    return br;
}

// Fixed-order sum of NV interleaved partials (part[b*NV + k], b < nb) in every
// block; result broadcast to all threads.
template <int NV>
__device__ __forceinline__ void reduce_partials(const double* __restrict__ part, int nb, double (&out)[NV],
                                                double* red) {
    double acc[NV];
    for (int k = 0; k < NV; k++) acc[k] = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x)
        for (int k = 0; k < NV; k++) acc[k] += part[(size_t) NV * b + k];
    for (int k = 0; k < NV; k++) {
        double a = acc[k];
        for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
        if ((threadIdx.x & 63) == 0) red[(threadIdx.x >> 6) * NV + k] = a;
    }
    __syncthreads();
    for (int k = 0; k < NV; k++) {
        double t = 0.0;
        for (int w = 0; w < (int) (blockDim.x >> 6); w++) t += red[w * NV + k];
        out[k] = t;
    }
    __syncthreads();
}

template <int NV>
__device__ __forceinline__ void write_partials(const double (&v)[NV], double* __restrict__ part, double* red) {
    for (int k = 0; k < NV; k++) {
        double a = v[k];
        for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
        if ((threadIdx.x & 63) == 0) red[(threadIdx.x >> 6) * NV + k] = a;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double t = 0.0;
        for (int w = 0; w < (int) (blockDim.x >> 6); w++) t += red[w * NV + threadIdx.x];
        part[(size_t) NV * blockIdx.x + threadIdx.x] = t;
    }
}

__device__ __forceinline__ int block_uniform_done(CgScalars* sc) {
    __shared__ int s_done;
    if (threadIdx.x == 0) s_done = *(volatile int*) &sc->done;
    __syncthreads();
    return s_done;
}

// acc + sum_k val[k] x[col[k]] over the row's SELL entries, gathers issued in
// batches of 4 for memory-level parallelism.  NT: the matrix is read with
// nontemporal loads (the FP64 solve's apply: its 10 bytes an entry do not
// fit the Infinity Cache beside the solver's vectors, and streaming them
// keeps the vectors and coarse levels cached: 2M FP64 step -6 %; the FP32
// matrix does fit and is read normally, as is the FP64 residual's, where
// nontemporal loads made the mixed step 2 % slower).
template <typename T, typename IDX, bool NT = false>
__device__ __forceinline__ T sell_row(const int* __restrict__ slice_pos, const IDX* __restrict__ col,
                                      const int* __restrict__ anc, const T* __restrict__ val,
                                      const T* __restrict__ x, int row, T acc) {
    const int sl = row >> 6, lane = row & 63;
    const int s0 = slice_pos[sl], w = slice_pos[sl + 1] - s0;
    const size_t base = (size_t) s0 * 64 + lane;
    int lo, hi;
    sell_anchors<IDX>(anc, row, lo, hi);
    int k = 0;
    for (; k + 4 <= w; k += 4) {
        const size_t i0 = base + (size_t) k * 64;
        const int c0 = sell_col<IDX, NT>(col, i0, row, lo, hi), c1 = sell_col<IDX, NT>(col, i0 + 64, row, lo, hi);
        const int c2 = sell_col<IDX, NT>(col, i0 + 128, row, lo, hi), c3 = sell_col<IDX, NT>(col, i0 + 192, row, lo, hi);
        const T v0 = ld_stream<NT>(val + i0), v1 = ld_stream<NT>(val + i0 + 64);
        const T v2 = ld_stream<NT>(val + i0 + 128), v3 = ld_stream<NT>(val + i0 + 192);
        const T x0 = x[c0], x1 = x[c1], x2 = x[c2], x3 = x[c3];
        acc += v0 * x0;
        acc += v1 * x1;
        acc += v2 * x2;
        acc += v3 * x3;
    }
    for (; k < w; k++) {
        const size_t i0 = base + (size_t) k * 64;
        acc += ld_stream<NT>(val + i0) * x[sell_col<IDX, NT>(col, i0, row, lo, hi)];
    }
    return acc;
}


// ---- resident CG (resident.hip) ----
//
// Exchange memory of the resident CG's workgroups: tagged words (a 32-bit
// value below a 32-bit tag) in two alternating halves.
struct CgExchange {
    unsigned long long* w;     // 2 x w_half: A r of every row
    unsigned long long* part;  // 2 x p_half: 3 partial sums of every block
    size_t w_half, p_half;
    int halo_max;              // most halo rows a block takes (resident_halo_rows() at most)
};
// LDS the kernel needs for segments of at most max_rows rows; 0 if it cannot
// take them.
size_t resident_lds(int max_rows, int tsize);
int resident_halo_rows();
// Lets the kernel of this shape use its LDS (once per device before a launch).
template <typename T, typename IDX>
hipError_t resident_prepare(int mean_width);
// Enqueues the whole CG (every iteration up to each segment's stop) as one
// launch of total_blocks workgroups, one per block of the layout.  All of
// them must be able to run at once.
template <typename T, typename IDX>
hipError_t resident_launch(const Seg& sg, int total_blocks, const int* slice_off, const IDX* col, const int* anc,
                           const T* val, const T* r, T* y, const double* dgl, CgScalars* sc, const CgExchange& x,
                           int mean_width, size_t lds, hipStream_t st);

}  // namespace mps
