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

// Row range of a block: contiguous within the segment, whole multiples of
// 64 rows from the segment start, XCD-grouped.
__device__ __forceinline__ BlockRows block_rows(const Seg& sg, int block) {
    BlockRows br;
    br.seg = seg_of_block(sg, block);
    br.b0 = sg.blk_off[br.seg];
    br.v = block - br.b0;
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
__device__ __forceinline__ BlockRows block_rows(const Seg& sg) { return block_rows(sg, blockIdx.x); }

// a of the lane CTRL places up in the row of 16 (0 past its end).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double a) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(a), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(a), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// Sum over the wavefront by the tree a += a[lane + 32], + 16, ... + 1, valid
// in lane 0: the sums of a __shfl_down loop bit for bit, with register moves
// (lane swaps of gfx950 for 32 and 16, DPP row shifts for 8 to 1) in place of
// LDS permutes, whose latency is several times an add's.
__device__ __forceinline__ double wave_sum(double a) {
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(a), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(a), false, false);
        a += __hiloint2double((int) hi[1], (int) lo[1]);
    }
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(a), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(a), false, false);
        a += __hiloint2double((int) hi[1], (int) lo[1]);
    }
    a += dpp_f64<0x108>(a);
    a += dpp_f64<0x104>(a);
    a += dpp_f64<0x102>(a);
    a += dpp_f64<0x101>(a);
    return a;
}

// wave_sum of three values at once: a's sum in lane 0, b's in lane 32, c's in
// lane 16.  The first two levels' lane swaps put different values into the
// halves and rows that a single sum leaves idle (after the level of 32 a sum
// lives in half the lanes, after 16 in a quarter), so three trees cost little
// more than one; each value is still added in the order of its own tree.
__device__ __forceinline__ double wave_sum3(double a, double b, double c) {
    auto swap_add32 = [](double x, double y) {  // x[i] + x[i + 32] below lane 32, y's above
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(y), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(y), false, false);
        return __hiloint2double((int) hi[0], (int) lo[0]) + __hiloint2double((int) hi[1], (int) lo[1]);
    };
    const double ab = swap_add32(a, b), cc = swap_add32(c, 0.0);
    double t;
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(ab), __double2loint(cc), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(ab), __double2hiint(cc), false, false);
        t = __hiloint2double((int) hi[0], (int) lo[0]) + __hiloint2double((int) hi[1], (int) lo[1]);
    }
    t += dpp_f64<0x108>(t);
    t += dpp_f64<0x104>(t);
    t += dpp_f64<0x102>(t);
    t += dpp_f64<0x101>(t);
    return t;
}
// The value of wave_sum3 (0, 1, 2) a lane holds, -1 for none.
__device__ __forceinline__ int sum3_of_lane(int lane) {
    return lane == 0 ? 0 : (lane == 32 ? 1 : (lane == 16 ? 2 : -1));
}

// Each wavefront's sums of NV values into red[wavefront * NV + k].
template <int NV>
__device__ __forceinline__ void wave_partials(const double (&v)[NV], double* red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if constexpr (NV == 3) {
        const double t = wave_sum3(v[0], v[1], v[2]);
        const int k = sum3_of_lane(lane);
        if (k >= 0) red[w * 3 + k] = t;
    } else {
        for (int k = 0; k < NV; k++) {
            const double a = wave_sum(v[k]);
            if (lane == 0) red[w * NV + k] = a;
        }
    }
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
    wave_partials<NV>(acc, red);
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
    wave_partials<NV>(v, red);
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


// FP64 CG restarts from the current iterate when the true residual of the
// recurrence's answer misses the tolerance.
constexpr int kMaxRestarts = 3;

// ---- resident solves (resident.hip) ----
//
// Exchange memory of the workgroups: tagged words (a 32-bit value below a
// 32-bit tag) in two alternating halves.
struct CgExchange {
    unsigned long long* w;     // 2 halves x 2 words x w_rows: a value of every row
    unsigned long long* part;  // 2 halves x p_sums places: 3 partial sums of every block or wavefront
    size_t w_rows, p_sums;
    int halo_max;              // lowers the halo rows a workgroup takes (tests)
};
// Options of a solve, read by its launch (pinned host memory).
struct ResidentIn {
    double tol2;           // tolerance^2
    double eta2;           // inner tolerance^2 (mixed)
    int max_iterations;    // <= 0: 2 x the segment's rows
    int max_refinements;   // restarts (FP64) or refinements (mixed) at most
    unsigned tag0;         // the launch's exchange tags follow it
    unsigned poison;       // the tag of a workgroup that gave up
    unsigned seq;          // the solve's number
};
// Results of a segment, written by its last workgroup (pinned host memory).
struct ResidentOut {
    double bn2;            // ||b||^2
    double rho2_start;     // residual^2 of the start
    double rho2;           // true residual^2 of the result
    int iterations;
    int rounds;            // restarts or refinements
    int converged;
    int bail;              // some workgroup gave up: x is not set
    unsigned seq;          // ResidentIn::seq, written last
};
// Everything a launch receives (compared as bytes: captured graphs bake it in).
struct ResidentArgs {
    Seg sg;
    const int* slice_pos;
    const void* col;       // IDX
    const int* anc;
    const void* val;       // T
    const double* val64;
    const int* row_slot;
    const int32_t* id;     // null without a warm start
    const double* b;       // by slot
    const double* pprev;
    const double* pprev2;
    const double* sdiag;
    const double* dgl;
    double* x;             // by slot
    CgExchange X;
    int* count;            // per segment: workgroups that have left
    const ResidentIn* in;
    ResidentOut* out;
};
// Shape of a launch: workgroups per block of the layout (1 or kResSplit),
// matrix entries a thread holds in registers, dynamic LDS.
constexpr int kResSplit = 4;
struct ResidentShape {
    int split;  // 0: the kernel does not take this system
    int emax;
    size_t lds;
};
// The shape for segments of at most max_rows rows in at most max_nb blocks,
// total_rows and total_blocks in all, mean_width entries a row of entry_bytes
// each (value and column), with at most `most` workgroups at once.
ResidentShape resident_shape(int dim, int max_rows, int max_nb, int total_rows, int total_blocks, int mean_width,
                             int entry_bytes, int most, bool mixed);
// Tags a launch may use: its iterations and rounds bound its exchanges.
long long resident_tags(long long max_iterations, int max_rounds);
// Places for partial sums (CgExchange::p_sums) a launch needs, and the words
// both halves of them take.
size_t resident_sums(int total_blocks);
size_t resident_sum_words(size_t p_sums);
// Lets the kernel of this shape use its LDS (once before its first launch).
template <typename T, typename IDX>
hipError_t resident_prepare(const ResidentShape& s);
// Enqueues the solve of every segment as one launch of `grid` workgroups
// (split x blocks), all of which must be able to run at once.
// T: double, the FP64 path; float, the mixed path.
template <typename T, typename IDX>
hipError_t resident_launch(const ResidentShape& s, int grid, const ResidentArgs& a, hipStream_t st);

}  // namespace mps
