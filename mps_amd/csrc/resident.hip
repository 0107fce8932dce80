// resident.hip — the Jacobi-scaled conjugate gradients of small and middle
// systems as one launch.
//
// Run by launches, an iteration is two dependent kernels (k_cg_apply,
// k_cg_step): 8-11 us whatever the size up to some 30k rows, nearly all of it
// launch, block start-up and first loads.  Here every block of the same
// layout stays on its CU for the whole solve: one row a thread, the row's
// matrix entries and its p, s, y in registers, r of the block's rows and of
// the rows they couple to (the halo) in LDS.  An iteration exchanges A r of
// the halo rows and each block's three partial sums once, and every block
// applies the update to its halo rows itself (s = A r + beta s,
// r -= alpha s), so one exchange an iteration is enough.
//
// The exchange is of tagged words: 32 bits of the value below a 32-bit tag,
// stored and polled as relaxed device-scope 64-bit atomics.  A word carries
// its own readiness, so it needs no flag, fence or counter after it, and one
// store-to-load latency is the whole exchange (measured between 64 blocks
// spread over the 8 XCDs: 2.3 us an iteration with the reductions, 3.0 us
// between 256).  Two halves alternate: a block writes a half again only
// after it has every block's partials of the iteration between, which each
// block sends after it has read the half.
//
// Measured (2D, FP64, launches -> resident): 2,520 rows of 28 entries at
// machine epsilon 3.87 -> 1.60 ms a step of ~280 iterations; 32k rows of 12,
// ~21,500 iterations of a gradient evaluation 112 -> 59 ms.
//
// Sums are taken in the order and with the arithmetic of the two kernels, so
// the iterates are theirs bit for bit, and an ensemble member keeps its solo
// run's bits.
//
// Every block must be on a CU at once (the host launches no more than fit
// and counts the blocks in flight); a wait is bounded all the same: a block
// that waits too long, or whose halo does not fit, raises `bail`, tells its
// segment through a poisoned tag and leaves, and the host then solves by
// launches.
#pragma clang fp contract(off)

#include "cg_device.hpp"

namespace mps {

constexpr int kResHalo = 8;                           // halo rows a thread updates
constexpr int kResHaloRows = kResHalo * kCgBlock;     // halo rows of a block at most
constexpr int kResMaxRows = 131072;                   // rows of a segment (bits of the halo map)
constexpr long long kResWait = 5000000;               // ticks of the 100 MHz clock a wait may take (50 ms)

__device__ __forceinline__ void put_word(unsigned long long* p, unsigned v, unsigned tag) {
    __hip_atomic_store(p, ((unsigned long long) tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long get_word(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned tag_of(unsigned long long w) { return (unsigned) (w >> 32); }

// A value of T in kWords<T> tagged words.
template <typename T>
constexpr int kWords = (int) (sizeof(T) / 4);
template <typename T>
__device__ __forceinline__ void put_value(unsigned long long* p, T v, unsigned tag) {
    if constexpr (sizeof(T) == 8) {
        const unsigned long long b = (unsigned long long) __double_as_longlong(v);
        put_word(p, (unsigned) b, tag);
        put_word(p + 1, (unsigned) (b >> 32), tag);
    } else {
        put_word(p, __float_as_uint(v), tag);
    }
}
template <typename T>
__device__ __forceinline__ T value_of(const unsigned long long* w) {
    if constexpr (sizeof(T) == 8)
        return __longlong_as_double((long long) ((w[1] << 32) | (w[0] & 0xffffffffull)));
    else
        return __uint_as_float((unsigned) w[0]);
}

// A bounded wait: expired() every poll; true once it has taken too long.
struct Wait {
    int n = 0;
    long long t0 = 0;
    __device__ __forceinline__ bool expired() {
        if ((++n & 63) != 0) return false;
        const long long t = wall_clock64();
        if (n == 64) t0 = t;
        return t - t0 > kResWait;
    }
};

// acc + sum of val[k] * x[idx[k]] in entry order, each product and sum
// rounded by itself as sell_row does (contraction is off here).
template <typename T, int EMAX>
__device__ __forceinline__ T resident_row(const T (&v)[EMAX], const unsigned (&ix)[EMAX / 2],
                                          const T* __restrict__ x, int w, T acc) {
#pragma unroll
    for (int k = 0; k < EMAX; k += 4) {
        if (k < w) {
            T xv[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const unsigned pair = ix[(k + q) / 2];
                xv[q] = x[(k + q) & 1 ? pair >> 16 : pair & 0xffffu];
            }
#pragma unroll
            for (int q = 0; q < 4; q++) acc += v[k + q] * xv[q];  // entries past w: value 0, own row
        }
    }
    return acc;
}

template <typename T, typename IDX, int EMAX>
__global__ void __launch_bounds__(kCgBlock) k_cg_resident(Seg sg, const int* __restrict__ slice_pos,
                                                          const IDX* __restrict__ col, const int* __restrict__ anc,
                                                          const T* __restrict__ val, const T* __restrict__ r_in,
                                                          T* __restrict__ y_io, const double* __restrict__ dgl,
                                                          CgScalars* scs, CgExchange X) {
#pragma clang fp contract(fast)
    static_assert(EMAX % 4 == 0, "entries are taken four at a time");
    constexpr bool kWeighted = sizeof(T) == 8;  // the FP64 solve stops on the unscaled residual
    constexpr int NW = kCgBlock / 64;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double s_wave[3 * NW], s_red[3 * NW];
    __shared__ int s_scan[NW + 1];
    __shared__ int s_bad;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const BlockRows br = block_rows(sg);
    CgScalars* sc = scs + br.seg;
    if (block_uniform_done(sc)) return;
    const int base = sg.row_off[br.seg];
    const int rows = sg.row_off[br.seg + 1] - base;
    const int nb = br.nb;
    const int own = br.r1 - br.r0;
    const int words = (rows + 31) >> 5;
    T* const x = (T*) smem;                                             // r: own rows, then the halo
    unsigned* const bits = (unsigned*) (smem + sizeof(T) * (kCgBlock + kResHaloRows));
    unsigned short* const pre = (unsigned short*) (bits + words);
    int* const hcol = (int*) x;                                         // while the halo is listed
    const unsigned tag0 = sc->tag0;
    const int max_iter = sc->max_iter;
    const double thr = sc->thr;
    const unsigned poison = tag0 + (unsigned) max_iter + 3u;
    const int row = br.r0 + tid;
    const bool live = tid < own;

    // ---- the row's entries, and the halo: the rows of the segment outside
    // the block that some entry names, numbered in row order
    for (int i = tid; i < words; i += kCgBlock) bits[i] = 0;
    if (tid == 0) s_bad = 0;
    int w = 0, lo = 0, hi = 0;
    size_t eb = 0;
    if (live) {
        const int sl = row >> 6;
        const int s0 = slice_pos[sl];
        w = slice_pos[sl + 1] - s0;
        eb = (size_t) s0 * 64 + (row & 63);
        sell_anchors<IDX>(anc, row, lo, hi);
    }
    T v[EMAX];
    int c[EMAX];
#pragma unroll
    for (int k = 0; k < EMAX; k++) {
        v[k] = (T) 0;
        c[k] = row;
        if (k < w) {
            v[k] = val[eb + (size_t) k * 64];
            c[k] = sell_col<IDX>(col, eb + (size_t) k * 64, row, lo, hi);
        }
    }
    __syncthreads();
    auto mark = [&](int cc) {
        if (cc < br.r0 || cc >= br.r1) atomicOr(&bits[(cc - base) >> 5], 1u << ((cc - base) & 31));
    };
    if (live) {
#pragma unroll
        for (int k = 0; k < EMAX; k++)
            if (k < w) mark(c[k]);
        for (int k = EMAX; k < w; k++) mark(sell_col<IDX>(col, eb + (size_t) k * 64, row, lo, hi));
    }
    __syncthreads();
    const int per = (words + kCgBlock - 1) / kCgBlock;
    int cnt = 0;
    for (int i = 0; i < per; i++) {
        const int q = tid * per + i;
        if (q < words) cnt += __popc(bits[q]);
    }
    int inc = cnt;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) s_scan[wid] = inc;
    __syncthreads();
    int off = inc - cnt, H = 0;
    for (int k = 0; k < NW; k++) {
        if (k < wid) off += s_scan[k];
        H += s_scan[k];
    }
    const bool fits = H <= X.halo_max;  // block-uniform
    int hc[kResHalo];
    T hs[kResHalo];
    if (fits) {
        for (int i = 0; i < per; i++) {
            const int q = tid * per + i;
            if (q >= words) break;
            unsigned m = bits[q];
            pre[q] = (unsigned short) off;
            while (m) {
                hcol[off++] = base + 32 * q + __builtin_ctz(m);
                m &= m - 1;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kResHalo; i++) {
            const int h = i * kCgBlock + tid;
            hc[i] = h < H ? hcol[h] : -1;
            hs[i] = (T) 0;
        }
        __syncthreads();
    }
    // place in x of column cc
    auto place = [&](int cc) -> unsigned {
        if (cc >= br.r0 && cc < br.r1) return (unsigned) (cc - br.r0);
        const int q = cc - base;
        return (unsigned) (kCgBlock + pre[q >> 5] + __popc(bits[q >> 5] & ((1u << (q & 31)) - 1u)));
    };
    unsigned ix[EMAX / 2];
    T r = (T) 0, p = (T) 0, s = (T) 0, y = (T) 0;
    double dg = 0.0;
    if (fits) {
#pragma unroll
        for (int k = 0; k < EMAX; k += 2) {
            const unsigned a = live && k < w ? place(c[k]) : (unsigned) tid;
            const unsigned b = live && k + 1 < w ? place(c[k + 1]) : (unsigned) tid;
            ix[k / 2] = a | (b << 16);
        }
        if (live) {
            r = r_in[row];
            y = y_io[row];
            if (kWeighted) dg = dgl[row];
        }
        x[tid] = r;
#pragma unroll
        for (int i = 0; i < kResHalo; i++)
            if (hc[i] >= 0) x[kCgBlock + i * kCgBlock + tid] = r_in[hc[i]];
        __syncthreads();
    }
    auto leave = [&]() {  // block-uniform
        if (tid == 0) atomicOr(&sc->bail, 1);
        if (tid < 2 && nb > 1) put_word(X.part + (size_t) tid * X.p_half + (size_t) blockIdx.x * 6, 0u, poison);
    };
    if (!fits) {
        leave();
        return;
    }

    // ---- iterations
    double gam_old = 0.0, alp_old = 0.0;
    for (int it = 1;; it++) {
        const unsigned tag = tag0 + (unsigned) it;
        unsigned long long* const xw = X.w + (size_t) (it & 1) * X.w_half;
        unsigned long long* const xp = X.part + (size_t) (it & 1) * X.p_half;
        // A r of the own row (unit diagonal)
        T ar = resident_row<T, EMAX>(v, ix, x, w, r);
        for (int k = EMAX; k < w; k++) {
            const size_t e = eb + (size_t) k * 64;
            const T one[4] = {val[e], (T) 0, (T) 0, (T) 0};
            const unsigned at[2] = {place(sell_col<IDX>(col, e, row, lo, hi)) | ((unsigned) tid << 16),
                                    (unsigned) tid | ((unsigned) tid << 16)};
            ar = resident_row<T, 4>(one, at, x, 1, ar);
        }
        if (live && nb > 1) put_value<T>(xw + (size_t) row * kWords<T>, ar, tag);
        // the block's partial sums: r.r, (A r).r and the stopping norm
        double part[3] = {0.0, 0.0, 0.0};
        if (live) {
            const double r2 = (double) r * (double) r;
            part[0] += (double) r * (double) r;
            part[1] += (double) ar * (double) r;
            part[2] += kWeighted ? dg * r2 : r2;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            double a = part[k];
            for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
            if (lane == 0) s_wave[wid * 3 + k] = a;
        }
        __syncthreads();
        double sum[3];
        T hw[kResHalo];
        if (nb == 1) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                double t = 0.0;
                for (int q = 0; q < NW; q++) t += s_wave[q * 3 + k];
                sum[k] = t;
            }
        } else {
            if (tid < 3) {
                double t = 0.0;
                for (int q = 0; q < NW; q++) t += s_wave[q * 3 + tid];
                put_value<double>(xp + (size_t) blockIdx.x * 6 + 2 * tid, t, tag);
            }
            bool bad = false;
            double acc[3] = {0.0, 0.0, 0.0};
            if (tid < nb) {
                const unsigned long long* q = xp + (size_t) (br.b0 + tid) * 6;
                unsigned long long m[6];
                Wait wt;
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (int k = 0; k < 6; k++) m[k] = get_word(q + k);
#pragma unroll
                    for (int k = 0; k < 6; k++) ok = ok && tag_of(m[k]) == tag;
                    if (ok) break;
                    if (tag_of(m[0]) == poison || wt.expired()) {
                        bad = true;
                        break;
                    }
                }
#pragma unroll
                for (int k = 0; k < 3; k++) acc[k] += value_of<double>(m + 2 * k);
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                double a = acc[k];
                for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
                if (lane == 0) s_red[wid * 3 + k] = a;
            }
            // A r of the thread's halo rows
            {
                Wait wt;
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (int i = 0; i < kResHalo; i++) {
                        if (hc[i] < 0) continue;
                        unsigned long long m[kWords<T>];
#pragma unroll
                        for (int k = 0; k < kWords<T>; k++) m[k] = get_word(xw + (size_t) hc[i] * kWords<T> + k);
#pragma unroll
                        for (int k = 0; k < kWords<T>; k++) ok = ok && tag_of(m[k]) == tag;
                        hw[i] = value_of<T>(m);
                    }
                    if (ok) break;
                    if (wt.expired()) {
                        bad = true;
                        break;
                    }
                }
            }
            if (bad) s_bad = 1;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 3; k++) {
                double t = 0.0;
                for (int q = 0; q < NW; q++) t += s_red[q * 3 + k];
                sum[k] = t;
            }
            if (s_bad) {
                leave();
                return;
            }
        }
        const double g = sum[0], dd = sum[1], rho = sum[2];
        const bool first = it == 1;
        const bool conv = rho <= thr;
        if (conv || it > max_iter || !(rho == rho)) {
            if (live) y_io[row] = y;
            if (br.v == 0 && tid == 0) {
                sc->done = 1;
                sc->converged = conv ? 1 : 0;
                sc->rho2 = rho;
                sc->fin = it - 1;
            }
            return;
        }
        const double b = first ? 0.0 : g / gam_old;
        const double a = first ? g / dd : g / (dd - b * g / alp_old);
        gam_old = g;
        alp_old = a;
        const T alpha = (T) a, beta = (T) b;
        p = first ? r : r + beta * p;
        s = first ? ar : ar + beta * s;
        y = y + alpha * p;
        r = r - alpha * s;
        x[tid] = r;
#pragma unroll
        for (int i = 0; i < kResHalo; i++) {
            if (hc[i] < 0) continue;
            T* const xh = x + kCgBlock + i * kCgBlock + tid;
            hs[i] = first ? hw[i] : hw[i] + beta * hs[i];
            *xh = *xh - alpha * hs[i];
        }
        __syncthreads();
    }
}

size_t resident_lds(int max_rows, int tsize) {
    if (max_rows > kResMaxRows) return 0;
    const size_t words = (size_t) (max_rows + 31) / 32;
    return (size_t) tsize * (kCgBlock + kResHaloRows) + words * 4 + ((words * 2 + 15) & ~(size_t) 15);
}

int resident_halo_rows() { return kResHaloRows; }

// Entries held in registers: 16 covers a 2D system at 2.1 l0 (12-14 a row),
// 36 one at 3.1 l0 (28-32) and 3D at 2.1 l0 (32-34); a wider row reads the
// rest from memory every iteration.
constexpr int kResFew = 16, kResMany = 36;

template <typename T, typename IDX>
hipError_t resident_prepare(int mean_width) {
    const int bytes = (int) resident_lds(kResMaxRows, (int) sizeof(T));
    return hipFuncSetAttribute(mean_width <= kResFew ? (const void*) k_cg_resident<T, IDX, kResFew>
                                                     : (const void*) k_cg_resident<T, IDX, kResMany>,
                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

template <typename T, typename IDX>
hipError_t resident_launch(const Seg& sg, int total_blocks, const int* slice_off, const IDX* col, const int* anc,
                           const T* val, const T* r, T* y, const double* dgl, CgScalars* sc, const CgExchange& x,
                           int mean_width, size_t lds, hipStream_t st) {
    if (mean_width <= kResFew)
        hipLaunchKernelGGL((k_cg_resident<T, IDX, kResFew>), dim3(total_blocks), dim3(kCgBlock), lds, st, sg, slice_off,
                           col, anc, val, r, y, dgl, sc, x);
    else
        hipLaunchKernelGGL((k_cg_resident<T, IDX, kResMany>), dim3(total_blocks), dim3(kCgBlock), lds, st, sg,
                           slice_off, col, anc, val, r, y, dgl, sc, x);
    return hipGetLastError();
}

#define RESIDENT_INST(T, IDX)                                                                                       \
    template hipError_t resident_prepare<T, IDX>(int);                                                              \
    template hipError_t resident_launch<T, IDX>(const Seg&, int, const int*, const IDX*, const int*, const T*,      \
                                                const T*, T*, const double*, CgScalars*, const CgExchange&, int,    \
                                                size_t, hipStream_t);
RESIDENT_INST(double, short)
RESIDENT_INST(double, unsigned short)
RESIDENT_INST(double, int)
RESIDENT_INST(float, short)
RESIDENT_INST(float, unsigned short)
RESIDENT_INST(float, int)
#undef RESIDENT_INST

}  // namespace mps
