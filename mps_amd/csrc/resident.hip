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
// store-to-load latency is the whole exchange (1.4-1.5 us between 2 to 64
// workgroups spread over the 8 XCDs; on one XCD it is the same).  Two halves alternate: a block writes a half again only
// after it has every block's partials of the iteration between, which each
// block sends after it has read the half.
//
// Measured (2D, FP64, launches -> resident): 2,520 rows of 28 entries at
// machine epsilon 3.80 -> 1.28 ms a step of ~280 iterations; 32k rows of 12,
// ~10,700 iterations of a gradient evaluation 111 -> 44 ms.  What an
// iteration spends now (2.4 GHz cycles, FP64, 64 blocks): row product and
// wavefront sums 1700, exchange 3500 (one uncached store and load), adding
// the sums up 900, three divisions 700, updates 800.
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

constexpr int kResHalo = 8;               // halo rows a thread updates
constexpr int kResMaxRows = 131072;       // rows of a segment (bits of the halo map)
constexpr long long kResWait = 5000000;   // ticks of the 100 MHz clock a wait may take (50 ms)
constexpr int kResWaves = kCgBlock / 64;  // wavefronts of a block of the layout
constexpr int kResMaxBlocks = 256;        // blocks of a segment
constexpr int kResSplitSums = 128;        // wavefronts of a segment with split blocks
// Words from one place of partial sums to the next: three doubles are six;
// at eight a place has a 64-byte line to itself and is sent by one store of
// six lanes.
constexpr int kSumWords = 8;

__device__ __forceinline__ void put_word(unsigned long long* p, unsigned v, unsigned tag) {
    __hip_atomic_store(p, ((unsigned long long) tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long get_word(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The word at a byte offset from a base that is the same in every lane.
__device__ __forceinline__ unsigned long long get_word_at(const unsigned long long* base, unsigned bytes) {
    return get_word((const unsigned long long*) ((const char*) base + bytes));
}
__device__ __forceinline__ unsigned tag_of(unsigned long long w) { return (unsigned) (w >> 32); }

// A value of T in kWords<T> tagged words, `stride` words apart: a word of all
// rows, then the next, so that a wavefront's words share cache lines (these
// accesses bypass the caches, every line is a request of its own).
template <typename T>
constexpr int kWords = (int) (sizeof(T) / 4);
template <typename T>
__device__ __forceinline__ void put_value(unsigned long long* p, size_t stride, T v, unsigned tag) {
    if constexpr (sizeof(T) == 8) {
        const unsigned long long b = (unsigned long long) __double_as_longlong(v);
        put_word(p, (unsigned) b, tag);
        put_word(p + stride, (unsigned) (b >> 32), tag);
    } else {
        put_word(p, __float_as_uint(v), tag);
    }
}
// A wavefront's three sums as wave_sum3 leaves them (lanes 0, 32, 16), sent
// by six lanes.
__device__ __forceinline__ void send_sums(unsigned long long* p, double ws, unsigned tag) {
    const int lane = threadIdx.x & 63;
    const int from = lane >> 1 == 0 ? 0 : (lane >> 1 == 1 ? 32 : 16);
    const int lo = __builtin_amdgcn_ds_bpermute(4 * from, __double2loint(ws));
    const int hi = __builtin_amdgcn_ds_bpermute(4 * from, __double2hiint(ws));
    if (lane < 6) put_word(p + lane, (unsigned) (lane & 1 ? hi : lo), tag);
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
template <typename T>
__device__ __forceinline__ T add_product(T acc, T v, T x) {
    acc += v * x;
    return acc;
}
template <typename T, int EMAX>
__device__ __forceinline__ T resident_row(const T (&v)[EMAX], const unsigned (&ix)[EMAX / 2],
                                          const T* __restrict__ x, T acc) {
    T xv[EMAX];
#pragma unroll
    for (int k = 0; k < EMAX; k++) {
        const unsigned pair = ix[k / 2];
        xv[k] = x[k & 1 ? pair >> 16 : pair & 0xffffu];
    }
#pragma unroll
    for (int k = 0; k < EMAX; k++) acc += v[k] * xv[k];  // entries past the row's: value 0, own row
    return acc;
}

// BT rows a workgroup.  BT == kCgBlock: one workgroup a block of the layout;
// it sends the block's three sums, and every workgroup adds the blocks' sums
// up as k_cg_step does.  BT < kCgBlock: kCgBlock / BT workgroups a block, the
// wavefronts' sums are sent, and every workgroup adds them up to the blocks'
// sums first, in k_cg_apply's order.
//
// Every thread sends its own row and polls right after.  A wavefront's loads
// and stores complete in order, so its first poll also waits for its stores'
// acknowledgement; a load that bypasses the L2s takes as long anyway (2500
// cycles) and mostly finds the others' words in that time.  Separate sending
// and polling wavefronts were slower (2,520 rows 26.1 -> 30.5 ms per 20
// steps): the poll sampled memory too early and had to be repeated.
template <typename T, typename IDX, int EMAX, int BT>
__global__ void __launch_bounds__(BT)
    k_cg_resident(Seg sg, const int* __restrict__ slice_pos, const IDX* __restrict__ col, const int* __restrict__ anc,
                  const T* __restrict__ val, const T* __restrict__ r_in, T* __restrict__ y_io,
                  const double* __restrict__ dgl, CgScalars* scs, CgExchange X) {
#pragma clang fp contract(fast)
    static_assert(EMAX % 2 == 0, "two places share a word");
    constexpr bool kWeighted = sizeof(T) == 8;  // the FP64 solve stops on the unscaled residual
    constexpr int NW = BT / 64;
    constexpr int kSplit = kCgBlock / BT;
    constexpr bool kByWave = kSplit > 1;
    constexpr int kHaloRows = kResHalo * BT;
    // sums sent per workgroup: its block's, or its wavefronts'; and the most
    // a workgroup waits for
    constexpr int kSent = kByWave ? NW : 1;
    constexpr int kMaxSums = kByWave ? kResSplitSums : kResMaxBlocks;
    constexpr int kPoll = kMaxSums * kSumWords / BT;  // words of them a thread polls
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) unsigned s_sum[kMaxSums * 6];  // the doubles of all sums, 3 a place
    __shared__ __align__(16) double s_wave[3][NW];
    __shared__ int s_scan[NW];
    __shared__ int s_bad;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    BlockRows br = block_rows(sg, blockIdx.x / kSplit);
    CgScalars* sc = scs + br.seg;
    if (block_uniform_done(sc)) return;
    const int base = sg.row_off[br.seg];
    const int rows = sg.row_off[br.seg + 1] - base;
    const int nb = br.nb;
    if (kByWave) {  // this workgroup's share of the block
        const int part = blockIdx.x % kSplit;
        br.r0 = br.r0 + part * BT < br.r1 ? br.r0 + part * BT : br.r1;
        br.r1 = br.r0 + BT < br.r1 ? br.r0 + BT : br.r1;
    }
    const int own = br.r1 - br.r0;
    const bool alone = !kByWave && nb == 1;  // the segment is this workgroup's
    const int words = (rows + 31) >> 5;
    T* const x = (T*) smem;  // r: own rows, then the halo
    unsigned* const bits = (unsigned*) (smem + sizeof(T) * (BT + kHaloRows));
    unsigned short* const pre = (unsigned short*) (bits + words);
    int* const hcol = (int*) x;  // while the halo is listed
    const unsigned tag0 = sc->tag0;
    const int max_iter = sc->max_iter;
    const double thr = sc->thr;
    const unsigned poison = tag0 + (unsigned) max_iter + 3u;
    const int row = br.r0 + tid;
    const bool live = tid < own;
    // the sums this thread waits for, and where this workgroup's go
    const int nsum = kByWave ? nb * kResWaves : nb;
    const size_t sum0 = (size_t) br.b0 * (kByWave ? kResWaves : 1);
    const size_t mine = (size_t) blockIdx.x * kSent;

    // ---- the halo: the rows of the segment outside the workgroup's that
    // some entry names, numbered in row order
    for (int i = tid; i < words; i += BT) bits[i] = 0;
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
    int c[EMAX];
#pragma unroll
    for (int k = 0; k < EMAX; k++) c[k] = k < w ? sell_col<IDX>(col, eb + (size_t) k * 64, row, lo, hi) : row;
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
    const int per = (words + BT - 1) / BT;
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
    auto leave = [&]() {  // every thread of the workgroup
        if (tid == 0) atomicOr(&sc->bail, 1);
        if (tid < 2 * kSent * kSumWords && !alone) {
            const int half = tid / (kSent * kSumWords), at = tid % (kSent * kSumWords);
            put_word(X.part + (size_t) half * kSumWords * X.p_sums + mine * kSumWords + at, 0u, poison);
        }
    };
    if (H > kHaloRows || H > X.halo_max) {  // uniform in the workgroup
        leave();
        return;
    }
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
    int hc[kResHalo];
    T hs[kResHalo];
#pragma unroll
    for (int i = 0; i < kResHalo; i++) {
        const int h = i * BT + tid;
        hc[i] = h < H ? hcol[h] : -1;
        hs[i] = (T) 0;
    }
    __syncthreads();
    // place in x of column cc
    auto place = [&](int cc) -> unsigned {
        if (cc >= br.r0 && cc < br.r1) return (unsigned) (cc - br.r0);
        const int q = cc - base;
        return (unsigned) (BT + pre[q >> 5] + __popc(bits[q >> 5] & ((1u << (q & 31)) - 1u)));
    };
    unsigned ix[EMAX / 2];
    T v[EMAX];
    T r = (T) 0, p = (T) 0, s = (T) 0, y = (T) 0;
    double dg = 0.0;
#pragma unroll
    for (int k = 0; k < EMAX; k += 2) {
        const unsigned a = live && k < w ? place(c[k]) : (unsigned) tid;
        const unsigned b = live && k + 1 < w ? place(c[k + 1]) : (unsigned) tid;
        ix[k / 2] = a | (b << 16);
    }
#pragma unroll
    for (int k = 0; k < EMAX; k++) v[k] = k < w ? val[eb + (size_t) k * 64] : (T) 0;
    if (live) {
        r = r_in[row];
        y = y_io[row];
        if (kWeighted) dg = dgl[row];
    }
    x[tid] = r;
#pragma unroll
    for (int i = 0; i < kResHalo; i++)
        if (hc[i] >= 0) x[BT + i * BT + tid] = r_in[hc[i]];
    __syncthreads();

    // ---- iterations
    double gam_old = 0.0, alp_old = 0.0;
    for (int it = 1;; it++) {
        const unsigned tag = tag0 + (unsigned) it;
        unsigned long long* const xw = X.w + (size_t) (it & 1) * 2 * X.w_rows;
        unsigned long long* const xp = X.part + (size_t) (it & 1) * kSumWords * X.p_sums;
        // A r of the own row (unit diagonal)
        T ar = resident_row<T, EMAX>(v, ix, x, r);
        for (int k = EMAX; k < w; k++) {
            const size_t e = eb + (size_t) k * 64;
            ar = add_product(ar, val[e], x[place(sell_col<IDX>(col, e, row, lo, hi))]);
        }
        if (live && !alone) put_value<T>(xw + row, X.w_rows, ar, tag);
        // the wavefronts' partial sums: r.r, (A r).r and the stopping norm
        double part[3] = {0.0, 0.0, 0.0};
        if (live) {
            const double r2 = (double) r * (double) r;
            part[0] += (double) r * (double) r;
            part[1] += (double) ar * (double) r;
            part[2] += kWeighted ? dg * r2 : r2;
        }
        const double ws = wave_sum3(part[0], part[1], part[2]);
        const int k3 = sum3_of_lane(lane);
        if (kByWave) {
            send_sums(xp + (mine + wid) * kSumWords, ws, tag);
        } else {
            if (k3 >= 0) s_wave[k3][wid] = ws;
            __syncthreads();
        }
        double sum[3];
        unsigned long long hm[kResHalo][kWords<T>];
        if (alone) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                double t = 0.0;
#pragma unroll
                for (int q = 0; q < NW; q++) t += s_wave[k][q];
                sum[k] = t;
            }
        } else {
            if (!kByWave && tid < 6) {
                double t = 0.0;
#pragma unroll
                for (int q = 0; q < NW; q++) t += s_wave[tid >> 1][q];
                put_word(xp + mine * kSumWords + tid, (unsigned) (tid & 1 ? __double2hiint(t) : __double2loint(t)), tag);
            }
            // wait for the sums and for A r of the thread's halo rows
            bool bad = false;
            unsigned long long m[kPoll];
            const bool sums = (tid & (kSumWords - 1)) < 6;
            {
                Wait wt;
                for (;;) {
                    bool ok = true;
#pragma unroll
                    for (int i = 0; i < kPoll; i++)
                        if (sums && i * BT + tid < nsum * kSumWords)
                            m[i] = get_word_at(xp + sum0 * kSumWords + (size_t) i * BT, (unsigned) tid * 8u);
#pragma unroll
                    for (int i = 0; i < kResHalo; i++)
                        if (i * BT < H && hc[i] >= 0) {
#pragma unroll
                            for (int k = 0; k < kWords<T>; k++)
                                hm[i][k] = get_word_at(xw + (size_t) k * X.w_rows, (unsigned) hc[i] * 8u);
                        }
#pragma unroll
                    for (int i = 0; i < kPoll; i++)
                        if (sums && i * BT + tid < nsum * kSumWords) {
                            ok = ok && tag_of(m[i]) == tag;
                            bad = bad || tag_of(m[i]) == poison;
                        }
#pragma unroll
                    for (int i = 0; i < kResHalo; i++)
                        if (i * BT < H && hc[i] >= 0) {
#pragma unroll
                            for (int k = 0; k < kWords<T>; k++) ok = ok && tag_of(hm[i][k]) == tag;
                        }
                    if (ok) break;
                    bad = bad || wt.expired();
                    if (bad) break;
                }
            }
#pragma unroll
            for (int i = 0; i < kPoll; i++) {
                const int at = i * BT + tid;
                if (sums && at < nsum * kSumWords) s_sum[at / kSumWords * 6 + at % kSumWords] = (unsigned) m[i];
            }
            if (bad) s_bad = 1;
            __syncthreads();
            // every wavefront adds them up: lane 0, 32, 16 of total hold the
            // segment's three sums
            const double* const ss = (const double*) s_sum;
            double total;
            if (kByWave) {
                // lanes 16 k + b: sum k of block b, then the blocks (16 at
                // most, so the tree's upper levels add zeros)
                static_assert(kResSplitSums <= 16 * kResWaves, "a row of lanes holds the blocks");
                const int k = lane < 16 ? 0 : (lane < 32 ? 2 : (lane < 48 ? 1 : 3));
                const int b = lane & 15;
                total = 0.0;
                if (k < 3 && b < nb) {
#pragma unroll
                    for (int q = 0; q < kResWaves; q++) total += ss[(b * kResWaves + q) * 3 + k];
                }
                total += 0.0;
                total += dpp_f64<0x108>(total);
                total += dpp_f64<0x104>(total);
                total += dpp_f64<0x102>(total);
                total += dpp_f64<0x101>(total);
            } else {
                total = 0.0;
                for (int q = 0; q < nb; q += 64) {  // the blocks of one wavefront of k_cg_step's reduction
                    const bool in = q + lane < nb;
                    const double* const c3 = ss + (q + lane) * 3;
                    total += wave_sum3(in ? c3[0] : 0.0, in ? c3[1] : 0.0, in ? c3[2] : 0.0);
                }
            }
            if (s_bad) {
                leave();
                return;
            }
            auto from = [&](int l) {
                return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(total), l),
                                        __builtin_amdgcn_readlane(__double2loint(total), l));
            };
            sum[0] = from(0);
            sum[1] = from(32);
            sum[2] = from(16);
        }
        const double g = sum[0], dd = sum[1], rho = sum[2];
        const bool first = it == 1;
        const bool conv = rho <= thr;
        if (conv || it > max_iter || !(rho == rho)) {
            if (live) y_io[row] = y;
            if (br.v == 0 && blockIdx.x % kSplit == 0 && tid == 0) {
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
            if (i * BT >= H || hc[i] < 0) continue;  // the first test is uniform
            T* const xh = x + BT + i * BT + tid;
            const T hw = value_of<T>(hm[i]);
            hs[i] = first ? hw : hw + beta * hs[i];
            *xh = *xh - alpha * hs[i];
        }
        __syncthreads();
    }
}

constexpr int kSplitThreads = kCgBlock / kResSplit;

static size_t resident_lds(int max_rows, int threads, int tsize) {
    const size_t words = (size_t) (max_rows + 31) / 32;
    return (size_t) tsize * (threads + kResHalo * threads) + words * 4 + ((words * 2 + 15) & ~(size_t) 15);
}

// Entries held in registers: 16 covers a 2D system at 2.1 l0 (12-14 a row),
// 36 one at 3.1 l0 (28-34) and 3D at 2.1 l0 (32-36); a wider row reads the
// rest from memory every iteration.
constexpr int kResFew = 16, kResMany = 36;

ResidentShape resident_shape(int max_rows, int max_nb, int total_blocks, int mean_width, int most, int tsize) {
    ResidentShape s{};
    if (max_rows > kResMaxRows || max_nb > kResMaxBlocks || total_blocks > most) return s;
    // Systems of few blocks leave the chip idle: four workgroups a block cut
    // the row products' LDS reads per CU.  A block alone needs no exchange
    // and stays whole; beyond 16 blocks the wavefronts' sums are more than
    // the threads of a split workgroup can wait for.
    s.split = max_nb > 1 && max_nb * kResWaves <= kResSplitSums && kResSplit * total_blocks <= most ? kResSplit : 1;
    s.emax = mean_width <= kResFew ? kResFew : kResMany;
    s.lds = resident_lds(max_rows, kCgBlock / s.split, tsize);
    return s;
}

size_t resident_sums(int total_blocks) { return (size_t) kResWaves * total_blocks; }
size_t resident_sum_words(size_t p_sums) { return 2 * (size_t) kSumWords * p_sums; }

template <typename T, typename IDX>
static const void* resident_kernel(const ResidentShape& s) {
    if (s.split > 1)
        return s.emax == kResFew ? (const void*) k_cg_resident<T, IDX, kResFew, kSplitThreads>
                                 : (const void*) k_cg_resident<T, IDX, kResMany, kSplitThreads>;
    return s.emax == kResFew ? (const void*) k_cg_resident<T, IDX, kResFew, kCgBlock>
                             : (const void*) k_cg_resident<T, IDX, kResMany, kCgBlock>;
}

template <typename T, typename IDX>
hipError_t resident_prepare(const ResidentShape& s) {
    return hipFuncSetAttribute(resident_kernel<T, IDX>(s), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int) resident_lds(kResMaxRows, kCgBlock / s.split, (int) sizeof(T)));
}

template <typename T, typename IDX>
hipError_t resident_launch(const ResidentShape& s, const Seg& sg, int total_blocks, const int* slice_off,
                           const IDX* col, const int* anc, const T* val, const T* r, T* y, const double* dgl,
                           CgScalars* sc, const CgExchange& x, hipStream_t st) {
    Seg a0 = sg;
    CgExchange a9 = x;
    void* args[] = {&a0, &slice_off, &col, &anc, &val, &r, &y, &dgl, &sc, &a9};
    return hipLaunchKernel(resident_kernel<T, IDX>(s), dim3(s.split * total_blocks), dim3(kCgBlock / s.split), args,
                           s.lds, st);
}

#define RESIDENT_INST(T, IDX)                                                                                      \
    template hipError_t resident_prepare<T, IDX>(const ResidentShape&);                                            \
    template hipError_t resident_launch<T, IDX>(const ResidentShape&, const Seg&, int, const int*, const IDX*,     \
                                                const int*, const T*, const T*, T*, const double*, CgScalars*,     \
                                                const CgExchange&, hipStream_t);
RESIDENT_INST(double, short)
RESIDENT_INST(double, unsigned short)
RESIDENT_INST(double, int)
RESIDENT_INST(float, short)
RESIDENT_INST(float, unsigned short)
RESIDENT_INST(float, int)
#undef RESIDENT_INST

}  // namespace mps
