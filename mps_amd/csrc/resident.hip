// resident.hip — the pressure solve of small and middle systems (start,
// Jacobi-scaled conjugate gradients, true residuals, restarts or refinements)
// as one launch.
//
// Run by launches, an iteration is two dependent kernels (k_cg_apply,
// k_cg_step): 8-11 us whatever the size up to some 30k rows, nearly all of it
// launch, block start-up and first loads, and every restart or refinement is
// five more launches and a host read.  Here every block of the same layout
// stays on its CU for the whole solve: one row a thread, the row's matrix
// entries (16 or 36, see resident_shape) and its p, s, y in registers, r of
// the block's rows and of the rows they couple to (the halo) in LDS.  512
// threads leave a thread 256 registers: whole blocks in FP64 spill 15 of them
// at 16 entries a row and some 100, 300 bytes a lane, at 36.  Even so 2D at
// 3.1 l0 takes 0.63 ms a step where the kernels take 0.94 (40k rows, 50
// iterations; the mixed kernel, which spills one at most, 0.57 and 1.05).  An
// iteration exchanges A r of the halo rows and each block's three partial sums
// once, and every block applies the update to its halo rows itself (s = A r +
// beta s, r -= alpha s), so one exchange an iteration is enough; a residual is
// one more, of r and its norm.
//
// The exchange is of tagged words: 32 bits of the value below a 32-bit tag,
// stored and polled as relaxed device-scope 64-bit atomics.  A word carries
// its own readiness, so it needs no flag, fence or counter after it, and one
// store-to-load latency is the whole exchange (1.4-1.5 us between 2 to 64
// workgroups spread over the 8 XCDs; on one XCD it is the same).  Two halves
// alternate: a block writes a half again only after it has every block's
// partials of the exchange between, which each block sends after it has read
// the half.  The exchange of y alone has no partials.  The one after it writes
// the half of the one before it, whose readers are the blocks that have a row
// of this block in their halo.  The matrix couples rows both ways (a pair is
// in range for both or for neither, and padding names its own row), so those
// are the blocks of this block's halo; they sent their y, which this block has
// by then, after they had read that half.
//
// Measured (2D, FP64, launches -> resident CG -> resident solve): 492 rows,
// ~60 iterations a step at machine epsilon 1.15 -> 0.78 -> 0.64 ms a step,
// export included; 2,520 rows of 28 entries, ~280 iterations 3.90 -> 1.28 ->
// 1.25 ms; 32k rows of 12, ~10,700 iterations of a gradient evaluation
// 112 -> 43.8 -> 43.2 ms.  What an iteration spends (2.4 GHz cycles, FP64, 64
// blocks): row product and wavefront sums 1700, exchange 3500 (one uncached
// store and load), adding the sums up 900, three divisions 700, updates 800.
//
// Sums are taken in the order and with the arithmetic of the two kernels, so
// the iterates are theirs bit for bit, and an ensemble member keeps its solo
// run's bits.
//
// Every block must be on a CU at once (the host launches no more than fit
// and counts the blocks in flight); a wait is bounded all the same: a block
// that waits too long, or whose halo does not fit, tells its segment through a
// poisoned tag and leaves, and the host then solves by launches.
#pragma clang fp contract(off)

#include <algorithm>
#include <cstring>

#include "cg_device.hpp"

namespace mps {

constexpr int kResHalo = 8;               // halo rows a thread updates
constexpr int kResMaxRows = 131072;       // rows of a segment (bits of the halo map)
constexpr int kResWaves = kCgBlock / 64;  // wavefronts of a block of the layout
constexpr int kResMaxBlocks = 256;        // blocks of a segment
constexpr int kResSplitSums = 128;        // wavefronts of a segment with split blocks
// Words of a place of partial sums: three doubles and two words of padding,
// so that a place has a 64-byte line to itself and is sent by one store of
// eight lanes.
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

// A uniform value the compiler may not compute with ahead of its use: the tests
// it would move out of the loops are more than the scalar registers hold.
__device__ __forceinline__ int at_use(int v) {
    v = __builtin_amdgcn_readfirstlane(v);
    asm volatile("" : "+s"(v));
    return v;
}

// The same for a value of every lane: a lane mask computed from it before is
// not kept for a later test.
__device__ __forceinline__ int at_use_v(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

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
// by eight lanes.
__device__ __forceinline__ void send_sums(unsigned long long* p, double ws, unsigned tag) {
    const int lane = threadIdx.x & 63;
    const int from = lane >> 1 == 1 ? 32 : (lane >> 1 == 2 ? 16 : 0);
    const int lo = __builtin_amdgcn_ds_bpermute(4 * from, __double2loint(ws));
    const int hi = __builtin_amdgcn_ds_bpermute(4 * from, __double2hiint(ws));
    if (lane < kSumWords) put_word(p + lane, (unsigned) (lane & 1 ? hi : lo), tag);
}
template <typename T>
__device__ __forceinline__ T value_of(const unsigned long long* w) {
    if constexpr (sizeof(T) == 8)
        return __longlong_as_double((long long) ((w[1] << 32) | (w[0] & 0xffffffffull)));
    else
        return __uint_as_float((unsigned) w[0]);
}

// acc + sum of val[k] * x[idx[k]] in entry order, each product and sum
// rounded by itself as sell_row does (contraction is off here).
template <typename T>
__device__ __forceinline__ T add_product(T acc, T v, T x) {
    acc += v * x;
    return acc;
}
template <typename T, int EMAX, typename X>
__device__ __forceinline__ T resident_row(const T (&v)[EMAX], const unsigned (&ix)[EMAX / 2], const X* x, T acc) {
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

// ---- the start and the FP64 residual, with k_cg_init's, k_residual64's and
// k_inner_init's arithmetic (no fused multiply-adds but where noted)

// The start of the solve at a row, scaled: 0, the previous solution or the
// line through the last two where both steps solved for this particle.
__device__ __forceinline__ double resident_start(const ResidentArgs& a, int row) {
    if (!a.pprev) return 0.0 / a.sdiag[row];
    const int id = a.id[a.row_slot[row]];
    const double p1 = a.pprev[id];
    double x0 = p1;
    if (a.pprev2) {
        const double p2 = a.pprev2[id];
        if (p1 != 0.0 && p2 != 0.0) x0 = 2.0 * p1 - p2;
    }
    return x0 / a.sdiag[row];
}
__device__ __forceinline__ double times(double a, double b) { return a * b; }
__device__ __forceinline__ double minus(double a, double b) { return a - b; }

// What the workgroups of a launch are to each other (uniform values).
struct ResidentPeers {
    unsigned long long* w;
    unsigned long long* part;
    unsigned w_rows, p_sums;
    unsigned tag0, poison;
    unsigned nval, nsum;  // exchanges of values and of sums so far
    int nb;               // blocks of the segment
    int sums;             // places of sums to wait for
    unsigned sum0, mine;  // the segment's first place, this workgroup's first
    int H;                // halo rows
};

template <int BT>
struct ResidentSize {
    static constexpr int waves = BT / 64;
    static constexpr int split = kCgBlock / BT;
    static constexpr bool by_wave = split > 1;
    static constexpr int halo_rows = kResHalo * BT;
    // sums sent per workgroup: its block's, or its wavefronts'; and the most
    // a workgroup waits for
    static constexpr int sent = by_wave ? waves : 1;
    static constexpr int max_sums = by_wave ? kResSplitSums : kResMaxBlocks;
    static constexpr int poll = max_sums * kSumWords / BT;  // words of them a thread polls
};

template <int BT>
struct ResidentLds {
    unsigned sum[ResidentSize<BT>::max_sums * kSumWords];  // all sums as they are sent
    double wave[3][ResidentSize<BT>::waves];
    int scan[ResidentSize<BT>::waves];
    int bad;
};

// One exchange.  VALS: sends the thread's row value `own` and receives those
// of its halo rows (hc) in `got`.  SUMS: adds `part` up over the segment.
// Every thread of every workgroup of the segment calls it; false (uniform in
// the workgroup) once a wait has failed.
template <typename V, bool VALS, bool SUMS, int BT>
__device__ __forceinline__ bool resident_exchange(ResidentPeers& P, ResidentLds<BT>& L, bool alone, int row, bool live,
                                                  V own, const int (&hc)[kResHalo], V (&got)[kResHalo],
                                                  const double (&part)[3], double (&sum)[3]) {
    using S = ResidentSize<BT>;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const unsigned vtag = P.tag0 + 2u * P.nval + 2u, stag = P.tag0 + 2u * P.nsum + 1u;
    unsigned long long* const xw = P.w + (size_t) ((P.nval & 1u) * 2u * P.w_rows);
    unsigned long long* const xp = P.part + (size_t) ((P.nsum & 1u) * kSumWords * P.p_sums);
    if (VALS) P.nval++;
    if (SUMS) P.nsum++;
    if (VALS && live && !alone) put_value<V>(xw + row, P.w_rows, own, vtag);
    if (SUMS) {
        const double ws = wave_sum3(part[0], part[1], part[2]);
        if (S::by_wave) {
            send_sums(xp + (P.mine + wid) * kSumWords, ws, stag);
        } else {
            const int k3 = sum3_of_lane(lane);
            if (k3 >= 0) L.wave[k3][wid] = ws;
            __syncthreads();
            if (alone) {
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    double t = 0.0;
#pragma unroll
                    for (int q = 0; q < S::waves; q++) t += L.wave[k][q];
                    sum[k] = t;
                }
                return true;
            }
            if (tid < kSumWords) {
                double t = 0.0;
#pragma unroll
                for (int q = 0; q < S::waves; q++) t += L.wave[tid < 6 ? tid >> 1 : 0][q];
                put_word(xp + P.mine * kSumWords + tid, (unsigned) (tid & 1 ? __double2hiint(t) : __double2loint(t)),
                         stag);
            }
        }
    }
    if (alone) return true;
    // No lane is masked off (a mask is two scalar registers, and there are not
    // enough for all of them): a lane past the end of the sums polls a word of
    // the first place again, one past the halo its own row.
    bool bad = false;
    unsigned long long m[S::poll], hm[kResHalo][kWords<V>];
    unsigned at[S::poll];  // word of the sums
    if (SUMS) {
        const int nw = at_use(P.sums) * kSumWords;
#pragma unroll
        for (int i = 0; i < S::poll; i++) {
            const unsigned q = (unsigned) (i * BT + tid);
            at[i] = q < (unsigned) nw ? q : (unsigned) tid & (kSumWords - 1);
        }
    }
    // A poll that samples memory just before the others' words arrive costs
    // a whole round trip more, so the first one waits some 1000 cycles (one
    // trip down): 2,520 rows 24.3 -> 23.4 ms per 20 steps, 32k rows 42.8 ->
    // 40.9 ms an evaluation; 640 cycles give half of it, 1500 lose it again.
    __builtin_amdgcn_s_sleep(16);
    BoundedWait wt;
    for (;;) {
        if (SUMS) {
#pragma unroll
            for (int i = 0; i < S::poll; i++)
                if (i * BT < at_use(P.sums) * kSumWords) m[i] = get_word_at(xp + P.sum0 * kSumWords, at[i] * 8u);
        }
        if (VALS) {
#pragma unroll
            for (int i = 0; i < kResHalo; i++)
                if (i * BT < at_use(P.H)) {
#pragma unroll
                    for (int k = 0; k < kWords<V>; k++)
                        hm[i][k] = get_word_at(xw + k * P.w_rows, (unsigned) hc[i] * 8u);
                }
        }
        unsigned off = 0;  // zero when every tag is there
        if (SUMS) {
#pragma unroll
            for (int i = 0; i < S::poll; i++)
                if (i * BT < at_use(P.sums) * kSumWords) {
                    off |= tag_of(m[i]) ^ stag;
                    bad = bad || tag_of(m[i]) == P.poison;
                }
        }
        if (VALS) {
#pragma unroll
            for (int i = 0; i < kResHalo; i++)
                if (i * BT < at_use(P.H)) {
#pragma unroll
                    for (int k = 0; k < kWords<V>; k++) off |= tag_of(hm[i][k]) ^ vtag;
                }
        }
        if (off == 0) break;
        bad = bad || wt.expired();
        if (bad) break;
    }
    if (VALS) {
#pragma unroll
        for (int i = 0; i < kResHalo; i++)
            if (i * BT < at_use(P.H)) got[i] = value_of<V>(hm[i]);
    }
    if (SUMS) {
#pragma unroll
        for (int i = 0; i < S::poll; i++)
            if (i * BT < at_use(P.sums) * kSumWords) L.sum[at[i]] = (unsigned) m[i];
    }
    if (bad) L.bad = 1;
    __syncthreads();
    if (SUMS) {
        // every wavefront adds them up: lane 0, 32, 16 of total hold the
        // segment's three sums
        const double* const ss = (const double*) L.sum;
        double total = 0.0;
        if (S::by_wave) {
            // lanes 16 k + b: sum k of block b (in k_cg_apply's order), then
            // the blocks (16 at most, so the tree's upper levels add zeros)
            static_assert(kResSplitSums <= 16 * kResWaves, "a row of lanes holds the blocks");
            const int k = lane < 16 ? 0 : (lane < 32 ? 2 : (lane < 48 ? 1 : 3));
            const int b = lane & 15;
            if (k < 3 && b < P.nb) {
#pragma unroll
                for (int q = 0; q < kResWaves; q++) total += ss[(b * kResWaves + q) * (kSumWords / 2) + k];
            }
            total += 0.0;
            total += dpp_f64<0x108>(total);
            total += dpp_f64<0x104>(total);
            total += dpp_f64<0x102>(total);
            total += dpp_f64<0x101>(total);
        } else {
            for (int q = 0; q < P.nb; q += 64) {  // the blocks of one wavefront of k_cg_step's reduction
                const bool in = q + lane < P.nb;
                const double* const c3 = ss + (q + lane) * (kSumWords / 2);
                total += wave_sum3(in ? c3[0] : 0.0, in ? c3[1] : 0.0, in ? c3[2] : 0.0);
            }
        }
        auto from = [&](int l) {
            return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(total), l),
                                    __builtin_amdgcn_readlane(__double2loint(total), l));
        };
        sum[0] = from(0);
        sum[1] = from(32);
        sum[2] = from(16);
    }
    return !L.bad;
}

// BT rows a workgroup.  BT == kCgBlock: one workgroup a block of the layout;
// it sends the block's three sums, and every workgroup adds the blocks' sums
// up as k_cg_step does.  BT < kCgBlock: kCgBlock / BT workgroups a block, each
// wavefront sends its own sums, and every workgroup adds them up to the
// blocks' sums first, in k_cg_apply's order.
//
// Every thread sends its own row and polls right after.  A wavefront's loads
// and stores complete in order, so its first poll also waits for its stores'
// acknowledgement; a load that bypasses the L2s takes as long anyway (2500
// cycles) and mostly finds the others' words in that time.  Separate sending
// and polling wavefronts were slower (2,520 rows 26.1 -> 30.5 ms per 20
// steps): the poll sampled memory too early and had to be repeated.
template <typename T, typename IDX, int EMAX, int BT>
__global__ void __launch_bounds__(BT) k_solve_resident(ResidentArgs arg) {
#pragma clang fp contract(fast)
    static_assert(EMAX % 2 == 0, "two places share a word");
    using S = ResidentSize<BT>;
    constexpr bool kMixed = sizeof(T) == 4;
    constexpr int NW = S::waves;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ ResidentLds<BT> L;
    __shared__ ResidentIn in;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    // What only the start, the residuals and the end need is read from LDS
    // where it is used: the scalar registers do not hold all of it.
    __shared__ ResidentArgs A;
    static_assert(sizeof(ResidentArgs) % 4 == 0, "copied by words");
    for (int i = tid; i < (int) (sizeof(ResidentArgs) / 4); i += BT)
        ((unsigned*) &A)[i] = ((const unsigned*) &arg)[i];
    __syncthreads();
    const IDX* const col = (const IDX*) A.col;
    const T* const val = (const T*) A.val;
    BlockRows br = block_rows(arg.sg, blockIdx.x / S::split);
    const int base = arg.sg.row_off[br.seg];
    const int rows = arg.sg.row_off[br.seg + 1] - base;
    if (S::by_wave) {  // this workgroup's share of the block
        const int part = blockIdx.x % S::split;
        br.r0 = br.r0 + part * BT < br.r1 ? br.r0 + part * BT : br.r1;
        br.r1 = br.r0 + BT < br.r1 ? br.r0 + BT : br.r1;
    }
    const int own = br.r1 - br.r0;
    const bool alone = !S::by_wave && br.nb == 1;  // the segment is this workgroup's
    const int words = (rows + 31) >> 5;
    // gathered values: own rows, then the halo (FP64 residuals and starts use
    // the same places as doubles)
    typedef T __attribute__((may_alias)) TAlias;
    typedef double __attribute__((may_alias)) DAlias;
    TAlias* const x = (TAlias*) smem;
    DAlias* const xd = (DAlias*) smem;
    unsigned* const bits = (unsigned*) (smem + sizeof(double) * (BT + S::halo_rows));
    unsigned short* const pre = (unsigned short*) (bits + words);
    int* const hcol = (int*) x;  // while the halo is listed
    // the options come from host memory: one read of a few lanes a workgroup
    static_assert(sizeof(ResidentIn) % 4 == 0 && sizeof(ResidentIn) / 4 <= 64, "read by one wavefront");
    if (tid < (int) (sizeof(ResidentIn) / 4)) ((unsigned*) &in)[tid] = ((const volatile unsigned*) A.in)[tid];
    __syncthreads();
    const int max_it = in.max_iterations > 0 ? in.max_iterations : 2 * rows;
    ResidentPeers P;
    P.w = arg.X.w;
    P.part = arg.X.part;
    P.w_rows = (unsigned) arg.X.w_rows;
    P.p_sums = (unsigned) arg.X.p_sums;
    P.tag0 = in.tag0;
    P.poison = in.poison;
    P.nval = P.nsum = 0;
    P.nb = br.nb;
    P.sums = __builtin_amdgcn_readfirstlane(S::by_wave ? br.nb * kResWaves : br.nb);
    P.sum0 = (unsigned) br.b0 * (S::by_wave ? kResWaves : 1);
    P.mine = blockIdx.x * S::sent;
    const int row = br.r0 + tid;
    const bool live = tid < own;

    // ---- results
    __shared__ double s_bn2, s_start;  // ||b||^2 and the start's residual
    if (tid == 0) s_bn2 = s_start = 0.0;
    double rho2 = 0.0;
    int total_it = 0, rounds = 0;
    bool conv = false;
    // The last workgroup of the segment to leave writes the results: the host
    // reads them once every workgroup is done, or one of them has given up.
    auto leave = [&](bool gave_up) {  // every thread of the workgroup
        if (gave_up && !alone && tid < 2 * S::sent * kSumWords) {
            const int half = tid / (S::sent * kSumWords), at = tid % (S::sent * kSumWords);
            put_word(P.part + (size_t) (half * kSumWords * P.p_sums + P.mine * kSumWords + at), 0u, P.poison);
        }
        if (tid == 0) {
            // count: arrivals in the low half, of which gave up in the high
            const int add = 1 + (gave_up ? 1 << 16 : 0);
            const int was = __hip_atomic_fetch_add(&A.count[br.seg], add, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            const int now = was + add;
            if ((now & 0xffff) == br.nb * S::split) {
                __hip_atomic_store(&A.count[br.seg], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                volatile ResidentOut* const o = A.out + br.seg;
                o->bn2 = s_bn2;
                o->rho2_start = s_start;
                o->rho2 = rho2;
                o->iterations = total_it;
                o->rounds = rounds;
                o->converged = conv ? 1 : 0;
                o->bail = now >> 16 ? 1 : 0;
                __hip_atomic_store(&A.out[br.seg].seq, in.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    };

    // ---- the halo: the rows of the segment outside the workgroup's that
    // some entry names, numbered in row order
    for (int i = tid; i < words; i += BT) bits[i] = 0;
    if (tid == 0) L.bad = 0;
    int w = 0, lo = 0, hi = 0;
    size_t eb = 0;
    if (live) {
        const int sl = row >> 6;
        const int s0 = A.slice_pos[sl];
        w = A.slice_pos[sl + 1] - s0;
        eb = (size_t) s0 * 64 + (row & 63);
        sell_anchors<IDX>(A.anc, row, lo, hi);
    }
    // entries past the row's: own row, value 0, by bit masks for the same
    // reason as in the exchange
    int c[EMAX];
#pragma unroll
    for (int k = 0; k < EMAX; k++) c[k] = row;
    if (w > 0) {
#pragma unroll
        for (int k = 0; k < EMAX; k++) {
            const int n = at_use_v(w), q = k < n ? k : n - 1, in_row = (k - n) >> 31;  // all ones inside the row
            c[k] = (sell_col<IDX>(col, eb + (size_t) q * 64, row, lo, hi) & in_row) | (row & ~in_row);
        }
    }
    __syncthreads();
    auto mark = [&](int cc) {
        if (cc < br.r0 || cc >= br.r1) atomicOr(&bits[(cc - base) >> 5], 1u << ((cc - base) & 31));
    };
    if (live) {
#pragma unroll
        for (int k = 0; k < EMAX; k++) mark(c[k]);
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
    if (lane == 63) L.scan[wid] = inc;
    __syncthreads();
    int off = inc - cnt, H = 0;
    for (int k = 0; k < NW; k++) {
        if (k < wid) off += L.scan[k];
        H += L.scan[k];
    }
    H = __builtin_amdgcn_readfirstlane(H);
    P.H = H;
    if (H > S::halo_rows || H > arg.X.halo_max) {  // uniform in the workgroup
        leave(true);
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
#pragma unroll
    for (int i = 0; i < kResHalo; i++) {
        const int h = i * BT + tid;
        hc[i] = h < H ? hcol[h] : (live ? row : br.r0);  // past the halo: a row of the workgroup
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
#pragma unroll
    for (int k = 0; k < EMAX; k += 2) {
        const unsigned a = live ? place(at_use_v(c[k])) : (unsigned) tid;
        const unsigned b = live ? place(at_use_v(c[k + 1])) : (unsigned) tid;
        ix[k / 2] = a | (b << 16);
    }
#pragma unroll
    for (int k = 0; k < EMAX; k++) v[k] = (T) 0;
    if (w > 0) {
#pragma unroll
        for (int k = 0; k < EMAX; k++) {
            const int n = at_use_v(w), q = k < n ? k : n - 1;
            const T one = val[eb + (size_t) q * 64];
            v[k] = k < n ? one : (T) 0;
        }
    }
    // A times the gathered values, own value `mid` (unit diagonal)
    auto row_product = [&](T mid) {
        T acc = resident_row<T, EMAX>(v, ix, x, mid);
        for (int k = EMAX; k < w; k++) {
            const size_t e = eb + (size_t) k * 64;
            acc = add_product(acc, val[e], x[place(sell_col<IDX>(col, e, row, lo, hi))]);
        }
        return acc;
    };
    auto row_product64 = [&](double mid) {
        if constexpr (!kMixed) {
            return row_product(mid);
        } else {  // the FP64 matrix, once a refinement, from memory
            double acc = mid;
            for (int k = 0; k < w; k++) {
                const size_t e = eb + (size_t) k * 64;
                acc = add_product(acc, A.val64[e], xd[place(sell_col<IDX>(col, e, row, lo, hi))]);
            }
            return acc;
        }
    };

    // ---- start: y = x0 / s, bhat = s b, ||b||^2
    double y = 0.0, dg = 0.0;
    double part[3] = {0.0, 0.0, 0.0}, sum[3];
    if (live) {
        const double b = A.b[A.row_slot[row]];
        dg = A.dgl[row];
        y = resident_start(A, row);
        part[0] += times(b, b);
    }
    T tnone[kResHalo] = {};
    if (!resident_exchange<T, false, true, BT>(P, L, alone, row, live, (T) 0, hc, tnone, part, sum)) {
        leave(true);
        return;
    }
    const double bn2 = sum[0], thr = in.tol2 * bn2;
    if (tid == 0) s_bn2 = bn2;
    if (bn2 == 0.0) y = 0.0;  // Eigen: a zero right-hand side gives x = 0
    xd[tid] = y;
#pragma unroll
    for (int i = 0; i < kResHalo; i++)
        if (i * BT < at_use(H)) xd[BT + i * BT + tid] = bn2 == 0.0 ? 0.0 : resident_start(A, hc[i]);
    __syncthreads();

    // ---- solves and true residuals
    T r = (T) 0;
    T hr[kResHalo];  // received r, A r or y of the halo rows
    bool stalled = false;
    for (int pass = 0;; pass++) {
        // FP64 residual of y (gathered in xd); r of the CG to the halo rows
        part[0] = part[1] = part[2] = 0.0;
        r = (T) 0;
        if (live) {
            const double acc = row_product64(y);
            const double r64 = minus(times(A.b[A.row_slot[row]], A.sdiag[row]), acc);
            r = (T) r64;
            part[0] += dg * (r64 * r64);
            part[1] += (double) r * (double) r;
        }
        if (!resident_exchange<T, true, true, BT>(P, L, alone, row, live, r, hc, hr, part, sum)) {
            leave(true);
            return;
        }
        const double before = rho2;
        rho2 = sum[0];
        conv = s_bn2 == 0.0 || rho2 <= thr;
        int inner_max = max_it - total_it;
        double inner_thr = thr;
        if (pass == 0) {
            if (tid == 0) s_start = rho2;
        } else if (!kMixed) {
            rounds += pass > 1;
            stalled = pass > 1 && !(rho2 <= 0.25 * before);
        } else {
            rounds++;
        }
        if (conv || stalled || total_it >= max_it || (kMixed ? rounds >= in.max_refinements : pass > in.max_refinements)) break;
        bool skip = false;
        if (kMixed) {
            // reduce the inner residual by eta, or by what the outer loop
            // still needs when that is less
            double red2 = in.eta2;
            const double need = thr / rho2;
            if (need > red2) red2 = need * 0.25;
            inner_thr = sum[1] * red2;
            skip = !(sum[1] > 0.0);
        }
        // gather places hold r (xd's readers are past the exchange's barrier)
        x[tid] = r;
#pragma unroll
        for (int i = 0; i < kResHalo; i++)
            if (i * BT < at_use(H)) x[BT + i * BT + tid] = hr[i];
        __syncthreads();
        // CG from r; e: the correction (mixed), else y itself
        T p = (T) 0, s = (T) 0, e = kMixed ? (T) 0 : (T) y;
        T hs[kResHalo] = {};
        double gam_old = 0.0, alp_old = 0.0;
        int it = 1;
        for (; !skip; it++) {
            // A r of the own row, and the sums r.r, (A r).r and the stopping norm
            const T ar = row_product(r);
            part[0] = part[1] = part[2] = 0.0;
            if (live) {
                const double r2 = (double) r * (double) r;
                part[0] += (double) r * (double) r;
                part[1] += (double) ar * (double) r;
                part[2] += kMixed ? r2 : dg * r2;
            }
            if (!resident_exchange<T, true, true, BT>(P, L, alone, row, live, ar, hc, hr, part, sum)) {
                leave(true);
                return;
            }
            const double g = sum[0], dd = sum[1], rho = sum[2];
            const bool first = it == 1;
            if (rho <= inner_thr || it > inner_max || !(rho == rho)) break;
            const double b = first ? 0.0 : g / gam_old;
            const double a = first ? g / dd : g / (dd - b * g / alp_old);
            gam_old = g;
            alp_old = a;
            const T alpha = (T) a, beta = (T) b;
            p = first ? r : r + beta * p;
            s = first ? ar : ar + beta * s;
            e = e + alpha * p;
            r = r - alpha * s;
            x[tid] = r;
#pragma unroll
            for (int i = 0; i < kResHalo; i++) {
                if (i * BT >= at_use(H)) continue;
                TAlias* const xh = x + BT + i * BT + tid;
                hs[i] = first ? hr[i] : hr[i] + beta * hs[i];
                *xh = *xh - alpha * hs[i];
            }
            __syncthreads();
        }
        total_it += skip ? 0 : it - 1;
        if (kMixed)
            y = y + (double) e;
        else
            y = (double) e;
        // y of the halo rows for the residual
        double hy[kResHalo];
        if (!resident_exchange<double, true, false, BT>(P, L, alone, row, live, y, hc, hy, part, sum)) {
            leave(true);
            return;
        }
        __syncthreads();  // every row product of the CG is done with x
        xd[tid] = y;
#pragma unroll
        for (int i = 0; i < kResHalo; i++)
            if (i * BT < at_use(H)) xd[BT + i * BT + tid] = hy[i];
        __syncthreads();
    }
    if (live) A.x[A.row_slot[row]] = times(y, A.sdiag[row]);
    __threadfence();  // x before the count
    __syncthreads();
    leave(false);
}

constexpr int kSplitThreads = kCgBlock / kResSplit;

static size_t resident_lds(int max_rows, int threads) {
    const size_t words = (size_t) (max_rows + 31) / 32;
    return sizeof(double) * threads * (1 + kResHalo) + words * 4 + ((words * 2 + 15) & ~(size_t) 15);
}

// Entries held in registers: 16 covers a 2D system at 2.1 l0 (12-14 a row),
// 36 one at 3.1 l0 (28-34) and 3D at 2.1 l0 (32-36); a wider row reads the
// rest from memory every iteration, one entry after the other, with its place
// looked up anew.  That pays up to some width and, where less than half of a row
// is held, while the L2s (4 MB an XCD) keep what is read again; beyond, the
// kernels win, which gather by fours with more wavefronts.  The FP64 kernel's
// spilled registers want their part of the L2s; in 3D the columns' anchors make
// what is read again dearer.  Measured, ms a step by kernels / resident, 25-45
// iterations a solve, graphs captured before:
//   entries a row          FP64                             mixed
//   2D  48   124k rows     1.27 / 1.12                      1.32 / 0.98
//       68   59k           1.30 / 1.33                      1.27 / 1.13
//       68   124k          1.57 / 1.57                      1.56 / 1.51
//       88                 32k 1.23 / 1.20, 39k 1.29 / 1.46   62k 1.51 / 1.36, 89k 1.61 / 1.70
//       97   20k           1.24 / 1.23                      1.36 / 1.35
//       103  12k           1.34 / 1.36                      1.40 / 1.42
//       119  9k            1.35 / 1.45                      1.46 / 1.55
//       158  12k           1.60 / 1.88                      1.73 / 2.11
//       119  714, split    1.04 / 1.07                      1.15 / 1.23
//       119  7k, split     1.29 / 1.27                      1.40 / 1.40
//       209  7k, split     2.00 / 2.16                      2.11 / 2.38
//   3D  92   (2.9 l0)      20k 2.09 / 2.04, 32k 2.19 / 2.32   46k 2.31 / 2.25
//       95   (3.1 l0, 630) 1.34 / 1.51                      1.58 / 1.69
//       111  5k, split     2.11 / 2.05                      2.28 / 2.20
//       115                12k 2.20 / 2.29, 36k 2.71 / 3.45   36k 2.62 / 2.73
constexpr int kResFew = 16, kResMany = 36;
// the widest mean row; in 3D split blocks of kResWide3Rows rows take up to kResWide3
constexpr int kResWide = 93, kResWide3 = 144, kResWide3Rows = 4096;
constexpr double kResReread64 = 16.5e6, kResReread32 = 24e6;  // bytes read again an iteration

ResidentShape resident_shape(int dim, int max_rows, int max_nb, int total_rows, int total_blocks, int mean_width,
                             int entry_bytes, int most, bool mixed) {
    ResidentShape s;
    std::memset(&s, 0, sizeof s);  // compared as bytes
    if (max_rows > kResMaxRows || max_nb > kResMaxBlocks || total_blocks > most) return s;
    // Systems of few blocks leave the chip idle: four workgroups a block cut
    // the row products' LDS reads per CU.  A block alone needs no exchange
    // and stays whole; beyond 16 blocks the wavefronts' sums are more than
    // the threads of a split workgroup can wait for.
    s.split = max_nb > 1 && max_nb * kResWaves <= kResSplitSums && kResSplit * total_blocks <= most ? kResSplit : 1;
    s.emax = mean_width <= kResFew ? kResFew : kResMany;
    const double reread = (double) std::max(mean_width - s.emax, 0) * entry_bytes * total_rows;
    const int widest = dim == 3 && s.split > 1 && total_rows >= kResWide3Rows ? kResWide3 : kResWide;
    if (mean_width > widest ||
        (mean_width > 2 * s.emax && reread > (mixed ? kResReread32 : kResReread64))) {
        s.split = 0;
        return s;
    }
    s.lds = resident_lds(max_rows, kCgBlock / s.split);
    return s;
}

// Every exchange takes one value tag and one sums tag (odd and even); a solve
// makes one for ||b||^2, one a residual, one an iteration, one that sees the
// stop of each CG and one for the new iterate.
long long resident_tags(long long max_iterations, int max_rounds) {
    return 2 * (max_iterations + 4ll * (max_rounds + 2)) + 16;
}

size_t resident_sums(int total_blocks) { return (size_t) kResWaves * total_blocks; }
size_t resident_sum_words(size_t p_sums) { return 2 * (size_t) kSumWords * p_sums; }

template <typename T, typename IDX>
static const void* resident_kernel(const ResidentShape& s) {
    if (s.split > 1)
        return s.emax == kResFew ? (const void*) k_solve_resident<T, IDX, kResFew, kSplitThreads>
                                 : (const void*) k_solve_resident<T, IDX, kResMany, kSplitThreads>;
    return s.emax == kResFew ? (const void*) k_solve_resident<T, IDX, kResFew, kCgBlock>
                             : (const void*) k_solve_resident<T, IDX, kResMany, kCgBlock>;
}

template <typename T, typename IDX>
hipError_t resident_prepare(const ResidentShape& s) {
    return hipFuncSetAttribute(resident_kernel<T, IDX>(s), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int) resident_lds(kResMaxRows, kCgBlock / s.split));
}

template <typename T, typename IDX>
hipError_t resident_launch(const ResidentShape& s, int grid, const ResidentArgs& a, hipStream_t st) {
    ResidentArgs arg = a;
    void* args[] = {&arg};
    return hipLaunchKernel(resident_kernel<T, IDX>(s), dim3(grid), dim3(kCgBlock / s.split), args, s.lds, st);
}

#define RESIDENT_INST(T, IDX)                                        \
    template hipError_t resident_prepare<T, IDX>(const ResidentShape&); \
    template hipError_t resident_launch<T, IDX>(const ResidentShape&, int, const ResidentArgs&, hipStream_t);
RESIDENT_INST(double, short)
RESIDENT_INST(double, unsigned short)
RESIDENT_INST(double, int)
RESIDENT_INST(float, short)
RESIDENT_INST(float, unsigned short)
RESIDENT_INST(float, int)
#undef RESIDENT_INST

}  // namespace mps
