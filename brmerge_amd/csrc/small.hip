// Short-row products in two launches and one host round trip.
//
// A product whose rows are all short (at most G = 64, or 32, lists and
// products) spends more on the general pipeline's dozen launches and two
// host round trips than on its kernels.  Such a product runs as:
//   1. one fill of the words through which the workgroups' places in C
//      are handed on;
//   2. k_small<G, P>: each workgroup takes a run of consecutive rows, in P
//      passes of one row per group of G lanes.  The passes are batched stage
//      by stage -- all row pointers, then all list descriptors, then all B
//      entries -- so that each dependent load is issued for every pass before
//      the first one is waited on.  Each group checks its rows' own indices,
//      finds the list offsets by a group scan (no global product scan) and
//      merges the row in registers with the short tier's code
//      (short_merge.h).  Every workgroup publishes its nnz, one wavefront of
//      the grid scans these as they come and publishes each workgroup's place,
//      and every row is written straight from registers into C, with C's row
//      pointer.  Workgroups past the row workgroups check all of B, a B row
//      per thread at a time (row pointers, column range, sorted rows), as the
//      general validation does.
// C is allocated beforehand for G entries per row, a bound of nnz(C) when
// every row is short.  The scanning wavefront writes the totals and flags to
// host memory, read once the stream has ended: a row with more than G lists or
// products, or a B row with more than 64 entries, sets a flag, and the product
// then goes through the general pipeline instead.
#include <limits.h>

#include <algorithm>

#include "brm_device.h"
#include "kernels.h"
#include "short_merge.h"

namespace brm {
namespace {

// One word per workgroup for what it adds (own) and, per row workgroup, one
// for what comes before it (pre).  The top bit marks a word as published; below
// it the flags (SMALL_BAD, SMALL_MISS), products (from bit SC_IP) and nnz(C).
// Each word carries its own value, so relaxed atomics (no cache invalidation
// or write-back) are enough.
constexpr int SC_IP = 28, SC_FLAGS = 2 * SC_IP;
constexpr uint64_t SC_SET = 1ull << 63, SC_LATE = 1ull << 62, SC_VAL = (1ull << SC_FLAGS) - 1ull;
static_assert((int64_t)SMALL_MAX_ROWS * BRM_WAVE < ((int64_t)1 << SC_IP), "two counts in a word");

__device__ __forceinline__ uint64_t sc_load(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sc_store(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The scanner (one wavefront, workgroup 0): reads the workgroups' own words
// in order as they appear and publishes each one's prefix.  A row workgroup
// then waits for one word.  (Decoupled look-back, every workgroup reading back
// to the nearest prefix, had the thousand resident workgroups poll the same
// cache lines past the L2 caches: with it A * P of a 27-point operator on 96^3
// points and an aggregation took 272 us, with the scanner 210, without any
// wait 180.)
// Workgroups start about in the order of their index, but nothing promises
// it, so both waits are bounded: after more looks without a new word of a row
// workgroup than an unpublished word says (the knob small_looks, which the host
// fills the words with) the scanner marks the rest late, and the product is left
// to the general pipeline.  (As an argument of the kernel the number makes the
// row workgroups of <64, 2> take 82 scalar registers instead of 80: one of them
// fits a CU then instead of two, and 16,384 rows of 64 products take 18.5 us
// instead of 14.3.)  The others' words come without any bound on the looks:
// these workgroups wait for nothing, and by then nobody waits for them.
// nrow words of row workgroups, then those of the others.
__device__ void scan_workgroups(const uint64_t* own, uint64_t* pre, int nrow, int n, SmallResult* res) {
    const int lane = lane_id();
    uint64_t sum = 0;
    unsigned flags = 0;
    int looks = 0;  // without a new word
    for (int base = 0; base < n;) {
        const uint64_t v = sc_load(&own[min(base + lane, n - 1)]);
        const uint64_t gap = __ballot((v & SC_SET) == 0 || base + lane >= n);
        const int got = gap ? __ffsll((long long)gap) - 1 : BRM_WAVE;  // words up to the first unpublished one
        if (got == 0) {
            if (base >= nrow || ++looks <= __builtin_amdgcn_readfirstlane((int)v)) continue;
            for (int q = base + lane; q < nrow; q += BRM_WAVE) sc_store(&pre[q], SC_SET | SC_LATE);
            flags |= SMALL_LATE;
            break;
        }
        looks = 0;
        const uint64_t mine = lane < got ? v & SC_VAL : 0;
        const unsigned f = lane < got ? (unsigned)(v >> SC_FLAGS) : 0u;
        if (__ballot(f & SMALL_BAD)) flags |= SMALL_BAD;
        if (__ballot(f & SMALL_MISS)) flags |= SMALL_MISS;
        const uint64_t inc = wave_incl_scan(mine);
        if (lane < got && base + lane < nrow) sc_store(&pre[base + lane], SC_SET | (sum + inc - mine));
        sum += wave_last(inc);
        base += got;
    }
    if (lane == 0) {
        res->nnz = (int64_t)(sum & ((1ull << SC_IP) - 1ull));
        res->ip = (int64_t)(sum >> SC_IP);
        res->flags = (int)flags;
        res->done = 1;
    }
}

// The flags of the workgroup's threads, in every thread (fl: one word per
// wavefront).
template <int NW>
__device__ unsigned block_flags(bool bad, bool miss, unsigned* fl) {
    const unsigned mine = (__ballot(bad) != 0ull ? SMALL_BAD : 0u) | (__ballot(miss) != 0ull ? SMALL_MISS : 0u);
    if (lane_id() == 0) fl[threadIdx.x / BRM_WAVE] = mine;
    __syncthreads();
    unsigned f = 0u;
#pragma unroll
    for (int i = 0; i < NW; ++i) f |= fl[i];
    return f;
}

// The prefix of workgroup b (called by one wavefront); 0 and *late when it
// does not come.
__device__ uint64_t await_prefix(const uint64_t* pre, int b, bool* late) {
    for (int looks = 0; looks < 4 * SMALL_LOOKS; ++looks) {
        const uint64_t v = sc_load(&pre[b]);
        if (v & SC_SET) {
            *late = (v & SC_LATE) != 0;
            return *late ? 0 : v & SC_VAL;
        }
        __builtin_amdgcn_s_sleep(2);
    }
    *late = true;
    return 0;
}

// Workgroup shape per group size: threads and passes.  A workgroup takes
// RPP * P consecutive rows (RPP rows per pass); wavefront 0 scans them, R per
// lane.
constexpr int SM_NT32 = 512;   // G = 32
constexpr int SM_NT64 = 1024;  // G = 64
constexpr int SM_P = 4;
// B rows longer than this are left to the general pipeline's validation.
constexpr int SM_BROW_MAX = 64;

template <int G, int P_>
struct SmallShape {
    static constexpr int NT = G == 32 ? SM_NT32 : SM_NT64;  // threads
    static constexpr int P = P_;                             // passes
    static constexpr int WPB = NT / BRM_WAVE;                // wavefronts
    static constexpr int RPW = BRM_WAVE / G;                 // rows per wavefront and pass
    static constexpr int RPP = WPB * RPW;                    // rows per pass
    static constexpr int ROWS = RPP * P;                     // rows per workgroup
    static constexpr int R = (ROWS + BRM_WAVE - 1) / BRM_WAVE;  // rows per lane of the scan
    static_assert(R * BRM_WAVE == ROWS || ROWS < BRM_WAVE, "row layout");
};

template <int G, int P>
__global__ __launch_bounds__((SmallShape<G, P>::NT)) void k_small(RowArgs a, int nnzA, int nnzB, int row_blocks,
                                                              int64_t* __restrict__ crpt, int* __restrict__ ccol,
                                                              double* __restrict__ cval, SmallResult* __restrict__ res,
                                                              uint64_t* __restrict__ own) {
    using S = SmallShape<G, P>;
    const int lane = lane_id();
    const int w = (int)(threadIdx.x / BRM_WAVE);
    const int words = (int)gridDim.x - 1;
    uint64_t* pre = own + words;
    if (blockIdx.x == 0) {
        if (w == 0) scan_workgroups(own, pre, row_blocks, words, res);
        return;
    }
    __shared__ unsigned fl[S::WPB];
    const int b = (int)blockIdx.x - 1;
    if (b >= row_blocks) {
        // ---- B: a row per thread at a time; entries 8 at a time (indices
        // clamped into the row, so that every load is in bounds)
        const int64_t step = (int64_t)(words - row_blocks) * S::NT;
        bool bad = false, lng = false;
        for (int64_t r = (int64_t)(b - row_blocks) * S::NT + threadIdx.x; r <= a.K; r += step) {
            if (r == a.K) {
                bad |= a.brpt[0] != 0 || a.brpt[a.K] != nnzB || a.arpt[0] != 0 || a.arpt[a.M] != nnzA;
                continue;
            }
            const int b0 = a.brpt[r], b1 = a.brpt[r + 1];
            if (b0 < 0 || b0 > b1 || b1 > nnzB) {
                bad = true;
            } else if (b1 - b0 > SM_BROW_MAX) {
                lng = true;
            } else {
                int prev = -1;
                for (int k0 = b0; k0 < b1; k0 += 8) {
                    int c[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) c[j] = a.bcol[min(k0 + j, b1 - 1)];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        if (k0 + j < b1) {
                            bad |= c[j] <= prev || c[j] >= a.N;
                            prev = c[j];
                        }
                    }
                }
            }
        }
        const unsigned f = block_flags<S::WPB>(bad, lng, fl);
        if (threadIdx.x == 0) sc_store(&own[b], SC_SET | (uint64_t)f << SC_FLAGS);
        return;
    }
    __shared__ int rcnt[S::ROWS];      // nnz of the workgroup's rows
    __shared__ int rip[S::ROWS];       // their products
    __shared__ int64_t rbase[S::ROWS];  // their C offsets
    __shared__ ListSlot slots[S::NT];
    const int gl = lane & (G - 1);
    const int gbase = lane & ~(G - 1);
    const uint64_t gmask = (~0ull >> (BRM_WAVE - G)) << gbase;
    const int slot = w * S::RPW + lane / G;  // the group's row within a pass
    bool bad = false, miss = false;
    // ---- stage 1: row pointers (all passes' loads first), checked before
    // they are followed; the checks use | and & so that no branch separates
    // one pass's loads from the next
    int a0[P], a1[P], L[P];
    bool ok[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int row = min(b * S::ROWS + p * S::RPP + slot, a.M - 1);
        a0[p] = a.arpt[row];
        a1[p] = a.arpt[row + 1];
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int row = b * S::ROWS + p * S::RPP + slot;
        const bool has = row < a.M;
        const bool rb = has & ((a0[p] < 0) | (a0[p] > a1[p]) | (a1[p] > nnzA));
        const bool ms = has & !rb & (a1[p] - a0[p] > G);
        bad |= rb;
        miss |= ms;
        ok[p] = has & !rb & !ms;
        L[p] = ok[p] ? a1[p] - a0[p] : 0;
    }
    // ---- stage 2: list descriptors (A column and value, B row bounds)
    int acl[P];
    double lav[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int idx = gl < L[p] ? a0[p] + gl : 0;  // nnz(A) >= 1
        acl[p] = a.acol[idx];
        lav[p] = a.aval[idx];
    }
    int lbst[P], lend[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const bool cok = (gl < L[p]) & (acl[p] >= 0) & (acl[p] < a.K);
        const int cc = cok ? acl[p] : 0;  // K >= 1
        lbst[p] = a.brpt[cc];
        lend[p] = a.brpt[cc + 1];
    }
    // ---- stage 3: list offsets, each lane's product, its B entry.  A list
    // that is malformed or longer than G counts as G + 1 entries: its row is
    // not merged, and the group's sum stays within int
    int pl[P], bcl[P], ipn[P];
    double pav[P], bvl[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const bool v = gl < L[p];
        const bool lbad = v & ((acl[p] < 0) | (acl[p] >= a.K) | (lbst[p] < 0) | (lbst[p] > lend[p]) |
                               (lend[p] > nnzB));
        bad |= lbad;
        const int bl = v ? (lbad ? G + 1 : min(lend[p] - lbst[p], G + 1)) : 0;
        const int incl = group_incl_scan<G>(bl);
        int ip = __builtin_amdgcn_readlane(incl, BRM_WAVE - 1);
        if (G < BRM_WAVE) ip = (int)of_half((uint32_t)__builtin_amdgcn_readlane(incl, G - 1), (uint32_t)ip, gbase);
        miss |= ip > G;
        ipn[p] = ip > G ? 0 : ip;
        const int off = incl - bl;
        const ListSlot ls = list_of<G>(&slots[w * BRM_WAVE], gl, gbase, (bl > 0) & (off < G), off, lbst[p], lav[p]);
        pl[p] = ls.q;
        pav[p] = ls.av;
        const int bi = gl < ipn[p] ? ls.rel + gl : 0;  // nnz(B) >= 1
        bcl[p] = a.bcol[bi];
        bvl[p] = a.bval[bi];
    }
    // ---- stage 4: the merges
    const bool narrow = short_keys_fit<G>(a.N);
    ShortMerged m[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const bool act = gl < ipn[p];
        m[p] = short_merge<true, G>(act ? bcl[p] : INT_MAX, pl[p], act ? fmul(pav[p], bvl[p]) : 0.0, act, ipn[p], gl,
                                    gbase, gmask, narrow);
        if (gl == 0) {
            rcnt[p * S::RPP + slot] = ipn[p] > 0 ? m[p].nout : 0;
            rip[p * S::RPP + slot] = ipn[p];
        }
    }
    const unsigned flags = block_flags<S::WPB>(bad, miss, fl);
    // ---- the workgroup's rows in C: a scan over its rows, behind the
    // workgroups before it; C's row pointer from wavefront 0
    if (w == 0) {
        int64_t local = 0, ips = 0;
#pragma unroll
        for (int j = 0; j < S::R; ++j) {
            if (lane * S::R + j >= S::ROWS) continue;
            local += rcnt[lane * S::R + j];
            ips += rip[lane * S::R + j];
        }
        const int64_t inc = wave_incl_scan(local);
        const int64_t agg = wave_last(inc);
        ips = wave_sum(ips);
        if (lane == 0)
            sc_store(&own[b], SC_SET | (uint64_t)flags << SC_FLAGS | (uint64_t)ips << SC_IP | (uint64_t)agg);
        bool late = false;
        const uint64_t before = await_prefix(pre, b, &late);
        const int64_t base = (int64_t)(before & ((1ull << SC_IP) - 1ull));
        int64_t off = base + inc - local;
#pragma unroll
        for (int j = 0; j < S::R; ++j) {
            const int k = lane * S::R + j;
            if (k >= S::ROWS) continue;
            const int row = b * S::ROWS + k;
            rbase[k] = off;
            if (row < a.M) crpt[row] = off;
            off += rcnt[k];
            if (row == a.M - 1) crpt[a.M] = off;
        }
        if (lane == 0 && late) res->late = 1;
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (ipn[p] > 0 && m[p].alive) {
            const int64_t cb = rbase[p * S::RPP + slot];
            ccol[cb + m[p].idx] = m[p].col;
            cval[cb + m[p].idx] = m[p].val;
        }
    }
}

template <int G, int P>
int64_t row_blocks_of(int M) {
    return ((int64_t)M + SmallShape<G, P>::ROWS - 1) / SmallShape<G, P>::ROWS;
}

// Workgroups for the K rows of B and the ends of the row pointers: SM_BMAX at
// most, each of which takes rows in turn, as the scanner looks at every one's
// word.  2,048 rows of 8 products, B of 2e7 rows of 2 entries: 326 us with
// a workgroup per 512 rows (the scanner alone goes through 39,063 words), now 110.
constexpr int SM_BMAX = 2048;
template <int G>
int64_t b_blocks_of(int K) {
    constexpr int NT = SmallShape<G, 1>::NT;
    return std::min(((int64_t)K + 1 + NT - 1) / NT, (int64_t)SM_BMAX);
}

template <int G, int P>
hipError_t launch_small_gp(const RowArgs& a, int64_t nnzA, int64_t nnzB, int64_t* crpt, int* ccol, double* cval,
                           SmallResult* res, uint64_t* own, hipStream_t s) {
    using S = SmallShape<G, P>;
    const int64_t rb = row_blocks_of<G, P>(a.M);
    const int64_t bb = b_blocks_of<G>(a.K);
    if (1 + rb + bb > INT32_MAX || nnzA > INT32_MAX || nnzB > INT32_MAX) return hipErrorInvalidValue;
    ProfScope ps_("k_small", s);
    k_small<G, P><<<(unsigned)(1 + rb + bb), S::NT, 0, s>>>(a, (int)nnzA, (int)nnzB, (int)rb, crpt, ccol, cval, res, own);
    return hipGetLastError();
}

// Passes per workgroup: the fewest that leave at most SM_FEW workgroups (two
// per CU), else SM_P.  Few rows are a matter of latency, which passes add to;
// many workgroups a matter of handing the places on, 8 ns each.  k_small, us:
//   rows     products each | P = 1    2      4      8
//   2,048    64            | 7.3             10.6
//   16,384   64            | 19.9     15.5   17.6
//   884,736  27            |          327    210    247
constexpr int SM_FEW = 512;
template <int G>
int passes_of(int M) {
    return row_blocks_of<G, 1>(M) <= SM_FEW ? 1 : row_blocks_of<G, 2>(M) <= SM_FEW ? 2 : SM_P;
}

template <int G>
hipError_t launch_small_g(const RowArgs& a, int64_t nnzA, int64_t nnzB, int64_t* crpt, int* ccol, double* cval,
                          SmallResult* res, uint64_t* own, hipStream_t s) {
    switch (passes_of<G>(a.M)) {
        case 1: return launch_small_gp<G, 1>(a, nnzA, nnzB, crpt, ccol, cval, res, own, s);
        case 2: return launch_small_gp<G, 2>(a, nnzA, nnzB, crpt, ccol, cval, res, own, s);
        default: return launch_small_gp<G, SM_P>(a, nnzA, nnzB, crpt, ccol, cval, res, own, s);
    }
}

template <int G>
int64_t words_of(int M, int K) {
    const int p = passes_of<G>(M);
    const int64_t rb = p == 1 ? row_blocks_of<G, 1>(M) : p == 2 ? row_blocks_of<G, 2>(M) : row_blocks_of<G, SM_P>(M);
    return 2 * rb + b_blocks_of<G>(K);
}

}  // namespace

int64_t small_words(int M, int K, int group) { return group == 32 ? words_of<32>(M, K) : words_of<64>(M, K); }

hipError_t launch_small(const RowArgs& a, int64_t nnzA, int64_t nnzB, int64_t* crpt, int* ccol, double* cval,
                        SmallResult* res, uint64_t* words, int group, hipStream_t s) {
    if (a.M < 1 || a.K < 1 || nnzA < 1 || nnzB < 1) return hipErrorInvalidValue;
    hipError_t e = launch_fill_i64((int64_t*)words, small_words(a.M, a.K, group), params().small_looks, s);
    if (e != hipSuccess) return e;
    return group == 32 ? launch_small_g<32>(a, nnzA, nnzB, crpt, ccol, cval, res, words, s)
                       : launch_small_g<64>(a, nnzA, nnzB, crpt, ccol, cval, res, words, s);
}

}  // namespace brm
