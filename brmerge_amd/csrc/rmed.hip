// Register tier for small medium rows: one wavefront per row, the row's
// products held in registers (R per lane, ip <= 64 R <= 2048, at most 64
// lists; R = 32 only with bitmap ranks).
//
//   1. every lane l < L holds list l's product offset, B row start and A
//      value; the non-empty lists mark their first product in an LDS bitmap
//      and describe themselves in an LDS table, so each product finds its
//      list by a popcount rank and loads its B entry; value = a * b (rounded,
//      BRMerge-SpGEMM/inc/spgemm.h:621).
//   Sort variant (R <= 16): keys = (column, list position, index), 32-bit
//   when the column fits beside 6 bits of list position and log2(64 R) bits
//   of index (half the shuffles and compares), else 64-bit;
//   2. a bitonic sort over the 64 R keys (cross-lane steps with shuffles,
//      intra-lane steps between registers) orders the products by column,
//      and within a column by list position;
//   3. the sorted keys and the values go to LDS; the first product of every
//      column run sums its run as the aligned binary tree over list
//      positions does (siblings added left + right, a node with one present
//      child passes it through, spgemm.h:639-707) -- a single pass that
//      keeps one pending left subtree per height;
//   4. run heads are compacted with ballots and written to C (Precise), or
//      to C-bar with the row length (Upper).
//   Bitmap variant (R >= 4): popcount ranks over LDS bitmaps in levels of
//   64-way fan-out give each product its output position; products (still in
//   registers) are bucketed by position into the ranks' LDS, and each bucket
//   is folded in list-position order -- no sort.
// The symbolic count of these rows (k_rmed_count) uses the same list lookup
// and bitmaps.
#include <limits.h>

#include <algorithm>
#include <type_traits>

#include "brm_device.h"
#include "bucket_sum.h"
#include "kernels.h"

namespace brm {
namespace {

constexpr int RM_LOGL = 6;  // list positions < 64: six tree levels

__device__ __forceinline__ uint64_t shfl_xor_key(uint64_t x, int m) {
    const int lo = __shfl_xor((int)(uint32_t)x, m, BRM_WAVE);
    const int hi = __shfl_xor((int)(uint32_t)(x >> 32), m, BRM_WAVE);
    return ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
}
__device__ __forceinline__ uint32_t shfl_xor_key(uint32_t x, int m) {
    return (uint32_t)__shfl_xor((int)x, m, BRM_WAVE);
}

// Key layout: column | list position (LP_BITS) | product index (J_BITS).
template <int R, typename KT>
struct RmKey {
    static constexpr int J_BITS = sizeof(KT) == 8 ? 16 : (R == 2 ? 7 : R == 4 ? 8 : R == 8 ? 9 : 10);
    static constexpr int LP_BITS = sizeof(KT) == 8 ? 16 : 6;
    static constexpr int COL_SHIFT = J_BITS + LP_BITS;
    // Largest column a key holds.  A valid key is all ones only as the
    // last product (j = 64 R - 1) of a row of 64 R products, which has no
    // all-ones filler keys.
    static constexpr int64_t COL_MAX = sizeof(KT) == 8 ? INT32_MAX : ((int64_t)1 << (32 - COL_SHIFT)) - 1;
    __device__ static KT make(int col, int lp, int j) {
        return ((KT)(uint32_t)col << COL_SHIFT) | ((KT)lp << J_BITS) | (KT)j;
    }
    __device__ static uint32_t col(KT k) { return (uint32_t)(k >> COL_SHIFT); }
    __device__ static int lp(KT k) { return (int)((k >> J_BITS) & (((KT)1 << LP_BITS) - 1)); }
    __device__ static int j(KT k) { return (int)(k & (((KT)1 << J_BITS) - 1)); }
};

template <int R, typename KT>
struct RmSmem {
    double val[64 * R];  // first: the bitmap path's val is the same array
    KT key[64 * R];
};

// Stage 1: the row's non-empty lists, k-th at ent[k] (B row start less the
// list's first product, list position, A value); bit j of start is set when a
// non-empty list begins at product j + 1.  Overlays the start of each
// variant's LDS.
struct RmListEnt {
    int b;
    int lp;
    double sc;
};
struct RmLists {
    unsigned start[64];  // 64-bit words, low half first
    RmListEnt ent[64];
};
static_assert(sizeof(RmLists) <= sizeof(RmSmem<2, uint32_t>), "list table fits the smallest variant");

// Bitmap variant: popcount ranks over LDS bitmaps give every product its
// output position, products are bucketed by position and each bucket is
// summed in list-position order -- O(ip) work instead of a sort.
//
// Ranks come in levels of 64-way fan-out.  The top level has one bit per
// 2^SH columns of the row's own column span, SH the least of 0, 6, 12, 18
// for which the span fits rb_words<R>() words of 64 bits; each level below holds one
// 64-bit word per bit set above it (at most one per product), so its words
// are numbered by the popcount ranks of the level above, and the ranks of
// the last level (SH = 0) are the output positions.  A banded row takes one
// level of a few words whatever N is, a row spread over 2^20 columns two,
// over 2^26 three.  The levels share one LDS area (a level is dead once its
// ranks are in registers), and phase B (the buckets) reuses it; the products
// stay in registers until phase B places them.
//
// Measured on MI355X, against a flat bitmap in up to two chunks or two fixed
// levels (one wave scan per 64 words, two atomics per product, pending
// subtrees in registers) and a 64-bit bitonic sort above 2^20 columns, one
// row per wavefront: 1.15e6 rows of 257-512 products, N <= 65,536: 3.45 ->
// 3.01 ms and 1,312 -> 810 VALU instructions per row; 1.30e6 rows of 65-256
// products, N = 1.5e6: 4.04 -> 1.68 ms, and their count 1.07 (hash) -> 0.82.
// Then, several rows per wavefront (rm_rows), products without lanes of
// their own as repeats of the last one, and as many registers as the row
// needs (rm_step): 3.01 -> 2.32 ms and 750 instructions, count 0.82 -> 0.62 ms.
// The vector units are then busy 0.68 of the time (0.74 at R = 4), and bank
// conflicts take a fifth of the LDS cycles.
template <int R>
constexpr int rb_words() {
    return R < 4 ? 256 : 64 * R;  // words of one level: at least one per product
}
template <int R>
struct RbRanks {
    unsigned w[2 * rb_words<R>()];  // 64-bit words, low half first
    unsigned rank[rb_words<R>()];   // bits set before the low half | before the high half << 16
};
// Columns of the outputs: 16 bits while B has at most RB_NARROW columns.
constexpr int RB_NARROW = 1 << 16;
template <int R, bool WIDE>
struct RbBuckets {
    union {
        unsigned cnt[64 * R];    // contributions of each output, until the offsets are known
        double val[64 * R];      // contributions, bucket by bucket
    };
    unsigned short off[64 * R + 2];  // bucket offsets
    typename std::conditional<WIDE, int, unsigned short>::type oc[64 * R];  // output columns
    unsigned char lp[64 * R + 8];  // list position of each contribution (read 8 at a time)
};
template <int R, bool WIDE>
union RbSmem {
    RbRanks<R> a;
    RbBuckets<R, WIDE> b;
    RmLists l;
};
static_assert(64 * 32 <= 0xffff, "bucket offsets in 16 bits");

// The lane, as a value the compiler does not carry across rows: left alone it
// keeps every lane-dependent address and bound of the row loop in a register
// (tens of them).
__device__ __forceinline__ int rm_lane() {
    int l = lane_id();
    asm volatile("" : "+v"(l));
    return l;
}

// The rows of one wavefront: entries k0 .. k0 + n of the row list, one per
// lane.  Everything that names a row's data (its A entries, products, place
// in C) is loaded for all of them at once: three dependent trips to memory
// per wavefront instead of per row.
struct RmRows {
    int n;  // uniform
    int row, a0;
    unsigned lic;  // lists (7 bits) | products << 7 (12 bits) | capacity in C << 19 (13 bits, saturated)
    int64_t out;   // numeric: first entry in C (Upper: in C-bar)
};
__device__ __forceinline__ int lic_lists(unsigned x) { return (int)(x & 127u); }
__device__ __forceinline__ int lic_products(unsigned x) { return (int)((x >> 7) & 4095u); }
__device__ __forceinline__ int lic_cap(unsigned x) { return (int)(x >> 19); }
static_assert(WMED_LMAX < 128 && WMED_CAP_BITMAP < 4096, "row sizes in one word");

// Entry of the row list that workgroup b of nb takes, in steps of rpw rows.
// Consecutive workgroups go to the eight XCDs in turn; each XCD gets one
// contiguous share of the list, so that the rows of B its rows share are
// fetched into one L2 instead of eight.
__device__ __forceinline__ int64_t rm_first(unsigned b, unsigned nb, int rpw) {
    const unsigned x = b & 7u, q = nb >> 3, r = nb & 7u;
    return (int64_t)(x * q + min(x, r) + (b >> 3)) * rpw;
}

template <bool NUMERIC>
__device__ __forceinline__ RmRows rm_rows(const int* __restrict__ rows, int nrows, int rpw, const RowArgs& a,
                                          const OutArgs& o) {
    const int lane = rm_lane();
    const int64_t k0 = rm_first(blockIdx.x, gridDim.x, rpw);
    RmRows w;
    w.n = (int)min((int64_t)rpw, (int64_t)nrows - k0);
    const int64_t k = k0 + min(lane, w.n - 1);
    w.row = rows[k];
    w.a0 = a.arpt[w.row];
    const int a1 = a.arpt[w.row + 1];
    const int64_t base = a.ipA[w.a0];
    const int ip = (int)(a.ipA[a1] - base);
    int cap = ip;
    w.out = base;
    if (NUMERIC && !o.upper) {
        w.out = o.crpt[w.row];
        cap = (int)min(o.crpt[w.row + 1] - w.out, (int64_t)8191);
    }
    w.lic = (unsigned)(a1 - w.a0) | ((unsigned)ip << 7) | ((unsigned)cap << 19);
    return w;
}

// One row's lists, one per lane: B row range and A value.  Fetched in two
// dependent steps while the row before is worked on.
struct RmList {
    int col;  // A column, until bounds()
    int bst, len;
    double sc;
    template <bool VALS>
    __device__ __forceinline__ void entry(const RowArgs& a, int a0, int L) {
        const int i = a0 + min(lane_id(), L - 1);
        col = a.acol[i];
        if (VALS) sc = a.aval[i];
    }
    __device__ __forceinline__ void bounds(const RowArgs& a, int L) {
        bst = a.brpt[col];
        len = a.brpt[col + 1] - bst;
        if (lane_id() >= L) len = 0;
    }
};

// Stage 1 of a row of ip products: product j = 64 r + lane reads B entry
// bi[r] of the non-empty list ent[k[r]]; lanes past the row take its last
// product.  The k-th non-empty list fills table entry k and marks its first
// product (but product 0) in a bitmap; product j's list is then the entry
// numbered by the marks at or before j (v_mbcnt).
template <int R, bool VALS>
__device__ __forceinline__ void rm_products(const RmList& l, int ip, RmLists& ls, int (&bi)[R], int (&lp)[R],
                                            int (&k)[R]) {
    const int lane = rm_lane();
    if (lane < 2 * R) ls.start[lane] = 0u;
    const int off = wave_incl_scan(l.len) - l.len;
    const uint64_t nzl = __ballot(l.len > 0);
    wave_lds_sync();  // start words cleared
    if (l.len > 0) {
        if (off > 0) atomicOr(&ls.start[(off - 1) >> 5], 1u << ((off - 1) & 31));
        ls.ent[__builtin_amdgcn_mbcnt_hi((unsigned)(nzl >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)nzl, 0u))] =
            RmListEnt{l.bst - off, lane, VALS ? l.sc : 0.0};
    }
    wave_lds_sync();
    unsigned before = 0u;  // marks in the words before
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const unsigned lo = ls.start[2 * r], hi = ls.start[2 * r + 1];
        k[r] = (int)__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, before));
        before += __popc(lo) + __popc(hi);
        lp[r] = ls.ent[k[r]].lp;
        bi[r] = ls.ent[k[r]].b + min(r * 64 + lane, ip - 1);
    }
    wave_lds_sync();
}

// Products per lane a row of the kernel for 64 CAP products may run with: the
// least of four steps that holds it (three at CAP = 4), so that no register
// holds nothing but lanes past the row (a row of 300 products at CAP = 8
// takes 5 steps of 64, not 8).
template <int CAP>
constexpr int rm_step() {
    return CAP <= 8 ? 1 : CAP / 8;
}

// Minimum and maximum of the products' columns over the wavefront.
template <int R>
__device__ __forceinline__ void col_range(const int (&col)[R], int& cmn, int& cmx) {
    cmn = INT_MAX;
    cmx = -1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        cmn = min(cmn, col[r]);
        cmx = max(cmx, col[r]);
    }
    // prefix extremes with DPP moves; the last lane holds the wavefront's
    auto mn = [](int x, int y) { return min(x, y); };
    auto mx = [](int x, int y) { return max(x, y); };
    cmn = mn(cmn, dpp_mov<0x111, 0xF>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x111, 0xF>(cmx, -1));
    cmn = mn(cmn, dpp_mov<0x112, 0xF>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x112, 0xF>(cmx, -1));
    cmn = mn(cmn, dpp_mov<0x114, 0xF>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x114, 0xF>(cmx, -1));
    cmn = mn(cmn, dpp_mov<0x118, 0xF>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x118, 0xF>(cmx, -1));
    cmn = mn(cmn, dpp_mov<0x142, 0xA>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x142, 0xA>(cmx, -1));
    cmn = mn(cmn, dpp_mov<0x143, 0xC>(cmn, INT_MAX));
    cmx = mx(cmx, dpp_mov<0x143, 0xC>(cmx, -1));
    cmn = wave_last(cmn);
    cmx = wave_last(cmx);
}

// The top level of a row with columns in [cmn, cmx]: its shift, and the
// words it takes.  (Here and below: R products per lane, LDS sized for CAP
// products per lane.)
template <int CAP>
__device__ __forceinline__ int top_level(int cmn, int cmx, int& nw) {
    int sh = 0;
    while (((cmx >> sh) - (cmn >> sh)) >> 6 >= rb_words<CAP>()) sh += 6;
    nw = (((cmx >> sh) - (cmn >> sh)) >> 6) + 1;
    return sh;
}

// One level: bit idx[r] of every product lane < ip - r * 64 set in nw words
// of cleared bitmap.  Returns with the bits visible to the wavefront.
template <int R, int CAP>
__device__ __forceinline__ void level_bits(RbRanks<CAP>& A, const int (&idx)[R], int ip, int nw) {
    const int lane = rm_lane();
    unsigned long long* w64 = reinterpret_cast<unsigned long long*>(A.w);
#pragma unroll 1
    for (int i = 0; i < nw; i += BRM_WAVE) w64[i + lane] = 0ull;  // rb_words is a whole number of steps
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        // lanes past the row would all set their last product's bit again, one
        // after the other: only the trailing registers can hold any
        if (r < R - rm_step<CAP>() || lane < ip - r * 64) atomicOr(&A.w[idx[r] >> 5], 1u << (idx[r] & 31));
    }
    wave_lds_sync();
}

// Ranks of the nw words (exclusive prefix of their popcounts, one per half
// word), two steps of 64 words per wave scan (16 bits each: a step holds at
// most 4,096 bits); returns the number of bits set.
template <int CAP>
__device__ __forceinline__ int level_ranks(RbRanks<CAP>& A, int nw) {
    const int lane = rm_lane();
    const unsigned long long* w64 = reinterpret_cast<const unsigned long long*>(A.w);
    int tot = 0;
#pragma unroll 1
    for (int i = 0; i < nw; i += 2 * BRM_WAVE) {
        const bool two = i + BRM_WAVE < nw;  // uniform
        const unsigned long long x = w64[i + lane];
        const unsigned long long y = two ? w64[i + BRM_WAVE + lane] : 0ull;
        const int xl = __popc((unsigned)x), yl = __popc((unsigned)y);
        const int xc = xl + __popc((unsigned)(x >> 32)), yc = yl + __popc((unsigned)(y >> 32));
        const int inc = wave_incl_scan(xc | (yc << 16));
        const int all = wave_last(inc);
        const int ex = tot + (inc & 0xffff) - xc;
        A.rank[i + lane] = (unsigned)(ex | ((ex + xl) << 16));
        tot += all & 0xffff;
        if (two) {
            const int ey = tot + (int)((unsigned)inc >> 16) - yc;
            A.rank[i + BRM_WAVE + lane] = (unsigned)(ey | ((ey + yl) << 16));
            tot += (int)((unsigned)all >> 16);
        }
    }
    wave_lds_sync();
    return tot;
}

// Every product's rank among the bits set: into idx.
template <int R, int CAP>
__device__ __forceinline__ void level_lookup(const RbRanks<CAP>& A, int (&idx)[R]) {
    const unsigned short* rk = reinterpret_cast<const unsigned short*>(A.rank);
#pragma unroll
    for (int r = 0; r < R; ++r) idx[r] = rk[idx[r] >> 5] + popc_below(A.w[idx[r] >> 5], (unsigned)idx[r]);
    wave_lds_sync();  // read before the area is cleared or reused
}

// Output position of every product, of column col[r]: into pos; returns the
// number of outputs.
template <int R, int CAP>
__device__ __forceinline__ int rmed_ranks(const int (&col)[R], int ip, RbRanks<CAP>& A, int (&pos)[R]) {
    int cmn, cmx, nw;
    col_range<R>(col, cmn, cmx);
    int s = top_level<CAP>(cmn, cmx, nw);
    const int top = cmn >> s;
#pragma unroll
    for (int r = 0; r < R; ++r) pos[r] = (col[r] >> s) - top;
#pragma unroll 1
    for (;;) {  // uniform: one to four levels
        level_bits<R, CAP>(A, pos, ip, nw);
        // the bit indices only: their LDS addresses are formed again for the
        // lookup rather than kept in R registers (25 spills at R = 8)
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(pos[r]));
        nw = level_ranks<CAP>(A, nw);
        level_lookup<R, CAP>(A, pos);
        if (s == 0) return nw;
        s -= 6;
#pragma unroll
        for (int r = 0; r < R; ++r) pos[r] = pos[r] * 64 + ((col[r] >> s) & 63);
    }
}

// The row's outputs from its products (column col[r], list position lp[r],
// value prod[r], output position pos[r]): nout of them at out .. out + cap of
// C or C-bar.
template <int R, int CAP, bool WIDE>
__device__ __forceinline__ void rmed_outputs(const int (&col)[R], const int (&lp)[R], const double (&prod)[R],
                                             int (&pos)[R], int ip, int nout, int row, int64_t out, int dcap,
                                             const OutArgs& o, RbBuckets<CAP, WIDE>& B) {
    const int lane = rm_lane();
    // ---- ranks are dead from here on: contributions per output; a
    // product's arrival is its place in its bucket (kept above the position)
#pragma unroll 1
    for (int i = lane; i < nout; i += BRM_WAVE) B.cnt[i] = 0u;
    wave_lds_sync();
    int most = 0;  // largest arrival of this lane's products
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (lane < ip - r * 64) {
            const int arr = (int)atomicAdd(&B.cnt[pos[r]], 1u);
            most = max(most, arr);
            if (arr == 0) B.oc[pos[r]] = (typename std::conditional<WIDE, int, unsigned short>::type)col[r];
            pos[r] |= arr << 16;
        }
    }
    int* dcol = o.ccol + out;
    double* dval = o.cval + out;
    const int nst = min(nout, dcap);
    if (__ballot(most >= 2) == 0ull) {
        // ---- at most two contributions per output: the first to arrive
        // waits at the output's place, the second is added to it there
        const bool pairs = __ballot(most == 1) != 0ull;
        wave_lds_sync();  // counters are dead: values take their place
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (lane < ip - r * 64 && pos[r] < 0x10000) {
                B.val[pos[r]] = prod[r];
                if (pairs) B.lp[pos[r]] = (unsigned char)lp[r];
            }
        }
        wave_lds_sync();
        if (pairs) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (lane < ip - r * 64 && pos[r] >= 0x10000) {
                    const int q = pos[r] & 0xffff;
                    const double x = B.val[q];
                    B.val[q] = (int)B.lp[q] < lp[r] ? fadd(x, prod[r]) : fadd(prod[r], x);
                }
            }
            wave_lds_sync();
        }
#pragma unroll 1
        for (int q = lane; q < nst; q += BRM_WAVE) {
            dcol[q] = (int)B.oc[q];
            dval[q] = B.val[q];
        }
    } else {
        // ---- bucket offsets (exclusive scan of the counters, two steps of
        // 64 buckets per wave scan), then every product to its slot
        wave_lds_sync();
        int tot = 0;
#pragma unroll 1
        for (int i = lane; i - lane < nout; i += 2 * BRM_WAVE) {
            const int x = i < nout ? (int)B.cnt[i] : 0, y = i + BRM_WAVE < nout ? (int)B.cnt[i + BRM_WAVE] : 0;
            const int inc = wave_incl_scan(x | (y << 16));
            const int all = wave_last(inc);
            if (i < nout) B.off[i] = (unsigned short)(tot + (inc & 0xffff) - x);
            tot += all & 0xffff;
            if (i + BRM_WAVE < nout) B.off[i + BRM_WAVE] = (unsigned short)(tot + (int)((unsigned)inc >> 16) - y);
            tot += (int)((unsigned)all >> 16);
        }
        const unsigned short* off = B.off;
        if (lane == 0) B.off[nout] = (unsigned short)ip;
        wave_lds_sync();  // counters are dead: values take their place
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (lane < ip - r * 64) {
                const int slot = off[pos[r] & 0xffff] + (pos[r] >> 16);
                B.val[slot] = prod[r];
                B.lp[slot] = (unsigned char)lp[r];
            }
        }
        wave_lds_sync();
#pragma unroll 1
        for (int q = lane; q < nst; q += BRM_WAVE) {
            const int s = off[q];
            const int m = off[q + 1] - s;
            double v = B.val[s];
            if (m == 2) {
                const double y = B.val[s + 1];
                v = B.lp[s] < B.lp[s + 1] ? fadd(v, y) : fadd(y, v);
            } else if (m > 2) {
                v = rb_bucket_sum(B.lp + s, B.val + s, m);
            }
            dcol[q] = (int)B.oc[q];
            dval[q] = v;
        }
    }
    if (lane == 0) {
        if (o.upper) o.rowlen[row] = nout;
        else if (nout != dcap) atomicOr(o.err, (int)DERR_COUNT_MISMATCH);
    }
}

// Bitonic sort of the wavefront's first 64 rr keys (rr <= R, a power of
// two, uniform), element i = r * 64 + lane; registers r >= rr are untouched.
template <int R, typename KT>
__device__ __forceinline__ void wave_bitonic_sort(KT (&key)[R], int rr) {
    constexpr int N = 64 * R;
    const int lane = rm_lane();
    const int nrt = 64 * rr;
#pragma unroll
    for (int k = 2; k <= N; k <<= 1) {
        if (k > nrt) break;
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= 64) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int rp = r ^ (j >> 6);
                    if (r < rp && rp < rr) {
                        const int i = r * 64 + lane;
                        const bool asc = (i & k) == 0;
                        const KT x = key[r], y = key[rp];
                        const bool sw = asc ? (x > y) : (x < y);
                        key[r] = sw ? y : x;
                        key[rp] = sw ? x : y;
                    }
                }
            } else {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (r >= rr) break;
                    const int i = r * 64 + lane;
                    const bool asc = (i & k) == 0;
                    const bool lower = (lane & j) == 0;
                    const KT x = key[r];
                    const KT y = shfl_xor_key(x, j);
                    const KT mn = x < y ? x : y;
                    const KT mx = x < y ? y : x;
                    key[r] = (lower == asc) ? mn : mx;
                }
            }
        }
    }
}

// The sort variant of a row's outputs (stages 2 to 4 above).
template <int R, typename KT>
__device__ __forceinline__ void rmed_sort(const int (&col)[R], const int (&lp)[R], const double (&prod)[R], int ip,
                                          int row, int64_t out, int dcap, const OutArgs& o, RmSmem<R, KT>& sm) {
    using Key = RmKey<R, KT>;
    const int lane = rm_lane();
    KT key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = r * 64 + lane;
        key[r] = j < ip ? Key::make(col[r], lp[r], j) : ~(KT)0;
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (r * 64 < ip) sm.val[r * 64 + lane] = prod[r];

    // ---- 2. sort by (column, list position): only the registers the row uses
    int rr = 1;
    while (64 * rr < ip) rr <<= 1;
    wave_bitonic_sort<R, KT>(key, rr);

    // ---- 3. run heads; sums of the runs
#pragma unroll
    for (int r = 0; r < R; ++r) sm.key[r * 64 + lane] = key[r];
    __syncthreads();
    bool head[R];
    int nout = 0;
    int idx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = r * 64 + lane;
        const uint32_t c = Key::col(key[r]);
        const bool valid = i < ip;
        const bool h = valid && (i == 0 || Key::col(sm.key[i - 1]) != c);
        head[r] = h;
        const uint64_t bal = __ballot(h);
        idx[r] = nout + __popcll(bal & ((1ull << lane) - 1ull));
        nout += __popcll(bal);
    }
    int* dcol = o.ccol + out;
    double* dval = o.cval + out;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (!head[r]) continue;
        const int i = r * 64 + lane;
        const uint32_t c = Key::col(key[r]);
        int prev = Key::lp(key[r]);
        double cur = sm.val[Key::j(key[r])];
        double lv[RM_LOGL];
        unsigned pend = 0u;
        for (int q = i + 1; q < ip; ++q) {
            const KT kq = sm.key[q];
            if (Key::col(kq) != c) break;
            const int l = Key::lp(kq);
            const int d = 31 - __clz(prev ^ l);
            double v = cur;
#pragma unroll
            for (int h = 0; h < RM_LOGL; ++h)
                if (h < d && ((pend >> h) & 1u)) v = fadd(lv[h], v);
#pragma unroll
            for (int h = 0; h < RM_LOGL; ++h)
                if (h == d) lv[h] = v;
            pend = (pend & ~((1u << d) - 1u)) | (1u << d);
            cur = sm.val[Key::j(kq)];
            prev = l;
        }
        double v = cur;
#pragma unroll
        for (int h = 0; h < RM_LOGL; ++h)
            if ((pend >> h) & 1u) v = fadd(lv[h], v);
        if (idx[r] < dcap) {
            dcol[idx[r]] = (int)c;
            dval[idx[r]] = v;
        }
    }
    if (lane == 0) {
        if (o.upper) o.rowlen[row] = nout;
        else if (nout != dcap) atomicOr(o.err, (int)DERR_COUNT_MISMATCH);
    }
}

// Waves per SIMD the register allocation must leave room for.
template <int R>
constexpr int rm_waves() {
    return R <= 4 ? 8 : R == 8 ? 6 : R == 16 ? 4 : 2;
}

// MODE 0: sort; 1: bitmap ranks (B of at most RB_NARROW columns); 2: bitmap
// ranks, any number of columns.
// One row of ip <= 64 R products: its lists in `l`, its outputs at out ..
// out + cap.  The next row's lists (nL of them from A entry na0) are fetched
// into l beside this row's work: its A entries beside this row's B entries,
// its B row ranges beside the buckets.
template <int R, int CAP, typename KT, int MODE, typename SH>
__device__ __forceinline__ void rmed_row(const RowArgs& a, const OutArgs& o, RmList& l, int na0, int nL, int row,
                                         int ip, int64_t out, int cap, SH& shm) {
    RmLists& ls = *reinterpret_cast<RmLists*>(&shm);
    int bi[R], lp[R], k[R];
    rm_products<R, true>(l, ip, ls, bi, lp, k);
    int col[R];
    double prod[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        col[r] = a.bcol[bi[r]];
        prod[r] = a.bval[bi[r]];
    }
    l.entry<true>(a, na0, nL);
    // the lists' A values are read from the table only now, so that they take
    // no registers while the loads are in flight
#pragma unroll
    for (int r = 0; r < R; ++r) prod[r] = fmul(ls.ent[k[r]].sc, prod[r]);
    wave_lds_sync();  // the table is read before its area is reused
    if constexpr (MODE != 0) {
        // list positions stay in registers as they are: left to itself the
        // compiler carries their derivation along (245 VGPRs instead of 120
        // at R = 16, spills at R = 32)
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(lp[r]));
        int pos[R];
        const int nout = rmed_ranks<R, CAP>(col, ip, shm.a, pos);
        l.bounds(a, nL);
        rmed_outputs<R, CAP, MODE == 2>(col, lp, prod, pos, ip, nout, row, out, cap, o, shm.b);
    } else {
        l.bounds(a, nL);
        rmed_sort<R, KT>(col, lp, prod, ip, row, out, cap, o, shm);
    }
}

template <int CAP, typename KT, int MODE>
__global__ __launch_bounds__(BRM_WAVE, rm_waves<CAP>()) void k_rmed(const int* __restrict__ rows, int nrows, int rpw,
                                                                    RowArgs a, OutArgs o) {
    // one of the layouts, sized for the variant; the list table of stage 1
    // overlays the start of each
    __shared__ typename std::conditional<MODE == 0, RmSmem<CAP, KT>, RbSmem<CAP, MODE == 2>>::type shm;
    const RmRows w = rm_rows<true>(rows, nrows, rpw, a, o);
    RmList l;
    const int L0 = lic_lists((unsigned)__builtin_amdgcn_readlane((int)w.lic, 0));
    l.entry<true>(a, __builtin_amdgcn_readlane(w.a0, 0), L0);
    l.bounds(a, L0);
#pragma unroll 1
    for (int i = 0; i < w.n; ++i) {
        const unsigned lic = (unsigned)__builtin_amdgcn_readlane((int)w.lic, i);
        const int row = __builtin_amdgcn_readlane(w.row, i), ip = lic_products(lic), cap = lic_cap(lic);
        const int64_t out = readlane64(w.out, i);
        const int j = min(i + 1, w.n - 1);
        const int na0 = __builtin_amdgcn_readlane(w.a0, j);
        const int nL = lic_lists((unsigned)__builtin_amdgcn_readlane((int)w.lic, j));
        constexpr int S = rm_step<CAP>();
        if constexpr (MODE == 0 || CAP < 4) {
            rmed_row<CAP, CAP, KT, MODE>(a, o, l, na0, nL, row, ip, out, cap, shm);
        } else {
            if (ip > 64 * (CAP - S)) rmed_row<CAP, CAP, KT, MODE>(a, o, l, na0, nL, row, ip, out, cap, shm);
            else if (ip > 64 * (CAP - 2 * S))
                rmed_row<CAP - S, CAP, KT, MODE>(a, o, l, na0, nL, row, ip, out, cap, shm);
            else if (CAP == 4 || ip > 64 * (CAP - 3 * S))
                rmed_row<CAP - 2 * S, CAP, KT, MODE>(a, o, l, na0, nL, row, ip, out, cap, shm);
            else if constexpr (CAP > 4)
                rmed_row<CAP - 3 * S, CAP, KT, MODE>(a, o, l, na0, nL, row, ip, out, cap, shm);
        }
        wave_lds_sync();  // outputs read before the next row's list table
    }
}

// Symbolic count of register-tier rows: the row's length is the number of
// bits set in the last level of the numeric variant's bitmaps.
template <int R>
union RcSmem {
    RmLists l;
    RbRanks<R> a;
};

template <int R, int CAP>
__device__ __forceinline__ int rmed_row_count(const RowArgs& a, RmList& l, int na0, int nL, int ip, RcSmem<CAP>& sh) {
    int bi[R], lp[R], k[R];
    rm_products<R, false>(l, ip, sh.l, bi, lp, k);
    int col[R];
#pragma unroll
    for (int r = 0; r < R; ++r) col[r] = a.bcol[bi[r]];
    l.entry<false>(a, na0, nL);
    int cmn, cmx, nw;
    col_range<R>(col, cmn, cmx);
    l.bounds(a, nL);
    int s = top_level<CAP>(cmn, cmx, nw);
    const int top = cmn >> s;
    int idx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) idx[r] = (col[r] >> s) - top;
#pragma unroll 1
    for (;;) {  // uniform
        level_bits<R, CAP>(sh.a, idx, ip, nw);
        if (s == 0) break;
        nw = level_ranks<CAP>(sh.a, nw);
        level_lookup<R, CAP>(sh.a, idx);
        s -= 6;
#pragma unroll
        for (int r = 0; r < R; ++r) idx[r] = idx[r] * 64 + ((col[r] >> s) & 63);
    }
    const int lane = rm_lane();
    int cnt = 0;
    const unsigned long long* w64 = reinterpret_cast<const unsigned long long*>(sh.a.w);
#pragma unroll 1
    for (int q = 0; q < nw; q += BRM_WAVE) cnt += __popcll(w64[q + lane]);
    return wave_sum(cnt);
}

template <int CAP>
__global__ __launch_bounds__(BRM_WAVE) void k_rmed_count(const int* __restrict__ rows, int nrows, int rpw, RowArgs a,
                                                         int64_t* __restrict__ nnzrow) {
    __shared__ RcSmem<CAP> sh;
    const RmRows w = rm_rows<false>(rows, nrows, rpw, a, OutArgs{});
    RmList l;
    const int L0 = lic_lists((unsigned)__builtin_amdgcn_readlane((int)w.lic, 0));
    l.entry<false>(a, __builtin_amdgcn_readlane(w.a0, 0), L0);
    l.bounds(a, L0);
    int mine = 0;  // lane i: the count of row i
#pragma unroll 1
    for (int i = 0; i < w.n; ++i) {
        const int ip = lic_products((unsigned)__builtin_amdgcn_readlane((int)w.lic, i));
        const int j = min(i + 1, w.n - 1);
        const int na0 = __builtin_amdgcn_readlane(w.a0, j);
        const int nL = lic_lists((unsigned)__builtin_amdgcn_readlane((int)w.lic, j));
        constexpr int S = rm_step<CAP>();
        int cnt = 0;
        if constexpr (CAP < 4) {
            cnt = rmed_row_count<CAP, CAP>(a, l, na0, nL, ip, sh);
        } else {
            if (ip > 64 * (CAP - S)) cnt = rmed_row_count<CAP, CAP>(a, l, na0, nL, ip, sh);
            else if (ip > 64 * (CAP - 2 * S)) cnt = rmed_row_count<CAP - S, CAP>(a, l, na0, nL, ip, sh);
            else if (CAP == 4 || ip > 64 * (CAP - 3 * S)) cnt = rmed_row_count<CAP - 2 * S, CAP>(a, l, na0, nL, ip, sh);
            else if constexpr (CAP > 4) cnt = rmed_row_count<CAP - 3 * S, CAP>(a, l, na0, nL, ip, sh);
        }
        if (lane_id() == i) mine = cnt;
        wave_lds_sync();  // words read before the next row's list table
    }
    if (lane_id() < w.n) nnzrow[w.row] = mine;
}

// Rows per wavefront: RM_RPW once that still leaves twice the wavefronts the
// chip holds, fewer (down to one) for shorter lists.  One row per wavefront
// waits on six dependent trips to memory for 75% of its cycles; on the
// 192-pair batch's plan 1, 4, 8 and 16 rows took 5.05, 4.40, 4.36 and 4.45 ms.
constexpr int RM_RPW = 8;
template <int R>
int rm_rpw(int n) {
    const int fill = 2 * 256 * 4 * rm_waves<R>();
    return std::max(1, std::min(RM_RPW, n / fill));
}
inline unsigned rm_blocks(int n, int rpw) { return (unsigned)(((int64_t)n + rpw - 1) / rpw); }

template <int R>
hipError_t rmed_count_t(const int* rows, int n, const RowArgs& a, int64_t* nnzrow, hipStream_t s) {
    const int64_t ch = launch_chunk(BRM_WAVE);
    for (int64_t b = 0; b < n; b += ch) {
        const int c = (int)std::min<int64_t>(ch, n - b);
        const int rpw = rm_rpw<R>(c);
        k_rmed_count<R><<<rm_blocks(c, rpw), BRM_WAVE, 0, s>>>(rows + b, c, rpw, a, nnzrow);
    }
    return hipGetLastError();
}

template <int R>
hipError_t rmed_t(const int* rows, int n, const RowArgs& a, const OutArgs& o, hipStream_t s) {
    const int64_t ch = launch_chunk(BRM_WAVE);
    const bool narrow = a.N <= 0 || (int64_t)a.N - 1 <= RmKey<R, uint32_t>::COL_MAX;
    const int mode = params().wmed_bitmap != 1 || R < 4 ? 0 : a.N <= RB_NARROW ? 1 : 2;
    // rows of more than 1024 products are binned only where the ranks run
    if (R > 16 && mode == 0) return hipErrorInvalidValue;
    for (int64_t b = 0; b < n; b += ch) {
        const int c = (int)std::min<int64_t>(ch, n - b);
        const int rpw = rm_rpw<R>(c);
        const unsigned nb = rm_blocks(c, rpw);
        if constexpr (R >= 4) {
            if (mode == 1) {
                k_rmed<R, uint32_t, 1><<<nb, BRM_WAVE, 0, s>>>(rows + b, c, rpw, a, o);
                continue;
            }
            if (mode == 2) {
                k_rmed<R, uint32_t, 2><<<nb, BRM_WAVE, 0, s>>>(rows + b, c, rpw, a, o);
                continue;
            }
        }
        if constexpr (R <= 16) {
            if (narrow) k_rmed<R, uint32_t, 0><<<nb, BRM_WAVE, 0, s>>>(rows + b, c, rpw, a, o);
            else k_rmed<R, uint64_t, 0><<<nb, BRM_WAVE, 0, s>>>(rows + b, c, rpw, a, o);
        }
    }
    return hipGetLastError();
}

}  // namespace

// B of at most RM_WIDE columns: rows of up to WMED_CAP_BITMAP products.
constexpr int RM_WIDE = 1 << 20;

int rmed_auto_cap(int N) {
    // With bitmap ranks rows of up to WMED_CAP_BITMAP products while B has at
    // most RM_WIDE columns (rows of 1025-2048 products: 2,048 products per
    // wavefront ran faster than the workgroup LDS tier).  Otherwise the sort's
    // limits: 1024 products while 32-bit keys hold N columns beside 16 bits of
    // position and index, else 512.  Above RM_WIDE columns that is not the
    // ranks' own limit, which serve any N: the rows between run faster with
    // wmed_cap 1024 than in the LDS tier (200,000 rows of 600 products, 1.5e6
    // columns: 1.09 ms against 19.0; 120,000 of 990: 0.97 against 15.9).
    if (params().wmed_bitmap == 1 && N <= RM_WIDE) return WMED_CAP_BITMAP;
    return (int64_t)N - 1 <= RmKey<16, uint32_t>::COL_MAX ? 1024 : 512;
}

int rmed_max_cap(int N) {
    return params().wmed_bitmap == 1 && N <= RM_WIDE ? WMED_CAP_BITMAP : WMED_CAP;
}

hipError_t launch_rmed_count(const int* rows, int n, const RowArgs& a, int64_t* nnzrow, hipStream_t s, int cap) {
    if (n <= 0) return hipSuccess;
    ProfScope ps_("k_rmed_count", s);
    if (cap <= 128) return rmed_count_t<2>(rows, n, a, nnzrow, s);
    if (cap <= 256) return rmed_count_t<4>(rows, n, a, nnzrow, s);
    if (cap <= 512) return rmed_count_t<8>(rows, n, a, nnzrow, s);
    if (cap <= 1024) return rmed_count_t<16>(rows, n, a, nnzrow, s);
    return rmed_count_t<32>(rows, n, a, nnzrow, s);
}

hipError_t launch_rmed_numeric(const int* rows, int n, const RowArgs& a, const OutArgs& o, hipStream_t s, int cap) {
    if (n <= 0) return hipSuccess;
    ProfScope ps_("k_rmed", s);
    if (cap <= 128) return rmed_t<2>(rows, n, a, o, s);
    if (cap <= 256) return rmed_t<4>(rows, n, a, o, s);
    if (cap <= 512) return rmed_t<8>(rows, n, a, o, s);
    if (cap <= 1024) return rmed_t<16>(rows, n, a, o, s);
    return rmed_t<32>(rows, n, a, o, s);
}

}  // namespace brm
