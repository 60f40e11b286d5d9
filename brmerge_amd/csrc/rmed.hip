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

// Stage 1: the row's non-empty lists, k-th at ent[k] (first product, list
// position, B row start, A value); bit j of start is set when a non-empty
// list begins at product j.  Overlays the start of each variant's LDS.
struct RmListEnt {
    int off_lp;  // first product | list position << 16
    int bst;
    double sc;
};
struct RmLists {
    unsigned long long start[32];
    RmListEnt ent[64];
};
static_assert(sizeof(RmLists) <= sizeof(RmSmem<2, uint32_t>), "list table fits the smallest variant");

// Bitmap variant: popcount ranks over LDS bitmaps give every product its
// output position, products are bucketed by position and each bucket is
// summed in list-position order -- O(ip) work instead of a sort.
//
// Ranks come in levels of 64-way fan-out.  The top level has one bit per
// 2^SH columns of the row's own column span, SH the least of 0, 6, 12, 18
// for which the span fits RB_NW words of 64 bits; each level below holds one
// 64-bit word per bit set above it (at most one per product), so its words
// are numbered by the popcount ranks of the level above, and the ranks of
// the last level (SH = 0) are the output positions.  A banded row takes one
// level of a few words whatever N is, a row spread over 2^20 columns two,
// over 2^26 three.  The levels share one LDS area (a level is dead once its
// ranks are in registers), and phase B (the buckets) reuses it; the products
// stay in registers until phase B places them.
//
// Measured on MI355X (kernel time, before: a flat bitmap in up to two chunks
// or two fixed levels, one wave scan per 64 words, two atomics per product,
// pending subtrees in registers; a 64-bit bitonic sort above 2^20 columns):
// 1.15e6 rows of 257-512 products, N <= 65,536: 3.45 -> 3.01 ms, 1,312 -> 810
// VALU instructions per row; 1.30e6 rows of 65-256 products, N = 1.5e6: 4.04
// -> 1.68 ms, and their count 1.07 (hash) -> 0.82 ms.
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
    double val[64 * R];         // contributions, bucket by bucket
    unsigned cnt[32 * R + 1];   // 16-bit bucket counters, then offsets, two per word (bucket 2i low, 2i + 1 high)
    typename std::conditional<WIDE, int, unsigned short>::type oc[64 * R];
    unsigned char lp[64 * R];   // list position of each contribution
};
template <int R, bool WIDE>
union RbSmem {
    RbRanks<R> a;
    RbBuckets<R, WIDE> b;
    RmLists l;
};
static_assert(64 * 32 <= 0xffff, "bucket offsets in 16 bits");

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Sum of one bucket (m >= 3 contributions from distinct lists) as the
// aligned tree over list positions: one pass over the contributions in list
// order with the pending left subtrees on a stack.  The pending heights
// shrink towards the top of the stack, so one bit mask holds them; when the
// next list first differs from the last one at bit d, the pending subtrees
// below height d are complete on its left and are added (left + right), and
// the sum waits at height d.  The stack takes the place of contributions
// already read (LDS), which keeps a push to about a dozen instructions (with
// the stack in registers, one slot per height, every push selects over all
// heights).
__device__ double rb_bucket_sum(unsigned char* lp, double* val, int m) {
    int prev = lp[0];
    // contributions placed by one register step of the wavefront may be out
    // of list order: order the bucket first
    for (int t = 1; t < m; ++t) {
        const int l = lp[t];
        if (l < prev) {
            const double x = val[t];
            int u = t;
            for (; u > 0 && (int)lp[u - 1] > l; --u) {
                lp[u] = lp[u - 1];
                val[u] = val[u - 1];
            }
            lp[u] = (unsigned char)l;
            val[u] = x;
        } else {
            prev = l;
        }
    }
    prev = lp[0];
    double cur = val[0];
    unsigned pend = 0u;
    int top = 0;
    for (int t = 1; t < m; ++t) {
        const int l = lp[t];
        const double x = val[t];
        const unsigned bit = 1u << (31 - __clz(prev ^ l));
        unsigned low = pend & (bit - 1u);
        pend = (pend & ~(bit - 1u)) | bit;
        while (low) {
            cur = fadd(val[--top], cur);
            low &= low - 1u;
        }
        val[top++] = cur;
        cur = x;
        prev = l;
    }
    while (top > 0) cur = fadd(val[--top], cur);
    return cur;
}

// Stage 1 of a row (A entries a0 .. a0 + L, products base .. base + ip):
// product j = 64 r + lane (j < ip) reads B entry bi[r] of list lp[r], whose
// A value is sv[r] (VALS).  The k-th non-empty list marks its first product
// in a bitmap and fills table entry k; product j's list is then entry
// (non-empty lists starting at or before j) - 1.  Ends with the table read
// and its LDS free for reuse.
template <int R, bool VALS>
__device__ __forceinline__ void rm_products(const RowArgs& a, int a0, int L, int64_t base, int ip, RmLists& ls,
                                            int (&bi)[R], int (&lp)[R], double (&sv)[R]) {
    const int lane = lane_id();
    if (lane < R) ls.start[lane] = 0ull;
    int off = 0, bst = 0, len = 0;
    double sc = 0.0;
    if (lane < L) {
        off = (int)(a.ipA[a0 + lane] - base);
        len = (int)(a.ipA[a0 + lane + 1] - base) - off;
        bst = a.brpt[a.acol[a0 + lane]];
        if (VALS) sc = a.aval[a0 + lane];
    }
    const uint64_t nzl = __ballot(len > 0);
    wave_lds_sync();  // start words cleared
    if (len > 0) {
        atomicOr(&ls.start[off >> 6], 1ull << (off & 63));
        ls.ent[__popcll(nzl & ((1ull << lane) - 1ull))] = RmListEnt{off | (lane << 16), bst, sc};
    }
    wave_lds_sync();
    const uint64_t upto = ~0ull >> (63 - lane);  // bits 0..lane
    int before = 0;                               // non-empty lists starting before product 64 r
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = r * 64 + lane;
        lp[r] = 0;
        bi[r] = 0;
        sv[r] = 0.0;
        if (r * 64 >= ip) continue;  // uniform
        const uint64_t w = ls.start[r];
        if (j < ip) {
            const RmListEnt e = ls.ent[before + __popcll(w & upto) - 1];
            lp[r] = e.off_lp >> 16;
            bi[r] = e.bst + j - (e.off_lp & 0xffff);
            if (VALS) sv[r] = e.sc;
        }
        before += __popcll(w);
    }
    wave_lds_sync();  // the table is read before its area is reused
}

// Bits of w below bit b (b taken mod 32).
__device__ __forceinline__ int popc_below(unsigned w, unsigned b) {
    return __popc(__builtin_amdgcn_ubfe(w, 0u, b & 31u));
}

// Minimum and maximum of the products' columns over the wavefront.
template <int R>
__device__ __forceinline__ void col_range(const int (&col)[R], int ip, int& cmn, int& cmx) {
    const int lane = lane_id();
    cmn = INT_MAX;
    cmx = -1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r * 64 + lane < ip) {
            cmn = min(cmn, col[r]);
            cmx = max(cmx, col[r]);
        }
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
// words it takes.
template <int R>
__device__ __forceinline__ int top_level(int cmn, int cmx, int& nw) {
    int sh = 0;
    while (((cmx >> sh) - (cmn >> sh)) >> 6 >= rb_words<R>()) sh += 6;
    nw = (((cmx >> sh) - (cmn >> sh)) >> 6) + 1;
    return sh;
}

// One level: bit idx[r] of every product r * 64 + lane < ip set in nw words
// of cleared bitmap.  Returns with the bits visible to the wavefront.
template <int R>
__device__ __forceinline__ void level_bits(RbRanks<R>& A, const int (&idx)[R], int ip, int nw) {
    const int lane = lane_id();
    unsigned long long* w64 = reinterpret_cast<unsigned long long*>(A.w);
#pragma unroll 1
    for (int i = 0; i < nw; i += BRM_WAVE) w64[i + lane] = 0ull;  // rb_words is a whole number of steps
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (r * 64 + lane < ip) atomicOr(&A.w[idx[r] >> 5], 1u << (idx[r] & 31));
    wave_lds_sync();
}

// Ranks of the nw words (exclusive prefix of their popcounts, one per half
// word), two steps of 64 words per wave scan (16 bits each: a step holds at
// most 4,096 bits); returns the number of bits set.
template <int R>
__device__ __forceinline__ int level_ranks(RbRanks<R>& A, int nw) {
    const int lane = lane_id();
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
template <int R>
__device__ __forceinline__ void level_lookup(const RbRanks<R>& A, int (&idx)[R], int ip) {
    const int lane = lane_id();
    const unsigned short* rk = reinterpret_cast<const unsigned short*>(A.rank);
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (r * 64 + lane < ip) idx[r] = rk[idx[r] >> 5] + popc_below(A.w[idx[r] >> 5], (unsigned)idx[r]);
    wave_lds_sync();  // read before the area is cleared or reused
}

// Products of product indices 64 r + lane < ip: column col[r], list position
// lp[r], value prod[r].
template <int R, bool WIDE>
__device__ __forceinline__ void rmed_bitmap(const int (&col)[R], const int (&lp)[R], const double (&prod)[R], int ip,
                                            int row, int64_t base, const OutArgs& o, RbSmem<R, WIDE>& sh) {
    const int lane = lane_id();
    int pos[R];
    int nout;
    {
        int cmn, cmx, nw;
        col_range<R>(col, ip, cmn, cmx);
        int s = top_level<R>(cmn, cmx, nw);
        const int top = cmn >> s;
#pragma unroll
        for (int r = 0; r < R; ++r) pos[r] = (col[r] >> s) - top;
#pragma unroll 1
        for (;;) {  // uniform: one to four levels
            level_bits<R>(sh.a, pos, ip, nw);
            nout = level_ranks<R>(sh.a, nw);
            level_lookup<R>(sh.a, pos, ip);
            if (s == 0) break;
            s -= 6;
            nw = nout;
#pragma unroll
            for (int r = 0; r < R; ++r) pos[r] = pos[r] * 64 + ((col[r] >> s) & 63);
        }
    }
    // ---- ranks are dead from here on: contributions per output; a
    // product's arrival is its place in its bucket (kept above the position)
    RbBuckets<R, WIDE>& B = sh.b;
    const int ncw = (nout + 1) >> 1;
#pragma unroll 1
    for (int i = lane; i < ncw; i += BRM_WAVE) B.cnt[i] = 0u;
    wave_lds_sync();
    int most = 0;  // largest arrival of this lane's products
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r * 64 + lane < ip) {
            const unsigned sft = (unsigned)(pos[r] & 1) << 4;
            const int arr = (int)((atomicAdd(&B.cnt[pos[r] >> 1], 1u << sft) >> sft) & 0xffffu);
            most = max(most, arr);
            if (arr == 0) B.oc[pos[r]] = (typename std::conditional<WIDE, int, unsigned short>::type)col[r];
            pos[r] |= arr << 16;
        }
    }
    int* dcol;
    double* dval;
    int64_t dcap;
    if (!o.upper) {
        const int64_t cb = o.crpt[row];
        dcol = o.ccol + cb;
        dval = o.cval + cb;
        dcap = o.crpt[row + 1] - cb;
    } else {
        dcol = o.ccol + base;
        dval = o.cval + base;
        dcap = ip;
    }
    const int nst = (int)min((int64_t)nout, dcap);
    if (__ballot(most >= 2) == 0ull) {
        // ---- at most two contributions per output: the first to arrive
        // waits at the output's place, the second is added to it there
        const bool pairs = __ballot(most == 1) != 0ull;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r * 64 + lane < ip && pos[r] < 0x10000) {
                B.val[pos[r]] = prod[r];
                if (pairs) B.lp[pos[r]] = (unsigned char)lp[r];
            }
        }
        wave_lds_sync();
        if (pairs) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (r * 64 + lane < ip && pos[r] >= 0x10000) {
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
        // 128 buckets per wave scan), then every product to its slot
        wave_lds_sync();
        int tot = 0;
#pragma unroll 1
        for (int i = 0; i < ncw; i += 2 * BRM_WAVE) {
            const int p = i + lane, q = i + BRM_WAVE + lane;
            const unsigned x = p < ncw ? B.cnt[p] : 0u, y = q < ncw ? B.cnt[q] : 0u;
            const int x0 = (int)(x & 0xffffu), y0 = (int)(y & 0xffffu);
            const int xt = x0 + (int)(x >> 16), yt = y0 + (int)(y >> 16);
            const int inc = wave_incl_scan(xt | (yt << 16));
            const int all = wave_last(inc);
            const int ex = tot + (inc & 0xffff) - xt;
            tot += all & 0xffff;
            const int ey = tot + (int)((unsigned)inc >> 16) - yt;
            tot += (int)((unsigned)all >> 16);
            if (p < ncw) B.cnt[p] = (unsigned)(ex | ((ex + x0) << 16));
            if (q < ncw) B.cnt[q] = (unsigned)(ey | ((ey + y0) << 16));
        }
        unsigned short* off = reinterpret_cast<unsigned short*>(B.cnt);
        if (lane == 0) off[nout] = (unsigned short)ip;
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if (r * 64 + lane < ip) {
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
        else if ((int64_t)nout != dcap) atomicOr(o.err, (int)DERR_COUNT_MISMATCH);
    }
}

// Bitonic sort of the wavefront's first 64 rr keys (rr <= R, a power of
// two, uniform), element i = r * 64 + lane; registers r >= rr are untouched.
template <int R, typename KT>
__device__ __forceinline__ void wave_bitonic_sort(KT (&key)[R], int rr) {
    constexpr int N = 64 * R;
    const int lane = lane_id();
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

// Waves per SIMD the register allocation must leave room for.
template <int R>
constexpr int rm_waves() {
    return R <= 4 ? 8 : R == 8 ? 6 : R == 16 ? 4 : 2;
}

// MODE 0: sort; 1: bitmap ranks (B of at most RB_NARROW columns); 2: bitmap
// ranks, any number of columns.
template <int R, typename KT, int MODE>
__global__ __launch_bounds__(BRM_WAVE, rm_waves<R>()) void k_rmed(const int* __restrict__ rows, int nrows, RowArgs a, OutArgs o) {
    using Key = RmKey<R, KT>;
    // one of the layouts, sized for the variant; the list table of stage 1
    // overlays the start of each
    __shared__ typename std::conditional<MODE == 0, RmSmem<R, KT>, RbSmem<R, MODE == 2>>::type shm;
    RmSmem<R, KT>& sm = *reinterpret_cast<RmSmem<R, KT>*>(&shm);
    RmLists& ls = *reinterpret_cast<RmLists*>(&shm);
    const int lane = lane_id();
    const int row = rows[blockIdx.x];
    const int a0 = a.arpt[row];
    const int L = a.arpt[row + 1] - a0;
    const int64_t base = a.ipA[a0];
    const int ip = (int)(a.ipA[a0 + L] - base);

    // ---- 1. list descriptors in lanes, products in registers
    int bi[R], lp[R];
    double sv[R];
    rm_products<R, true>(a, a0, L, base, ip, ls, bi, lp, sv);
    int col[R];
    double prod[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        col[r] = 0;
        prod[r] = 0.0;
        if (r * 64 + lane < ip) {
            col[r] = a.bcol[bi[r]];
            prod[r] = fmul(sv[r], a.bval[bi[r]]);
        }
    }

    // ---- bitmap ranks instead of a sort
    if constexpr (MODE != 0) {
        // list positions stay in registers as they are: left to itself the
        // compiler carries their derivation along (245 VGPRs instead of 120
        // at R = 16, spills at R = 32)
#pragma unroll
        for (int r = 0; r < R; ++r) asm volatile("" : "+v"(lp[r]));
        rmed_bitmap<R, MODE == 2>(col, lp, prod, ip, row, base, o, shm);
        return;
    }
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
    int* dcol;
    double* dval;
    int64_t dcap;
    if (!o.upper) {
        const int64_t cb = o.crpt[row];
        dcol = o.ccol + cb;
        dval = o.cval + cb;
        dcap = o.crpt[row + 1] - cb;
    } else {
        const int64_t cb = base;
        dcol = o.ccol + cb;
        dval = o.cval + cb;
        dcap = ip;
    }
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
        else if ((int64_t)nout != dcap) atomicOr(o.err, (int)DERR_COUNT_MISMATCH);
    }
}

// Symbolic count of register-tier rows: the row's length is the number of
// bits set in the last level of the numeric variant's bitmaps.
template <int R>
union RcSmem {
    RmLists l;
    RbRanks<R> a;
};

template <int R>
__global__ __launch_bounds__(BRM_WAVE) void k_rmed_count(const int* __restrict__ rows, int nrows, RowArgs a,
                                                         int64_t* __restrict__ nnzrow) {
    __shared__ RcSmem<R> sh;
    const int lane = lane_id();
    const int row = rows[blockIdx.x];
    const int a0 = a.arpt[row];
    const int L = a.arpt[row + 1] - a0;
    const int64_t base = a.ipA[a0];
    const int ip = (int)(a.ipA[a0 + L] - base);
    int bi[R], lp[R];
    double sv[R];
    rm_products<R, false>(a, a0, L, base, ip, sh.l, bi, lp, sv);
    int col[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        col[r] = 0;
        if (r * 64 + lane < ip) col[r] = a.bcol[bi[r]];
    }
    int cmn, cmx, nw;
    col_range<R>(col, ip, cmn, cmx);
    int s = top_level<R>(cmn, cmx, nw);
    const int top = cmn >> s;
    int idx[R];
#pragma unroll
    for (int r = 0; r < R; ++r) idx[r] = (col[r] >> s) - top;
#pragma unroll 1
    for (;;) {  // uniform
        level_bits<R>(sh.a, idx, ip, nw);
        if (s == 0) break;
        nw = level_ranks<R>(sh.a, nw);
        level_lookup<R>(sh.a, idx, ip);
        s -= 6;
#pragma unroll
        for (int r = 0; r < R; ++r) idx[r] = idx[r] * 64 + ((col[r] >> s) & 63);
    }
    int cnt = 0;
    const unsigned long long* w64 = reinterpret_cast<const unsigned long long*>(sh.a.w);
#pragma unroll 1
    for (int i = 0; i < nw; i += BRM_WAVE) cnt += __popcll(w64[i + lane]);
    cnt = wave_sum(cnt);
    if (lane == 0) nnzrow[row] = cnt;
}

template <int R>
hipError_t rmed_count_t(const int* rows, int n, const RowArgs& a, int64_t* nnzrow, hipStream_t s) {
    const int64_t ch = launch_chunk(BRM_WAVE);
    for (int64_t b = 0; b < n; b += ch) {
        const int c = (int)std::min<int64_t>(ch, n - b);
        k_rmed_count<R><<<c, BRM_WAVE, 0, s>>>(rows + b, c, a, nnzrow);
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
        if constexpr (R >= 4) {
            if (mode == 1) {
                k_rmed<R, uint32_t, 1><<<c, BRM_WAVE, 0, s>>>(rows + b, c, a, o);
                continue;
            }
            if (mode == 2) {
                k_rmed<R, uint32_t, 2><<<c, BRM_WAVE, 0, s>>>(rows + b, c, a, o);
                continue;
            }
        }
        if constexpr (R <= 16) {
            if (narrow) k_rmed<R, uint32_t, 0><<<c, BRM_WAVE, 0, s>>>(rows + b, c, a, o);
            else k_rmed<R, uint64_t, 0><<<c, BRM_WAVE, 0, s>>>(rows + b, c, a, o);
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
    // wavefront ran faster than the workgroup LDS tier).  Otherwise 1024
    // products while 32-bit sort keys hold N columns beside 16 bits of
    // position and index, else 512.
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
