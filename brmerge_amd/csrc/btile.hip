// Column-tile group merge for long rows (the long-row engine where its
// tables pay; bmerge.hip has the engine without them).
//
// As in bmerge.hip one workgroup materialises one tree node from up to
// BGROUP_KMAX sorted child lists (B rows read in place and scaled, or nodes
// of the previous pass), in rounds that rank the round's columns with an LDS
// bitmap and sum each column's contributions by the aligned tree over list
// positions.  There a round loads windows of every child and takes the part
// below the smallest window end, about half of what it loads; here a round's
// columns are chosen first, so that it loads exactly what it takes:
//   - the columns are cut into nb blocks of about equal share of B's entries
//     (k_colblocks), and a table holds where each block begins in every B
//     row (k_btab); a node of one pass writes the same table row for itself,
//     from its bitmap ranks, for the next pass;
//   - wavefront 0, one child per lane, reads the table at eight block
//     boundaries ahead and takes the furthest with at most BT_W elements in
//     all children; a block too full for a round is cut by a search for a
//     column in every child.
// Products go from registers straight to their slot in their column's bucket:
// the bucket counters hold one 16-bit count per wavefront, so that a bucket
// fills nearly in list order, elements being numbered child by child.
//
// What bounds it: LDS instructions and the barriers of a round, while B stays
// in the caches (R-MAT of 2^18 rows); at 2^20 rows also HBM, 3.8 TB/s of it
// where a copy reaches 4.6.  Hence 2,048 elements a round in under 40 KB, four
// workgroups per CU (three: 44.4 ms against 38.9 on R-MAT, 2^18 rows); the
// next round's loads in flight over this round's sums, and the plan of the
// round after it by wavefront 0 while the others sum (37.6 ms to 35.2; it had
// been a fifth of a round).  The whole product with it, before and after:
// R-MAT of 2^18 rows, 16 per row 61.9 ms to 35.1; 2^14 rows 2.51 to 1.64.
#include <limits.h>
#include <stddef.h>

#include <algorithm>

#include "brm_device.h"
#include "bucket_sum.h"
#include "kernels.h"

namespace brm {
namespace {

constexpr int BT_NT = 256;
constexpr int BT_NW = BT_NT / BRM_WAVE;
constexpr int BT_W = 2048;             // elements of a round
constexpr int BT_IPT = BT_W / BT_NT;   // per thread
constexpr int BT_SPAN = 1 << 16;       // columns of a round
constexpr int BT_WORDS = BT_SPAN / 64;
constexpr int BT_WPT = BT_WORDS / BT_NT;
constexpr int BT_K = BGROUP_KMAX;
constexpr int BT_CAND = 8;             // block boundaries looked at per plan
// Buckets of more contributions than this are summed by 16 lanes (dense over
// the list ids) instead of by one thread.  R-MAT of 2^18 rows, ms at 4, 6, 8,
// 12, 16: 38.8, 37.8, 37.6, 38.4, 39.2.
constexpr int BT_THREAD_M = 8;
constexpr int BT_BIGMAX = BT_W / (BT_THREAD_M + 1) + 1;
constexpr int BT_MIDMAX = BT_W / 3 + 1;
static_assert(BT_K == BRM_WAVE && BT_NW == 4, "one child per lane, one count field per wavefront");
static_assert(BT_WPT == 4 && BT_IPT == 8, "16-byte LDS accesses per thread");

struct BtSmem {
    union {
        unsigned long long cnt[BT_W];  // per output: 16-bit counts of the four wavefronts, then their slots
        double val[BT_W];              // contributions, bucket by bucket
    };
    unsigned short ocol[BT_W];         // output columns less the round's first
    unsigned long long bm[BT_WORDS];   // bitmap of the round's columns; scratch of the big sums
    union {
        unsigned rank[BT_WORDS];       // bits before the low | before the high half of each word
        struct {                       // the output phase, when the ranks are dead
            unsigned short mid[BT_MIDMAX];           // outputs of 3 .. BT_THREAD_M contributions
            unsigned short big[BT_BIGMAX];           // outputs of more
        } q;
    };
    unsigned short off[BT_W + 2];      // bucket offsets
    unsigned char lid[BT_W + 8];       // list id of each contribution (read 8 at a time)
    // the window to fetch next: its non-empty children in order (scales and
    // list ids: of the window fetched last)
    const int* cptr[BT_K];             // element e of the window at cptr[q][e]
    const double* vptr[BT_K];
    double scale[BT_K];
    unsigned char clid[BT_K];
    alignas(8) unsigned mark[BT_W / 32];          // bit e: a child other than the first begins at element e + 1
    int wn, c_lo, bh;                  // elements, first column, last block boundary reached
    int nmid, nbig, bnext;
    int red_a[BT_NW], red_b[BT_IPT * BT_NW];
};
static_assert(sizeof(BtSmem) <= 160 * 1024 / 4, "four workgroups per CU");
static_assert(offsetof(BtSmem, bm) % 16 == 0 && offsetof(BtSmem, rank) % 16 == 0,
              "16-byte accesses");

// The workspace buffers that hold the nodes of the pass before.
struct BtBufs {
    int *col0, *col1;
    double *val0, *val1;
};

// How far each child has come: wavefront 0, one child per lane.
struct BtPlan {
    const int* tp;      // the child's table row: element index at every block boundary
    int cur, end;       // next element, one past the last
    int cand[BT_CAND];  // element index at boundaries b0 + g, b0 + 2 g, ...
    int cbv;            // lane i: column of the i-th of them
    int b0;             // last boundary reached (uniform, as all below)
    int c_cur;          // first column of the next round
    int g;              // boundaries per step
    int64_t left;       // elements left in all children
    // the planned window's scales and list ids, for bt_scales
    double scale;
    int lid, q;         // q: the child's place in the window, -1 for none
};

__device__ __forceinline__ void bt_candidates(BtPlan& p, int k, const int* __restrict__ cb, int nb) {
    p.cbv = cb[min(p.b0 + (min(lane_id(), BT_CAND - 1) + 1) * p.g, nb)];
    if (lane_id() < k) {
#pragma unroll
        for (int i = 0; i < BT_CAND; ++i) p.cand[i] = p.tp[min(p.b0 + (i + 1) * p.g, nb)];
    }
}

// Minimum over the wavefront (DPP prefix minimum, then the last lane).
__device__ __forceinline__ int wave_min(int x) {
    x = min(x, dpp_mov<0x111, 0xF>(x, INT_MAX));  // row_shr:1
    x = min(x, dpp_mov<0x112, 0xF>(x, INT_MAX));  // row_shr:2
    x = min(x, dpp_mov<0x114, 0xF>(x, INT_MAX));  // row_shr:4
    x = min(x, dpp_mov<0x118, 0xF>(x, INT_MAX));  // row_shr:8
    x = min(x, dpp_mov<0x142, 0xA>(x, INT_MAX));  // row_bcast15 into rows 1 and 3
    x = min(x, dpp_mov<0x143, 0xC>(x, INT_MAX));  // row_bcast31 into rows 2 and 3
    return wave_last(x);
}

// First element of [lo, hi) whose column is at least c (hi when none is).
__device__ __forceinline__ int bt_lower(const int* col, int lo, int hi, int c) {
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (col[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Chooses the next round and publishes its window but for the scales and list
// ids, which the round before still reads (wavefront 0; seen by the others
// after the next barrier).  wn = 0 when nothing is left.
__device__ __forceinline__ void bt_plan(BtSmem& g, BtPlan& p, const Child* __restrict__ children, int k,
                                        const RowArgs& a, const BtBufs& bufs, const int* __restrict__ cb, int nb) {
    const int lane = lane_id();
    // where the child's elements are: read again by every plan (from L1) rather
    // than held in registers across the round
    const Child& ch = children[min(lane, k - 1)];
    const Src src = ch.src;
    const int lid = ch.lid;
    const bool virt = src.kind == SRC_VIRTUAL;
    const int* ccol = virt ? a.bcol : (src.buf ? bufs.col1 : bufs.col0) + src.off;
    const double* cval = virt ? a.bval : (src.buf ? bufs.val1 : bufs.val0) + src.off;
    const int N = a.N;
    int hi = p.cur, bh = p.b0, c_hi = p.c_cur, total = 0;
    int c_lo = p.c_cur, taken = 0;
    while (p.left > 0) {
        if (p.left <= BT_W && N - p.c_cur <= BT_SPAN) {
            hi = p.end;
            bh = nb;
            c_hi = N;
        } else {
            int nf = 0;  // boundaries with at most BT_W elements before them (the counts ascend)
            int tot0 = 0;
#pragma unroll
            for (int i = 0; i < BT_CAND; ++i) {
                const int s = wave_sum(lane < k ? min(p.cand[i] - p.cur, 1 << 24) : 0);
                if (i == 0) tot0 = s;
                nf += s <= BT_W ? 1 : 0;
            }
            const int cbv = p.cbv;
            const int ns = __popcll(__ballot(lane < BT_CAND && cbv - p.c_cur <= BT_SPAN));
            const int best = min(nf, ns) - 1;
            if (best >= 0) {
                hi = p.cand[0];
#pragma unroll
                for (int i = 1; i < BT_CAND; ++i) {
                    hi = i <= best ? p.cand[i] : hi;
                    asm volatile("" : "+v"(hi));  // selects, not an indexed copy of cand in scratch memory
                }
                bh = min(p.b0 + (best + 1) * p.g, nb);
                c_hi = __builtin_amdgcn_readlane(cbv, best);
                taken = (best + 1) * p.g;
            } else if (p.g > 1) {
                p.g = max(1, p.g / BT_CAND);
                bt_candidates(p, k, cb, nb);
                continue;
            } else {
                // the next block alone is too full, or too wide: a part of
                // it, from the first column any child has
                p.c_cur = c_lo = max(p.c_cur, wave_min(p.cur < p.end ? ccol[p.cur] : INT_MAX));
                const int c_end = __builtin_amdgcn_readlane(cbv, 0);
                int w = c_end - p.c_cur;
                if (tot0 > BT_W) w = (int)((double)w * (0.8 * BT_W / tot0));
                w = min(max(w, 1), BT_SPAN);
                // one column (of at most BT_K children) always fits; a block
                // that ends before the first column holds nothing
                for (hi = p.cur, c_hi = c_end; c_end > p.c_cur;) {
                    c_hi = p.c_cur + w;
                    hi = lane < k ? bt_lower(ccol, p.cur, p.cand[0], c_hi) : p.cur;
                    if (wave_sum(min(hi - p.cur, 1 << 24)) <= BT_W || w == 1) break;
                    w >>= 1;
                }
                bh = c_hi >= c_end ? min(p.b0 + 1, nb) : p.b0;
            }
        }
        if (lane >= k) hi = p.cur;
        total = wave_sum(hi - p.cur);
        if (total > 0) break;
        // nothing in these columns: the round begins behind them
        p.b0 = bh;
        p.c_cur = c_lo = max(p.c_cur, c_hi);
        bt_candidates(p, k, cb, nb);
    }
    const int len = hi - p.cur;
    const int o = wave_incl_scan(len) - len;
    const uint64_t nz = __ballot(len > 0);
    g.mark[lane] = 0u;
    p.q = -1;
    static_assert(BT_W / 32 == BRM_WAVE, "one mark word per lane");
    wave_lds_sync();
    if (len > 0) {
        const int q = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(nz >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)nz, 0u));
        g.cptr[q] = ccol + (p.cur - o);
        g.vptr[q] = cval + (p.cur - o);
        p.scale = virt ? src.scale : 1.0;  // a product by 1.0 is the value itself
        p.lid = lid;
        p.q = q;
        if (o > 0) atomicOr(&g.mark[(o - 1) >> 5], 1u << ((o - 1) & 31));
    }
    if (lane == 0) {
        g.wn = total;
        g.c_lo = c_lo;
        g.bh = bh;
    }
    p.cur = hi;
    p.left -= total;
    // the next plan's boundaries: eight steps to a sixth more than a round, at
    // this round's elements per block
    if (taken > 0 && total > 0)
        p.g = min((int)((float)taken * (1.17f * BT_W / BT_CAND) / (float)total) + 1, nb);
    p.c_cur = max(p.c_cur, c_hi);
    p.b0 = bh;
    if (p.left > 0) bt_candidates(p, k, cb, nb);  // for the plan of the round after
}

__device__ __forceinline__ void bt_scales(BtSmem& g, const BtPlan& p) {
    if (p.q >= 0) {
        g.scale[p.q] = p.scale;
        g.clid[p.q] = (unsigned char)p.lid;
    }
}

// The lane, and the thread, as values the compiler does not carry from one
// phase of a round to the next: left alone it keeps every address and bound
// that derives from them in a register.
__device__ __forceinline__ int bt_lane() {
    int l = lane_id();
    asm volatile("" : "+v"(l));
    return l;
}
__device__ __forceinline__ int bt_thread() {
    int l = (int)threadIdx.x;
    asm volatile("" : "+v"(l));
    return l;
}

// Element bt_first(wv, i) + lane (0 <= i < BT_IPT) belongs to lane `lane` of
// wavefront wv: each wavefront owns one contiguous run, so that elements are
// in child order across the wavefronts too.
__device__ __forceinline__ int bt_first(int wv, int i) { return wv * (BT_IPT * BRM_WAVE) + i * BRM_WAVE; }

// The published window's elements into registers; rq: the element's child.
// Elements at or past wn repeat the last one.
__device__ __forceinline__ void bt_fetch(const BtSmem& g, int wn, int wv, int (&rc)[BT_IPT], double (&rv)[BT_IPT],
                                         int (&rq)[BT_IPT]) {
    const int lane = bt_lane();
    const int pc = __popc(g.mark[lane]);
    const int before = wave_incl_scan(pc) - pc;
#pragma unroll
    for (int i = 0; i < BT_IPT; ++i) {
        const int wd = wv * BT_IPT + i;
        const unsigned long long m = reinterpret_cast<const unsigned long long*>(g.mark)[wd];
        rq[i] = (int)__builtin_amdgcn_mbcnt_hi(
            (unsigned)(m >> 32),
            __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)__builtin_amdgcn_readlane(before, 2 * wd)));
    }
#pragma unroll
    for (int i = 0; i < BT_IPT; ++i) {
        const int e = min(bt_first(wv, i) + lane, wn - 1);
        rc[i] = g.cptr[rq[i]][e];
        rv[i] = g.vptr[rq[i]][e];
    }
}

template <int CTRL>
__device__ __forceinline__ double dpp_d(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xF, 0xF, false),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xF, 0xF, false));
}

// Sums of four buckets by one wavefront, one per row of 16 lanes (m = 0: no
// bucket): each row places its contributions by list id in BT_K slots of its
// own, lanes add their four slots, and the tree over the row's lanes is
// finished with DPP moves; the sums end in each row's last lane.  Slots
// without a contribution hold -0.0 (on entry and on return): x + -0.0 is x for
// every x, zeros of both signs included, and -0.0 + -0.0 is -0.0, so a node
// with one present child passes it through by a plain add.  (With presence
// flags a level took a dozen instructions instead of three.)
__device__ __forceinline__ double bt_wave_sum4(const double* val, const unsigned char* lid, int s, int m,
                                               double* dense) {
    const int hl = lane_id() & 15;
    double* dn = dense + (lane_id() >> 4) * BT_K;
    static_assert(BT_K == 64, "four slots per lane");
    for (int i = hl; i < m; i += 16) dn[lid[s + i]] = val[s + i];
    wave_lds_sync();
    double2* d2 = reinterpret_cast<double2*>(dn) + 2 * hl;
    const double2 x = d2[0], y = d2[1];
    wave_lds_sync();
    d2[0] = d2[1] = double2{-0.0, -0.0};
    double v = fadd(fadd(x.x, x.y), fadd(y.x, y.y));
    // lane i takes lane i - S; only lanes i % (2 S) == 2 S - 1 are used further
    v = fadd(dpp_d<0x111>(v), v);  // row_shr:1
    v = fadd(dpp_d<0x112>(v), v);  // row_shr:2
    v = fadd(dpp_d<0x114>(v), v);  // row_shr:4
    v = fadd(dpp_d<0x118>(v), v);  // row_shr:8
    wave_lds_sync();
    return v;
}

__global__ __launch_bounds__(BT_NT, 4) void k_btile(const GroupTask* __restrict__ tasks,
                                                    const int* __restrict__ order,
                                                    const Child* __restrict__ children, RowArgs a, TileTabs tt,
                                                    BtBufs bufs, int64_t* __restrict__ slots, int64_t* counters, OutArgs o) {
    extern __shared__ __align__(16) unsigned char smraw[];
    BtSmem& g = *reinterpret_cast<BtSmem*>(smraw);
    const int t = threadIdx.x, lane = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(t / BRM_WAVE);
    const GroupTask T = tasks[order ? order[blockIdx.x] : (int)blockIdx.x];
    const int k = T.nchild, nb = tt.nb;
    BtPlan p{};
    int64_t in_total = 0;
    if (wv == 0) {
        if (lane < k) {
            const Child c = children[T.cbase + lane];
            const bool virt = c.src.kind == SRC_VIRTUAL;
            p.tp = (virt ? tt.brow : tt.node) + (int64_t)c.tab * (nb + 1);
            p.cur = p.tp[0];
            p.end = p.tp[nb];
        }
        in_total = wave_sum((int64_t)(p.end - p.cur));
        p.left = in_total;
        p.g = (int)min((int64_t)nb, max((int64_t)1, (int64_t)nb * (BT_W + BT_W / 4) / (BT_CAND * max(in_total, (int64_t)1))));
        bt_candidates(p, k, tt.cb, nb);
        bt_plan(g, p, children + T.cbase, k, a, bufs, tt.cb, nb);
        bt_scales(g, p);
    }
    if (t == 0) g.nbig = g.nmid = g.bnext = 0;
#pragma unroll
    for (int i = 0; i < BT_WPT; ++i) g.bm[t * BT_WPT + i] = 0ull;

    int* dc;
    double* dv;
    int64_t dcap = INT64_MAX;
    int* own = nullptr;  // this node's table row
    if (T.final_dst) {
        dc = o.ccol + T.dst_off;
        dv = o.cval + T.dst_off;
        if (!o.upper) dcap = o.crpt[T.row + 1] - o.crpt[T.row];
    } else {
        dc = (T.dst_buf ? bufs.col1 : bufs.col0) + T.dst_off;
        dv = (T.dst_buf ? bufs.val1 : bufs.val0) + T.dst_off;
        own = tt.node + T.tab * (nb + 1);
        if (t == 0) own[0] = 0;
    }
    __syncthreads();
    int rc[BT_IPT], rq[BT_IPT];
    double rv[BT_IPT];
    int wn = g.wn, c_lo = g.c_lo, bh = g.bh;
    if (wn > 0) bt_fetch(g, wn, wv, rc, rv, rq);
    __syncthreads();
    if (wv == 0 && wn > 0) bt_plan(g, p, children + T.cbase, k, a, bufs, tt.cb, nb);
    int64_t out_n = 0;
    int rounds = 0, bw = 0;  // bw: last boundary written to `own`
    while (wn > 0) {
        rounds++;
        // ---- products; the round's columns
        {
            const int ln = bt_lane();
#pragma unroll
            for (int i = 0; i < BT_IPT; ++i) {
                rv[i] = fmul(g.scale[rq[i]], rv[i]);
                rq[i] = g.clid[rq[i]];
                rc[i] -= c_lo;
                if (ln < wn - bt_first(wv, i))
                    atomicOr(reinterpret_cast<unsigned*>(g.bm) + (rc[i] >> 5), 1u << (rc[i] & 31));
            }
        }
        // the columns only: their LDS addresses are formed again below
#pragma unroll
        for (int i = 0; i < BT_IPT; ++i) asm volatile("" : "+v"(rc[i]));
        __syncthreads();
        if (wv == 0) bt_scales(g, p);  // of the next window
        // ---- ranks of the bitmap words
        int nout;
        {
            const int th = bt_thread();
            unsigned pc[2 * BT_WPT], sum = 0u;
            {
                const uint4* w = reinterpret_cast<const uint4*>(g.bm) + th * (BT_WPT / 2);
                const uint4 x = w[0], y = w[1];
                const unsigned h[2 * BT_WPT] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
                for (int i = 0; i < 2 * BT_WPT; ++i) {
                    pc[i] = sum;
                    sum += __popc(h[i]);
                }
            }
            const unsigned ex = (unsigned)block_excl_scan_1b<BT_NT>((int)sum, g.red_a, &nout) * 0x10001u;
            uint4 r;
            r.x = ex + (pc[0] | (pc[1] << 16));
            r.y = ex + (pc[2] | (pc[3] << 16));
            r.z = ex + (pc[4] | (pc[5] << 16));
            r.w = ex + (pc[6] | (pc[7] << 16));
            reinterpret_cast<uint4*>(g.rank)[th] = r;
#pragma unroll
            for (int i = 0; i < BT_IPT; ++i)
                if (i * BT_NT < nout) g.cnt[i * BT_NT + th] = 0ull;  // uniform
        }
        __syncthreads();
        // ---- output positions; contributions per output and wavefront
        const unsigned short* rk = reinterpret_cast<const unsigned short*>(g.rank);
        const unsigned* bm32 = reinterpret_cast<const unsigned*>(g.bm);
        int pos[BT_IPT];
#pragma unroll
        for (int i = 0; i < BT_IPT; ++i) pos[i] = rk[rc[i] >> 5] + popc_below(bm32[rc[i] >> 5], (unsigned)rc[i]);
        const int lnp = bt_lane();
#pragma unroll
        for (int i = 0; i < BT_IPT; ++i) {
            if (lnp < wn - bt_first(wv, i)) {
                unsigned* half = reinterpret_cast<unsigned*>(g.cnt) + (wv >> 1);  // this wavefront's half word
                const int arr = (int)((atomicAdd(half + 2 * pos[i], 1u << (16 * (wv & 1))) >> (16 * (wv & 1))) & 0xffffu);
                if (arr == 0) g.ocol[pos[i]] = (unsigned short)rc[i];
                pos[i] |= (arr << 16) | (rq[i] << 24);  // at most BT_K arrivals
            }
        }
        // ---- where the blocks that begin in this round do in the node
        if (own) {
            for (int b = bw + 1 + t; b <= bh; b += BT_NT) {
                const int x = tt.cb[b] - c_lo;
                int r = nout;
                if (x <= 0) r = 0;
                else if (x < BT_SPAN) r = rk[x >> 5] + popc_below(bm32[x >> 5], (unsigned)x);
                own[b] = (int)out_n + r;
            }
        }
        bw = max(bw, bh);
        __syncthreads();
        // ---- bucket offsets: step i of wavefront wv holds 64 consecutive
        // outputs from (4 i + wv) * 64 (conflict-free LDS; eight outputs in a row
        // per thread would be 16 ways), two steps to a wave scan; every
        // wavefront's first slot of each bucket replaces its count
        {
            const int ln = bt_lane();
            int inc[BT_IPT / 2];
#pragma unroll
            for (int h = 0; h < BT_IPT / 2; ++h) {
                inc[h] = 0;
                if (2 * h * BT_NT < nout) {  // uniform
                    int m2[2];
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int oi = ((2 * h + j) * BT_NW + wv) * BRM_WAVE + ln;
                        const unsigned long long x = oi < nout ? g.cnt[oi] : 0ull;
                        const unsigned y = (unsigned)x + (unsigned)(x >> 32);
                        m2[j] = (int)((y & 0xffffu) + (y >> 16));
                    }
                    inc[h] = wave_incl_scan(m2[0] | (m2[1] << 16));
                    if (ln == BRM_WAVE - 1) {
                        g.red_b[2 * h * BT_NW + wv] = inc[h] & 0xffff;
                        g.red_b[(2 * h + 1) * BT_NW + wv] = (int)((unsigned)inc[h] >> 16);
                    }
                }
            }
            __syncthreads();
            const int steps = (nout + BT_NT - 1) / BT_NT;
            const int v = ln < (steps + (steps & 1)) * BT_NW ? g.red_b[ln] : 0;
            const int pre = wave_incl_scan(v) - v;
            if (t == 0) g.off[nout] = (unsigned short)wn;
#pragma unroll
            for (int h = 0; h < BT_IPT / 2; ++h) {
                if (2 * h * BT_NT < nout) {  // uniform
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int oi = ((2 * h + j) * BT_NW + wv) * BRM_WAVE + ln;
                        if (oi < nout) {
                            const unsigned long long x = g.cnt[oi];
                            const unsigned y = (unsigned)x + (unsigned)(x >> 32);
                            const int m = (int)((y & 0xffffu) + (y >> 16));
                            const int ex = __builtin_amdgcn_readlane(pre, (2 * h + j) * BT_NW + wv) +
                                           (j ? (int)((unsigned)inc[h] >> 16) : inc[h] & 0xffff) - m;
                            // exclusive prefix over the four counts (0, c0,
                            // c0 + c1, c0 + c1 + c2), plus the bucket's offset
                            unsigned long long f = x << 16;
                            f += f << 16;
                            f += f << 32;
                            g.cnt[oi] = f + (((unsigned long long)((unsigned)ex * 0x10001u) << 32) |
                                             ((unsigned)ex * 0x10001u));
                            g.off[oi] = (unsigned short)ex;
                        }
                    }
                }
            }
        }
        __syncthreads();
        // ---- contributions to their slots (the values take the counters' place)
#pragma unroll
        for (int i = 0; i < BT_IPT; ++i)
            pos[i] = (pos[i] & 0x3f000000) |
                     (reinterpret_cast<const unsigned short*>(g.cnt)[4 * (pos[i] & 0xffff) + wv] + ((pos[i] >> 16) & 0xff));
        __syncthreads();
        {
            const int ln = bt_lane();
#pragma unroll
            for (int i = 0; i < BT_IPT; ++i) {
                if (ln < wn - bt_first(wv, i)) {
                    g.val[pos[i] & 0xffff] = rv[i];
                    g.lid[pos[i] & 0xffff] = (unsigned char)(pos[i] >> 24);
                }
            }
        }
        const int nwn = g.wn, nc_lo = g.c_lo, nbh = g.bh;
        if (nwn > 0) bt_fetch(g, nwn, wv, rc, rv, rq);
        __syncthreads();
        // ---- one output per thread (coalesced stores) for one or two
        // contributions; outputs with more are queued, so that the lanes of a
        // wavefront take the same path
        for (int oi = bt_thread(); oi < nout; oi += BT_NT) {
            const int s = g.off[oi];
            const int m = g.off[oi + 1] - s;
            if (m > 2) {
                if (m > BT_THREAD_M) g.q.big[atomicAdd(&g.nbig, 1)] = (unsigned short)oi;
                else g.q.mid[atomicAdd(&g.nmid, 1)] = (unsigned short)oi;
                continue;
            }
            const int s1 = s + m - 1;
            const double v0 = g.val[s], v1 = g.val[s1];
            const unsigned l0 = g.lid[s], l1 = g.lid[s1];
            const double v = m == 2 ? (l0 < l1 ? fadd(v0, v1) : fadd(v1, v0)) : v0;
            const int64_t q = out_n + oi;
            if (q < dcap) {
                dc[q] = c_lo + (int)g.ocol[oi];
                dv[q] = v;
            }
        }
        __syncthreads();
        // ---- wavefront 0 plans the round after the next, the others sum the
        // buckets of 3 to BT_THREAD_M; all of them then the larger ones
        if (wv == 0) {
            if (nwn > 0) bt_plan(g, p, children + T.cbase, k, a, bufs, tt.cb, nb);
        } else {
            const int nmid = g.nmid;
            for (int b = bt_thread() - BRM_WAVE; b < nmid; b += BT_NT - BRM_WAVE) {
                const int oi = g.q.mid[b];
                const int s = g.off[oi];
                const double v = rb_bucket_sum(g.lid + s, g.val + s, g.off[oi + 1] - s);
                const int64_t q = out_n + oi;
                if (q < dcap) {
                    dc[q] = c_lo + (int)g.ocol[oi];
                    dv[q] = v;
                }
            }
        }
        {
            // the bitmap is free until the next round: each wavefront's share
            // is its scratch; then cleared
            double* dense = reinterpret_cast<double*>(&g.bm[wv * (BT_WORDS / BT_NW)]);
            static_assert(4 * BT_K <= BT_WORDS / BT_NW, "scratch fits a wavefront's share");
            const int nbig = g.nbig;
            if (nbig > 0) {
                double2* d2 = reinterpret_cast<double2*>(dense) + 2 * lane;
                d2[0] = d2[1] = double2{-0.0, -0.0};
                wave_lds_sync();
                for (;;) {  // four at a time, claimed from a shared counter
                    int b = 0;
                    if (lane == 0) b = atomicAdd(&g.bnext, 4);
                    b = __builtin_amdgcn_readfirstlane(b);
                    if (b >= nbig) break;
                    const int bi = b + (lane >> 4);
                    const int oi = bi < nbig ? g.q.big[bi] : 0;
                    const int s = g.off[oi];
                    const int m = bi < nbig ? g.off[oi + 1] - s : 0;
                    const double v = bt_wave_sum4(g.val, g.lid, s, m, dense);
                    const int64_t q = out_n + oi;
                    if ((lane & 15) == 15 && m > 0 && q < dcap) {
                        dc[q] = c_lo + (int)g.ocol[oi];
                        dv[q] = v;
                    }
                }
            }
            static_assert(BT_WPT * BRM_WAVE == BT_WORDS / BT_NW, "a wavefront clears its own bitmap words");
#pragma unroll
            for (int i = 0; i < BT_WPT / 2; ++i)
                reinterpret_cast<uint4*>(g.bm)[bt_thread() * (BT_WPT / 2) + i] = uint4{0u, 0u, 0u, 0u};
        }
        out_n += nout;
        wn = nwn;
        c_lo = nc_lo;
        bh = nbh;
        __syncthreads();
        if (t == 0) g.nbig = g.nmid = g.bnext = 0;  // read by every wavefront before the barrier
    }
    if (own)
        for (int b = bw + 1 + t; b <= nb; b += BT_NT) own[b] = (int)out_n;
    if (t == 0) {
        if (T.final_dst) {
            if (o.upper) o.rowlen[T.row] = out_n;
            else if (out_n != dcap) atomicOr(o.err, (int)DERR_COUNT_MISMATCH);
        } else {
            slots[T.slot] = out_n;
        }
        atomicAdd((unsigned long long*)&counters[CNT_GRP_IN], (unsigned long long)in_total);
        atomicAdd((unsigned long long*)&counters[CNT_GRP_OUT], (unsigned long long)out_n);
        atomicAdd((unsigned long long*)&counters[CNT_ROUNDS], (unsigned long long)rounds);
    }
}

// ---------------------------------------------------------------- tables
// Column blocks of about equal share of B's entries: cb[0] = 0 .. cb[nb] = N,
// non-decreasing, from a histogram of evenly spaced entries over CB_BINS equal
// column bins (one workgroup).  Which columns a block holds is a matter of
// speed only.
constexpr int CB_NT = 1024;
constexpr int CB_BINS = 1 << 15;
constexpr int CB_SAMPLES = 1 << 16;

__global__ __launch_bounds__(CB_NT) void k_colblocks(RowArgs a, int shift, int nb, int* __restrict__ cb) {
    extern __shared__ __align__(16) unsigned char smraw[];
    int* bins = reinterpret_cast<int*>(smraw);
    int* red = bins + CB_BINS;
    const int t = threadIdx.x;
    for (int i = t; i < CB_BINS; i += CB_NT) bins[i] = 0;
    __syncthreads();
    const int64_t nnz = a.brpt[a.K];
    const int S = (int)min(nnz, (int64_t)CB_SAMPLES);
    for (int i0 = t; i0 < S; i0 += 8 * CB_NT) {
        int c[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) c[j] = a.bcol[(int64_t)min(i0 + j * CB_NT, S - 1) * nnz / S];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (i0 + j * CB_NT < S) atomicAdd(&bins[c[j] >> shift], 1);
    }
    __syncthreads();
    constexpr int PER = CB_BINS / CB_NT;
    int sum = 0;
    for (int i = 0; i < PER; ++i) sum += bins[t * PER + i];
    int tot;
    int64_t before = block_excl_scan<CB_NT>(sum, red, &tot);
    for (int i = 0; i < PER; ++i) {
        const int64_t after = before + bins[t * PER + i];
        const int64_t c = min(((int64_t)(t * PER + i) + 1) << shift, (int64_t)a.N);
        for (int64_t q = before * nb / S + 1; q <= after * nb / S; ++q)
            if (q < nb) cb[q] = (int)c;
        before = after;
    }
    if (t == 0) {
        cb[0] = 0;
        cb[nb] = a.N;
    }
}

// Table rows of B: tab[r * (nb + 1) + b] = index in B of row r's first entry
// with a column of at least cb[b].  One wavefront per row, 64 boundaries per
// step, each by a binary search in the row.
__global__ __launch_bounds__(BT_NT) void k_btab(RowArgs a, const int* __restrict__ cb, int nb, int64_t r0,
                                                int* __restrict__ tab) {
    const int64_t r = r0 + (int64_t)blockIdx.x * BT_NW + threadIdx.x / BRM_WAVE;
    if (r >= a.K) return;
    const int b0 = a.brpt[r], b1 = a.brpt[r + 1];
    int* row = tab + r * (nb + 1);
    for (int b = lane_id(); b <= nb; b += BRM_WAVE) row[b] = b0 < b1 ? bt_lower(a.bcol, b0, b1, cb[b]) : b0;
}

}  // namespace

// Boundaries worth their table for long rows of long_ip products.  An entry
// of the table costs about 3 ps and a product 8 ps, so the table is held to
// an eighth of the products (5 % of the time) and 1,024 blocks; finer blocks
// fill the rounds no better.  Measured by number of blocks, ms (engine
// without tables | 128, 256, 512, 1024, 2048, 4096):
//   2^18 rows, 3.8e9 long products   62.0 | 36.3, 35.5, 35.3, 35.1, 36.5, 39.1
//   2^17 rows, 1.3e9                 26.3 | 15.3, 15.0, 14.8, 14.8, 15.4, 16.5
//   2^14 rows, 5.1e7                 2.51 | 1.63, 1.63, 1.64, 1.66, 1.72, 1.81
// With fewer than 64 blocks' worth of products the engine without tables runs.
int tile_blocks(int64_t long_ip, int K, int N) {
    int nb = 1024;
    while (nb >= 64 && (int64_t)nb * std::max(K, 1) > long_ip / 8) nb >>= 1;
    return nb >= 64 && N >= 1 ? nb : 0;
}

hipError_t launch_tile_tables(const RowArgs& a, int nb, int* cb, int* brow, hipStream_t s) {
    constexpr int lds = (CB_BINS + CB_NT / BRM_WAVE + 2) * (int)sizeof(int);
    static SmemLimit lim;
    if (hipError_t e = lim.raise((const void*)k_colblocks, lds); e != hipSuccess) return e;
    int shift = 0;
    while (((int64_t)a.N - 1) >> shift >= CB_BINS) ++shift;
    {
        ProfScope ps_("k_colblocks", s);
        k_colblocks<<<1, CB_NT, lds, s>>>(a, shift, nb, cb);
    }
    {
        ProfScope ps_("k_btab", s);
        const int64_t ch = launch_chunk(BRM_WAVE) / BT_NW * BT_NW;
        const int64_t step = std::max<int64_t>(ch, BT_NW);
        for (int64_t r = 0; r < a.K; r += step)
            k_btab<<<(unsigned)((std::min<int64_t>(step, a.K - r) + BT_NW - 1) / BT_NW), BT_NT, 0, s>>>(a, cb, nb, r,
                                                                                                       brow);
    }
    return hipGetLastError();
}

hipError_t launch_btile(const GroupTask* tasks, int64_t n, const Child* children, const RowArgs& a,
                        const TileTabs& tt, int* const ws_col[2], double* const ws_val[2], int64_t* slots,
                        int64_t* counters, const OutArgs& o, hipStream_t s, const int* order) {
    if (n <= 0) return hipSuccess;
    static SmemLimit lim;
    if (hipError_t e = lim.raise((const void*)k_btile, (int)sizeof(BtSmem)); e != hipSuccess) return e;
    {
        ProfScope ps_("k_btile", s);
        const int64_t ch = launch_chunk(BT_NT);
        for (int64_t b = 0; b < n; b += ch)
            k_btile<<<(unsigned)std::min<int64_t>(ch, n - b), BT_NT, sizeof(BtSmem), s>>>(
                order ? tasks : tasks + b, order ? order + b : nullptr, children, a, tt,
                BtBufs{ws_col[0], ws_col[1], ws_val[0], ws_val[1]}, slots, counters, o);
    }
    return hipGetLastError();
}

}  // namespace brm
